"""SAF3R_FAULT_INJECT by an entry's name also fails the forms of that entry that take host lists or typed parameters,
which are the ones the plugin calls (CPU: an injected entry fails before it looks at its arguments)."""
from importlib import import_module

import pytest

FORMS = {"saf3r_pack_qkv_typed": "saf3r_pack_qkv", "saf3r_probe_scores_host": "saf3r_probe_scores",
         "saf3r_keyset_build_host": "saf3r_keyset_build", "saf3r_keyset_gather_host": "saf3r_keyset_gather"}


@pytest.mark.parametrize("form", sorted(FORMS))
def test_injection_reaches_every_form_of_an_entry(pkg, monkeypatch, form):
    lib = import_module(pkg.__name__ + "._lib").load()

    def call(name):
        fn = getattr(lib, name)
        return fn(*[None if t.__name__ == "c_void_p" else 0 for t in fn.argtypes])
    base = FORMS[form]
    for named in (base, form, "all"):
        monkeypatch.setenv("SAF3R_FAULT_INJECT", named)
        assert call(form) == 4 and form.encode() in lib.saf3r_last_error(), named
        assert call(base) == (1 if named == form else 4), named
    for other in ("saf3r_pack", "saf3r_keyset", base + "_", form + "_host", "_host"):
        monkeypatch.setenv("SAF3R_FAULT_INJECT", other)
        assert call(form) == 1 and call(base) == 1, other
