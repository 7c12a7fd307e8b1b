"""The Python extension of the linears (relax_amd/_calls.so): it is used for the torch it was compiled for, and without it the linears
take the general path."""
import sys
import types

import pytest

torch = pytest.importorskip("torch")


@pytest.fixture
def fresh(monkeypatch):
    import relax_amd
    from relax_amd import _lib

    monkeypatch.setattr(_lib, "_calls", None)
    monkeypatch.delattr(relax_amd, "_calls", raising=False)
    return _lib


def test_it_is_used(fresh):
    m = fresh.calls()
    assert m.torch_version == str(torch.__version__)
    assert fresh.calls() is m


@pytest.mark.parametrize("module", [None, types.ModuleType("_calls"), types.SimpleNamespace(torch_version="0.0.0")],
                         ids=["missing", "of unknown version", "of another torch"])
def test_without_it_every_call_is_left_to_the_general_path(fresh, monkeypatch, module):
    import relax_amd

    monkeypatch.setitem(sys.modules, "relax_amd._calls", module)
    if module is not None:
        monkeypatch.setattr(relax_amd, "_calls", module, raising=False)
    with pytest.warns(RuntimeWarning, match="relax_amd.build"):
        m = fresh.calls()
    assert fresh.calls() is m  # (and no second warning)
    assert m.q4g32_linear(*range(6)) is None and m.fpA_intB_gemm(*range(11)) is None and m.gptq_linear(*range(9)) is None
    # what the general path refuses is refused with its own message
    from relax_amd import ops

    w = torch.zeros(8, 4, dtype=torch.int32)
    with pytest.raises(ValueError, match="device tensor"):
        ops.q4g32_linear(w, w, w)
