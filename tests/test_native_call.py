"""The two ways into the C ABI (aiter_amd/_lib.py): the native caller and
ctypes take the same arguments and report the same errors.  On the CPU: every
call here is refused before anything is launched."""
import ctypes

import pytest
import torch

from aiter_amd import _lib


class _Sub(torch.Tensor):
    pass


def _outcome(name, args):
    try:
        _lib.call(name, *args)
    except Exception as e:
        return type(e), str(e)
    return None


X = torch.zeros(4, 64, dtype=torch.bfloat16)
CALLS = [("moe_sum", (X, X)), ("moe_sum", (X, None)), ("moe_sum", (None, None)), ("moe_sum", (X,)),
         ("moe_sum", (X, 1.5)), ("moe_sum", (X.as_subclass(_Sub), X)), ("moe_sum", (X.to(torch.complex64), X)),
         ("moe_sum", (torch.zeros([1] * 9), X)), ("moe_sum", (X[:0], X[:, ::2])),
         ("moe_sum", (X.to("meta"), X)), ("dynamic_mxfp4_quant", (X, X, X, 1 << 40)),
         ("dynamic_mxfp4_quant", (X, X, X, True)), ("dynamic_mxfp4_quant", (X, X, X, 1.0)),
         ("gemm_a16w16_asm", (X, X, X, None, None, 0, "näme", 1)),
         ("gemm_a16w16_asm", (X, X, X, None, None, 0, "\ud800", 1)),
         ("gemm_a4w4_asm", (X, X, X, X, X, "", None, 1, 0.5, 1, 0)),
         ("gemm_a4w4_asm", (X, X, X, X, X, "", None, "1", 0.5, 1, 0))]


@pytest.mark.parametrize("i", range(len(CALLS)))
def test_native_and_ctypes_agree(i, monkeypatch):
    name, args = CALLS[i]
    _lib.lib()
    native = _outcome(name, args)
    monkeypatch.delitem(_lib._native, name)
    assert native is not None and native == _outcome(name, args)


def test_every_launching_entry_is_native():
    _lib.lib()
    launching = {n for n, (args, _) in _lib.SIGNATURES.items() if args and args[-1] is ctypes.c_void_p and
                 args[0] is _lib._T and not n.startswith("hbm_")}
    assert launching == set(_lib._native)


def test_missing_native_module_raises(monkeypatch):
    def missing(name):
        raise ImportError("no such module")

    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(_lib.importlib, "import_module", missing)
    with pytest.raises(RuntimeError, match="_native.so is not built"):
        _lib.lib()


@pytest.mark.parametrize("version,ok", [(torch.__version__, True), ("1.2.3+rocm7.0", False)])
def test_module_of_another_torch_raises(version, ok, monkeypatch):
    """The module reads torch's C++ objects: one that was compiled for another
    minor version is refused."""
    _lib.lib()
    real = _lib.importlib.import_module("aiter_amd._native")
    assert real.torch_version == torch.__version__

    class Other:
        torch_version = version

    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(_lib.importlib, "import_module", lambda name: Other)
    if ok:
        _lib.lib()
    else:
        with pytest.raises(RuntimeError, match="built for torch 1.2.3"):
            _lib.lib()
