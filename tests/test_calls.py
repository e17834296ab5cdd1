"""The compiled bindings against ctypes over the argument forms both take, and the
refusals of each (no device needed: size queries and calls that fail their checks)."""
import ctypes

import pytest
import torch

from voom_amd import _lib, ops


def test_size_queries_agree_with_ctypes():
    for name, args in (("voom_paged_gqa_workspace_bytes", (16, 32, 8, 128, 0)),
                       ("voom_paged_gqa_workspace_bytes", (1, 9, 3, 64, 7)),
                       ("voom_mla_head_weights_bytes", (128, 512, 128)),
                       ("voom_paged_gqa_workspace_bytes", (0, 32, 8, 128, -1))):
        assert getattr(_lib.calls(), name)(*args) == getattr(_lib.lib(), name)(*args)
    assert _lib.calls().voom_abi_version() == _lib.lib().voom_abi_version()
    # integers are cut to the parameter's width
    wide = (1 << 32) + 16
    name = "voom_paged_gqa_workspace_bytes"
    assert (getattr(_lib.calls(), name)(wide, 32, 8, 128, 0)
            == getattr(_lib.lib(), name)(wide, 32, 8, 128, 0))


@pytest.mark.parametrize("form", [int, ctypes.c_void_p, lambda p: (ctypes.c_byte * 64)()])
def test_pointer_forms_reach_the_same_check(form):
    x = torch.zeros(64, dtype=torch.bfloat16)
    args = (form(x.data_ptr()), x, x.data_ptr(), 0, 8, 32, None)  # rows 0: refused
    with pytest.raises(ValueError, match="row count"):
        _lib.call("voom_linear_rows", *args)
    with pytest.raises(ValueError, match="null pointer"):
        _lib.call("voom_linear_rows", None, *args[1:])


def test_refused_arguments():
    with pytest.raises((TypeError, ctypes.ArgumentError)):
        _lib.call("voom_linear_rows", None, None, None, 1.5, 8, 8, None)
    with pytest.raises((TypeError, ctypes.ArgumentError)):
        _lib.call("voom_linear_rows", None, None)
    with pytest.raises((TypeError, ctypes.ArgumentError)):
        _lib.call("voom_linear_rows", object(), None, None, 1, 8, 8, None)


def test_require_device():
    assert ops._require_device() is None and ops._require_device(None, None) is None
    with pytest.raises(ValueError, match="ROCm device tensors"):
        ops._require_device(None, torch.zeros(4))
    with pytest.raises(AttributeError):
        ops._require_device(4)

    class Sub(torch.Tensor):
        pass

    with pytest.raises(ValueError, match="ROCm device tensors"):
        ops._require_device(torch.zeros(4).as_subclass(Sub))
    with pytest.raises(ValueError, match="row count"):
        x = torch.zeros(64, dtype=torch.bfloat16).as_subclass(Sub)
        _lib.call("voom_linear_rows", x, x, x, 0, 8, 32, None)


@pytest.mark.gpu
def test_require_device_on_the_device():
    class Sub(torch.Tensor):
        pass

    x = torch.zeros((4, 4), device="cuda")
    for t in (x, x.as_subclass(Sub), torch.nn.Parameter(x)):
        assert ops._require_device(None, t, x) == x.device
        with pytest.raises(ValueError, match="contiguous"):
            ops._require_device(x, t.t())
        with pytest.raises(ValueError, match="ROCm device tensors"):
            ops._require_device(t, torch.zeros(4))
