"""The Python side of the native calls of csrc/host_calls.cpp, as far as it shows without a GPU."""
import pytest
import torch
import torch.nn.functional as F

from actnn_amd import _lib
from actnn_amd.cpp_extension import backward_func as ext_bf


@pytest.fixture
def nothing_built(monkeypatch):
    def missing():
        raise RuntimeError("not built")
    monkeypatch.setattr(_lib, "load", missing)
    monkeypatch.setattr(_lib, "load_host", missing)


def test_batch_norm_of_cpu_tensors_needs_nothing_built(nothing_built):
    x, one, zero = torch.randn(4, 8, 6, 6), torch.ones(8), torch.zeros(8)
    affine = (one, zero, zero, one)
    assert ext_bf._bn_geometry(x) is None
    assert not ext_bf.hip_batch_norm_applies(x, *affine)
    assert not ext_bf.hip_batch_norm_minmax_applies(x, *affine)
    assert not ext_bf.hip_batch_norm_pack_applies(x, *affine)
    assert ext_bf.hip_batch_norm_quantize_geometry(x, *affine) is None
    y, mean, invstd = ext_bf.native_batch_norm(x, *affine, False, 0.1, 1e-5)
    assert torch.allclose(y, F.batch_norm(x, zero, one, one, zero, False, 0.1, 1e-5))
    gi, _, _ = ext_bf.native_batch_norm_backward(torch.ones_like(x), x, one, zero, one, mean, invstd, False, 1e-5,
                                                 [True, True, True])
    assert torch.allclose(gi, torch.full_like(x, (1 + 1e-5) ** -0.5))
