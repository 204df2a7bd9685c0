"""The Python side of the native calls of csrc/host_calls.cpp, as far as it shows without a GPU."""
import os

import pytest
import torch
import torch.nn.functional as F

from actnn_amd import _lib
from actnn_amd.cpp_extension import _glue
from actnn_amd.cpp_extension import backward_func as ext_bf
from actnn_amd.cpp_extension import quantization as ext_q


@pytest.fixture
def nothing_built(monkeypatch):
    def missing():
        raise RuntimeError("not built")
    monkeypatch.setattr(_lib, "load", missing)
    monkeypatch.setattr(_lib, "load_host", missing)
    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(_lib, "_host", None)


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


class _Recorder:
    def __getattr__(self, name):
        return lambda *args: (name, args[2:] if name.endswith("backward") else args[1:])


@pytest.mark.parametrize("window,stride,want", [((3, 2), (2, 1, 7), (3, 2, 2, 1, 1, 0, 1, 2)), ((3, 2, 9), (2,), None),
                                                ((3,), (2, 1, 7, 7), None)])
def test_pool_arguments_keep_their_places(monkeypatch, window, stride, want):
    """The native calls count their arguments: one more in one tuple must not stand in for one that another lacks.  The window has
    two values; of the others the first two are read, as ever."""
    monkeypatch.setattr(_glue, "host", lambda: _Recorder())
    x = torch.zeros(2, 4, 8, 8)
    padding, dilation = (1, 0, 5), [1, 2, 5]
    if want is None:
        with pytest.raises(ValueError):
            ext_q.max_pool2d_forward(x, window, stride, padding[:2], dilation[:2])
        return
    assert ext_q.max_pool2d_forward(x, window, stride, padding, dilation) == ("max_pool2d_forward", (False, *want, False))
    got = ext_q.max_pool2d_backward(x, x.to(torch.int8), x.shape, window, stride, padding)
    assert got == ("max_pool2d_backward", (False, False, 2, 4, 8, 8, *want[:6]))
    with pytest.raises(ValueError):
        ext_q.max_pool2d_backward(x, x.to(torch.int8), x.shape[1:], (3, 2, 2), (2, 1), (1, 0))


@pytest.mark.parametrize("shape,bits,what", [((4, 6, 100), 4, "two dimensions, got 3"), ((600,), 4, "two dimensions, got 1"),
                                             ((4, 600), 3, "8 % bits must be 0, got 3"), ((4, 600), 0, "got 0"), ((4, 600), 16, "got 16")])
def test_refusal_of_rows_at_one_width_says_what_is_wrong(shape, bits, what):
    with pytest.raises(RuntimeError, match=what):
        ext_q.quantize_rows_fixed(torch.zeros(shape), bits, None, torch.float32)


@pytest.mark.parametrize("fails", [None, "hipcc", "g++"])
def test_a_build_replaces_both_files_or_none(monkeypatch, tmp_path, fails):
    paths = [str(tmp_path / name) for name in ("libactnn_hip.so", "_host.so")]
    monkeypatch.setattr(_lib, "_HERE", str(tmp_path))
    monkeypatch.setattr(_lib, "LIB_PATH", paths[0])
    monkeypatch.setattr(_lib, "HOST_PATH", paths[1])
    for path in paths:
        with open(path, "w") as f:
            f.write("old")

    def compile_(cmd, verbose):
        if cmd[0] == fails:
            raise RuntimeError(f"{fails} failed")
        with open(cmd[cmd.index("-o") + 1], "w") as f:
            f.write("new")
        return ""
    monkeypatch.setattr(_lib, "_run", compile_)
    if fails:
        with pytest.raises(RuntimeError):
            _lib.build()
    else:
        _lib.build()
    assert [open(path).read() for path in paths] == ["old" if fails else "new"] * 2
    assert sorted(os.listdir(tmp_path)) == ["_host.so", "libactnn_hip.so"]


@pytest.mark.parametrize("broken", [None, "load", "load_host"])
def test_a_build_loads_what_it_built(monkeypatch, broken):
    import __graft_entry__
    from oracle import build_ref
    loaded = []
    monkeypatch.setattr(_lib, "build", lambda verbose=False: None)
    monkeypatch.setattr(build_ref, "build", lambda: None)
    for name in ("load", "load_host"):
        def load(name=name, real=getattr(_lib, name)):
            if name == broken:
                raise ImportError(f"{name}: undefined symbol")
            loaded.append(name)
            return real()
        monkeypatch.setattr(_lib, name, load)
    monkeypatch.setattr(_lib, "_host", None)
    if broken:
        with pytest.raises(ImportError):
            __graft_entry__.build()
    else:
        __graft_entry__.build()
        assert set(loaded) == {"load", "load_host"}


@pytest.mark.parametrize("there", [(), ("LIB_PATH",), ("HOST_PATH",), ("LIB_PATH", "HOST_PATH")])
def test_tests_build_where_a_file_is_missing(monkeypatch, tmp_path, there):
    import conftest
    built = []
    monkeypatch.setattr(_lib, "build", lambda: built.append(True))
    for name in ("LIB_PATH", "HOST_PATH"):
        monkeypatch.setattr(_lib, name, str(tmp_path / name))
        if name in there:
            (tmp_path / name).touch()

    class Config:
        def addinivalue_line(self, *line):
            pass
    conftest.pytest_configure(Config())
    assert len(built) == (len(there) < 2)
