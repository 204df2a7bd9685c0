"""The native calls of csrc/host_calls.cpp: what they take over from Python besides the kernels' results (which the tests of
each operator check) - stream, generator, tensor classes, and the refusals."""
import pytest
import torch

import actnn_amd.cpp_extension.quantization as ext_q
from actnn_amd.cpp_extension import backward_func as ext_bf
from actnn_amd.qscheme import AllocationArgs

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _rows(N, F, bits=4):
    torch.manual_seed(0)
    return ext_q.quantize_rows_fixed(torch.randn(N, F, device=DEV), bits, None, torch.bfloat16)


def _compress(x, known):
    rows = x.reshape(256, -1)
    alloc = AllocationArgs(256, 1.0, None, 8, 2.0)
    ranges = torch.aminmax(rows.reshape(-1, 256), dim=1) if known else None
    packed, bits, scale, mn = ext_q.quantize_activation_device(rows, 256, ranges, alloc)
    back = ext_q.unpack_rows_mixed(packed, bits, scale, mn.view(scale.shape), 256, rows.shape[1], rows.dtype)
    return packed, bits, scale, mn, back


def _compress_fixed(x):
    rows = x.reshape(256, -1)
    packed, scale, mn = ext_q.quantize_rows_fixed(rows, 4, None, rows.dtype)
    back = ext_q.unpack_rows_fixed(packed, 4, scale, mn, 256, rows.shape[1], rows.dtype)
    return packed[:-1], scale, mn, back                # (the last byte is spare)


def _relu(x):
    y, mask = ext_q.relu_forward(x)
    return y, mask, ext_q.relu_backward(x, mask)


def _dropout(x):
    y, mask = ext_q.dropout_forward(x, 0.25)
    return y, mask, ext_q.dropout_backward(x, mask, 0.25)


def _pool(x, channels_last, nibble):
    x = x.contiguous(memory_format=torch.channels_last) if channels_last else x
    window = (3, 3), (2, 2), (1, 1)
    y, idx = ext_q.max_pool2d_forward(x, *window, (1, 1), nibble)
    return y, idx, ext_q.max_pool2d_backward(y, idx, x.shape, *window, channels_last)


def _batch_norm(x):
    weight, bias, mean, var = (torch.full((64,), v, device=DEV) for v in (1.0, 0.5, 0.0, 1.0))
    y, save_mean, invstd, mn, mx = ext_bf.hip_batch_norm_forward(x, weight, bias, mean, var, 0.1, 1e-5, True)
    return (y, save_mean, invstd, mn, mx, mean, var, *ext_bf.hip_batch_norm_backward(x, y, weight, save_mean, invstd, True))


def _batch_norm_packed(x, relu):
    x = x.contiguous(memory_format=torch.channels_last)
    weight, bias, mean, var = (torch.full((64,), v, device=DEV) for v in (1.0, 0.5, 0.0, 1.0))
    geo = ext_bf.hip_batch_norm_quantize_geometry(x, weight, bias, mean, var)
    got = ext_bf.hip_batch_norm_forward_quantize(x, geo, weight, bias, mean, var, 0.1, 1e-5, AllocationArgs(256, 1.0, None, 8, 2.0),
                                                 relu, x if relu else None)
    y, save_mean, invstd, mn, mx, bits, packed, scale = got[:8]
    stream = _Stream((packed, bits, scale, mn.view(scale.shape)))
    stream.memory_format = torch.channels_last
    back = ext_bf.hip_batch_norm_backward_packed(x.shape, stream, y, weight, save_mean, invstd, True, got[8] if relu else None)
    return (*got, mean, var, *back)


class _Stream(tuple):
    pass


@pytest.mark.parametrize("operator", [lambda x: _compress(x, False), lambda x: _compress(x, True), _compress_fixed, _relu, _dropout,
                                      lambda x: _pool(x, False, False), lambda x: _pool(x, False, True), lambda x: _pool(x, True, False),
                                      lambda x: _pool(x, True, True), _batch_norm, lambda x: _batch_norm_packed(x, False),
                                      lambda x: _batch_norm_packed(x, True)],
                         ids=["compress", "compress known ranges", "compress fixed", "relu", "dropout", "pool", "pool nibbles",
                              "pool channels last", "pool channels last nibbles", "batch norm", "batch norm packed",
                              "batch norm relu packed"])
def test_calls_run_on_the_current_stream(operator):
    """Forward and backward of each native call behind work that only calls on the same stream come behind."""
    x = torch.randn(256, 64, 16, 16, device=DEV).to(torch.bfloat16)
    ahead = torch.randn(1 << 24, device=DEV)
    torch.cuda.manual_seed(5)
    expected = operator(x)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        late = torch.zeros_like(x)                     # what a call on another stream would read
        side.synchronize()
        for _ in range(40):                            # (about a millisecond)
            ahead.mul_(1.0009765625)
        late.copy_(x)
        torch.cuda.manual_seed(5)
        got = operator(late)
    side.synchronize()
    assert len(got) == len(expected)
    for i, (a, b) in enumerate(zip(got, expected)):
        assert torch.equal(a, b), i


@pytest.mark.parametrize("draws", [1, 3])
def test_each_call_advances_the_generator_as_one_draw(draws):
    gen = torch.cuda.default_generators[0]
    torch.manual_seed(7)
    gen.set_offset(40)
    got = [ext_q.dropout_forward(torch.ones(4096, device=DEV), 0.5)[0] for _ in range(draws)]
    assert gen.get_offset() == 40 + 4 * draws
    gen.set_offset(40)
    assert torch.equal(ext_q.dropout_forward(torch.ones(4096, device=DEV), 0.5)[0], got[0])
    assert draws == 1 or not torch.equal(got[0], got[1])


class _Named(torch.Tensor):
    pass


@pytest.mark.parametrize("make", [lambda x: x, lambda x: torch.nn.Parameter(x), lambda x: x.as_subclass(_Named)],
                         ids=["tensor", "parameter", "subclass"])
def test_tensor_classes_come_back_as_empty_like_makes_them(make):
    x = torch.randn(2048, device=DEV)
    given = make(x.clone())
    with torch.no_grad():
        y, mask = ext_q.relu_forward(given)
        back = ext_q.relu_backward(given, mask)
        z, kept = ext_q.dropout_forward(given, 0.5)
        scaled = ext_q.dropout_backward(given, kept, 0.5)
        for got in (y, back, z, scaled):
            assert type(got) is type(torch.empty_like(given)) and not got.requires_grad
    for got in (y, back):
        assert torch.equal(got.as_subclass(torch.Tensor), torch.relu(x))
    assert torch.equal(z.as_subclass(torch.Tensor), scaled.as_subclass(torch.Tensor))
    assert torch.isin(z.as_subclass(torch.Tensor) / x, torch.tensor([0.0, 2.0], device=DEV)).all()


@pytest.mark.parametrize("operator", ["relu", "dropout"])
@pytest.mark.parametrize("order", ["transposed", "channels last", "default", "misaligned"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_gradient_of_a_tensor_class_in_any_order(operator, order, dtype):
    """A gradient that is an instance of a subclass keeps its class; its values come back in their places whatever its strides are."""
    shape = (6, 16, 5, 7)
    x = torch.randn(shape, device=DEV, dtype=dtype)
    if operator == "relu":
        y, mask = ext_q.relu_forward(x)
        factor = (x > 0).to(dtype)
    else:
        factor, mask = ext_q.dropout_forward(torch.ones_like(x), 0.5)                # 0 and 2
    values = torch.randn(shape, device=DEV, dtype=dtype)
    grad = {"transposed": lambda: values.permute(3, 2, 1, 0).contiguous().permute(3, 2, 1, 0),
            "channels last": lambda: values.contiguous(memory_format=torch.channels_last), "default": values.clone,
            "misaligned": lambda: torch.cat([values.new_zeros(1), values.flatten()])[1:].view(shape)}[order]()
    for given in (grad, grad.as_subclass(_Named)):
        got = ext_q.relu_backward(given, mask) if operator == "relu" else ext_q.dropout_backward(given, mask, 0.5)
        assert torch.equal(got.as_subclass(torch.Tensor), values * factor)
        assert type(got) is type(given) and got.is_contiguous()
    leaf = (x if operator == "relu" else torch.ones_like(x)).requires_grad_()
    out = ext_q.act_quantized_relu(leaf) if operator == "relu" else ext_q.act_quantized_dropout(leaf, 0.5)
    factor = factor if operator == "relu" else out.detach()
    (got,) = torch.autograd.grad(out, leaf, grad.as_subclass(_Named))
    assert torch.equal(got.as_subclass(torch.Tensor), values * factor)


def test_misaligned_input_is_copied():
    x = torch.randn(4097, device=DEV)[1:]
    y, mask = ext_q.relu_forward(x)
    assert torch.equal(y, torch.relu(x))
    g = torch.randn(4097, device=DEV)[1:]
    assert torch.equal(ext_q.relu_backward(g, mask), torch.where(x > 0, g, torch.zeros_like(g)))


@pytest.mark.parametrize("wrong,what", [("data", "data"), ("scale", "scale"), ("min", "min"), ("short", "too short"), ("N", "shape mismatch"),
                                        ("dtype", "type of min")])
def test_restoring_what_does_not_fit_is_refused(wrong, what):
    N, F = 5, 700
    packed, scale, mn = _rows(N, F)
    args = dict(packed=packed, bits=4, scale=scale, mn=mn, N=N, F=F, dtype=torch.float32)
    args.update({"data": dict(packed=packed.cpu()), "scale": dict(scale=scale.int()), "min": dict(mn=None),
                 "short": dict(packed=packed[:-300]), "N": dict(N=N + 1), "dtype": dict(mn=mn.float())}[wrong])
    with pytest.raises(RuntimeError, match=what):
        ext_q.unpack_rows_fixed(**args)
    bits = torch.full((N,), 4, dtype=torch.int32, device=DEV)
    groups = N * ((F + 255) // 256)
    args.update(bits=bits)
    if args["packed"] is not None and wrong != "data":
        args["packed"] = torch.zeros(groups * 32 - (8 if wrong == "short" else 0), dtype=torch.int32, device=DEV)
    with pytest.raises(RuntimeError, match=what):
        ext_q.unpack_rows_mixed(**args)


@pytest.mark.parametrize("shape,fmt,want", [((4, 8, 3, 5), None, (4, 8, 15, False)), ((4, 8, 3, 5), torch.channels_last, (4, 8, 15, True)),
                                            ((6, 7), None, (6, 7, 1, False)), ((2, 8, 2, 3, 4), torch.channels_last_3d, (2, 8, 24, True)),
                                            ((2, 1, 3, 5), torch.channels_last, (2, 1, 15, False)), ((0, 8, 3, 5), None, None)])
def test_batch_norm_geometry(shape, fmt, want):
    x = torch.zeros(shape, device=DEV)
    x = x if fmt is None else x.contiguous(memory_format=fmt)
    assert ext_bf._bn_geometry(x) == want
    assert ext_bf._bn_geometry(x.cpu()) is None and ext_bf._bn_geometry(x.double()) is None
    if want is not None and len(shape) > 2 and shape[1] > 1:
        assert ext_bf._bn_geometry(x.transpose(0, 2)) is None
    one = torch.ones(shape[1], device=DEV)
    assert ext_bf.hip_batch_norm_applies(x, one, None, one, one) == (want is not None)
    assert not ext_bf.hip_batch_norm_applies(x, one.half(), None, one, one)
    assert not ext_bf.hip_batch_norm_applies(x, one.cpu(), None, one, one)
