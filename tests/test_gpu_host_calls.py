"""The native calls of csrc/host_calls.cpp: what they take over from Python besides the kernels' results (which the tests of
each operator check) - stream, generator, tensor classes, and the refusals."""
import pytest
import torch

import actnn_amd.cpp_extension.quantization as ext_q
from actnn_amd.cpp_extension import backward_func as ext_bf
from actnn_amd.cpp_extension import _glue

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _rows(N, F, bits=4):
    torch.manual_seed(0)
    return ext_q.quantize_rows_fixed(torch.randn(N, F, device=DEV), bits, None, torch.bfloat16)


def test_calls_run_on_the_current_stream():
    x = torch.randn(1 << 22, device=DEV)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(20):                            # work in front, that only calls on this stream come behind
            x = x * 1.0009765625
        y, mask = _glue.host().relu_forward(x)
    side.synchronize()
    assert torch.equal(y, torch.relu(x))


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


def test_tensor_classes_come_back_as_empty_like_makes_them():
    class Named(torch.Tensor):
        pass
    x = torch.randn(2048, device=DEV)
    for given in (x, torch.nn.Parameter(x.clone()), x.clone().as_subclass(Named)):
        y, _ = ext_q.relu_forward(given.detach() if type(given) is torch.nn.Parameter else given)
        assert type(y) is type(torch.empty_like(given.detach()))
        assert torch.equal(y.as_subclass(torch.Tensor), torch.relu(given.detach()).as_subclass(torch.Tensor))


class _Named(torch.Tensor):
    pass


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
