"""``minimax(data) -> (min, max)``: row-wise min/max of a [M, D] device tensor
(reference: cpp_extension/minimax.cc:7-16)."""
import torch

from . import _glue as g
from .._lib import check
from ..utils import channels_last_format


def minimax(data):
    g.check_float(data, "data")                        # minimax.cc:8
    if data.dim() != 2:
        raise RuntimeError("The dimension of data is not correct!")
    M, D = data.shape
    mn = torch.empty(M, dtype=data.dtype, device=data.device)
    mx = torch.empty(M, dtype=data.dtype, device=data.device)
    with g.on_device(data.device):
        check(g.lib().actnn_minimax(data.data_ptr(), mn.data_ptr(), mx.data_ptr(), M, D,
                                    g.DTYPE_CODE[data.dtype], g.stream_ptr(data.device)), "minimax")
    return mn, mx


def range_sqr(mn, mx, N, factor=1.0, mult=None):
    """fp32 [N]: factor * mult * sum over the groups of sample n of (mx - mn)^2, in one kernel
    (reference: the tensor expression of qscheme.py:80-82).  mn / mx: the [N * G] outputs of
    ``minimax``; mult: None, a 0-dim fp32 device tensor or an fp32 device tensor of N values."""
    g.check_float(mn, "min")
    if mx.dtype != mn.dtype or mx.shape != mn.shape or mn.numel() % max(N, 1) != 0:
        raise RuntimeError("range_sqr: min and max do not match")
    mn = mn.contiguous()
    mx = mx.contiguous()
    G = mn.numel() // N if N else 0
    out = torch.empty(N, dtype=torch.float32, device=mn.device)
    mult_ptr, per_sample = None, 0
    if mult is not None:
        if mult.dtype != torch.float32 or mult.device != mn.device or mult.numel() not in (1, N):
            raise RuntimeError("range_sqr: mult must be fp32 on the same device with 1 or N values")
        mult = mult.contiguous()
        mult_ptr, per_sample = mult.data_ptr(), int(mult.numel() == N and N != 1)
    with g.on_device(mn.device):
        check(g.lib().actnn_range_sqr(mn.data_ptr(), mx.data_ptr(), out.data_ptr(), N, G, float(factor),
                                      mult_ptr, per_sample, g.DTYPE_CODE[mn.dtype], g.stream_ptr(mn.device)),
              "range_sqr")
    return out


def sample_sqnorm(x):
    """fp32 [N]: squared L2 norm of every sample of a dense tensor (any layout: the sum does not
    care about the order), one pass at memory speed."""
    N = x.shape[0]
    F = x.numel() // max(N, 1)
    elems = 16 // x.element_size()
    dense = x.is_contiguous() or channels_last_format(x) is not None
    if (N == 0 or N > 65535 or F % elems != 0 or x.dtype not in g.DTYPE_CODE or not x.is_cuda
            or not dense or x.data_ptr() % 16 != 0):
        return torch.linalg.vector_norm(x.reshape(N, -1), dim=1, dtype=torch.float32).square()
    slices = max(1, min(64, F // 8192))
    part = torch.empty(N, slices, dtype=torch.float32, device=x.device)
    with g.on_device(x.device):
        check(g.lib().actnn_sample_sqnorm(x.data_ptr(), part.data_ptr(), N, F, slices,
                                          g.DTYPE_CODE[x.dtype], g.stream_ptr(x.device)), "sample_sqnorm")
    return part.sum(1) if slices > 1 else part.view(N)


def _sums_pay(N, F, size, with_sqnorm):
    """Where row_column_sums is the faster way (us, its two kernels / torch's sum over the rows, and with the
    norms / the sum and sample_sqnorm; f16 unless said).  From 2^20 elements on, where it was first 5 us ahead
    ([1024,1024] 5.7 / 10.3).  Its second kernel walks N / 16 partial rows for a column, so tall and
    narrow tensors lose: [32768,64] 19.0 / 11.6, [65535,256] 34.7 / 31.4, but [16384,256] 12.4 / 24.2,
    [8192,64] 8.1 / 9.7; beyond 128 MB torch reads as fast: f32 [16384,4096] 49.2 / 46.9, [16384,2048]
    28.5 / 31.6, f32 [4096,16384] 46 / 169.  The norms cost it little: [65535,64] 40.4 / 52.4, [65535,32]
    48.8 / 47.3."""
    if N * F < 1 << 20 or N > 65535:
        return False
    if with_sqnorm:
        return F >= 64
    return 128 <= N <= 32768 and F >= N / 128 and (N <= 4096 or N * F * size <= 1 << 27)


def row_column_sums(x, with_sqnorm):
    """(sum over the rows of a [N, F] tensor in its dtype, squared norm of every row as sample_sqnorm gives it
    or None) from one read, or None where the kernel does not apply or does not pay: ragged rows, rows too long
    for a block, under a graph of the backward pass, and for a batch of gradients at once
    (torch.autograd.grad with is_grads_batched), which has no memory to read."""
    if (x.dim() != 2 or x.dtype not in g.DTYPE_CODE or not x.is_cuda or not x.is_contiguous() or torch.is_grad_enabled()
            or not _sums_pay(x.shape[0], x.shape[1], x.element_size(), with_sqnorm)
            or not g.has_storage(x) or x.data_ptr() % 16 != 0):
        return None
    N, F = x.shape
    elems = 16 // x.element_size()
    if F % elems != 0 or (with_sqnorm and F > 1024 * elems):
        return None
    columns = torch.empty(F, dtype=x.dtype, device=x.device)
    sq = torch.empty(N, dtype=torch.float32, device=x.device) if with_sqnorm else None
    part = torch.empty((N + 15) // 16, F, dtype=torch.float32, device=x.device)
    with g.on_device(x.device):
        check(g.lib().actnn_row_column_sums(x.data_ptr(), columns.data_ptr(), sq.data_ptr() if with_sqnorm else None,
                                            part.data_ptr(), N, F, g.DTYPE_CODE[x.dtype], g.stream_ptr(x.device)),
              "row_column_sums")
    return columns, sq


def row_column_sums_transposed(x, with_columns, with_sqnorm):
    """(sum over the rows or None, squared norm of every row or None, the rows turned over: [F, N rounded up to 64],
    zero behind row N) of a 16-bit [N, F] tensor from one read, or None where row_column_sums says None for the
    tensor's form.  The sums' order is another one than row_column_sums'."""
    if (x.dim() != 2 or x.dtype not in (torch.float16, torch.bfloat16) or not x.is_cuda or not x.is_contiguous()
            or torch.is_grad_enabled() or x.shape[1] % 8 != 0 or x.numel() == 0
            or not g.has_storage(x) or x.data_ptr() % 16 != 0):
        return None
    N, F = x.shape
    ld = (N + 63) // 64 * 64
    out = torch.empty(F, ld, dtype=x.dtype, device=x.device)
    columns = torch.empty(F, dtype=x.dtype, device=x.device) if with_columns else None
    sq = torch.empty(N, dtype=torch.float32, device=x.device) if with_sqnorm else None
    part = torch.empty(ld // 64, F, dtype=torch.float32, device=x.device) if with_columns else None
    sq_part = torch.empty((F + 255) // 256, N, dtype=torch.float32, device=x.device) if with_sqnorm else None
    ptr = lambda t: t.data_ptr() if t is not None else None
    with g.on_device(x.device):
        check(g.lib().actnn_row_column_sums_transposed(
            x.data_ptr(), ptr(columns), ptr(sq), out.data_ptr(), ptr(part), ptr(sq_part), N, F, ld, g.DTYPE_CODE[x.dtype],
            g.stream_ptr(x.device)), "row_column_sums_transposed")
    return columns, sq, out
