"""Rows of any length (not whole groups of 256, any element address): the row kernels against the
composition of minimax, pack and unpack on the zero-padded rows, which the oracle tests pin."""
import pytest
import torch

from actnn_amd import ops, qscheme
from actnn_amd.conf import config
from actnn_amd.cpp_extension import minimax as ext_minimax
from actnn_amd.cpp_extension import quantization as ext_q

pytestmark = pytest.mark.gpu

DTYPES = [torch.float32, torch.float16, torch.bfloat16]
# (a block packs 4096 elements of a row in fp32, 8192 in 16 bits: the longest rows take several, the last one ragged)
SHAPES = [(8, 1), (1, 9), (3, 3), (2, 7), (5, 255), (3, 256), (4, 257), (9, 2049), (2, 4093), (65, 300), (7, 512),
          (3, 4097), (2, 8193), (3, 20001)]


def _rows(N, F, dtype, shift, seed):
    """[N, F] whose first element lies `shift` elements behind an allocation's start."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    flat = torch.randn(N * F + shift, generator=gen, device="cuda") * 3 + 1
    return flat.to(dtype)[shift:].view(N, F)


def _padded(x):
    N, F = x.shape
    G = (F + 255) // 256
    return torch.cat([x, torch.zeros(N, G * 256 - F, dtype=x.dtype, device=x.device)], 1).view(N, G, 256)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("bits", [1, 2, 4, 8])
def test_fixed_width_rows_equal_the_padded_composition(dtype, bits):
    for i, (N, F) in enumerate(SHAPES):
        for shift in (0, 1):
            x = _rows(N, F, dtype, shift, 17 * i + shift)
            groups = _padded(x)
            G = groups.shape[1]
            mn, mx = ext_minimax.minimax(groups.view(-1, 256))
            mn, mx = mn.view(N, G, 1), mx.view(N, G, 1)
            torch.manual_seed(i)
            want, want_scale = ext_q.pack_single_precision(groups, mn, mx, bits, True)
            store = ops._stored_dtype(dtype)
            want_scale, want_mn = want_scale.to(store), mn.to(store)
            torch.manual_seed(i)
            packed, scale, low = ext_q.quantize_rows_fixed(x, bits, None, store)
            used = packed.numel() - 1                            # the last byte belongs to no element
            assert torch.equal(packed[:used], want[:used]), (N, F, shift)
            assert torch.equal(scale, want_scale) and torch.equal(low, want_mn), (N, F, shift)
            back = ext_q.unpack_rows_fixed(packed, bits, scale, low, N, F, dtype)
            full = ext_q.unpack_single_precision(want, bits, want_scale.to(dtype), want_mn.to(dtype), N, G, 256)
            assert torch.equal(back, full.view(N, -1)[:, :F]), (N, F, shift)


@pytest.mark.parametrize("dtype", DTYPES)
def test_fixed_width_rows_with_known_ranges(dtype):
    x = _rows(6, 1024, dtype, 0, 3)
    mn, mx = ext_minimax.minimax(x.view(-1, 256))
    store = ops._stored_dtype(dtype)
    torch.manual_seed(5)
    want = ext_q.quantize_rows_fixed(x, 4, None, store)
    torch.manual_seed(5)
    got = ext_q.quantize_rows_fixed(x, 4, (mn, mx), store)
    assert torch.equal(got[0][:-1], want[0][:-1]) and torch.equal(got[1], want[1]) and torch.equal(got[2], want[2])


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("channels_last", [False, True])
def test_special_values_survive_the_one_pass(dtype, channels_last):
    """Constant groups, infinities and NaNs: as the general path (taken for a noisy group size switch) leaves them."""
    config.reset()
    config.activation_compression_bits = [4]
    try:
        x = torch.randn(3, 8, 13, 7, device="cuda").to(dtype)
        x[0] = 2.5
        x[1, :, :2] = float("nan")
        x[2, 0, 0, 0] = float("inf")
        if channels_last:
            x = x.contiguous(memory_format=torch.channels_last)
        torch.manual_seed(1)
        saved = ops.quantize_saved(x, None)
        torch.manual_seed(1)
        groups, bits, mn, mx = ops.no_scheme_compute_quantization_bits(x)
        want, scale = ext_q.pack_single_precision(groups, mn, mx, bits, True)
        store = ops._stored_dtype(dtype)
        assert torch.equal(saved[0][:-1], want[:-1])
        assert torch.equal(saved[2].nan_to_num(7.0), scale.to(store).nan_to_num(7.0))
        assert torch.equal(saved[3].nan_to_num(7.0), mn.to(store).nan_to_num(7.0))
        assert ops.dequantize_activation(saved, x.shape).stride() == x.stride()
    finally:
        config.reset()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("initial,avg", [(8, 2.0), (8, 3.7), (2, 1.3)])
def test_rows_at_widths_of_their_own_equal_the_padded_composition(dtype, initial, avg):
    for i, (N, F) in enumerate(SHAPES):
        for shift in (0, 1):
            x = _rows(N, F, dtype, shift, 31 * i + shift)
            groups = _padded(x)
            G = groups.shape[1]
            mn, mx = ext_minimax.minimax(groups.view(-1, 256))
            C, bits = qscheme.allocate_bits_on_device(mn, mx, N, F, 1.0, None, initial, avg)
            mn, mx = mn.view(N, G, 1), mx.view(N, G, 1)
            torch.manual_seed(i)
            want, want_scale = ext_q.pack_mixed_precision(groups, mn, mx, bits, True)
            alloc = qscheme.AllocationArgs(N, 256 / F, None, initial, avg)
            alloc.store_dtype = store = ops._stored_dtype(dtype)
            torch.manual_seed(i)
            packed, bits2, scale, low = ext_q.quantize_activation_device(x, N, None, alloc)
            assert torch.equal(bits2, bits) and torch.equal(packed, want), (N, F, shift)
            want_scale, want_mn = want_scale.to(store), mn.to(store)
            assert torch.equal(scale, want_scale) and torch.equal(low.view(N, G, 1), want_mn), (N, F, shift)
            back = ext_q.unpack_rows_mixed(packed, bits2, scale, low.view(N, G, 1), N, F, dtype)
            full = ext_q.unpack_mixed_precision(want, bits, want_scale.to(dtype), want_mn.to(dtype), N, G, 256)
            assert torch.equal(back, full.view(N, -1)[:, :F]), (N, F, shift)


@pytest.mark.parametrize("dtype", DTYPES)
def test_rows_end_at_every_place_in_a_line(dtype):
    # the restored rows start anywhere in a line of 128 bytes (odd lengths) and end within, at and behind units of
    # a wave (1024 elements in fp32, 2048 in 16 bits); what lies behind the last row stays as it was
    for F in (1, 2, 31, 63, 64, 65, 1023, 1024, 1025, 1057, 2047, 2049, 2081, 3001):
        N = 67
        x = _rows(N, F, dtype, 0, F)
        if x.numel() < 8:
            continue
        alloc = qscheme.AllocationArgs(N, 256 / F, None, 8, 3)
        alloc.store_dtype = store = ops._stored_dtype(dtype)
        packed, bits, scale, low = ext_q.quantize_activation_device(x, N, None, alloc)
        low = low.view(N, -1, 1)
        G = (F + 255) // 256
        want = ext_q.unpack_mixed_precision(packed, bits, scale.to(dtype), low.to(dtype), N, G, 256).view(N, -1)[:, :F]
        room = torch.full((N * F + 256,), 7.0, dtype=dtype, device="cuda")
        prefix = ext_q._bits_info(bits)[1]
        code = ext_q.g.DTYPE_CODE
        rc = ext_q.g.lib().actnn_unpack_mixed_rows(packed.data_ptr(), bits.data_ptr(), prefix.data_ptr(), scale.data_ptr(),
                                                   low.data_ptr(), room.data_ptr(), N, F, code[dtype], code[store],
                                                   torch.cuda.current_stream().cuda_stream)
        assert rc == 0
        assert torch.equal(room[:N * F].view(N, F), want), F
        assert bool((room[N * F:] == 7).all()), F


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("F", [257, 1001, 2049, 8193])
def test_odd_rows_on_both_sides_of_the_line_between_the_stores(dtype, F):
    # up to 96 MiB restored rows are stored through the caches, larger ones past them, from LDS at per-sample widths:
    # the same values either way, and nothing behind the last row
    size = torch.empty(0, dtype=dtype).element_size()
    at_most = (96 << 20) // (F * size)
    code = ext_q.g.DTYPE_CODE
    store = ops._stored_dtype(dtype)
    for N in (at_most, at_most + 1):
        x = _rows(N, F, dtype, 0, F)
        G = (F + 255) // 256
        room = torch.full((N * F + 256,), 7.0, dtype=dtype, device="cuda")
        stream = torch.cuda.current_stream().cuda_stream
        bits = 1 + torch.arange(N, dtype=torch.int32) % 8
        dev_bits = ext_q.attach_bits_host(bits.cuda(), bits)
        padded = _padded(x)
        mn, mx = ext_minimax.minimax(padded.view(-1, 256))
        mn, mx = mn.view(N, G, 1), mx.view(N, G, 1)
        packed, scale = ext_q.pack_mixed_precision(padded, mn, mx, dev_bits, True)
        prefix = ext_q._bits_info(dev_bits)[1]
        want = ext_q.unpack_mixed_precision(packed, dev_bits, scale, mn, N, G, 256).view(N, -1)[:, :F]
        assert ext_q.g.lib().actnn_unpack_mixed_rows(packed.data_ptr(), dev_bits.data_ptr(), prefix.data_ptr(), scale.data_ptr(),
                                                     mn.data_ptr(), room.data_ptr(), N, F, code[dtype], code[dtype], stream) == 0
        assert torch.equal(room[:N * F].view(N, F), want) and bool((room[N * F:] == 7).all()), N
        packed, scale, low = ext_q.quantize_rows_fixed(x, 4, None, store)
        want = ext_q.unpack_single_precision(packed, 4, scale.to(dtype), low.to(dtype), N, G, 256).view(N, -1)[:, :F]
        room.fill_(7.0)
        assert ext_q.g.lib().actnn_unpack_single_rows(packed.data_ptr(), 4, scale.data_ptr(), low.data_ptr(), room.data_ptr(),
                                                      N, F, code[dtype], code[store], stream) == 0
        assert torch.equal(room[:N * F].view(N, F), want) and bool((room[N * F:] == 7).all()), N


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("N,F", [(1, 256), (7, 300), (63, 512), (64, 257), (65, 4096), (130, 1000), (2050, 264)])
@pytest.mark.parametrize("avg", [2, 5])
def test_rows_with_the_samples_contiguous(dtype, N, F, avg):
    # (both widths of a wave's halves up to 2, up to 4 and above; ragged last tiles of 64 samples and 256 features)
    x = _rows(N, F, dtype, 0, N + F) * torch.exp(torch.randn(N, 1, device="cuda", generator=torch.Generator("cuda").manual_seed(F))).to(dtype)
    alloc = qscheme.AllocationArgs(N, 256 / F, None, 8, avg)
    alloc.store_dtype = dtype
    packed, bits, scale, low = ext_q.quantize_activation_device(x, N, None, alloc)
    low = low.view(N, -1, 1)
    want = ext_q.unpack_rows_mixed(packed, bits, scale, low, N, F, dtype)
    got = ext_q.unpack_rows_mixed_transposed(packed, bits, scale, low, N, F)
    assert got.shape == (F, (N + 63) // 64 * 64) and torch.equal(got[:, :N].t(), want)
    assert not got[:, N:].any()                              # the columns behind the last sample are zero


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("N,F", [(1024, 1024), (1025, 2048), (2047, 1000), (150, 8192), (16384, 72)])
def test_row_and_column_sums_from_one_read(dtype, N, F):
    x = _rows(N, F, dtype, 0, N)
    with_sq = F <= 1024 * 16 // x.element_size()
    with torch.no_grad():
        got = ext_minimax.row_column_sums(x, with_sq)
    assert got is not None
    # fp32 sums of N terms in runs of 16, then 16 partial sums side by side: under 2 * (16 + N / 256 + 5) roundings
    exact, weight = x.double().sum(0), x.double().abs().sum(0)
    eps = {torch.float32: 2.0 ** -24, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}[dtype]
    bound = 2 * (21 + N / 256) * 2.0 ** -24 * weight + eps * exact.abs()
    assert bool(((got[0].double() - exact).abs() <= bound).all())
    assert got[0].dtype == dtype
    if with_sq:
        slices = max(1, min(64, F // 8192))
        if slices == 1:
            assert torch.equal(got[1], ext_minimax.sample_sqnorm(x))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("N,F", [(1, 8), (63, 248), (64, 256), (65, 264), (2050, 1000), (4096, 512)])
def test_sums_and_the_rows_turned_over_from_one_read(dtype, N, F):
    x = _rows(N, F, dtype, 0, N + F)
    with torch.no_grad():
        columns, sq, turned = ext_minimax.row_column_sums_transposed(x, True, True)
        none = ext_minimax.row_column_sums_transposed(x, False, False)
    assert turned.shape == (F, (N + 63) // 64 * 64) and torch.equal(turned[:, :N].t(), x) and not turned[:, N:].any()
    assert none[0] is None and none[1] is None and torch.equal(none[2], turned)
    # columns: 8 rows, 8 of those, then tiles of 64 rows 16 side by side; squares: 8 products in a lane, 32
    # lanes, then tiles of 256 columns one after the other
    exact, weight = x.double().sum(0), x.double().abs().sum(0)
    eps = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}[dtype]
    bound = (8 + 3 + N / 1024 + 5) * 2.0 ** -24 * weight + eps * exact.abs()
    assert columns.dtype == dtype and bool(((columns.double() - exact).abs() <= bound).all())
    exact = x.double().square().sum(1)
    assert bool(((sq.double() - exact).abs() <= (8 + 5 + F / 256 + 1) * 2.0 ** -24 * exact).all())
