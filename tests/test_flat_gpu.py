"""The flat INT4 forward (widths or groups that are not multiples of eight):
the row form, the GEMM and the fallback, at the edges of their columns, rows
and K chunks, with the last codes in a partial dword and groups that straddle
rows.  The oracle is x . (code * scale) in 64 bits; each output may be off by
a rounding per addition (K of them, in any order) of at most sum |x w|.
"""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _check(sgq, dev, M, K, N, G, seed=3, poke=None):
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed)
    qw = sgq.quantize_int4(torch.randn(K, N, generator=gen, device=dev) * 0.02, G, keep_qdata=False)
    x = torch.randn(M, K, generator=gen, device=dev)
    b = torch.randn(1, N, generator=gen, device=dev)
    w = sgq.dequantize_int4(qw).double()
    for bias in (b, None):
        y = sgq.quantized_matmul_int4(x, qw, bias).double()
        ref, mag = x.double() @ w, x.double().abs() @ w.abs()
        if bias is not None:
            ref, mag = ref + bias.double(), mag + bias.double().abs()
        bound = (K + 2) * 2.0**-24 * mag
        assert bool(((y - ref).abs() <= bound).all()), float(((y - ref).abs() / bound).max())


@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 8, 9, 31, 33])
@pytest.mark.parametrize("K,N,G", [(1, 9, 32), (7, 13, 8), (511, 63, 32), (513, 65, 12), (1025, 127, 128),
                                   (64, 129, 30), (100, 1001, 64), (2048, 4099, 32)])
def test_rows(sgq, dev, M, K, N, G):
    _check(sgq, dev, M, K, N, G)


@pytest.mark.parametrize("M,K,N,G", [(64, 33, 32771, 32), (500, 95, 4001, 128), (2048, 130, 1027, 24),
                                     (257, 1, 8195, 64)])
def test_gemm(sgq, dev, M, K, N, G):
    _check(sgq, dev, M, K, N, G)


@pytest.mark.parametrize("M,K,N,G", [(1, 1, 9, 32), (40, 3, 4001, 24), (5000, 15, 9, 12), (300, 40, 33, 32),
                                     (9000, 64, 17, 32), (9000, 20, 8193, 32), (33, 2, 70001, 8)])
def test_short_k(sgq, dev, M, K, N, G):
    """Few products per output: a thread per output, tiles where there are many rows."""
    _check(sgq, dev, M, K, N, G)


@pytest.mark.parametrize("M,K,N,G", [(M, K, N, 32) for M, K in ((1, 4095), (2, 4097), (4, 8193), (5, 2047), (8, 2049), (9, 4097))
                                     for N in (33, 32801 if M < 9 else 16411)])
def test_k_chunks(sgq, dev, M, K, N, G):
    """x restaged in LDS: K around one and two chunks of 4096 rows (2048 from five
    batch rows on), workgroups of 64 and of 128 columns."""
    _check(sgq, dev, M, K, N, G)


def _queued_us(fn, reps=20):
    fn()
    best = float("inf")
    for _ in range(5):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        torch.cuda.synchronize()
        a.record()
        for _ in range(reps):
            fn()
        b.record()
        b.synchronize()
        best = min(best, a.elapsed_time(b) * 1000 / reps)
    return best


@pytest.mark.parametrize("M,K,N,few,most", [(20306, 15, 9, 64, 4), (39, 6, 9671, 1, 2)])
def test_short_k_costs_few_launches(sgq, dev, M, K, N, few, most):
    """Some hundred thousand products of a short K take about a launch's time,
    as a few rows do (measured 1.0 to 1.2 times; the row form 9 and 2.7)."""
    qw = sgq.quantize_int4(torch.randn(K, N, device=dev), 24, keep_qdata=False)
    x = torch.randn(M, K, device=dev)
    base = _queued_us(lambda: sgq.quantized_matmul_int4(x[:few], qw))
    assert _queued_us(lambda: sgq.quantized_matmul_int4(x, qw)) < most * base


@pytest.mark.parametrize("M,K,N,G", [(3, 50, 5, 32), (4, 40, 33, 7), (2, 16, 40, 5)])
def test_narrow_and_small_groups(sgq, dev, M, K, N, G):
    _check(sgq, dev, M, K, N, G)


@pytest.mark.parametrize("M,K,N", [(3, 70, 1001), (230, 70, 8193)])
def test_non_finite(sgq, dev, M, K, N):
    """Infinities and NaNs of x and of the last scale reach the outputs that use them, and no others."""
    gen = torch.Generator(device=dev)
    gen.manual_seed(4)
    qw = sgq.quantize_int4(torch.randn(K, N, generator=gen, device=dev) * 0.02, 32, keep_qdata=False)
    x = torch.randn(M, K, generator=gen, device=dev)
    x[0, 5], x[2, 69] = float("inf"), float("nan")
    qw.scales[-1] = float("inf")
    y = sgq.quantized_matmul_int4(x, qw)
    code, scale = sgq.unpack_codes(qw).double(), qw.scales.double()
    w = (code.reshape(-1) * scale.repeat_interleave(32)[: K * N]).reshape(K, N)
    ref = torch.stack([(x[m].double()[:, None] * w).sum(0) for m in range(M)])
    assert torch.equal(torch.isnan(y), torch.isnan(ref)) and torch.equal(torch.isinf(y), torch.isinf(ref))


def test_wide_row(sgq, dev):
    """Columns past the row kernels' grid: one product each, so the result is exact."""
    N = (1 << 27) + 1
    gen = torch.Generator(device=dev)
    gen.manual_seed(6)
    qw = sgq.quantize_int4(torch.randn(1, N, generator=gen, device=dev) * 0.02, 32, keep_qdata=False)
    x = torch.full((1, 1), 1.5, device=dev)
    assert torch.equal(sgq.quantized_matmul_int4(x, qw), x * sgq.dequantize_int4(qw).reshape(1, N))
