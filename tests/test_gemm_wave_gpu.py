"""The INT4 GEMM of independent wavefront tiles (scale columns of a multiple of
four strips) at the edges of its tiles: rows around 32 and 64, column blocks
past the weight, scale groups of 32 to 128 columns, K shorter than its K ranges,
with a partial stage, odd (rows of x at any 4-byte address), with and without a
K split over workgroups.

The oracle is x . dequantize(W) in 64 bits.  Each output is bounded on its own:
an accumulator takes three MFMA additions per 32 k, each of which may round or
truncate (2^-23 of at most sum |x w|), the K ranges, splits, product and
epilogue add a few more roundings.
"""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _check(y, x, w, b, K, splits=16 + 4, floor=0.0):
    x, w = x.double(), w.double()
    ref, mag = x @ w, x.abs() @ w.abs()
    if b is not None:
        ref, mag = ref + b.double(), mag + b.double().abs()
    bound = (3 * -(-K // 32) + splits + 4) * 2.0**-23 * mag + floor
    bad = ((y.double() - ref).abs() > bound).sum()
    assert int(bad) == 0, (int(bad), float(((y.double() - ref).abs() / bound).max()))


def _inputs(sgq, dev, M, K, N, G, seed, offset=0):
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed)
    w = torch.randn(K, N, generator=gen, device=dev) * 0.02
    flat = torch.randn(M * K + offset, generator=gen, device=dev)
    b = torch.randn(1, N, generator=gen, device=dev)
    return flat[offset:].reshape(M, K), sgq.quantize_int4(w, G, keep_qdata=False), b


@pytest.mark.parametrize("G,N", [(32, 32), (32, 160), (64, 64), (64, 320), (96, 288), (128, 128), (128, 384)])
@pytest.mark.parametrize("M,K", [(129, 16), (160, 33), (191, 64), (193, 95), (256, 1000), (130, 2049)])
def test_tile_edges(sgq, dev, M, K, G, N):
    for offset in (0, 1):  # x at a 16-byte and at a 4-byte address
        x, qw, b = _inputs(sgq, dev, M, K, N, G, M + K + N, offset)
        _check(sgq.quantized_matmul_int4(x, qw, b), x, sgq.dequantize_int4(qw), b, K)
        _check(sgq.quantized_matmul_int4(x, qw), x, sgq.dequantize_int4(qw), None, K)


@pytest.mark.parametrize("M,K,N,G", [(2048, 160, 4096, 128), (2049, 97, 4224, 128), (40, 4096, 4096, 32),
                                     (1025, 512, 5632, 64), (33, 8200, 1152, 128),
                                     (1100, 97, 4224, 32), (1100, 512, 4096, 128), (1100, 513, 4096, 128),
                                     (2049, 33, 4160, 64), (2081, 512, 4128, 96), (1020, 64, 4096, 32), (1020, 70, 4096, 128)])
def test_large_grids(sgq, dev, M, K, N, G):
    """Four row blocks per wavefront, grids without a K split, small batches over
    long K, a short K in one and two ranges per workgroup."""
    x, qw, b = _inputs(sgq, dev, M, K, N, G, 5)
    _check(sgq.quantized_matmul_int4(x, qw, b), x, sgq.dequantize_int4(qw), b, K)


@pytest.mark.parametrize("scheme", [0, 1])
@pytest.mark.parametrize("M,K,N", [(1100, 97, 4101), (2050, 33, 4099), (2051, 30, 4224), (140, 1, 9), (133, 66, 1002)])
def test_int8_rows_at_any_address(sgq, dev, scheme, M, K, N):
    """INT8 rows that are no multiple of four floats: a partial stage whose quads
    reach into the next row, rows of y at any address, one to four last columns."""
    gen = torch.Generator(device=dev)
    gen.manual_seed(M + N)
    qw = sgq.quantize_int8(torch.randn(K, N, generator=gen, device=dev) * 0.02, scheme, keep_qdata=False)
    flat = torch.randn(M * K + 1, generator=gen, device=dev)
    b = torch.randn(1, N, generator=gen, device=dev)
    out = torch.full((M * N + 3,), 7.0, device=dev)
    for x in (flat[:-1].reshape(M, K), flat[1:].reshape(M, K)):
        for bias in (b, None):
            y = out[1 : 1 + M * N].view(M, N)
            sgq.quantized_matmul_int8(x, qw, bias, y)
            _check(y, x, sgq.dequantize_int8(qw), bias, K)
    assert out[0] == 7 and bool((out[1 + M * N :] == 7).all())


@pytest.mark.parametrize("G", [32, 128])
def test_short_k_keeps_up_with_memory(sgq, dev, G):
    """A product of one 32-k stage over many tiles is bound by writing y: measured
    1.6 to 1.8 times a copy of y, 2.9 to 3.4 with four K ranges per workgroup; the
    bound lies between."""
    M, K, N = 2048, 24, 8192
    x, qw, b = _inputs(sgq, dev, M, K, N, G, 12)
    y, z = torch.zeros(M, N, device=dev), torch.zeros(M, N, device=dev)
    copy = _us(lambda: z.copy_(y))
    assert _us(lambda: sgq.quantized_matmul_int4(x, qw, b, y)) < 2.3 * copy


@pytest.mark.parametrize("bits,G,M,K,N", [(4, 32, 140, 300, 256), (4, 64, 140, 300, 256), (4, 128, 140, 300, 256),
                                          (8, 0, 140, 301, 250), (8, 1, 140, 301, 250), (4, 32, 24, 4096, 4096),
                                          (8, 1, 24, 1030, 2048)])
def test_non_finite_inputs(sgq, dev, bits, G, M, K, N):
    """Infinities and NaNs land where x . (q * s) puts them: rows with one, with
    infinities of both signs, with a NaN in the last, partial run of k, and all NaN."""
    gen = torch.Generator(device=dev)
    gen.manual_seed(7)
    w = torch.randn(K, N, generator=gen, device=dev) * 0.02
    qw = sgq.quantize_int8(w, G) if bits == 8 else sgq.quantize_int4(w, G)
    x = torch.randn(M, K, generator=gen, device=dev)
    x[3, 17], x[11, K - 1], x[M - 1, 0] = float("inf"), float("nan"), -float("inf")
    x[5, 2], x[5, K - 2], x[7] = float("inf"), -float("inf"), float("nan")
    y = sgq.quantized_matmul(x, qw).double()
    ref = x.double().cpu() @ sgq.dequantize_codes(qw).double().cpu()
    ref = ref.to(dev)
    assert torch.equal(torch.isnan(y), torch.isnan(ref))
    assert torch.equal(torch.isinf(y), torch.isinf(ref))
    fin = torch.isfinite(ref)
    assert torch.equal(torch.sign(y[~fin & ~torch.isnan(ref)]), torch.sign(ref[~fin & ~torch.isnan(ref)]))


def _us(fn, reps=20):
    """The fastest of five queues of `reps` calls, us a call."""
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


@pytest.mark.parametrize("G,M,K,N", [(32, 256, 2048, 5632), (64, 256, 2048, 5632), (32, 24, 4096, 4096)])
def test_nan_rows_are_no_slower(sgq, dev, G, M, K, N):
    """A batch with inactive sequences holds rows of NaN; each of their outputs
    is recomputed, which must end as soon as it is known to be NaN (measured
    1.0 times the clean batch, 6 to 12 with whole sums)."""
    x, qw, b = _inputs(sgq, dev, M, K, N, G, 11)
    clean = _us(lambda: sgq.quantized_matmul_int4(x, qw, b))
    x[::8] = float("nan")
    assert _us(lambda: sgq.quantized_matmul_int4(x, qw, b)) < 2 * clean + 10


@pytest.mark.parametrize("M,K,N,G", [(256, 1000, 256, 32), (256, 1000, 256, 64), (256, 1000, 288, 96),
                                     (24, 4096, 4096, 32), (24, 4096, 4096, 64), (32, 2048, 5632, 128)])
def test_small_products(sgq, dev, M, K, N, G):
    """Products near fp32's smallest normal number (|x s| about 2^-126) keep
    their bits, on the wavefront tiles and the skinny kernel's super-block
    form; one below it may lose a subnormal's last place (2^-149, times a code
    of up to 8)."""
    x, qw, b = _inputs(sgq, dev, M, K, N, G, 8)
    x = x * 2.0**-118
    _check(sgq.quantized_matmul_int4(x, qw), x, sgq.dequantize_int4(qw), None, K, floor=K * 8 * 2.0**-149)


@pytest.mark.parametrize("bits,G", [(4, 128), (4, 32), (4, 24), (8, 0), (8, 1)])
@pytest.mark.parametrize("M,K,N", [(130, 256, 384), (300, 2048, 768), (1100, 96, 4224), (2051, 35, 4224), (182, 20, 1080)])
def test_gated_epilogue(sgq, dev, M, K, N, bits, G):
    """The gated MLP of GEMM batches: the up projection's epilogue multiplies
    by silu of the gate projection, the same values as the two forwards and an
    elementwise product (expf and the division are a few ulp from torch's)."""
    gen = torch.Generator(device=dev)
    gen.manual_seed(9)
    w = [torch.randn(K, N, generator=gen, device=dev) * 0.02 for _ in range(2)]
    b = [torch.randn(1, N, generator=gen, device=dev) for _ in range(2)]
    x = torch.randn(M, K, generator=gen, device=dev)
    q = [sgq.quantize_int8(v, G) if bits == 8 else sgq.quantize_int4(v, G) for v in w]
    gate, up = (sgq.quantized_matmul(x, q[i], b[i]).double() for i in range(2))
    h = sgq.quantized_swiglu(x, q[0], q[1], b[0], b[1])
    ref = gate / (1 + torch.exp(-gate)) * up
    assert float(((h.double() - ref).abs() / ref.abs().clamp_min(1e-30)).max()) < 16 * 2.0**-24


def test_rows_past_one_launch(sgq, dev):
    """More 64-row tiles than a launch takes: the second half's rows and outputs follow the first's."""
    M, K = (1 << 29) + 70, 5
    if torch.cuda.mem_get_info()[0] < 32 << 30:
        pytest.skip("needs 32 GiB of free GPU memory")
    gen = torch.Generator(device=dev)
    gen.manual_seed(5)
    x = torch.empty((M, K), device=dev)
    x.copy_(torch.arange(K, device=dev).float().expand(M, K))
    rows = torch.randn(200, K, generator=gen, device=dev)
    at = [0, (1 << 28) - 100, 1 << 28, M - 200]
    for a in at:
        x[a : a + 200] = rows
    qw = sgq.quantize_int8(torch.randn(K, 1, generator=gen, device=dev) * 0.02, 1)
    y, w = sgq.quantized_matmul_int8(x, qw), sgq.dequantize_int8(qw)
    for a in at[:1] + at[2:]:
        _check(y[a : a + 200], x[a : a + 200], w, None, K)
    _check(y[at[1] : at[1] + 100], x[at[1] : at[1] + 100], w, None, K)
    assert torch.equal(y[1000:2000], y[-2000:-1000])
