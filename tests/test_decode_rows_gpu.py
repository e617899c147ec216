"""Block decode of batches past the GEMV form, at real widths: the skinny kernel's
super-block form (q, k and v in a launch, the gated product, residuals with and
without a K split), the GEMM of wavefront tiles and the fp32 MFMA GEMM with
three weights, K splits, the gate and residuals in their epilogues, and a
projection left to the GEMV.  The reference is the block in 64 bits from the
dequantized weights; the error bound is the one of the block tests, the
largest difference of a row over its largest value at most 1e-5.
"""
import ctypes
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

TOL = 1e-5
EPS = 1e-5
GEMV, GEMM, GEMM_OTHER, SKINNY = 0, 1, 2, 4
# B, D, H, heads, G, and the forward plan (kernel, K split over workgroups) of
# q, k and v side by side, o, gate, down on a full device
CASES = [
    (17, 2048, 5632, 16, 32, [(SKINNY, False), (GEMV, False), (SKINNY, False), (SKINNY, True)]),
    (32, 2048, 5632, 16, 128, [(SKINNY, False), (GEMV, False), (SKINNY, False), (SKINNY, True)]),
    (32, 4096, 4096, 32, 128, [(SKINNY, False), (SKINNY, True), (SKINNY, True), (SKINNY, True)]),
    (32, 8192, 2048, 64, 64, [(SKINNY, False), (SKINNY, False), (SKINNY, True), (SKINNY, False)]),
    (33, 2048, 5632, 16, 32, [(GEMM_OTHER, True), (GEMV, False), (GEMM_OTHER, True), (GEMM_OTHER, True)]),
    (33, 1024, 8192, 8, 128, [(GEMV, False), (GEMV, False), (GEMM, True), (GEMM, True)]),
    (48, 2048, 5632, 16, 24, [(GEMM_OTHER, True), (GEMV, False), (GEMM_OTHER, True), (GEMM_OTHER, True)]),
    (40, 4096, 11008, 32, 128, [(GEMM, True), (GEMM, True), (GEMM, True), (GEMM, True)]),
    (300, 512, 1408, 8, 64, [(GEMM_OTHER, True), (GEMM_OTHER, True), (GEMM_OTHER, True), (GEMM_OTHER, True)]),
]
IDS = [f"{c[0]}x{c[1]}x{c[2]}g{c[4]}" for c in CASES]


@pytest.mark.parametrize("B,D,H,heads,G,plans", CASES, ids=IDS)
def test_plans(sgq, B, D, H, heads, G, plans):
    """The shapes reach what the module says (on a full device)."""
    lib = sgq.load_library()
    for (K, N), (path, split) in zip([(D, 3 * D), (D, D), (D, H), (H, D)], plans):
        p, ks = ctypes.c_int(), ctypes.c_int()
        assert lib.sgq_linear_plan(4, B, K, N, G, 256, ctypes.byref(p), ctypes.byref(ks)) == 0
        assert (p.value, ks.value > 1) == (path, split), (K, N, p.value, ks.value)


def _row_err(y, ref):
    return float(((y.double() - ref).abs().amax(-1) / ref.abs().amax(-1)).max())


@pytest.mark.parametrize("bias", [True, False])
@pytest.mark.parametrize("B,D,H,heads,G,plans", CASES, ids=IDS)
def test_block_rows(sgq, dev, B, D, H, heads, G, plans, bias):
    import soverign_grad_amd.decode as decode

    gen = torch.Generator(device=dev)
    gen.manual_seed(B + D + G)

    def normal(*shape, std=1.0):
        return torch.randn(*shape, generator=gen, device=dev) * std

    q, b = {}, {}
    for p, (K, N) in decode.projection_shapes(D, H).items():
        q[p] = sgq.quantize_int4(normal(K, N, std=0.02), G)
        b[p] = normal(N, std=0.05) if bias else None
    n1, n2 = 1 + normal(D, std=0.1), 1 + normal(D, std=0.1)
    blk = decode.QuantizedLLaMABlock.from_codes({p: w.qdata for p, w in q.items()}, {p: w.scales for p, w in q.items()},
                                                b, n1, n2, heads, G, EPS)
    x, ctx = normal(B, D), 21
    k, v = normal(B, ctx + 3, D), normal(B, ctx + 3, D)
    pos = torch.randint(0, ctx + 1, (B,), generator=gen, device=dev, dtype=torch.int32)
    pos[0], pos[B // 2] = ctx, -1  # an inactive sequence in the middle
    k64, v64, kept = k.double(), v.double(), (k.clone(), v.clone())
    y = blk.decode(x, k, v, pos, ctx + 1)

    def proj(a, p):
        r = a @ sgq.dequantize_int4(q[p]).double()
        return r if b[p] is None else r + b[p].double()

    def rms(a, g):
        return a / torch.sqrt((a * a).mean(-1, keepdim=True) + EPS) * g.double()

    n = rms(x.double(), n1)
    qh, kn, vn = proj(n, "q"), proj(n, "k"), proj(n, "v")
    att = torch.zeros_like(qh)
    live = [i for i in range(B) if i != B // 2]
    for i in live:
        t = int(pos[i])
        k64[i, t], v64[i, t] = kn[i], vn[i]
        score = (k64[i, : t + 1] @ qh[i]) / math.sqrt(D // heads)
        att[i] = torch.softmax(score, 0) @ v64[i, : t + 1]
    h = x.double() + proj(att, "out")
    n = rms(h, n2)
    g = proj(n, "gate")
    ref = h + proj(g / (1 + torch.exp(-g)) * proj(n, "up"), "down")

    assert bool(torch.isnan(y[B // 2]).all())
    assert _row_err(y[live], ref[live]) <= TOL
    at = [(i, int(pos[i])) for i in live]
    for got, new, old in ((k, kn, kept[0]), (v, vn, kept[1])):
        assert _row_err(torch.stack([got[i, t] for i, t in at]), new[live]) <= TOL
        for i, t in at:
            old[i, t] = got[i, t]
        assert torch.equal(got, old)  # and no other row of the cache moved
