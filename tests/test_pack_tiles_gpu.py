"""The pack kernels at the edges of their tiles (32 rows by 128 columns): codes,
scales, strips, k-octet copy, gap and device scales, from x (one pass, or with
scales found first) and from codes, bit for bit against the oracle's codes and
the numpy models of the layouts."""
import numpy as np
import pytest
import torch

import helpers

pytestmark = pytest.mark.gpu

KS = [1, 16, 31, 33, 100]


def _x(synth, K, N, seed):
    W = synth.normal((K, N), seed, synth.STREAM_W, 0.0, 0.02)
    W.reshape(-1)[:: 7 * N + 3] = 0.0
    W[0, 0] = np.nan  # NaN never wins the maximum and takes the largest code
    return W


@pytest.mark.parametrize("N,G", [(8, 8), (120, 8), (128, 128), (136, 8), (144, 16), (160, 32), (192, 64), (384, 128),
                                 (120, 24), (136, 128), (256, 256), (24, 32)])
@pytest.mark.parametrize("K", KS)
def test_int4_tiles(sgq, dev, oracle, synth, K, N, G):
    W = _x(synth, K, N, 40 + N)
    q, s = oracle.quantize_int4(W, G)
    flat = torch.from_numpy(np.r_[np.float32(0), W.reshape(-1)]).to(dev)
    for x in (torch.from_numpy(W).to(dev), flat[1:].reshape(K, N)):  # 16-byte and 4-byte addresses
        qw = sgq.quantize_int4(x, G)
        assert helpers.same_bits(qw.qdata.cpu().numpy(), q) and helpers.same_bits(qw.scales.cpu().numpy(), s)
        for got in (qw, sgq.pack_int4(qw.qdata, qw.scales, G), sgq.quantize_int4(x, G, keep_qdata=False)):
            assert np.array_equal(got.packed.cpu().numpy(), helpers.model_pack_i4_tiled(q, G))
            ds = helpers.model_devscales_i4(s, K, N, G).reshape(-1)
            assert helpers.same_bits(got.devscales.cpu().numpy()[: ds.size], ds)


@pytest.mark.parametrize("N", [1, 4, 127, 128, 129, 131, 260])
@pytest.mark.parametrize("K", KS)
@pytest.mark.parametrize("scheme", [0, 1])
def test_int8_tiles(sgq, dev, oracle, synth, K, N, scheme):
    W = _x(synth, K, N, 60 + N)
    q, s = oracle.quantize_int8(W, scheme)
    flat = torch.from_numpy(np.r_[np.float32(0), W.reshape(-1)]).to(dev)
    for x in (torch.from_numpy(W).to(dev), flat[1:].reshape(K, N)):
        qw = sgq.quantize_int8(x, scheme)
        assert helpers.same_bits(qw.qdata.cpu().numpy(), q) and helpers.same_bits(qw.scales.cpu().numpy(), s)
        for got in (qw, sgq.pack_int8(qw.qdata, qw.scales, scheme)):
            assert np.array_equal(got.packed.cpu().numpy()[: helpers.model_pack_i8(q).size], helpers.model_pack_i8(q))


@pytest.mark.parametrize("K,N", [(1, 65541), (65541, 2), (65541, 3), (65541, 16), (65541, 17), (524291, 4), (524291, 5)])
@pytest.mark.parametrize("scheme", [0, 1])
def test_int8_narrow(sgq, dev, oracle, synth, K, N, scheme):
    """Both sides of the line between the tiles and a thread per chunk."""
    W = _x(synth, K, N, 80 + N)
    q, s = oracle.quantize_int8(W, scheme)
    qw = sgq.quantize_int8(torch.from_numpy(W).to(dev), scheme)
    assert helpers.same_bits(qw.qdata.cpu().numpy(), q) and helpers.same_bits(qw.scales.cpu().numpy(), s)
    for got in (qw, sgq.pack_int8(qw.qdata, qw.scales, scheme), sgq.quantize_int8(torch.from_numpy(W).to(dev), scheme, keep_qdata=False)):
        assert np.array_equal(got.packed.cpu().numpy()[: helpers.model_pack_i8(q).size], helpers.model_pack_i8(q))
    bad = qw.qdata.clone()
    bad[-1, -1] = 0.5
    with pytest.raises(sgq.SGQError):
        sgq.pack_int8(bad, qw.scales, scheme)


def test_int8_narrow_is_no_slower_than_square(sgq, dev):
    """A column of 2^20 weights quantizes like a square of them (measured about the
    same; in tiles of 128 columns 3.2 times)."""
    def us(K, N):
        w = torch.randn(K, N, device=dev)
        best = float("inf")
        for _ in range(6):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            torch.cuda.synchronize()
            a.record()
            for _ in range(20):
                sgq.quantize_int8(w, 0, keep_qdata=False)
            b.record()
            b.synchronize()
            best = min(best, a.elapsed_time(b) * 1000 / 20)
        return best

    assert us(1 << 20, 1) < 2 * us(1 << 10, 1 << 10)


# Narrow weights whose tiles, 256 threads each, pass 2^32 threads: the last tile's
# rows and the first of the second launch come out like the first rows.
@pytest.mark.parametrize("bits,N", [(8, 1), (8, 5), (4, 8)])
def test_more_tiles_than_one_launch(sgq, dev, bits, N):
    K = (1 << 29) + 40
    if torch.cuda.mem_get_info()[0] < 64 << 30:
        pytest.skip("needs 64 GiB of free GPU memory")
    x = torch.empty((K, N), device=dev)
    rows = torch.arange(37, device=dev)
    small = ((rows[:, None] * 3 + torch.arange(N, device=dev)) % 15 - 7).float()
    at = [0, 1 << 27, (1 << 29) - 64, K - 37]  # 2^27 rows are the tiles of a launch
    x.zero_()
    for a in at:
        x[a : a + 37] = small
    qw = sgq.quantize_int8(x, 0, keep_qdata=False) if bits == 8 else sgq.quantize_int4(x, 8, keep_qdata=False)
    del x
    w = (sgq.dequantize_int8 if bits == 8 else sgq.dequantize_int4)(qw)
    want = w[:37].clone()
    assert (want - small).abs().max().item() <= 7.0 / (127 if bits == 8 else 7) / 2 + 1e-5
    for a in at:
        assert torch.equal(w[a : a + 37], want)
    assert not w[1 << 28 : (1 << 28) + 64].any()
