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
