"""The INT8 skinny kernel with one, two and four column blocks per workgroup, at
widths with a partial strip, column block and workgroup, against x . (code *
scale) in 64 bits.  Sixteen wavefronts each add K / 512 k blocks of three MFMA
terms, then sixteen partial sums; each addition may round or truncate."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,K,N", [(16, 512, 11008), (16, 513, 11009), (9, 1024, 11003), (17, 519, 11010), (5, 2048, 20001),
                                   (16, 1024, 5632), (12, 1027, 5633), (33, 1024, 4097), (100, 1024, 4093),
                                   (16, 4096, 1024), (128, 1024, 1021)])
@pytest.mark.parametrize("scheme", [0, 1])
def test_column_blocks(sgq, dev, M, K, N, scheme):
    path, ks = ctypes.c_int(), ctypes.c_int()
    assert sgq.load_library().sgq_linear_plan(8, M, K, N, 0, 0, ctypes.byref(path), ctypes.byref(ks)) == 0
    assert path.value == 4
    gen = torch.Generator(device=dev)
    gen.manual_seed(M + N)
    qw = sgq.quantize_int8(torch.randn(K, N, generator=gen, device=dev) * 0.02, scheme, keep_qdata=False)
    x, b = torch.randn(M, K, generator=gen, device=dev), torch.randn(1, N, generator=gen, device=dev)
    w = sgq.dequantize_int8(qw).double()
    ref, mag = x.double() @ w + b.double(), x.double().abs() @ w.abs() + b.double().abs()
    bound = (3 * -(-K // 512) + 20) * 2.0**-23 * mag
    y = sgq.quantized_matmul_int8(x, qw, b).double()
    assert bool(((y - ref).abs() <= bound).all()), float(((y - ref).abs() / bound).max())
