"""rms_norm over row lengths at the edges of its forms (quads kept in registers from
192 up to 2048 and 8192 floats, the scalar loop for the rest), in place and from an
address that is no multiple of 16, against 64 bits.  The sum of squares is D
positive terms in any order (relative error at most D * 2^-24, typically far
less: D / 256 per thread), then a division, a square root and two products."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [1, 3, 4, 188, 192, 196, 1020, 2044, 2048, 2052, 4099, 8188, 8192, 8196])
@pytest.mark.parametrize("rows", [1, 33])
def test_rows(sgq, dev, rows, D):
    import soverign_grad_amd.decode as decode

    gen = torch.Generator(device=dev)
    gen.manual_seed(D)
    x = torch.randn(rows * D + 1, generator=gen, device=dev)[1:].reshape(rows, D)
    g = torch.randn(D, generator=gen, device=dev)
    ref = x.double() / torch.sqrt((x.double() ** 2).mean(1, keepdim=True) + 1e-5) * g.double()
    y = decode.rms_norm(x, g, 1e-5)
    assert bool(((y.double() - ref).abs() <= (D // 256 + 24) * 2.0**-24 * ref.abs()).all())
    decode.rms_norm(x, g, 1e-5, out=x)
    assert torch.equal(x, y)
