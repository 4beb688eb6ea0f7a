"""kad_axial_sums: row and column sums of an NHWC map against float64, at the channel counts where
the split of a line over the block's threads changes (one piece, a wave of pieces, more than a block)
and on both load widths (16-byte pieces, single elements)."""
import pytest
import torch

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -24


@pytest.mark.parametrize('dt', [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize('c,cs,shift', [(1, 8, 0), (12, 16, 0), (12, 12, 0), (40, 48, 8), (65, 67, 1), (300, 304, 0),
                                        (513, 520, 0), (1030, 1032, 0), (2060, 2064, 0)])
@pytest.mark.parametrize('h,w', [(1, 5), (9, 130)])
def test_axial_sums_nhwc(dt, c, cs, shift, h, w):
    from kadconv import _ext
    g = torch.Generator().manual_seed(c + h)
    flat = torch.randn(2 * h * w * cs + shift, generator=g).to(dt)
    buf = flat[shift:].view(2, h, w, cs)
    x = flat.cuda()[shift:].view(2, h, w, cs)
    rows, cols = (torch.full((2, k, c), float('nan'), device='cuda') for k in (h, w))
    print(f'axial nhwc {dt} c {c} cs {cs} {h}x{w}', flush=True)
    _ext.axial_sums(x, c, rows, cols)
    torch.cuda.synchronize()
    xd = buf[..., :c].double()
    # n - 1 additions in fp32, in any order: |d| <= n eps sum |x|
    for got, dim, n in ((rows, 2, w), (cols, 1, h)):
        bound = n * EPS * xd.abs().sum(dim) + 1e-30
        assert ((got.cpu().double() - xd.sum(dim)).abs() <= bound).all()
