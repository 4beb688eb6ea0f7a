"""kad_to_nhwc's 16-bit path for planes of any size against a permutation, bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DT = {'f16': torch.float16, 'bf16': torch.bfloat16}


@pytest.mark.parametrize('dt', ['f16', 'bf16'])
@pytest.mark.parametrize('n,c,h,w', [(1, 1, 1, 1), (2, 3, 1, 7), (3, 70, 5, 13), (2, 64, 9, 7), (1, 65, 1, 129),
                                     (2, 130, 25, 25), (1, 40, 50, 50), (5, 9, 3, 21)])
def test_to_nhwc_any_plane(dt, n, c, h, w):
    from kadconv import _ext
    x = torch.randn(n, c, h, w, generator=torch.Generator().manual_seed(c + w)).to(DT[dt]).cuda()
    cs = (c + 7) // 8 * 8
    out = torch.full((n, h, w, cs), float('nan'), dtype=DT[dt], device='cuda')
    print(f'to_nhwc {dt} {n, c, h, w}', flush=True)
    _ext.to_nhwc(x, out)
    torch.cuda.synchronize()
    assert torch.equal(out[..., :c], x.permute(0, 2, 3, 1)) and out[..., c:].abs().sum().item() == 0
