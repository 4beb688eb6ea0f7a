"""kad_dcn_prep against the separate conversions and kad_dcn_pack_weights, bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DT = {'f16': torch.float16, 'bf16': torch.bfloat16}


def _odd(t, shift):
    """t's values in memory that starts `shift` elements past an aligned address."""
    buf = torch.empty(t.numel() + shift, dtype=t.dtype, device='cuda')
    buf[shift:] = t.flatten().cuda()
    return buf[shift:].view(t.shape)


@pytest.mark.parametrize('dt', ['f16', 'bf16'])
@pytest.mark.parametrize('shift', [0, 3])
@pytest.mark.parametrize('n,cin,cout,h,w,mask,bias', [(1, 1, 1, 1, 1, True, True), (2, 33, 17, 5, 7, True, False),
                                                      (1, 64, 300, 12, 19, False, True), (3, 40, 16, 16, 16, False, False)])
def test_dcn_prep(dt, shift, n, cin, cout, h, w, mask, bias):
    from kadconv import _ext
    g = torch.Generator().manual_seed(cin + cout)
    mk = lambda *s: _odd(torch.randn(*s, generator=g).to(DT[dt]), shift)  # noqa: E731
    off, wt = mk(n, 18, h, w), mk(cout, cin, 3, 3)
    m = mk(n, 9, h, w) if mask else None
    b = mk(cout) if bias else None
    print(f'dcn prep {dt} {n, cin, cout, h, w} shift {shift}', flush=True)
    off32, m32, b32, wp = _ext.dcn_prep(off, m, wt, b)
    assert torch.equal(off32, off.float()) and torch.equal(wp, _ext.dcn_pack_weights(wt, DT[dt]))
    for got, src in ((m32, m), (b32, b)):
        assert got is None if src is None else torch.equal(got, src.float())
