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


@pytest.mark.parametrize('dt', ['f16', 'f32'])
def test_deform_conv2d_bias_length(dt):
    """A bias shorter than Cout is refused on the device too; one that has more elements uses the first Cout."""
    import kadconv
    dtype = {**DT, 'f32': torch.float32}[dt]
    x, off = torch.randn(1, 8, 5, 6).to('cuda', dtype), torch.randn(1, 18, 5, 6).to('cuda', dtype)
    w, b = torch.randn(40, 8, 3, 3).to('cuda', dtype), torch.randn(48).to('cuda', dtype)
    with pytest.raises(ValueError, match='bias has 1 elements for 40'):
        kadconv.deform_conv2d(x, off, w, b[:1], padding=1)
    assert torch.equal(kadconv.deform_conv2d(x, off, w, b, padding=1),
                       kadconv.deform_conv2d(x, off, w, b[:40].contiguous(), padding=1))
