"""The fp32 1x1 GEMM and 3x3 convolution kernels at the edges of their tiles and of their split of the
contraction (one, two and four shares by the number of blocks), against float64 torch: fp32 sums of K
products of unit-variance terms scaled to unit variance, max|d| <= 1e-5 of the output scale (K <= 2600:
sqrt(K) * 2^-24 is 3e-6)."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


def _close(got, ref, what):
    err = (got.double().cpu() - ref).abs().max().item()
    assert err <= 1e-5 * ref.abs().max().item(), f'{what}: max|d| = {err:.3e}'


@pytest.mark.parametrize('layout', ['nchw', 'nhwc'])
@pytest.mark.parametrize('n,cin,cout,h,w', [(1, 4, 3, 1, 3), (2, 20, 40, 5, 7), (1, 36, 65, 9, 31), (3, 16, 64, 25, 25),
                                            (2, 100, 33, 64, 64), (1, 48, 72, 190, 181), (2, 260, 130, 33, 35)])
def test_gemm_f32(layout, n, cin, cout, h, w):
    from kadconv import _ext, ops
    g = torch.Generator().manual_seed(cin + cout)
    x = torch.randn(n, cin, h, w, generator=g)
    wt = torch.randn(cout, cin, 1, 1, generator=g) / cin ** 0.5
    b = torch.randn(cout, generator=g)
    ref = F.silu(F.conv2d(x.double(), wt.double(), b.double()))
    print(f'gemm_f32 {layout} {n, cin, cout, h, w}', flush=True)
    xd = x.cuda()
    if layout == 'nhwc':
        xd = xd.contiguous(memory_format=torch.channels_last)
    _close(ops.conv1x1(xd, wt.cuda(), b.cuda(), act='silu'), ref, layout)
    if layout == 'nhwc':  # a channel slice of a wider buffer on both sides
        cs, os = cin + 12, (cout + 7) // 8 * 8 + 8
        xw = torch.full((n, h, w, cs), float('nan'), device='cuda')
        xw[..., 4:4 + cin] = x.permute(0, 2, 3, 1).cuda()
        out = torch.full((n, h, w, os), 7.0, device='cuda')
        wp = _ext.gemm_pack_weights(wt.cuda(), torch.float32)
        _ext.gemm1x1_nhwc(xw[..., 4:4 + cin], cin, wp, cout, out[..., :cout], bias=b.cuda(), act=_ext.KAD_ACT_SILU)
        _close(out[..., :cout].permute(0, 3, 1, 2), ref, 'slice')
        assert (out[..., cout:(cout + 7) // 8 * 8] == 0).all() and (out[..., (cout + 7) // 8 * 8:] == 7.0).all()


@pytest.mark.parametrize('n,cin,cout,h,w,stride', [(1, 3, 5, 4, 3, 1), (2, 24, 40, 9, 11, 1), (1, 40, 70, 33, 17, 2),
                                                   (2, 72, 64, 64, 65, 1), (1, 16, 33, 230, 170, 1),
                                                   (3, 288, 20, 8, 8, 2)])
@pytest.mark.parametrize('act', [0, 1, 2])
def test_conv3_f32(n, cin, cout, h, w, stride, act):
    from kadconv import _ext
    from tests._util import nhwc_padded
    g = torch.Generator().manual_seed(cin * cout)
    x = torch.randn(n, cin, h, w, generator=g)
    wt = torch.randn(cout, cin, 3, 3, generator=g) / (9 * cin) ** 0.5
    b = torch.randn(cout, generator=g)
    ref = F.conv2d(x.double(), wt.double(), b.double(), stride=stride, padding=1)
    ref = (ref, F.relu(ref), F.silu(ref))[act]
    code = (_ext.KAD_ACT_NONE, _ext.KAD_ACT_RELU, _ext.KAD_ACT_SILU)[act]
    print(f'conv3_f32 {n, cin, cout, h, w, stride, act}', flush=True)
    out = torch.full((n, ref.shape[2], ref.shape[3], cout + 5), 7.0, device='cuda')
    _ext.conv_fwd(nhwc_padded(x.cuda()), cin, _ext.dcn_pack_weights(wt.cuda(), torch.float32), cout, out[..., :cout],
                  stride=stride, pad=1, bias=b.cuda(), act=code)
    _close(out[..., :cout].permute(0, 3, 1, 2), ref, 'conv')
    assert (out[..., cout:] == 7.0).all()


@pytest.mark.parametrize('op', ['gemm', 'conv'])
@pytest.mark.parametrize('n,cin,cout,h,w', [
    (1, 16, 16, 50, 50), (2, 512, 20, 40, 41),                          # one k-step; up to 32 columns, many steps
    (2, 17, 16, 33, 9), (1, 32, 4, 90, 91), (8, 16, 16, 50, 50),        # convolutions of the general kernel
    (8, 33, 16, 46, 51), (8, 33, 16, 64, 64), (1, 33, 17, 128, 130)])   # and just past its rule
def test_splits_f32(op, n, cin, cout, h, w):
    """Both sides of the choice of the split and of the general convolution for up to 16 output channels."""
    (test_gemm_f32('nchw', n, cin, cout, h, w) if op == 'gemm' else test_conv3_f32(n, cin, cout, h, w, 1, 2))
