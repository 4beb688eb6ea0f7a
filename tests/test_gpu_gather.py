"""Edges of the gathering deformable convolution and of its fused squeeze-excitation tail,
against the CPU oracle (tolerances of tests/_util.check_close: fp32 1e-4 of the output scale,
16-bit 1e-2).  Output channels around the 16 / 32 / 96 / 128-channel borders of the dispatch and of
the column blocks, input channels that leave a 64-byte step partly empty, odd and even counts of
steps, tiles with one row, stride 2 (footprints larger than the prefetch registers hold, one LDS
buffer instead of two), samples far outside the tile and the image."""
import pytest
import torch
import torch.nn.functional as F

from oracle import kadconv_oracle as O
from tests._util import check_close, nhwc_padded, quant

pytestmark = pytest.mark.gpu

DT = {'f32': torch.float32, 'f16': torch.float16, 'bf16': torch.bfloat16}


def _case(N, C, Co, H, W, stride, off_std, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    Ho, Wo = (H - 1) // stride + 1, (W - 1) // stride + 1
    x = torch.randn(N, C, H, W, generator=g)
    ow = torch.randn(18, C, 3, 3, generator=g) * (off_std / (9 * C) ** 0.5)
    ob = torch.randn(18, generator=g) * 0.3
    w = (torch.rand(Co, C, 3, 3, generator=g) * 2 - 1) / (9 * C) ** 0.5
    b = torch.randn(Co, generator=g) * 0.1
    mask = torch.rand(N, 9, Ho, Wo, generator=g)
    off = F.conv2d(quant(x, dtype), quant(ow, dtype), ob.double(), stride=stride, padding=1)
    ref = O.deform_conv2d(quant(x, dtype), off, quant(w, dtype), b.double(), stride=stride, padding=1,
                          mask=mask.double())
    return x, ow, ob, w, b, mask, off, ref


@pytest.mark.parametrize('dt', ['f16', 'bf16', 'f32'])
@pytest.mark.parametrize('mode', ['dsc', 'dcn'])
@pytest.mark.parametrize('shape,stride,off_std', [
    ((2, 8, 17, 11, 13), 1, 2.0), ((1, 24, 32, 16, 9), 1, 2.0), ((2, 31, 33, 12, 25), 1, 3.0),
    ((1, 65, 96, 20, 21), 1, 2.0), ((1, 33, 97, 9, 30), 1, 2.0), ((1, 130, 129, 14, 11), 1, 2.0),
    ((1, 48, 48, 1, 200), 1, 1.0), ((1, 40, 40, 50, 2), 1, 40.0), ((2, 16, 20, 25, 41), 2, 2.0),
    ((1, 20, 36, 5, 257), 2, 2.0), ((1, 72, 64, 67, 9), 2, 30.0)])
def test_gather_edges(dt, mode, shape, stride, off_std):
    from kadconv import _ext
    dtype = DT[dt]
    N, C, Co, H, W = shape
    x, ow, ob, w, b, mask, off, ref = _case(*shape, stride, off_std, dtype, seed=sum(shape))
    Ho, Wo = ref.shape[2:]
    print(f'gather {dt} {mode} {shape} stride={stride} off_std={off_std}', flush=True)
    xq = nhwc_padded(x.to(dtype).cuda())
    md = mask.permute(0, 2, 3, 1).contiguous().cuda()
    wp = _ext.dcn_pack_weights(w.to(dtype).cuda(), dtype)
    for layout in (_ext.KAD_NCHW, _ext.KAD_NHWC):
        cs = (Co + 7) // 8 * 8
        out = torch.empty(N, Co, Ho, Wo, dtype=dtype, device='cuda') if layout == _ext.KAD_NCHW else \
            torch.full((N, Ho, Wo, cs), 7.0, dtype=dtype, device='cuda')
        if mode == 'dsc':
            owp = _ext.dcn_pack_weights(ow.to(dtype).cuda(), dtype)
            _ext.dsc_fwd(xq, C, owp, ob.cuda(), md, (Ho * Wo * 9, 9, 1), wp, Co, out, stride=stride, bias=b.cuda(),
                         out_layout=layout)
        else:
            _ext.dcn_fwd(xq, C, off.float().permute(0, 2, 3, 1).contiguous().cuda(), (Ho * Wo * 18, 18, 1), md,
                         (Ho * Wo * 9, 9, 1), wp, Co, out, stride=stride, bias=b.cuda(), out_layout=layout)
        torch.cuda.synchronize()
        if layout == _ext.KAD_NHWC:
            assert (out[..., Co:] == 7.0).all()  # channels past Cout belong to the caller
            out = out[..., :Co].permute(0, 3, 1, 2)
        check_close(out, ref, dtype, f'{dt} {mode} {shape} layout {layout}')


@pytest.mark.parametrize('dt', ['f16', 'bf16', 'f32'])
@pytest.mark.parametrize('mode', ['dsc', 'dcn'])
@pytest.mark.parametrize('shape', [(2, 16, 16, 13, 21), (1, 17, 1, 9, 10), (2, 24, 15, 17, 11), (1, 33, 16, 12, 25),
                                   (1, 64, 9, 20, 7), (1, 130, 16, 11, 14), (1, 145, 16, 14, 9)])
def test_narrow_outputs(dt, mode, shape):
    """Up to 16 output channels: the narrow kernel and the gathering one with 16 columns, on both sides of
    the rule between them (half-chunks of 16 input channels, 128 channels)."""
    test_gather_edges(dt, mode, shape, 1, 2.0)


@pytest.mark.parametrize('dt', ['f16', 'bf16'])
@pytest.mark.parametrize('shape', [(2, 12, 16, 60, 64), (1, 40, 15, 64, 70), (1, 144, 16, 48, 61)])
def test_narrow_outputs_far_offsets(dt, shape):
    """The narrow kernel with offsets from memory, one, three and nine half-chunks, samples beyond the
    region that a tile stages."""
    test_gather_edges(dt, 'dcn', shape, 1, 12.0)


@pytest.mark.parametrize('c,hid', [(10, 32), (16, 16), (40, 40), (86, 86), (90, 91), (128, 128), (85, 7)])
def test_se_tail_sizes(c, hid):
    """Fused squeeze-excitation with weights that fit the LDS beside the partials and ones that do not
    (c = 90 x 91 and 128 x 128 take the general tail): att against the oracle's MLP on the mean of the
    kernel's own output, to fp32 rounding of sums of at most 128 terms (1e-5 on values in (0, 1))."""
    from kadconv import _ext
    dtype = torch.float16
    N, H, W = 3, 33, 47
    x, ow, ob, w, b, mask, _, _ = _case(N, c, c, H, W, 1, 2.0, dtype, seed=c + hid)
    g = torch.Generator().manual_seed(c * hid)
    w1, b1 = torch.randn(hid, c, generator=g) / c ** 0.5, torch.randn(hid, generator=g) * 0.1
    w2, b2 = torch.randn(c, hid, generator=g) / hid ** 0.5, torch.randn(c, generator=g) * 0.1
    print(f'se tail c={c} hid={hid}', flush=True)
    att = torch.empty(N, c, device='cuda')
    count = torch.zeros(N, dtype=torch.int32, device='cuda')
    gap = torch.empty(N, _ext.dcn_tiles(H, W), c, device='cuda')
    out = torch.empty(N, c, H, W, dtype=dtype, device='cuda')
    for _ in range(2):  # the counters are left zero
        att.fill_(-1)
        _ext.dsc_fwd(nhwc_padded(x.to(dtype).cuda()), c, _ext.dcn_pack_weights(ow.to(dtype).cuda(), dtype), ob.cuda(),
                     mask.permute(0, 2, 3, 1).contiguous().cuda(), (H * W * 9, 9, 1),
                     _ext.dcn_pack_weights(w.to(dtype).cuda(), dtype), c, out, bias=b.cuda(),
                     out_layout=_ext.KAD_NCHW, gap_partial=gap,
                     se=(w1.cuda(), b1.cuda(), w2.cuda(), b2.cuda(), att, count))
        torch.cuda.synchronize()
        m = out.double().cpu().mean((2, 3))
        ref = torch.sigmoid(F.linear(torch.relu(F.linear(m, w1.double(), b1.double())), w2.double(), b2.double()))
        assert (att.double().cpu() - ref).abs().max().item() <= 1e-5
    assert (count == 0).all()


@pytest.mark.parametrize('dt', ['f16', 'f32'])
@pytest.mark.parametrize('mode', ['dsc', 'dcn'])
@pytest.mark.parametrize('c,hid', [(300, 64), (513, 40), (4100, 4100), (4600, 4600), (7000, 16), (11760, 16)])
def test_se_tail_wide(dt, mode, c, hid):
    """The general tail of the fused squeeze-excitation, up to the widest layers the entry points take
    (Cout + hidden + 512 floats in 48 KB): att against the MLP in 64 bits on the mean of the kernel's own
    output.  Each weight row has 16 nonzeros, half of W1's among the last 64 channels.  Bound: the mean
    rounded in at most 16 steps, each layer's in at most 24 (adding a zero is exact) on the sums' absolute
    terms, sigmoid's slope 1 / 4, and 4 units for the sigmoid itself."""
    from kadconv import _ext
    dtype = DT[dt]
    N, C, H, W = 2, 8, 9, 11
    g = torch.Generator().manual_seed(c + hid)
    x = torch.randn(N, C, H, W, generator=g)
    w = torch.randn(c, C, 3, 3, generator=g) / (9 * C) ** 0.5
    def sparse(rows, cols):
        at = torch.cat((torch.randint(cols, (rows, 8), generator=g), cols - 1 - torch.randint(min(64, cols), (rows, 8), generator=g)), 1)
        return torch.zeros(rows, cols).scatter_(1, at, torch.randn(rows, 16, generator=g))

    w1, b1, w2, b2 = sparse(hid, c), torch.randn(hid, generator=g), sparse(c, hid), torch.randn(c, generator=g)
    print(f'wide se tail {dt} {mode} c={c} hid={hid}', flush=True)
    att = torch.full((N, c), -1.0, device='cuda')
    gap = torch.empty(N, _ext.dcn_tiles(H, W), c, device='cuda')
    out = torch.empty(N, c, H, W, dtype=dtype, device='cuda')
    kw = dict(out_layout=_ext.KAD_NCHW, gap_partial=gap,
              se=(w1.cuda(), b1.cuda(), w2.cuda(), b2.cuda(), att, torch.zeros(N, dtype=torch.int32, device='cuda')))
    xq, wp = nhwc_padded(x.to(dtype).cuda()), _ext.dcn_pack_weights(w.to(dtype).cuda(), dtype)
    ow = torch.randn(18, C, 3, 3, generator=g) / (9 * C) ** 0.5
    if mode == 'dsc':
        _ext.dsc_fwd(xq, C, _ext.dcn_pack_weights(ow.to(dtype).cuda(), dtype), None, None, None, wp, c, out, **kw)
    else:
        off = torch.randn(N, H, W, 18, generator=g).cuda()
        _ext.dcn_fwd(xq, C, off, (H * W * 18, 18, 1), None, None, wp, c, out, **kw)
    torch.cuda.synchronize()
    m, u = out.double().cpu().mean((2, 3)), 2.0 ** -24
    w1, b1, w2, b2 = (t.double() for t in (w1, b1, w2, b2))
    h = torch.relu(F.linear(m, w1, b1))
    ref = torch.sigmoid(F.linear(h, w2, b2))
    em = 16 * u * out.double().abs().cpu().mean((2, 3))
    eh = F.linear(em, w1.abs()) + 24 * u * (F.linear(m.abs(), w1.abs()) + b1.abs())
    tol = (F.linear(eh, w2.abs()) + 24 * u * (F.linear(h, w2.abs()) + b2.abs())) / 4 + 4 * u
    d = (att.double().cpu() - ref).abs()
    assert (d <= tol).all(), f'max excess {(d - tol).max().item():.2e}, max d {d.max().item():.2e}, tol {tol.max().item():.2e}'
