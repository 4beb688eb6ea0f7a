"""Parity of the fused HIP forwards (kadconv.enable_fast_inference, kadconv.ops,
kadconv.blocks) against the CPU oracle, at the sizes of the benchmark.

Weights are generated by state-dict name (oracle.make_*_state), loaded into
the product modules, and the modules are cast to the run dtype; the oracle
then runs in float64 on exactly those (quantised) weights and inputs.
Tolerances: fp32 max|d| <= 1e-4 max|ref|; fp16/bf16 max|d| <= 1e-2."""
import pytest
import torch

from kadconv import synthetic as S
from oracle import kadconv_oracle as O
from tests._util import check_close, quant

pytestmark = pytest.mark.gpu

DT = {'f32': torch.float32, 'f16': torch.float16, 'bf16': torch.bfloat16}


def _sd64(module):
    return {k: v.detach().double().cpu() for k, v in module.state_dict().items()}


def _kadconv(dim, dtype, seed=0, offset_std_px=None, se_min_hidden=32, n=3):
    import kadconv
    m = kadconv.KADConv(dim, n=n, se_min_hidden=se_min_hidden)
    sd = S.make_kadconv_state(dim, n=n, seed=seed, offset_std_px=offset_std_px, se_min_hidden=se_min_hidden)
    missing, unexpected = m.load_state_dict(sd, strict=False)
    assert not unexpected and all(k.endswith('num_batches_tracked') for k in missing)
    return m.to('cuda', dtype).eval()


def _x(shape, dtype, seed=0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(dtype)


@pytest.mark.parametrize('dt,shape', [
    ('f32', (1, 64, 80, 80)),       # config 1 shape, on the GPU path
    ('f16', (1, 64, 80, 80)),
    ('bf16', (2, 48, 37, 29)),      # odd sizes: floor pooling, ragged tiles
    ('f32', (2, 48, 37, 29)),
    ('f16', (8, 256, 100, 100)),    # metric config
])
def test_kadconv_fast_matches_oracle(dt, shape):
    import kadconv
    dtype = DT[dt]
    print(f'kadconv dt={dt} shape={shape}', flush=True)
    m = _kadconv(shape[1], dtype, seed=1)
    sd = _sd64(m)
    x = _x(shape, dtype, seed=2)
    kadconv.enable_fast_inference(m)
    with torch.no_grad():  # twice: the second call runs on recycled buffers (no reliance on fresh memory)
        got = m(x.cuda())
        got2 = m(x.cuda())
    torch.cuda.synchronize()
    ref = O.kadconv_forward(sd, x.double())
    check_close(got, ref, dtype, f'kadconv {dt} {shape}')
    check_close(got2, ref, dtype, f'kadconv {dt} {shape} (second call)')


@pytest.mark.parametrize('dt,n,shape', [('f16', 1, (2, 32, 24, 20)), ('f16', 2, (2, 48, 37, 29)),
                                         ('bf16', 2, (1, 40, 16, 40)), ('f32', 1, (1, 24, 13, 18))])
def test_kadconv_fewer_branches(dt, n, shape):
    """KADConv(dim, n) with n = 1 or 2: the pyramid's missing pooled branches (their
    waves and staging) and the shorter stream schedule."""
    import kadconv
    dtype = DT[dt]
    print(f'kadconv n={n} dt={dt} shape={shape}', flush=True)
    m = _kadconv(shape[1], dtype, seed=11, n=n)
    sd = _sd64(m)
    x = _x(shape, dtype, seed=12)
    kadconv.enable_fast_inference(m)
    with torch.no_grad():
        got = m(x.cuda())
    torch.cuda.synchronize()
    check_close(got, O.kadconv_forward(sd, x.double(), n=n), dtype, f'kadconv n={n} {dt} {shape}')


@pytest.fixture(params=['grouped', 'streams'])
def schedule(request, monkeypatch):
    """Both forward schedules of a KADConv layer: 'grouped' (this size of layer runs every stage as
    one launch on the caller's stream) and 'streams' (branch chains forked onto side streams, the
    schedule the KADConv(256) metric runs)."""
    from kadconv import fused
    if request.param == 'streams':
        monkeypatch.setattr(fused, 'GROUPED', False)
    return request.param


def test_kadconv_channels_last_and_disable_roundtrip(schedule):
    import kadconv
    dtype = torch.float16
    m = _kadconv(64, dtype, seed=3)
    sd = _sd64(m)
    x = _x((2, 64, 40, 48), dtype, seed=4)
    kadconv.enable_fast_inference(m)
    xc = x.cuda().contiguous(memory_format=torch.channels_last)
    print(f'channels_last schedule={schedule}', flush=True)
    with torch.no_grad():
        got = m(xc)
    assert got.is_contiguous(memory_format=torch.channels_last)
    ref = O.kadconv_forward(sd, x.double())
    check_close(got, ref, dtype, 'channels_last')
    assert hasattr(m, '_kad_plan')
    kadconv.disable_fast_inference(m)
    assert 'forward' not in vars(m) and not hasattr(m, '_kad_plan')


@pytest.mark.parametrize('dim,hw', [(64, (40, 48)), (96, (32, 36))])
def test_kadconv_channels_last_slices_in_place(schedule, dim, hw):
    """A channels-last input that is a channel slice of a wider NHWC buffer, written in place into
    a channel slice of another (the way KAD-CNet's concat buffers are used), on both schedules:
    the slice equals the oracle and the rest of the output buffer is untouched."""
    import kadconv
    dtype = torch.float16
    m = _kadconv(dim, dtype, seed=5)
    sd = _sd64(m)
    kadconv.enable_fast_inference(m)
    H, W = hw
    x = _x((2, dim, H, W), dtype, seed=6)
    big_in = torch.randn(2, H, W, dim + 24, generator=torch.Generator().manual_seed(7)).to('cuda', dtype)
    big_in[..., 16:16 + dim] = x.permute(0, 2, 3, 1).cuda()
    big_out = torch.full((2, H, W, dim + 40), 7.0, dtype=dtype, device='cuda')
    xin = big_in[..., 16:16 + dim].permute(0, 3, 1, 2)
    out = big_out[..., 8:8 + dim].permute(0, 3, 1, 2)
    print(f'channels_last slices schedule={schedule} dim={dim} hw={hw}', flush=True)
    with torch.no_grad():
        m._kad_plan.forward(xin, out=out)
    torch.cuda.synchronize()
    check_close(out, O.kadconv_forward(sd, x.double()), dtype, 'channels-last slice in place')
    assert (big_out[..., :8] == 7).all() and (big_out[..., 8 + dim:] == 7).all(), 'wrote outside its slice'


def test_plain_forward_on_gpu_uses_hip_deform():
    """The un-switched module (plain torch composition + HIP deform_conv2d)."""
    dtype = torch.float32
    m = _kadconv(32, dtype, seed=5)
    sd = _sd64(m)
    x = _x((2, 32, 24, 20), dtype, seed=6)
    with torch.no_grad():
        got = m(x.cuda())
    check_close(got, O.kadconv_forward(sd, x.double()), dtype, 'plain gpu')


@pytest.mark.parametrize('dt', ['f16', 'bf16'])
def test_kadconv_metric_state(dt):
    """The metric's exact workload: KADConv(256) at [8,256,100,100] with the bench's
    weights (kadconv.synthetic.make_metric_kadconv_state: conv_offset ~ N(0, 2/sqrt(9c)),
    offsets ~2 px, identity BN, unit branch scale), against the float64 oracle."""
    import kadconv
    dtype = DT[dt]
    print(f'kadconv metric state {dt}', flush=True)
    m = kadconv.KADConv(256)
    m.load_state_dict(S.make_metric_kadconv_state(256), strict=False)
    m = m.to('cuda', dtype).eval()
    sd = _sd64(m)
    x = torch.randn(8, 256, 100, 100, generator=torch.Generator().manual_seed(0)).to(dtype)
    kadconv.enable_fast_inference(m)
    with torch.no_grad():
        got = m(x.cuda())
    torch.cuda.synchronize()
    check_close(got, O.kadconv_forward(sd, x.double()), dtype, f'kadconv metric state {dt}')


@pytest.mark.parametrize('dt', ['f16', 'bf16', 'f32'])
@pytest.mark.parametrize('C,H', [(128, 100), (256, 50), (512, 25)])
def test_dsc_config2(dt, C, H):
    """Standalone DSC, batch 8, offsets ~N(0, 2) px."""
    import kadconv
    dtype = DT[dt]
    print(f'dsc dt={dt} C={C} H={H}', flush=True)
    d = kadconv.DSC(C, C)
    sd = S.make_dsc_state(C, C, seed=C, offset_std_px=2.0)
    d.load_state_dict(sd, strict=False)
    d = d.to('cuda', dtype).eval()
    sd = _sd64(d)
    x = _x((8, C, H, H), dtype, seed=C + 1)
    off = torch.nn.functional.conv2d(x.double(), sd['conv_offset.weight'], sd['conv_offset.bias'], padding=1)
    std = off.std().item()
    assert 1.6 < std < 2.4, std                         # offsets ~N(0, 2) px
    assert (off.abs() > 3).float().mean() > 0.05       # out-of-bounds samples occur at the borders
    kadconv.enable_fast_inference(d)
    with torch.no_grad():
        got = d(x.cuda())
    torch.cuda.synchronize()
    check_close(got, O.dsc_forward(sd, '', x.double()), dtype, f'dsc {dt} C={C}')


@pytest.mark.parametrize('layout', ['nchw', 'nhwc'])
@pytest.mark.parametrize('C,split', [(128, False), (130, True)])
def test_dsc_f32_conv_offset_launch(layout, C, split):
    """fp32 DSC: above 128 channels conv_offset is a launch of its own."""
    import kadconv
    d = kadconv.DSC(C, C)
    sd = S.make_dsc_state(C, C, seed=C, offset_std_px=2.0)
    d.load_state_dict(sd, strict=False)
    d = kadconv.enable_fast_inference(d.to('cuda').eval())
    x = _x((2, C, 13, 21), torch.float32, seed=C + 1)
    xd = x.cuda() if layout == 'nchw' else x.cuda().contiguous(memory_format=torch.channels_last)
    y = torch.zeros(2, 13, 21, (C + 7) // 8 * 8, device='cuda')
    st = d._kad_plan.stages(y, 2, 13, 21, torch.empty(2, C, 13, 21, device='cuda'), 0)
    assert any(name == 'conv_offset' for name, _ in st) == split
    with torch.no_grad():
        got = d(xd)
    check_close(got, O.dsc_forward(_sd64(d), '', x.double()), torch.float32, f'dsc f32 C={C} {layout}')


@pytest.mark.parametrize('dt,shape', [('f16', (16, 512, 50, 50)), ('f32', (2, 40, 9, 13)),
                                      ('bf16', (3, 72, 20, 21))])
def test_conv1x1_silu(dt, shape):
    """1x1 conv + SiLU, W ~ N(0, 0.02)."""
    import kadconv
    dtype = DT[dt]
    g = torch.Generator().manual_seed(7)
    N, C, H, W = shape
    m = kadconv.Conv1x1SiLU(C, C)
    with torch.no_grad():
        m.conv.weight.copy_(torch.randn(C, C, 1, 1, generator=g) * 0.02)
        m.conv.bias.copy_(torch.randn(C, generator=g) * 0.02)
    m = m.to('cuda', dtype).eval()
    x = _x(shape, dtype, seed=8)
    with torch.no_grad():
        got = m(x.cuda())
        got_cl = m(x.cuda().contiguous(memory_format=torch.channels_last))
    w = m.conv.weight.detach().double().cpu()
    b = m.conv.bias.detach().double().cpu()
    ref = O.conv1x1_silu(x.double(), w, b)
    check_close(got, ref, dtype, f'conv1x1 {dt}')
    check_close(got_cl, ref, dtype, f'conv1x1 channels_last {dt}')


@pytest.mark.parametrize('dt,n,cin,cout,h,w,act,bias', [
    ('f16', 2, 64, 96, 16, 16, 'silu', True),     # P % 8 == 0: 16-byte pixel runs
    ('bf16', 1, 72, 300, 10, 30, None, True),     # P % 8 == 4: 8-byte runs; Cout past one 256 block
    ('f16', 3, 40, 24, 9, 12, 'silu', False),     # Cin padded to 64, no bias, ragged 108-pixel tile
    ('f16', 2, 512, 512, 25, 26, 'silu', True),   # deep K, 650-pixel images
    ('f16', 2, 48, 40, 7, 9, 'silu', True),       # P % 4 != 0: general kernel
    # launches of >= 1024 128-pixel blocks take the 128-pixel tile (the cases above the 64-pixel one)
    ('f16', 8, 256, 512, 100, 100, 'silu', True),  # P % 8 == 0
    ('bf16', 16, 128, 1024, 50, 50, None, True),   # P % 8 == 4, ragged last tile, four channel blocks
])
def test_conv1x1_shapes(dt, n, cin, cout, h, w, act, bias):
    """kadconv.ops.conv1x1 (NCHW fast path and the general kernel) against
    F.conv2d (+ SiLU) in float64 on the quantised operands."""
    import torch.nn.functional as F
    from kadconv import ops
    dtype = DT[dt]
    g = torch.Generator().manual_seed(cin + cout + h)
    x = torch.randn(n, cin, h, w, generator=g).to(dtype)
    # outputs ~N(0, 0.3): |y| < 2, where a bf16 output's rounding stays below 1e-2
    wt = (torch.randn(cout, cin, 1, 1, generator=g) * (0.3 / cin ** 0.5)).to(dtype)
    b = torch.randn(cout, generator=g) * 0.1 if bias else None
    print(f'conv1x1 {dt} n={n} cin={cin} cout={cout} {h}x{w} act={act} bias={bias}', flush=True)
    got = ops.conv1x1(x.cuda(), wt.cuda(), None if b is None else b.cuda(), act=act)
    torch.cuda.synchronize()
    ref = F.conv2d(x.double(), wt.double(), None if b is None else b.double())
    if act == 'silu':
        ref = F.silu(ref)
    check_close(got, ref, dtype, f'conv1x1 {dt} {cin}->{cout} {h}x{w}')


@pytest.mark.parametrize('dt,shape', [('f16', (16, 1024, 25, 25)), ('f32', (2, 48, 7, 9)), ('bf16', (4, 96, 12, 12))])
def test_squeeze_excitation(dt, shape):
    """SE with reduction 16."""
    import kadconv
    dtype = DT[dt]
    C = shape[1]
    torch.manual_seed(9)
    m = kadconv.SqueezeExcitation(C, reduction=16).to('cuda', dtype).eval()
    x = _x(shape, dtype, seed=10)
    with torch.no_grad():
        got = m(x.cuda())
        got_cl = m(x.cuda().contiguous(memory_format=torch.channels_last))
    p = {k: v.detach().double().cpu() for k, v in m.state_dict().items()}
    ref = O.se_forward(x.double(), p['fc.0.weight'], p['fc.0.bias'], p['fc.2.weight'], p['fc.2.bias'])
    check_close(got, ref, dtype, f'se {dt}')
    check_close(got_cl, ref, dtype, f'se channels_last {dt}')


@pytest.mark.parametrize('dt,shape,red', [
    ('f16', (1, 5, 5, 3), 2),       # 75 elements: per-plane pool and scale (no 16-byte pieces)
    ('bf16', (3, 40, 2, 3), 4),     # 6-pixel planes: per-plane kernels
    ('f32', (2, 300, 9, 9), 16),    # C > 256: one tile slice per channel in the MLP
    ('f16', (2, 24, 3, 7), 4),      # 21-pixel planes, pieces straddling plane boundaries
    ('f32', (2, 320, 5, 6), 8),     # wide MLP kernel: C % 64 == 0, 40 hidden units
    ('bf16', (3, 1024, 4, 4), 16),  # wide MLP kernel at its largest C, 64 hidden units
    ('f16', (3, 6, 9, 9), 2),       # 81-pixel planes: layer 2 in the scale, pieces straddling planes
    ('bf16', (4, 34, 13, 5), 8),    # 65-pixel planes, 33 planes per scale block
    ('f16', (2, 64, 3, 3), 16),     # two-launch NCHW SE: 9-pixel planes, 4 hidden units
    ('bf16', (1, 32, 1, 8), 8),     # ... one piece per plane
    ('f32', (3, 96, 7, 11), 4),     # ... 77-pixel planes, fp32 pieces, 24 hidden units
])
def test_squeeze_excitation_edges(dt, shape, red):
    import kadconv
    dtype = DT[dt]
    torch.manual_seed(sum(shape))
    m = kadconv.SqueezeExcitation(shape[1], reduction=red).to('cuda', dtype).eval()
    x = _x(shape, dtype, seed=sum(shape))
    print(f'se {dt} {shape} r={red}', flush=True)
    with torch.no_grad():
        got = m(x.cuda())
    torch.cuda.synchronize()
    p = {k: v.detach().double().cpu() for k, v in m.state_dict().items()}
    ref = O.se_forward(x.double(), p['fc.0.weight'], p['fc.0.bias'], p['fc.2.weight'], p['fc.2.bias'])
    check_close(got, ref, dtype, f'se {dt} {shape}')


def test_se_nchw_repeat_and_graph():
    """kad_se_nchw (two launches, layer-1 shares in a per-call workspace): calls with a larger and
    then a smaller batch, graph replays with eager calls between them; every result is
    bit-identical to the first eager one of its input (fixed-order sums)."""
    import kadconv
    dtype = torch.float16
    torch.manual_seed(3)
    m = kadconv.SqueezeExcitation(1024, reduction=16).to('cuda', dtype).eval()
    xa = _x((16, 1024, 25, 25), dtype, seed=4).cuda()
    xb = _x((4, 1024, 25, 25), dtype, seed=5).cuda()
    with torch.no_grad():
        ra, rb = m(xa), m(xb)
        s = torch.cuda.Stream()
        s.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            m(xa)
        torch.cuda.current_stream().wait_stream(s)
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            ya = m(xa)
        for _ in range(3):
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(ya, ra)
            assert torch.equal(m(xb), rb)
    p = {k: v.detach().double().cpu() for k, v in m.state_dict().items()}
    ref = O.se_forward(xb.double().cpu(), p['fc.0.weight'], p['fc.0.bias'], p['fc.2.weight'], p['fc.2.bias'])
    check_close(rb, ref, dtype, 'se nchw small batch')


@pytest.mark.parametrize('n,c,hid,tiles', [(16, 1024, 64, 1), (3, 86, 32, 40), (5, 300, 18, 3), (2, 1000, 63, 1),
                                           (1, 7, 2, 5), (40, 1024, 64, 1), (2, 2048, 128, 1)])
def test_se_mlp_ws_matches_single_launch(n, c, hid, tiles):
    """kad_se_mlp_ws (each layer spread over the batch, hidden activations in a
    caller buffer) against kad_se_mlp (one block per image) and a float64 MLP on
    the same partial sums; shapes past the split path's limits (C > 1024,
    hid > 64) run kad_se_mlp and leave the workspace untouched.
    Tolerance: 1e-5 absolute on att (fp32 sums of <= 2048 terms)."""
    from kadconv import _ext
    dev = 'cuda'
    g = torch.Generator().manual_seed(n * 131 + c + hid)
    partial = torch.randn(n, tiles, c, generator=g).to(dev)
    w1 = (torch.randn(hid, c, generator=g) / c ** 0.5).to(dev)
    b1 = (torch.randn(hid, generator=g) * 0.1).to(dev)
    w2 = (torch.randn(c, hid, generator=g) / hid ** 0.5).to(dev)
    b2 = (torch.randn(c, generator=g) * 0.1).to(dev)
    inv = 1.0 / (tiles * 7.0)
    att_a = torch.full((n, c), float('nan'), device=dev)
    att_b = torch.full((n, c), float('nan'), device=dev)
    hidden = torch.full((n, hid), -1.0, device=dev)
    print(f'se_mlp_ws n={n} c={c} hid={hid} tiles={tiles}', flush=True)
    _ext.se_mlp(partial, tiles, inv, w1, b1, w2, b2, att_a, n, c, hid)
    _ext.se_mlp_ws(partial, tiles, inv, w1, b1, w2, b2, att_b, n, c, hid, hidden)
    torch.cuda.synchronize()
    gm = partial.double().sum(1) * inv
    h = torch.relu(gm @ w1.double().t() + b1.double())
    ref = torch.sigmoid(h @ w2.double().t() + b2.double())
    assert (att_a.double() - ref).abs().max().item() <= 1e-5
    assert (att_b.double() - ref).abs().max().item() <= 1e-5
    split = c <= 1024 and hid <= 64
    if split:
        assert (hidden.double() - h).abs().max().item() <= 1e-5
    else:
        assert (hidden == -1.0).all()


@pytest.mark.parametrize('dt,shape,c2', [('f16', (8, 256, 100, 100), 512), ('f32', (2, 24, 36, 44), 40),
                                         ('bf16', (1, 32, 27, 19), 16)])
def test_kaddown(dt, shape, c2):
    """KADDown (see oracle.kaddown_forward)."""
    import kadconv
    dtype = DT[dt]
    m = kadconv.KADDown(shape[1], c2)
    m.load_state_dict(S.make_kaddown_state(shape[1], c2, seed=11))
    m = m.to('cuda', dtype).eval()
    sd = _sd64(m)
    x = _x(shape, dtype, seed=12)
    with torch.no_grad():
        got = m(x.cuda())
    check_close(got, O.kaddown_forward(sd, x.double()), dtype, f'kaddown {dt}')


@pytest.mark.parametrize('dt,shape,c2,nb,cl', [
    ('f16', (2, 20, 32, 48), 72, 3, False),    # K = 60 (Cin padding), fast GEMM (P = 384)
    ('bf16', (2, 16, 20, 28), 300, 2, True),   # two branches, channels-last input and output
    ('f16', (1, 8, 17, 23), 24, 3, False),     # odd sizes: scalar input pass, general GEMM
    ('f32', (1, 8, 10, 12), 16, 3, False),     # 5 x 6 output planes: vector input pass, element resize loop
])
def test_kaddown_variants(dt, shape, c2, nb, cl):
    import kadconv
    dtype = DT[dt]
    m = kadconv.KADDown(shape[1], c2, n=nb)
    m.load_state_dict(S.make_kaddown_state(shape[1], c2, seed=nb, n=nb))
    m = m.to('cuda', dtype).eval()
    sd = _sd64(m)
    x = _x(shape, dtype, seed=nb + 20)
    xd = x.cuda()
    if cl:
        xd = xd.contiguous(memory_format=torch.channels_last)
    print(f'kaddown {dt} {shape} -> {c2} nb={nb} channels_last={cl}', flush=True)
    with torch.no_grad():
        got = m(xd)
    torch.cuda.synchronize()
    if cl:
        assert got.is_contiguous(memory_format=torch.channels_last)
    check_close(got, O.kaddown_forward(sd, x.double(), n=nb), dtype, f'kaddown {dt} nb={nb}')


def test_deform_conv2d_functional_torchvision_layout():
    import kadconv
    g = torch.Generator().manual_seed(13)
    x = torch.randn(2, 12, 15, 17, generator=g)
    off = torch.randn(2, 18, 15, 17, generator=g) * 3
    mask = torch.rand(2, 9, 15, 17, generator=g)
    w = torch.randn(20, 12, 3, 3, generator=g) * 0.1
    b = torch.randn(20, generator=g)
    got = kadconv.deform_conv2d(x.cuda(), off.cuda(), w.cuda(), b.cuda(), padding=1, mask=mask.cuda())
    ref = O.deform_conv2d(x.double(), off.double(), w.double(), b.double(), padding=1, mask=mask.double())
    check_close(got, ref, torch.float32, 'deform_conv2d')
    with pytest.raises(ValueError):
        kadconv.deform_conv2d(x.cuda(), off[:, :9].cuda(), w.cuda(), b.cuda(), padding=1)


@pytest.mark.parametrize('layout', ['nchw', 'nhwc'])
def test_graph_replay_matches_eager(schedule, layout):
    """The bench times HIP-graph replays of the fused forward (branch chains on forked side streams
    for the metric layer; grouped launches for small layers): on both schedules and both input
    layouts, every replay, with eager work and synchronisation in between, must equal the eager
    forward bit for bit (deterministic kernels)."""
    import kadconv
    mf = torch.channels_last if layout == 'nhwc' else torch.contiguous_format
    m = _kadconv(64, torch.float16, seed=3)
    kadconv.enable_fast_inference(m)
    static_x = _x((2, 64, 40, 36), torch.float16, seed=0).cuda().contiguous(memory_format=mf)
    print(f'graph replay schedule={schedule} layout={layout}', flush=True)
    with torch.no_grad():
        s = torch.cuda.Stream()
        s.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            m(static_x)
        torch.cuda.current_stream().wait_stream(s)
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            static_y = m(static_x)
        for seed in (1, 2, 3):
            xin = _x((2, 64, 40, 36), torch.float16, seed=seed).cuda().contiguous(memory_format=mf)
            ref = m(xin).clone()          # eager, same module
            torch.cuda.synchronize()
            static_x.copy_(xin)
            g.replay()
            torch.cuda.synchronize()
            print(f'graph replay seed={seed}', flush=True)
            assert torch.equal(static_y, ref), f'replay {seed} differs from eager'
    sd = _sd64(m)
    ref64 = O.kadconv_forward(sd, xin.double().cpu())
    check_close(static_y, ref64, torch.float16, 'graph replay vs oracle')


@pytest.mark.parametrize('layout', ['nchw', 'nhwc'])
def test_merge_channel_window(layout):
    """kad_branch_merge with a channel window writes exactly [c_begin, c_end):
    bilinear (align_corners=False) upsample x att + residual inside, the rest untouched."""
    import torch.nn.functional as F
    from kadconv import _ext
    g = torch.Generator().manual_seed(7)
    N, C, H, W, c_off, c, h, w = 2, 24, 13, 18, 5, 11, 7, 9
    z = torch.randn(N, h, w, 16, generator=g)
    z[..., c:] = 0
    att = torch.rand(N, c, generator=g)
    res = torch.randn(N, C, H, W, generator=g)
    up = F.interpolate(z[..., :c].permute(0, 3, 1, 2).double(), size=(H, W), mode='bilinear', align_corners=False)
    exp = res.double().clone()
    exp[:, c_off:c_off + c] += att.double()[:, :, None, None] * up
    dev = 'cuda'
    if layout == 'nchw':
        out = torch.full((N, C, H, W), 9.0, device=dev)
        resd, lay = res.to(dev), _ext.KAD_NCHW
    else:
        out = torch.full((N, H, W, C), 9.0, device=dev)
        resd, lay = res.permute(0, 2, 3, 1).contiguous().to(dev), _ext.KAD_NHWC
    _ext.branch_merge(out, lay, [{'z': z.to(dev), 'c': c, 'c_off': c_off, 'att': att.to(dev)}], residual=resd,
                      channels=(c_off, c_off + c))
    torch.cuda.synchronize()
    got = out.cpu().double() if layout == 'nchw' else out.cpu().double().permute(0, 3, 1, 2)
    assert (got[:, :c_off] == 9.0).all() and (got[:, c_off + c:] == 9.0).all()
    assert torch.allclose(got[:, c_off:c_off + c], exp[:, c_off:c_off + c], atol=1e-5)


@pytest.mark.parametrize('dt', ['f32', 'f16', 'bf16'])
@pytest.mark.parametrize('N,H,W', [(2, 13, 18), (3, 40, 40)])
@pytest.mark.parametrize('inplace,wide', [(False, False), (True, False), (True, True)])
def test_merge_nhwc_vector_branches(dt, N, H, W, inplace, wide):
    """kad_branch_merge, NHWC, window and channel count multiples of 8 (the one-thread-per-8-
    channels kernel) with every kind of branch: at the output's resolution (optionally read in
    place from the output's own channel window, as the channels-last KAD-Conv does), upsampled
    maps whose channel windows start at offsets that are not multiples of 8 (aligned pieces read
    with a shift), a map whose channel stride is not a multiple of 8 (element loads), and channels
    no branch covers (gate x residual).  wide: output and residual are channel slices of wider
    NHWC buffers (out_cs / res_cs), the neighbouring channels untouched.  Reference: F.interpolate
    in float64 on the dtype-rounded inputs; tolerance fp32 1e-5, fp16/bf16 1e-2 absolute."""
    import torch.nn.functional as F
    from kadconv import _ext
    dtype, dev = DT[dt], 'cuda'
    g = torch.Generator().manual_seed(N * 1000 + H + int(inplace))
    C = 64
    res = torch.randn(N, C, H, W, generator=g) * 0.25
    gate = torch.rand(C, generator=g) + 0.5
    exp_q = quant(res, dtype).clone()
    obuf = torch.full((N, H, W, C + 16 if wide else C), 9.0, dtype=dtype, device=dev)
    out = obuf[..., 8:8 + C] if wide else obuf
    brs = []
    # (c_off, c, cs, branch resolution, coeff); channels 61 .. 63 belong to no branch
    for c_off, c, cs, (h, w), coeff in [(0, 13, 16, (H, W), 1.0), (13, 22, 24, ((H + 1) // 2, (W + 1) // 2), 0.7),
                                        (35, 9, 12, ((H + 3) // 4, (W + 3) // 4), 1.3),
                                        (44, 17, 24, ((H + 3) // 4, (W + 3) // 4), 0.9)]:
        z = torch.randn(N, h, w, cs, generator=g) * 0.25
        att = torch.rand(N, c, generator=g)
        zc = quant(z[..., :c], dtype).permute(0, 3, 1, 2)
        up = zc if (h, w) == (H, W) else F.interpolate(zc, size=(H, W), mode='bilinear', align_corners=False)
        exp_q[:, c_off:c_off + c] += coeff * att.double()[:, :, None, None] * up
        if inplace and (h, w) == (H, W):
            out[..., c_off:c_off + c] = z[..., :c].to(dtype).to(dev)
            zd = out[..., c_off:c_off + c]
        else:
            zd = z.to(dtype).to(dev)
        brs.append({'z': zd, 'c': c, 'c_off': c_off, 'att': att.to(dev), 'coeff': coeff})
    exp_q *= gate.double()[None, :, None, None]
    print(f'merge nhwc vec {dt} {N}x{H}x{W} inplace={inplace}', flush=True)
    resd = res.permute(0, 2, 3, 1).contiguous().to(dtype).to(dev)
    if wide:  # the residual as a slice too, at another stride
        rbuf = torch.zeros(N, H, W, C + 24, dtype=dtype, device=dev)
        rbuf[..., 16:16 + C] = resd
        resd = rbuf[..., 16:16 + C]
    _ext.branch_merge(out, _ext.KAD_NHWC, brs, residual=resd, gate=gate.to(dev))
    torch.cuda.synchronize()
    got = out.cpu().double().permute(0, 3, 1, 2)
    if wide:
        assert (obuf[..., :8] == 9.0).all() and (obuf[..., 8 + C:] == 9.0).all()
    tol = 1e-5 if dtype == torch.float32 else 1e-2
    err = (got - exp_q).abs().max().item()
    assert err <= tol, f'max|d| = {err:.3e}'


@pytest.mark.parametrize('dt', ['f32', 'f16', 'bf16'])
@pytest.mark.parametrize('H,W,hw', [(16, 50, [(8, 25), (4, 12)]), (8, 1200, [(4, 600), (2, 300)]),
                                    (130, 8, [(65, 4), (32, 2)]), (100, 100, [(50, 50), (25, 25)])])
def test_merge_band_nchw(dt, H, W, hw):
    """kad_branch_merge, NCHW, disjoint branch windows on planes of a multiple of 8
    pixels (the 2 KB-run kernel): out[c] = gate[c] * (residual + coeff * att *
    bilinear_up(z)) (align_corners=False, kad_conv.py:117-121) in each branch's
    window, the channels outside every window untouched.  Runs of 1024 pixels
    span many rows (W = 8), exactly a row and a bit (W = 1000s) or ~10 rows.
    Reference: F.interpolate in float64 on the dtype-rounded inputs; tolerance
    fp32 1e-5, fp16/bf16 1e-2 absolute (values |v| < 4)."""
    import torch.nn.functional as F
    from kadconv import _ext
    dtype, dev = DT[dt], 'cuda'
    g = torch.Generator().manual_seed(H * 131 + W)
    N, C = 2, 40
    spans = [(3, 13), (16, 19)]           # (c_off, c)
    res = torch.randn(N, C, H, W, generator=g) * 0.25   # |out| < 2.5: bf16 output rounding < 1e-2
    gate = torch.rand(C, generator=g) + 0.5
    exp_q = quant(res, dtype).clone()
    brs = []
    for (c_off, c), (h, w), coeff in zip(spans, hw, (0.7, 1.3)):
        cs = (c + 7) // 8 * 8
        z = torch.randn(N, h, w, cs, generator=g) * 0.25
        z[..., c:] = 0
        att = torch.rand(N, c, generator=g)
        up = F.interpolate(quant(z[..., :c], dtype).permute(0, 3, 1, 2), size=(H, W), mode='bilinear',
                           align_corners=False)
        exp_q[:, c_off:c_off + c] += coeff * att.double()[:, :, None, None] * up
        brs.append({'z': z.to(dtype).to(dev), 'c': c, 'c_off': c_off, 'att': att.to(dev), 'coeff': coeff})
    exp_q *= gate.double()[None, :, None, None]
    out = torch.full((N, C, H, W), 9.0, dtype=dtype, device=dev)
    print(f'merge band {dt} {H}x{W}', flush=True)
    _ext.branch_merge(out, _ext.KAD_NCHW, brs, residual=res.to(dtype).to(dev), gate=gate.to(dev),
                      channels=(3, 35))
    torch.cuda.synchronize()
    got = out.cpu().double()
    assert (got[:, :3] == 9.0).all() and (got[:, 35:] == 9.0).all()
    tol = 1e-5 if dtype == torch.float32 else 1e-2
    err = (got[:, 3:35] - exp_q[:, 3:35]).abs().max().item()
    assert err <= tol, f'max|d| = {err:.3e}'


@pytest.mark.parametrize('edt', [torch.float16, torch.float32])
@pytest.mark.parametrize('n,c,h,w', [(2, 86, 25, 25), (1, 200, 13, 40), (3, 512, 9, 17)])
def test_lcsa_mask_split_matches_single(edt, n, c, h, w):
    """kad_lcsa_mask_split (the channel contraction split over blocks, partial logits
    added in split order by a second launch) against kad_lcsa_mask on the same
    inputs, for several split counts including one chunk per split.  Both sum
    the same fp32 products, only grouped differently: |d| <= 1e-5 after the
    sigmoid.  The unsplit kernel itself is pinned against the oracle by the DSC
    and KADConv parity tests (which also run the split path where the plan
    picks it)."""
    from kadconv import _ext
    dev = 'cuda'
    g = torch.Generator().manual_seed(c + h)
    arow = torch.randn(n, h, c, generator=g).to(dev)
    colm = torch.randn(n, w, c, generator=g).to(dev)
    params = (torch.randn(_ext.lcsa_params_elems(c), generator=g) * 0.3).to(dev)
    emat, ebias = _ext.lcsa_pack(params, c, edt)
    ref = torch.empty(n, h, w, 9, device=dev)
    _ext.lcsa_mask(arow, colm, params, emat, ebias, ref, n, c, h, w)
    nk = (c + 31) // 32
    for ks in sorted({2, 3, nk, _ext.lcsa_mask_splits(n, c, h, w)}):
        if ks < 2 or ks > nk:
            continue
        print(f'lcsa split {edt} n={n} c={c} {h}x{w} ksplit={ks}', flush=True)
        work = torch.full((_ext.lcsa_mask_work_elems(n, h, w, ks),), float('nan'), device=dev)
        got = torch.full((n, h, w, 9), float('nan'), device=dev)
        _ext.lcsa_mask(arow, colm, params, emat, ebias, got, n, c, h, w, ks, work)
        torch.cuda.synchronize()
        err = (got - ref).abs().max().item()
        assert err <= 1e-5, f'ksplit={ks}: max|d| = {err:.3e}'


@pytest.mark.parametrize('dt', ['f32', 'f16', 'bf16'])
@pytest.mark.parametrize('shape', [(2, 5, 100, 100), (3, 7, 13, 9), (1, 3, 1, 12288), (2, 4, 110, 111)])
def test_axial_sums_nchw(dt, shape):
    """kad_axial_sums_nchw: row sums [N, H, C] and column sums [N, W, C] of an
    NCHW map (LCSA's pool_h / pool_w numerators, kad_conv.py:26-27) against
    float64 sums of the same dtype-rounded input; both the 4-element and the
    scalar plane loads (H*W % 4 != 0), the largest plane.  Tolerance: 1e-5
    relative to the largest |sum| (fp32 sums of at most 12288 values)."""
    from kadconv import _ext
    dtype, dev = DT[dt], 'cuda'
    N, C, H, W = shape
    g = torch.Generator().manual_seed(H * W + C)
    x = torch.randn(N, C, H, W, generator=g).to(dtype)
    rows = torch.full((N, H, C), float('nan'), device=dev)
    cols = torch.full((N, W, C), float('nan'), device=dev)
    print(f'axial nchw {dt} {shape}', flush=True)
    _ext.axial_sums_nchw(x.to(dev), rows, cols)
    torch.cuda.synchronize()
    xd = x.double()
    for got, ref, what in [(rows, xd.sum(3).permute(0, 2, 1), 'rows'), (cols, xd.sum(2).permute(0, 2, 1), 'cols')]:
        err = (got.cpu().double() - ref).abs().max().item()
        assert err <= 1e-5 * max(ref.abs().max().item(), 1.0), f'{what}: max|d| = {err:.3e}'


@pytest.mark.parametrize('dt', ['f32', 'f16', 'bf16'])
@pytest.mark.parametrize('shape', [(2, 5, 100, 100), (3, 7, 13, 9), (1, 86, 25, 25), (2, 4, 110, 111)])
def test_axial_means_equal_sums_then_prep(dt, shape):
    """kad_axial_means (NHWC) and kad_axial_means_nchw write LCSA's arow / colm in one launch;
    they must equal kad_axial_sums(_nchw) followed by kad_lcsa_prep of that one slice bit for
    bit (the same sums times the same 1/W, 1/H)."""
    from kadconv import _ext
    from tests._util import nhwc_padded
    dtype, dev = DT[dt], 'cuda'
    N, C, H, W = shape
    g = torch.Generator().manual_seed(H * W + C + 1)
    x = torch.randn(N, C, H, W, generator=g).to(dtype).to(dev)
    xh = nhwc_padded(x)
    print(f'axial means {dt} {shape}', flush=True)
    for layout in ('nchw', 'nhwc'):
        rows = torch.empty(N, H, C, device=dev)
        cols = torch.empty(N, W, C, device=dev)
        arow_ref = torch.full((N, H, C), float('nan'), device=dev)
        colm_ref = torch.full((N, W, C), float('nan'), device=dev)
        arow = torch.full((N, H, C), float('nan'), device=dev)
        colm = torch.full((N, W, C), float('nan'), device=dev)
        if layout == 'nchw':
            _ext.axial_sums_nchw(x, rows, cols)
            _ext.axial_means_nchw(x, arow, colm)
        else:
            _ext.axial_sums(xh, C, rows, cols)
            _ext.axial_means(xh, C, arow, colm)
        _ext.lcsa_prep(rows, 1, cols, 1, arow_ref, colm_ref, N, C, H, W)
        torch.cuda.synchronize()
        assert torch.equal(arow, arow_ref) and torch.equal(colm, colm_ref), layout


@pytest.mark.parametrize('dt', ['f32', 'f16', 'bf16'])
@pytest.mark.parametrize('shape', [(2, 37, 16, 10), (1, 130, 7, 9), (3, 64, 100, 100), (1, 8, 1, 8)])
def test_to_nhwc(dt, shape):
    """kad_to_nhwc: NCHW -> NHWC with the channel stride padded to a multiple of 8
    and the pad channels written 0 (bit-exact copy); the 16-byte path (planes of
    a multiple of 8 pixels) and the element path."""
    from kadconv import _ext
    dtype, dev = DT[dt], 'cuda'
    N, C, H, W = shape
    x = torch.randn(*shape, generator=torch.Generator().manual_seed(C * H)).to(dtype)
    cs = (C + 7) // 8 * 8
    out = torch.full((N, H, W, cs), float('nan'), dtype=dtype, device=dev)
    _ext.to_nhwc(x.to(dev), out)
    torch.cuda.synchronize()
    got = out.cpu()
    assert torch.equal(got[..., :C], x.permute(0, 2, 3, 1)), 'values'
    assert (got[..., C:] == 0).all(), 'pad channels'


@pytest.mark.parametrize('dt', ['f32', 'f16', 'bf16'])
@pytest.mark.parametrize('shape,wide', [((2, 12, 20, 18), 12), ((1, 21, 7, 9), 33), ((3, 10, 25, 25), 10), ((1, 1, 3, 5), 4)])
def test_nhwc_pad(dt, shape, wide):
    """kad_nhwc_pad: a channels-last tensor (pixel stride = C, or the first C channels of a wider
    channels-last buffer) -> NHWC with the channel stride padded to a multiple of 8, pad channels 0,
    bit-exact, in one launch; and ops._nhwc_view takes it for a channels-last input."""
    from kadconv import _ext, ops
    dtype, dev = DT[dt], 'cuda'
    N, C, H, W = shape
    base = torch.randn(N, wide, H, W, generator=torch.Generator().manual_seed(C * H + wide)).to(dtype)
    buf = base.to(dev).contiguous(memory_format=torch.channels_last)
    x = buf[:, :C]                       # NCHW-shaped view of channels-last memory, pixel stride `wide`
    cs = (C + 7) // 8 * 8
    out = torch.full((N, H, W, cs), float('nan'), dtype=dtype, device=dev)
    _ext.nhwc_pad(x.permute(0, 2, 3, 1), out)
    v, vcs = ops._nhwc_view(x)
    torch.cuda.synchronize()
    ref = base[:, :C].permute(0, 2, 3, 1)
    got = out.cpu()
    assert torch.equal(got[..., :C], ref) and (got[..., C:] == 0).all()
    if C % 8 == 0 and wide == C:
        assert v.data_ptr() == buf.data_ptr()          # already usable: no copy
    else:
        assert vcs == cs and torch.equal(v.cpu(), got)


def test_empty_batch():
    """A batch of 0 images: DSC, deform_conv2d and the blocks give the empty
    output of the module's shape, as torchvision's deform_conv2d and the plain
    PyTorch modules do; KADConv raises, as the reference's module does (its SE
    reshape .view(x.size(0), -1, 1, 1) of 0 elements, KAD-Conv/kadconv/kad_conv.py:117)."""
    import kadconv
    from kadconv import ops
    dev = 'cuda'
    m = _kadconv(32, torch.float16)
    kadconv.enable_fast_inference(m)
    d = kadconv.DSC(16, 24).to(dev).eval()
    kadconv.enable_fast_inference(d)
    with torch.no_grad():
        with pytest.raises(RuntimeError):
            m(torch.empty(0, 32, 24, 20, dtype=torch.float16, device=dev))
        assert d(torch.empty(0, 16, 9, 7, device=dev)).shape == (0, 24, 9, 7)
        y = ops.deform_conv2d(torch.empty(0, 8, 10, 12, device=dev), torch.empty(0, 18, 10, 12, device=dev),
                              torch.randn(5, 8, 3, 3, device=dev), padding=1)
        assert y.shape == (0, 5, 10, 12)
        assert kadconv.Conv1x1SiLU(8, 12).to(dev).eval()(torch.empty(0, 8, 6, 6, device=dev)).shape == (0, 12, 6, 6)
        assert kadconv.SqueezeExcitation(32).to(dev).eval()(torch.empty(0, 32, 6, 6, device=dev)).shape == (0, 32, 6, 6)
        assert kadconv.KADDown(8, 16).to(dev).eval()(torch.empty(0, 8, 16, 16, device=dev)).shape == (0, 16, 8, 8)
    torch.cuda.synchronize()


def test_graph_survives_larger_eager_batch():
    """A graph captured at batch 1, then an eager forward at batch 2 (which needs
    larger SE arrival counters), then the batch-1 graph replayed: the replay must
    still equal the eager batch-1 forward (the counters it captured stay alive)."""
    import kadconv
    m = _kadconv(48, torch.float16, seed=21)
    kadconv.enable_fast_inference(m)
    x1 = _x((1, 48, 32, 40), torch.float16, seed=22).cuda()
    x2 = _x((2, 48, 32, 40), torch.float16, seed=23).cuda()
    with torch.no_grad():
        static_x = x1.clone()
        s = torch.cuda.Stream()
        s.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            m(static_x)
        torch.cuda.current_stream().wait_stream(s)
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            static_y = m(static_x)
        ref1 = m(x1).clone()
        for rep in range(3):
            y2 = m(x2).clone()           # eager, larger batch, between the replays
            torch.cuda.synchronize()
            g.replay()
            torch.cuda.synchronize()
            print(f'graph after larger batch: replay {rep}', flush=True)
            assert torch.equal(static_y, ref1), f'replay {rep} differs from eager'
    sd = _sd64(m)
    check_close(y2, O.kadconv_forward(sd, x2.double().cpu()), torch.float16, 'eager batch 2')


@pytest.mark.parametrize('n,shape', [(4, (1, 8, 32, 32)), (3, (1, 4, 520, 520))])
def test_kaddown_outside_one_pass_kernel(n, shape):
    """KADDown with more branches than the one-pass input kernel covers (n = 4), or
    planes whose pools exceed its LDS staging (520 x 520), takes the plain
    composition instead of raising, and still matches the oracle."""
    import kadconv
    dtype = torch.float32
    m = kadconv.KADDown(shape[1], 6, n=n)
    m.load_state_dict(S.make_kaddown_state(shape[1], 6, seed=n, n=n))
    m = m.to('cuda', dtype).eval()
    sd = _sd64(m)
    x = _x(shape, dtype, seed=n)
    print(f'kaddown plain route n={n} {shape}', flush=True)
    with torch.no_grad():
        got = m(x.cuda())
    torch.cuda.synchronize()
    check_close(got, O.kaddown_forward(sd, x.double(), n=n), dtype, f'kaddown n={n}')
