"""The workloads this framework is timed on: its layers, its operators and its detector, through the
public entry points, at the sizes of its benchmark, its tests and the KAD-CNet-S configuration.

    listed()            the fixed cases
    draw(rng)           one more case of the same ranges
    prepare(case, s)    inputs and layers of a case on the GPU, made from the seed
    run(state)          one pass
    work(case)          bytes and flops that one pass cannot do without
    tolerance(case)     how far another correct implementation at the same precision may be
    exact(case, s)      the same outputs in 64 bits, from plain torch on the CPU

``call`` says how the program calls: 'graph' replays a HIP graph captured once (how the benchmark and
a serving loop run a layer of fixed shape), 'eager' calls the layer or the operator itself.
"""
import functools
import math
import os
import sys

import torch
import torch.nn.functional as F

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), 'kad-conv_amd'))

DTYPES = {'f32': torch.float32, 'f16': torch.float16, 'bf16': torch.bfloat16}
BN_EPS = 1e-3
NET_CLASSES, NET_BOX = 20, 64
NET_GFLOP_800 = 38.87  # of one 3 x 800 x 800 image: convolutions, Linears and deformable 3 x 3, 2 per multiply-add


def listed():
    return [
        # The headline layer: KADConv(256) on the [8, 256, 100, 100] neck map of a detector, served in fp16.
        dict(name='kadconv256_100_f16', op='kadconv', n=8, c=256, h=100, w=100, dtype='f16', layout='nchw', call='graph'),
        # A KAD-Conv layer of a channels-last bf16 network, ragged map and a width that is not a multiple of 8 per branch.
        dict(name='kadconv96_cl_bf16', op='kadconv', n=4, c=96, h=75, w=61, dtype='bf16', layout='nhwc', call='graph'),
        # The smallest layer call: one image in fp32, called directly (the sanity configuration, 64 channels at 80 x 80).
        dict(name='kadconv64_n1_f32', op='kadconv', n=1, c=64, h=80, w=80, dtype='f32', layout='nchw', call='eager'),
        # A standalone deformable convolution at the finest neck scale.
        dict(name='dsc128_100_f16', op='dsc', n=8, c=128, h=100, w=100, dtype='f16', layout='nchw', call='graph'),
        # The same at the coarsest scale: many channels, few pixels.
        dict(name='dsc512_25_bf16', op='dsc', n=8, c=512, h=25, w=25, dtype='bf16', layout='nchw', call='graph'),
        # A detector's narrow channels-last deformable convolution (KAD-CNet-S, first branch at 100 x 100).
        dict(name='dsc12_cl_f16', op='dsc', n=16, c=12, h=100, w=100, dtype='f16', layout='nhwc', call='graph'),
        # The operator in place of torchvision's, called with the offsets and masks of a program's own network.
        dict(name='dcn256_50_f16', op='dcn', n=8, c=256, h=50, w=50, dtype='f16', layout='nchw', call='eager'),
        # The stride-2 multi-branch downsampler between two neck scales.
        dict(name='down256_512_f16', op='down', n=8, c=256, c2=512, h=100, w=100, dtype='f16', layout='nchw', call='graph'),
        # A fused 1 x 1 convolution + SiLU.
        dict(name='conv1x1_512_50_f16', op='conv1x1', n=16, c=512, c2=512, h=50, w=50, dtype='f16', layout='nchw', call='graph'),
        # A squeeze-excitation block.
        dict(name='se1024_25_f16', op='se', n=16, c=1024, h=25, w=25, dtype='f16', layout='nchw', call='graph'),
        # The detector on a batch of 800 x 800 images in fp16.
        dict(name='net_b16_800_f16', op='net', n=16, c=3, h=800, w=800, dtype='f16', layout='nchw', call='graph'),
        # The detector on one 512 x 512 image in fp32: the protocol of the reference's published frame rate.
        dict(name='net_b1_512_f32', op='net', n=1, c=3, h=512, w=512, dtype='f32', layout='nchw', call='graph'),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A layer, block, operator or detector call: maps of 20 to 120 pixels a side (odd ones too), batches of 1 to 16,
    the channel range of each operator, every data type, both layouts."""
    op = rng.choice(['kadconv', 'kadconv', 'kadconv', 'dsc', 'dsc', 'dsc', 'dcn', 'down', 'conv1x1', 'se', 'net'])
    dtype = rng.choice(['f16', 'f16', 'bf16', 'f32'])
    if op == 'net':
        side = lambda: 32 * rng.randint(8, 25)  # noqa: E731
        n = rng.choice([1, 2, 4, 8])
        return dict(op=op, n=n, c=3, h=side(), w=side(), dtype=dtype, layout='nchw', call='graph')
    h = rng.randint(20, 120)
    w = h if rng.random() < 0.5 else rng.randint(20, 120)
    n = _log_int(rng, 1, 16)
    c = {'kadconv': lambda: _log_int(rng, 32, 288), 'dsc': lambda: _log_int(rng, 10, 512),
         'dcn': lambda: 8 * _log_int(rng, 4, 48), 'down': lambda: 8 * _log_int(rng, 8, 48),
         'conv1x1': lambda: 8 * _log_int(rng, 8, 96), 'se': lambda: 16 * _log_int(rng, 4, 64)}[op]()
    while n * c * h * w > 8 * 256 * 100 * 100:  # no larger than the headline layer's map
        n, h, w = max(1, n // 2), max(20, h * 3 // 4), max(20, w * 3 // 4)
    case = dict(op=op, n=n, c=c, h=h, w=w, dtype=dtype, layout='nchw', call=rng.choice(['graph', 'graph', 'eager']))
    if op in ('kadconv', 'dsc', 'conv1x1'):
        case['layout'] = rng.choice(['nchw', 'nchw', 'nhwc'])
    if op == 'down':
        case['c2'] = 2 * c
    if op == 'conv1x1':
        case['c2'] = 8 * _log_int(rng, 8, 96)
    return case


# ------------------------------------------------------------------ weights, by parameter name
def _uni(g, *shape, fan):
    return (torch.rand(*shape, generator=g) * 2 - 1) / math.sqrt(fan)


def _near_one(g, *shape):
    return 1 + 0.2 * (torch.rand(*shape, generator=g) * 2 - 1)


def _dsc_weights(g, c, p=''):
    """kaiming-uniform weights; conv_offset ~ N(0, 2 / sqrt(9 c)), so that a unit-variance input moves the samples by about 2 px"""
    r = p + 'RCA_mask.excite.'
    return {p + 'weight': _uni(g, c, c, 3, 3, fan=9 * c), p + 'bias': _uni(g, c, fan=9 * c),
            p + 'conv_offset.weight': torch.randn(18, c, 3, 3, generator=g) * (2 / math.sqrt(9 * c)),
            p + 'conv_offset.bias': torch.zeros(18),
            r + '0.weight': _uni(g, c, 1, 1, 11, fan=11), r + '0.bias': _uni(g, c, fan=11),
            r + '1.weight': _near_one(g, c), r + '1.bias': 0.1 * torch.randn(c, generator=g),
            r + '1.running_mean': 0.1 * torch.randn(c, generator=g), r + '1.running_var': _near_one(g, c),
            r + '3.weight': _uni(g, c, 1, 11, 1, fan=11), r + '3.bias': _uni(g, c, fan=11),
            r + '4.weight': _uni(g, 9, c, 1, 1, fan=c), r + '4.bias': _uni(g, 9, fan=c)}


def _widths(c):
    return [c - 2 * (c // 3), c // 3, c // 3]


def _weights(case):
    """The layer's parameters (fp32, CPU): the same for every seed, as a program's are."""
    g = torch.Generator().manual_seed(17 * case['c'] + 1)
    c, op = case['c'], case['op']
    if op == 'dsc':
        return _dsc_weights(g, c)
    if op == 'kadconv':
        sd = {}
        for i, b in enumerate(_widths(c)):
            p, hid = f'convs.{i}.', max(32, b)
            sd.update({p + '0.weight': _uni(g, b, c, 1, 1, fan=c), p + '0.bias': _uni(g, b, fan=c)})
            sd.update(_dsc_weights(g, b, p + '1.'))
            sd.update({p + '2.weight': _near_one(g, b), p + '2.bias': 0.1 * torch.randn(b, generator=g),
                       p + '2.running_mean': 0.1 * torch.randn(b, generator=g), p + '2.running_var': _near_one(g, b),
                       f'fc.{i}.0.weight': _uni(g, hid, b, fan=b), f'fc.{i}.0.bias': _uni(g, hid, fan=b),
                       f'fc.{i}.2.weight': _uni(g, b, hid, fan=hid), f'fc.{i}.2.bias': _uni(g, b, fan=hid),
                       f'weight.{i}.0.weight': _near_one(g, 1, b, 1, 1)})
        return sd
    if op == 'dcn':
        return {'weight': _uni(g, c, c, 3, 3, fan=9 * c), 'bias': _uni(g, c, fan=9 * c)}
    if op == 'down':
        sd = {'alpha': torch.randn(3, generator=g), 'gate': torch.randn(case['c2'], generator=g)}
        for i in range(3):
            sd.update({f'proj.{i}.weight': _uni(g, case['c2'], c, 1, 1, fan=c), f'proj.{i}.bias': _uni(g, case['c2'], fan=c)})
        return sd
    if op == 'conv1x1':
        return {'conv.weight': _uni(g, case['c2'], c, 1, 1, fan=c / 3), 'conv.bias': _uni(g, case['c2'], fan=c)}
    hid = max(1, c // 16)  # se
    return {'fc.0.weight': _uni(g, hid, c, fan=c / 3), 'fc.0.bias': _uni(g, hid, fan=c),
            'fc.2.weight': _uni(g, c, hid, fan=hid / 3), 'fc.2.bias': _uni(g, c, fan=hid)}


# ------------------------------------------------------------------ inputs and layers
def _inputs(case, seed):
    """(x, offset, mask): unit-variance feature maps, or images in [0, 1); offset (about 2 px) and mask for the operator alone."""
    g = torch.Generator('cuda').manual_seed(seed)
    n, c, h, w = (case[k] for k in 'nchw')
    kw = dict(generator=g, device='cuda')
    dt = DTYPES[case['dtype']]
    if case['op'] == 'net':
        return torch.rand(n, c, h, w, **kw).to(dt), None, None
    x = torch.randn(n, c, h, w, **kw).to(dt)
    if case['layout'] == 'nhwc':
        x = x.contiguous(memory_format=torch.channels_last)
    if case['op'] != 'dcn':
        return x, None, None
    return x, (2 * torch.randn(n, 18, h, w, **kw)).to(dt), torch.rand(n, 9, h, w, **kw).to(dt)


@functools.lru_cache(maxsize=1)
def _net_model():
    import kadcnet
    return kadcnet.build_kadcnet_s(seed=0).fuse().eval()


def _layer(case):
    """The eval-mode layer of a case on the GPU, on its fast path, as a callable of the inputs."""
    import copy

    import kadconv
    dt = DTYPES[case['dtype']]
    if case['op'] == 'net':
        import kadcnet
        m = copy.deepcopy(_net_model()).to('cuda', dt).eval()
        return kadcnet.enable_fast_inference(m)
    sd = _weights(case)
    if case['op'] == 'dcn':
        weight, bias = (sd[k].to('cuda', dt) for k in ('weight', 'bias'))
        return lambda x, offset, mask: kadconv.deform_conv2d(x, offset, weight, bias, padding=1, mask=mask)
    m = {'kadconv': lambda: kadconv.KADConv(case['c']), 'dsc': lambda: kadconv.DSC(case['c'], case['c']),
         'down': lambda: kadconv.KADDown(case['c'], case['c2']), 'conv1x1': lambda: kadconv.Conv1x1SiLU(case['c'], case['c2']),
         'se': lambda: kadconv.SqueezeExcitation(case['c'])}[case['op']]()
    m.load_state_dict(sd, strict=False)  # BatchNorm's num_batches_tracked stays
    m = m.to('cuda', dt).eval()
    return kadconv.enable_fast_inference(m) if case['op'] in ('kadconv', 'dsc') else m


def prepare(case, seed):
    f = _layer(case)
    args = [t for t in _inputs(case, seed) if t is not None]
    state = {'layer': f, 'args': args}
    with torch.no_grad():
        if case['call'] == 'graph':
            side = torch.cuda.Stream()
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side):
                for _ in range(2):
                    f(*args)
            torch.cuda.current_stream().wait_stream(side)
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                out = f(*args)
            state.update(graph=graph, out=out)
    return state


def run(state):
    if 'graph' in state:
        state['graph'].replay()
        return state['out']
    with torch.no_grad():
        return state['layer'](*state['args'])


# ------------------------------------------------------------------ what a pass needs, and how exact it is
def _dsc_flops(px, c):
    """conv_offset and the deformable 3 x 3 on px pixels of c channels (bilinear blends 2 x 4 x 9 c, LCSA's strips 2 x 20 c)"""
    return px * (2 * 9 * c * (c + 18) + 72 * c + 40 * c)


def work(case):
    op, n, c, h, w = (case[k] for k in ('op', 'n', 'c', 'h', 'w'))
    e = 4 if case['dtype'] == 'f32' else 2
    px = n * h * w
    if op == 'net':
        head = n * (h * w // 64 + h * w // 256 + h * w // 1024)
        return {'bytes': e * (3 * px + head * (4 + NET_CLASSES + NET_BOX + NET_CLASSES)),
                'flops': NET_GFLOP_800 * 1e9 * px / 640000}
    if op == 'kadconv':
        fl = sum(_dsc_flops(n * (h >> i) * (w >> i), b) + 2 * c * b * n * (h >> i) * (w >> i) for i, b in enumerate(_widths(c)))
        par = sum(b * c + 9 * b * b + 162 * b + 2 * b * max(32, b) for b in _widths(c))
        return {'bytes': e * (2 * px * c + par), 'flops': fl}
    if op == 'dsc':
        return {'bytes': e * (2 * px * c + 9 * c * c + 162 * c), 'flops': _dsc_flops(px, c)}
    if op == 'dcn':
        return {'bytes': e * (px * (2 * c + 27) + 9 * c * c), 'flops': px * (18 * c * c + 72 * c)}
    if op == 'down':
        po, c2 = n * (h // 2) * (w // 2), case['c2']
        return {'bytes': e * (px * c + po * c2 + 3 * c * c2), 'flops': 2 * c * c2 * n * sum((h >> k) * (w >> k) for k in (1, 2, 3))}
    if op == 'conv1x1':
        return {'bytes': e * (px * (c + case['c2']) + c * case['c2']), 'flops': 2 * px * c * case['c2']}
    return {'bytes': e * 2 * px * c, 'flops': 2 * px * c}  # se


# (rel, max) per operator and type: about four times the distance of the kernels from exact() over some 40 cases of these
# ranges (the detector: from its own layers in 64 bits, image by image).  A KADConv's output is mostly its residual, so its
# relative error is below a DSC's; the detector's bf16 rounding travels through 22 layers.
TOLERANCES = {
    'f32': {'kadconv': (1e-6, 1e-5), 'dsc': (2e-5, 2e-4), 'dcn': (2e-5, 2e-4), 'down': (3e-6, 2e-5),
            'conv1x1': (2e-6, 1e-5), 'se': (5e-7, 2e-6), 'net': (1e-5, 1e-4)},
    'f16': {'kadconv': (7e-4, 3e-3), 'dsc': (2e-3, 1e-2), 'dcn': (2e-3, 1.2e-2), 'down': (1.5e-3, 1e-2),
            'conv1x1': (9e-4, 2e-3), 'se': (9e-4, 2e-3), 'net': (6e-3, 4e-2)},
    'bf16': {'kadconv': (5e-3, 2e-2), 'dsc': (1e-2, 5e-2), 'dcn': (1e-2, 6e-2), 'down': (1.2e-2, 8e-2),
             'conv1x1': (7e-3, 1.6e-2), 'se': (7e-3, 1.6e-2), 'net': (0.03, 0.3)},
}


def tolerance(case):
    rel, most = TOLERANCES[case['dtype']][case['op']]
    return {'rel': rel, 'max': most}


# ------------------------------------------------------------------ the same in 64 bits
def _bn(x, sd, p):
    return F.batch_norm(x, sd[p + 'running_mean'], sd[p + 'running_var'], sd[p + 'weight'], sd[p + 'bias'], False, 0.0, BN_EPS)


def _deform(x, offset, weight, bias, mask):
    """Modulated deformable 3 x 3, padding 1: bilinear samples with zeros outside (grid_sample's corners are pixel centres)."""
    n, c, h, w = x.shape
    gy, gx = torch.meshgrid(torch.arange(h, dtype=x.dtype), torch.arange(w, dtype=x.dtype), indexing='ij')
    out = bias.view(1, -1, 1, 1)
    for k in range(9):
        y, z = gy + k // 3 - 1 + offset[:, 2 * k], gx + k % 3 - 1 + offset[:, 2 * k + 1]
        grid = torch.stack((2 * z / (w - 1) - 1, 2 * y / (h - 1) - 1), dim=-1)
        v = F.grid_sample(x, grid, mode='bilinear', padding_mode='zeros', align_corners=True) * mask[:, k:k + 1]
        out = out + F.conv2d(v, weight[:, :, k // 3, k % 3, None, None])
    return out


def _dsc(x, sd, p=''):
    c, r = x.shape[1], p + 'RCA_mask.excite.'
    offset = F.conv2d(x, sd[p + 'conv_offset.weight'], sd[p + 'conv_offset.bias'], padding=1)
    t = x.mean(3, keepdim=True) + x.mean(2, keepdim=True)
    t = F.conv2d(t, sd[r + '0.weight'], sd[r + '0.bias'], padding=(0, 5), groups=c)
    t = F.conv2d(F.relu(_bn(t, sd, r + '1.')), sd[r + '3.weight'], sd[r + '3.bias'], padding=(5, 0), groups=c)
    mask = torch.sigmoid(F.conv2d(t, sd[r + '4.weight'], sd[r + '4.bias']))
    return _deform(x, offset, sd[p + 'weight'], sd[p + 'bias'], mask)


def _attention(x, w1, b1, w2, b2):
    a = torch.sigmoid(F.linear(F.relu(F.linear(x.mean((2, 3)), w1, b1)), w2, b2))
    return x * a[:, :, None, None]


def exact(case, seed):
    if case['op'] == 'net':
        return None  # 22 layers on the CPU in 64 bits take longer than a check should
    dt = DTYPES[case['dtype']]
    sd = {k: v.to(dt).double() for k, v in _weights(case).items()}  # the values that the layer holds
    x, offset, mask = (None if t is None else t.double().cpu().contiguous() for t in _inputs(case, seed))
    op = case['op']
    if op == 'dsc':
        return _dsc(x, sd)
    if op == 'dcn':
        return _deform(x, offset, sd['weight'], sd['bias'], mask)
    if op == 'conv1x1':
        return F.silu(F.conv2d(x, sd['conv.weight'], sd['conv.bias']))
    if op == 'se':
        return _attention(x, *(sd[k] for k in ('fc.0.weight', 'fc.0.bias', 'fc.2.weight', 'fc.2.bias')))
    outs = []
    if op == 'down':
        a = torch.softmax(sd['alpha'], 0)
        size = (case['h'] // 2, case['w'] // 2)
        for i in range(3):
            z = F.conv2d(F.avg_pool2d(x, 2 << i), sd[f'proj.{i}.weight'], sd[f'proj.{i}.bias'])
            outs.append(a[i] * (z if i == 0 else F.interpolate(z, size=size, mode='bilinear', align_corners=False)))
        return sum(outs) * torch.sigmoid(sd['gate']).view(1, -1, 1, 1)
    for i in range(3):
        p = f'convs.{i}.'
        z = F.conv2d(F.avg_pool2d(x, 1 << i) if i else x, sd[p + '0.weight'], sd[p + '0.bias'])
        z = F.relu(_bn(_dsc(z, sd, p + '1.'), sd, p + '2.')) * sd[f'weight.{i}.0.weight']
        z = _attention(z, *(sd[f'fc.{i}.{k}'] for k in ('0.weight', '0.bias', '2.weight', '2.bias')))
        outs.append(z if i == 0 else F.interpolate(z, size=x.shape[2:], mode='bilinear', align_corners=False))
    return torch.cat(outs, 1) + x
