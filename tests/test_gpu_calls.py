"""A small KAD-Conv layer's recorded launches (kad_run_calls) against the same stages launched one by
one: bit for bit, over layouts, channel slices, types and odd sizes, with another input and other
buffers than those recorded, under graph replay, and with more geometries than a plan keeps."""
import copy

import pytest
import torch

pytestmark = pytest.mark.gpu
DT = {'f32': torch.float32, 'f16': torch.float16, 'bf16': torch.bfloat16}


def _layer(dim, dtype):
    import kadconv
    from kadconv import synthetic as S
    m = kadconv.KADConv(dim)
    m.load_state_dict(S.make_kadconv_state(dim, seed=dim), strict=False)
    return kadconv.enable_fast_inference(m.to('cuda', dtype).eval())


def _input(n, c, h, w, dtype, layout, seed):
    x = torch.randn(n, c, h, w, generator=torch.Generator().manual_seed(seed)).to('cuda', dtype)
    if layout == 'nhwc':
        x = x.contiguous(memory_format=torch.channels_last)
    if layout == 'slice':  # a channel slice of a wider channels-last buffer
        wide = torch.randn(n, h, w, c + 16, device='cuda').to(dtype)
        wide[..., 8:8 + c] = x.permute(0, 2, 3, 1)
        x = wide[..., 8:8 + c].permute(0, 3, 1, 2)
    if layout == 'strided':  # neither: made contiguous on entry
        x = torch.cat((x, x), 3)[..., :w]
    return x


@pytest.mark.parametrize('dt', ['f32', 'f16', 'bf16'])
@pytest.mark.parametrize('layout', ['nchw', 'nhwc', 'slice', 'strided'])
@pytest.mark.parametrize('dim,n,h,w', [(32, 1, 16, 16), (48, 2, 21, 37), (96, 1, 5, 7), (130, 2, 20, 12)])
def test_recorded_calls_match_stages(dt, layout, dim, n, h, w):
    m = _layer(dim, DT[dt])
    plan = m._kad_plan
    print(f'calls {dt} {layout} {dim, n, h, w}', flush=True)
    with torch.no_grad():
        keep = [m(_input(n, dim, h, w, DT[dt], layout, 0)) for _ in range(2)]  # records, then replays
        assert [v is not None for v in plan._lists.values()] == [True]
        for seed in (1, 2):
            x = _input(n, dim, h, w, DT[dt], layout, seed)
            st, ref = plan.schedule_grouped(x)
            for _, fn in st:
                fn()
            got = m(x)
            keep.append(got)
            assert got.stride() == ref.stride() and torch.equal(got, ref)


def test_recorded_calls_graph_and_bound():
    from kadconv import fused
    m = _layer(48, torch.float16)
    plan = m._kad_plan
    with torch.no_grad():
        for k in range(fused.MAX_LISTS + 3):
            for _ in range(2):
                m(_input(1, 48, 8 + k, 9, torch.float16, 'nchw', k))
        assert len(plan._lists) == fused.MAX_LISTS
        x = _input(1, 48, 30, 31, torch.float16, 'nchw', 0)
        for _ in range(2):
            m(x)
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            y = m(x)
        for seed in (3, 4, 5):
            x.copy_(_input(1, 48, 30, 31, torch.float16, 'nchw', seed))
            g.replay()
            ref = m(x.clone())
            torch.cuda.synchronize()
            assert torch.equal(y, ref)


def test_copied_plan_records_its_own_calls():
    m = _layer(48, torch.float32)
    x = _input(1, 48, 9, 12, torch.float32, 'nchw', 0)
    with torch.no_grad():
        ref = [m(x) for _ in range(3)][-1]
        plan = copy.deepcopy(m._kad_plan)
        assert len(m._kad_plan._lists) == 1 and not plan._lists
        del m
        for _ in range(3):
            assert torch.equal(plan.forward(x), ref)


@pytest.mark.parametrize('dt', ['f32', 'f16', 'bf16'])
@pytest.mark.parametrize('dim,n,h,w', [(48, 2, 21, 37), (130, 1, 20, 12)])
@pytest.mark.parametrize('place', ['x first', 'out first', 'two buffers'])
def test_recorded_calls_with_out(dt, dim, n, h, w, place):
    """forward(x, out=) on channel slices, x and out of one wide buffer (the detector's concats) or of two:
    every call on buffers of its own, bit for bit as the stages one by one; nothing else is written."""
    dtype, cs = DT[dt], (dim + 7) // 8 * 8
    plan = _layer(dim, dtype)._kad_plan
    wide = 2 * cs + 24
    ax, ao = {'x first': (8, cs + 16), 'out first': (cs + 16, 8), 'two buffers': (8, 16)}[place]
    print(f'calls out {dt} {dim, n, h, w} {place}', flush=True)

    def buffers(seed):
        g = torch.Generator().manual_seed(seed)
        bx = torch.randn(n, h, w, wide, generator=g).to('cuda', dtype)
        bo = bx if place != 'two buffers' else torch.randn(n, h, w, wide, generator=g).to('cuda', dtype)
        return bx, bo, bx[..., ax:ax + dim].permute(0, 3, 1, 2), bo[..., ao:ao + dim].permute(0, 3, 1, 2)

    past = []
    with torch.no_grad():
        for seed in range(4):
            bx, bo, x, out = buffers(seed)
            rx, ro, x2, out2 = buffers(seed)
            st, _ = plan.schedule_grouped(x2, out2)
            for _, fn in st:
                fn()
            assert plan.forward(x, out=out) is out
            assert torch.equal(bx, rx) and torch.equal(bo, ro)   # the slices and all around them
            past.append((bx, bo, bx.clone(), bo.clone()))
        assert len(plan._lists) == 1
        for bx, bo, cx, co in past:
            assert torch.equal(bx, cx) and torch.equal(bo, co)
