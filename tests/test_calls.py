"""kad_run_calls' own checks (no GPU: nothing is launched before they fail)."""
import ctypes

import pytest

from kadconv import _ext


def _run(blob, calls, relocs, bases):
    b = ctypes.create_string_buffer(blob, max(len(blob), 1))
    c, r = (_ext.Call * max(len(calls), 1))(*calls), (_ext.Reloc * max(len(relocs), 1))(*relocs)
    p = (ctypes.c_void_p * max(len(bases), 1))(*bases)
    return _ext.load().kad_run_calls(ctypes.addressof(b), len(blob), ctypes.addressof(c), len(calls),
                                     ctypes.addressof(r), len(relocs), p, len(bases), None)


def test_empty_list():
    assert _run(b'\0' * 16, [], [_ext.Reloc(8, 4, 0)], [64]) == 0


@pytest.mark.parametrize('call', [_ext.Call(9, 1, 0, 0), _ext.Call(-1, 1, 0, 0), _ext.Call(_ext.CALL_DSC, 0, 0, 0),
                                  _ext.Call(_ext.CALL_DSC, 3, 0, 0), _ext.Call(_ext.CALL_DSC, 1 << 30, 0, 0),
                                  _ext.Call(_ext.CALL_MERGE, 1, 8, 0), _ext.Call(_ext.CALL_PYRAMID, 1, -8, 0),
                                  _ext.Call(_ext.CALL_LCSA_PREP, 1, 4, 0)])
def test_calls_out_of_range(call):
    assert _run(b'\0' * ctypes.sizeof(_ext.MergeArgs), [call], [], []) < 0


@pytest.mark.parametrize('reloc', [_ext.Reloc(16, 0, 0), _ext.Reloc(-8, 0, 0), _ext.Reloc(4, 0, 0),
                                   _ext.Reloc(0, 0, 1), _ext.Reloc(0, 0, -1)])
def test_relocations_out_of_range(reloc):
    assert _run(b'\0' * 16, [], [reloc], [64]) < 0


def test_blob_too_large():
    assert _run(b'\0' * 16392, [], [], []) < 0


def test_struct_layouts():
    """The ctypes mirrors of kad_call, kad_reloc and kad_scale_args have C's layout (8-byte pointers)."""
    assert (_ext.Call.args.offset, ctypes.sizeof(_ext.Call)) == (8, 24)
    assert (_ext.Reloc.add.offset, _ext.Reloc.base.offset, ctypes.sizeof(_ext.Reloc)) == (8, 16, 24)
    assert (_ext.ScaleArgs.n.offset, ctypes.sizeof(_ext.ScaleArgs)) == (24, 56)


def _find(pointers, spans):
    """[(offset in the blob, base, offset from it)] of kad_find_relocs for a blob of these pointers."""
    import array
    blob = array.array('q', pointers).tobytes()
    at, sp = array.array('q', range(0, len(blob), 8)), array.array('q', [v for s in spans for v in s])
    out = (_ext.Reloc * len(pointers))()
    n = _ext.load().kad_find_relocs(blob, len(blob), at.buffer_info()[0], len(at), sp.buffer_info()[0], len(spans), out)
    return n if n < 0 else [(r.at, r.base, r.add) for r in out[:n]]


def test_find_relocs():
    spans = [(4096, 100, 0, 0), (8192, 64, 0, 1), (9000, 16, 256, 1)]
    assert _find([0, 4096, 4100, 4195, 4196, 8200, 9015, 9016, 5], spans) == [
        (8, 0, 0), (16, 0, 4), (24, 0, 99), (40, 1, 8), (48, 1, 271)]
    assert _find([0, 7], spans) == []


@pytest.mark.parametrize('x,out', [(4096, 4128), (4128, 4096)])
def test_find_relocs_of_interleaved_slices(x, out):
    """Input and output are channel slices of one buffer: each span holds the other's start."""
    spans = [(x, 4000, 0, 0), (out, 4000, 0, 1)]
    assert _find([x, out, x], spans) == [(0, 0, 0), (8, 1, 0), (16, 0, 0)]
    assert _find([max(x, out) + 16], spans) < 0       # could be either's: refused
    assert _find([x], [(x, 4000, 0, 0), (x, 4000, 0, 1)]) < 0


@pytest.mark.parametrize('at', [-8, 9, 16])
def test_find_relocs_outside_the_blob(at):
    import array
    a, sp, out = array.array('q', [at]), array.array('q', [0, 1, 0, 0]), (_ext.Reloc * 1)()
    assert _ext.load().kad_find_relocs(b'\1' * 16, 16, a.buffer_info()[0], 1, sp.buffer_info()[0], 1, out) < 0


def test_call_layout():
    """One kad_call per call at its structs' place, and the places of all their pointers."""
    calls, at = _ext._call_layout(((_ext.CALL_DSC, _ext.DcnArgs * 2, 0), (_ext.CALL_LCSA_MASK, _ext.LcsaArgs * 1, 5),
                                   (_ext.CALL_MERGE, _ext.MergeArgs, 0)))
    dcn, lcsa = ctypes.sizeof(_ext.DcnArgs), ctypes.sizeof(_ext.LcsaArgs)
    assert [(c.fn, c.count, c.args, c.arg) for c in calls] == [
        (_ext.CALL_DSC, 2, 0, 0), (_ext.CALL_LCSA_MASK, 1, 2 * dcn, 5), (_ext.CALL_MERGE, 1, 2 * dcn + lcsa, 0)]
    assert _ext.DcnArgs.se_att.offset in at and dcn + _ext.DcnArgs.x.offset in at
    assert 2 * dcn + _ext.LcsaArgs.mask.offset in at
    merge = 2 * dcn + lcsa + _ext.MergeArgs.br_z.offset
    assert merge in at and merge + 8 in at
    words = sum(1 for st, k in ((_ext.DcnArgs, 2), (_ext.LcsaArgs, 1), (_ext.MergeArgs, 1)) for _ in range(k)
                for n, t in st._fields_ for _ in range(1 if t is ctypes.c_void_p else
                                                       t._length_ if isinstance(t, type) and issubclass(t, ctypes.Array)
                                                       and t._type_ is ctypes.c_void_p else 0))
    assert len(at) == len(set(at)) == words
