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
