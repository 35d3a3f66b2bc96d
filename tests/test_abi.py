"""CPU checks of the C-ABI library: it loads, exports every symbol declared in
include/dqh.h, and its descriptor layout matches the Python mirror. No compute."""

import ctypes
import os
import re

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared_symbols():
    src = open(os.path.join(ROOT, 'include', 'dqh.h')).read()
    return sorted(set(re.findall(r'\b(dqh_[a-z0-9_]+)\s*\(', src)))


def test_library_exports_every_declared_symbol():
    from dynamiqs_amd import _native

    lib = ctypes.CDLL(_native.LIB_PATH)
    names = _declared_symbols()
    assert len(names) >= 7
    for name in names:
        assert hasattr(lib, name), name
    assert set(names) <= set(_native.SYMBOLS), set(names) - set(_native.SYMBOLS)


def test_descriptor_layout_matches_mirror():
    from dynamiqs_amd import _native

    lib = _native.lib()
    assert lib.dqh_sizeof_me_inst() == _native.ME_INST_DTYPE.itemsize
    assert lib.dqh_me_work_elems(64, 2, 0) == 11 * 64 * 64
    src = open(os.path.join(ROOT, 'include', 'dqh.h')).read()
    body = src[src.index('typedef struct dqh_me_inst') : src.index('} dqh_me_inst;')]
    fields = re.findall(r'\b(?:int64_t|double|uint64_t)\s+([a-zA-Z0-9_, ]+);', body)
    names = [f.strip() for group in fields for f in group.split(',')]
    assert names == list(_native.ME_INST_DTYPE.names)


def test_rouchon1_expectations_without_saves_are_refused():
    """Before any work, and without a division by the number of saves."""
    from dynamiqs_amd import _native
    from dynamiqs_amd.integrators.dia import DiaRouchon1

    p = DiaRouchon1()
    p.nb = p.n = p.n_true = 64
    p.ninst = p.nsets = p.nE = 1
    p.EopsT = p.expects = 16
    p.ops[0].nops = p.ops[0].noff[0] = 1
    for nsave in (0, -1):
        p.nsave = nsave
        assert _native.lib().dqh_mesolve_rouchon1_dia(ctypes.byref(p), None) == -1
        assert b'nsave >= 1' in _native.lib().dqh_last_error()


def test_no_fallback_when_library_missing(monkeypatch, tmp_path):
    import pytest

    from dynamiqs_amd import _native

    monkeypatch.setattr(_native, '_lib', None)
    monkeypatch.setattr(_native, 'LIB_PATH', str(tmp_path / 'missing.so'))
    with pytest.raises(RuntimeError, match='missing'):
        _native.lib()
