"""libspk.so loads and exports every symbol include/spk.h declares; its
host-only parts (variogram parsing, nugget check) work without a GPU."""
import ctypes
import re
import subprocess
import sys
from pathlib import Path

import numpy as np
import pytest

from spinterps_amd import _lib

HEADER = Path(__file__).resolve().parents[1] / 'include' / 'spk.h'


def declared_symbols():
    txt = HEADER.read_text()
    txt = re.sub(r'/\*.*?\*/', '', txt, flags=re.S)
    return sorted(set(re.findall(r'\b(spk_[a-z0-9_]+)\s*\(', txt)))


def test_library_exports_every_declared_symbol():
    h = ctypes.CDLL(str(_lib.LIB_PATH))
    syms = declared_symbols()
    assert len(syms) >= 20
    missing = [s for s in syms if not hasattr(h, s)]
    assert not missing, missing
    # and the binding declares a signature for each of them
    assert not [s for s in syms if s not in _lib.SIGNATURES]


def test_vg_parse_matches_reference_grammar():
    v = _lib.parse_vg('0.1 Nug(0.0) + 0.9 Sph(25000.0)')
    assert v.n == 2
    assert list(v.type)[:2] == [1, 2]
    assert list(v.sill)[:2] == [0.1, 0.9]
    assert list(v.range)[:2] == [1e-5, 25000.0]   # pyx:183 clamp
    assert v.sill_sum == 0.1 + 0.9
    assert v.range_max_raw == 25000.0
    v = _lib.parse_vg(' 2.5 Gau(1e4)+3 Exp(7) ')
    assert v.n == 2 and v.range[0] == 1e4 and v.sill[1] == 3.0
    for bad in ['1 Foo(2)', '1  Sph(2)', 'Sph(2)', 'nan', '1 Sph 2', 'x Sph(2)']:
        with pytest.raises(ValueError):
            _lib.parse_vg(bad)


def test_nuggetness_host():
    out = ctypes.c_int()
    f = _lib.lib().spk_vg_full_nuggetness
    for s, mvv, exp in [('1.0 Nug(0.0)', 0.0, 1),
                        ('0.1 Nug(0.0) + 0.9 Sph(25.0)', 0.0, 0),
                        ('0.0 Sph(25.0)', 0.0, 1),
                        ('2.0 Sph(25.0)', 30.0, 1),
                        ('nan', 0.0, 0)]:
        assert f(s.encode(), mvv, ctypes.byref(out)) == 0
        assert out.value == exp, s


def test_vg_array_layout():
    arr = _lib.vg_array(['1 Sph(2)', '3 Exp(4) + 1 Nug(0)', '1 Sph(2)'])
    assert arr.dtype.itemsize == ctypes.sizeof(_lib.SpkVg)
    assert arr['n'].tolist() == [1, 2, 1]
    assert arr['sill'][1, :2].tolist() == [3.0, 1.0]
    assert arr['type'][1, :2].tolist() == [3, 1]


def test_f32_out_struct_layout():
    """SpkF32Out mirrors include/spk.h's spk_f32_out: two host pointers,
    two int32 flags, two doubles (40 bytes, the doubles 8-aligned)."""
    S = _lib.SpkF32Out
    assert ctypes.sizeof(S) == 40
    assert S.est32.offset == 0 and S.var32.offset == 8
    assert S.has_min.offset == 16 and S.has_max.offset == 20
    assert S.min_cut.offset == 24 and S.max_cut.offset == 32


def test_first_context_loads_the_library():
    """A process whose first library call makes a context (as an IDW call
    or a variogram fit does) does not wait on its own lock: context() holds
    it while the library is loaded under it.  Without a GPU the context
    itself is refused."""
    code = ('from spinterps_amd import _lib\n'
            'try:\n    _lib.context(0)\nexcept Exception:\n    pass\n'
            'assert _lib._lib is not None\n')
    subprocess.run([sys.executable, '-c', code], check=True, timeout=60,
                   cwd=Path(__file__).resolve().parents[1])
