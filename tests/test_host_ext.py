"""CPU checks of the entry points of include/leniax_amd_ext.h: exported, bound, and with the conventions for
empty and negative batches of the others (no device call on these paths)."""
import ctypes
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_entry_points_take_empty_batches_and_refuse_negative_ones():
    from leniax_amd import _lib
    if not _lib.available():
        pytest.skip('libleniax_amd.so not built')
    L_ = _lib.lib()
    rule = _lib.lx_rule()
    rule.ndim, rule.C, rule.K, rule.average = 2, 1, 1, 1
    rule.dims[0], rule.dims[1] = 64, 64
    r, N, size = ctypes.byref(rule), None, ctypes.c_size_t(0)
    calls = {
        'lx_update_dt': lambda B: L_.lx_update_dt(r, N, B, N, 0, N, 0, N, 0, 0.1, N, N, N, N, N),
        'lx_potential_direct_adjoint_size':
            lambda B: L_.lx_potential_direct_adjoint_size(r, B, 27, 27, ctypes.byref(size)),
        'lx_potential_direct_adjoint_work':
            lambda B: L_.lx_potential_direct_adjoint_work(r, N, B, N, 27, 27, N, N, N, N, N),
    }
    text = re.sub(r'/\*.*?\*/', '', open(os.path.join(ROOT, 'include', 'leniax_amd_ext.h')).read(), flags=re.S)
    assert set(re.findall(r'\b(lx_[a-z0-9_]+)\s*\(', text)) == set(calls)
    for name, fn in calls.items():
        assert fn(0) == _lib.LX_OK, name
        assert fn(-1) != _lib.LX_OK, name
