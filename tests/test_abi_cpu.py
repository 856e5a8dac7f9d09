"""The C ABI library loads without a GPU and exports every entry point that
include/percolate_hip.h declares; host-only entry points and argument
checks work without a device."""
import ctypes
import os
import re

import pytest

from pypercolate_amd import _native as nat

HEADER = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                      'include', 'percolate_hip.h')


def declared_functions():
    text = open(HEADER).read()
    text = re.sub(r'/\*.*?\*/', '', text, flags=re.S)
    return sorted(set(re.findall(r'\b(pc_[a-z0-9_]+)\s*\(', text)))


def test_header_declares_functions():
    names = declared_functions()
    assert 'pc_sweep' in names and 'pc_microcanonical_sums' in names
    assert len(names) >= 10


def test_library_exports_every_declared_symbol():
    lib = nat.load_library()
    for name in declared_functions():
        assert hasattr(lib, name), name


def test_binding_table_matches_header():
    assert sorted(nat.SIGNATURES) == declared_functions()


def test_host_only_entry_points():
    lib = nat.load_library()
    assert lib.pc_abi_version() >= 1
    assert lib.pc_record_bytes(65536) == 4
    assert lib.pc_record_bytes(65537) == 8
    a, b = ctypes.c_int64(), ctypes.c_int64()
    assert lib.pc_binomial_window(32512, 0.5, ctypes.byref(a), ctypes.byref(b)) == 0
    sigma = (32512 * 0.25) ** 0.5
    assert a.value <= 16256 - 12 * sigma and a.value + b.value - 1 >= 16256 + 12 * sigma
    assert lib.pc_binomial_window(10, 0.0, ctypes.byref(a), ctypes.byref(b)) == 0
    assert a.value == 0 and b.value == 11


def test_argument_errors_without_gpu():
    lib = nat.load_library()
    rc = lib.pc_sweep(0, 1, None, None, 0, None, 1, 1, None, 1, None, None, 0, 0, 0,
                      None, None)
    assert rc == nat.PC_EINVAL
    assert b'num_nodes' in lib.pc_last_error()
    rc = lib.pc_sweep(16, 1, None, None, 0, None, 1, 1, None, 1, None, None, 0, 99,
                      0, None, None)
    assert rc == nat.PC_EINVAL and b'merge_rounds' in lib.pc_last_error()
    rc = lib.pc_sweep(20000, 1, None, None, 0, None, 1, 1, None, 1, None, None, 0,
                      0, nat.PC_STATE_LDS, None, None)
    assert rc == nat.PC_EINVAL
    with pytest.raises(ValueError):
        nat.check(rc, 'pc_sweep')
    # both wave flags at once is not a mode
    rc = lib.pc_sweep(16, 1, None, None, 0, None, 1, 1, None, 1, None, None, 0,
                      0, nat.PC_SWEEP_WAVES_MASK, None, None)
    assert rc == nat.PC_EINVAL and b'state_mode' in lib.pc_last_error()
    rc = lib.pc_binomial_window(10, 1.5, ctypes.byref(ctypes.c_int64()),
                                ctypes.byref(ctypes.c_int64()))
    assert rc == nat.PC_EINVAL
    rc = lib.pc_microcanonical_sums(1 << 22, 10, 1, None, 1, None, None, None,
                                    None, 0, None)
    assert rc == nat.PC_EOVERFLOW


def _tiled(length, runs, nbytes, mode=nat.PC_STATE_AUTO, span_first=0):
    lib = nat.load_library()
    at_once = ctypes.c_uint32(99)
    assert lib.pc_sweep_lattice_tiled_runs(length, span_first, runs, nbytes, mode,
                                           ctypes.byref(at_once)) == 0
    return at_once.value


def _lattice_bytes(length, runs):
    b = ctypes.c_uint64()
    assert nat.load_library().pc_sweep_lattice_workspace_size(
        length, runs, nat.PC_STATE_AUTO, ctypes.byref(b)) == 0
    return b.value


@pytest.mark.parametrize('length,runs', [
    (65, 1), (65, 600), (80, 40), (95, 1024), (96, 1500), (100, 3), (127, 700), (128, 200),
    (128, 1025), (128, 10000), (129, 5), (129, 300), (130, 7), (136, 9), (181, 40), (192, 3),
    (200, 12), (255, 2), (256, 200), (257, 8), (264, 30), (300, 2), (400, 300), (512, 2),
    (513, 2), (700, 80), (725, 2), (1000, 1), (1024, 1000), (1100, 1), (2048, 1)])
def test_lattice_sweep_in_tiles(length, runs):
    """With the workspace it asks for, the lattice sweep goes in tiles at
    every size of its range; in slabs of four runs on with less, and not at
    all below that, in other modes or with sides joined from the first
    merge on."""
    full = _lattice_bytes(length, runs)
    assert 0 < _tiled(length, runs, full) <= runs + 7
    assert _tiled(length, runs, full, nat.PC_STATE_HBM) == 0
    assert _tiled(length, runs, full, nat.PC_STATE_AUTO | nat.PC_SWEEP_TWO_WAVES) == 0
    assert _tiled(length, runs, full, span_first=1) == 0
    assert _tiled(length, runs, 0) == 0
    bonds = 8 * length * (length - 1)        # a run's list, in bytes
    assert _tiled(length, runs, min(runs, 3) * bonds) == 0
    if runs >= 30:
        assert 4 <= _tiled(length, runs, full // 2) < runs


@pytest.mark.parametrize('length,runs', [(1, 1), (16, 40), (64, 1), (64, 10000), (65, 1025),
                                         (95, 4000), (2049, 1), (2052, 3), (16384, 1)])
def test_lattice_sweep_not_in_tiles(length, runs):
    assert _tiled(length, runs, 1 << 40) == 0
