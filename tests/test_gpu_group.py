"""Grouping by key (k_group_rank, k_group_scan, k_group_place), which orders
the realisations of a wavefront by start key and the per-primitive log by
primitive, and the log's two routes: up to 16,384 keys grouped, beyond by a
radix sort."""
import ctypes as C

import numpy as np
import pytest

import ssol_ctypes as L
import ssol_scene as S
import test_zz_no_alloc as N

pytestmark = pytest.mark.gpu

U32P = C.POINTER(C.c_uint32)


# blocks of 4096 items; 16 keys per thread of the scan
@pytest.mark.parametrize("n,nkeys", [(1, 1), (63, 1), (4095, 15), (4096, 16384), (4097, 16383),
                                     (100_003, 17), (300_000, 10_003)])
def test_groups_are_whole_and_in_key_order(gpu, n, nkeys):
    lib = L.Scene(S.config2(0, n_helio=1, radius=60.0, rcv_size=8.0, rcv_cells=1))
    lib.solve(1000, seed=1)
    hip, ctx = N._hip(), N._ctx(lib)
    hip.ssolh_test_group.argtypes = [C.c_void_p, C.c_uint32, C.c_uint32, U32P, U32P, U32P]
    key = np.random.default_rng(n).integers(0, nkeys, n, dtype=np.uint32)
    key[-1] = nkeys - 1
    order, off = np.zeros(n, np.uint32), np.zeros(nkeys + 1, np.uint32)
    p = lambda a: a.ctypes.data_as(U32P)
    assert hip.ssolh_test_group(ctx, n, nkeys, p(key), p(order), p(off)) == 0
    assert np.array_equal(off, np.concatenate([[0], np.cumsum(np.bincount(key, minlength=nkeys))]))
    assert np.array_equal(np.sort(order), np.arange(n))
    assert np.array_equal(key[order], np.sort(key))
    key[0] = nkeys
    assert hip.ssolh_test_group(ctx, n, nkeys, p(key), p(order), p(off)) != 0
    lib.close()


# ssolh_solve_noalloc keeps no log: its entries are added one by one. Sums of
# n terms of one sign in two orders differ by at most 2 n 2^-53 relative. Logs
# of 2^18 records on are in 16 segments.
@pytest.mark.parametrize("n", [60_000, 262_144])
@pytest.mark.parametrize("cells,keys", [(64, 16384), (65, 16900)])
def test_log_routes_match_atomics(gpu, cells, keys, n):
    spec = S.config2(0, n_helio=40, radius=150.0, rcv_size=8.0, rcv_cells=cells)
    lib = L.Scene(spec)
    lib.solve(1000, seed=1)
    hip, ctx = N._hip(), N._ctx(lib)
    a = N.SolveArgs(n, 2**62, 3, 0, 0, 0, 0, 0)
    ref, got = N.Out(spec, lib), N.Out(spec, lib)
    assert hip.ssolh_solve(ctx, C.byref(a)) == 0, hip.ssolh_last_error()
    assert hip.ssolh_tallies_download(ctx, C.byref(ref.t)) == 0
    assert hip.ssolh_solve_noalloc(ctx, C.byref(a), C.byref(got.t)) == 0, hip.ssolh_last_error()
    assert len(ref.prim) == keys * 20 and np.count_nonzero(ref.prim) > 1000
    N._same(got, ref, 2 * n * 2.0 ** -53)
    lib.close()


# Paths between two diffuse walls meet more primitives than they hold pending
# entries for: the rest, logged one by one, against atomics (sums of at most
# n = 400,000 terms of one sign in two orders: 2 n 2^-53 = 8.9e-11 relative)
@pytest.mark.parametrize("precision", [0, 1])
def test_spilled_entries_match_atomics(gpu, precision):
    wall = S.matte(0.7)
    obj = S.Object([(S.grid_mesh(4.0, 4.0, 9, 9), wall, wall)])
    floor = S.Instance(obj, S.IDENTITY, receiver_mask=S.FRONT | S.BACK, per_primitive=1)
    roof = S.Instance(obj, S.transform(None, (3.0, 0.0, 1.5)), receiver_mask=S.FRONT | S.BACK,
                      per_primitive=1, sample=0)
    spec = S.Scene([floor, roof], S.Sun("directional", (0, 0, -1), 1000.0,
                                        S.Spectrum([1.0], [1.0])), None, name="walls")
    lib = L.Scene(spec)
    lib.solve(1000, seed=1)
    hip, ctx = N._hip(), N._ctx(lib)
    a = N.SolveArgs(100_000, 2**62, 3, 0, precision, 0, 1, 0)
    ref, got = N.Out(spec, lib), N.Out(spec, lib)
    assert hip.ssolh_solve(ctx, C.byref(a)) == 0, hip.ssolh_last_error()
    assert hip.ssolh_tallies_download(ctx, C.byref(ref.t)) == 0
    assert hip.ssolh_solve_noalloc(ctx, C.byref(a), C.byref(got.t)) == 0, hip.ssolh_last_error()
    assert ref.t.pending_spills == got.t.pending_spills > 1000
    N._same(got, ref, 8.9e-11)
    lib.close()
