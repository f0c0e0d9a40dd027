"""The fold of the striped tallies (k_fold). A solve folds every tally's
stripes into one buffer; ssolh_solve_noalloc folds them in place and, in its
64 MiB, with fewer stripes where the tallies are large. Both run the same
realisations, so the folded tallies agree up to the order of the FP64
additions, at sizes on both sides of the kernel's tiles (1024 / min(16,
stripes) elements): receivers of 2 to 2,178 triangles, 1 to 130 sampled
instances (300: several shares of the instances in k_fold_rcv, which sums the
receiver tally from the sampled x receiver one). Order of additions: sums of at most n = 60,000 terms of one sign
in two orders differ by at most 2 n 2^-53 = 1.3e-11 relative; counts are
equal."""
import ctypes as C

import numpy as np
import pytest

import ssol_ctypes as L
import ssol_scene as S
import test_zz_no_alloc as N

pytestmark = pytest.mark.gpu

REALISATIONS = 60_000


@pytest.mark.parametrize("heliostats,cells", [(1, 1), (2, 7), (25, 8), (63, 33), (130, 9),
                                              (300, 4)])
def test_fold_into_buffer_matches_fold_in_place(gpu, heliostats, cells):
    spec = S.config2(0, n_helio=heliostats, radius=40.0 + 20.0 * heliostats ** 0.5, rcv_size=8.0,
                     rcv_cells=cells)
    lib = L.Scene(spec)
    lib.solve(1000, seed=1)
    hip, ctx = N._hip(), N._ctx(lib)
    a = N.SolveArgs(REALISATIONS, 2**62, 3, 0, 0, 0, 0, 0)
    ref, got = N.Out(spec, lib), N.Out(spec, lib)
    assert hip.ssolh_solve(ctx, C.byref(a)) == 0, hip.ssolh_last_error()
    assert hip.ssolh_tallies_download(ctx, C.byref(ref.t)) == 0
    assert hip.ssolh_solve_noalloc(ctx, C.byref(a), C.byref(got.t)) == 0, hip.ssolh_last_error()
    assert ref.t.realisation_count == REALISATIONS and int(ref.cnt.sum()) == REALISATIONS
    assert ref.t.segments > REALISATIONS
    assert ref.rcv.any() and ref.samp.any() and ref.prim.any()
    N._same(got, ref, 1.3e-11)
    for o in (ref, got):
        per_instance = o.sxr[:heliostats * 40].reshape(heliostats, 40)
        assert np.count_nonzero(per_instance[:, 0]) == heliostats
        assert np.allclose(o.rcv[:40], per_instance.sum(axis=0), rtol=1e-13, atol=0)
    lib.close()


@pytest.mark.parametrize("suns", [1, 3, 65])
def test_fold_keeps_the_suns_apart(gpu, suns):
    """The global tally of a batch has a row of 16 doubles per sun."""
    spec = S.config2(0, n_helio=10, radius=120.0)
    lib = L.Scene(spec)
    dirs = [S.sun_dir_from(170.0 + 0.3 * j, 50.0 + 0.1 * j) for j in range(suns)]
    counts = [300 + 7 * j for j in range(suns)]
    res, got = lib.solve_sun_batch(dirs, counts, seed=2)
    assert got == counts
    area = lib.solve(1000, seed=1).sampled_area
    for g in res:
        sinks = sum(g[f][0] for f in ("absorbed_by_receivers", "missing", "shadowed",
                                      "extinguished_by_atmosphere", "other_absorbed"))
        # the sun's angular blur: sinks against the main direction's flux
        assert np.isclose(sinks, spec.sun.dni * area * g["cos_factor"][0], rtol=1e-2)
    lib.close()
