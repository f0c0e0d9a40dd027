"""Estimators take their memory from those released before: each keeps its
own values whatever the order of solves and releases, also where the next
solve's tallies need more or fewer words than a spare block holds."""
import gc

import numpy as np
import pytest

import ssol_ctypes as L
import ssol_scene as S

pytestmark = pytest.mark.gpu


def _values(spec, est):
    rcv = spec.instances[-1]
    prims = est.primitives(rcv, rcv.object.sshapes[0][0], S.FRONT, "incoming_flux")
    return np.concatenate([[v for f in sorted(g) for v in g[f]] for g in
                           [est.global_(), est.receiver(rcv, S.FRONT)]] + [np.ravel(prims)])


@pytest.mark.parametrize("released", [(), (0,), (2, 0, 1), (0, 1, 2, 3)])
def test_estimators_keep_their_values(gpu, released):
    spec = S.config2(0, n_helio=5, radius=80.0, rcv_size=8.0, rcv_cells=6)
    lib = L.Scene(spec)
    ests = {k: lib.solve(3000 + k, seed=k) for k in range(4)}
    want = {k: _values(spec, e) for k, e in ests.items()}
    for k in released:
        del ests[k]
        gc.collect()
    more = [lib.solve(2000 + k, seed=9 + k) for k in range(3)]
    for k, e in ests.items():
        assert np.array_equal(_values(spec, e), want[k])
    again = [_values(spec, lib.solve(2000 + k, seed=9 + k)) for k in range(3)]
    for e, a in zip(more, again):  # the same paths, added in another order
        assert np.allclose(_values(spec, e), a, rtol=1e-9, atol=1e-12)
    assert all(not np.array_equal(again[0], a) for a in again[1:])
    lib.close()
