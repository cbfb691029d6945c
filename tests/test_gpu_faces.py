"""The staged MUSCL faces (face_tile) at the sizes where a tile can go wrong: rows shorter than a
stencil, rows of a tile's length and one off it, tiles of a single face, tails along each axis; a box
inside the block; against the oracle's faces to the bit, by the sweep of one axis (pga_flux) and by the
launch over all three (pga_faces), which write no other face. A trace species decaying into the
subnormals, zero slopes and signed zeros are among the cells."""

import numpy as np
import pytest

import support as sp
from oracle import oracle as O
from peregrine_amd import native
from test_gpu_parity import _case, _prepared, dev  # noqa: F401

pytestmark = pytest.mark.gpu

SIZES = [(1, 1, 1), (1, 90, 2), (2, 3, 61), (15, 16, 17), (16, 33, 2), (255, 2, 3), (256, 1, 2), (300, 5, 1), (64, 7, 31)]


@pytest.mark.parametrize("gas,primary,limiter", [("h2o2", "hllc", "koren"), ("binary", "rusanov", "vanleer"),
                                                 ("air-tpg", "hllc", "superbee"), ("air-cpg", "rusanov", "mc")])
@pytest.mark.parametrize("n", SIZES)
def test_faces_of_every_tile_match(dev, gas, primary, limiter, n):  # noqa: F811
    cfg, sim, nc, oc = _case(gas, "muscl", primary, limiter)
    hb = sp.HostBlock(n, sim.ng, sim.ne, 2, jostle=0.2, seed=5)
    q = sp.smooth_prims(hb.xcc, sim.ne, ns=sim.ns)
    if sim.ns > 1:
        q[..., 5:] *= 0.1
        # a front falling through the subnormals, and a species that is nowhere
        front = 10.0 ** -(3.0 * np.indices(q.shape[:3]).sum(axis=0) + 290.0)
        q[..., 5] = np.where(np.indices(q.shape[:3])[0] % 2, front, 0.0)
        if sim.ns > 2:
            q[..., 6] = 0.0
    q[::2, ..., 3] = -0.0
    _prepared(sim, oc, hb, q)
    ng, L = hb.ng, native.lib()
    dQv, dSt = dev.put(hb.regs[0]), dev.put(hb.state)
    dS = [dev.put(s) for s in hb.S]
    for inner in (False, True):
        start, ext = [ng] * 3, list(n)
        if inner:
            # a box inside the block: a cell in from the low ends where there is one to spare
            start = [ng + (m > 1) for m in n]
            ext = [max(1, m - 2) for m in n]
        boxes = [(start, [e + (a == b) for b, e in enumerate(ext)]) for a in range(3)]
        want = []
        for a, (s, e) in enumerate(boxes):
            F = np.full_like(hb.F[a], 7.0)
            O.lib.pgo_flux(oc.ref, a, O.arr(hb.regs[0]), O.arr(hb.state), O.arr(hb.S[a]), O.arr(F), O.box(s, e))
            want.append(F)
        one = [dev.put(np.full_like(f, 7.0)) for f in hb.F]
        for a, (s, e) in enumerate(boxes):
            native.check(L.pga_flux(nc.handle, a, dev.view(dQv), dev.view(dSt), dev.view(dS[a]), dev.view(one[a]),
                                    native.box(s, e), None), "pga_flux")
        every = [dev.put(np.full_like(f, 7.0)) for f in hb.F]
        none = native.View()
        native.check(L.pga_faces(nc.handle, dev.view(dQv), dev.view(dSt), (native.View * 3)(*map(dev.view, dS)),
                                 (native.View * 3)(*map(dev.view, every)),
                                 (native.Box * 3)(*[native.box(s, e) for s, e in boxes]), 0, 0.0, none, none, none,
                                 none, None, None), "pga_faces")
        for a in range(3):
            np.testing.assert_array_equal(dev.get(one[a]), want[a])
            np.testing.assert_array_equal(dev.get(every[a]), want[a])
