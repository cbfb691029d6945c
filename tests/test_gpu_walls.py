"""A block's walls in one launch (pga_wall_mirrors, pga_wall_fluxes) against a call per wall, to the
bit: every face a wall, of different kinds, on blocks one cell thin, with tails of a workgroup, and
across its edge."""

import ctypes

import numpy as np
import pytest

import support as sp
from peregrine_amd import get_backend, get_solver, mesher, native

pytestmark = pytest.mark.gpu

KINDS = {1: ("slp-adia-wall", {}), 2: ("slp-isot-wall", {"T": 350.0}), 3: ("no-slp-adia-wall", {}),
         4: ("no-slp-isot-wall", {"T": 420.0}), 5: ("mov-adia-wall", {"u": 20.0, "v": 0.0, "w": -4.0}),
         6: ("mov-isot-wall", {"u": 5.0, "v": 2.0, "w": 0.0, "T": 500.0})}


@pytest.mark.parametrize("gas,trans", [("binary", None), ("air-tpg", "constant"), ("h2o2", "kinetic-theory")])
@pytest.mark.parametrize("n", [(1, 1, 1), (300, 1, 2), (5, 33, 16), (16, 16, 1)])
def test_every_wall_in_one_launch_is_a_call_per_wall(gpu, gas, trans, n):
    cfg = sp.config(gas, recon="muscl", primary="hllc", limiter="koren", trans=trans)
    for f, (kind, values) in KINDS.items():
        if trans is None and f > 2:
            kind, values = KINDS[1 + f % 2]
        cfg["bcvals"][f"w{f}"] = {"kind": kind, **values}
    mesh = mesher.CubeMesher(blkdims=[m + 1 for m in n], lengths=[0.01 * m for m in n], periodic=[False] * 3,
                             bcnames={f: f"w{f}" for f in KINDS})
    mb = get_solver(cfg, mesh, get_backend("mi355x", cfg))
    blk = mb.blocks[0]
    mb.set_prims([sp.smooth_prims(blk.xcc.get(), mb.sim.ne, ns=mb.sim.ns)])
    if trans:
        mb.transport(0)
    outs = []
    faces = (blk.iF, blk.jF, blk.kF)
    for each in (False, True):
        # every halo spoiled first: what the walls do not write would show as the spoilt value
        rng = np.random.default_rng(5)
        for arr in (blk.Q, blk.state, *faces):
            host = arr.get().copy()
            spoilt = rng.random(host.shape)
            if arr in (blk.Q, blk.state):
                spoilt[blk.interior] = host[blk.interior]
            arr.set(spoilt)
        nw, axes, head = mb._walls(blk)
        visc = mb.sim.viscous
        if each:
            for axis, side, wall in blk.walls:
                S = (blk.iS, blk.jS, blk.kS)[axis].view()
                mb._call("pga_wall_mirror", mb.case.handle, axis, side, ctypes.byref(wall), native.ints(n), mb.ng,
                         blk.Q.view(), blk.state.view(), S)
                mb._call("pga_wall_flux", mb.case.handle, axis, side, ctypes.byref(wall), native.ints(n), mb.ng,
                         blk.Q.view(), blk.state.view(), blk.trstate.view() if visc else native.View(),
                         blk.xcc.view(), blk.xf[axis].view() if visc else native.View(), S, faces[axis].view())
        else:
            mb.wall_halos(0)
            S, F = ((native.View * nw)(*[arr[a].view() for a in axes]) for arr in ((blk.iS, blk.jS, blk.kS), faces))
            xf = (native.View * nw)(*[blk.xf[a].view() for a in axes]) if visc else None
            mb._call("pga_wall_fluxes", *head, blk.Q.view(), blk.state.view(),
                     blk.trstate.view() if visc else native.View(), blk.xcc.view(), xf, S, F)
        outs.append([arr.get().copy() for arr in (blk.Q, blk.state, *faces)])
    for a, b in zip(*outs):
        np.testing.assert_array_equal(a, b)
    # the mirror wrote its halos: a slip wall's halo cell holds the first cell's density
    g = mb.ng
    Q = outs[0][0]
    assert np.all(Q[g - 1, g:-g, g:-g, 0] == Q[g, g:-g, g:-g, 0])
