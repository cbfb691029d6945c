"""The halo pass and the rates in one launch (pga_halo_rates) against a launch each, to the bit, on blocks
with tails of a workgroup, of one workgroup, and without a halo to fill."""

import numpy as np
import pytest

import support as sp
from peregrine_amd import get_backend, get_solver, mesher

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,periodic", [((2, 2, 2), True), ((5, 33, 4), True), ((64, 4, 2), True), ((7, 3, 16), False)])
def test_one_launch_is_the_two(gpu, n, periodic):
    cfg = sp.config("h2o2", recon="muscl", primary="hllc", limiter="koren", chem=True)
    cfg["bcvals"]["wall"] = {"kind": "slp-adia-wall"}
    mesh = mesher.CubeMesher(mbdims=[2, 1, 1] if periodic else [1, 1, 1], blkdims=[m + 1 for m in n],
                             lengths=[0.01 * m for m in n], periodic=[periodic] * 3, defaultbc="wall")
    mb = get_solver(cfg, mesh, get_backend("mi355x", cfg))
    mb.set_prims([sp.reacting_flow(blk.xcc.get(), n[0], [0.01 * m for m in n]) for blk in mb.blocks])
    start = [(blk.Q.get().copy(), blk.state.get().copy()) for blk in mb.blocks]
    found = []
    for one in (False, True):
        for blk, (Q, st) in zip(mb.blocks, start):
            # halos spoiled, their T kept: what the pass does not write would show
            q, s = np.full_like(Q, 3.0), np.full_like(st, 3.0)
            q[blk.interior], s[blk.interior] = Q[blk.interior], st[blk.interior]
            s[..., 1] = st[..., 1]
            blk.Q.set(q)
            blk.state.set(s)
            blk.rates.set(np.full_like(blk.rates.get(), 5.0))
        mb._halo_pass(0, rates=one)
        if not one:
            for blk in mb.blocks:
                mb.chemistry_source(blk, blk.Q.view(), blk.rates.view(), False)
        found.append([a.get() for blk in mb.blocks for a in (blk.Q, blk.state, blk.rates)])
    for want, got in zip(*found):
        np.testing.assert_array_equal(got, want)
