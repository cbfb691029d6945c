"""The halo's gradients stored by the partner's own launch (pga_transport_grads_slabs) against the gradients
and their exchange, to the bit: periodic blocks, a lattice, blocks relabelled against each other with walls
around them, on both sides of the size the two kernels share a launch to."""

import numpy as np
import pytest

import support as sp
from peregrine_amd import get_backend, get_solver, mesher

pytestmark = pytest.mark.gpu


def _mesh(kind, n):
    if kind == "reoriented":
        return sp.ReorientedPair(n, mbdims=[2, 1, 1], blkdims=[6, 3, 2], lengths=[2.0, 1.0, 1.0], defaultbc="wall")
    mb = [1, 1, 1] if kind == "block" else [2, 1, 1]
    return mesher.CubeMesher(mbdims=mb, blkdims=[m + 1 for m in n], lengths=[0.01 * m for m in n], periodic=[True] * 3)


@pytest.mark.parametrize("gas,trans", [("air-tpg", "constant"), ("binary", "constant"), ("h2o2", "kinetic-theory")])
@pytest.mark.parametrize("kind,n", [("block", (2, 2, 2)), ("block", (5, 33, 4)), ("block", (41, 40, 41)),
                                    ("lattice", (7, 3, 16)), ("reoriented", "123"), ("reoriented", "231"),
                                    ("reoriented", "426"), ("reoriented", "612")])
def test_the_slabs_gradients_are_the_exchanged_ones(gpu, gas, trans, kind, n):
    if kind == "reoriented" and n not in sp.orientations():
        n = sp.orientations()[int(n) % len(sp.orientations())]
    cfg = sp.config(gas, recon="muscl", primary="hllc", limiter="koren", trans=trans)
    cfg["bcvals"]["wall"] = {"kind": "slp-adia-wall"}
    mb = get_solver(cfg, _mesh(kind, n), get_backend("mi355x", cfg))
    mb.set_prims([sp.smooth_prims(blk.xcc.get(), mb.sim.ne, ns=mb.sim.ns) for blk in mb.blocks])
    found = []
    for way in (mb.gradients, mb.transport_gradients):
        for blk in mb.blocks:
            blk.grads.set(np.full(blk.grads.get().shape, 3.0))
        way(0)
        found.append([blk.grads.get() for blk in mb.blocks])
    for want, got in zip(*found):
        assert (want != 3.0).any()
        np.testing.assert_array_equal(got, want)
