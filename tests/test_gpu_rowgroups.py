"""The stage's rows in groups (a block below 2^17 cells) against the reference's sequence of launches, to the
bit: a thread a row, uneven last groups, one cell to a side, and both sides of the size where groups end."""

import numpy as np
import pytest

import support as sp
from peregrine_amd import get_backend, get_solver, mesher

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(2, 2, 2), (17, 45, 40), (41, 40, 50), (64, 64, 32), (64, 64, 33)])
def test_a_stage_by_row_groups_is_the_sequence(gpu, n):
    out = []
    for fused in (True, False):
        cfg = sp.config("h2o2", recon="muscl", primary="hllc", limiter="koren", chem=True, dt=1e-8)
        cfg["backend-mi355x"]["fused-stage"] = fused
        mesh = mesher.CubeMesher(blkdims=[m + 1 for m in n], lengths=[0.01] * 3, periodic=[True] * 3)
        mb = get_solver(cfg, mesh, get_backend("mi355x", cfg))
        mb.set_prims([sp.reacting_flow(mb.blocks[0].xcc.get(), n[0], [0.01] * 3)])
        for _ in range(2):
            mb.step(1e-8)
        blk = mb.blocks[0]
        out.append((blk.Q.get()[blk.interior], blk.state.get()[blk.interior]))
    for got, want in zip(*out):
        np.testing.assert_array_equal(got, want)
