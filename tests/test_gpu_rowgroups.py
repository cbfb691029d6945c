"""The stage's rows in groups (a block below 2^17 cells) against the reference's sequence of launches, to the
bit: a thread a row, uneven last groups, one cell to a side, and both sides of the size where groups end."""

import numpy as np
import pytest

import support as sp
from peregrine_amd import get_backend, get_solver, mesher
from test_gpu_parity import _rowerr, _run_pair

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


def test_a_long_line_along_k_steps_as_the_oracle(gpu):
    """Nine species on 5100 cells one to a plane, whose thirteen rows in groups of their own would take more of
    the grid's z than a box's planes may: the walled line by the fused stage, within the reacting case's bound."""
    L = (0.01, 0.01, 0.4)
    mb, hb = _run_pair("h2o2", "muscl", "hllc", "koren", True, "tvd-rk3", (1, 1, 5100), 3, 1e-9,
                       lambda x: sp.reacting_flow(x, 1, L), L, walls=range(6))
    assert mb.fused
    g = hb.ng
    got = mb.blocks[0].Q.get()[g:-g, g:-g, g:-g].transpose(3, 2, 1, 0)
    assert _rowerr(got, hb.regs[0][hb.interior()]) < 1e-10
