"""A mechanism of more species than the main library's nine on the device, by the library built for it."""

import numpy as np
import pytest

import support as sp
from test_gpu_parity import _rowerr, _run_pair, dev  # noqa: F401

pytestmark = [pytest.mark.gpu, pytest.mark.timeout(600)]


def test_a_reacting_step_of_fourteen_species_matches(dev, tmp_path):  # noqa: F811
    """Ten steps by the fused stage against the oracle, within the bound of the nine-species case."""
    n, L = 20, (0.01,) * 3

    def prims(x):
        q9 = sp.reacting_flow(x, n, L)
        q = np.zeros(x.shape[:3] + (18,))
        q[..., :13], q[..., 13:] = q9, 1e-5
        q[..., 12] = 1e-5
        return q

    mb, hb = _run_pair("h2o2", "muscl", "hllc", "koren", True, "tvd-rk3", (n, n, n), 10, 1e-8, prims, L,
                       species=sp.grown_mechanism(tmp_path, 14, 20))
    g = hb.ng
    got = mb.blocks[0].Q.get()[g:-g, g:-g, g:-g].transpose(3, 2, 1, 0)
    err = _rowerr(got, hb.regs[0][hb.interior()])
    print(f"14 species 10 steps: {err:.3e}")
    assert err < 1e-10
