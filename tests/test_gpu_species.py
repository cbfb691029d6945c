"""A mechanism of more species than the main library's nine on the device, by the library built for it: the
staged faces where a tile's LDS grows with the species, and a reacting step."""

import numpy as np
import pytest

import support as sp
from oracle import oracle as O
from peregrine_amd import native
from peregrine_amd.backend import Mi355xBackend
from peregrine_amd.simulator import NativeCase, get_simulator
from test_gpu_parity import _prepared, _rowerr, _run_pair, dev  # noqa: F401

pytestmark = [pytest.mark.gpu, pytest.mark.timeout(600)]


@pytest.mark.parametrize("n", [(64, 8, 12), (50, 16, 10), (33, 4, 65)])
def test_faces_of_fourteen_species_match(dev, n, tmp_path):  # noqa: F811
    """Rows of 49 to 64 faces with few along the axis, which take the widest tile of fewer species; to the
    bit, by one axis and by all three at once."""
    cfg = sp.config("h2o2", recon="muscl", primary="hllc", limiter="koren", chem=True)
    cfg["mixture"]["species"] = sp.grown_mechanism(tmp_path, 14, 20)
    sim = get_simulator(cfg)
    nc, oc = NativeCase(sim, Mi355xBackend(cfg)), O.OracleCase(sim.mixture, "muscl", "koren", "hllc")
    assert sim.ns == 14 and nc.L is not native.lib()
    hb = sp.HostBlock(n, sim.ng, sim.ne, 2, jostle=0.2, seed=5)
    _prepared(sim, oc, hb, sp.smooth_prims(hb.xcc, sim.ne, ns=sim.ns))
    dQv, dSt = dev.put(hb.regs[0]), dev.put(hb.state)
    dS = [dev.put(s) for s in hb.S]
    boxes = [([hb.ng] * 3, [e + (a == b) for b, e in enumerate(n)]) for a in range(3)]
    one, every = ([dev.put(np.full_like(f, 7.0)) for f in hb.F] for _ in range(2))
    none = native.View()
    for a, (s, e) in enumerate(boxes):
        native.check(nc.L.pga_flux(nc.handle, a, dev.view(dQv), dev.view(dSt), dev.view(dS[a]), dev.view(one[a]),
                                   native.box(s, e), None), "pga_flux", nc.L)
    native.check(nc.L.pga_faces(nc.handle, dev.view(dQv), dev.view(dSt), (native.View * 3)(*map(dev.view, dS)),
                                (native.View * 3)(*map(dev.view, every)),
                                (native.Box * 3)(*[native.box(s, e) for s, e in boxes]), 0, 0.0, none, none, none,
                                none, None, None), "pga_faces", nc.L)
    for a, (s, e) in enumerate(boxes):
        want = np.full_like(hb.F[a], 7.0)
        O.lib.pgo_flux(oc.ref, a, O.arr(hb.regs[0]), O.arr(hb.state), O.arr(hb.S[a]), O.arr(want), O.box(s, e))
        np.testing.assert_array_equal(dev.get(one[a]), want)
        np.testing.assert_array_equal(dev.get(every[a]), want)


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
