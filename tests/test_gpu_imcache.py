"""The implicit form's caches past 64 KB of LDS a workgroup, and past all of it (then in the work array): the
matrices against the oracle's, and a step of a table of blocks against the same blocks in turn."""

import ctypes

import numpy as np
import pytest

import support as sp
from oracle import oracle as O
from peregrine_amd import get_backend, get_solver, mesher, native
from peregrine_amd.backend import Mi355xBackend
from peregrine_amd.simulator import NativeCase, get_simulator
from test_gpu_implicit import _device_y
from test_gpu_parity import dev  # noqa: F401

pytestmark = [pytest.mark.gpu, pytest.mark.timeout(600)]

SIZES = [sp.CACHE_PAST_64K, sp.CACHE_PAST_LDS]


def _config(directory, nr):
    cfg = sp.config("h2o2", recon="muscl", primary="hllc", limiter="koren", chem=True)
    cfg["mixture"]["species"] = sp.recombination_mechanism(directory, nr)
    cfg["chem-integration"]["kind"] = "implicit"
    return cfg


def _prims(x, seed=2):
    q = np.zeros(x.shape[:3] + (7,))
    r = np.random.default_rng(seed)
    q[..., 0] = 101325.0
    q[..., 1:4] = r.uniform(-5.0, 5.0, x.shape[:3] + (3,))
    q[..., 4] = r.uniform(1200.0, 3000.0, x.shape[:3])
    q[..., 5], q[..., 6] = r.uniform(1e-3, 0.05, x.shape[:3]), 0.2
    return q


@pytest.mark.parametrize("nr", SIZES)
def test_matrices_are_the_oracles(dev, nr, tmp_path):  # noqa: F811
    """Every cell's matrix within 1e-12 of its columns' largest entries, as the H2/O2 case's are, over a
    partial last workgroup; and a guard past the work array as it was."""
    import torch

    cfg = _config(tmp_path, nr)
    sim = get_simulator(cfg)
    nc, oc = NativeCase(sim, Mi355xBackend(cfg)), O.OracleCase(sim.mixture, "muscl", "koren", "hllc")
    ncell = (5, 13, 2)
    hb = sp.HostBlock(ncell, 0, sim.ne, 1)
    O.lib.pgo_fromprims(oc.ref, O.arr(sp.to_dev(_prims(np.zeros(ncell + (3,))))), O.arr(hb.regs[0]), O.arr(hb.state),
                        O.box((0, 0, 0), ncell))
    box, cells, nv, dt = native.box((0, 0, 0), ncell), int(np.prod(ncell)), sim.ns + 1, 1e-6
    groups = -(-cells // 16)
    nwork = int(nc.L.pga_implicit_worksize(nc.handle, box))
    assert (nwork > groups * nv * nv * 16 + 3 * nv * cells) == (nr == sp.CACHE_PAST_LDS)
    work = torch.full((nwork + 4096,), -7.0, dtype=torch.float64, device="cuda")
    sweeps = torch.zeros(cells, dtype=torch.int32, device="cuda")
    out = dev.put(np.zeros((sim.ns - 1,) + hb.regs[0].shape[1:]))
    ddt = dev.put(np.array([dt]))
    opts = native.ImplicitOpts(1, 8, 1e-13)
    native.check(nc.L.pga_implicit(nc.handle, ctypes.byref(opts), dev.view(dev.put(hb.regs[0])),
                                   dev.view(dev.put(hb.state)), dev.view(out), 0, sweeps.data_ptr(), cells,
                                   work.data_ptr(), nwork, ddt.data_ptr(), box, None), "pga_implicit", nc.L)
    w = work.cpu().numpy()
    assert (w[nwork:] == -7.0).all()
    A = w[:groups * nv * nv * 16].reshape(groups, nv, nv, 16).transpose(0, 3, 1, 2).reshape(-1, nv, nv)[:cells]
    y, rho = _device_y((hb.regs[0].reshape(sim.ne, -1), hb.state[1].reshape(-1)), sim)
    for c in range(cells):
        want = oc.implicit_matrix(rho[c], y[:, c].astype(np.float32).astype(np.float64), dt)
        assert (np.abs(A[c] - want).max(axis=0) <= 1e-12 * np.abs(want).max(axis=0)).all()
    taken = sweeps.cpu().numpy()
    assert (taken >= 1).all() and (taken <= 8).all()


@pytest.mark.parametrize("nr", SIZES)
def test_a_table_of_blocks_steps_as_the_blocks_in_turn(dev, nr, tmp_path):  # noqa: F811
    """Three steps, two parts each, the later ones replayed from a graph, to the bit."""
    out = []
    for batched in ("auto", False):
        cfg = _config(tmp_path, nr)
        cfg["chem-integration"]["implicit-parts"] = 2
        cfg["backend-mi355x"]["batched"] = batched
        mesh = mesher.CubeMesher(mbdims=[2, 1, 1], blkdims=[8, 6, 4], lengths=[0.01] * 3, periodic=[True] * 3)
        mb = get_solver(cfg, mesh, get_backend("mi355x", cfg))
        mb.set_prims([_prims(b.xcc.get(), n) for n, b in enumerate(mb.blocks)])
        assert mb.batched == (batched == "auto")
        for _ in range(3):
            mb.step(1e-8)
        assert mb.replays > 0
        out.append([a.get()[b.interior] for b in mb.blocks for a in (b.Q, b.state)])
        mb.release()
    for got, want in zip(*out):
        assert np.isfinite(got).all()
        np.testing.assert_array_equal(got, want)
