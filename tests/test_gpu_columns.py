"""The implicit form's matrices at the edges of its launches' shapes: 64 cells a workgroup of the species
columns, 16 a group of the work array, 256 a tile of the whole evaluations."""

import ctypes

import numpy as np
import pytest

import support as sp
from oracle import oracle as O
from peregrine_amd import native
from test_gpu_implicit import _device_y
from test_gpu_parity import _case, _hot_and_cold, dev  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ncell", [(1, 1, 1), (63, 1, 1), (4, 8, 2), (5, 13, 1), (257, 1, 1)])
def test_matrices_of_every_cell_and_nothing_past_them(dev, ncell):
    """Each cell's matrix against pgo_implicit_matrix at its y rounded to FP32: the same rates and steps,
    the species columns' sums in the same order, so within 1e-12 of a column's largest entry as the
    matrices of a whole block are; and a guard past the work array as it was."""
    import torch

    cfg, sim, nc, oc = _case("h2o2", chem=True)
    q = _hot_and_cold(sim, ncell, radicals=1e-3)
    hb = sp.HostBlock(ncell, 0, sim.ne, 1)
    O.lib.pgo_fromprims(oc.ref, O.arr(sp.to_dev(q)), O.arr(hb.regs[0]), O.arr(hb.state), O.box((0, 0, 0), ncell))
    L = native.lib()
    box = native.box((0, 0, 0), ncell)
    cells, nv, dt = int(np.prod(ncell)), sim.ns + 1, 1e-7
    groups = -(-cells // 16)
    nwork = int(L.pga_implicit_worksize(nc.handle, box))
    work = torch.full((nwork + 4096,), -7.0, dtype=torch.float64, device="cuda")
    sweeps = torch.zeros(cells, dtype=torch.int32, device="cuda")
    out = dev.put(np.zeros((sim.ns - 1,) + hb.regs[0].shape[1:]))
    ddt = dev.put(np.array([dt]))
    opts = native.ImplicitOpts(1, 8, 1e-13)
    native.check(L.pga_implicit(nc.handle, ctypes.byref(opts), dev.view(dev.put(hb.regs[0])), dev.view(dev.put(hb.state)),
                                dev.view(out), 0, sweeps.data_ptr(), cells, work.data_ptr(), nwork, ddt.data_ptr(), box,
                                None), "pga_implicit")
    w = work.cpu().numpy()
    assert (w[nwork:] == -7.0).all()
    A = w[:groups * nv * nv * 16].reshape(groups, nv, nv, 16).transpose(0, 3, 1, 2).reshape(-1, nv, nv)[:cells]
    y, rho = _device_y((hb.regs[0].reshape(sim.ne, -1), hb.state[1].reshape(-1)), sim)
    for c in range(cells):
        want = oc.implicit_matrix(rho[c], y[:, c].astype(np.float32).astype(np.float64), dt)
        assert (np.abs(A[c] - want).max(axis=0) <= 1e-12 * np.abs(want).max(axis=0)).all()
    taken = sweeps.cpu().numpy()
    assert (taken >= 1).all() and (taken <= 8).all()
