"""The slabs a block's gradients are stored into (Solver._gradient_slabs) on the CPU: every interface that faces
the block, in a lattice and across every orientation, found without a walk over the lattice."""

from types import SimpleNamespace

import pytest

import support as sp
from peregrine_amd import mesher, native
from peregrine_amd.solver import Block, Solver, placement


class _Block(Block):
    """A block that counts the reads of its interfaces."""

    reads = 0

    @property
    def faces(self):
        self.reads += 1
        return self._faces

    @faces.setter
    def faces(self, faces):
        self._faces = faces


class _Lattice:
    def __init__(self):
        self.blocks, self.ng = [], 2

    def add_blk(self):
        blk = _Block(len(self.blocks), self)
        # a view by which a slab's destination is told
        blk.grads = SimpleNamespace(view=lambda n=blk.nblki: native.View(sj=n + 1))
        self.blocks.append(blk)
        return blk


def _meshes():
    yield mesher.CubeMesher(blkdims=[5, 4, 6], periodic=[True, False, True], defaultbc="wall")
    yield mesher.CubeMesher(mbdims=[3, 4, 5], blkdims=[4, 4, 4], periodic=[True, False, True], defaultbc="wall")
    yield mesher.CubeMesher(mbdims=[2, 1, 1], blkdims=[4, 4, 4], periodic=[True] * 3)
    for S in sp.orientations():
        yield sp.ReorientedPair(S, mbdims=[2, 1, 1], blkdims=[6, 4, 3], lengths=[2.0, 1.3, 0.7], defaultbc="wall")


@pytest.mark.parametrize("mesh", _meshes())
def test_every_interface_that_faces_a_block(mesh):
    mb = _Lattice()
    mesh.fill(mb)
    for blk in mb.blocks:
        want = sorted((dst.nblki, *map(tuple, placement(dst, f, blk, 1))) for dst in mb.blocks
                      for f in dst.faces.values() if f.nbr == blk.nblki)
        for b in mb.blocks:
            b.reads = 0
        n, views, *p = Solver._gradient_slabs(mb, blk, False)
        got = sorted((views[m].sj - 1, *(tuple(a[3 * m:3 * m + 3]) for a in p)) for m in range(n))
        assert got == want and n <= 6
        assert sum(b.reads for b in mb.blocks) <= 7
        assert Solver._gradient_slabs(mb, blk, True)[0] == 0
