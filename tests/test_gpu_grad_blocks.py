"""Integration-point gradients at the edges of the gradient kernel's blocks
(csrc/k_grad.hip): 64 tets to a block for the four- and five-point rules, 256
for the one-point rule, results leaving through LDS in parts of a block.

The kernel evaluates the reference's operations in the reference's order, so
every value equals the oracle's, on curved edges too.
"""
import numpy as np
import pytest

from core_amd import mesh, spr
from oracle import oracle as O

pytestmark = pytest.mark.gpu

# tets kept of a box: below a block, around a part of one, around a block of
# either size, several and a remainder
NT = [1, 15, 17, 63, 64, 65, 255, 256, 257, 641]


def _part(nt, order, with_edges):
    h = mesh.box(5, order=2, jitter=0.25, seed=3)
    rng = np.random.default_rng(nt)
    xyz = h.xyz.copy()
    xyz[h.nv:] += 0.01 * rng.standard_normal((h.ne, 3))  # curved edges
    # the part's own vertices and edges, renumbered in order of first id
    v, tv = np.unique(h.tv[:nt], return_inverse=True)
    e, te = np.unique(h.te[:nt], return_inverse=True)
    vmap = np.full(h.nv, -1)
    vmap[v] = np.arange(v.size)
    if order == 2:
        x = np.concatenate([xyz[v], xyz[h.nv + e]])
    else:
        x = xyz[v]
    if order == 1 and not with_edges:
        return mesh.HostMesh(tv.reshape(-1, 4), x, 1)
    return mesh.HostMesh(tv.reshape(-1, 4), x, order, te=te.reshape(-1, 6), ev=vmap[h.ev[e]])


@pytest.mark.parametrize("nt", NT)
def test_blocks_bitwise(gpu, nt):
    rng = np.random.default_rng(100 + nt)
    for order, edges in [(1, False), (1, True), (2, True)]:
        h = _part(nt, order, edges)
        om = O.Mesh(h.tv, h.xyz, order, te=h.te, ev=h.ev)
        m = spr.Mesh(h)
        for forder in (1, 2) if edges else (1,):
            for nc in (1, 3, 9):
                vals = rng.standard_normal((h.nv + (h.ne if forder == 2 else 0), nc))
                f = m.createLagrangeField("u", nc, forder, vals)
                for ipo in (1, 2, 3):
                    what = (nt, order, edges, forder, nc, ipo)
                    if order == 1 and forder == 2 and nc != 9:  # refused, as before
                        with pytest.raises(spr.SPRError):
                            spr.getGradIPField(f, "g", ipo)
                        continue
                    g = spr.getGradIPField(f, "g", ipo)
                    assert np.array_equal(g.numpy(), O.grad_ip(om, forder, vals, ipo)), what
                    m.destroyField(g)
                m.destroyField(f)
