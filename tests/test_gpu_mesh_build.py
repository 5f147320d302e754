"""The device's straight-sided test and slot layout (csrc/k_mesh.hip
k_straight, csrc/k_tile.hip k_tile_union).

The fast form takes sample points from the vertices' affine map where every
edge node is its edge's midpoint, from the Lagrange-2 map otherwise; the
exact form always takes the latter.  One edge node moved by a tenth of the
edge's length moves its tets' sample points by 1e-2 of it, so a test that
misses the edge shows at 1e-4 or more of the field; the forms' rounding on
these meshes stays below 1e-8 (condition numbers below 1e7 times 1e-16).
"""
import numpy as np
import pytest

from core_amd import mesh, spr
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,tet", [(2, None), (2, 0), (3, 63), (3, 64), (4, 255), (4, 256), (4, 383)])
def test_one_curved_edge(gpu, n, tet):
    h = mesh.box(n, order=2, jitter=0.2, seed=5)
    xyz = h.xyz.copy()
    if tet is not None:  # the last edge of that tet
        e = h.te[tet, 5]
        a, b = xyz[h.ev[e, 0]], xyz[h.ev[e, 1]]
        xyz[h.nv + e] += 0.1 * np.cross(b - a, [0.48, 0.6, 0.64])
    h = mesh.HostMesh(h.tv, xyz, 2, te=h.te, ev=h.ev)
    m = spr.Mesh(h)
    x = h.ip_points(2)
    ip = np.stack([np.sin(3 * x[..., 0] + x[..., 1]), x[..., 1] * x[..., 2], np.cos(2 * x[..., 2])], -1)
    f = m.createIPField("f", 3, 2, ip)
    r = spr.recoverField(f, form="fp64f")
    got = r.numpy()
    m.destroyField(r)
    ref = O.recover(O.Mesh(h.tv, h.xyz, 2, te=h.te, ev=h.ev), ip)
    assert np.array_equal(spr.recoverField(f, form="fp64").numpy(), ref)
    assert np.abs(got - ref).max() <= 1e-8 * np.abs(ref).max()
