"""More sets of one row bucket than the exact fits' workspace holds at a time
(csrc/k_qr.hip, QR_CHUNK = 12288): a box of 26^3 cubes has 25^3 = 15,625 inner
vertices of 24 tets, 96 rows each.  The exact form is bit-identical to the
oracle's, the chunks' seams included.
"""
import numpy as np
import pytest

from core_amd import mesh, spr
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def test_two_chunks_bitwise(gpu):
    h = mesh.box(26, order=2, jitter=0.2, seed=4)
    om = O.Mesh(h.tv, h.xyz, 2, te=h.te, ev=h.ev)
    m = spr.Mesh(h)
    x = h.ip_points(2)
    ip = np.sin(3 * x[..., :1] + x[..., 1:2] * x[..., 2:])
    r = spr.recoverField(m.createIPField("f", 1, 2, ip), form="fp64").numpy()
    nv = h.nv
    assert np.array_equal(r[:nv], O.recover(om, ip, 0, nv)[:nv])
