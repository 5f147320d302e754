"""Sets that grow above 32 rows in the exact form and refits of more than 32
rows in the fast forms (csrc/k_exact.hip, k_exact_fit): up to 1,024 sets of at
most 96 rows are fitted beside the larger ones in one launch (the only one up to
1,024 patches), more of them by a launch of their own.  All values are the oracle's, bit for bit.
"""
import numpy as np
import pytest

from core_amd import mesh, spr
from oracle import oracle as O
from test_gpu_rank_test_values import _min_ratio

pytestmark = pytest.mark.gpu


def _check(h, om, ip_order, q, nc, form="fp64", at=slice(None)):
    ip = np.random.default_rng(h.nt + nc).standard_normal((h.nt, q, nc))
    m = spr.Mesh(h)
    got = spr.recoverField(m.createIPField("f", nc, ip_order, ip), form=form).numpy()
    st = m.last_stats()
    m.close()
    assert np.array_equal(got[at], O.recover(om, ip)[at])
    return st


# an undistorted box grows most edge sets to 9-18 tets, 36 to 72 rows at four
# points (729, 1,331 and 4,913 patches)
@pytest.mark.parametrize("n", [4, 5, 8])
@pytest.mark.parametrize("nc", [1, 11])
def test_lattice_exact(gpu, n, nc):
    h = mesh.box(n, order=2)
    st = _check(h, O.Mesh(h.tv, h.xyz, 2, te=h.te, ev=h.ev), 2, 4, nc)
    assert st["expanded"] > 400


def fan(k, copies):
    """`copies` fans of k tets around one edge and a tet on an outer face.  The
    k centroids lie in a plane, so at one point per tet the fan's sets lack rank
    until they hold all k + 1 tets."""
    t = 2 * np.pi * np.arange(k) / k
    xyz = np.vstack([np.stack([np.cos(t), np.sin(t), 0 * t], 1), [[0, 0, 0], [0, 0, 1], [1.5, 0.4, 1.2]]])
    tv = np.array([[k, i, (i + 1) % k, k + 1] for i in range(k)] + [[0, 1, k + 1, k + 2]])
    n = len(xyz)
    return mesh.HostMesh(np.vstack([tv + c * n for c in range(copies)]),
                         np.vstack([xyz * (1 + 0.05 * c) + [4.0 * c, 0, 0] for c in range(copies)]), 1)


# sets on both sides of the lists' limits (64, 96, 128, 192 rows), on meshes on
# both sides of 1,024 patches
@pytest.mark.parametrize("rows", [33, 64, 65, 96, 97, 128, 129, 180])
@pytest.mark.parametrize("many", [False, True])
def test_fans_exact(gpu, rows, many):
    k = rows - 1
    h = fan(k, 1 + 1024 // (k + 3) if many else 1)
    om = O.Mesh(h.tv, h.xyz, 1)
    off, _ = O.patch_sets(om, 1)
    assert (h.nv > 1024) == many and (np.diff(off) == rows).sum() > h.nv // 2
    st = _check(h, om, 1, 1, 5)
    assert st["expanded"] > h.nv // 2


# a box bent into thin sheets: vertex sets of 96 rows and edge sets between
# have full rank and pivots far below 1e-6 (729 and 2,197 patches)
@pytest.mark.parametrize("form", ["fp64f", "fp32r"])
@pytest.mark.parametrize("n", [4, 6])
def test_refits(gpu, n, form):
    h = mesh.box(n, order=2)
    v = h.xyz[:h.nv].copy()
    v[:, 2] = 1e-3 * v[:, 2] + v[:, 0] ** 2 + v[:, 1] ** 2
    h = mesh.HostMesh(h.tv, np.vstack([v, v[h.ev[:, 0]] * 0.5 + v[h.ev[:, 1]] * 0.5]), 2, te=h.te, ev=h.ev)
    om = O.Mesh(h.tv, h.xyz, 2, te=h.te, ev=h.ev)
    x = h.ip_points(2)
    off, idx = O.vertex_tets(om)
    sets, _ = O.patch_sets(om, 4)
    at = [p for p in range(h.nv) if off[p + 1] - off[p] > 8 and sets[p + 1] - sets[p] == off[p + 1] - off[p]
          and _min_ratio(x[idx[off[p]:off[p + 1]]].reshape(-1, 3) - h.xyz[p]) < 1e-8]
    assert at
    _check(h, om, 2, 4, 9, form=form, at=at)
