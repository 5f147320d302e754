"""Values of the patches whose initial set passes the batched rank test
(csrc/k_qr.hip, k_rank_test) and is kept.  On a box whose nodes are moved off
the lattice by 1e-4 to 1e-2 of a cell, most sets have full rank with pivots far
below what the fast forms certify, next to sets that lack rank or rows.

A patch whose smallest Cholesky pivot keeps less than 1e-6 of its diagonal is
queued for the test; if the set passes, the fit of the kept set meets the same
small pivot and hands it to the exact kernel, so the value equals the oracle's
bit for bit.  The patches are picked here: initial set kept by the oracle,
pivot ratio below 1e-8 in FP64 (its rounding, some tens of 2^-53 times the
growth of the factorisation, is far below the gap to 1e-6).  A wrong place in
the set storage, a wrong patch id or a wrong tet gives another set's value.
"""
import numpy as np
import pytest

from core_amd import mesh, spr
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _min_ratio(x):
    """Smallest pivot over its diagonal of the Gram matrix of the ten
    monomials at the centred points x."""
    a = np.stack([np.ones(len(x)), x[:, 0], x[:, 1], x[:, 2], x[:, 0] * x[:, 1], x[:, 1] * x[:, 2],
                  x[:, 2] * x[:, 0], x[:, 0] ** 2, x[:, 1] ** 2, x[:, 2] ** 2], 1)
    g = a.T @ a
    diag = g.diagonal().copy()
    low = 1.0
    for k in range(10):
        r = g[k, k] / diag[k]
        low = min(low, r)
        if not r > 0:
            break
        g[k + 1:, k + 1:] -= np.outer(g[k + 1:, k], g[k, k + 1:]) / g[k, k]
    return low


def kept_patches(h, om, q):
    """Patches that keep an initial set with a pivot ratio below 1e-8."""
    x = h.ip_points(2)[:, :q]  # the first points of the mesh order's rule
    off, idx = O.patch_sets(om, q)
    init = []
    for o, i in (O.vertex_tets(om), O.edge_tets(om)):
        init += [i[o[k]:o[k + 1]] for k in range(len(o) - 1)]
    keep = []
    for p, s in enumerate(init):
        if 10 <= q * len(s) <= 32 and np.array_equal(s, idx[off[p]:off[p + 1]]):
            if _min_ratio(x[s].reshape(-1, 3) - h.xyz[p]) < 1e-8:
                keep.append(p)
    return np.array(keep, int)


@pytest.mark.parametrize("form", ["fp64f", "fp32r"])
@pytest.mark.parametrize("n,jitter,ip_order", [(8, 1e-2, 1), (8, 1e-3, 1), (3, 1e-3, 2), (6, 1e-4, 2), (7, 1e-2, 2)])
def test_kept_sets_bitwise(gpu, n, jitter, ip_order, form):
    h = mesh.box(n, order=2, jitter=jitter, seed=7)
    om = O.Mesh(h.tv, h.xyz, 2, te=h.te, ev=h.ev)
    q = {1: 1, 2: 4}[ip_order]
    keep = kept_patches(h, om, q)
    assert keep.size > 0
    ip = np.random.default_rng(n).standard_normal((h.nt, q, 3))
    m = spr.Mesh(h)
    got = spr.recoverField(m.createIPField("f", 3, ip_order, ip), form=form).numpy()
    ref = O.recover(om, ip)
    assert np.array_equal(got[keep], ref[keep])
    m.close()
