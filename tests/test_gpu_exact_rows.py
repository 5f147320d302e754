"""The exact fits (csrc/k_qr.hip) at the edges of their row buckets.

A star mesh has one vertex in T tets, so at one point per tet that vertex's
fit has exactly T rows: sizes on both sides of every bucket limit (16, 24, 32,
64, 96, 128, 192 rows), with 4- and 10-term fits and component counts on both
sides of a wave's lanes.  The recovered field must equal the oracle's bit for
bit.  A mesh whose large sets outnumber the sets of one launch sequence (the
allocation-free entry point holds about 3,800 of them) must equal the
recovery that takes them in one.
"""
import ctypes

import numpy as np
import pytest
import torch

import smb_util
from core_amd import _lib, mesh, spr, workloads
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _star(tets, order):
    tv, xyz = smb_util.star(tets // 2 + 2)  # 2 k - 4 tets
    assert np.bincount(tv.ravel()).max() == tets
    if order == 1:
        return mesh.HostMesh(tv, xyz, 1)
    pairs = np.sort(tv[:, mesh.TET_EDGE_VERTS].reshape(-1, 2), axis=1)
    ev, te = np.unique(pairs, axis=0, return_inverse=True)
    mid = xyz[ev[:, 0]] * 0.5 + xyz[ev[:, 1]] * 0.5
    return mesh.HostMesh(tv, np.vstack([xyz, mid]), 2, te=te.reshape(-1, 6), ev=ev, ne=ev.shape[0])


ROWS = [16, 18, 24, 26, 32, 34, 64, 66, 96, 98, 128, 130, 190, 192]


# 194: the large-set kernel's first size (order 1: on an order-2 star some
# edge's set grows to all tets, and sets that grow hold at most 192)
@pytest.mark.parametrize("tets,order", [(t, o) for t in ROWS for o in (1, 2)] + [(194, 1)])
def test_bucket_edges_bitwise(gpu, tets, order):
    h = _star(tets, order)
    om = O.Mesh(h.tv, h.xyz, order, te=h.te, ev=h.ev)
    m = spr.Mesh(h)
    rng = np.random.default_rng(tets + order)
    for nc in (1, 9, 10, 11, 27):
        ip = rng.standard_normal((h.nt, 1, nc))
        f = m.createIPField("f%d" % nc, nc, 1, ip)
        r = spr.recoverField(f)
        assert np.array_equal(r.numpy(), O.recover(om, ip)), (tets, order, nc)
    m.close()


def test_sets_in_several_sequences(gpu):
    h = mesh.box(20, order=2, jitter=0.25, seed=workloads.C5)
    m = spr.Mesh(h)
    f = m.createIPField("eps", 9, 2, workloads.strain_field(h.ip_points(2)))
    ref = spr.recoverField(f)
    out = torch.full_like(ref.data, float("nan"))
    torch.cuda.synchronize()
    _lib.check(_lib.lib().sprg_recover_noalloc(m.handle, 2, 9, ctypes.c_void_p(f.data.data_ptr()),
                                               ctypes.c_void_p(out.data_ptr()), spr.FORMS["fp64"]))
    assert torch.equal(out, ref.data)
    m.close()
