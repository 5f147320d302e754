"""An exact-form batch beside eager exact calls of its context, which share the
workspace of the exact fits with the batch's first lane: an eager call on a
mesh with more large sets (27 vertices of 96 rows in the batch's largest mesh,
1,331 in the eager one) moves it, and the next batch call must record again.
Every replay equals the per-mesh calls, with eager work between the replays."""
import numpy as np
import pytest
import torch

from core_amd import _lib, mesh, spr, workloads

pytestmark = pytest.mark.gpu


def test_workspace_moves_between_replays(gpu, monkeypatch):
    monkeypatch.setattr(spr, "_CTX", {})  # a context of its own, with no workspace yet
    hosts = [mesh.box(n, order=2, jitter=0.2, seed=workloads.C4 + n) for n in (4, 3, 2, 3, 4)]
    ms = [spr.Mesh(h) for h in hosts]
    fs = [m.createIPField("eps", 9, 2, workloads.strain_field(h.ip_points(2))) for m, h in zip(ms, hosts)]
    batch = spr.Batch(ms)
    outs = batch.size_fields(fs, adapt_ratio=0.05)
    first = [o.clone() for o in outs]
    big = mesh.box(12, order=2, jitter=0.2, seed=workloads.C5)
    mb = spr.Mesh(big)
    fb = mb.createIPField("eps", 9, 2, workloads.strain_field(big.ip_points(2)))
    for k in range(4):
        if k == 1:
            mb.destroyField(spr.recoverField(fb))
        for o in outs:
            o.fill_(-1.0)
        torch.cuda.synchronize()
        outs = batch.size_fields(fs, adapt_ratio=0.05, outputs=outs)
        assert all(torch.equal(o, r) for o, r in zip(outs, first)), k
    for m, f, r in zip(ms, fs, first):
        assert np.array_equal(spr.getSPRSizeField(f, 0.05).numpy()[:, 0], r.cpu().numpy())
    ctx = spr.context(0)
    batch.close()
    for m in ms + [mb]:
        m.close()
    _lib.check(_lib.lib().sprg_ctx_destroy(ctx))
