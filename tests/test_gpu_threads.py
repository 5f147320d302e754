"""Exact-form calls of two threads on two meshes of one context, which share
the workspace of the exact fits: each call's result equals the same call
alone, bit for bit.  The second mesh has sets of more rows and more of them,
so the first calls also replace the buffer."""
import threading

import numpy as np
import pytest
import torch

from core_amd import mesh, spr, workloads

pytestmark = pytest.mark.gpu


def test_two_threads_one_context(gpu):
    hosts = [mesh.box(n, order=2, jitter=j, seed=workloads.C5) for n, j in ((6, 0.2), (12, 0.25))]
    ms = [spr.Mesh(h) for h in hosts]
    fs = [m.createIPField("eps", 9, 2, workloads.strain_field(h.ip_points(2))) for m, h in zip(ms, hosts)]
    got, errors = [[], []], []

    def both(i):
        out = []
        for call in (spr.recoverField, lambda f: spr.getSPRSizeField(f, 0.05)):
            r = call(fs[i])
            out.append(r.numpy())
            ms[i].destroyField(r)
        return out

    def work(i):
        try:
            for _ in range(20):
                got[i].append(both(i))
        except Exception as e:
            errors.append(e)

    torch.cuda.synchronize()
    ts = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not errors
    for i in range(2):
        r, s = both(i)
        assert len(got[i]) == 20
        assert all(np.array_equal(a, r) and np.array_equal(b, s) for a, b in got[i])
        ms[i].close()
