"""The exact fits' shared workspace on the CPU emulation of the library
(tests/emu/build.py): two host threads on one context, and a device that
grants only part of what is asked for.  The meshes are P1 stars, whose centre
vertex has more than 32 rows, so that its fit takes the three-launch path
through the workspace; "large" takes a star beyond the exact kernels' rows.  Started by tests/test_emu_workspace.py in a child
process with AddressSanitizer preloaded, with one check's name."""
import ctypes
import os
import sys
import threading

import numpy as np

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(os.path.dirname(HERE))
sys.path.insert(0, ROOT)
from core_amd import _lib  # noqa: E402

_lib.LIB_PATH = os.path.join(HERE, "_build", "libsprgpu_emu.so")
from core_amd import mesh, workloads  # noqa: E402
from oracle import oracle as O  # noqa: E402

sys.path.insert(0, os.path.dirname(HERE))
import smb_util  # noqa: E402

L = _lib.lib()
vp = ctypes.c_void_p
SHAPE = (ctypes.c_int64 * 5)(64, 24, 16, 8, 12)  # small persistent grids: the emulator walks every block


def P(a):
    return vp(a.ctypes.data)


def check(name, ok):
    print(("PASS " if ok else "FAIL ") + name, flush=True)
    if not ok:
        sys.exit(1)


class Stars:
    """k disjoint stars of `tets` tets each, as one order-1 mesh."""

    def __init__(self, ctx, k, tets, seed):
        tv, xyz = smb_util.star(tets // 2 + 2)
        n = xyz.shape[0]
        self.h = mesh.HostMesh(np.vstack([tv + i * n for i in range(k)]),
                               np.vstack([xyz * (1 + 0.1 * i) + [3.0 * i, 0, 0] for i in range(k)]), 1)
        h = self.h
        self.m = vp()
        _lib.check(L.sprg_mesh_create(ctx, h.nv, h.nt, 0, P(h.tv), None, P(h.xyz), 1, ctypes.byref(self.m)))
        _lib.check(L.sprg_mesh_set_shape(self.m, SHAPE, 5))
        self.ip = np.ascontiguousarray(np.random.default_rng(seed).standard_normal((h.nt, 1, 3)))
        self.om = O.Mesh(h.tv, h.xyz, 1)
        self.ref = O.recover(self.om, self.ip)

    def recover(self):
        out = np.full((self.h.nv, 3), np.nan)
        _lib.check(L.sprg_recover(self.m, 1, 3, P(self.ip), P(out), 0))
        return out

    def size(self, form=0):
        s = np.full(self.h.nv, np.nan)
        diag = np.zeros(4)
        _lib.check(L.sprg_spr_size(self.m, 1, 3, P(self.ip), 0.1, P(s), form, P(diag)))
        return s

    def close(self):
        L.sprg_mesh_destroy(self.m)


def threads(ctx):
    # one context, two threads, a mesh each: their launches alternate.  The
    # larger sets of the second mesh also make it replace the buffer.
    a, b = Stars(ctx, 1, 40, 1), Stars(ctx, 2, 90, 2)
    got = [[], []]

    def work(i, s):
        for _ in range(3):
            got[i].append((s.recover(), s.size()))

    ts = [threading.Thread(target=work, args=(i, s)) for i, s in enumerate((a, b))]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for i, s in enumerate((a, b)):
        size = s.size()  # alone
        check("mesh %d: three calls beside another thread's" % i,
              len(got[i]) == 3 and all(np.array_equal(r, s.ref) and np.array_equal(z, size) for r, z in got[i]))
    a.close()
    b.close()


def limit(nbytes):
    L.emu_malloc_limit(ctypes.c_size_t(nbytes))


FREE = 2**64 - 1


def refused(ctx):
    # four sets of 40 rows: 4,224 bytes of workspace each (the reflectors, R's
    # top and Q of a 4-term fit of up to 64 rows)
    one = 8 * (4 * 64 + 16 + 64 * 4)
    s = Stars(ctx, 4, 40, 3)
    s.size(form=2)  # everything but the exact fits' workspace is there now
    limit(2 * one)
    check("half of the workspace granted", np.array_equal(s.recover(), s.ref))
    limit(0)
    for k in range(2):
        check("nothing granted beside it, call %d" % k, np.array_equal(s.recover(), s.ref))
    limit(FREE)
    check("all granted again", np.array_equal(s.recover(), s.ref))
    # a set that the buffer at hand does not hold, on a device without room
    big = Stars(ctx, 1, 180, 4)
    big.size(form=2)
    limit(0)
    out = np.zeros((big.h.nv, 3))
    check("no room for one set: refused",
          L.sprg_recover(big.m, 1, 3, P(big.ip), P(out), 0) == _lib.SPRG_ENOMEM)
    limit(FREE)
    check("granted once there is room", np.array_equal(big.recover(), big.ref))
    check("and the smaller sets still fit", np.array_equal(s.recover(), s.ref))
    big.close()
    # batches: recorded once, then replayed, with part of the workspace, and
    # recorded again where an eager call has moved the context's
    parts = [Stars(ctx, 4, 40 + 2 * i, 5 + i) for i in range(5)]
    want = [p.size() for p in parts]
    fresh = vp()
    _lib.check(L.sprg_ctx_create(0, ctypes.byref(fresh)))
    for p in parts:
        p.close()
    parts = [Stars(fresh, 4, 40 + 2 * i, 5 + i) for i in range(5)]
    for p in parts:
        p.size(form=2)
    arr = (vp * 5)(*[p.m.value for p in parts])
    b = vp()
    _lib.check(L.sprg_batch_create(fresh, 5, arr, ctypes.byref(b)))
    outs = [np.zeros(p.h.nv) for p in parts]
    ips = (vp * 5)(*[p.ip.ctypes.data for p in parts])
    ops = (vp * 5)(*[o.ctypes.data for o in outs])
    t = np.zeros(1)
    limit(2 * one)
    graphs = []
    for k in range(4):
        for o in outs:
            o[:] = -1.0
        if k == 3:
            limit(FREE)
            Stars(fresh, 1, 40, 9).close()  # memory came back: the next call may ask for more
            check("mesh 0 alone", np.array_equal(parts[0].recover(), parts[0].ref))
        _lib.check(L.sprg_batch_size(b, 1, 3, ips, None, 0.1, 0.25, 2.0, ops, 0, P(t)))
        graphs.append(L.emu_graph_count())
        check("batch run %d equals the per-mesh calls" % k, all(np.array_equal(o, w) for o, w in zip(outs, want)))
    check("later runs replay: graphs recorded %s" % graphs, graphs[0] == graphs[1] == graphs[2])
    check("recorded again where the context's workspace moved", graphs[3] > graphs[2])
    L.sprg_batch_destroy(b)
    for p in parts + [s]:
        p.close()
    _lib.check(L.sprg_ctx_destroy(fresh))


def large(ctx):
    # a vertex of 136 tets at four points per tet, 544 rows: more than the exact
    # kernels take, so the exact form refuses it and the fast forms solve it
    # where its rank is certain and refuse it where it is not
    tv, xyz = smb_util.star(70)
    for skew, certain in ((1.0, True), (1e-4, False)):
        x = xyz.copy()
        x[:, 2] = x[:, 0] + skew * x[:, 2]  # pivot ratio about the skew squared
        h = mesh.HostMesh(tv, x, 1)
        om = O.Mesh(h.tv, h.xyz, 1)
        m = vp()
        _lib.check(L.sprg_mesh_create(ctx, h.nv, h.nt, 0, P(h.tv), None, P(h.xyz), 1, ctypes.byref(m)))
        _lib.check(L.sprg_mesh_set_shape(m, SHAPE, 5))
        ip = np.ascontiguousarray(workloads.strain_field(h.ip_points(2)))
        ref = O.recover(om, ip)
        for form in (0, 1, 2):
            out = np.full((h.nv, 9), np.nan)
            rc = L.sprg_recover(m, 2, 9, P(ip), P(out), form)
            st = np.zeros(7, np.int64)
            L.sprg_mesh_last_stats(m, P(st), 7)
            if form == 0 or not certain:
                check("544 rows, skew %g, form %d: refused" % (skew, form), rc == _lib.SPRG_EUNSUPPORTED)
            else:
                ok = rc == 0 and np.abs(out - ref).max() <= 1e-9 * np.abs(ref).max()
                check("544 rows, skew %g, form %d: solved, settled" % (skew, form), ok and st[3] == 0)
        L.sprg_mesh_destroy(m)


CHECKS = {"threads": threads, "refused": refused, "large": large}

if __name__ == "__main__":
    ctx = vp()
    _lib.check(L.sprg_ctx_create(0, ctypes.byref(ctx)))
    CHECKS[sys.argv[1]](ctx)
    _lib.check(L.sprg_ctx_destroy(ctx))
    print("ALL PASS", flush=True)
