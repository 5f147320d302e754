"""The exact fits' shared workspace on the CPU emulation of the library
(tests/emu/build.py): two host threads on one context, and a device that
grants only part of what is asked for.  The meshes are P1 stars, whose centre
vertex has more than 32 rows, so that its fit takes the three-launch path
through the workspace.  Started by tests/test_emu_workspace.py in a child
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

    def size(self):
        s = np.full(self.h.nv, np.nan)
        diag = np.zeros(4)
        _lib.check(L.sprg_spr_size(self.m, 1, 3, P(self.ip), 0.1, P(s), 0, P(diag)))
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


CHECKS = {"threads": threads}

if __name__ == "__main__":
    ctx = vp()
    _lib.check(L.sprg_ctx_create(0, ctypes.byref(ctx)))
    CHECKS[sys.argv[1]](ctx)
    _lib.check(L.sprg_ctx_destroy(ctx))
    print("ALL PASS", flush=True)
