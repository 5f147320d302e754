"""The fits of the expansion queue's sets (csrc/k_fast.hip, k_fast_sets): by
eight lanes a set up to 65536 queued sets, by a thread a set above.

On an undistorted lattice most edge patches are queued (about seven for each
cube of the box), so n = 20 lies below the line and n = 22 above it.  The fast
form's sets have pivot ratios above 1e-6 or take the exact kernel, which
bounds the difference to the exact form by about 1e6 times some tens of
2^-53: 1e-8 of the field.
"""
import numpy as np
import pytest

from core_amd import mesh, spr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nc", [1, 3, 9, 27])
@pytest.mark.parametrize("n,order,jitter", [(2, 2, 0.0), (20, 2, 0.0), (22, 2, 0.0), (6, 2, 0.25), (5, 1, 0.2)])
def test_expanded_sets(gpu, n, order, jitter, nc):
    h = mesh.box(n, order=order, jitter=jitter, seed=9)
    m = spr.Mesh(h)
    x = h.ip_points(2)
    k = np.linspace(0.5, 2.5, 3 * nc).reshape(nc, 3)
    f = m.createIPField("f", nc, 2, np.sin(x @ k.T))
    r = spr.recoverField(f, form="fp64f")
    got = r.numpy()
    st = m.last_stats()
    m.destroyField(r)
    assert st["status"] == 0 and st["expanded"] == st["queued_exact"] > 0
    if n >= 20:
        assert (st["queued_exact"] > 65536) == (n == 22)
    ref = spr.recoverField(f, form="fp64").numpy()
    assert np.abs(got - ref).max() <= 1e-8 * np.abs(ref).max()
