"""The batched rank test of the fast forms' uncertified initial sets
(csrc/k_qr.hip, k_rank_test).

On an unjittered lattice most edge patches' samples do not determine a
quadratic: the fast forms queue them, the rank test runs the reference's
recurrence on them, and the ones it rejects grow.  The patch sets are the
reference's, so the fast form's recovered field must follow the exact form's
(itself bit-identical to the oracle) to rounding, and every queued patch must
end with a set.  At one point per tet some square 10x10 sets pass the test
and keep their initial sets.
"""
import numpy as np
import pytest

from core_amd import mesh, spr
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form", ["fp64f", "fp32r"])
@pytest.mark.parametrize("n,jitter,ip_order", [(2, 0.0, 2), (5, 0.0, 2), (7, 0.0, 2), (3, 0.25, 1), (6, 0.2, 1),
                                               (5, 0.0, 1)])
def test_sets_and_values(gpu, n, jitter, ip_order, form):
    h = mesh.box(n, order=2, jitter=jitter, seed=7)
    om = O.Mesh(h.tv, h.xyz, 2, te=h.te, ev=h.ev)
    m = spr.Mesh(h)
    x = h.ip_points(ip_order)
    ip = np.stack([np.sin(3 * x[..., 0] + x[..., 1]), x[..., 1] * x[..., 2], np.cos(2 * x[..., 2])], -1)
    f = m.createIPField("f", 3, ip_order, ip)
    r = spr.recoverField(f, form=form)
    got = r.numpy()
    st = m.last_stats()
    m.destroyField(r)
    assert st["status"] == 0 and st["expanded"] == st["queued_exact"]
    if jitter == 0 and ip_order == 2 and n > 2:
        assert st["exact_tested"] > h.ne // 2
    ref = O.recover(om, ip)
    assert np.array_equal(spr.recoverField(f, form="fp64").numpy(), ref)
    assert np.isfinite(got).all()
    if ip_order == 2:
        # 1e-9 of the component scale: the bar of the fast forms' other tests
        # (square sets at one point per tet may be fitted with pivots down to
        # 1e-6 of their diagonals, so there the bar would measure the form's
        # conditioning and not the sets)
        assert np.max(np.abs(got - ref) / np.abs(ref).max(0)) <= 1e-9
    else:
        assert st["exact_tested"] > 0
    m.close()
