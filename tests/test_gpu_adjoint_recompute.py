"""The adjoint's recomputed states from the multi-step kernels (the state of every step stored) against
one launch per step: dJ/ds and dJ/du_in bit for bit, with a mask, a solid fraction and periodic
axes (one launch per step either way), at segment lengths that leave several remainders of the 7 steps
per launch.  J, summed over tiles instead of row blocks in the forward run, to 1e-12."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = {
    "tiles": (9, (61, 33, 1), (0, 0, 0), 23),
    "tiles_mask": (9, (40, 21, 1), (0, 0, 0), 9),
    "mask_touching": (9, (130, 18, 1), (0, 0, 0), 31),
    "periodic": (9, (45, 20, 1), (0, 1, 0), 8),
}


def run(L, prec, Q, n, per, K, mask):
    nx, ny, nz = n
    rng = np.random.default_rng(7)
    m = np.zeros((nz, ny, nx), np.uint8)
    if mask:
        m[:, ny // 2 - 1:ny // 2 + 2, nx // 3:nx // 3 + 3] = 1
        m[0, 0, nx // 2] = m[-1, -1, -1] = 1
    cfg = L.make_config(Q, nx, ny, nz, tau0=0.06, u0=0.05, precision=prec, body=L.BODY_MASK, perturb=1e-2, periodic=per)
    with L.Solver(cfg) as s:
        s.set_mask(m)
        s.set_solid_fraction(np.clip(0.3 * rng.standard_normal((nz, ny, nx)), 0, 1) * (1 - m))
        s.set_perturbation(rng.random((nz, ny, nx)) * 2 - 1)
        s.initialize()
        return s.adjoint(5, 31, 1.0, K)[:3]


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_recompute_equals_one_launch_per_step(pkg, monkeypatch, prec, case):
    L = pkg.lbm
    Q, n, per, K = CASES[case]
    a = run(L, L.PRECISIONS[prec], Q, n, per, K, "mask" in case)
    monkeypatch.setenv("LBM_TEMPORAL_BLOCKING", "0")
    b = run(L, L.PRECISIONS[prec], Q, n, per, K, "mask" in case)
    assert abs(a[0] - b[0]) <= 1e-12 * abs(b[0])
    assert np.array_equal(a[1], b[1]) and np.array_equal(a[2], b[2])
