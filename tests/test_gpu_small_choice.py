"""Small D2Q9 domains at the steps per launch and tile side chosen for them (10 steps on the smallest,
4 and fewer on the largest) against one launch per step: populations bit for bit, forces to the
summation order of FP64 partials (1e-12 of the largest: at most 2^18 terms' rounding, 2^-53 each)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["fp64", "fp32", "bf16s"])
@pytest.mark.parametrize("nx,ny,fi", [(7, 3, 1), (48, 32, 1), (301, 79, 10), (511, 131, 1), (700, 180, 3), (1000, 250, 1)])
def test_chosen_depth_equals_one_launch_per_step(pkg, monkeypatch, prec, nx, ny, fi):
    L = pkg.lbm
    got = []
    for tb in ("0", "1"):
        monkeypatch.setenv("LBM_TEMPORAL_BLOCKING", tb)
        cfg = L.make_config(9, nx, ny, 1, tau0=0.06, u0=0.05, precision=L.PRECISIONS[prec], body=L.BODY_ZCYL,
                            center=(nx / 4, ny / 2 - 0.5, 0), r2=(ny / 8) ** 2, perturb=1e-2, force_interval=fi)
        with L.Solver(cfg) as s:
            s.initialize().step(27)
            s.step(4)
            got.append((s.populations(), s.forces()))
    (a, fa), (b, fb) = got
    assert np.array_equal(a, b)
    assert fa.shape == fb.shape and np.array_equal(fa[:, 0], fb[:, 0])
    assert np.abs(fa - fb).max(initial=0) <= 1e-12 * max(np.abs(fa[:, 1:]).max(initial=0), 1.0)
