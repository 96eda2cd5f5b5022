"""Several D2Q9 steps per launch (k_tb2d) in every storage format and with a solid fraction, against
one launch per step: populations and fields bit for bit, forces to their summation order (per
tile).  A mask touching the inlet, the outlet and the walls, several tiles with ragged edges, and a
domain smaller than a tile's core; step counts that leave remainders of the launches."""
import numpy as np
import pytest

gpu = pytest.mark.gpu


@gpu
@pytest.mark.parametrize("n", [(101, 43), (30, 9)])
@pytest.mark.parametrize("sfrac", [False, True])
@pytest.mark.parametrize("prec", ["fp64", "fp32", "fp16s", "bf16s"])
def test_small_steps_equal_one_launch_per_step(pkg, monkeypatch, prec, sfrac, n):
    L = pkg.lbm
    nx, ny = n
    mask = np.zeros((1, ny, nx), np.uint8)
    mask[0, ny // 2, 1] = mask[0, 0, nx // 2] = mask[0, ny - 1, nx - 1] = 1
    mask[0, 3:6, nx - 1] = mask[0, 2:4, 0] = 1
    mask[0, ny // 2 - 1:ny // 2 + 2, nx // 3:nx // 3 + 3] = 1
    sf = np.clip(0.3 * np.random.default_rng(5).standard_normal((1, ny, nx)), 0, 1) * (1 - mask)
    cfg = L.make_config(9, nx, ny, 1, tau0=0.06, u0=0.05, precision=L.PRECISIONS[prec], body=L.BODY_MASK, perturb=1e-2,
                        force_interval=3)
    out = []
    for tb in ("0", "1"):
        monkeypatch.setenv("LBM_TEMPORAL_BLOCKING", tb)
        with L.Solver(cfg) as s:
            s.set_mask(mask)
            if sfrac:
                s.set_solid_fraction(sf)
            s.initialize()
            res = []
            for steps in (1, 2, 7, 23):
                s.step(steps)
                res += [s.populations(), *s.fields()]
            out.append((res, s.forces()))
    (ra, fa), (rb, fb) = out
    for x, y in zip(ra, rb):
        assert np.array_equal(x, y)
    assert fa.shape == fb.shape == (11, 4) and np.array_equal(fa[:, 0], fb[:, 0])
    assert np.abs(fa - fb).max() <= 1e-12 * np.abs(fa[:, 1:]).max()
