"""Several D2Q9 steps per pass on large domains (k_strip) against one launch per step, in every
storage format: populations and fields bit for bit, forces to their summation order (per wave).
Widths around the 58, 60 and 62 stored columns of a wave (4, 3 and 2 steps), domains smaller than a
wave or than the rows a run recomputes, walls, periodic axes, a mask touching inlet, outlet and
walls, a solid fraction; step counts that leave every remainder, force records in each of the
launch's steps."""
import numpy as np
import pytest

gpu = pytest.mark.gpu

CASES = {
    "walls": dict(n=(117, 43)),
    "one_strip": dict(n=(58, 21)),
    "one_column_more": dict(n=(59, 9), fi=2),
    "tiny": dict(n=(5, 3), mask=False),
    "tiny_periodic": dict(n=(5, 3), per=(1, 1), mask=False),
    "periodic_y": dict(n=(130, 37), per=(0, 1), fi=1),
    "periodic_x": dict(n=(61, 37), per=(1, 0), fi=4),
    "periodic": dict(n=(201, 70), per=(1, 1), fi=3),
    "solid_fraction": dict(n=(131, 50), sfrac=True, fi=3),
    "tall": dict(n=(70, 900), fi=5),
}


def run(L, prec, n, per=(0, 0), mask=True, sfrac=False, fi=3):
    nx, ny = n
    rng = np.random.default_rng(3)
    m = np.zeros((1, ny, nx), np.uint8)
    if mask:
        m[0, ny // 2, 1] = m[0, 0, nx // 2] = m[0, ny - 1, nx - 1] = 1
        m[0, 3:6, nx - 1] = m[0, 2:4, 0] = 1
        m[0, ny // 2 - 1:ny // 2 + 2, nx // 3:nx // 3 + 3] = 1
    cfg = L.make_config(9, nx, ny, 1, tau0=0.06, u0=0.05, precision=prec, body=L.BODY_MASK, perturb=1e-2, force_interval=fi,
                        periodic=(*per, 0))
    with L.Solver(cfg) as s:
        s.set_mask(m)
        if sfrac:
            s.set_solid_fraction(np.clip(0.3 * rng.standard_normal((1, ny, nx)), 0, 1) * (1 - m))
        s.set_perturbation(rng.random((1, ny, nx)) * 2 - 1)
        s.initialize()
        out = []
        for steps in (1, 3, 4, 5, 6, 19):
            s.step(steps)
            out += [s.populations(), *s.fields()]
        return out, s.forces()


@gpu
@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("prec", ["fp64", "fp32", "fp16s", "bf16s"])
def test_strips_equal_one_launch_per_step(pkg, monkeypatch, prec, case):
    L = pkg.lbm
    monkeypatch.setenv("LBM_TEMPORAL_BLOCKING", "0")
    a, fa = run(L, L.PRECISIONS[prec], **CASES[case])
    monkeypatch.setenv("LBM_TEMPORAL_BLOCKING", "2")
    b, fb = run(L, L.PRECISIONS[prec], **CASES[case])
    for x, y in zip(a, b):
        assert np.array_equal(x, y)
    assert fa.shape == fb.shape and np.array_equal(fa[:, 0], fb[:, 0])
    assert np.abs(fa - fb).max() <= 1e-12 * max(np.abs(fa[:, 1:]).max(), 1e-300)
