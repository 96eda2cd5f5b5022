"""Two D3Q27 steps per pass (pair_kernel.hpp) against one step per launch: populations and fields bit
for bit, forces included.  Sizes at the edges of the columns (64 x 8, FP64 32 x 13)
and of the runs of planes, walls, periodic axes, inlet and outlet columns with mask links, solid
fraction; odd step counts and force intervals, so that both paths mix within a run."""
import numpy as np
import pytest

gpu = pytest.mark.gpu

CASES = {
    "smaller_than_a_column": dict(n=(20, 12, 9), fi=5),
    "smallest": dict(n=(3, 3, 3), body=False),
    "smallest_periodic": dict(n=(3, 3, 3), per=(1, 1, 1), body=False),
    "ragged": dict(n=(70, 11, 10), per=(0, 1, 1), fi=2),
    "one_column_periodic_x": dict(n=(64, 8, 8), per=(1, 0, 0), fi=3),
    "one_more_than_a_column": dict(n=(65, 9, 40), per=(1, 1, 1)),
    "fp64_column_edges": dict(n=(33, 14, 7), fi=1),
    "solid_fraction": dict(n=(129, 28, 13), body=False, sfrac=True, fi=4),
    "noise_mask": dict(n=(67, 20, 11), noise=0.08, fi=3, inlet=1),
    "noise_mask_periodic": dict(n=(67, 20, 11), noise=0.08, per=(1, 1, 1), fi=3),
    "sphere": dict(n=(130, 37, 70), fi=10),
}


def run(L, prec, n, per=(0, 0, 0), body=True, noise=0.0, sfrac=False, fi=0, inlet=0):
    nx, ny, nz = n
    rng = np.random.default_rng(7)
    kind = L.BODY_MASK if noise else L.BODY_SPHERE if body else L.BODY_NONE
    cfg = L.make_config(27, nx, ny, nz, tau0=0.06, u0=0.05, precision=prec, periodic=per, body=kind, inlet=inlet,
                        center=(nx * 0.3, (ny - 1) / 2, (nz - 1) / 2), r2=(min(nx // 2, ny, nz) * 0.18) ** 2,
                        perturb=1e-2, force_interval=fi)
    with L.Solver(cfg) as s:
        if noise:
            s.set_mask(rng.random((nz, ny, nx)) < noise)
        if sfrac:
            s.set_solid_fraction(np.clip(0.3 * rng.standard_normal((nz, ny, nx)), 0, 1))
        s.set_perturbation(rng.random((nz, ny, nx)) * 2 - 1)
        s.initialize()
        out = []
        for steps in (7, 6, 1, 4):
            s.step(steps)
            out += [*s.fields(), s.populations()]
        return out, s.forces()


@gpu
@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("prec", ["fp64", "fp32", "fp16s", "bf16s"])
def test_two_steps_per_pass_equal_one(pkg, monkeypatch, prec, case):
    L = pkg.lbm
    monkeypatch.setenv("LBM_TWO_STEPS", "0")
    a, fa = run(L, L.PRECISIONS[prec], **CASES[case])
    monkeypatch.setenv("LBM_TWO_STEPS", "1")
    b, fb = run(L, L.PRECISIONS[prec], **CASES[case])
    for x, y in zip(a, b):
        assert np.array_equal(x, y)
    assert np.array_equal(fa, fb)
