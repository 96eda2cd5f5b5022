"""The reference's 2D step in one launch (k_ref_one) against the oracle's kernel sequence, at the sizes
where its source table can go wrong: the smallest box, bodies next to the inlet, the outlet and the
walls, a body spanning the channel, no body; one call per step and several, and the staged calls in
between.  Bounds of the FP64 parity tests: 1e-13 on fields and populations, 1e-11 on forces."""
import numpy as np
import pytest

gpu = pytest.mark.gpu

CASES = {
    "smallest": (3, 3, None),
    "no_body": (20, 9, None),
    "disk": (131, 37, (40.0, 18.0, 25.0)),
    "at_inlet": (40, 21, (0.0, 10.0, 9.0)),
    "at_outlet": (40, 21, (39.0, 8.0, 9.0)),
    "at_wall": (50, 16, (20.0, 0.0, 5.0)),
    "corner": (30, 12, (29.0, 11.0, 6.0)),
    "across": (64, 9, (30.0, 4.0, 49.0)),
}


def rel(a, b):
    n = np.linalg.norm(np.ravel(b))
    return np.linalg.norm(np.ravel(a) - np.ravel(b)) / (n if n > 0 else 1.0)


@gpu
@pytest.mark.parametrize("case", CASES)
def test_one_launch_reference_step(pkg, orc, case):
    L = pkg.lbm
    nx, ny, body = CASES[case]
    kw = dict(tau0=0.06, u0=0.05, force_interval=1)
    if body:
        kw.update(body=L.BODY_SPHERE, center=(body[0], body[1], 0.0), r2=body[2])
    ran = np.random.default_rng(11).integers(0, 100, (ny + 4, nx + 4), dtype=np.int32)
    o = orc.RefState(orc.make_cfg(9, nx, ny, **kw), ran=ran)
    with L.Solver(L.make_config(9, nx, ny, bc_mode=L.BC_REFERENCE, **kw)) as s:
        s.set_ran(ran)
        s.initialize()
        s.step(1)
        s.step(4)
        for stage in (s.collide, s.boundary, s.stream, s.update):
            stage()
        s.step(3)
        o.step(9)
        assert rel(s.populations(), o.populations()) <= 1e-13
        for a, b in zip(s.fields(), o.fields()):
            assert rel(a, b) <= 1e-13
        f, g = s.forces(), o.forces()
        assert f.shape == g.shape == (9, 4) and np.array_equal(f[:, 0], g[:, 0])
        assert np.abs(f - g).max() <= 1e-11 * max(np.abs(g[:, 1:]).max(), 1e-300)
