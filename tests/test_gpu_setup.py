"""The device classification of the nodes: the counts of solid nodes and of fluid nodes with a solid
neighbour against a host count, at row lengths around the launch's block of 256 nodes, with the mask on
every edge and corner (so that periodic axes wrap into it) and with the body formulas."""
import itertools

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def counts(solid, periodic):
    """solid: (nz, ny, nx) bool; fluid nodes with a solid neighbour among the 26 (8 in 2D)"""
    near = np.zeros_like(solid)
    per = periodic[::-1]
    pad = [(0, 0) if solid.shape[a] == 1 and a == 0 else (1, 1) for a in range(3)]
    p = np.zeros([n + a + b for n, (a, b) in zip(solid.shape, pad)], bool)
    idx = [np.arange(-a, n + b) for n, (a, b) in zip(solid.shape, pad)]
    inside = [(i >= 0) & (i < n) | bool(w) for i, n, w in zip(idx, solid.shape, per)]
    p[:] = solid[np.ix_(*[i % n for i, n in zip(idx, solid.shape)])]
    p &= inside[0][:, None, None] & inside[1][None, :, None] & inside[2][None, None, :]
    for d in itertools.product(*[range(-a, b + 1) for a, b in pad]):
        if any(d):
            near |= p[tuple(slice(a + k, a + k + n) for k, (a, _), n in zip(d, pad, solid.shape))]
    return int(solid.sum()), int((near & ~solid).sum())


@pytest.mark.parametrize("precision", ["fp64", "fp32", "fp16s"])
@pytest.mark.parametrize("Q,nx,ny,nz,periodic", [
    (9, 255, 7, 1, (0, 0, 0)), (9, 256, 5, 1, (0, 1, 0)), (9, 257, 6, 1, (1, 1, 0)), (9, 513, 4, 1, (1, 0, 0)),
    (27, 31, 7, 5, (0, 0, 0)), (27, 64, 5, 6, (0, 1, 1)), (27, 257, 6, 4, (1, 1, 1)), (27, 33, 4, 5, (1, 0, 0)),
])
def test_node_counts(pkg, Q, nx, ny, nz, periodic, precision):
    lbm = pkg.lbm
    rng = np.random.default_rng(nx + ny)
    solid = rng.random((nz, ny, nx)) < 0.05
    solid[0, 0, 0] = solid[-1, -1, -1] = solid[-1, 0, nx // 2] = True
    cfg = lbm.make_config(Q, nx, ny, nz, tau0=0.1, u0=0.03, precision=lbm.PRECISIONS[precision], periodic=periodic,
                          body=lbm.BODY_MASK)
    with lbm.Solver(cfg) as s:
        s.set_mask(solid)
        info = s.initialize().info()
    assert (info.solid_nodes, info.boundary_nodes) == counts(solid, periodic)


@pytest.mark.parametrize("body", ["sphere", "zcyl"])
@pytest.mark.parametrize("Q", [9, 27])
def test_body_counts(pkg, Q, body):
    lbm = pkg.lbm
    nx, ny, nz = 70, 24, 24 if Q == 27 else 1
    c, r2 = (20.3, 11.5, 12.25), 5.7 ** 2
    cfg = lbm.make_config(Q, nx, ny, nz, tau0=0.1, u0=0.03, body=lbm.BODY_SPHERE if body == "sphere" else lbm.BODY_ZCYL,
                          center=c, r2=r2)
    z, y, x = np.meshgrid(np.arange(nz), np.arange(ny), np.arange(nx), indexing="ij")
    r = (x - c[0]) ** 2 + (y - c[1]) ** 2
    if Q == 27 and body == "sphere":
        r = r + (z - c[2]) ** 2
    with lbm.Solver(cfg) as s:
        info = s.initialize().info()
    assert (info.solid_nodes, info.boundary_nodes) == counts(r <= r2, (0, 0, 0))
