"""The reverse sweep of one residual at the edges of its tiles (cell counts
one below, at and one above a tile and a row pair, every tile shape, every
boundary type at either end of a line, a neighbour that is the cell itself),
against central differences of the oracle's residual along random
directions.  Bar 1e-7: a central difference of step h = 1e-5 of an O(1)
smooth function is off by about h^2 = 1e-10 and eps/h = 2e-11 of its scale."""
import numpy as np
import pytest

from sddc_amd import abi
from sddc_amd import mesh as M

pytestmark = pytest.mark.gpu

MESHES = [   # (N, mesh): tiles of 20, 16, 12 cells for N = 3, 4, 5
    (3, lambda: M.channel(19, 1, free_left=1)),
    (3, lambda: M.channel(10, 4, types=("WALL", "SYMP", "INLE", "WALL"))),
    (4, lambda: M.channel(17, 3, seed=5)),
    (4, lambda: M.periodic_square(1, 3, 0.1, 0.3)),
    (5, lambda: M.channel(1, 1, types=("SYMP", "OUTL", "WALL", "INLE"))),
    (5, lambda: M.periodic_square(13, 3, 1.3, 0.3)),
]


@pytest.mark.parametrize("shape", [abi.SD2D_TILE_STRIPS, abi.SD2D_TILE_BLOCKS,
                                   abi.SD2D_TILE_ROWPAIRS])
@pytest.mark.parametrize("k", range(len(MESHES)))
def test_residual_pullback_at_tile_edges(k, shape):
    from oracle.oracle import Oracle
    from sddc_amd.solver import Sd2d
    N, mk = MESHES[k]
    m = mk()
    case = M.build_case(m, M.RunParams(N=N, dt=1e-3, dxcycl=m.dxcycl, dycycl=m.dycycl))
    print(f"[gpu-adjoint-tiles] {m.name} N={N} shape={shape}", flush=True)
    Q = M.smooth_perturbed_state(case, 0.05, seed=4)
    mx = [2.5, 1.4, 2.5, 1.4]
    rng = np.random.default_rng(k)
    rb = np.asfortranarray(rng.standard_normal(Q.shape))
    V = rng.standard_normal(Q.shape)
    g, o = Sd2d(case, tile_shape=shape), Oracle(case)
    g.set_state(Q, mx)
    qb, _, _ = g.compresid_vjp(rb)

    def value(h):
        o.set_state(np.asfortranarray(Q + h * V), mx)
        return float((o.compresid()[0] * rb).sum())

    h = 1e-5
    fd = (value(h) - value(-h)) / (2 * h)
    scale = np.linalg.norm(qb) * np.linalg.norm(V)
    assert abs(float((qb * V).sum()) - fd) <= 1e-7 * scale
