"""The viscous kernels at the edges of their tiles: cell counts one below, at
and one above a tile and a pair of rows, every tile shape, walls at either
end of a line, both line families crossing tiles.  Against the oracle to
1e-12 per variable (the bar of the device's residual: the arithmetic is
double throughout, and sums of at most 2(N+1) products per point)."""
import numpy as np
import pytest

from sddc_amd import abi
from sddc_amd import mesh as M
from tests.util import per_var_error

pytestmark = pytest.mark.gpu

MESHES = [   # (N, mesh): tiles of 20, 16, 12 cells for N = 3, 4, 5
    (3, lambda: M.channel(19, 1, free_left=1)),
    (3, lambda: M.channel(10, 4, types=("WALL", "WALL", "INLE", "WALL"))),
    (4, lambda: M.channel(17, 3, seed=5)),
    (4, lambda: M.ogrid(3, 16, 0.5, 4.0)),
    (5, lambda: M.channel(1, 1, types=("WALL", "OUTL", "WALL", "INLE"))),
    (5, lambda: M.periodic_square(13, 3, 1.3, 0.3)),
    (5, lambda: M.ogrid(2, 25, 2.0, 3.0)),
]


@pytest.mark.parametrize("shape", [abi.SD2D_TILE_STRIPS, abi.SD2D_TILE_BLOCKS,
                                   abi.SD2D_TILE_ROWPAIRS])
@pytest.mark.parametrize("k", range(len(MESHES)))
def test_viscous_residual_at_tile_edges(k, shape):
    from oracle.oracle import Oracle
    from sddc_amd.solver import Sd2d
    N, mk = MESHES[k]
    m = mk()
    case = M.build_case(m, M.RunParams(N=N, dt=1e-3, mu=0.01, eta0=0.02, dxcycl=m.dxcycl,
                                       dycycl=m.dycycl))
    print(f"[gpu-viscous-tiles] {m.name} N={N} shape={shape}", flush=True)
    Q0 = M.smooth_perturbed_state(case, 0.05, seed=4)
    g, o = Sd2d(case, tile_shape=shape), Oracle(case)
    for s in (g, o):
        s.set_state(Q0, [0, 0, 0, 0])
    rg, ng = g.compresid()
    ro, no = o.compresid()
    assert per_var_error(rg, ro)[0].max() <= 1e-12
    assert per_var_error(ng.reshape(18, -1, order="F"), no.reshape(18, -1, order="F"))[0].max() <= 1e-12
    g.step(1)
    o.step(1)
    assert np.isfinite(g.get_state()[0]).all()
    assert per_var_error(g.get_state()[0] - Q0, o.get_state()[0] - Q0)[0].max() <= 1e-11
