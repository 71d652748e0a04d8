"""The two FP64 forms of the stage kernel on one mesh: rows a few cells longer than
a multiple of half a tile take more than 256 tiles in row pairs (the line kernel)
and about 210 in compact blocks (one wavefront per flux-point number), on a device
of 256 CUs.  Both integrators, every face type, with norms and the AV sensor:
states, maxima and sensor are equal bit for bit, the norms (summed per tile in
another order) to 1e-12, and the state, maxima and norms of each agree with the
oracle to the bars of test_gpu_parity."""
import numpy as np
import pytest

from oracle.oracle import Oracle
from sddc_amd import abi
from sddc_amd import mesh as M
from tests.util import per_var_error

pytestmark = pytest.mark.gpu

# row length, rows: ceil(R / H) * rows / 2 = 260 tiles, H = 10, 8, 6 cells a row
ROWS = {3: (31, 130), 4: (33, 104), 5: (19, 130)}


def _case(N, kind, k_stage):
    R, rows = ROWS[N]
    if kind == "channel":
        m = M.channel(R, rows, lx=2.0, ly=8.0, seed=5, free_left=rows // 3)
    elif kind == "ogrid":
        m = M.ogrid(rows, R, 0.5, 15.0)
    else:
        m = M.periodic_square(R, rows, 2.0, 8.0)
    p = M.RunParams(N=N, dt=4e-5 if kind == "ogrid" else 2e-4, k_stage=k_stage,
                    dxcycl=m.dxcycl, dycycl=m.dycycl)
    case = M.build_case(m, p)
    return case, M.smooth_perturbed_state(case, 0.05, seed=1)


def test_tile_counts():
    cells = {3: 20, 4: 16, 5: 12}
    for N, (R, rows) in ROWS.items():
        h = cells[N] // 2
        assert -(-R // h) * (rows // 2) == 260 and -(-R * rows // cells[N]) <= 256


@pytest.mark.parametrize("k_stage", [3, 5], ids=["RK_S5P3", "FiveStageRk"])
@pytest.mark.parametrize("kind", ["channel", "ogrid", "periodic"])
@pytest.mark.parametrize("N", [3, 4, 5])
def test_line_and_point_kernel(N, kind, k_stage):
    from sddc_amd.solver import Sd2d
    print(f"[stage kernels] N={N} {kind} k_stage={k_stage}", flush=True)
    case, Q0 = _case(N, kind, k_stage)
    o = Oracle(case)
    o.set_state(Q0, [0, 0, 0, 0])
    o.step(3, 2)
    Qo, mo = o.get_state()
    do = o.diag()
    res = []
    for shape in (abi.SD2D_TILE_ROWPAIRS, abi.SD2D_TILE_BLOCKS):
        g = Sd2d(case, tile_shape=shape)
        g.set_state(Q0, [0, 0, 0, 0])
        g.step(3, 2)             # norms on the first and third step, none on the second
        Q, mx = g.get_state()
        sm = g.get_av()[0]
        d = g.diag()
        g.close()
        res.append((Q, mx, sm, np.array([d["resid_rms"], d["divb_rms"]])))
        e = per_var_error(Q - Q0, Qo - Q0)[0]
        assert e.max() <= 1e-11, (shape, e)
        np.testing.assert_allclose(mx, mo, rtol=1e-13, atol=0)
        assert d["norms_valid"] == 1
        np.testing.assert_allclose(res[-1][3], [do["resid_rms"], do["divb_rms"]], rtol=1e-10)
    for a, b in zip(res[0][:3], res[1][:3]):
        assert np.array_equal(a, b, equal_nan=True)
    np.testing.assert_allclose(res[0][3], res[1][3], rtol=1e-12)
