"""The stage kernel that the groups of an ensemble take (one kernel for at most a
tile per CU where the groups leave the chip to each other, else the line kernel):
groups of one, two and three orders on both sides of that rule, and rebuilt by the
tile-shape trial, equal the runs made alone bit for bit."""
import numpy as np
import pytest

from sddc_amd import mesh as M

pytestmark = pytest.mark.gpu

CELLS = {3: 20, 4: 16, 5: 12}          # cells of a tile


def _case(N, tiles, kind):
    """About `tiles` tiles of order N: a channel (every face type) or an O-grid."""
    n = tiles * CELLS[N]
    if kind == "channel":
        ny = max(4, int(np.sqrt(n / 2)))
        m = M.channel(max(4, n // ny), ny, seed=3, free_left=2)
    else:
        m = M.ogrid(max(4, n // 96), 96, 0.5, 6.0)
    return M.build_case(m, M.RunParams(N=N, dt=2e-4, dxcycl=m.dxcycl, dycycl=m.dycycl))


@pytest.mark.parametrize("tiles", [{4: 250}, {3: 120, 4: 120, 5: 120}, {4: 250, 5: 250},
                                   {3: 250, 4: 250, 5: 250}, {3: 100, 4: 640}, {3: 190, 4: 640, 5: 190}],
                         ids=lambda t: "+".join(f"N{n}x{k}" for n, k in t.items()))
def test_members_equal_runs_alone(tiles):
    from sddc_amd.solver import Sd2d, Sd2dEnsemble
    print(f"[ensemble kernels] {tiles}", flush=True)
    cases = []
    for N, t in tiles.items():           # two members a group, of unlike sizes and kinds
        cases += [_case(N, 2 * t // 3, "channel"), _case(N, t - 2 * t // 3, "ogrid")]
    q = [M.smooth_perturbed_state(c, 0.02, seed=i) for i, c in enumerate(cases)]
    ens = Sd2dEnsemble(cases)
    for i, s in enumerate(q):
        ens.set_state(i, s, [0, 0, 0, 0])
    ens.step(2)
    ens.tune(1)
    ens.step(2)
    for i, c in enumerate(cases):
        g = Sd2d(c)
        g.set_state(q[i], [0, 0, 0, 0])
        g.step(4)
        a, ma = g.get_state()
        b, mb = ens.get_state(i)
        assert np.isfinite(a).all()
        assert np.array_equal(a, b) and np.array_equal(ma, mb), (i, c.N, c.ncell)
        g.close()
    ens.close()
