"""The compact metric table (one metric vector per flux-point position, shared
by the lines of a family) against the full one.  A mesh takes the full table
as soon as one vector differs between two lines of one cell, so the same mesh
with the last bit of one such value of one cell flipped runs the general path:
away from that cell the results must be bit for bit the same."""
import dataclasses

import numpy as np
import pytest

from sddc_amd import abi
from sddc_amd import mesh as M

pytestmark = pytest.mark.gpu


def _pair(N, **kw):
    m = M.ogrid(14, 25, 0.5, 4.0)
    case = M.build_case(m, M.RunParams(N=N, dt=2e-4, **kw))
    s1 = case.s1.copy(order="F")
    cell = case.ncell - 3                       # on the outer ring
    s1[0, 0, 1, 1, cell] = np.nextafter(s1[0, 0, 1, 1, cell], np.inf)
    return case, dataclasses.replace(case, s1=s1)


INNER = 25 * 8                                  # eight inner rings: six rings from the change


@pytest.mark.parametrize("style", ["fp64", "mixed", "rk4", "viscous"])
@pytest.mark.parametrize("N", [3, 4, 5])
def test_compact_equals_full(N, style):
    from sddc_amd.solver import Sd2d
    print(f"[gpu-metric-table] N={N} {style}", flush=True)
    kw = {"k_stage": 5} if style == "rk4" else ({"mu": 0.01, "eta0": 0.02} if style == "viscous" else {})
    out = []
    for case in _pair(N, **kw):
        Q = M.smooth_perturbed_state(case, 0.05, seed=1)
        g = Sd2d(case, precision=abi.SD2D_MIXED if style == "mixed" else abi.SD2D_FP64)
        g.set_state(Q, [0, 0, 0, 0])
        r, nab = g.compresid()
        g.set_state(Q, [2.0, 1.0, 2.0, 1.0])
        g.step(1, 1)
        res = [r, nab, g.get_state()[0], g.get_av()[0]]
        if style == "fp64":
            g.set_state(Q, [2.0, 1.0, 2.0, 1.0])
            res.append(g.compresid_vjp(np.asfortranarray(Q * Q))[0])
            g.set_state(Q, [2.0, 1.0, 2.0, 1.0])
            g.fwd(1, 1)
            res.append(g.vjp(None, 1.0)[0])
        out.append(res)
    for a, b in zip(*out):
        assert np.array_equal(a[..., :INNER], b[..., :INNER])
        assert np.isfinite(a).all()


def test_ensemble_of_both_kinds():
    """A group whose members are of both kinds takes the full table for all;
    its members equal single runs bit for bit."""
    from sddc_amd.solver import Sd2d, Sd2dEnsemble
    a, b = _pair(4)
    c = M.build_case(M.ogrid(5, 12, 0.5, 6.0, curved=True), M.RunParams(N=4, dt=2e-4, curve_wall=1))
    cases = [a, b, c]
    q = [M.smooth_perturbed_state(x, 0.05, seed=2) for x in cases]
    e = Sd2dEnsemble(cases)
    for i in range(3):
        e.set_state(i, q[i], [0, 0, 0, 0])
    e.step(3)
    for i, x in enumerate(cases):
        g = Sd2d(x)
        g.set_state(q[i], [0, 0, 0, 0])
        g.step(3)
        s, mx = g.get_state()
        t, my = e.get_state(i)
        assert np.array_equal(s, t) and np.array_equal(mx, my)
