"""The adjoint of runs whose state was set with the local maxima (eigvmax,
umax) apart from the pair the first c_h is formed from (eigvmax_g, umax_g):
a maximum that came from the caller is a constant, one that a flux point
attained is not.  Against central differences of the device's own forward
(bar 1e-5, h = 1e-6, as the steps of test_gpu_adjoint)."""
import numpy as np
import pytest

from tests.util import make_case

pytestmark = pytest.mark.gpu

# eigvmax, umax, eigvmax_g, umax_g: no point reaches the caller's local maxima
# (c_h of the second evaluation on is formed from them); only the wave speed's;
# local maxima below the pair (every maximum restarts from the first
# evaluation's points)
MAXIMA = {"local above": [50.0, 20.0, 6.0, 2.0], "eigvmax above": [50.0, 0.0, 6.0, 2.0],
          "local below": [0.0, 0.0, 50.0, 20.0]}


@pytest.mark.parametrize("name", ["ogrid4x8_N4", "channel5x4_N3", "periodic4x4_N5"])
@pytest.mark.parametrize("which", MAXIMA)
def test_vjp_with_maxima_set_apart(name, which):
    from sddc_amd.solver import Sd2d
    print(f"[gpu-adj-maxima] {name} {which}", flush=True)
    case, Q0 = make_case(name)
    mx = MAXIMA[which]
    rng = np.random.default_rng(7)
    C = np.asfortranarray(rng.standard_normal(Q0.shape))
    V = np.asfortranarray(rng.standard_normal(Q0.shape)) * \
        np.abs(Q0).max(axis=(1, 2, 3))[:, None, None, None]
    nsteps, jbar = 3, 2.0
    g = Sd2d(case)

    def F(Q):
        g.set_state(Q, mx)
        J = g.fwd(nsteps, 2)
        return np.sum(C * g.get_state()[0]) + jbar * J

    F(Q0)
    Qf, mf = g.get_state()
    qb0, _, _ = g.vjp(C, jbar)
    # the context is as after fwd
    Qv, mv = g.get_state()
    assert np.array_equal(Qv, Qf) and np.array_equal(mv, mf)
    h = 1e-6
    fd = (F(Q0 + h * V) - F(Q0 - h * V)) / (2 * h)
    ad = float(np.sum(qb0 * V))
    print(f"[gpu-adj-maxima] adjoint {ad:.12e} fd {fd:.12e}", flush=True)
    assert abs(ad - fd) <= 1e-5 * abs(fd), (ad, fd)
    g.close()
