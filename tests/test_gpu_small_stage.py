"""The stage kernel of small meshes (one wavefront per flux-point number)
against the line kernel: the same run alone (at most 256 tiles) and as every
member of an ensemble of more than 256 tiles.  Both sum every point's fluxes
in one order and an ensemble's members are bitwise the runs made alone, so
the states and maxima are equal."""
import numpy as np
import pytest

from sddc_amd import mesh as M
from tests.util import make_case

pytestmark = pytest.mark.gpu

LARGE = {  # exactly 256 tiles; rows padded to the tile; the widest tile
    "periodic64x64_N4": (lambda: M.periodic_square(64, 64), dict(N=4, dt=1e-3)),
    "ogrid4x193_N5": (lambda: M.ogrid(4, 193, 5.0, 6.0), dict(N=5, dt=5e-4)),
    "channel41x37_N3": (lambda: M.channel(41, 37, seed=3, free_left=2), dict(N=3, dt=5e-4)),
}


def _case(name):
    if name not in LARGE:
        return make_case(name)
    mk, kw = LARGE[name]
    m = mk()
    case = M.build_case(m, M.RunParams(dxcycl=m.dxcycl, dycycl=m.dycycl, **kw))
    return case, M.smooth_perturbed_state(case, 0.05, seed=1)


@pytest.mark.parametrize("name,copies", [
    ("channel5x4_N3", 260), ("periodic6x5_N4", 130), ("ogrid_curved4x8_N4", 130),
    ("channel7x6_N5", 65), ("periodic64x64_N4", 2), ("ogrid4x193_N5", 5),
    ("channel41x37_N3", 4)])
def test_alone_equals_line_kernel(name, copies):
    from sddc_amd.solver import Sd2d, Sd2dEnsemble
    print(f"[small stage] {name}", flush=True)
    case, Q0 = _case(name)
    g = Sd2d(case)
    g.set_state(Q0, [0, 0, 0, 0])
    g.step(3)
    Qs, ms = g.get_state()
    g.close()
    ens = Sd2dEnsemble([case] * copies)
    for i in range(copies):
        ens.set_state(i, Q0, [0, 0, 0, 0])
    ens.step(3)
    for i in (0, copies - 1):
        Qe, me = ens.get_state(i)
        assert np.array_equal(Qe, Qs) and np.array_equal(me, ms), (name, i)
    ens.close()
