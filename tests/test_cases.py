"""The bytes a stage has to move: which metric table a mesh takes."""
import dataclasses

import numpy as np
import pytest

from sddc_amd import cases
from sddc_amd import mesh as M
from tests.util import CASES, make_case


@pytest.mark.parametrize("name", sorted(CASES))
def test_lines_share(name):
    case, _ = make_case(name)
    assert cases.lines_share_metrics(case) == ("curved" not in name)


@pytest.mark.parametrize("which", ["s1", "s2"])
def test_one_bit_apart(which):
    case = M.build_case(M.ogrid(3, 9, 0.5, 4.0), M.RunParams(N=4, dt=1e-3))
    s = getattr(case, which).copy(order="F")
    i = (0, 1, 2, 3, 7) if which == "s1" else (1, 0, 2, 3, 7)
    s[i] = np.nextafter(s[i], np.inf)
    assert not cases.lines_share_metrics(dataclasses.replace(case, **{which: s}))
    full = cases.alg_bytes_per_dof_stage(4)
    assert full - cases.alg_bytes_per_dof_stage(4, lines_share=True) == 8 * 4 * 3 * 5 / 16
