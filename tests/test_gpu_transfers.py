"""State-sized copies through the pinned ring (sd2d_xfer.hpp): the round trip
is bit for bit at the sizes where its path changes (below and above 1 MiB, 3
MiB, the ring's 32 MiB and the upload's 64 MiB; whole and ragged last chunks),
and with several contexts copying from several threads at once."""
import threading

import numpy as np
import pytest

from sddc_amd import mesh as M

pytestmark = pytest.mark.gpu


def _context(nx, ny, N):
    from sddc_amd.solver import Sd2d
    m = M.periodic_square(nx, ny)
    p = M.RunParams(N=N, dxcycl=m.dxcycl, dycycl=m.dycycl, dt=1e-4)
    return Sd2d(M.build_case(m, p))


def _state(g, seed):
    return np.asfortranarray(np.random.default_rng(seed).random((g.nc, g.N, g.N, 9)).T)


# N = 5: 1800 bytes a cell, N = 3: 648
@pytest.mark.parametrize("nx,ny,N", [(97, 6, 5), (53, 11, 5), (32, 52, 3), (83, 21, 5), (85, 22, 5),
                                     (137, 136, 5), (167, 113, 5), (200, 187, 5)])
def test_round_trip(nx, ny, N):
    print(f"[gpu-transfers] {nx}x{ny} N={N}", flush=True)
    g = _context(nx, ny, N)
    for seed in (1, 2):
        q = _state(g, seed)
        g.set_state(q, [1.0, 0.5, 2.0, 0.25])
        r, mx = g.get_state()
        assert np.array_equal(r, q)
        assert np.array_equal(mx, [1.0, 0.5, 2.0, 0.25])
    g.close()


def test_several_threads():
    ctx = [_context(60 + 7 * k, 50, 5) for k in range(4)]
    bad = []

    def work(k):
        try:
            for i in range(6):
                q = _state(ctx[k], 10 * k + i)
                ctx[k].set_state(q)
                if not np.array_equal(ctx[k].get_state()[0], q):
                    bad.append((k, i))
        except Exception as e:   # reported by the assertion below
            bad.append((k, repr(e)))

    th = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad, bad
    for c in ctx[:3]:
        c.close()
    q = _state(ctx[3], 99)       # the ring outlives the contexts that are gone
    ctx[3].set_state(q)
    assert np.array_equal(ctx[3].get_state()[0], q)
    ctx[3].close()
    g = _context(60, 50, 5)      # and is there again after the last one went
    q = _state(g, 100)
    g.set_state(q)
    assert np.array_equal(g.get_state()[0], q)
