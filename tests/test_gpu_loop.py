"""The device loop's control inside the first stage of a step (march kernel) and in a kernel of its own
(strip kernel), over every way to drive a run: one fv2d_advance by step count, short ones by end
time (whose last chunk queues steps past the end), and the host-driven loop of fv2d_compute_dt and
fv2d_step, mixed with each other. Same dt sequence, time and fields, bit for bit."""
import numpy as np
import pytest

from fv2d_amd import problems as P
from fv2d_amd.capi import FP32, FP64, TS_EULER, TS_RK2
from fv2d_amd.solver import Solver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("chunk_rows", [0, 4])
@pytest.mark.parametrize("precision", [FP64, FP32])
@pytest.mark.parametrize("ts", [TS_EULER, TS_RK2])
@pytest.mark.parametrize("nx,ny", [(2, 3), (61, 40), (300, 7)])
def test_loop_forms_agree(nx, ny, ts, precision, chunk_rows, gpu_lib):
    p = P.kh_params(N=2, Nx=nx, Ny=ny, time_stepping=ts, precision=precision, chunk_rows=chunk_rows, CFL=0.3)
    q0, n = P.random_state(p, seed=nx), 37
    with Solver(p, gpu_lib) as a, Solver(p, gpu_lib) as b, Solver(p, gpu_lib) as c:
        for s in (a, b, c):
            s.set_prim(q0)
        t, dts, counts, k = a.advance(max_steps=n)
        assert k == n and len(dts) == n
        # by end times that fall between two steps, with and without a step limit
        tb, done, got = 0.0, 0, np.zeros(3, dtype=int)
        ends = np.concatenate([[0.0], np.cumsum(dts)])
        for upto, limit in ((1, 0), (2, 50), (9, 0), (9, 0), (20, 11), (37, 0)):
            tend = ends[upto] - 0.5 * dts[upto - 1] + p.epsilon
            tb, _, cnt, m = b.advance(tend=tend, max_steps=limit, t0=tb, record_dts=False)
            done += m
            got += cnt
            assert done == upto
            if upto < n:
                assert b.compute_dt()[0] == dts[upto]
        assert tb == t and tuple(got) == tuple(counts)
        # the host loop, with a device loop in the middle
        tc = 0.0
        for k in range(n):
            if k == 15:
                tc, d, _, m = c.advance(max_steps=6, t0=tc)
                assert m == 6 and np.array_equal(d, dts[15:21])
            if 15 <= k < 21:
                continue
            dt, _ = c.compute_dt()
            assert dt == dts[k]
            c.step(dt)
            tc += dt
        assert tc == t
        qa = a.get_prim()
        assert np.array_equal(qa, b.get_prim()) and np.array_equal(qa, c.get_prim())
        assert a.compute_dt()[0] == b.compute_dt()[0] == c.compute_dt()[0]
