"""Host <-> device copies of the state (fv2d_set_prim, fv2d_get_prim, fv2d_get_cons) at the sizes where
the copy path changes (one runtime copy, pinned pieces of 1 / 2 / 4 MB on one or more threads) and with
ragged last pieces: what was uploaded comes back bit for bit, also from two host threads at once."""
import threading

import numpy as np
import pytest

from fv2d_amd import problems as P
from fv2d_amd.solver import Solver

pytestmark = pytest.mark.gpu

SHAPES = [(64, 64), (256, 256), (257, 256), (331, 283), (512, 512), (625, 629), (1021, 613), (1448, 1449), (2000, 1500)]


def round_trip(nx, ny, gpu_lib, times=2):
    p = P.kh_params(N=2, Nx=nx, Ny=ny)
    with Solver(p, gpu_lib) as s:
        for seed in range(times):
            q = P.random_state(p, seed=seed)
            s.set_prim(q)
            assert np.array_equal(s.get_prim(), q)
            u = s.get_cons()
            assert np.array_equal(u[0], q[0]) and np.array_equal(u[1], q[0] * q[1])


@pytest.mark.parametrize("nx,ny", SHAPES)
def test_round_trip(nx, ny, gpu_lib):
    round_trip(nx, ny, gpu_lib)


def test_two_threads(gpu_lib):
    errors = []

    def work(nx, ny):
        try:
            round_trip(nx, ny, gpu_lib, times=3)
        except BaseException as e:  # noqa: BLE001 (reported below)
            errors.append(e)

    ts = [threading.Thread(target=work, args=a) for a in ((1021, 613), (1448, 1449))]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not errors, errors
