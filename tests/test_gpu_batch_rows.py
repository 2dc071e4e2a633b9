"""Task height of batched march jobs: chosen for the whole work list from the jobs it holds, so the
same job runs in tasks of 4, 8 or 16 rows, also changing between launches. Bit for bit the job with a
task height of its own, in lists from one small job (more items than max_items counts) to a full chip."""
import numpy as np
import pytest

from fv2d_amd import problems as P
from fv2d_amd.capi import FP32, FP64, BatchConfig
from fv2d_amd.solver import Batch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [FP64, FP32])
@pytest.mark.parametrize("nx,ny,jobs,max_items", [(61, 70, 1, 2), (2, 3, 9, 9), (130, 133, 40, 1 << 18),
                                                  (300, 203, 60, 1 << 18), (190, 37, 300, 1 << 18)])
def test_height_of_the_list(nx, ny, jobs, max_items, precision, gpu_lib):
    def run(seg, stagger):
        p = P.kh_params(N=2, Nx=nx, Ny=ny, precision=precision, CFL=0.3, seg_rows=seg)
        q0 = P.random_state(p, seed=nx)
        cfg = BatchConfig.defaults(precision=precision, max_jobs=jobs, steps_per_launch=2,
                                   max_items=1 << 18 if seg else max_items)
        with Batch(cfg, lib=gpu_lib) as b:
            ids = []
            for k in range(jobs):
                ids.append(b.submit(p, q=q0, max_steps=5 + k % 2))
                if stagger and k in (0, jobs // 2):
                    b.launch(1)
            while b.run(1):
                pass
            return [b.collect(i)[0] for i in sorted({*ids[:2], *ids[-2:]})]

    for x, y in zip(run(0, True), run(16, False)):
        assert np.array_equal(x, y)
