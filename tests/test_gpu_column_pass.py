"""2D column pass and the x-pass's two forms at the edges of their ranges, against
the FP64 oracle: the shortest and longest columns (one wavefront and more per
team), unequal extents, and batches whose rows share blocks across members.
Tolerance 1e-12 on states of order one after 3 RK4 steps: a few hundred
roundings of 1e-16 each, far below it; FP32-bulk increments are dt times
single-precision products, 1e-2 x 1e-7 x 12 stages, below 1e-6."""
import numpy as np
import pytest

import oracle_lib as O
import psgpu_amd as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,batch", [(16, 16, 1), (16, 64, 3), (64, 16, 1), (16, 16, 130), (1024, 32, 1),
                                         (32, 1024, 1), (256, 512, 9), (128, 256, 2)])
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_2d_steps_at_edges(gpu, nx, ny, batch, prec):
    alpha = ny / nx
    g = O.grid2(nx, ny, alpha)
    z0 = np.stack([O.ic_ns2d_cfg(g, 91 + m % 5, 1.0) for m in range(batch)])
    with P.Stepper(flavour="ns2d", nx=nx, ny=ny, n=ny, alpha=alpha, v2=1 / 40, dt=0.01, force="kolmogorov", kf=4.0,
                   ampfor=-2.0, batch=batch, precision=prec) as s:
        for m in range(batch):
            s.set_state(z0[m][None], m)
        s.run(3)
        got = [s.get_state(m)[0] for m in range(batch)]
    orc = O.NS2D(ny, v2=1 / 40, dt=0.01, alpha=alpha, nx=nx)
    want = [orc.run(z0[m], 3) for m in range(min(batch, 5))]
    tol = 1e-12 if prec == "fp64" else 1e-6
    for m in range(batch):
        w = want[m % 5]
        assert np.abs(got[m] - w).max() <= tol * np.abs(w).max(), m
