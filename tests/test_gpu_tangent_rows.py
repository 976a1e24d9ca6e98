"""The combined base + perturbation x-pass (six fields in, four out) over blocks of
neighbouring rows: from 2048 rows on, the rows of several members in one block and a
last block that is partly empty, and a single 1024^2 member; and over one row a block
at its longest row.  The perturbation of member 0 against the recorded replay of a
single-member context (an x-pass of three fields, one row a block) and central
differences of the FP64 oracle, the base flows of the other members against the oracle.
Three RK4 steps of states of order one: 1e-12 leaves hundreds of FP64 roundings, twice
that for the two products of the linearised term; FP32-bulk increments are dt times
single-precision products, 1e-2 x 1e-7 x 12 stages, below 1e-6 and again twice that.
The differences with eps 1e-5 are off by eps^2 and by 1e-16 / eps a rounding: 1e-8."""
import numpy as np
import pytest

import oracle_lib as O
import psgpu_amd as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,batch", [(16, 16, 129), (32, 16, 129), (64, 16, 129), (128, 16, 129), (256, 32, 65),
                                         (512, 16, 129), (1024, 16, 65), (1024, 1024, 1), (1024, 64, 1)])
@pytest.mark.parametrize("prec,tol", [("fp64", 2e-12), ("fp32", 2e-6)])
def test_tangent_over_rows_of_many_members(gpu, nx, ny, batch, prec, tol):
    alpha, steps, dt = ny / nx, 3, 0.005
    g = O.grid2(nx, ny, alpha)
    z = np.stack([O.ic_ns2d_cfg(g, 31 + m, 1.0) for m in range(3)])
    d = O.ic_ns2d_cfg(g, 47, 1.0)
    kw = dict(flavour="ns2d", nx=nx, ny=ny, n=ny, alpha=alpha, v2=1 / 40, dt=dt, force="kolmogorov", kf=4.0, ampfor=-2.0,
              precision=prec)
    T = steps * dt * (1 + 1e-9)   # the period's integer part is the step count
    with P.Stepper(batch=batch, **kw) as s:
        for m in range(1, batch):
            s.set_state(z[m % 3][None], m)
        z1, dz1 = s.tangent(z[0][None], d[None], T, dt)
        others = {m: s.get_state(m)[0] for m in {1, 2, batch - 2, batch - 1} if 0 < m < batch}
    with P.Stepper(batch=1, **kw) as s:
        z2, dz2 = s.tangent_many(z[0][None], d[None, None], T, dt)
    assert np.abs(z1 - z2).max() <= tol * np.abs(z2).max()
    assert np.abs(dz1 - dz2).max() <= tol * np.abs(dz2).max()
    orc = O.NS2D(ny, v2=1 / 40, dt=T / steps, alpha=alpha, nx=nx)
    want = [orc.run(z[m], steps) for m in range(3 if others else 1)]
    assert np.abs(z1[0] - want[0]).max() <= tol * np.abs(want[0]).max()
    for m, got in others.items():
        assert np.abs(got - want[m % 3]).max() <= tol * np.abs(want[m % 3]).max(), m
    eps = 1e-5
    fd = (orc.run(z[0] + eps * d, steps) - orc.run(z[0] - eps * d, steps)) / (2 * eps)
    assert np.abs(dz1[0] - fd).max() <= max(tol, 1e-8) * np.abs(fd).max()
