"""Boussinesq passes at the edges of their dispatch, against the FP64 oracle: the
z-inverse with its fields split over blocks (few blocks) and whole, short and long
transforms, ragged kx tiles and batches, both precisions, the default x-pass shape
of every rule, and rough states (neither solenoidal nor masked).  Two steps of
states of order one: 1e-12 leaves hundreds of FP64 roundings; in FP32-bulk each
increment is dt times single-precision products, 1e-3 x 1e-6, below 1e-7."""
import numpy as np
import pytest

import oracle_lib as O
import psgpu_amd as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,batch", [((32, 32, 32), 1), ((16, 64, 16), 2), ((64, 32, 256), 1), ((32, 16, 512), 1),
                                     ((128, 64, 64), 5), ((256, 32, 32), 2), ((16, 32, 1024), 1)])
@pytest.mark.parametrize("prec,tol", [("fp64", 1e-12), ("fp32", 1e-7)])
def test_steps_match_oracle(gpu, n, batch, prec, tol):
    kw = dict(flavour="bous", nx=n[0], ny=n[1], nz=n[2], alpha=n[1] / n[0], v2=0.01, sc=2.0, ri=0.7, theta=0.9,
              dt=1e-3, force="kolmogorov")
    with P.Stepper(batch=batch, precision=prec, **kw) as s:
        rng = np.random.default_rng(11)
        z = [(rng.standard_normal((4, s.nkt)) + 1j * rng.standard_normal((4, s.nkt))) / np.sqrt(s.nkt)
             for _ in range(batch)]
        for m in range(batch):
            s.set_state(z[m], m)
        s.run(2)
        got = [s.get_state(m) for m in range(batch)]
    orc = O.BOUS(n[1], v2=0.01, dt=1e-3, sc=2.0, ri=0.7, theta=0.9, alpha=n[1] / n[0], nx=n[0], ny=n[1], nz=n[2])
    for m in (0, batch - 1):
        want = orc.run(z[m], 2)
        assert np.abs(got[m] - want).max() <= tol * np.abs(want).max()
