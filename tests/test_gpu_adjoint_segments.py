"""The adjoint sweep's segments: every checkpoint interval gives the same bits (the
recomputed states are those recorded), for intervals that divide the steps, leave
one step over, hold a single step or exceed the run, and the residual gradient's
flow is the adjoint's."""
import numpy as np
import pytest

import oracle_lib as O
import psgpu_amd as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("steps", [1, 7])
def test_checkpoint_interval_changes_nothing(gpu, steps, prec):
    with P.Stepper(flavour="ns3d", n=32, v2=0.01, dt=0.01, precision=prec) as s:
        rng = np.random.default_rng(steps)
        z, lam = ((rng.standard_normal((3, s.nkt)) + 1j * rng.standard_normal((3, s.nkt))) * s.mask / np.sqrt(s.nkt)
                  for _ in range(2))
        s.set_state(z)
        s.run(steps)
        flow = s.get_state()
        z0, l0 = s.adjoint(z, lam, steps, 100)
        assert np.isfinite(l0).all() and np.abs(l0).max() > 0
        assert np.abs(z0 - flow).max() <= (1e-13 if prec == "fp64" else 1e-6) * np.abs(flow).max()
        for ckpt in (1, 2, 3, 4, 7):
            zc, lc = s.adjoint(z, lam, steps, ckpt)
            assert np.array_equal(zc, z0) and np.array_equal(lc, l0), ckpt
            assert np.array_equal(s.get_state(), z0)


@pytest.mark.parametrize("n", [(64, 16, 32), (128, 32, 16), (256, 16, 16), (1024, 16, 16)])
@pytest.mark.parametrize("prec,tol", [("fp64", 1e-11), ("fp32", 1e-5)])
def test_adjoint_transposes_the_tangent_at_every_row_length(gpu, n, prec, tol):
    # unit directions: hundreds of roundings of the two inner products
    g = O.grid3(*n, n[1] / n[0])
    L = O.tables(g)[3].astype(float)
    z = O.ic_solenoidal(g, 3, 0.5)
    v, w = (d / np.sqrt(np.sum(np.abs(d) ** 2)) for d in (O.ic_solenoidal(g, 4, 0.5), O.ic_solenoidal(g, 5, 0.5)))
    with P.Stepper(flavour="ns3d", nx=n[0], ny=n[1], nz=n[2], alpha=n[1] / n[0], v2=0.02, dt=0.004,
                   force="kolmogorov", precision=prec) as s:
        _, jv = s.tangent_steps(z, v, 5)
        _, jtw = s.adjoint(z, w, 5, 2)
    lhs, rhs = (float(np.sum((np.conj(a) * b).real * L[None])) for a, b in ((jv, w), (v, jtw)))
    assert abs(lhs - rhs) <= tol, (lhs, rhs)
