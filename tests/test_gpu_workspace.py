"""Device memory of the workspaces that a context allocates on first use, against
what their kernels read and write: the tangent linear keeps one perturbation state
and what its scheme stores (3D Heun one right-hand side, 2D RK4 one running sum) and
its pass buffers; the adjoint sweep's workspace stays with the context up to 1 GiB,
serves sweeps of other lengths, and a larger one is given back."""
import numpy as np
import pytest
import torch

import psgpu_amd as P

pytestmark = pytest.mark.gpu

GRAIN = 2 << 20   # an allocation is a whole number of these


def free():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def rough(s, seed):
    rng = np.random.default_rng(seed)
    return (rng.standard_normal((s.nf, s.nkt)) + 1j * rng.standard_normal((s.nf, s.nkt))) / np.sqrt(s.nkt)


@pytest.mark.parametrize("kw", [dict(flavour="ns3d", n=128), dict(flavour="ns2d", n=1024, batch=4)])
def test_tangent_keeps_what_it_uses(gpu, kw):
    with P.Stepper(v2=0.01, dt=1e-3, **kw) as s:
        z, d = rough(s, 1), rough(s, 2)
        two = s.nf == 1
        go = (lambda: s.tangent(z, d, 2e-3, 1e-3)) if two else (lambda: s.tangent_steps(z, d, 2))
        s.set_graph(0)
        s.timederiv(z)   # the kernels used and the staging of host arrays are there before
        before = free()
        go()
        used = before - free()
        n, g = kw["n"], s.grid
        ix, b = n // 3 + 1, kw.get("batch", 1)
        iy, xp = 2 * (n // 3) + 1, (ix + 15) // 16 * 16
        state = 16 * s.nf * s.nkt * b
        if two:
            buffers = 10 * 16 * ix * (n + 8) * b
        else:
            buffers = 16 * (12 * n * iy * xp + 18 * n * n * xp)
        assert used <= 2 * state + buffers + 6 * GRAIN, (used, state, buffers)
        assert used >= buffers


def test_adjoint_workspace_is_kept_and_given_back(gpu):
    n, gib = 128, 1 << 30
    with P.Stepper(flavour="ns3d", n=n, v2=0.01, dt=1e-3) as s:
        z, lam = rough(s, 3) * s.mask, rough(s, 4) * s.mask
        state = 16 * 3 * s.nkt
        states = lambda steps, k: -(-steps // min(k, steps)) + 2 * min(k, steps) + 2
        assert states(40, 40) * state > gib > states(40, 10) * state
        s.adjoint(z, lam, 1, 1)
        base = free() + states(1, 1) * state
        want = s.adjoint(z, lam, 40, 10)
        for steps, k in ((40, 10), (40, 4), (7, 3)):   # the smaller sweeps use the kept workspace
            got = s.adjoint(z, lam, steps, k)
            assert abs(base - free() - states(40, 10) * state) <= 2 * GRAIN, (steps, k)
            if steps == 40:
                assert all(np.array_equal(a, b) for a, b in zip(got, want)), k
        got = s.adjoint(z, lam, 40, 40)                # larger than 1 GiB: given back
        assert all(np.array_equal(a, b) for a, b in zip(got, want))
        assert base - free() <= 2 * GRAIN
        got = s.adjoint(z, lam, 40, 10)                # and a later sweep allocates again
        assert all(np.array_equal(a, b) for a, b in zip(got, want))
        assert abs(base - free() - states(40, 10) * state) <= 2 * GRAIN
    # the context's memory goes with it
    assert free() >= base
