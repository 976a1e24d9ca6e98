"""Device memory of the workspaces that a context allocates on first use, against
what their kernels read and write: the tangent linear keeps one perturbation state
and what its scheme stores (3D Heun one right-hand side, 2D RK4 one running sum) and
its pass buffers."""
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
