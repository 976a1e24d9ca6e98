"""Two-kernel 3D stepper (small grids, default shapes) against the five pencil
passes and the FP64 oracle, over the forms that it accepts: every extent it takes
beside every other, both precisions and flavours, the three forcings, batches,
and states that are neither solenoidal nor masked (the kx = 0 plane then holds
values in the half that the Hermitian fill replaces).  States are of order one
after 3 steps of dt 1e-3: 1e-12 leaves hundreds of FP64 roundings, and FP32-bulk
rounds the state itself, 3 steps of 1e-7 each."""
import numpy as np
import pytest

import oracle_lib as O
import psgpu_amd as P

pytestmark = pytest.mark.gpu

SHAPES = [(32, 32, 32), (64, 64, 64), (32, 64, 128), (128, 32, 64), (64, 128, 32), (32, 128, 64), (128, 64, 32),
          (64, 32, 128), (128, 128, 64), (64, 128, 128)]


def rough(st, seed):
    rng = np.random.default_rng(seed)
    return (rng.standard_normal((3, st.nkt)) + 1j * rng.standard_normal((3, st.nkt))) / np.sqrt(st.nkt)


def run(n, prec, flavour, force, batch, variant, states, steps, graph=16):
    with P.Stepper(flavour=flavour, nx=n[0], ny=n[1], nz=n[2], n=n[1], alpha=n[1] / n[0], v2=0.01, dt=1e-3, force=force,
                   precision=prec, batch=batch) as s:
        s.set_variant(variant)
        s.set_graph(graph)
        if states is None:
            states = [rough(s, 7 + m) for m in range(batch)]
        for m in range(batch):
            s.set_state(states[m], m)
        s.run(steps)
        return states, [s.get_state(m) for m in range(batch)]


def off(a, b):
    return max(np.abs(x - y).max() / np.abs(y).max() for x, y in zip(a, b))


@pytest.mark.parametrize("n", SHAPES)
@pytest.mark.parametrize("prec,tol", [("fp64", 1e-12), ("fp32", 1e-6)])
def test_matches_pencil_passes(gpu, n, prec, tol):
    for flavour, force, batch in (("ns3d", "kolmogorov", 1), ("euler", "none", 2), ("ns3d", "gmres", 3)):
        states, a = run(n, prec, flavour, force, batch, 0, None, 3)
        _, b = run(n, prec, flavour, force, batch, 1, states, 3)
        assert off(a, b) <= tol, (flavour, force, batch)


@pytest.mark.parametrize("n", [(32, 32, 32), (64, 32, 32), (32, 64, 32)])
@pytest.mark.parametrize("flavour,force,code", [("ns3d", "dns", 1), ("ns3d", "kolmogorov", 3), ("euler", "none", 0)])
def test_rough_states_match_oracle(gpu, n, flavour, force, code):
    states, a = run(n, "fp64", flavour, force, 1, 0, None, 3)
    orc = O.NS3D(n[1], v2=0.01, dt=1e-3, force=code, alpha=n[1] / n[0], nx=n[0], ny=n[1], nz=n[2],
                 flavour=1 if flavour == "euler" else 0)
    assert off(a, [orc.run(states[0], 3)]) <= 1e-12


def test_layout_follows_the_variant(gpu):
    """One context stepping with the two kernels, the pencil passes and the two kernels
    again, over a change of dt, equals fresh contexts doing each part."""
    n = (64, 64, 64)
    with P.Stepper(flavour="ns3d", n=64, v2=0.01, dt=1e-3) as s:
        z = rough(s, 3)
        s.set_state(z)
        want = z
        for variant, dt in ((0, 1e-3), (1, 1e-3), (0, 2e-3), (0, 1e-3)):
            s.set_variant(variant)
            s.set_dt(dt)
            s.run(19)
            with P.Stepper(flavour="ns3d", n=64, v2=0.01, dt=dt) as f:
                f.set_variant(2)
                f.set_state(want)
                f.run(19)
                want = f.get_state()
            assert off([s.get_state()], [want]) <= 1e-12
