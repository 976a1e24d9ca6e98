"""The ends of a run.  The steppers whose update makes the next stage's fields make
none after a run's last step; a run of any length, in one call or step by step, by
direct launches or with captured steps in the middle (that end with the run, or leave
steps over), is the same flow, and so are the tangent about a running base and about
a recorded one.  States of order one over up to 11 steps: 1e-12 leaves hundreds of
FP64 roundings; FP32-bulk (1e-6) rounds products of dt 1e-3 or 5e-3 in each step."""
import numpy as np
import pytest

import oracle_lib as O
import psgpu_amd as P

pytestmark = pytest.mark.gpu

CASES = [dict(flavour="ns2d", n=64, batch=3, v2=1 / 40, dt=0.005, kf=4.0, ampfor=-2.0),
         dict(flavour="ns2d", n=1024, v2=1 / 40, dt=0.002, kf=4.0, ampfor=-2.0),
         dict(flavour="ns3d", n=32, batch=2, v2=0.02, dt=1e-3), dict(flavour="euler", n=64, v2=0.0, dt=1e-3, force="none"),
         dict(flavour="ns3d", n=16, v2=0.02, dt=1e-3), dict(flavour="bous", n=32, v2=0.02, dt=1e-3, ri=0.5)]


def start(s):
    if s.nf == 1:
        return O.ic_ns2d_cfg(O.grid2(s.cfg.nx, s.cfg.ny), 17, 1.0)[None]
    z = np.zeros((s.nf, s.nkt), np.complex128)
    z[:3] = O.ic_solenoidal(O.grid3(s.cfg.nx, s.cfg.ny, s.cfg.nz), 17, 0.5)[:3]
    if s.nf == 4:
        z[3] = 0.1 * z[0]
    return z


@pytest.mark.parametrize("kw", CASES)
@pytest.mark.parametrize("prec,tol", [("fp64", 1e-12), ("fp32", 1e-6)])
def test_a_run_may_be_cut_anywhere(gpu, kw, prec, tol):
    with P.Stepper(precision=prec, **kw) as s:
        z = start(s)
        last = s.cfg.batch - 1

        def flow(graph, *chunks):
            s.set_graph(graph)
            for m in range(s.cfg.batch):
                s.set_state(z * (1.0 - 0.1 * m), m)
            for n in chunks:
                s.run(n)
            return np.stack([s.get_state(0), s.get_state(last)])

        want = flow(0, *[1] * 11)
        size = np.abs(want).max()
        for graph, chunks in ((0, (11,)), (0, (5, 6)), (4, (11,)), (4, (9, 2)), (4, (5, 5, 1)), (10, (11,))):
            assert np.abs(flow(graph, *chunks) - want).max() <= tol * size, (graph, chunks)


@pytest.mark.parametrize("graph", [0, 4])
@pytest.mark.parametrize("prec,tol", [("fp64", 1e-12), ("fp32", 1e-6)])
def test_tangents_of_any_length(gpu, graph, prec, tol):
    kw = dict(flavour="ns2d", n=64, v2=1 / 40, dt=0.005, kf=4.0, ampfor=-2.0, precision=prec)
    with P.Stepper(**kw) as s:
        s.set_graph(graph)
        g = O.grid2(64, 64)
        z, d = O.ic_ns2d_cfg(g, 3, 1.0), O.ic_ns2d_cfg(g, 4, 1.0)
        for T in (0.005, 0.0255, 0.0457):        # whole steps and a short last one (policy 1)
            z1, d1 = s.tangent(z[None], d[None], T * (1 + 1e-9), 0.005, 1)
            z2, d2 = s.tangent_many(z[None], np.stack([d, d])[:, None], T * (1 + 1e-9), 0.005, 1)
            zf = s.flow_map(z[None], T * (1 + 1e-9), 0.005, 1)
            assert np.abs(z1 - zf).max() <= tol * np.abs(zf).max(), T
            assert np.abs(z2 - zf).max() <= tol * np.abs(zf).max(), T
            assert np.abs(d2 - d1).max() <= 2 * tol * np.abs(d1).max(), T


@pytest.mark.parametrize("nx,ny", [(16, 16), (32, 64), (64, 32), (128, 128), (256, 256), (64, 512), (32, 1024)])
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_captured_steps_at_the_end_give_the_bits_of_direct_launches(gpu, nx, ny, prec):
    # the last stage of direct launches only updates, that of captured steps also transforms
    g = O.grid2(nx, ny, ny / nx)
    z, d = O.ic_ns2d_cfg(g, 5, 1.0), O.ic_ns2d_cfg(g, 6, 1.0)
    with P.Stepper(flavour="ns2d", nx=nx, ny=ny, n=ny, alpha=ny / nx, v2=1 / 40, dt=0.005, kf=4.0, ampfor=-2.0,
                   precision=prec) as s:
        out = []
        for graph in (0, 4):
            s.set_graph(graph)
            s.set_dt(0.005)   # the tangents leave their own
            s.set_state(z[None])
            s.run(9)
            out.append((s.get_state(),) + s.tangent(z[None], d[None], 9.5 * 0.005, 0.005)
                       + s.tangent_many(z[None], d[None, None], 9.5 * 0.005, 0.005))
    for a, b in zip(*out):
        assert np.array_equal(a, b)
