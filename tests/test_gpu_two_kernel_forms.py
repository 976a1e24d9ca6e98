"""Two-kernel 3D stepper: its two block forms at the largest z tile (128 points in y
and z: two kx columns a block in FP64, three in FP32), each case shown to take the
two-kernel path, over flavours, forcings and member strides; tolerances of the
comparison over all extents.  And a single context of the default stepper is not
slower than the pencil passes where the z kernel has the fewest blocks."""
import time

import pytest

import psgpu_amd as P
import test_gpu_two_kernel_step as forms

pytestmark = pytest.mark.gpu


def kernels(n, prec, flavour, force, batch):
    with P.Stepper(flavour=flavour, nx=n[0], ny=n[1], nz=n[2], n=n[1], alpha=n[1] / n[0], v2=0.01, dt=1e-3, force=force,
                   precision=prec, batch=batch) as s:
        s.profile()
        s.run(1)
        return {r["kernel"] for r in s.profile_report()}


@pytest.mark.parametrize("n,prec,flavour,force,batch", [
    ((32, 128, 128), "fp64", "euler", "none", 2), ((32, 128, 128), "fp64", "ns3d", "gmres", 2),
    ((64, 128, 128), "fp64", "euler", "none", 1), ((64, 128, 128), "fp64", "ns3d", "gmres", 1),
    ((32, 128, 128), "fp32", "euler", "none", 3), ((64, 128, 128), "fp32", "ns3d", "gmres", 2),
    ((64, 128, 128), "fp32", "euler", "none", 2), ((128, 128, 128), "fp32", "ns3d", "kolmogorov", 1)])
def test_largest_z_tiles_match_pencil_passes(gpu, n, prec, flavour, force, batch):
    assert {"xy", "z_update"} <= kernels(n, prec, flavour, force, batch)
    states, a = forms.run(n, prec, flavour, force, batch, 0, None, 3)
    _, b = forms.run(n, prec, flavour, force, batch, 1, states, 3)
    assert forms.off(a, b) <= (1e-12 if prec == "fp64" else 1e-6)


@pytest.mark.parametrize("n,prec,batch", [((32, 128, 128), "fp64", 1), ((64, 128, 128), "fp64", 1), ((64, 128, 128), "fp32", 2)])
def test_one_context_is_not_slower(gpu, n, prec, batch):
    with P.Stepper(flavour="ns3d", nx=n[0], ny=n[1], nz=n[2], n=n[1], alpha=n[1] / n[0], v2=0.01, dt=1e-3, precision=prec,
                   batch=batch) as s:
        z = forms.rough(s, 1)
        for m in range(batch):
            s.set_state(z, m)
        best = {0: 1e9, 1: 1e9}
        for _ in range(6):
            # slab variant 1 covers all 128 planes at once: the pencil passes in their default shapes
            for slab in best:
                s.set_variant(slab, 2)
                s.run(33)
                s.sync()
                t = time.perf_counter()
                s.run(64)
                s.sync()
                best[slab] = min(best[slab], time.perf_counter() - t)
        assert best[0] <= best[1], best
