"""Small fleets on the GPU run the lane-group kernels (two or four lanes per vehicle); results have the bits
of the one-lane kernels, which a fleet bucket set to two waves per SIMD runs at any size."""
import ctypes
import os

import numpy as np
import pytest

from conftest import DATA

import lfdm_amd
from lfdm_amd import workloads as W
from lfdm_amd._lib import lib
from lfdm_amd.solver import Fleet, SolverHalfImplicitGPU, TMeasy, TMeasyNr

pytestmark = pytest.mark.gpu

# One vehicle, around a wavefront, and either side of the sizes where the choice changes on 1,024 SIMDs
# (four lanes up to 16,384 at one and 32,768 at two wavefronts per SIMD, two lanes up to 65,536).
SIZES = [1, 65, 16384, 16385, 32769, 65536, 65537]


def fleet(dof, nr, n):
    d = os.path.join(DATA, f"{dof}dof", "Sedan" if nr else "HMMWV")
    flat = lfdm_amd.params_from_json(dof, f"{d}/vehicle.json", f"{d}/tmeasyNr.json" if nr else f"{d}/tmeasy.json",
                                     f"{d}/suspension.json" if dof == 24 else None, int(nr))
    fl = W.knot_fleet(n, flat, seed=n, dof=dof, tire_nr=nr)
    s = SolverHalfImplicitGPU(dof, n)
    s.construct_flat(flat, n, None, TMeasyNr if nr else TMeasy)
    s.set_overrides(fl["ovr"])
    s.initialize_batch(W.initial_speed_records(n, flat, dof, seed=3, tire_nr=nr))
    s.set_controls_knots(fl["ns"], fl["ds"], fl["np"], fl["dp"], fl["knots"])
    s.set_horizons(np.random.default_rng(n).integers(0, 61, n))
    return s


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("dof,nr", [(11, False), (11, True), (18, False), (18, True), (24, False), (24, True)])
def test_lane_groups_give_the_one_lane_bits(dof, nr, n):
    s = fleet(dof, nr, n)
    init = s.get_states()
    with Fleet([s]) as f:
        f.set_config(0, 64, 0, 2)  # one lane per vehicle
        f.run(60)
        f.synchronize()
        ref = s.get_states()
        s.set_states(init)
        f.set_config(0, 128, 25, 0)  # the automatic choice, in three launches of two-wavefront blocks
        f.run(60)
        f.synchronize()
        got = s.get_states()
    s.close()
    assert n < 64 or not np.array_equal(ref, init)
    np.testing.assert_array_equal(got, ref)


@pytest.mark.parametrize("mode", ["table", "steps"])
@pytest.mark.parametrize("dof,n", [(11, 100), (11, 32769), (18, 100), (18, 16385), (24, 100), (24, 16385)])
def test_controls_looked_up_ahead_give_the_one_lane_bits(dof, n, mode):
    """Driver rows and per-step controls held a step ahead (one wavefront per SIMD) and not, in three launches,
    with horizons: 60 steps over a table of 30 rows, some out of order, the last before the end."""
    d = os.path.join(DATA, f"{dof}dof", "HMMWV")
    flat = lfdm_amd.params_from_json(dof, f"{d}/vehicle.json", f"{d}/tmeasy.json",
                                     f"{d}/suspension.json" if dof == 24 else None)
    rng = np.random.default_rng(n)
    rows = np.column_stack([np.linspace(0.002, 0.05, 30), rng.random((30, 3)) - [0.5, 0.0, 0.0]])
    rows[8:12, 0] = rows[[10, 8, 11, 9], 0]
    s = SolverHalfImplicitGPU(dof, n)
    s.construct_flat(flat, n, rows, TMeasy)
    s.set_overrides(W.knot_fleet(n, flat, seed=n, dof=dof)["ovr"])
    s.initialize_batch(W.initial_speed_records(n, flat, dof, seed=3))
    if mode == "steps":
        s.set_controls_steps(rng.random((60, 3, n)) - np.array([0.5, 0.0, 0.0])[:, None])
    s.set_horizons(rng.integers(0, 61, n))
    init = s.get_states()
    with Fleet([s]) as f:
        f.set_config(0, 64, 0, 2)  # one lane per vehicle
        f.run(60)
        f.synchronize()
        ref = s.get_states()
        s.set_states(init)
        f.set_config(0, 64, 25, 0)
        f.run(60)
        f.synchronize()
        got = s.get_states()
    s.close()
    assert not np.array_equal(ref, init)
    np.testing.assert_array_equal(got, ref)


@pytest.mark.parametrize("budget", [0, 1])
def test_adjoint_lane_groups_give_the_one_lane_bits(budget):
    """Trajectories and gradients of fleets at the sizes where the forward's and the reverse's lanes change,
    against the same vehicles at the head of a fleet of more than one wavefront per SIMD (one lane each);
    budget 1 makes every backward group a single segment, recomputed but for the last."""
    import torch

    from lfdm_amd.mpc import moving_start
    from lfdm_amd.torch_ops import make_solver, rollout

    flat = lfdm_amd.params_from_json(18, W.HMMWV_VEH, W.HMMWV_TIRE)
    steps, big = 40, 65_600
    g = torch.Generator(device="cuda").manual_seed(9)
    rand = lambda *s: torch.rand(s, generator=g, dtype=torch.float64, device="cuda")  # noqa: E731
    ctrl = torch.stack([rand(steps, big) - 0.5, rand(steps, big), 0.3 * rand(steps, big)], 1)
    par = torch.from_numpy(W.default_overrides(flat, big)).cuda() * (0.9 + 0.2 * rand(7, big))
    init = (moving_start(flat, 1)[0].cuda()[None] * (0.5 + rand(big, 1))).contiguous()
    gxy = rand(steps, 2, big) - 0.5

    def gradients(n):
        s = make_solver(flat, n)
        s.adjoint_set_tape_budget(budget)
        x = [t[..., :n].contiguous().requires_grad_(True) for t in (ctrl, par)] + [
            init[:n].contiguous().requires_grad_(True)]
        xy = rollout(s, *x, 16)
        out = [xy.detach(), *torch.autograd.grad(xy, x, gxy[..., :n].contiguous())]
        torch.cuda.synchronize()
        s.close()
        return out

    ref = gradients(big)
    for n in (1, 65, 16384, 16385, 32768, 32769, 65536):
        for name, a, b in zip(("xy", "controls", "parameters", "records"), gradients(n), ref):
            b = b[:n] if name == "records" else b[..., :n]
            assert torch.equal(a, b), (name, n)


def test_step_jacobian_does_not_depend_on_the_fleet():
    """Jacobians of 1, 64 and 65 vehicles are those of the same vehicles in a fleet of 200."""
    import torch

    from lfdm_amd.mpc import moving_start
    from lfdm_amd.torch_ops import make_solver

    flat = lfdm_amd.params_from_json(18, W.HMMWV_VEH, W.HMMWV_TIRE)
    big = 200
    g = torch.Generator(device="cuda").manual_seed(4)
    init = (moving_start(flat, 1)[0].cuda()[None] *
            (0.5 + torch.rand((big, 1), generator=g, dtype=torch.float64, device="cuda"))).contiguous()
    ctrl = torch.rand((3, big), generator=g, dtype=torch.float64, device="cuda")

    def jacobian(n):
        s = make_solver(flat, n)
        s.set_states_device(init[:n].contiguous().data_ptr())
        c = ctrl[:, :n].contiguous()
        jac = torch.full((21, 24, n), float("nan"), dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        assert s.step_jacobian(c.data_ptr(), jac.data_ptr()) == (21, 24)
        s.synchronize()
        s.close()
        return jac

    ref = jacobian(big)
    assert torch.isfinite(ref).all()
    for n in (1, 64, 65):
        assert torch.equal(jacobian(n), ref[..., :n]), n


@pytest.mark.parametrize("dof,n", [(11, 40_000), (18, 20_000), (18, 65_536), (24, 40_000)])
def test_functor_launches_take_the_one_lane_occupancy(dof, n):
    """A caller's controls functor has one-lane kernels only: one wavefront per SIMD on fleets that fill no more,
    whatever the lane-group kernels of such a fleet are built for."""
    s = fleet(dof, False, n)
    size, block, grid, stream = 8, ctypes.c_int(), ctypes.c_int(), ctypes.c_void_p()
    begin = lib.lfdm_functor_chunk_begin
    begin.argtypes = [ctypes.c_void_p, ctypes.c_double, ctypes.c_int, ctypes.c_void_p, ctypes.c_int] + [ctypes.c_void_p] * 3
    out = [ctypes.addressof(v) for v in (block, grid, stream)]
    raw = (ctypes.c_char * 4096)()
    while begin(s._h, 0.0, 1, raw, size, *out) != 0:
        size += 8
        assert size < 4096
    _, waves, lanes, strict = np.frombuffer(raw, np.int32, 4, size - 16)  # the launch record's last fields
    s.close()
    assert (waves, lanes, strict) == (1, 1, 0)
