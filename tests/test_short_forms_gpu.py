"""The whole-solve kernels of the small systems take short forms of the division, the square root, the logarithm and the
exponential where an iteration's operands are in their ranges, and the general forms otherwise: results at and across the
edges of those ranges against the scalar C oracle, bit for bit."""
import pytest
import torch

import torchode_amd as to
from helpers import assert_identical, c_oracle_solve, gpu_solve

pytestmark = pytest.mark.gpu

# (tolerances and exponents: inside the ranges; at their edges; absolute tolerance zero or below 2^-40; relative tolerance
# above 1/16; exponents of the error ratio above 1/2)
CONTROLLERS = {
    "inside": dict(kind="pid", atol=1e-6, rtol=1e-4, pcoeff=0.2, icoeff=0.5, dcoeff=0.05),
    "edge": dict(kind="pid", atol=2.0**-40, rtol=2.0**-4, pcoeff=1.0, icoeff=1.5, dcoeff=0.0),
    "tiny-atol": dict(kind="integral", atol=1e-13, rtol=1e-4),
    "large-rtol": dict(kind="integral", atol=1e-4, rtol=0.07),
    "steep": dict(kind="pid", atol=1e-5, rtol=1e-3, pcoeff=1.2, icoeff=1.6, dcoeff=0.1),
}


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("controller", CONTROLLERS)
@pytest.mark.parametrize("name,method", [("vdp", "tsit5"), ("lorenz", "dopri5"), ("linear_decay", "tsit5"), ("linear_decay", "dopri5")])
def test_ranges_of_the_controller(name, method, controller, dtype):
    w = to.workloads.make(name, batch=130, dtype=dtype)
    spec = CONTROLLERS[controller]
    ref = c_oracle_solve(w.f, w.y0, w.t_eval, method, spec)
    for fast in ("one", True):
        assert_identical(gpu_solve(w.f, w.y0, w.t_eval, method, spec, fast=fast), ref)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("features", [1, 2, 3, 4, 8])
def test_scaled_errors_of_every_size(features, dtype):
    """Linear decay from states of 2^-140 ... 2^100 in one wavefront, some exactly zero: scaled errors that are zero, far
    below and above the range of the short forms, next to ordinary ones; evaluation points from the first step on."""
    B = 97
    g = torch.Generator().manual_seed(5)
    exponent = torch.linspace(-140, 100, B, dtype=torch.float64)[torch.randperm(B, generator=g)]
    y0 = (torch.randn((B, features), generator=g, dtype=torch.float64) * 2.0 ** exponent[:, None]).to(dtype)
    y0[::7, 0] = 0.0
    y0[5] = 0.0
    f = to.LinearDecay((torch.rand((B, features), generator=g, dtype=torch.float64) * 3 + 0.1).to(dtype))
    t_eval = (torch.rand((B, 1), generator=g, dtype=torch.float64) * torch.tensor([[0.0, 1e-30, 1e-9, 0.01, 0.3, 0.31, 0.9, 1.0]], dtype=torch.float64)).to(dtype)
    spec = dict(kind="pid", atol=1e-6, rtol=1e-4, pcoeff=0.2, icoeff=0.5, dcoeff=0.05)
    for method in ("dopri5", "tsit5"):
        ref = c_oracle_solve(f, y0, t_eval, method, spec)
        for fast in ("one", True):
            assert_identical(gpu_solve(f, y0, t_eval, method, spec, fast=fast), ref)


@pytest.mark.parametrize("form", range(10), ids=[f"{name}-{dtype}" for dtype in ("f32", "f64") for name in ("reciprocal", "root", "over-root-2", "over-root-3", "quotient")])
def test_forms_against_the_compilers(form):
    """float32 over every value of the form's range, float64 and quotients on 2^28 pseudo-random operands: not one result
    that differs from the division's or the square root's (ids in the order of the library's forms)."""
    from torchode_amd import _lib

    mismatches = torch.zeros(1, dtype=torch.int32, device="cuda")
    _lib.check(_lib.load().tode_check_short_forms(form, 1 << 28, mismatches.data_ptr(), _lib.stream_of(mismatches)), "tode_check_short_forms")
    assert int(mismatches) == 0


@pytest.mark.parametrize("form", [10, 11, 12, 13], ids=["power-f32", "power-f64", "sum-f32", "sum-f64"])
def test_powers_and_sums_against_their_general_forms(form):
    """2^26 pairs of a base -- any bits, or from around the short forms' range -- and an exponent of either kind; as many
    values summed over wavefronts."""
    from torchode_amd import _lib

    mismatches = torch.zeros(1, dtype=torch.int32, device="cuda")
    _lib.check(_lib.load().tode_check_short_forms(form, 1 << 26, mismatches.data_ptr(), _lib.stream_of(mismatches)), "tode_check_short_forms")
    assert int(mismatches) == 0


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("n", [16, 64])
@pytest.mark.parametrize("controller", CONTROLLERS)
def test_step_factor_of_a_grid(controller, n, dtype):
    """The grid kernel forms the powers of its step factor on lanes of one wavefront; the per-call operators form them one
    after the other: the same bits, whichever exponents are zero or outside the short forms' range."""
    spec = dict(CONTROLLERS[controller])
    B, F = 5, n * n
    g = torch.Generator().manual_seed(n)
    y0 = torch.rand((B, F), generator=g, dtype=torch.float64).to(dtype).cuda()
    f = to.ReactionDiffusion(torch.tensor([1e-3, 3e-3, 1e-2, 3e-2, 1e-1], dtype=dtype).cuda(), n)
    t_eval = torch.linspace(0.0, 1.0, 7, dtype=dtype).repeat(B, 1).cuda()
    make = to.PIDController if spec.pop("kind") == "pid" else to.IntegralController
    solver = to.AutoDiffAdjoint(to.Tsit5(), make(**spec))
    fused = solver.solve(to.InitialValueProblem(y0, t_eval=t_eval), to.ODETerm(f))
    per_call = solver._solve_protocol(to.InitialValueProblem(y0, t_eval=t_eval), to.ODETerm(f), to.ODETerm(f), None, None)
    assert torch.equal(fused.ys, per_call.ys) and torch.equal(fused.status, per_call.status)
    for key in ("n_steps", "n_accepted", "n_initialized"):
        assert torch.equal(fused.stats[key], per_call.stats[key])
