"""The two-wavefront kernel with a sample's features on lanes of their own (the choice for small batches): the edges of its
groups of 32 and 16 samples and of the batch sizes that take it, against the scalar C oracle and the other kernels."""
import pytest
import torch

import torchode_amd as to
from helpers import assert_identical, c_oracle_solve, gpu_solve
from torchode_amd import _lib

pytestmark = pytest.mark.gpu
PID = dict(kind="pid", atol=1e-6, rtol=1e-4, pcoeff=0.2, icoeff=0.5, dcoeff=0.05)


def lanes_solve(*args, **kwargs):
    """gpu_solve with this form asked for (an error where it does not cover the problem)."""
    real = _lib.set_fast_kernel_variant
    _lib.set_fast_kernel_variant = lambda v: real(3 if v == 2 else v)
    try:
        return gpu_solve(*args, fast="two", **kwargs)
    finally:
        _lib.set_fast_kernel_variant = real


def problem(name, B, dtype, E):
    if name.startswith("linear_decay"):
        F = int(name[-1])
        g = torch.Generator().manual_seed(B)
        f = to.LinearDecay((torch.rand((B, F), generator=g, dtype=torch.float64) * 5 + 0.1).to(dtype))
        y0 = torch.randn((B, F), generator=g, dtype=torch.float64).to(dtype)
        t1 = torch.rand((B, 1), generator=g, dtype=torch.float64) + 1
    else:
        w = to.workloads.make(name, batch=B, dtype=dtype)
        f, y0, t1 = w.f, w.y0, 0.25 * w.t_eval[:, -1:].double()
    return f, y0, (t1 * torch.linspace(0, 1, E, dtype=torch.float64)[None, :]).to(dtype)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("B", [1, 15, 17, 31, 33, 65])
@pytest.mark.parametrize("name", ["vdp", "lorenz", "linear_decay2", "linear_decay3", "linear_decay4"])
def test_groups_that_are_not_full(name, B, dtype):
    f, y0, t_eval = problem(name, B, dtype, 7)
    t_eval[::2] = t_eval[::2, -1:] - t_eval[::2]  # every other sample backwards in time
    if name == "lorenz":
        t_eval *= 0.05
    for method, spec in (("tsit5", PID), ("dopri5", dict(kind="integral", atol=1e-5, rtol=1e-3))):
        assert_identical(lanes_solve(f, y0, t_eval, method, spec), c_oracle_solve(f, y0, t_eval, method, spec))


@pytest.mark.parametrize("name,dtype,last", [("vdp", torch.float32, 32768), ("lorenz", torch.float64, 8192), ("linear_decay2", torch.float32, 12288), ("linear_decay4", torch.float64, 16384)])
def test_last_batch_size_of_the_form(name, dtype, last):
    f, y0, t_eval = problem(name, last + 1, dtype, 5)
    cut = lambda x, n: None if x is None else x[:n].contiguous()
    g = {to.VanDerPol: lambda n: to.VanDerPol(f.mu[:n]), to.Lorenz63: lambda n: to.Lorenz63(f.rho[:n]), to.LinearDecay: lambda n: to.LinearDecay(f.k[:n])}[type(f)]
    ref = gpu_solve(f, y0, t_eval, "tsit5", PID, fast="one")
    sol = lanes_solve(g(last), cut(y0, last), cut(t_eval, last), "tsit5", PID)
    assert torch.equal(sol.ys, ref.ys[:last]) and all(torch.equal(sol.stats[k].cpu(), ref.stats[k][:last].cpu()) for k in ("n_steps", "n_accepted", "n_initialized"))
    assert _lib.last_solve_kernel_name() == "tode::solve_pair_kernel"
    after = lanes_solve(f, y0, t_eval, "tsit5", PID)  # (one sample more is not covered: the call goes to the general kernel)
    assert _lib.last_solve_kernel_name() == "tode::solve_kernel"
    assert torch.equal(after.ys, ref.ys)


# Evaluation points of 32 samples (lanes) or 64 (one sample per lane) per workgroup, beside step records of 6 to 21 KB in LDS: numbers of
# points that a small batch keeps there too, with 64 KB and up to the last byte of its budget, and the next one, which
# is read from memory.
@pytest.mark.parametrize("form, dtype, n_eval", [
    ("lanes", torch.float32, 700), ("lanes", torch.float32, 1226), ("lanes", torch.float32, 1227), ("lanes", torch.float64, 588), ("lanes", torch.float64, 589),
    ("two", torch.float32, 300), ("two", torch.float32, 594), ("two", torch.float32, 595), ("two", torch.float64, 275), ("two", torch.float64, 276),
], ids=str)  # fmt: skip
def test_evaluation_points_up_to_the_size_of_lds(form, dtype, n_eval):
    f, y0, t_eval = problem("vdp", 70, dtype, n_eval)
    solve = lanes_solve if form == "lanes" else lambda *args: gpu_solve(*args, fast="two")
    for method, spec in (("tsit5", PID), ("dopri5", dict(kind="integral", atol=1e-5, rtol=1e-3))):
        assert_identical(solve(f, y0, t_eval, method, spec), c_oracle_solve(f, y0, t_eval, method, spec))
        assert _lib.last_solve_kernel_name() == "tode::solve_pair_kernel"


def test_rows_of_more_than_two_to_the_24_values():
    """Offsets into a workgroup's block of the output are 32 bits wide: 32 samples of that many values are within them."""
    f, y0, t_eval = problem("vdp", 2, torch.float32, 2**23 + 1)
    ref = c_oracle_solve(f, y0, t_eval, "tsit5", PID)
    assert_identical(gpu_solve(f, y0, t_eval, "tsit5", PID), ref)
    assert _lib.last_solve_kernel_name() == "tode::solve_pair_kernel"
