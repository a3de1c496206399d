"""The one-kernel reverse sweep of the small systems against gradients it gave before, bit for bit.

The sweep goes through powers of error ratios that are themselves near rounding, so the order of its sums -- an iteration's
evaluation points one by one into the cotangents of the stages -- decides a sample's float32 gradient to a few percent.
Results from one build to the next therefore differ visibly unless that order is kept; nothing on the CPU has the same
bits to compare with (torch sums the same terms in another order), hence the stored values.

    python tests/test_reverse_sweep_bits_gpu.py

writes tests/stored/reverse_sweep_gradients.json on a machine with a GPU (float.hex of every value)."""
import json
import os
import sys

import pytest
import torch

if __name__ != "__main__":
    pytestmark = pytest.mark.gpu
GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "stored", "reverse_sweep_gradients.json")

# (system, features, method, controller, dtype, evaluation points)
CASES = {
    "vdp-f32-tsit5-pid": ("vdp", 2, "Tsit5", "pid", "float32", 50),
    "vdp-f64-dopri5-integral": ("vdp", 2, "Dopri5", "integral", "float64", 33),
    "vdp-f32-dopri5-pid-end": ("vdp", 2, "Dopri5", "pid", "float32", 0),
    "lorenz-f32-dopri5-integral": ("lorenz", 3, "Dopri5", "integral", "float32", 20),
    "lorenz-f64-tsit5-pid": ("lorenz", 3, "Tsit5", "pid", "float64", 41),
    "decay1-f32-tsit5-integral": ("decay", 1, "Tsit5", "integral", "float32", 25),
    "decay3-f64-tsit5-integral": ("decay", 3, "Tsit5", "integral", "float64", 40),
    "decay4-f32-dopri5-integral": ("decay", 4, "Dopri5", "integral", "float32", 30),
    "decay8-f32-tsit5-pid": ("decay", 8, "Tsit5", "pid", "float32", 30),
}
B = 19


def gradients(case):
    """y0's and the parameters' gradients, of the first solve of a solver and of the second (their records come from different
    kernels, with the same bits in them)."""
    import torchode_amd as to

    system, F, method, control, dtype, E = CASES[case]
    dtype = getattr(torch, dtype)
    g = torch.Generator().manual_seed(7)
    rand = lambda lo, hi, *shape: (lo + (hi - lo) * torch.rand(shape, generator=g, dtype=torch.float64)).to(dtype).cuda()
    y0, t1 = rand(-1.5, 1.5, B, F).requires_grad_(), rand(1.0, 3.0, B)
    par, f = {"vdp": (rand(0.5, 5.0, B), to.VanDerPol), "lorenz": (rand(20.0, 30.0, B), to.Lorenz63), "decay": (rand(0.1, 5.0, B, F), to.LinearDecay)}[system]
    cotangent = rand(-1.0, 1.0, B, max(E, 1), F)
    par.requires_grad_()
    if system == "lorenz":
        t1 = t1 * 0.25
    # (multiples of 1/64: the same values wherever they are formed)
    times = dict(t_eval=t1[:, None] * (torch.arange(E, device="cuda").to(dtype) / 64)) if E else dict(t_start=torch.zeros_like(t1), t_end=t1)
    controller = to.PIDController(1e-6, 1e-4, 0.2, 0.5, 0.05) if control == "pid" else to.IntegralController(1e-5, 1e-3)
    solver = to.AutoDiffAdjoint(getattr(to, method)(), controller)
    for attempt in range(2):
        sol = solver.solve(to.InitialValueProblem(y0, **times), to.ODETerm(f(par)))
        assert int(sol.status.abs().sum()) == 0
        yield torch.autograd.grad(sol.ys, [y0, par], cotangent)


@pytest.mark.parametrize("case", CASES)
def test_bits_of_the_gradients(case):
    with open(GOLDEN) as file:
        want = json.load(file)[case]
    for attempt, grads in enumerate(gradients(case)):
        for name, x, values in zip(("y0", "parameters"), grads, want):
            stored = torch.tensor([float.fromhex(v) for v in values], dtype=torch.float64)
            got = x.detach().double().cpu().flatten()
            assert bool(got.isfinite().all())
            assert torch.equal(got, stored), (attempt, name, float((got - stored).norm() / stored.norm()))


# (rows of four doubles hand over the most: 69 632 bytes of LDS)
IN_TWO = dict(CASES, **{"vdp-f64-tsit5-pid": ("vdp", 2, "Tsit5", "pid", "float64", 33), "decay4-f64-tsit5-pid": ("decay", 4, "Tsit5", "pid", "float64", 30), "decay4-f64-dopri5-integral": ("decay", 4, "Dopri5", "integral", "float64", 30)})


@pytest.mark.parametrize("case", ["vdp-f32-tsit5-pid", "vdp-f64-dopri5-integral", "vdp-f64-tsit5-pid", "lorenz-f32-dopri5-integral", "lorenz-f64-tsit5-pid", "decay1-f32-tsit5-integral", "decay4-f32-dopri5-integral",
                                  "decay3-f64-tsit5-integral", "decay4-f64-tsit5-pid", "decay4-f64-dopri5-integral"])  # fmt: skip
def test_one_wavefront_and_two(case):
    """Samples of a batch of 1025 groups of 64 (one wavefront to a group) and the same in batches of 1 to 512 groups (two), of 513
    and of 1024 (two in float32): the same gradients, bit for bit, points in order and swapped, some samples over before the others."""
    import torchode_amd as to

    system, F, method, control, dtype, E = IN_TWO[case]
    dtype, B = getattr(torch, dtype), 1025 * 64 - 5
    g = torch.Generator("cuda").manual_seed(11)
    rand = lambda lo, hi, *shape: (lo + (hi - lo) * torch.rand(shape, generator=g, dtype=torch.float64, device="cuda")).to(dtype)
    y0, t1 = rand(-1.5, 1.5, B, F), rand(0.5, 1.5, B) * (0.25 if system == "lorenz" else 1)
    t1[7::64] *= 1e-3
    par, f = {"vdp": (rand(0.5, 3.0, B), to.VanDerPol), "lorenz": (rand(20.0, 30.0, B), to.Lorenz63), "decay": (rand(0.1, 5.0, B, F), to.LinearDecay)}[system]
    cotangent = rand(-1.0, 1.0, B, max(E, 1), F)
    t_eval = t1[:, None] * (torch.arange(E, device="cuda").to(dtype) / 64) if E else None
    if E:
        t_eval[64 * 3 + 2] = t_eval[64 * 3 + 2].flip(0)
    controller = to.PIDController(1e-6, 1e-4, 0.2, 0.5, 0.05) if control == "pid" else to.IntegralController(1e-5, 1e-3)

    def gradients_of(rows):
        y, p = y0[rows].clone().requires_grad_(), par[rows].clone().requires_grad_()
        times = dict(t_start=torch.zeros_like(t1[rows]), t_end=t1[rows]) if not E else dict(t_eval=t_eval[rows], t_start=torch.zeros_like(t1[rows]), t_end=t1[rows])
        sol = to.AutoDiffAdjoint(getattr(to, method)(), controller).solve(to.InitialValueProblem(y, **times), to.ODETerm(f(p)))
        assert not sol.status.any()
        return [sol.ys.detach(), sol.stats["n_steps"], *torch.autograd.grad(sol.ys, [y, p], cotangent[rows])]

    whole = gradients_of(slice(0, B))
    for rows in (slice(0, 1), slice(60, 391), slice(128, 128 + 64 * 64), slice(B - 64 * 512, B), slice(0, 64 * 512 + 1), slice(0, 64 * 1024)):
        for found, expected in zip(gradients_of(rows), whole):
            assert torch.equal(found, expected[rows]), (case, rows)


if __name__ == "__main__":
    result = {case: [[float(v).hex() for v in x.double().flatten().tolist()] for x in next(gradients(case))] for case in CASES}
    with open(sys.argv[1] if len(sys.argv) > 1 else GOLDEN, "w") as file:
        json.dump(result, file, indent=0)
        file.write("\n")
