"""What this solver's users have it do, as cases that can be timed: whole solves of a batch of initial value problems
through ``AutoDiffAdjoint.solve``, forward and with gradients, with the built-in right-hand sides and with a user's own.

``listed()`` names the standing cases, ``draw(rng)`` gives another one of the same ranges, ``prepare(case, seed)`` makes
what a program has in hand before the call (tensors on the GPU, the term, the solver), ``run(state)`` is one solve (or one
solve and its backward pass), ``work(case)`` what it cannot do without and ``tolerance(case)`` how far two correct results
may be apart.  The distributions are those of ``torchode_amd.workloads`` (there drawn on the CPU for parity fixtures, here
on the GPU from the seed); the fixed sizes are the benchmark's configurations and sizes of the tests between them.
"""
import math

import torch

import torchode_amd as to

# Adaptive steps a sample takes on average (counted on these distributions): enters the estimate of the work only.
MEAN_STEPS = {"decay": 12, "vdp": 67, "lorenz": 31, "diffusion": 3, "network": 3}
CONTROL = {
    "decay": dict(atol=1e-6, rtol=1e-3),
    "vdp": dict(atol=1e-6, rtol=1e-4),
    "lorenz": dict(atol=1e-5, rtol=1e-3),
    "diffusion": dict(atol=1e-5, rtol=1e-3),
    "network": dict(atol=1e-5, rtol=1e-3),
}


def _case(system, B, F, E, *, H=0, use="solve", f="builtin", dtype="f32", method="dopri5", control="integral", inputs="float32", through_control=True):
    """system: which differential equation; B: batch, F: state values per sample, E: evaluation points (0: the end point
    alone), H: hidden units of the network; use: "solve" or "gradient" (solve and backward pass); f: "builtin" or
    "callable" (the same equation as a user's own function of torch operations); inputs: of the network's matrix products;
    through_control: whether gradients count the step sizes as functions of the inputs (the library's default)."""
    return dict(
        system=system, B=B, F=F, E=E, H=H, use=use, f=f, dtype=dtype, method=method, control=control, inputs=inputs, through_control=through_control
    )


def listed():
    pid = dict(method="tsit5", control="pid")
    return [
        # a small problem in double precision, as in a notebook or a test: launches and latency are all there is
        dict(_case("decay", 256, 4, 10, dtype="f64"), name="decay_f64_small"),
        # the benchmark's headline: a parameter study of a two-dimensional oscillator
        dict(_case("vdp", 65536, 2, 50, **pid), name="vdp_f32"),
        # the same in double precision, a batch that fills no power of two
        dict(_case("vdp", 20011, 2, 33, dtype="f64", **pid), name="vdp_f64_ragged"),
        # an ensemble of a million trajectories of a three-dimensional system
        dict(_case("lorenz", 1048576, 3, 20), name="lorenz_f32_large"),
        # the same system where only the state at t_end is asked for
        dict(_case("lorenz", 40009, 3, 0), name="lorenz_f32_end_point"),
        # a discretised partial differential equation: long rows, a dense output of most of a gigabyte
        dict(_case("diffusion", 512, 64 * 64, 100, **pid), name="diffusion_f32"),
        # a neural differential equation: inference with float32 matrix products
        dict(_case("network", 4096, 64, 20, H=256), name="network_f32"),
        # the reduced-precision variant on a larger, ragged batch
        dict(_case("network", 20011, 64, 20, H=256, inputs="bfloat16"), name="network_bf16_ragged"),
        # sensitivities of the oscillator to its start and its parameter: forward and backward
        dict(_case("vdp", 65536, 2, 50, use="gradient", **pid), name="vdp_f32_gradient"),
        # one training step's solve and backward pass of the neural differential equation
        dict(_case("network", 4096, 64, 20, H=256, use="gradient"), name="network_f32_training"),
        # a right-hand side that the user wrote in torch operations, many small steps
        dict(_case("vdp", 4096, 2, 50, f="callable", **pid), name="user_vdp_f32"),
        # a user's own torch network as right-hand side, few steps on longer rows
        dict(_case("network", 4096, 64, 20, H=256, f="callable"), name="user_network_f32"),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(["decay", "vdp", "vdp", "lorenz", "lorenz", "diffusion", "network", "network", "small_gradient", "network_gradient", "user"])
    steps = dict(method=rng.choice(["dopri5", "tsit5"]), control=rng.choice(["integral", "pid"]))
    dtype = rng.choice(["f32", "f32", "f64"])
    E = rng.choice([0, rng.randint(2, 60), rng.randint(2, 60), rng.randint(2, 60)])
    if kind == "decay":
        return _case("decay", _log_int(rng, 17, 200000), rng.choice([1, 2, 3, 4, 8]), rng.randint(2, 40), dtype=dtype, **steps)
    if kind == "vdp":
        return _case("vdp", _log_int(rng, 100, 120000), 2, E, dtype=dtype, **steps)
    if kind == "lorenz":
        return _case("lorenz", _log_int(rng, 100, 120000 if E == 0 else 900000), 3, min(E, 30), dtype=dtype, **steps)
    if kind == "diffusion":
        n = rng.choice([16, 32, 64, 64])
        return _case("diffusion", _log_int(rng, 9, 500 * (64 // n) ** 2 // (2 if dtype == "f64" else 1)), n * n, rng.randint(2, 100), dtype=dtype, **steps)
    if kind == "network":
        steps["control"] = "integral"
        F, H = rng.choice([(64, 256), (64, 256), (rng.randint(4, 63), rng.randint(16, 255))])
        return _case("network", _log_int(rng, 100, 60000), F, rng.randint(2, 40), H=H, inputs=rng.choice(["float32", "float32", "bfloat16"]), **steps)
    if kind == "small_gradient":
        system, F = rng.choice([("vdp", 2), ("vdp", 2), ("decay", 4), ("decay", 3)])
        return _case(system, _log_int(rng, 100, 60000), F, rng.randint(2, 50), use="gradient", dtype=dtype, **steps)
    if kind == "network_gradient":
        steps["control"] = "integral"
        F, H = rng.choice([(64, 256), (64, 256), (rng.randint(4, 63), rng.randint(16, 255))])
        return _case("network", _log_int(rng, 60, 12000), F, rng.randint(2, 30), H=H, use="gradient", through_control=rng.random() < 0.5, **steps)
    if rng.random() < 0.5:
        return _case("vdp", _log_int(rng, 100, 4000), 2, rng.randint(2, 50), f="callable", dtype=dtype, **steps)
    return _case("network", _log_int(rng, 100, 4000), rng.randint(8, 100), rng.randint(2, 40), H=rng.randint(16, 256), f="callable", **steps)


def prepare(case, seed):
    B, F, E, H = case["B"], case["F"], case["E"], case["H"]
    dtype = torch.float64 if case["dtype"] == "f64" else torch.float32
    g = torch.Generator("cuda").manual_seed(seed)
    rand = lambda *shape: torch.rand(shape, generator=g, dtype=torch.float64, device="cuda")
    randn = lambda *shape: torch.randn(shape, generator=g, dtype=torch.float64, device="cuda")
    uniform = lambda a, b, *shape: a + (b - a) * rand(*shape)
    log_uniform = lambda a, b, *shape: uniform(math.log(a), math.log(b), *shape).exp()
    system, gradient = case["system"], case["use"] == "gradient"
    if system == "decay":
        params, y0, t1 = [log_uniform(0.1, 10.0, B, F)], randn(B, F), uniform(5.0, 5.0, B)
    elif system == "vdp":
        params, y0, t1 = [uniform(0.5, 5.0, B)], uniform(-2.0, 2.0, B, F), uniform(8.0, 12.0, B)
    elif system == "lorenz":
        params, y0, t1 = [uniform(20.0, 30.0, B)], randn(B, F) + torch.tensor([0.0, 1.0, 20.0], dtype=torch.float64, device="cuda"), uniform(2.0, 2.0, B)
    elif system == "diffusion":
        n = math.isqrt(F)
        params, t1 = [log_uniform(1e-3, 1e-1, B)], uniform(1.0, 1.0, B)
        y0 = uniform(0.0, 1.0, B, n, n).to(dtype)
        kernel = torch.exp(-0.125 * torch.arange(-6, 7, device="cuda", dtype=torch.float64) ** 2)
        for dim in (1, 2):  # a smooth field: one separable periodic blur of width 2
            y0 = sum(float(w / kernel.sum()) * torch.roll(y0, s - 6, dim) for s, w in enumerate(kernel))
        y0 = y0.reshape(B, F)
    else:
        bound1, bound2 = math.sqrt(6.0 / (F + 1 + H)), math.sqrt(6.0 / (H + F))
        params = [uniform(-bound1, bound1, H, F + 1), torch.zeros(H, device="cuda"), uniform(-bound2, bound2, F, H), torch.zeros(F, device="cuda")]
        y0, t1 = randn(B, F), uniform(1.0, 1.0, B)
    params = [p.to(dtype).contiguous() for p in params]
    y0, t1 = y0.to(dtype).contiguous(), t1.to(dtype)
    state = dict(y0=y0, params=params, gradient=gradient)
    if E > 0:
        frac = torch.arange(E, dtype=torch.float64, device="cuda") / (E - 1)
        state["times"] = dict(t_eval=(t1.double()[:, None] * frac[None, :]).to(dtype).contiguous())
    else:
        state["times"] = dict(t_start=torch.zeros_like(t1), t_end=t1)
    if gradient:
        for x in [y0, *params]:
            x.requires_grad_()
        state["cotangent"] = randn(B, E, F).to(dtype)  # d loss / d ys

    if case["f"] == "callable" and system == "vdp":
        (mu,) = params
        f = lambda t, y: torch.stack((y[:, 1], mu * (1 - y[:, 0] ** 2) * y[:, 1] - y[:, 0]), dim=1)
    elif case["f"] == "callable":
        W1, b1, W2, b2 = params
        f = lambda t, y: torch.nn.functional.linear(torch.tanh(torch.nn.functional.linear(torch.cat((y, t[:, None]), dim=1), W1, b1)), W2, b2)
    elif system == "network":
        f = to.MLPField(*params, matrix_inputs=case["inputs"])
    elif system == "diffusion":
        f = to.ReactionDiffusion(params[0], math.isqrt(F))
    else:
        f = {"decay": to.LinearDecay, "vdp": to.VanDerPol, "lorenz": to.Lorenz63}[system](params[0])
    state["term"] = to.ODETerm(f)
    tolerances = CONTROL[system]
    controller = to.PIDController(**tolerances, pcoeff=0.2, icoeff=0.5, dcoeff=0.0) if case["control"] == "pid" else to.IntegralController(**tolerances)
    state["solver"] = to.AutoDiffAdjoint(
        to.Tsit5() if case["method"] == "tsit5" else to.Dopri5(), controller, backprop_through_step_size_control=case["through_control"]
    )
    return state


def run(state):
    problem = to.InitialValueProblem(state["y0"], **state["times"])
    if not state["gradient"]:
        with torch.no_grad():
            solution = state["solver"].solve(problem, state["term"])
    else:
        solution = state["solver"].solve(problem, state["term"])
    out = dict(ys=solution.ys, status=solution.status, **solution.stats)
    if state["gradient"]:
        inputs = [state["y0"], *state["params"]]
        out["gradients"] = torch.autograd.grad(solution.ys, inputs, state["cotangent"])
        out["ys"] = solution.ys.detach()
    return out


def work(case):
    B, F, E, H = case["B"], case["F"], case["E"], case["H"]
    size = 8 if case["dtype"] == "f64" else 4
    per_sample = {"decay": F, "vdp": 1, "lorenz": 1, "diffusion": 1, "network": 0}[case["system"]]
    weights = H * (F + 1) + H + F * H + F if case["system"] == "network" else 0
    inputs = B * (F + max(E, 2) + per_sample) + weights
    values = inputs + B * max(E, 1) * F
    f_flops = {"decay": F, "vdp": 5, "lorenz": 8, "diffusion": 9 * F, "network": 2 * (H * (F + 1) + F * H)}[case["system"]]
    steps = MEAN_STEPS[case["system"]]
    flops = B * ((2 + 6 * steps) * f_flops + steps * 70 * F)
    if case["use"] == "gradient":  # ys' cotangent in; the gradients of y0 and the parameters out; the stages once more and their products
        values += B * E * F + B * (F + per_sample) + weights
        flops *= 4
    size_of_calls = 0
    if case["f"] == "callable":  # a user's f takes y and returns its derivative through memory
        size_of_calls = B * (2 + 6 * steps) * 2 * F * size
    return {"bytes": values * size + B * 4 * 8 + size_of_calls, "flops": flops}


def tolerance(case):
    # The small systems and the grid: every operation and its order is fixed (the results are those of the reference's
    # operations on the host, bit for bit, and the tests hold them to it), and the step sizes of an adaptive solve amplify
    # any other rounding: float32 against float64 of the same inputs differs in half of the step counts.
    if case["use"] == "solve" and (case["system"] != "network"):
        return "exact"
    # Their gradients, taken through the controller's powers of error ratios that are themselves near rounding: two of the
    # library's own reverse sweeps differ by up to 2e-2 (single samples by 0.6) in float32, by 1e-9 in float64.
    if case["system"] != "network":
        return {"rel": 3e-2, "max": 0.99} if case["dtype"] == "f32" else {"rel": 1e-6, "max": 1e-4}
    # bfloat16 matrix inputs: float32 against float64 sums move a few roundings of the hidden layer to the other side
    # (8e-4, single values 9e-3; 2e-2 of the step counts).
    if case["inputs"] == "bfloat16":
        return {"rel": 3e-3, "max": 4e-2, "differ": 8e-2}
    # Gradients of the network: float32 against float64 2e-4 (single values 3e-2 through the step sizes).
    if case["use"] == "gradient":
        return {"rel": 8e-4, "max": 0.12, "differ": 4e-3}
    # Matrix cores against the vendor library's products: 4e-6 (single values 2.4e-4; 1.2e-3 of the step counts).
    return {"rel": 1.6e-5, "max": 1e-3, "differ": 5e-3}
