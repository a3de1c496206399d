"""The reverse sweep's kernels for the perceptron (tode_mlp_stages, tode_mlp_stages_backward, tode_mlp_weight_gradients)
against the same sweep with torch's evaluations of the network and autograd's vector-Jacobian products, over the same
record, at the edges of their tiles: one sample, a full tile of 16 and one more, more tiles than workgroups; one
feature, rows that are no multiple of four, all 64; one hidden unit, 255, 256."""
import math
import types

import pytest
import torch

import torchode_amd as to
from torchode_amd import _lib

pytestmark = pytest.mark.gpu


def _gradients(B, F, H, E, method, controller, through, network, hook=False):
    g = torch.Generator("cuda").manual_seed(B + F + H)
    rand = lambda *shape: torch.rand(shape, generator=g, dtype=torch.float64, device="cuda")
    bound = lambda n, *shape: ((2 * rand(*shape) - 1) * math.sqrt(6.0 / n)).float().requires_grad_()
    weights = [bound(F + 1 + H, H, F + 1), bound(F + 1 + H, H), bound(F + H, F, H), bound(F + H, F)]
    y0 = (2 * rand(B, F) - 1).float().requires_grad_()
    t1 = (0.5 + 0.5 * rand(B)).float()
    times = dict(t_eval=(t1[:, None] * torch.linspace(0, 1, E, device="cuda")[None, :])) if E else dict(t_start=torch.zeros_like(t1), t_end=t1)
    f = to.MLPField(*weights)
    if hook:
        f.register_forward_hook(lambda module, inputs, output: 2 * output)
    solver = to.AutoDiffAdjoint(method(), controller(), backprop_through_step_size_control=through)
    solver.backward_network_kernels = network
    sol = solver.solve(to.InitialValueProblem(y0, **times), to.ODETerm(f))
    cotangent = (2 * rand(*sol.ys.shape) - 1).float()
    return torch.autograd.grad(sol.ys, [y0, *weights], cotangent)


@pytest.mark.parametrize("method, controller", [(to.Dopri5, lambda: to.IntegralController(1e-5, 1e-3)), (to.Tsit5, lambda: to.PIDController(1e-5, 1e-3, 0.2, 0.5, 0.0))],
                         ids=["dopri5-integral", "tsit5-pid"])  # fmt: skip
@pytest.mark.parametrize("B, F, H, E", [(1, 1, 1, 4), (16, 64, 256, 7), (17, 63, 255, 0), (33, 6, 3, 5), (4113, 64, 256, 3), (300, 4, 100, 20)])
def test_network_kernels_against_autograd(B, F, H, E, method, controller):
    """Same record, same decisions.  With the step sizes held constant the two differ by the roundings of float32 sums of at
    most 6 * 4113 rows or 256 units: 2^-24 times the square root of their number, with a factor of two in hand for
    products of several such sums, 2e-5 of the 2-norm.  Through the step size rule those are amplified by the
    derivatives of powers of error ratios (2e-2, as for the other pairs of sweeps)."""
    for through, bound in ((False, 2e-5), (True, 2e-2)):
        got = _gradients(B, F, H, E, method, controller, through, True)
        want = _gradients(B, F, H, E, method, controller, through, False)
        for a, b in zip(got, want):
            assert a.shape == b.shape and bool(a.isfinite().all())
            assert float((a.double() - b.double()).norm()) <= bound * float(b.double().norm()), (through, tuple(a.shape))


def test_a_hook_on_the_network_is_called():
    """A hook that doubles what the network returns: the sweep evaluates the module then, and both settings agree exactly."""
    got, want = (_gradients(17, 8, 16, 4, to.Dopri5, lambda: to.IntegralController(1e-5, 1e-3), False, network, hook=True) for network in (True, False))
    for a, b in zip(got, want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("B, F, H", [(1, 3, 5), (50, 64, 256)])
def test_a_solve_of_more_steps_than_the_first_record_holds(B, F, H):
    """Tight tolerances: more iterations than the record's first size, so the first solve is repeated with a longer one and
    the next solve of the same solver fits at once; every pass returns the same bits, and the gradients are those of the
    per-step path with torch's products.  (At these tolerances the error estimate is float32 rounding, so the two may take
    other steps: each is within 2^-24 times the some hundred roundings per step of 10 to 100 steps, 6e-4, of the same solution.)"""
    g = torch.Generator("cuda").manual_seed(B)
    rand = lambda *shape: (math.sqrt(6.0 / sum(shape)) * (2 * torch.rand(shape, generator=g, device="cuda") - 1)).requires_grad_()
    weights = [rand(H, F + 1), rand(H), rand(F, H), rand(F)]
    y0, cotangent = rand(B, F), rand(B, 6, F).detach()
    t_eval = torch.linspace(0, 3, 6, device="cuda").repeat(B, 1)
    results = {}
    for network in (True, False):
        solver = to.AutoDiffAdjoint(to.Tsit5(), to.IntegralController(1e-8, 1e-7), backprop_through_step_size_control=False)
        solver.backward_network_kernels = network
        for attempt in range(2):
            sol = solver.solve(to.InitialValueProblem(y0, t_eval=t_eval), to.ODETerm(to.MLPField(*weights)))
            assert int(sol.status.abs().sum()) == 0 and int(sol.stats["n_steps"].max()) > 8
            results[network, attempt] = torch.autograd.grad(sol.ys, [y0, *weights], cotangent)
        if network:
            assert list(solver._record_entries.values()) == [int(sol.stats["n_steps"].max()) + 5]
    for a, b, c in zip(results[True, 0], results[True, 1], results[False, 0]):
        assert torch.equal(a, b)
        assert float((a.double() - c.double()).norm()) <= 1e-3 * float(c.double().norm())


def test_gradient_of_y0_alone():
    """No weight wants a gradient: no outer products, and the same bits for y0."""
    g = torch.Generator("cuda").manual_seed(5)
    rand = lambda *shape: 2 * torch.rand(shape, generator=g, device="cuda") - 1
    B, F, H = 19, 10, 24
    weights = [rand(H, F + 1), rand(H), rand(F, H), rand(F)]
    y0, t_eval, cotangent = rand(B, F).requires_grad_(), torch.linspace(0, 1, 5, device="cuda").repeat(B, 1), rand(B, 5, F)
    results = []
    for wanted in (False, True):
        f = to.MLPField(*(w.clone().requires_grad_(wanted) for w in weights))
        solver = to.AutoDiffAdjoint(to.Tsit5(), to.IntegralController(1e-5, 1e-3))
        sol = solver.solve(to.InitialValueProblem(y0, t_eval=t_eval), to.ODETerm(f))
        results.append(torch.autograd.grad(sol.ys, y0, cotangent)[0])
    assert torch.equal(*results) and float(results[0].abs().max()) > 0


@pytest.mark.parametrize("times", [False, True], ids=["constant-times", "time-gradients"])
@pytest.mark.parametrize("F, E", [(64, 63), (64, 65), (100, 130), (64, 0)])
@pytest.mark.parametrize("method", [to.Dopri5, to.Tsit5], ids=["dopri5", "tsit5"])
def test_points_of_long_rows_as_sums(method, F, E, times):
    """The dense output's reverse on rows of a wavefront each, its marks looked at 64 at a time: fewer and more points than
    that, a row that is no multiple of 64, no points; against the sweep in torch operations (float64, the bound of the other
    comparisons of the two with the steps held constant)."""
    g = torch.Generator("cuda").manual_seed(F + E)
    rand = lambda *shape: torch.rand(shape, generator=g, dtype=torch.float64, device="cuda")
    B = 3
    rate, y0 = (0.5 + rand(F)).requires_grad_(), rand(B, F).requires_grad_()
    t1 = 0.5 + rand(B)
    if E:
        given = dict(t_eval=t1[:, None] * torch.linspace(0, 1, E, dtype=torch.float64, device="cuda")[None, :])
    else:
        given = dict(t_start=torch.zeros_like(t1), t_end=t1)
    given = {k: v.clone().requires_grad_(times) for k, v in given.items()}
    wrt = [rate, y0, *(given.values() if times else ())]
    cotangent = rand(B, max(E, 1), F)
    results = []
    for kernels in (True, False):
        solver = to.AutoDiffAdjoint(method(), to.IntegralController(1e-6, 1e-4), backprop_through_step_size_control=False)
        solver.backward_kernels = kernels
        sol = solver.solve(to.InitialValueProblem(y0, **given), to.ODETerm(lambda t, y: -rate * y * y + torch.sin(t)[:, None]))
        results.append(torch.autograd.grad(sol.ys, wrt, cotangent))
    for got, want in zip(*results):
        assert float((got - want).abs().max()) <= 1e-9 * float(want.abs().max())


@pytest.mark.parametrize("method", [to.Dopri5, to.Tsit5], ids=["dopri5", "tsit5"])
def test_points_of_long_rows_are_added_up_in_the_time_type(method):
    """float64 times and float32 data, a step with 100 000 points and the same cotangent at each: the gradient of t_start is
    -sum(g f) exactly, f being constant.  Added up in float32 it would be off by some 2^-24 per added point in one
    direction; the interpolant's coefficients (weights of up to 30, rounded to float32, where all but one should be zero)
    leave 30 * 2^-24 times a few."""
    E, F = 100_000, 64
    c = torch.arange(64, 64 + F, device="cuda") / 64
    t_eval = torch.linspace(0.001, 0.999, E, dtype=torch.float64, device="cuda").repeat(2, 1)
    t_start = torch.zeros(2, dtype=torch.float64, device="cuda", requires_grad=True)
    t_end, dt0 = torch.full_like(t_start, 2.0).detach(), torch.ones_like(t_start).detach()
    solver = to.AutoDiffAdjoint(method(), to.IntegralController(1e-5, 1e-3), backprop_through_step_size_control=False)
    y0 = torch.zeros(2, F, device="cuda")
    sol = solver.solve(to.InitialValueProblem(y0, t_start, t_end, t_eval), to.ODETerm(lambda t, y: c + 0 * y), dt0=dt0)
    (got,) = torch.autograd.grad(sol.ys, t_start, torch.full_like(sol.ys, 0.1))
    want = -float(torch.tensor(0.1)) * E * float(c.double().sum())
    assert float((got / want - 1).abs().max()) <= 1e-5


@pytest.mark.parametrize("method", [to.Dopri5, to.Tsit5], ids=["dopri5", "tsit5"])
def test_a_point_without_a_cotangent_adds_nothing(method):
    """A point so far in front of t_start that its position in the step is an infinity, and no cotangent at it, next to one
    that has one in the same step: gradients
    are those of the problem without the point."""
    B, F = 3, 70
    rate = torch.linspace(0.5, 1.5, F, device="cuda").requires_grad_()
    y0, t_start = torch.linspace(1, 2, B * F, device="cuda").reshape(B, F).requires_grad_(), torch.ones(B, device="cuda")
    points = torch.tensor([-3e38, 1.0001, 1.7, 2.0], device="cuda").repeat(B, 1)
    results = []
    for first in (0, 1):
        solver = to.AutoDiffAdjoint(method(), to.IntegralController(1e-5, 1e-3))
        sol = solver.solve(to.InitialValueProblem(y0, t_start, points[:, 3].contiguous(), points[:, first:].contiguous()), to.ODETerm(lambda t, y: -rate * y))
        cotangent = torch.ones_like(sol.ys)
        cotangent[:, : 1 - first] = 0
        results.append(torch.autograd.grad(sol.ys, [y0, rate], cotangent))
    for got, want in zip(*results):
        assert bool(want.isfinite().all()) and torch.equal(got, want)


def test_a_record_that_just_fits():
    """As many entries as the solve has iterations, and one for the state after them, are enough also where the sample with the
    most steps has landed past t_end and sits through one more iteration: the record is kept and the same."""
    g = torch.Generator("cuda").manual_seed(3)
    rand = lambda *shape: 2 * torch.rand(shape, generator=g, device="cuda") - 1
    B, F, H, E = 200, 8, 16, 5
    weights = [rand(H, F + 1), rand(H), rand(F, H), rand(F)]
    y0 = rand(B, F).requires_grad_()
    t_start, t_end = -0.3 - 0.1 * torch.rand(B, generator=g, device="cuda"), 1e-3 + 1e-3 * torch.rand(B, generator=g, device="cuda")
    t_eval = t_start[:, None] + (t_end - t_start)[:, None] * torch.linspace(0, 0.9, E, device="cuda")[None, :]
    solver = to.AutoDiffAdjoint(to.Dopri5(), to.IntegralController(1e-5, 1e-3))
    kept, real = [], solver._solve_recording_in_one_kernel
    solver._solve_recording_in_one_kernel = lambda *args: kept.append((real(*args), args[5])) or kept[-1][0]
    grads = []
    for attempt in range(2):
        sol = solver.solve(to.InitialValueProblem(y0, t_start, t_end, t_eval), to.ODETerm(to.MLPField(*weights)))
        grads.append(torch.autograd.grad(sol.ys, y0, torch.ones_like(sol.ys))[0])
        n = int(sol.stats["n_steps"].max())
        ((shape, entries),) = solver._record_entries.items()
        assert entries == n + 5
        solver._record_entries[shape] = n + 1
    assert [solution is not None for solution, _ in kept] == [True, True]
    record = kept[1][1].arrays
    assert record["t"].shape[0] == n + 1
    assert bool((record["t"][n] > t_end)[sol.stats["n_steps"] == n].any())  # (the case meant)
    for name, x in record.items():
        assert torch.equal(x, kept[0][1].arrays[name][: n + 1]), name
    assert torch.equal(*grads)


def test_memory_of_the_points_iterations(monkeypatch):
    """Which iteration wrote which point is found with memory for the times and the points, not for their product: 500 points
    and over 200 iterations of 1000 samples, 100 MB and more as one byte each, in a pass whose other buffers (rows of six
    evaluations, 12 MB, their outer products, 13 MB, two sets of cotangents, points, times) stay below 40 MB."""
    from torchode_amd.autodiff import NetworkSweep

    monkeypatch.setattr(NetworkSweep, "ROOM", 0)
    g = torch.Generator("cuda").manual_seed(2)
    rand = lambda *shape: 2 * torch.rand(shape, generator=g, device="cuda") - 1
    B, E = 1000, 500
    weights = [rand(4, 2).requires_grad_(), rand(4), rand(1, 4), rand(1)]
    t_eval = torch.linspace(0, 60, E, device="cuda").repeat(B, 1)
    solver = to.AutoDiffAdjoint(to.Tsit5(), to.IntegralController(1e-5, 1e-3, dt_max=0.3))
    problem, term = to.InitialValueProblem(rand(B, 1), t_eval=t_eval), to.ODETerm(to.MLPField(*weights))
    for attempt in range(2):
        sol = solver.solve(problem, term)
        assert int(sol.stats["n_steps"].max()) > 200
        torch.cuda.synchronize()
        held = torch.cuda.memory_allocated()
        torch.cuda.reset_peak_memory_stats()
        torch.autograd.grad(sol.ys, weights[0], torch.ones_like(sol.ys))
        assert torch.cuda.max_memory_allocated() - held < 40e6


def test_rows_that_do_not_fit_into_memory(monkeypatch):
    """Where the rows of all evaluations cannot be had the sweep takes those of one iteration at a time: the same gradient of y0,
    and the weights' with their rows added up in other shares (the bound of the comparison with autograd)."""
    case = (300, 64, 256, 9, to.Dopri5, lambda: to.IntegralController(1e-5, 1e-3), False, True)
    want = _gradients(*case)
    real, refused = torch.empty, []

    def empty(*args, **kwargs):
        shape = args[0] if args and isinstance(args[0], tuple) else ()
        if len(shape) == 3 and shape[0] > 7 and shape[1:] == (300, 256):  # (more than an iteration's evaluations of hidden units)
            refused.append(shape)
            raise torch.cuda.OutOfMemoryError("no room")
        return real(*args, **kwargs)

    monkeypatch.setattr(torch, "empty", empty)
    got = _gradients(*case)
    assert len(refused) == 1 and torch.equal(got[0], want[0])
    for a, b in zip(got, want):
        assert float((a.double() - b.double()).norm()) <= 2e-5 * float(b.double().norm())


@pytest.mark.parametrize("batch, points, iterations, sign", [(1, 1, 1, 1.0), (300, 7, 5, 1.0), (300, 7, 5, -1.0), (5, 3, 200, 1.0), (257, 64, 0, -1.0)])
def test_what_a_sweep_needs_of_its_record(batch, points, iterations, sign):
    """tode_mlp_sweep_begin against torch operations: points on recorded times, in front of the start and beyond the end, a first
    point at t_start, rejected steps (times that repeat), columns of a wider array as start and end, more points than
    iterations and the other way round."""
    g = torch.Generator().manual_seed(batch + points)
    steps = torch.rand(iterations, batch, generator=g) * (torch.rand(iterations, batch, generator=g) < 0.7)
    t = torch.cat([torch.randn(1, batch, generator=g), steps]).cumsum(0) if iterations else torch.randn(1, batch, generator=g)
    at = torch.rand(batch, points, generator=g) * (t[-1] - t[0])[:, None] * 1.4 + t[0][:, None] - 0.1
    on = torch.randint(0, iterations + 1, (batch, points), generator=g)
    at = torch.where(torch.rand(batch, points, generator=g) < 0.4, torch.gather(t.T, 1, on), at).sort(dim=1).values
    at[::2, 0] = torch.minimum(t[0], at[:, 0])[::2] if points > 1 else t[0][::2]
    t, at = sign * t, sign * at
    ends = torch.stack([t[0], t[0] + sign, t[0]], dim=1).contiguous().cuda()
    accepted = torch.cat([torch.zeros(1, batch, dtype=torch.int32), (steps > 0).to(torch.int32).cumsum(0).to(torch.int32)])
    later = sign * t[1:].T
    hit = torch.searchsorted(later.contiguous(), (sign * at).contiguous(), out_int32=True) if iterations else torch.zeros(batch, points, dtype=torch.int32)
    hit = torch.where(hit < iterations, hit, -1)
    hit[:, 0] = torch.where(at[:, 0] == t[0], -1, hit[:, 0])
    t_dev, at_dev, accepted_dev = t.contiguous().cuda(), at.contiguous().cuda(), accepted.cuda()
    new = lambda *shape, dtype=torch.int32: torch.full(shape, 7, dtype=dtype, device="cuda")
    hits, moved, t_start, t_end = new(batch, points), new(max(iterations, 1), batch), new(batch, dtype=torch.float32), new(batch, dtype=torch.float32)
    rc = _lib.load().tode_mlp_sweep_begin(
        batch, points, iterations, ends.data_ptr(), 3, ends.data_ptr() + 4, 3, at_dev.data_ptr(), t_dev.data_ptr(), accepted_dev.data_ptr(), hits.data_ptr(), moved.data_ptr(),
        t_start.data_ptr(), t_end.data_ptr(), _lib.stream_of(ends),
    )  # fmt: skip
    assert rc == 0
    assert torch.equal(hits.cpu(), hit) and torch.equal(t_start, ends[:, 0]) and torch.equal(t_end, ends[:, 1])
    if iterations:
        assert torch.equal(moved.cpu(), (accepted[1:] > accepted[:-1]).to(torch.int32))


def test_hidden_units_against_tanh_in_float64():
    """The gradient's kernels' tanh, seen through a network whose hidden unit u is tanh of state value u (one weight of one, the
    rest zeros: the matrix cores pass the value on exactly): magnitudes from 2^-20 to 10, the neighbours of 1, where its two forms
    meet, saturation and zero.  At most 2.5 units in the last place: 1.8 from the argument's, exponential's and reciprocal's
    roundings (a quarter of which reaches the result where the exponential form begins, less beyond) or 1.3 from the
    polynomial's, and half a unit from the last operation.  In the mean 0.35, where correct rounding has 0.25."""
    B = 4096
    g = torch.Generator("cuda").manual_seed(3)
    rand = lambda *shape: torch.rand(shape, generator=g, dtype=torch.float64, device="cuda")
    y = (2.0 ** (-20 + (20 + math.log2(10.0)) * rand(B, 64))).float()
    y[: B // 4] = (3 * torch.randn(B // 4, 64, generator=g, dtype=torch.float64, device="cuda")).float()
    near = (torch.ones(64, device="cuda").view(torch.int32) + torch.arange(-32, 32, device="cuda", dtype=torch.int32)).view(torch.float32)
    y[0], y[1], y[2] = near, -near, torch.linspace(8, 10, 64, device="cuda")
    y[3, :6] = torch.tensor([0.0, -0.0, 30.0, -30.0, 1e30, -1e30], device="cuda")
    y[4::2] = -y[4::2]
    W1 = torch.zeros(256, 65, device="cuda")
    W1[torch.arange(256), torch.arange(256) % 64] = 1.0
    zeros = lambda *shape: torch.zeros(shape, device="cuda")
    f = to.MLPField(W1, zeros(256), zeros(64, 256), zeros(64))
    packed = f.builtin_packed(y.device, torch.float32)
    t, dt, k0, k, inputs, times, hidden, unused = zeros(B), zeros(B), zeros(B, 64), zeros(6, B, 64), zeros(6, B, 64), zeros(6, B), zeros(6, B, 256) + 7, zeros(7, B, 64)
    p = _lib.MlpReverse(0, 64, 256, 1, B, packed.data_ptr(), packed.data_ptr(), t.data_ptr(), dt.data_ptr(), y.data_ptr(), k0.data_ptr(), k.data_ptr(), inputs.data_ptr(),
                        times.data_ptr(), hidden.data_ptr(), None, None, *([unused.data_ptr()] * 5))  # fmt: skip
    _lib.check(_lib.load().tode_mlp_stages(_lib.C.byref(p), _lib.stream_of(y)), "tode_mlp_stages")
    assert torch.equal(inputs, y.expand(6, B, 64))  # (steps of zero: every stage's input is the state)
    want = torch.tanh(y.double())
    _, exponent = torch.frexp(want)
    unit = torch.where(want == 0, 1.0, torch.ldexp(torch.ones_like(want), exponent - 24))
    off = (hidden.view(6, B, 4, 64).double() - want[None, :, None, :]).abs() / unit[None, :, None, :]
    print("units in the last place: most", float(off.max()), "mean", float(off.mean()))
    assert float(off.max()) <= 2.5 and float(off.mean()) <= 0.35


@pytest.mark.parametrize("control", ["integral", "pid"])
@pytest.mark.parametrize("points", ["usual", "many", "outside", "backwards", "few"])
@pytest.mark.parametrize("B, F, H", [(1, 1, 1), (17, 63, 255), (64, 4, 20), (4113, 64, 256)])
def test_all_iterations_in_one_kernel(monkeypatch, B, F, H, points, control):
    """The sweep over a whole record against the launches per iteration that the same cotangents take where times want gradients
    too: with the step sizes held constant the gradient of y0 bit for bit (rows of 64; shorter ones are swept by one thread, point by
    point), and the weights' from the same rows; through the step sizes, whose sums over a sample's features are added up in another order, to the bound of the comparison with autograd.
    Points: more than a wavefront has lanes, in front of the start and beyond the end, backwards in time, one alone; a cotangent at
    an address that is no multiple of 16 bytes, some of it zero."""
    from torchode_amd.autodiff import NetworkSweep

    g = torch.Generator("cuda").manual_seed(B + F)
    rand = lambda *shape: torch.rand(shape, generator=g, device="cuda")
    weights = [(math.sqrt(6.0 / (F + H)) * (2 * rand(*shape) - 1)).requires_grad_() for shape in ((H, F + 1), (H,), (F, H), (F,))]
    y0 = (2 * rand(B, F) - 1).requires_grad_()
    E = {"usual": 9, "many": 130, "outside": 12, "backwards": 7, "few": 2}[points]
    t1 = 0.5 + rand(B)
    at = t1[:, None] * torch.linspace(0, 1, E, device="cuda")
    if points == "outside":
        at = t1[:, None] * torch.linspace(0, 1.3, E, device="cuda")
        at[:, 0] = -1e-3  # (a tenth of a first step or less: powers of large positions cancel to nothing in either sweep)
    if points == "backwards":
        at, t1 = -at, -t1
    times = dict(t_eval=at, t_start=torch.zeros_like(t1), t_end=t1)
    cotangent = torch.empty(B * E * F + 1, device="cuda")[1:].view(B, E, F)
    cotangent.copy_((2 * rand(B, E, F) - 1) * (rand(B, E, 1) < 0.8))
    assert cotangent.data_ptr() % 16 and cotangent.is_contiguous()
    make = lambda: to.PIDController(1e-5, 1e-3, 0.2, 0.5, 0.05) if control == "pid" else to.IntegralController(1e-5, 1e-3)
    whole, calls = NetworkSweep.whole, []
    for through, bound in ((False, 2e-5), (True, 2e-2)):
        results = []
        for one_kernel in (True, False):
            monkeypatch.setattr(NetworkSweep, "whole", lambda *a: calls.append(whole(*a)) or calls[-1] if one_kernel else None)
            solver = to.AutoDiffAdjoint(to.Tsit5() if control == "pid" else to.Dopri5(), make(), backprop_through_step_size_control=through)
            sol = solver.solve(to.InitialValueProblem(y0, **times), to.ODETerm(to.MLPField(*weights)))
            assert not sol.status.any()
            results.append(torch.autograd.grad(sol.ys, [y0, *weights], cotangent))
        if not through and F == 64:
            assert torch.equal(results[0][0], results[1][0])
        for a, b in zip(*results):
            # (a single sample's sum over the points may cancel: the roundings of its terms, at most the root of their number times
            # the cotangent's norm, 2^-22 with the products behind them, are those of a result that does not)
            cancelled = bound / 2e-5 * 2.0**-22 * math.sqrt(E) * float(cotangent.double().norm())
            assert bool(a.isfinite().all()) and float((a.double() - b.double()).norm()) <= bound * float(b.double().norm()) + cancelled
    assert len(calls) == 2 and all(c is not None for c in calls)


def replay_with(mistake):
    """The oracle's loop, with one of the ways that a step size takes to later ones left out."""
    from torchode_amd.autodiff import Replay

    class Planted(Replay):
        def attempt(self, state):
            held = {"factor of the last ratio": "prev", "factor of the ratio before": "pprev"}.get(mistake)
            return super().attempt(state if held is None else dict(state, **{held: state[held].detach()}))

        def advance(self, state, attempt, *rest):
            ks, y1, ratio, dt_next = attempt
            if mistake == "ratio kept":
                attempt = (ks, y1, ratio.detach(), dt_next)
            if mistake == "ratio handed on":
                state = dict(state, prev=state["prev"].detach())
            return super().advance(state, attempt, *rest)

    return Planted


def in_float64(record, method, controller, tensors, t_eval, cotangent, through, dt0=None, mistake=None):
    """The gradients of y0 and the weights (``tensors``) over a record, its iterations as torch operations in float64 on the CPU."""
    from torchode_amd import autodiff

    y0, *weights = (x.detach().cpu().double() for x in tensors)
    states = [{k: v.cpu().double() if v.is_floating_point() else v.cpu() for k, v in state.items()} for state in record.trimmed(record.iterations)]
    params = [x.requires_grad_() for x in weights]
    problem, dt0 = to.InitialValueProblem(y0, t_eval=t_eval.double()), None if dt0 is None else dt0.double()
    replay = replay_with(mistake)(method, controller, to.ODETerm(to.MLPField(*params)), None, problem, through, dt0)
    adj, grads = autodiff.reverse_sweep_torch(replay, states, autodiff.simulate_hits(replay, states, t_eval.shape[1]), cotangent.double(), params)
    of_y0 = autodiff.SolveThroughLoop.start_backward(types.SimpleNamespace(dt0=dt0), replay, adj, y0, dt0, params, grads)
    return [of_y0, *grads]


def apart(gradients, want):
    return max(float((a.detach().cpu().double() - b).norm() / b.norm()) for a, b in zip(gradients, want))


MISTAKES = ["factor of the last ratio", "factor of the ratio before", "ratio kept", "ratio handed on"]


@pytest.mark.parametrize("F, H, method, first, until", [(64, 256, to.Tsit5, 0.2, 1.5), (7, 40, to.Tsit5, 0.4, 1.5), (64, 256, to.Dopri5, 0.2, 3), (33, 100, to.Dopri5, 0.2, 3)])
def test_controllers_history_in_one_kernel(monkeypatch, F, H, method, first, until):
    """A network with strong weights, large tolerances and a controller that looks far back: errors far above rounding, and
    gradients to which every way through the controller's history adds a hundredth or more.  Against the record's iterations as torch
    operations in float64 on the CPU, within 1e-3: the same in float32 comes to 5e-5, 2.4e-4, 3e-5 and 3e-5 of them; with one way
    through the history left out they are 1.9e-2 and more apart, which is looked at too."""
    from torchode_amd import autodiff

    whole, calls = autodiff.NetworkSweep.whole, []
    monkeypatch.setattr(autodiff.NetworkSweep, "whole", lambda *a: calls.append(whole(*a)) or calls[-1])
    B, E, g = 17, 3, torch.Generator().manual_seed(0)
    rand = lambda *shape: torch.rand(shape, generator=g, dtype=torch.float64)
    weights = [(4 * math.sqrt(6.0 / (F + H)) * (2 * rand(*shape) - 1)).float() for shape in ((H, F + 1), (H,), (F, H), (F,))]
    y0 = (2 * rand(B, F) - 1).float()
    t_eval = (until * (0.8 + 0.4 * rand(B, 1)) * torch.linspace(0, 1, E, dtype=torch.float64)).float()
    cotangent = (2 * rand(B, E, F) - 1).float()
    cotangent[:, 0] = 0  # (the point at the start)
    dt0, controller = torch.full((B,), first), to.PIDController(0.03, 0.03, 0.2, 0.4, -0.3)

    leaves = [x.cuda().requires_grad_() for x in (y0, *weights)]
    sol = to.AutoDiffAdjoint(method(), controller).solve(to.InitialValueProblem(leaves[0], t_eval=t_eval.cuda()), to.ODETerm(to.MLPField(*leaves[1:])), dt0=dt0.cuda())
    assert not sol.status.any()
    record = sol.ys.grad_fn.record
    found = torch.autograd.grad(sol.ys, leaves, cotangent.cuda())
    assert len(calls) == 1 and calls[0] is not None
    reference = lambda mistake=None: in_float64(record, method(), controller, leaves, t_eval, cotangent, True, dt0, mistake)
    want = reference()
    off = [apart(reference(mistake), want) for mistake in MISTAKES]
    print("iterations", record.iterations, "apart", apart(found, want), off)
    assert apart(found, want) <= 1e-3
    assert min(off) >= 1e-2


@pytest.mark.parametrize("method", [to.Dopri5, to.Tsit5])
@pytest.mark.parametrize("B, F, H, E", [(60, 10, 30, 5), (100, 4, 20, 12), (200, 63, 255, 9), (64, 17, 128, 29)])
def test_short_rows_against_float64(monkeypatch, B, F, H, E, method):
    """Rows shorter than 64 take five sums a feature over an iteration's points where the launches per iteration go point by point:
    with the step sizes held constant either is within 4.6e-6 of float64 over the same record (geometric means of 60 solves: y0
    4.5e-7 and 4.6e-7, W1 8.5e-7 and 8.6e-7), so four times that bounds both."""
    from torchode_amd.autodiff import NetworkSweep

    g = torch.Generator().manual_seed(B)
    randn = lambda *shape: torch.randn(shape, generator=g)
    tensors = [randn(B, F), *(scale * randn(*shape) for scale, shape in ((0.9 / math.sqrt(F), (H, F + 1)), (0.1, (H,)), (0.9 / math.sqrt(H), (F, H)), (0.1, (F,))))]
    t_eval, cotangent = torch.linspace(0, 1, E).repeat(B, 1), randn(B, E, F)
    cotangent[:, 0] = 0  # (the point at the start)
    whole = NetworkSweep.whole
    for one_kernel in (True, False):
        monkeypatch.setattr(NetworkSweep, "whole", whole if one_kernel else lambda *a: None)
        leaves, controller = [x.cuda().requires_grad_() for x in tensors], to.IntegralController(1e-5, 1e-3)
        sol = to.AutoDiffAdjoint(method(), controller, backprop_through_step_size_control=False).solve(to.InitialValueProblem(leaves[0], t_eval=t_eval.cuda()), to.ODETerm(to.MLPField(*leaves[1:])))
        record = sol.ys.grad_fn.record
        found = torch.autograd.grad(sol.ys, leaves, cotangent.cuda())
        difference = apart(found, in_float64(record, method(), controller, leaves, t_eval, cotangent, False))
        print("one kernel" if one_kernel else "per iteration", difference)
        assert difference <= 1.9e-5


def test_outer_products_of_a_record_beyond_its_room(monkeypatch):
    """A record whose rows do not all fit: the outer products are taken of as many iterations' rows at a time as do fit, and the
    gradients are those of the sweep that holds all rows."""
    from torchode_amd.autodiff import NetworkSweep

    B, F, H, lib = 40, 64, 256, _lib.load()
    g = torch.Generator("cuda").manual_seed(12)
    rand = lambda *shape: torch.rand(shape, generator=g, device="cuda")
    weights = [(math.sqrt(6.0 / (F + H)) * (2 * rand(*shape) - 1)).requires_grad_() for shape in ((H, F + 1), (H,), (F, H), (F,))]
    y0 = (2 * rand(B, F) - 1).requires_grad_()
    t_eval = 2 * torch.linspace(0, 1, 6, device="cuda").repeat(B, 1)
    cotangent = 2 * rand(B, 6, F) - 1
    outer, calls, results = lib.tode_mlp_outer_products, [], []
    monkeypatch.setattr(lib, "tode_mlp_outer_products", lambda p, rows, accumulate, stream: calls.append((rows, accumulate)) or outer(p, rows, accumulate, stream))
    for held in (None, 15):  # evaluations: two iterations and a remainder that no third fits into
        if held:
            monkeypatch.setattr(NetworkSweep, "ROOM", held * 4 * B * (2 * 256 + 3 * F + 1))
        solver = to.AutoDiffAdjoint(to.Dopri5(), to.IntegralController(1e-6, 1e-5), backprop_through_step_size_control=False)
        sol = solver.solve(to.InitialValueProblem(y0, t_eval=t_eval), to.ODETerm(to.MLPField(*weights)))
        results.append(torch.autograd.grad(sol.ys, [y0, *weights], cotangent))
    L = (int(sol.stats["n_f_evals"][0]) - 2) // 6
    assert L >= 5
    expected, rows = [], 0
    for evaluations in [6] * L + [1]:  # (the start of the loop: its one evaluation where the step rule wants no gradient)
        if rows + evaluations > 15:
            expected.append(rows)
            rows = 0
        rows += evaluations
    expected.append(rows)
    assert calls == [(B * n, int(i > 0)) for i, n in enumerate(expected)]  # (the sweep that holds all rows calls it from native code)
    for a, b in zip(*results):
        assert float((a.double() - b.double()).norm()) <= 2e-5 * float(b.double().norm())


@pytest.mark.parametrize("F, H", [(1, 1), (64, 256), (63, 255), (6, 40)])
def test_both_packings_in_one_launch(F, H):
    """The two orders straight from four tensors against the two packings of their concatenation."""
    g = torch.Generator("cuda").manual_seed(F)
    weights = [torch.randn(shape, generator=g, device="cuda") for shape in ((H, F + 1), (H,), (F, H), (F,))]
    weights[0] = torch.cat([weights[0], weights[0]], 1)[:, : F + 1]  # (not contiguous)
    f, lib = to.MLPField(*weights), _lib.load()
    forward, reverse = _lib.MLP_PACKED_SIZE["float32"], _lib.MLP_REVERSE_PACKED_SIZE
    raw, want = f.builtin_shared(), torch.full((forward + reverse,), 7.0, device="cuda")
    _lib.check(lib.tode_mlp_pack_weights_for(raw.data_ptr(), raw.numel(), F, 0, want.data_ptr(), _lib.stream_of(raw)), "tode_mlp_pack_weights_for")
    _lib.check(lib.tode_mlp_pack_weights_reverse(raw.data_ptr(), raw.numel(), F, want.data_ptr() + 4 * forward, _lib.stream_of(raw)), "tode_mlp_pack_weights_reverse")
    assert torch.equal(f.builtin_packed_both(), want)


def test_weights_written_between_the_passes(monkeypatch):
    """The reverse sweep goes by the forward pass's packing of the weights only while the weights are those: written in place or
    replaced in between, they are packed anew, and both sweeps take the new ones."""
    from torchode_amd.autodiff import NetworkSweep

    whole, results = NetworkSweep.whole, []
    for one_kernel in (True, False):
        monkeypatch.setattr(NetworkSweep, "whole", whole if one_kernel else lambda *a: None)
        for change in (lambda f: f.W1.mul_(1.01), lambda f: setattr(f, "W2", f.W2 * 0.99), lambda f: None):
            g = torch.Generator("cuda").manual_seed(9)
            rand = lambda *shape: 0.2 * (2 * torch.rand(shape, generator=g, device="cuda") - 1)
            f = to.MLPField(rand(256, 65), rand(256), rand(64, 256), rand(64))
            y0 = rand(40, 64).requires_grad_()
            solver = to.AutoDiffAdjoint(to.Dopri5(), to.IntegralController(1e-5, 1e-3), backprop_through_step_size_control=False)
            sol = solver.solve(to.InitialValueProblem(y0, t_eval=torch.linspace(0, 1, 5, device="cuda").repeat(40, 1)), to.ODETerm(f))
            with torch.no_grad():
                change(f)
            results.append(torch.autograd.grad(sol.ys, y0, torch.ones_like(sol.ys))[0])
    for a, b in zip(results[:3], results[3:]):
        assert torch.equal(a, b)
    assert not torch.equal(results[0], results[2]) and not torch.equal(results[1], results[2])
