"""``torchode_amd._host``, the native call around a whole solve's kernel: every form of problem that ``solve`` takes there against
the operator of PyTorch's dispatcher, which prepares the same kernel by itself -- the same bits -- and its refusals."""
import threading

import pytest
import torch

import torchode_amd as to
from torchode_amd import _lib, ops

pytestmark = pytest.mark.gpu


def through_the_operator(solver, problem, term, dt0):
    f, c = term.f, solver.step_size_controller
    kind, control = c.control_values()
    columns = [t if t.stride(0) >= 1 else t.contiguous() for t in (problem.t_start, problem.t_end)]
    mlp = f.builtin_kind == _lib.TERM_MLP
    params = None if mlp else f.builtin_params().to(problem.y0)
    shared = ops.mlp_pack_weights(f.builtin_shared(), _lib.MLP_INPUTS[f.matrix_inputs], problem.n_features) if mlp else None
    return ops.solve_builtin(
        problem.y0, *columns, problem.t_eval, dt0, params, shared, solver.step_method.method_id, f.builtin_kind,
        [float(x) for x in getattr(f, "builtin_scalars", lambda: ())()], kind, control, solver.max_steps, solver.use_fast_path,
    )  # fmt: skip


def forms(B, E, time_dtype):
    t1 = 1.0 + torch.arange(B, dtype=time_dtype, device="cuda") / max(B, 1)
    rows = t1[:, None] * torch.linspace(0, 1, E, dtype=time_dtype, device="cuda")
    wide = torch.full((B, 2 * E), 7.0, dtype=time_dtype, device="cuda")
    wide[:, ::2] = rows
    return {
        "points": dict(t_eval=rows),
        "points-strided": dict(t_eval=wide[:, ::2]),
        "points-transposed": dict(t_eval=rows.T.contiguous().T),
        "points-one-row": dict(t_eval=rows[:1].expand(B, E)),
        "points-backwards": dict(t_eval=rows.flip(1)),
        "range-in-points": dict(t_eval=rows, t_start=torch.zeros_like(t1) - 0.5, t_end=t1 + 0.25),
        "range": dict(t_start=torch.zeros_like(t1), t_end=t1),
        "range-expanded": dict(t_start=torch.zeros(1, dtype=time_dtype, device="cuda").expand(B), t_end=torch.ones(1, dtype=time_dtype, device="cuda").expand(B)),
        "no-range": dict(t_start=t1, t_end=t1),
        "points-in-no-order": dict(t_eval=rows[:, torch.randperm(E, generator=torch.Generator().manual_seed(1)).cuda()], t_start=torch.zeros_like(t1), t_end=t1),
    }


FORMS = ["points", "points-strided", "points-transposed", "points-one-row", "points-backwards", "range-in-points", "range", "range-expanded", "no-range", "points-in-no-order"]


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("dtype,time_dtype", [(torch.float32, torch.float32), (torch.float64, torch.float64), (torch.float64, torch.float32)], ids=["f32", "f64", "f64-t32"])
@pytest.mark.parametrize("B", [0, 1, 67])
def test_forms_of_a_problem(form, dtype, time_dtype, B):
    if B == 0 and form == "range-expanded":
        pytest.skip("an empty expanded range keeps its stride of zero, which the library refuses")
    g = torch.Generator().manual_seed(3)
    y0 = torch.randn((3, B), generator=g, dtype=torch.float64).to(dtype).cuda().T  # (not contiguous)
    # (parameters in another type than the state; Lorenz' equations, which have scalars too, leave every bound when followed
    # backwards for long, and their solve would take millions of ever smaller steps)
    rates = torch.rand((B, 3), generator=g, dtype=torch.float64).cuda()
    f = to.LinearDecay(rates) if form == "points-backwards" else to.Lorenz63(20 + 10 * rates[:, 0], beta=2.5)
    times = forms(B, 6, time_dtype)[form]
    step = torch.full((B,), -0.01 if form == "points-backwards" else 0.01, dtype=torch.float64, device="cuda")  # (in another type than the times)
    for options, dt0 in ((dict(), None), (dict(max_steps=3), None), (dict(), step)):
        solver = to.AutoDiffAdjoint(to.Tsit5(), to.PIDController(atol=1e-5, rtol=1e-3, pcoeff=0.2, icoeff=0.5, dcoeff=0.0), **options)
        problem, term = to.InitialValueProblem(y0, **times), to.ODETerm(f)
        ys, n_steps, n_accepted, n_initialized, status, iterations = through_the_operator(solver, problem, term, dt0)
        for _ in range(2):
            got = solver.solve(problem, term, dt0)
            assert torch.equal(got.stats["n_steps"], n_steps) and torch.equal(got.stats["n_accepted"], n_accepted)
            assert torch.equal(got.stats["n_initialized"], n_initialized) and torch.equal(got.status, status)
            assert got.stats["n_f_evals"].tolist() == [(2 if dt0 is None else 1) + 6 * int(iterations)] * B
            if not status.any():
                assert torch.equal(got.ys, ys)
            assert got.ys.shape == (B, times["t_eval"].shape[1] if "t_eval" in times else 1, 3) and got.ys.dtype == dtype


@pytest.mark.parametrize("system", ["network", "grid", "decay"])
def test_other_terms_and_reassigned_members(system):
    g = torch.Generator().manual_seed(4)
    rand = lambda *shape: torch.rand(shape, generator=g).cuda()
    B = 33
    y0 = rand(B, {"network": 17, "grid": 256, "decay": 2}[system])
    f = {
        "network": lambda: to.MLPField(rand(30, 18) - 0.5, rand(30), rand(17, 30) - 0.5, rand(17)),
        "grid": lambda: to.ReactionDiffusion(rand(B) * 0.1, 16),
        "decay": lambda: to.LinearDecay(rand(B, 2)),
    }[system]()
    solver, problem, term = to.AutoDiffAdjoint(to.Dopri5(), to.IntegralController(atol=1e-5, rtol=1e-3)), to.InitialValueProblem(y0, t_eval=rand(B, 5).sort(1).values), to.ODETerm(f)
    for change in (lambda: None, lambda: y0.mul_(0.5), lambda: setattr(problem, "y0", y0 + 1), lambda: next(iter(f.buffers())).mul_(0.9)):
        change()  # (nothing of an earlier solve of the same objects may be kept)
        ys, n_steps, *_ = through_the_operator(solver, problem, term, None)
        got = solver.solve(problem, term)
        assert torch.equal(got.ys, ys) and torch.equal(got.stats["n_steps"], n_steps)


def test_refusals():
    solver = to.AutoDiffAdjoint(to.Dopri5(), to.IntegralController(atol=1e-5, rtol=1e-3))
    y0, t = torch.ones((4, 2), device="cuda"), torch.zeros(4, device="cuda")
    with pytest.raises(AssertionError, match="batch size"):
        solver.solve(to.InitialValueProblem(y0, t, t + 1), to.ODETerm(to.VanDerPol(torch.ones(3, device="cuda"))))
    with pytest.raises(RuntimeError, match="GPU"):
        solver.solve(to.InitialValueProblem(y0.cpu(), t.cpu(), t.cpu() + 1), to.ODETerm(to.VanDerPol(torch.ones(4))))
    with pytest.raises(TypeError):
        _lib.load_host().solve(y0)
    with pytest.raises(TypeError):
        _lib.load_host().solve(*[None] * 24)


@pytest.mark.parametrize("limit,as_int", [(1e4, 10000), (3.9, 3), (True, 1), (torch.tensor(2.0), 2)])
def test_step_limit_as_any_number(limit, as_int):
    """``max_steps`` is taken as ``int(max_steps)`` says, with gradients and without."""
    y0, t_eval = torch.full((5, 2), 0.5, device="cuda"), torch.linspace(0, 3, 4, device="cuda").repeat(5, 1)
    make = lambda n: to.AutoDiffAdjoint(to.Dopri5(), to.IntegralController(atol=1e-6, rtol=1e-4), max_steps=n)
    for gradient in (False, True):
        a, b = (make(n).solve(to.InitialValueProblem(y0.clone().requires_grad_(gradient), t_eval=t_eval), to.ODETerm(to.VanDerPol(torch.ones(5, device="cuda")))) for n in (limit, as_int))
        assert torch.equal(a.status, b.status) and torch.equal(a.stats["n_steps"], b.stats["n_steps"])
        assert int(a.stats["n_steps"].max()) <= as_int and bool(a.status.any()) == (as_int < 10)
        written = torch.arange(4, device="cuda") < a.stats["n_initialized"][:, None]
        assert torch.equal(a.ys[written], b.ys[written])


def test_threads_and_streams():
    """Solves of several host threads, each on a stream of its own: the call releases the interpreter while it waits."""
    solver = to.AutoDiffAdjoint(to.Tsit5(), to.IntegralController(atol=1e-6, rtol=1e-4))
    wrong = []

    def work(seed):
        with torch.cuda.stream(torch.cuda.Stream()):
            g = torch.Generator("cuda").manual_seed(seed)
            mu, y0 = torch.rand(500, generator=g, device="cuda") * 4 + 0.5, torch.randn((500, 2), generator=g, device="cuda")
            term, t_eval = to.ODETerm(to.VanDerPol(mu)), torch.linspace(0, 6, 9, device="cuda").repeat(500, 1)
            first = solver.solve(to.InitialValueProblem(y0, t_eval=t_eval), term)
            for _ in range(20):
                again = solver.solve(to.InitialValueProblem(y0, t_eval=t_eval), term)
                if not torch.equal(first.ys, again.ys) or not torch.equal(first.stats["n_steps"], again.stats["n_steps"]):
                    wrong.append(seed)

    threads = [threading.Thread(target=work, args=(s,)) for s in range(6)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong


@pytest.mark.parametrize("method,controller", [(to.Dopri5, to.IntegralController), (to.Tsit5, to.IntegralController), (to.Heun, to.IntegralController), (to.Euler, to.FixedStepController)])
@pytest.mark.parametrize("dtype,time_dtype", [(torch.float32, torch.float32), (torch.float64, torch.float32)], ids=["f32", "f64-t32"])
def test_stages_around_a_users_function(method, controller, dtype, time_dtype):
    """A user's f gets fresh tensors at every stage, of its problem's types, that stay what they were; what it returns may be of
    another type, expanded or strided; the loop's result is that of the operator path, evaluation by evaluation."""
    seen = []

    def f(t, y):
        assert t.dtype == time_dtype and y.dtype == dtype and t.shape == (9,) and y.shape == (9, 3) and y.is_contiguous()
        seen.append((t, y, y.clone()))
        out = -y * (1 + t[:, None].to(dtype))
        return (out.double(), out[:, :1].expand(9, 3), out.T.contiguous().T)[len(seen) % 3] if method is not to.Euler else out

    g = torch.Generator().manual_seed(2)
    y0 = torch.rand((9, 1), generator=g, dtype=torch.float64).to(dtype).expand(9, 3).cuda()
    times = dict(t_eval=torch.linspace(0, 1, 5, dtype=time_dtype, device="cuda").repeat(9, 1))
    dt0 = torch.full((9,), 0.125, dtype=time_dtype, device="cuda") if controller is to.FixedStepController else None
    make = lambda: to.AutoDiffAdjoint(method(), controller() if dt0 is not None else controller(atol=1e-4, rtol=1e-3))
    found = make().solve(to.InitialValueProblem(y0, **times), to.ODETerm(f), dt0=dt0)
    assert len({id(y) for _, y, _ in seen}) == len(seen) and all(torch.equal(y, copy) for _, y, copy in seen)
    steps = found.stats["n_f_evals"][0].item()
    assert steps <= len(seen) <= steps + 12
    wanted = make()._solve_protocol(to.InitialValueProblem(y0, **times), to.ODETerm(f), to.ODETerm(f), dt0, None)
    assert torch.equal(found.stats["n_steps"], wanted.stats["n_steps"]) and torch.allclose(found.ys, wanted.ys, rtol=1e-5, atol=1e-6)
    with pytest.raises(ValueError):
        _lib.load_host().stage(0, 0, 1, y0, y0, None, None)
    state, control, y = _lib.StepState(), _lib.Controller(), torch.zeros((9, 3), device="cuda")
    for k in (y.cpu(), y.double(), y[:8], y.T.contiguous().T):
        with pytest.raises(ValueError, match="of y's shape"):
            _lib.load_host().stage(_lib.C.addressof(state), _lib.C.addressof(control), 1, y, y[:, 0], k, None)
    with pytest.raises(TypeError):
        _lib.load_host().stage(0, 0)


@pytest.mark.parametrize("evaluation", [0, 1, 4, 7])
def test_a_users_function_off_the_device_is_refused(evaluation):
    """f's result on the CPU, at the start, at a stage and at the last one of a step, is an error as in torch's own arithmetic."""
    seen = []

    def f(t, y):
        seen.append(None)
        return -y.cpu() if len(seen) > evaluation else -y

    problem = to.InitialValueProblem(torch.ones((5, 2), device="cuda"), t_eval=torch.linspace(0, 1, 3, device="cuda").repeat(5, 1))
    with torch.no_grad(), pytest.raises(RuntimeError, match="GPU"):
        to.AutoDiffAdjoint(to.Dopri5(), to.IntegralController(atol=1e-4, rtol=1e-3)).solve(problem, to.ODETerm(f))
    torch.cuda.synchronize()
