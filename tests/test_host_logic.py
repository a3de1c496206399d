"""CPU tests of the host side: problem validation, term bookkeeping, controller parameter
marshalling, dispatch guards, the C ABI's exported symbols, the seeded workloads and the
committed golden fixtures (checked here against the C oracle, on the GPU against the kernels)."""
import glob
import hashlib
import json
import os
import re

import pytest
import torch

import torchode_amd as to
from oracle import c_oracle
from torchode_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_problem_defaults_and_direction():
    t_eval = torch.tensor([[0.0, 1.0, 2.0], [5.0, 4.0, 1.0], [3.0, 3.0, 3.0]])
    p = to.InitialValueProblem(torch.zeros(3, 2), t_eval=t_eval)
    assert torch.equal(p.t_start, t_eval[:, 0]) and torch.equal(p.t_end, t_eval[:, -1])
    assert p.time_direction.tolist() == [1, -1, -1]  # t_end == t_start counts as backwards
    assert (p.batch_size, p.n_features, p.n_evaluation_points) == (3, 2, 3)
    p = to.InitialValueProblem(torch.zeros(2, 1, dtype=torch.float64), torch.zeros(2), torch.ones(2))
    assert p.n_evaluation_points == 0 and p.data_dtype == torch.float64 and p.time_dtype == torch.float32


@pytest.mark.parametrize(
    "kwargs",
    [
        dict(y0=torch.zeros(3), t_start=torch.zeros(3), t_end=torch.ones(3)),  # y0 not 2-D
        dict(y0=torch.zeros(3, 1), t_start=torch.zeros(2), t_end=torch.ones(2)),  # batch mismatch
        dict(y0=torch.zeros(3, 1), t_start=torch.zeros(3), t_end=torch.ones(3, dtype=torch.float64)),  # time dtypes
        dict(y0=torch.zeros(3, 1), t_eval=torch.zeros(3)),  # t_eval not 2-D
    ],
)
def test_problem_rejects_bad_shapes(kwargs):
    with pytest.raises((AssertionError, IndexError)):
        to.InitialValueProblem(**kwargs)


def test_term_counts_evaluations_on_cpu_tensor_and_passes_args_by_identity():
    seen = []
    term = to.ODETerm(lambda t, y, a: seen.append(a) or y, with_args=True)
    problem = to.InitialValueProblem(torch.zeros(4, 1), t_eval=torch.zeros(4, 2))
    stats = {}
    term.init(problem, stats)
    token = object()
    for _ in range(3):
        term.vf(problem.t_start, problem.y0, stats, token)
    assert stats["n_f_evals"].tolist() == [3, 3, 3, 3] and stats["n_f_evals"].device.type == "cpu"
    assert all(a is token for a in seen)
    quiet = to.ODETerm(lambda t, y: y, with_stats=False)
    stats = {}
    quiet.init(problem, stats)
    quiet.vf(problem.t_start, problem.y0, stats, None)
    assert stats == {}


def test_controller_struct_carries_float32_rounded_tolerances():
    c = to.PIDController(1e-6, 1e-4, 0.2, 0.5, 0.0, dt_max=0.5).c_struct()
    assert c.kind == _lib.CTRL_PID and c.has_dt_max == 1 and c.has_dt_min == 0 and c.dt_max == 0.5
    assert c.atol == float(torch.tensor(1e-6)) != 1e-6 and c.rtol == float(torch.tensor(1e-4)) != 1e-4
    assert (c.pcoeff, c.icoeff, c.dcoeff, c.safety, c.factor_min, c.factor_max) == (0.2, 0.5, 0.0, 0.9, 0.2, 10.0)
    i = to.IntegralController(1e-3, 1e-3, safety=0.8)
    assert i.c_struct().kind == _lib.CTRL_INTEGRAL and i.c_struct().safety == 0.8
    assert i.atol.dtype == torch.float32 and "atol" in dict(i.named_buffers())
    assert to.IntegralController(1e-3, 1e-3, norm=to.step_size_controllers.max_norm).fusable is False


def test_solve_refuses_cpu_tensors_and_grad():
    w = to.workloads.make("vdp", batch=4)
    solver = to.AutoDiffAdjoint(to.Tsit5(), to.PIDController(1e-6, 1e-4, 0.2, 0.5, 0.0))
    with pytest.raises(RuntimeError, match="AMD GPU"):
        solver.solve(to.InitialValueProblem(w.y0, t_eval=w.t_eval), to.ODETerm(w.f))
    assert solver.step_method.convergence_order() == 5 and solver.max_steps is None


def test_library_exports_every_declared_symbol():
    header = open(os.path.join(ROOT, "include", "torchode_amd.h")).read()
    header = re.sub(r"/\*.*?\*/", "", header, flags=re.S)
    declared = set(re.findall(r"\b(tode_[a-z0-9_]+)\s*\(", header))
    assert declared, "no declarations found"
    lib = _lib.load()
    for name in sorted(declared):
        assert hasattr(lib, name), f"{name} is declared in include/torchode_amd.h but not exported"
    assert declared == set(_lib.EXPORTS)
    assert lib.tode_abi_version() == _lib.ABI_VERSION == int(re.search(r"#define TODE_ABI_VERSION (\d+)", header).group(1))
    assert lib.tode_last_error() is not None


@pytest.mark.parametrize("name", ["HOST_LIB", "OPS_LIB"])
def test_libraries_between_pytorch_and_the_kernels_have_no_thread_local_storage(name):
    """Thread-local storage that a thread never reaches slows down every access of that thread to that of other libraries loaded at
    run time, PyTorch's among them: all its operations, for the rest of the process."""
    import struct

    from torchode_amd import build

    with open(getattr(build, name), "rb") as file:
        elf = file.read()
    assert elf[:6] == b"\x7fELF\x02\x01"
    (table,), (size, count) = struct.unpack_from("<Q", elf, 32), struct.unpack_from("<HH", elf, 54)
    kinds = [struct.unpack_from("<I", elf, table + i * size)[0] for i in range(count)]
    assert 1 in kinds and 7 not in kinds  # PT_LOAD, PT_TLS


def test_torch_operators_are_registered_for_the_gpu_only_with_tracing_rules():
    """libtorchode_amd_ops.so registers torch.ops.torchode_amd.solve_builtin / mlp_pack_weights: no CPU implementation
    (a call with CPU tensors fails in the dispatcher), and the shapes, dtypes and devices of the results for a tracer."""
    from torch._subclasses.fake_tensor import FakeTensorMode

    from torchode_amd import ops

    ops.load()
    op = torch.ops.torchode_amd.solve_builtin
    assert "CUDA" in torch._C._dispatch_dump("torchode_amd::solve_builtin") and "CPU:" not in torch._C._dispatch_dump("torchode_amd::solve_builtin")
    control = [1e-6, 1e-5, 0.0, 1.0, 0.0, 0.9, 0.2, 10.0, float("nan"), float("nan")]
    with FakeTensorMode():
        y0, t_eval = torch.empty(8, 3, device="cuda", dtype=torch.float64), torch.empty(8, 5, device="cuda", dtype=torch.float64)
        out = op(y0, t_eval[:, 0], t_eval[:, -1], t_eval, None, torch.empty(8, 1, device="cuda"), None, 1, 2, [10.0, 8 / 3], 0, control, -1, True)
        assert [tuple(o.shape) for o in out] == [(8, 5, 3), (8,), (8,), (8,), (8,), ()]
        assert [o.dtype for o in out] == [torch.float64] + [torch.long] * 5
        assert [o.device.type for o in out] == ["cuda"] * 5 + ["cpu"]
        end_only = op(y0, t_eval[:, 0], t_eval[:, -1], None, None, None, None, 1, 2, [10.0, 8 / 3], 0, control, -1, True)
        assert tuple(end_only[0].shape) == (8, 1, 3)
        packed = torch.ops.torchode_amd.mlp_pack_weights(torch.empty(256 * 65 + 256 + 64 * 256 + 64, device="cuda"), 1)
        assert tuple(packed.shape) == (_lib.MLP_PACKED_SIZE["bfloat16"],)
    y0, t_eval = torch.zeros(8, 3), torch.zeros(8, 5)
    with pytest.raises(NotImplementedError, match="CPU"):
        op(y0, t_eval[:, 0], t_eval[:, -1], t_eval, None, torch.zeros(8, 1), None, 1, 2, [10.0, 8 / 3], 0, control, -1, True)


def test_solve_workspace_size_and_argument_checks_of_the_one_call_entry_point():
    lib = _lib.load()
    a, c = _lib.SolveArgs(), _lib.Controller()
    assert lib.tode_solve_workspace_bytes(None) == -1
    a.dtype, a.batch, a.n_features, a.n_eval = _lib.DTYPES[torch.float64], 1000, 3, 0
    up = lambda n: (n + 255) // 256 * 256
    assert lib.tode_solve_workspace_bytes(_lib.C.byref(a)) == up(16) + up(5 * 1000 * 4) + up(1000 * 3 * 8)
    a.n_eval = 7
    need = lib.tode_solve_workspace_bytes(_lib.C.byref(a))
    assert need == up(16) + up(5 * 1000 * 4) + up(1000 * 7)
    it = _lib.C.c_int64(0)
    dummy = (_lib.C.c_double * 64)()
    p = _lib.C.addressof(dummy)
    assert lib.tode_solve_builtin_auto(_lib.C.byref(a), _lib.C.byref(c), p, p, p, p, p, need - 1, 1, None, _lib.C.byref(it)) == _lib.E_INVALID
    assert b"workspace" in lib.tode_last_error()
    assert lib.tode_solve_builtin_auto(_lib.C.byref(a), _lib.C.byref(c), p, p, p, p, None, need, 1, None, _lib.C.byref(it)) == _lib.E_INVALID
    assert lib.tode_solve_builtin_auto(_lib.C.byref(a), _lib.C.byref(c), p, p, p, p, p, need, 1, None, None) == _lib.E_INVALID
    a.term = 9
    assert lib.tode_solve_builtin_auto(_lib.C.byref(a), _lib.C.byref(c), p, p, p, p, p, need, 1, None, _lib.C.byref(it)) == _lib.E_INVALID
    assert b"unknown term" in lib.tode_last_error()
    a.term, a.dtype = _lib.TERM_MLP, _lib.DTYPES[torch.float64]  # the matrix-core kernel is float32: refused before anything is launched
    assert lib.tode_solve_builtin_auto(_lib.C.byref(a), _lib.C.byref(c), p, p, p, p, p, need, 1, None, _lib.C.byref(it)) == _lib.E_UNSUPPORTED


def test_whole_reverse_sweep_entry_point_checks_its_arguments_without_a_gpu():
    lib = _lib.load()
    a, c, adj = _lib.SolveArgs(), _lib.Controller(), _lib.SolveAdjoint()
    ref = lambda x: _lib.C.byref(x)
    assert lib.tode_solve_builtin_backward(None, None, None, None) == _lib.E_INVALID
    a.dtype, a.batch, a.n_features, a.n_eval, a.n_params, a.term = _lib.DTYPES[torch.float64], 100, 2, 0, 1, 1
    a.t_start_stride = a.t_end_stride = 1
    assert lib.tode_solve_backward_scratch_bytes(ref(a)) == 0  # (no evaluation points: no lists of them to work out)
    a.n_eval = 7
    assert lib.tode_solve_backward_scratch_bytes(ref(a)) == 2 * 100 * 7 * 4  # (two int32 lists [B,E], unless the caller hands them in)
    a.n_eval = 0
    assert lib.tode_solve_builtin_backward(ref(a), ref(c), ref(adj), None) == _lib.E_INVALID and b"record" in lib.tode_last_error()
    rec = _lib.SolveRecord()
    rec.capacity = 5
    a.record = _lib.C.addressof(rec)
    adj.iterations = 5
    assert lib.tode_solve_builtin_backward(ref(a), ref(c), ref(adj), None) == _lib.E_INVALID and b"entries" in lib.tode_last_error()
    adj.iterations = 4
    assert lib.tode_solve_builtin_backward(ref(a), ref(c), ref(adj), None) == _lib.E_INVALID  # null arrays
    a.dtype = _lib.dtype_code(torch.float32, torch.float64)
    assert lib.tode_solve_builtin_backward(ref(a), ref(c), ref(adj), None) == _lib.E_UNSUPPORTED and b"one dtype" in lib.tode_last_error()


def test_abi_argument_validation_without_a_gpu():
    """Null / inconsistent arguments are rejected before anything touches a device."""
    lib = _lib.load()
    a, c = _lib.SolveArgs(), _lib.Controller()
    assert lib.tode_solve_builtin(None, None, None) == -1
    a.batch, a.n_features, a.n_eval = 4, 2, 0
    assert lib.tode_solve_builtin(_lib.C.byref(a), _lib.C.byref(c), None) == -1
    assert b"null" in lib.tode_last_error()
    dummy = (_lib.C.c_double * 64)()
    for name in ("y0", "t_start", "t_end", "ys", "y_idle"):
        setattr(a, name, _lib.C.addressof(dummy))
    assert lib.tode_solve_builtin(_lib.C.byref(a), _lib.C.byref(c), None) == -1  # strides left at zero
    assert b"stride" in lib.tode_last_error()
    # n_eval == 0 through the fast entry point: y_idle is needed (every term takes that case; the next check is the flag block)
    a.term = _lib.TERM_MLP
    assert lib.tode_solve_builtin_fast(_lib.C.byref(a), _lib.C.byref(c), None, None, None, None, None) == -1
    assert b"flags" in lib.tode_last_error()
    a.term, a.y_idle = 1, None
    assert lib.tode_solve_builtin_fast(_lib.C.byref(a), _lib.C.byref(c), None, None, None, None, None) == -1
    assert b"y_idle" in lib.tode_last_error()
    a.y_idle = _lib.C.addressof(dummy)
    assert lib.tode_select_end_point(4, 2, 7, 3, _lib.C.addressof(dummy), _lib.C.addressof(dummy), _lib.C.addressof(dummy), None) == -1
    assert b"dtype" in lib.tode_last_error()
    assert lib.tode_select_end_point(4, 2, 0, 3, None, _lib.C.addressof(dummy), _lib.C.addressof(dummy), None) == -1
    assert lib.tode_select_end_point(0, 2, 0, 3, None, None, None, None) == 0
    a.n_features = 0
    assert lib.tode_solve_builtin(_lib.C.byref(a), _lib.C.byref(c), None) == -1
    assert b"bad sizes" in lib.tode_last_error()
    out = _lib.C.c_float()
    assert lib.tode_last_solve_kernel_ms(_lib.C.byref(out)) == -1


def test_workloads_are_deterministic_and_prefix_consistent():
    a = to.workloads.make("vdp", batch=300, dtype=torch.float64)
    b = to.workloads.make("vdp", batch=1000, dtype=torch.float64)
    assert torch.equal(a.y0, b.y0[:300]) and torch.equal(a.t_eval, b.t_eval[:300]) and torch.equal(a.f.mu, b.f.mu[:300])
    f32 = to.workloads.make("vdp", batch=300)
    assert f32.y0.dtype == torch.float32 and torch.equal(f32.y0, a.y0.float())
    assert torch.equal(a.t_eval[:, 0], torch.zeros(300, dtype=torch.float64))
    assert (a.bytes_step, a.bytes_dense) == (160, 1200) and (f32.bytes_step, f32.bytes_dense) == (88, 600)
    lz, ld = to.workloads.make("lorenz", batch=8), to.workloads.make("linear_decay")
    assert (lz.bytes_step, lz.bytes_dense) == (88, 320) and (ld.bytes_step, ld.bytes_dense) == (216, 400)
    assert ld.y0.shape == (256, 4) and ld.y0.dtype == torch.float64 and lz.t_eval.shape == (8, 20)


def test_builtin_terms_are_plain_torch_callables():
    w = to.workloads.make("lorenz", batch=5, dtype=torch.float64)
    t = torch.zeros(5, dtype=torch.float64)
    dy = w.f(t, w.y0)
    x, y, z = w.y0.T
    expect = torch.stack((10.0 * (y - x), x * (w.f.rho - z) - y, x * y - (8.0 / 3.0) * z), 1)
    assert torch.equal(dy, expect)
    assert w.f.builtin_params().shape == (5, 1) and w.f.builtin_kind == to.builtin_terms.TERM_LORENZ63


def _sha(t):
    return hashlib.sha256(t.contiguous().numpy().tobytes()).hexdigest()


GOLDEN = sorted(glob.glob(os.path.join(ROOT, "tests", "golden", "*.json")))


@pytest.mark.parametrize("path", [p for p in GOLDEN if p.endswith("_tolerance.json")], ids=os.path.basename)
def test_tolerance_fixture_inputs_and_workload_agree(path):
    """Vectors of the long-row workloads (ATen-op oracle, compared at 1e-4 on the GPU): here only that
    the seeded inputs are the ones the vectors were computed from, and that the vectors are complete."""
    g = json.load(open(path))
    w = to.workloads.make(g["workload"], batch=g["batch"], dtype=getattr(torch, g["dtype"]))
    assert {"y0": _sha(w.y0), "t_eval": _sha(w.t_eval)} == g["inputs_sha256"]
    assert (w.method, w.controller) == (g["method"], g["controller"])
    assert len(g["ys_points"]) == len(g["ys_values"]) == 2048 and len(g["n_steps"]) == g["batch"]
    assert all(s == 0 for s in g["status"]) and g["n_f_evals"] == 2 + 6 * max(g["n_steps"])


@pytest.mark.parametrize("path", [p for p in GOLDEN if not p.endswith(("_tolerance.json", "_mixed.json", "_fixed.json", "_low_order.json", "_early_stop.json"))], ids=os.path.basename)
def test_oracle_reproduces_golden_fixture(path):
    g = json.load(open(path))
    dtype = getattr(torch, g["dtype"])
    w = to.workloads.make(g["workload"], batch=g["batch"], dtype=dtype)
    assert {"y0": _sha(w.y0), "t_eval": _sha(w.t_eval), "params": _sha(w.f.builtin_params())} == g["inputs_sha256"]
    cfg = c_oracle.make_config(method=g["method"], term=g["workload"], nthreads=4, **g["controller"])
    out = c_oracle.solve(cfg, w.f.builtin_params(), w.y0, w.t_eval)
    for key in ("n_steps", "n_accepted", "n_initialized", "status"):
        if isinstance(g[key], dict):
            assert _sha(out[key]) == g[key]["sha256_int64"] and int(out[key].sum()) == g[key]["sum"], key
        else:
            assert out[key].tolist() == g[key], key
    assert _sha(out["ys"]) == g["ys_sha256"]
    assert int(out["n_f_evals"][0]) == g["n_f_evals"]
    got = [float(v).hex() for v in out["ys"][g["subset"]].flatten().tolist()]
    assert got == g["ys_subset"]
    assert float(out["ys"].double().abs().max()).hex() == g["ys_max_abs"]


@pytest.mark.parametrize("path", [p for p in GOLDEN if p.endswith("_early_stop.json")], ids=os.path.basename)
def test_oracle_reproduces_early_stop_fixture(path):
    """No evaluation points and every sample stopped by max_steps (tests/golden/make_golden.py::make_early_stop): the
    value returned is the last step's interpolant far outside its step, where the last place of Tsit5's dense-output
    weights shows in the result."""
    g = json.load(open(path))
    dtype = getattr(torch, g["dtype"])
    w = to.workloads.make(g["workload"], batch=g["batch"], dtype=dtype)
    t_start, t_end = w.t_eval[:, 0].clone(), w.t_eval[:, -1].clone()
    assert {"y0": _sha(w.y0), "t_start": _sha(t_start), "t_end": _sha(t_end), "params": _sha(w.f.builtin_params())} == g["inputs_sha256"]
    cfg = c_oracle.make_config(method=g["method"], term=g["workload"], nthreads=4, max_steps=g["max_steps"], **g["controller"])
    out = c_oracle.solve(cfg, w.f.builtin_params(), w.y0, None, t_start=t_start, t_end=t_end)
    for key in ("n_steps", "n_accepted", "n_initialized", "status"):
        assert out[key].tolist() == g[key], key
    assert all(s == 3 for s in g["status"]) and int(out["n_f_evals"][0]) == g["n_f_evals"] == 2 + 6 * g["max_steps"]
    assert [float(v).hex() for v in out["ys"].flatten().tolist()] == g["ys"] and _sha(out["ys"]) == g["ys_sha256"]


def test_mlp_weights_in_one_row_major_block():
    f = to.workloads.make("mlp", batch=4).f
    raw = f.builtin_shared()
    assert raw.shape == (256 * 65 + 256 + 64 * 256 + 64,)
    assert torch.equal(raw[: 256 * 65], f.W1.reshape(-1)) and torch.equal(raw[256 * 65 : 256 * 65 + 256], f.b1)
    assert torch.equal(raw[256 * 65 + 256 : -64], f.W2.reshape(-1)) and torch.equal(raw[-64:], f.b2)


def test_torch_compile_wrapper_hands_out_the_solvers_own_solve():
    """torch.compile(solver) wraps the module; `.solve` on the wrapper is the wrapped solver's bound
    method, so the idiom of the reference's README and tests/torch_script_test.py:17-21 runs this
    library's solve unchanged."""
    term = to.ODETerm(torch.nn.Linear(2, 2))
    for cls in (to.AutoDiffAdjoint, to.BacksolveAdjoint, to.JointBacksolveAdjoint):
        args = (to.Tsit5(), to.IntegralController(1e-3, 1e-3))
        solver = cls(*args) if cls is to.AutoDiffAdjoint else cls(term, *args)
        wrapped = torch.compile(solver)
        assert wrapped.solve.__self__ is solver and wrapped.solve.__func__ is cls.solve


@pytest.mark.parametrize("path", [p for p in GOLDEN if p.endswith("_mixed.json")], ids=os.path.basename)
def test_mixed_dtype_fixture_is_well_formed(path):
    """Vectors of the ATen-op oracle with time and data in different dtypes (tests/golden/make_golden.py::make_mixed);
    the inputs they belong to are the float64 workload rounded to the two dtypes."""
    g = json.load(open(path))
    time_dtype, data_dtype = getattr(torch, g["time_dtype"]), getattr(torch, g["data_dtype"])
    assert time_dtype != data_dtype
    w = to.workloads.make(g["workload"], batch=g["batch"], dtype=torch.float64)
    got = {"y0": _sha(w.y0.to(data_dtype)), "t_eval": _sha(w.t_eval.to(time_dtype)), "params": _sha(w.f.builtin_params().to(data_dtype))}
    assert got == g["inputs_sha256"]
    assert len(g["n_steps"]) == g["batch"] and all(s == 0 for s in g["status"]) and g["n_f_evals"] == 2 + 6 * max(g["n_steps"])


@pytest.mark.parametrize("path", [p for p in GOLDEN if p.endswith("_fixed.json")], ids=os.path.basename)
def test_fixed_step_fixture_is_well_formed_and_reproducible_here(path):
    """Vectors of the ATen-op oracle with the reference's FixedStepController (tests/golden/make_golden.py::make_fixed)."""
    g = json.load(open(path))
    dtype = getattr(torch, g["dtype"])
    w = to.workloads.make(g["workload"], batch=g["batch"], dtype=dtype)
    assert {k: v for k, v in g["inputs_sha256"].items() if k != "dt0"} == {"y0": _sha(w.y0), "t_eval": _sha(w.t_eval), "params": _sha(w.f.builtin_params())}
    assert g["n_steps"] == g["n_accepted"] and all(61 <= n <= 68 for n in g["n_steps"]) and g["n_f_evals"] == 1 + 6 * max(g["n_steps"])
    assert all(s == 0 for s in g["status"]) and all(n == 50 or n == 20 for n in g["n_initialized"])


@pytest.mark.parametrize("path", [p for p in GOLDEN if p.endswith("_low_order.json")], ids=os.path.basename)
def test_low_order_fixture_is_well_formed(path):
    """Vectors of the ATen-op oracle with Heun and Euler (tests/golden/make_golden.py::make_low_order): the inputs are
    the workload's, every sample finished, and the evaluation count follows from the step count (two per Heun step,
    one per Euler step, two more where the first step size is chosen automatically)."""
    g = json.load(open(path))
    w = to.workloads.make(g["workload"], batch=g["batch"], dtype=getattr(torch, g["dtype"]))
    assert g["inputs_sha256"] == {"y0": _sha(w.y0), "t_eval": _sha(w.t_eval), "params": _sha(w.f.builtin_params())}
    per_step, first = {"heun": 2, "euler": 1}[g["method"]], 2 if g["first_step_parts"] is None else 0
    assert g["n_f_evals"] == first + per_step * max(g["n_steps"]) and all(s == 0 for s in g["status"])
    assert all(n == w.t_eval.shape[1] for n in g["n_initialized"]) and g["ys_finite_fraction"] == 1.0
    assert g["bit_exact"] == (g["first_step_parts"] is not None)  # (the controller's own first step takes x ** 0.5)
    if g["controller"]["kind"] == "fixed" or g["method"] == "euler":
        assert g["n_steps"] == g["n_accepted"]  # nothing to reject without an error estimate or with fixed steps
    else:
        assert all(a <= n for a, n in zip(g["n_accepted"], g["n_steps"]))


def test_names_the_reference_keeps_in_its_adjoints_and_interpolation_modules():
    """``from torchode.adjoints import BacksolveAdjoint`` and the like keep working after the switch (reference
    adjoints.py:15, 322, 510; interpolation.py:8, 25)."""
    from torchode_amd import adjoints, backsolve, interpolation

    assert adjoints.BacksolveAdjoint is backsolve.BacksolveAdjoint and adjoints.JointBacksolveAdjoint is backsolve.JointBacksolveAdjoint
    assert callable(interpolation.poly3eval) and callable(interpolation.poly4eval)
    import importlib

    for module, name in (("tsit5", "Tsit5"), ("dopri5", "Dopri5"), ("heun", "Heun"), ("euler", "Euler")):
        assert getattr(importlib.import_module(f"torchode_amd.single_step_methods.{module}"), name) is getattr(to, name)
    with pytest.raises(NotImplementedError):
        adjoints.Adjoint().solve(None)
    with pytest.raises(AttributeError):
        adjoints.no_such_name


def test_typing_names_and_predicates():
    """reference typing.py:7-36 (the three predicates) and :44-95 (the tensor names, plain ``torch.Tensor`` here)."""
    from torchode_amd import typing as ty

    a, b, c = torch.zeros(2, 3), torch.zeros(2, 4), torch.zeros(2, 3, dtype=torch.float64)
    assert ty.same_shape(a, b, dim=0) and not ty.same_shape(a, b) and not ty.same_shape(a, b, dim=1) and ty.same_shape(a, c)
    assert ty.same_dtype(a, b) and not ty.same_dtype(a, b, c) and ty.same_device(a, b, c) and ty.same_dtype() and ty.same_shape(a)
    for name in ("DataTensor", "NormTensor", "SolutionDataTensor", "TimeTensor", "EvaluationTimesTensor", "AcceptTensor", "StatusTensor",
                 "InterpTimeTensor", "InterpDataTensor", "SampleIndexTensor"):  # fmt: skip
        assert getattr(ty, name) is torch.Tensor


def test_no_register_copy_ahead_of_the_exec_mask_restore(tmp_path):
    """The device assembly of every translation unit, searched for the one miscompilation met so far: copies of vector
    registers to accumulation registers placed at the end of a divergent region ahead of the instruction that restores
    the execution mask, which lanes that skipped the region then miss (torchode_amd/build.py).  Four instantiations of
    the one-kernel reverse sweep had it -- gradients of the parameters wrong by tens of per cent for samples without an
    evaluation point left, no error -- until the region was written as a loop the wavefront runs together."""
    import shutil

    from torchode_amd import build

    if shutil.which("hipcc") is None and not os.path.exists("/opt/rocm/bin/hipcc"):
        pytest.skip("no hipcc here")
    for path in build.emit_assembly(str(tmp_path)):
        assert build.copies_ahead_of_the_exec_restore(path) == [], path

