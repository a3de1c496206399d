"""The whole-solve kernels of the small systems, compiled for the host (tests/host_wavefront): with the address sanitizer and
one lane per wavefront, what their loops do on inputs whose times leave the range of the type; their short form of
the division; and their reverse sweep."""
import os
import re
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
# one-instruction maxima and minima in the kernels' source, and what they return for operands that the host compares
OPERATIONS = {"v_max": "fmax", "v_min": "fmin"}


@pytest.fixture(scope="module")
def sources(tmp_path_factory):
    """A copy of the kernels' sources that the host's compiler takes; returns the compiler's command up to its file."""
    if shutil.which("g++") is None:
        pytest.skip("no g++ here")
    build = tmp_path_factory.mktemp("host_wavefront")
    csrc = os.path.join(build, "torchode_amd", "csrc")
    shutil.copytree(os.path.join(ROOT, "torchode_amd", "csrc"), csrc)
    shutil.copytree(os.path.join(ROOT, "include"), os.path.join(build, "include"))

    def operation(m):
        a, b = (re.sub(r"\|(%\d)\|", r"fabs(\1)", x).replace("%1", "a").replace("%2", "b") for x in m.group(2).split(", "))
        return f"r = {OPERATIONS[m.group(1)]}({a}, {b});"

    for name in ("tode_math.h", "tode_solve.h", "tode_fast.hip", "tode_pair.hip", "tode_backward.hip"):
        path = os.path.join(csrc, name)
        text = open(path).read()
        text = re.sub(r'asm\("(v_max|v_min)_f\d\d %0, ([^"]*)" : [^;]*;', operation, text)
        text = re.sub(r'asm volatile\(""[^;]*;', "", text)
        text = text.replace("extern __shared__ __align__(16) unsigned char smem_raw[];", "unsigned char *const smem_raw = host::lds;")
        open(path, "w").write(text)
    return str(build), ["g++", "-std=c++17", "-w", "-ffp-contract=off", "-pthread", f"-I{os.path.join(HERE, 'host_wavefront')}", f"-I{csrc}"]


@pytest.fixture(scope="module")
def program(sources):
    build, compiler = sources
    out = os.path.join(build, "main")
    subprocess.run([*compiler, "-O1", "-g", "-fsanitize=address", os.path.join(HERE, "host_wavefront", "main.cpp"), "-o", out], check=True, timeout=600)

    def run(*args):
        env = dict(os.environ, ASAN_OPTIONS="verify_asan_link_order=0")
        r = subprocess.run([out, *map(str, args)], capture_output=True, text=True, timeout=120, env=env)
        assert r.returncode == 0, r.stderr[-3000:]
        flag, steps, initialized, value = r.stdout.split()
        return int(flag), int(steps), int(initialized), float(value)

    return run


KERNELS = [(kernel, method) for kernel in ("fast", "pair") for method in ("dopri5", "tsit5")]


@pytest.mark.parametrize("kernel, method", KERNELS)
def test_an_ordinary_solve(program, kernel, method):
    """The harness itself: exp(-1) to the tolerance, the point counted, no flag."""
    flag, steps, initialized, value = program(kernel, "f32", method, 1.0, 1.0, 0.0, 1.0, 2.0)
    assert (flag, initialized) == (0, 1) and steps > 3 and abs(value - 0.36787944) < 1e-4


@pytest.mark.parametrize("dtype, largest", [("f32", 3.4e38), ("f64", 1.79e308)])
@pytest.mark.parametrize("sign", [1, -1], ids=["forwards", "backwards"])
@pytest.mark.parametrize("kernel, method", KERNELS)
def test_a_time_range_beyond_the_largest_value(program, kernel, method, sign, dtype, largest):
    """t_end - t_start overflows and the error estimate is zero: the step grows to infinity, and the step after it is not a
    number and carries the time to infinity.  The loop over the evaluation points ends at the last one all the same (it wrote
    past the end of ys for ever when the point behind the last one was an infinity that an infinite time has reached), and the
    batch is handed to the general kernel."""
    flag, _, initialized, value = program(kernel, dtype, method, 0.0, 1.0, -sign * largest, 0.0, sign * largest)
    assert flag == 1 and initialized <= 1


@pytest.mark.parametrize("dtype, far", [("f32", -3e38), ("f32", -1e30), ("f64", -1e308)])
@pytest.mark.parametrize("kernel, method", KERNELS)
def test_a_point_far_in_front_of_the_start(program, kernel, method, dtype, far):
    """A point so far in front of t_start that its position in units of the first step overflows: extrapolated to an infinity, as
    by the division (the product with the step's reciprocal made it an infinity less an infinity)."""
    flag, _, initialized, value = program(kernel, dtype, method, 1.0, 1.0, 1.0, far, 2.0)
    assert (flag, initialized) == (0, 1) and abs(value) == float("inf")


def test_reverse_sweep_against_its_general_forms(sources):
    """The one-kernel reverse sweep against the per-iteration reverse on random records: the same bits, whatever rule sends an
    operand to a short form and a row of times to the walk or to the lists."""
    build, compiler = sources
    out = os.path.join(build, "sweep")
    subprocess.run([*compiler, "-O1", "-march=native", "-fsanitize=address", os.path.join(HERE, "host_wavefront", "sweep.cpp"), "-o", out], check=True, timeout=600)
    env = dict(os.environ, ASAN_OPTIONS="verify_asan_link_order=0")
    r = subprocess.run([out, "0", "2000"], capture_output=True, text=True, timeout=300, env=env)
    assert r.returncode == 0 and r.stdout.split() == ["4000", "0"], (r.stdout, r.stderr[-2000:])


def test_reverse_sweep_by_one_wavefront(sources):
    """The same where one wavefront does all of it, as for batches that fill the GPU (rows of up to four values; the test above
    has them in two)."""
    build, compiler = sources
    out = os.path.join(build, "sweep_by_one")
    subprocess.run([*compiler, "-O1", "-march=native", "-fsanitize=address", "-DTODE_PAIRED_SWEEP_GROUPS=0", os.path.join(HERE, "host_wavefront", "sweep.cpp"), "-o", out], check=True, timeout=600)
    env = dict(os.environ, ASAN_OPTIONS="verify_asan_link_order=0")
    r = subprocess.run([out, "0", "1000"], capture_output=True, text=True, timeout=300, env=env)
    assert r.returncode == 0 and r.stdout.split() == ["2000", "0"], (r.stdout, r.stderr[-2000:])


def test_quotients_next_to_a_rounding_boundary(sources):
    """The short form of the float32 quotient, given the correctly rounded reciprocal, on all 46 517 418 pairs of mantissas
    whose quotient lies so close to a boundary that the form's error could take it to the other side."""
    build, compiler = sources
    out = os.path.join(build, "quotients")
    subprocess.run([*compiler, "-O2", "-march=native", os.path.join(HERE, "host_wavefront", "quotients.cpp"), "-o", out], check=True, timeout=600)
    r = subprocess.run([out], capture_output=True, text=True, timeout=600, check=True)
    assert r.stdout.split() == ["46517418", "0"]
