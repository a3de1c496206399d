"""The loops of the whole-solve kernels of the small systems, compiled for the host with the address sanitizer, one lane per
wavefront (tests/host_wavefront): what they do on inputs whose times or states leave the range of the type."""
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
def program(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("no g++ here")
    build = tmp_path_factory.mktemp("host_wavefront")
    csrc = os.path.join(build, "torchode_amd", "csrc")
    shutil.copytree(os.path.join(ROOT, "torchode_amd", "csrc"), csrc)
    shutil.copytree(os.path.join(ROOT, "include"), os.path.join(build, "include"))

    def operation(m):
        a, b = (re.sub(r"\|(%\d)\|", r"fabs(\1)", x).replace("%1", "a").replace("%2", "b") for x in m.group(2).split(", "))
        return f"r = {OPERATIONS[m.group(1)]}({a}, {b});"

    for name in ("tode_math.h", "tode_solve.h", "tode_fast.hip", "tode_pair.hip"):
        path = os.path.join(csrc, name)
        text = open(path).read()
        text = re.sub(r'asm\("(v_max|v_min)_f\d\d %0, ([^"]*)" : [^;]*;', operation, text)
        text = re.sub(r'asm volatile\(""[^;]*;', "", text)
        text = text.replace("extern __shared__ __align__(16) unsigned char smem_raw[];", "unsigned char *const smem_raw = host::lds;")
        open(path, "w").write(text)
    out = os.path.join(build, "main")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-w", "-ffp-contract=off", "-fsanitize=address", "-pthread", f"-I{os.path.join(HERE, 'host_wavefront')}",
                    f"-I{csrc}", os.path.join(HERE, "host_wavefront", "main.cpp"), "-o", out], check=True, timeout=600)  # fmt: skip

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
