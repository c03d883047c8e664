"""What the host makes of a persistent launch's results when a bounded wait failed (CPU: the rules of the
launch headers, compiled with the host compiler).

A wait that fails marks the results of its launch whatever the controller's status says: the controller may
have taken its last verdict before (the dense output's stages of the last step), and only one workgroup
writes its status."""
import subprocess

import pytest

from conftest import PACKAGE_DIR

CSRC = PACKAGE_DIR / "csrc"


def run(tmp_path, body, *includes):
    """Compile and run a host program over the launch headers; its output's words."""
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    head = "".join(f'#include "{h}"\n' for h in includes)
    src.write_text(f"#include <stdio.h>\n{head}int main() {{\n{body}\nreturn 0; }}\n")
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", f"-I{CSRC}", "-o", str(exe),
                    str(src)], check=True)
    return subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split()


@pytest.mark.parametrize("status", ["RC_ST_OK", "RC_ST_MAX_STEPS", "RC_ST_NONFINITE"])
def test_trajectory_system_with_a_failed_wait(tmp_path, status):
    out = run(tmp_path, f"""
        double out[RC_OUT_STRIDE] = {{0}};
        out[RC_OUT_STATUS] = {status};
        const int without = rc_system_status(out);
        out[RC_OUT_WAIT_FAILED] = 1.0;   // by any workgroup, also after the last verdict
        printf("%d %d\\n", without == {status}, rc_system_status(out) == RC_ST_WAIT_LIMIT);""", "trajectory.h")
    assert out == ["1", "1"]


def test_trajectory_results_have_a_place_each(tmp_path):
    """The mark lies between the counters and the phase timers."""
    out = run(tmp_path, """
        printf("%d %d\\n", RC_OUT_WAIT_FAILED > RC_OUT_NEXTPOINT && RC_OUT_WAIT_FAILED < RC_OUT_TIMERS,
               RC_OUT_TIMERS + RC_NTIMERS <= RC_OUT_STRIDE);""", "trajectory.h")
    assert out == ["1", "1"]


def test_integration_launch_with_its_abort_word_set(tmp_path):
    """The action ODE's launch: another workgroup than the one that reports may have left early."""
    out = run(tmp_path, """
        printf("%d %d %d\\n", rc_launch_status(RC_ST_OK, 0) == RC_ST_OK, rc_launch_status(RC_ST_OK, 1) == RC_ST_WAIT_LIMIT,
               rc_launch_status(RC_ST_NONFINITE, 0) == RC_ST_NONFINITE);""", "trajectory.h")
    assert out == ["1", "1", "1"]


def test_each_equation_of_a_fused_launch_has_its_own_outcome(tmp_path):
    """Three equations of one launch: accepted, a wait that failed, a residual above the bar (and NaN).  Only
    the failed ones carry a code, so the evaluations beside them in a batch are complete."""
    out = run(tmp_path, """
        const double q[4][8] = {{0, 1, 17, 1e-14, 2.0, 1e-13, 0, 0}, {7, 0, 3, 0, 0, 0, 0, 0},
                                {0, 0, 200, 1e-3, 0.5, 1e-3, 0, 0}, {0, 0, 2, __builtin_nan(""), 1.0, __builtin_nan(""), 0, 0}};
        for (const double* o : q) printf("%d ", rc_gmres_code(rc_gmres_result(o), 2e-10, 10));
        const RcGmresResult r = rc_gmres_result(q[0]);
        printf("%d %d\\n", r.converged && r.matvecs == 17 && r.resid == 1e-14 && r.nb == 2.0 && r.true_res == 1e-13,
               rc_gmres_code({0, true, 1, 0.0, 2.0, 3e-10}, 2e-10, 10));""", "gmres.h")
    assert out == ["0", "7", "10", "10", "1", "0"]
