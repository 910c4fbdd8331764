"""Compile flags that results depend on (no GPU: the device code is compiled to LLVM IR, nothing runs)."""
import os
import subprocess

from kiln_amd import build


def test_nan_arithmetic_is_kept_where_results_rest_on_it(tmp_path):
    """linear_f32.hip recomputes the outputs whose sum is NaN. Compiled with NaNs declared impossible (the flag of the
    other kernels), inf - inf in its split of x and the loop that ends on a NaN would be the compiler's to fold away: no
    instruction of its device code may carry that promise (`nnan` or `fast`)."""
    out = tmp_path / "linear_f32.ll"
    subprocess.run([build.HIPCC, "-x", "hip", *build.flags("linear_f32.hip"), "--cuda-device-only", "-S", "-emit-llvm",
                    os.path.join(build.CSRC, "linear_f32.hip"), "-o", str(out)], check=True, capture_output=True)
    ir = out.read_text()
    assert "k_linear_x3" in ir and "fsub" in ir
    body = [ln for ln in ir.splitlines() if ln.startswith("  ")]
    assert not [ln for ln in body if " nnan " in ln or " fast " in ln]
    assert '"no-nans-fp-math"="true"' not in ir
