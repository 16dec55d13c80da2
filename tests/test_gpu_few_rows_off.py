"""The kernels that few_rows and few_rows_many took products over from.  They still run where those decline: activations or weights off 16 bytes,
a row length that is no whole number of super-blocks, prepared activations that a fixed scratch does not hold."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
TESTS = ("q4k_few_rows or few_rows_against or decoded_weights_gemm_split or kernel_chosen_for_a_shape or q4k_random_shapes or other_formats_random_shapes "
         "or int8_gemm_at_random_large_shapes or reference_model_shapes")


def test_products_of_few_rows_without_those_kernels():
    """The switch is read at the first product, hence the child process; the tests of those kernels name them there."""
    res = subprocess.run([sys.executable, "-m", "pytest", "-x", "-q", "-p", "no:cacheprovider", "tests/test_gpu_matmul.py", "-m", "gpu", "-k", TESTS], cwd=ROOT,
                         env=dict(os.environ, JQ_FEW_ROWS="0"), capture_output=True, text=True, timeout=110)
    assert res.returncode == 0 and " passed" in res.stdout, res.stdout[-3000:] + res.stderr[-1000:]
