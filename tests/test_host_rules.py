"""Host rules of the library that no GPU is needed for, compiled from its own sources into a small program."""
import os
import shutil
import subprocess

import pytest

from joshua_amd.build import HIPCC_FLAGS

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "joshua_amd", "csrc")


def run(tmp_path, text):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("no hipcc")
    src, exe = tmp_path / "rule.hip", tmp_path / "rule"
    src.write_text(text)
    res = subprocess.run([hipcc, *HIPCC_FLAGS, "-w", "-I", CSRC, "-I", os.path.join(ROOT, "include"), "-o", str(exe), str(src)],
                         capture_output=True, text=True, timeout=300)
    assert res.returncode == 0, res.stderr[-3000:]
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert res.returncode == 0, res.stdout + res.stderr
    return res.stdout


def test_capture_query_that_fails_does_not_fail_the_call(tmp_path):
    """A stream that cannot be asked whether it is captured (the null stream beside a blocking stream's capture) counts as captured."""
    assert "ok" in run(tmp_path, r"""
#include <hip/hip_runtime.h>
static hipError_t answer = hipSuccess;
static hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
static hipError_t asked(hipStream_t, hipStreamCaptureStatus *s) { return *s = status, answer; }
#define hipStreamIsCapturing asked
#include "split16.hip"
namespace jqh {
int fail(const char *, ...) { return 1; }
}
int main() {
    using namespace jqh;
    Split16Latent s{4, 640};
    s.ready = 300;
    split16_latent_overwrites(&s, 200, nullptr);
    if (s.ready != 200 || s.captured) return 1;
    answer = hipErrorStreamCaptureImplicit;
    split16_latent_overwrites(&s, 100, nullptr);
    if (s.ready != 100 || !s.captured) return 2;
    Split16Latent t{4, 640};
    answer = hipSuccess, status = hipStreamCaptureStatusActive;
    split16_latent_overwrites(&t, 0, nullptr);
    if (!t.captured) return 3;
    puts("ok");
}
""")


def test_offsets_of_the_f16_fp6_gemm_stay_in_their_registers(tmp_path):
    """Every byte that the kernel reads of a record's row group lies below 2^31 from its start, of 16 weight rows below 2^32, for the
    longest rows that the rule lets through, also where a paired matrix's rows lie two rows apart."""
    assert "ok" in run(tmp_path, r"""
#include <hip/hip_runtime.h>
#include "core.hpp"
#include "kernels_mfma_gemm_h6.hpp"
int main() {
    size_t longest = 0;
    for (size_t nb = 1; nb < (size_t)1 << 21; nb++)
        for (size_t apart : {144 * nb, 288 * nb})
            if (jq::h6_offsets_hold(nb, apart)) {
                longest = nb > longest ? nb : longest;
                if (nb * jq::H6_REC > 0x7FFFFFFFull || 15 * apart + 144 * nb > 0xFFFFFFFFull) return 1;
            }
    if (longest < 100000) return 2;
    puts("ok");
}
""")
