"""The measured-slower attention variants, which compile only with -DMXLLM_ATTN_EXPERIMENTS, still do (host syntax and
template checks; no GPU)."""
import os
import shutil
import subprocess

import pytest

from mxllm import _build

HIPCC = os.path.join(_build.ROCM, "bin", "hipcc")


@pytest.mark.skipif(shutil.which(HIPCC) is None, reason="no hipcc")
@pytest.mark.parametrize("src", ["attn_fwd.hip", "attn_bwd.hip"])
def test_attention_experiments_compile(src):
    kernels = os.path.join(_build.CSRC, "kernels")
    r = subprocess.run([HIPCC, "-fsyntax-only", "-std=c++17", f"--offload-arch={_build.ARCH}", "-DMXLLM_ATTN_EXPERIMENTS",
                        "-Wno-unused-result", f"-I{_build.CSRC}", f"-I{kernels}", os.path.join(kernels, src)],
                       capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr[-2000:]
