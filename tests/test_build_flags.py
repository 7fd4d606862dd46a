"""Code generation flags of the kernel files."""
import re
import subprocess

import pytest

from llm_weighted_consensus_amd import _build

FILES = ["attention_prefill.hip", "encoder_few.hip", "gemm1s.hip", "gemm2s.hip", "gemm8g.hip", "gemm8p.hip"]


@pytest.mark.parametrize("name", FILES)
def test_rewritten_kernels_hold_no_packed_fp32(name):
    """Built without packed fp32 instructions, beside the flags that a file has for other reasons."""
    flags = _build.PER_FILE_FLAGS[name]
    at = flags.index("-packed-fp32-ops") - 3
    assert flags[at:at + 4] == _build.NO_PACKED_FP32
    assert ("-amdgpu-mfma-vgpr-form=1" in flags) == (name == "attention_prefill.hip")


def test_prefill_attention_compiles_to_none(tmp_path):
    src, out = _build.CSRC / "kernels" / "attention_prefill.hip", tmp_path / "a.s"
    subprocess.run(["hipcc", f"--offload-arch={_build.ARCH}", "-O3", "-std=c++17", "-munsafe-fp-atomics", f"-I{src.parent}",
                    *_build.PER_FILE_FLAGS[src.name], "--cuda-device-only", "-S", str(src), "-o", str(out)], check=True,
                   stderr=subprocess.DEVNULL)
    asm = out.read_text()
    assert "v_mfma_f32_16x16x32_bf16" in asm and not re.search(r"v_pk_(add|mul|fma)_f32", asm)
