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


def _asm(name, tmp_path):
    src, out = _build.CSRC / "kernels" / name, tmp_path / "a.s"
    subprocess.run(["hipcc", f"--offload-arch={_build.ARCH}", "-O3", "-std=c++17", "-munsafe-fp-atomics", f"-I{src.parent}",
                    *_build.PER_FILE_FLAGS[src.name], "--cuda-device-only", "-S", str(src), "-o", str(out)], check=True,
                   stderr=subprocess.DEVNULL)
    return out.read_text()


def test_prefill_attention_compiles_to_none(tmp_path):
    asm = _asm("attention_prefill.hip", tmp_path)
    assert "v_mfma_f32_16x16x32_bf16" in asm and not re.search(r"v_pk_(add|mul|fma)_f32", asm)


def test_grouped_gemm_loops_start_on_a_cache_line(tmp_path):
    """The K loop of each gemm8g kernel: the block that a later branch goes back to over its 32 or 64 MFMAs."""
    kernels = re.findall(r"^(_ZN\w*gemm8g_kernel\w*):(.*?)s_endpgm", _asm("gemm8g.hip", tmp_path), re.S | re.M)
    assert len(kernels) == 6
    for name, body in kernels:
        parts = re.split(r"^(\.LBB\w+):", body, flags=re.M)
        labels, blocks = parts[1::2], parts[2::2]
        loops = [i for i, label in enumerate(labels) for j in range(i, len(labels))
                 if re.search(r"s_c?branch\w*\s+" + re.escape(label) + r"\b", blocks[j])
                 and "".join(blocks[i:j + 1]).count("v_mfma") >= 32]
        assert loops, name
        for i in loops:
            assert re.search(r"\.p2align\s+6", parts[2 * i].splitlines()[-1]), (name, labels[i])
