"""bench.py's view of the kernels: every attention kernel of the decode graph is filed under its family, and no entry of the
table names a kernel that is gone."""
import re
from pathlib import Path

import pytest

import bench

CSRC = Path(__file__).resolve().parent.parent / "inferred-thoughts_amd" / "csrc"


def kernels(pattern):
    """names of the kernels that the sources matching `pattern` define"""
    return {n for f in CSRC.glob(pattern) for n in re.findall(r"__global__[^;{]*?\bvoid\s+(\w+)\s*\(", f.read_text())}


def test_attention_kernels_have_their_family():
    names = (kernels("k_attn.hip") | kernels("k_attn_decode.hip")) - {"attend_exact_k"}     # (exact mode has no such profile)
    assert len(names) >= 5, names
    for n in names:
        assert bench.decode_family(f"void itk::(anonymous namespace)::{n}<256, 8, true>(itk::AttnArgs, int)", 65536) == "attend", n


@pytest.mark.parametrize("begin", sorted(bench.DECODE_FAMILIES))
def test_every_entry_names_a_kernel(begin):
    assert any(n.startswith(begin) for n in kernels("*.hip"))


def test_the_output_head_is_told_from_the_other_products():
    name = "void itk::(anonymous namespace)::fused_gemv_fast_k<8, 2, 64, false, false>(itk::FusedGemvP)"
    assert bench.decode_family(name, 524288).startswith("lm_head")
    assert bench.decode_family(name, 131072).startswith("fused_gemv")
    for n in kernels("k_attn_prefill.hip") | {"moe_group_k"}:                               # the prompt's
        assert bench.decode_family(f"void itk::(anonymous namespace)::{n}<256, 8>(itk::AttnArgs)", 1024) is None, n


@pytest.mark.parametrize("n_tokens,exact", [(100, False), (5700, False), (5700, True)])
def test_a_familys_rate_is_held_against_an_instruction_of_the_same_rate(n_tokens, exact):
    """The ceiling's instruction does as many multiply-accumulates a cycle as the one that the kernels issue."""
    per_cycle = {"int8_32x32x32": 1024, "int8_16x16x64": 1024, "int8_16x16x32": 512, "f16_32x32x16": 512, "f16_16x16x32": 512,
                 "f16_16x16x16": 256, "f32_16x16x4": 32}
    import inferred_hip as ih
    for family, (issued, ceiling) in bench.prefill_instructions(n_tokens, exact).items():
        assert ceiling in ih.Hip.MFMA_KINDS
        assert per_cycle[issued] == per_cycle[ceiling], family
    # (NVFP4 experts: k_gemm_f16.hip's 32x32x16 and, keeping the CPU path's bits, k_gemm.hip's experts_nvfp4_k)
    issued = bench.prefill_instructions(n_tokens, exact)["moe_glu"][0]
    source = (CSRC / "k_gemm.hip").read_text().split("void experts_nvfp4_k(")[1].split("\n}\n")[0] if exact else (CSRC / "k_gemm_f16.hip").read_text()
    assert issued.replace("f16_", "mfma_f32_") in source
    wide = bench.prefill_instructions(n_tokens, exact)["matmul (dense"][0] == "int8_32x32x32"
    assert wide == (n_tokens >= 512)       # (most dense rows of a pass of 512 tokens go through k_gemm.hip's 32x32x32 products)
