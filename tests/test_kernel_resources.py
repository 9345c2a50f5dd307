"""Register-allocation guard for the hot HIP kernels (CPU: hipcc cross-compiles gfx950).

A kernel that spills to scratch turns its K/V stream into extra memory round trips per lane; a
harmless-looking refactor (a by-reference lambda around the attention work unit) once made every
paged-attention instantiation spill 176 B/lane and run ~1.3x slower on MI355X.  This compiles the
kernels with the flags of the build and ``-Rpass-analysis=kernel-resource-usage`` and fails on any scratch use.
"""
import functools
import os
import re
import shutil
import subprocess
import tempfile

import pytest

from distributed_llm_amd._build import HIP_FLAGS

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
KERNELS = ["attention.hip", "gemv.hip", "skinny_gemm.hip", "sampling.hip", "moe.hip",
           "flash_prefill.hip", "tgemm.hip", "encoder.hip", "gqa.hip", "delta.hip", "mlstm_chunk.hip",
           "chunk_scan.hip", "scan_chunk.hip", "seqmix.hip", "elementwise.hip", "decode_gemm.hip", "moe_decode.hip", "f32_gemm.hip",
           "latent.hip", "wide_gemm.hip", "outer_scan.hip", "norm.hip", "rope_kv.hip", "cosine.hip"]
# measured exceptions (bytes/lane allowed): the d=64 flash prefill at 4 waves per SIMD (128-VGPR cap,
# two workgroups per CU) keeps ~5 values in scratch around the chunk loop and is still 1.14-1.17x
# faster than the spill-free one-workgroup build (profiles/r2_flash_prefill_microbench.md)
ALLOW = {r"flash_prefill_kernelILi64ELi4E": 32}


@functools.lru_cache(maxsize=None)
def _usage(src):
    path = os.path.join(ROOT, "csrc", "kernels", src)
    with tempfile.TemporaryDirectory() as tmp:
        r = subprocess.run([HIPCC, *HIP_FLAGS, "-I", os.path.dirname(path), "-c", path, "-o", os.path.join(tmp, "k.o"),
                            "-Rpass-analysis=kernel-resource-usage"], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr[-2000:]
    return r.stderr


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not available")
@pytest.mark.parametrize("src", KERNELS)
def test_no_scratch_spills(src):
    out = _usage(src)
    names = re.findall(r"Function Name: (\S+)", out)
    scratch = [int(x) for x in re.findall(r"ScratchSize \[bytes/lane\]: (\d+)", out)]
    assert names and len(names) == len(scratch)
    budget = lambda n: max([v for k, v in ALLOW.items() if re.search(k, n)] or [0])
    spilled = [(n, s) for n, s in zip(names, scratch) if s > budget(n)]
    assert not spilled, f"scratch spills: {spilled}"


# What a wave may hold of the registers, where one workgroup more or less on a CU is a round of the launch: (source, kernel, waves a SIMD)
WAVES = [
    ("seqmix.hip", r"norm_resadd_reg_kernelI\w\wLi(16|32)E", 4),      # 1000 rows of 5120: 15 us, 21 with three
    ("seqmix.hip", r"norm_resadd_reg_kernelI\w\wLi64E", 2),
    ("gqa.hip", r"paged_gqa_mfma_kernelILi(128|192)E", 2),      # 24 decode rows of 192-wide heads: 14 us, 20 with one
    ("gqa.hip", r"paged_gqa_mfma_kernelILi96E", 3),
    ("gqa.hip", r"gqa_few_kernel", 2),
    ("gqa.hip", r"gqa_cols_kernelILi(64|96)E", 4),      # 96 / 64 with slopes holds 124 of 128
    ("gqa.hip", r"gqa_cols_kernelILi(128|192)E", 2),
]


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not available")
@pytest.mark.parametrize("src,kernel,waves", WAVES)
def test_waves_of_a_simd(src, kernel, waves):
    out = _usage(src)
    got = {n: int(w) for n, w in re.findall(r"Function Name: (\S+).*?Occupancy \[waves/SIMD\]: (\d+)", out, re.S) if re.search(kernel, n)}
    assert got and min(got.values()) >= waves, got


def _registers(operand):
    m = re.fullmatch(r"([va])(?:\[(\d+):(\d+)\]|(\d+))", operand)
    return {(m[1], i) for i in range(int(m[2] or m[4]), int(m[3] or m[4]) + 1)} if m else set()


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not available")
def test_inline_products_of_wide_gemm(tmp_path):
    """The compiler does not know that the inline instruction of wide_gemm.hip is a matrix product and keeps no distance from it: a
    vector instruction must not write an operand within two wait states ahead of one, and from the first product up to the wait behind the
    last nothing else may touch the accumulators."""
    path, out = os.path.join(ROOT, "csrc", "kernels", "wide_gemm.hip"), tmp_path / "k.s"
    r = subprocess.run([HIPCC, *HIP_FLAGS, "-I", os.path.dirname(path), "--cuda-device-only", "-S", path, "-o", str(out)],
                       capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr[-2000:]
    kernels = 0
    for text in re.split(r"\n(?=_Z\w+:)", out.read_text().split(".section\t.AMDGPU.metadata")[0])[1:]:
        ins, at = [], {}
        for line in text.split("\n"):
            line = line.split(";")[0].strip()
            if re.fullmatch(r"\.L\w+:", line):
                at[line[:-1]] = len(ins)
            elif re.match(r"[a-z]\w+(\s|$)", line):
                ins.append((line.split()[0], re.split(r",\s*", line.split(None, 1)[1]) if " " in line or "\t" in line else []))
        mul = [i for i, (op, _) in enumerate(ins) if op.startswith("v_mfma")]
        if not mul:
            continue
        kernels += 1
        ways = {}      # instruction: where a jump comes from
        for i, (op, args) in enumerate(ins):
            if "branch" in op and args and args[-1] in at:
                ways.setdefault(at[args[-1]], []).append(i)

        def ahead(i, states):
            """Instructions that can run within ``states`` wait states ahead of instruction i."""
            if states <= 0 or i < 0:
                return
            for j in [i - 1] + ways.get(i, []):
                if j >= 0 and (j != i - 1 or ins[j][0] not in ("s_branch", "s_endpgm")):
                    yield j
                    yield from ahead(j, states - (1 + int(ins[j][1][0]) if ins[j][0] == "s_nop" else 1))

        for i in mul:
            read = set().union(*(_registers(a) for a in ins[i][1][1:]))
            for j in ahead(i, 2):
                op, args = ins[j]
                assert not (op.startswith("v_") and not op.startswith("v_mfma") and _registers(args[0]) & read), (ins[j], ins[i])
        # (program order is the order of the steps: the loop, the stage before the last, the last)
        end = next(i for i in range(mul[-1], len(ins)) if ins[i][0] == "s_nop" and ins[i + 1][0] == "s_nop")
        assert int(ins[end][1][0]) + int(ins[end + 1][1][0]) + 2 >= 18
        for i in range(mul[0], end):
            if i not in mul:
                assert not any(x[0] == "a" for arg in ins[i][1] for x in _registers(arg)), ins[i]
    assert kernels == 7      # the epilogues
