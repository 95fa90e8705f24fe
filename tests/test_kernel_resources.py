"""Register budgets the kernels' co-residency depends on, read from the gfx950
code objects of the built library (zealot_amd/_build/*.o).

A mixed runner step runs the chunk prefill (side stream) and the decode (cache
stream) together, each on part of every CU: one four-wave prefill workgroup and
two decode waves a CU.  The plan kernels are one 1024-thread workgroup (four
waves on every SIMD) that must start while those waves are resident; with more
than 64 VGPRs a lane the prefill plan cannot be placed beside a decode wave and
the chunks' attention runs after the decode instead of beside it (a regression
this file guards: 0.73 -> 0.87 ms a mixed step)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
BUILD = os.path.join(ROOT, "zealot_amd", "_build")
LLVM = "/opt/rocm/llvm/bin"
SIMD_VGPRS = 512  # unified VGPR + AGPR file of a gfx950 SIMD, per lane
GRANULE = 8


def _tools():
    bundler = os.path.join(LLVM, "clang-offload-bundler")
    readelf = os.path.join(LLVM, "llvm-readelf")
    objcopy = shutil.which("objcopy") or os.path.join(LLVM, "llvm-objcopy")
    if not all(os.path.exists(t) for t in (bundler, readelf, objcopy)):
        pytest.skip("ROCm LLVM tools not found")
    return bundler, readelf, objcopy


def kernel_registers(obj_name: str, tmp_path) -> dict:
    """{kernel symbol: (vgpr_count, agpr_count, private_segment_fixed_size)} of one object."""
    obj = os.path.join(BUILD, obj_name)
    if not os.path.exists(obj):
        pytest.skip(f"{obj_name} not built (run python -m zealot_amd.build)")
    bundler, readelf, objcopy = _tools()
    fb = tmp_path / (obj_name + ".fatbin")
    co = tmp_path / (obj_name + ".co")
    subprocess.run([objcopy, f"--dump-section=.hip_fatbin={fb}", obj, str(tmp_path / "scratch.o")], check=True,
                   capture_output=True)
    subprocess.run([bundler, "--unbundle", "--type=o", "--targets=hipv4-amdgcn-amd-amdhsa--gfx950",
                    f"--input={fb}", f"--output={co}"], check=True, capture_output=True)
    notes = subprocess.run([readelf, "--notes", str(co)], check=True, capture_output=True, text=True).stdout
    out, cur = {}, {}
    for line in notes.splitlines():
        s = line.strip()
        if s.startswith("- ") and cur:  # a new kernel's map starts
            if "name" in cur:
                out[cur["name"]] = (cur.get("vgpr", 0), cur.get("agpr", 0), cur.get("priv", 0))
            cur = {}
        s = s[2:] if s.startswith("- ") else s
        key, _, val = s.partition(":")
        val = val.strip()
        if key == ".name":
            cur["name"] = val
        elif key == ".vgpr_count":
            cur["vgpr"] = int(val)
        elif key == ".agpr_count":
            cur["agpr"] = int(val)
        elif key == ".private_segment_fixed_size":
            cur["priv"] = int(val)
    if "name" in cur:
        out[cur["name"]] = (cur.get("vgpr", 0), cur.get("agpr", 0), cur.get("priv", 0))
    return out


def _alloc(vgprs: int) -> int:
    return -(-vgprs // GRANULE) * GRANULE


def _one(regs: dict, needle: str):
    hits = [k for k in regs if needle in k]
    assert len(hits) == 1, f"{needle}: {hits}"
    return regs[hits[0]]


def _all(regs: dict, needle: str) -> dict:
    hits = {k: v for k, v in regs.items() if needle in k}
    assert hits, f"no kernel matching {needle}"
    return hits


# template arguments: cache type (0 f32, 1 bf16, 2 fp8), head size, heads a
# kv-head, planless, and for the decode row groups and shared prefixes
MIXED_DECODE = "decode_mfma_kernelILi1ELi128ELi4ELb0ELb0ELb0E"  # the mixed step's: bf16, planned


def test_plan_kernels_fit_beside_attention_waves(tmp_path):
    dec = kernel_registers("paged_decode.o", tmp_path)
    pre = kernel_registers("paged_prefill.o", tmp_path)
    plan = _one(dec, "11plan_kernelENS_6Params")
    pplan = _one(pre, "prefill_plan_kernel")
    decode = _one(dec, MIXED_DECODE)
    for name, (v, a, priv) in (("plan_kernel", plan), ("prefill_plan_kernel", pplan)):
        assert v + a <= 64, f"{name}: {v} VGPRs + {a} AGPRs a lane (at most 64)"
        assert priv == 0, f"{name} spills {priv} bytes a lane"
        # four of its waves on a SIMD beside one resident decode wave
        assert 4 * _alloc(v + a) + _alloc(decode[0] + decode[1]) <= SIMD_VGPRS


def test_attention_kernels_register_budgets(tmp_path):
    """The prefill kernel runs two waves a SIMD (two four-wave workgroups a
    CU), so a wave holds at most 256 registers; the planned decode kernel one
    wave a SIMD, the planless one two and more where LDS allows (20 KB a wave
    and less: everything but f32 at a head size of 128).  In a mixed step a
    prefill wave and a decode wave may share a SIMD.  No instantiation of
    either kernel spills."""
    dec = kernel_registers("paged_decode.o", tmp_path)
    pre = kernel_registers("paged_prefill.o", tmp_path)
    attention = {**_all(dec, "decode_mfma_kernel"), **_all(pre, "prefill_mfma_kernel")}
    for name, (v, a, priv) in attention.items():
        assert priv == 0, f"{name} spills {priv} bytes a lane"
        one_wave = "decode_mfma_kernelILi0ELi128E" in name
        assert _alloc(v + a) <= (SIMD_VGPRS if one_wave else SIMD_VGPRS // 2), f"{name}: {v} + {a}"
    decode = _one(dec, MIXED_DECODE)
    for planless in (0, 1):
        prefill = _one(pre, f"prefill_mfma_kernelILi1ELi128ELi4ELb{planless}E")
        assert _alloc(decode[0] + decode[1]) + _alloc(prefill[0] + prefill[1]) <= SIMD_VGPRS
