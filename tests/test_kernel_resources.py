"""Resource limits of the built gfx950 kernels, read from the code object's
AMDGPU metadata (no GPU needed).

A GEMM whose accumulators end up in scratch memory still computes the right
result but runs several times slower (the 256x256 QKV GEMM did, once, when its
epilogue loop was left rolled), so the parity tests cannot catch it; this test
does. It also checks the LDS and register budgets the kernels are written for.
"""
import os
import re
import shutil
import subprocess
import tempfile

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "rustane_amd", "libhip_bridge.so")
LLVM = "/opt/rocm/llvm/bin"
CSRC = os.path.join(ROOT, "rustane_amd", "csrc")


def _kernel_metadata():
    bundler = os.path.join(LLVM, "clang-offload-bundler")
    readelf = os.path.join(LLVM, "llvm-readelf")
    objcopy = shutil.which("objcopy") or os.path.join(LLVM, "llvm-objcopy")
    if not (os.path.exists(LIB) and os.path.exists(bundler) and os.path.exists(readelf)):
        pytest.skip("built library or ROCm LLVM tools not present")
    notes = ""
    with tempfile.TemporaryDirectory() as d:
        fat = os.path.join(d, "fat.bin")
        # objcopy rewrites its input file when no output file is named, which
        # would change the library under any process that has it mapped: write
        # the (unused) copy into the temporary directory instead.
        subprocess.run([objcopy, "--dump-section", f".hip_fatbin={fat}", LIB,
                        os.path.join(d, "lib_copy.so")], check=True,
                       capture_output=True)
        # one offload bundle per translation unit, concatenated; the bundler
        # reads only the first bundle of a file, so split them
        data = open(fat, "rb").read()
        magic = b"__CLANG_OFFLOAD_BUNDLE__"
        starts = [i for i in range(len(data)) if data.startswith(magic, i)]
        for n, (a, b) in enumerate(zip(starts, starts[1:] + [len(data)])):
            part, co = os.path.join(d, f"part{n}.bin"), os.path.join(d, f"part{n}.co")
            with open(part, "wb") as f:
                f.write(data[a:b])
            subprocess.run([bundler, "--type=o", "--unbundle", f"--input={part}", f"--output={co}",
                            "--targets=hipv4-amdgcn-amd-amdhsa--gfx950"], check=True,
                           capture_output=True)
            notes += subprocess.run([readelf, "--notes", co], check=True, capture_output=True,
                                    text=True).stdout
    kernels, cur = [], None
    for line in notes.splitlines():
        if line.startswith("  - "):  # a new entry of amdhsa.kernels
            cur = {}
            kernels.append(cur)
            line = "    " + line[4:]
        m = re.match(r"^    \.(\w+):\s+(\S+)", line)
        if cur is not None and m:
            cur[m.group(1)] = m.group(2)
    return [k for k in kernels if "name" in k]


def test_gemm_kernels_keep_accumulators_in_registers():
    ks = _kernel_metadata()
    gemms = [k for k in ks if "gemm_nt_kernel" in k["name"]]
    assert len(gemms) >= 7, "expected the GEMM tile instantiations in the library"
    for k in gemms:
        # a few spilled address registers outside the main loop are tolerated;
        # an accumulator tile in scratch would be >= 1 KiB
        assert int(k["private_segment_fixed_size"]) <= 128, (k["name"], k["private_segment_fixed_size"])


def test_register_array_kernels_use_no_scratch():
    """These keep tiles, rows or accumulators in registers up to the limit of
    their occupancy: nothing may be spilled, and an instance meant to run two
    workgroups of 4 waves to a CU needs at most 256 registers a lane."""
    ks = _kernel_metadata()
    for name, least in (("attn_prefill_kernel", 8), ("attn_bwd_dq_kernel", 4), ("attn_bwd_dkv_kernel", 4),
                        ("attn_decode_kernel", 8), ("ce_backward_kernel", 3), ("gemv_xreg_kernel", 11)):
        mine = [k for k in ks if name in k["name"]]
        assert len(mine) >= least, (name, len(mine))
        for k in mine:
            assert int(k["private_segment_fixed_size"]) == 0, (k["name"], k["private_segment_fixed_size"])
            two = ("attn_bwd_dq" in name or ("attn_bwd_dkv" in name and "Li4ELi1E" in k["name"]) or
                   ("attn_prefill" in name and "ELb0ELi" in k["name"]))
            if two:
                assert int(k["vgpr_count"]) <= 256, (k["name"], k["vgpr_count"])


def test_kernels_fit_the_cu():
    for k in _kernel_metadata():
        assert int(k["group_segment_fixed_size"]) <= 160 * 1024, k["name"]
        assert int(k["vgpr_count"]) <= 512, k["name"]
        assert k.get("uses_dynamic_stack", "false") == "false", k["name"]


def test_inline_asm_leaves_m0_to_the_compiler():
    """m0 cannot be listed as clobbered (the compiler reserves it and warns),
    so an asm block that writes it is invisible to code around it that uses it:
    the direct-to-LDS copies take it as an operand instead."""
    copies = 0
    for name in sorted(os.listdir(CSRC)):
        if not name.endswith((".hip", ".hpp")):
            continue
        text = open(os.path.join(CSRC, name)).read()
        for stmt in re.findall(r"\basm\b[^;]*;", text):
            template = "".join(re.findall(r'"((?:[^"\\]|\\.)*)"', stmt.split("::")[0]))
            assert not re.search(r"\bm0\b", template), (name, template)
            if re.search(r"buffer_load\w* .* lds\b", template):
                copies += 1
                assert '"{m0}"(' in stmt, (name, template)
    assert copies >= 2, "expected the direct-to-LDS copies in the sources"


def test_decode_gemvs_are_built_for_the_rows_they_get():
    """Split rows reach the projections of two-term layers and the logits, and
    QKV with low parts gets no others; the fragment-order gate is never written
    for one or two rows."""
    names = [k["name"] for k in _kernel_metadata() if re.search(r"gemv(_xreg)?_kernel", k["name"])]
    forms = {}
    for n in names:
        # <KS, U or XS, .., Epi, [PRO,] two flags>: the split flag is the last of
        # the register-row kernel's and the first of the plain kernel's
        m = re.search(r"gemv_(xreg_)?kernelI(?:Li\d+E)+NS_\d+(\w+?)(?:ILb(\d)ELi(\d)EE)?E(?:Li(\d+)E)?Lb(\d)ELb(\d)EE", n)
        assert m, n
        epi = m.group(2) + ("" if m.group(3) is None else f"<{m.group(3)},{m.group(4)}>")
        split = (m.group(7) if m.group(1) else m.group(6)) == "1"
        forms.setdefault(epi, set()).add((split, int(m.group(5) or 0)))
    few, wide = {(False, 3), (False, 4)}, {(False, 0), (False, 10)}  # PRO_NORM + rows
    assert forms == {
        "EpiResidual": {(False, 0), (False, 1), (True, 0)},
        "EpiSwiGLU": few | wide | {(True, 0)},
        "EpiSwiGLUFrag": wide,
        "EpiLogits": few | wide | {(True, 0)},
        "EpiQKVAt<1,0>": few | wide,
        "EpiQKVAt<1,1>": {(True, 0)},
    }, forms
