"""The hot GEMM kernels must fit the register file: a kernel that spills keeps running, only slower (its scratch
reloads wait behind the operand loads in flight), so nothing else would notice.  Compiles the two GEMM sources to
gfx950 assembly with the library's own flags (no GPU needed) and reads the kernel descriptors."""
import importlib.util
import os
import re
import shutil
import subprocess

import pytest

from conftest import ROOT

PKG = os.path.join(ROOT, "triton-int8_amd")


def _build_module():
    spec = importlib.util.spec_from_file_location("ti8_build", os.path.join(PKG, "build.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


def compile_to_asm(source, tmp_path):
    """Path of the gfx950 assembly of one kernel source, compiled with the library's own flags."""
    b = _build_module()
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    if not (os.path.exists(hipcc) or shutil.which(hipcc)):
        pytest.skip("hipcc not available")
    out = str(tmp_path / (source + ".s"))
    flags = [f for f in b.FLAGS if f not in ("-shared", "-fPIC")]
    res = subprocess.run([hipcc] + flags + ["--cuda-device-only", "-S", "-o", out, os.path.join(b.CSRC, source)],
                         stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert res.returncode == 0, res.stdout[-2000:]
    return out


def kernel_resources(source, tmp_path):
    out = compile_to_asm(source, tmp_path)
    kernels = {}
    for m in re.finditer(r"\.amdhsa_kernel (\S+)(.*?)\.end_amdhsa_kernel", open(out).read(), flags=re.S):
        body = m.group(2)
        kernels[m.group(1)] = {k: int(re.search(r"\.amdhsa_" + k + r" (\d+)", body).group(1))
                               for k in ("private_segment_fixed_size", "next_free_vgpr", "next_free_sgpr")}
    return kernels


def test_persistent_chain_kernel_does_not_spill(tmp_path):
    kernels = kernel_resources("gemm_chain.hip", tmp_path)
    chain = [v for k, v in kernels.items() if "gemm_i8_chain_kernel" in k]
    assert len(chain) == 1
    assert chain[0]["private_segment_fixed_size"] == 0, chain[0]     # no scratch
    assert chain[0]["next_free_vgpr"] <= 256                          # two waves per SIMD


def test_tiled_gemm_kernels_do_not_spill(tmp_path):
    kernels = kernel_resources("gemm.hip", tmp_path)
    # 256 x 256 and 256 x 128 tiles run 8 waves of up to 256 registers; only the literal-arithmetic kernel (not tuned) may spill
    hot = {k: v for k, v in kernels.items() if "gemm_i8" in k and "ELi3EEE" not in k}
    assert len(hot) >= 8
    for name, v in hot.items():
        assert v["private_segment_fixed_size"] == 0, (name, v)
        assert v["next_free_vgpr"] <= 256, (name, v)


def test_persistent_chain_kernel_waits_match_its_stores(tmp_path):
    """The persistent kernel lets its epilogue stores drain under the next tile's first K tile: it waits with
    `s_waitcnt vmcnt(n)`, n = the stores a wave issued last, for everything issued BEFORE them (the next tile's operand
    and factor loads).  That is only safe while n does not exceed the stores really emitted, so the count in the source
    (EPILOGUE_STORES = 16: one 16-byte store per lane and row) is checked against the code the toolchain produces:
    every variant of the epilogue must hold exactly 16 global stores, all of them 16 bytes wide, and the two waits
    must carry that count (plus the 4 operand loads issued behind the factor loads)."""
    text = open(compile_to_asm("gemm_chain.hip", tmp_path)).read()
    body = text[text.index("gemm_i8_chain_kernel"):]
    body = body[:body.index(".end_amdhsa_kernel")]
    src = open(os.path.join(PKG, "csrc", "gemm_chain.hip")).read()
    m = re.search(r"static_assert\(RPI == 8 && STORES_PER_PASS == 2 && EPILOGUE_STORES == (\d+)", src)
    assert m, "the source no longer pins EPILOGUE_STORES"
    stores_per_wave = int(m.group(1))
    stores = re.findall(r"^\s*(global_store_\w+|buffer_store_\w+|flat_store_\w+|scratch_store_\w+)", body, flags=re.M)
    assert stores and set(stores) == {"global_store_dwordx4"}, sorted(set(stores))
    variants = 8          # extra factor x row scales x column scales, each a compile-time copy of the store loop
    assert len(stores) == variants * stores_per_wave, (len(stores), stores_per_wave)
    # straight-line check: between two branch targets / branches no more than one variant's stores
    for block in re.split(r"^\.LBB\S+:|^\s*s_cbranch\w+|^\s*s_branch", body, flags=re.M):
        n = len(re.findall(r"^\s*global_store_dwordx4", block, flags=re.M))
        assert n in (0, stores_per_wave), n
    waits = set(re.findall(r"s_waitcnt vmcnt\((\d+)\)", body))
    assert str(stores_per_wave) in waits, waits              # first K tile of a tile: everything but the stores
    assert str(stores_per_wave + 4) in waits, waits          # next tile's factors: behind 4 operand loads and the stores
    assert all(int(w) <= stores_per_wave + 4 for w in waits), waits


def test_chain_kernel_with_a_bias_waits_like_the_one_without(tmp_path):
    """The same 16 stores of 16 bytes per wave and variant, nothing branching between them, no more waited for than without the bias,
    and no scratch."""
    text = open(compile_to_asm("gemm_chain.hip", tmp_path)).read()
    body = text[text.index("gemm_i8_chain_bias_kernel"):]
    body = body[:body.index(".end_amdhsa_kernel")]
    assert re.search(r"\.amdhsa_private_segment_fixed_size 0\b", body)
    stores = re.findall(r"^\s*(global_store_\w+|buffer_store_\w+|flat_store_\w+|scratch_store_\w+)", body, flags=re.M)
    assert stores == ["global_store_dwordx4"] * (8 * 16)
    for block in re.split(r"^\.LBB\S+:|^\s*s_cbranch\w+|^\s*s_branch", body, flags=re.M):
        assert len(re.findall(r"^\s*global_store_dwordx4", block, flags=re.M)) in (0, 16)
    waits = {int(w) for w in re.findall(r"s_waitcnt vmcnt\((\d+)\)", body)}
    assert {16, 20} <= waits and max(waits) == 20


VMEM = r"((?:global|buffer|flat|scratch)_(?:load|store|atomic)\w*)"


def kernel_bodies(source, tmp_path, name):
    text = open(compile_to_asm(source, tmp_path)).read()
    bodies = {m.group(1): m.group(0) for m in re.finditer(r"^(_Z\w*" + name + r"\w*):.*?\.end_amdhsa_kernel", text, flags=re.S | re.M)}
    assert bodies
    return bodies


def loops(body):
    """Text between a label and the last branch back to it."""
    for m in re.finditer(r"^(\.LBB\w+):", body, flags=re.M):
        back = list(re.finditer(r"^\s*s_c?branch\w* " + re.escape(m.group(1)) + r"\b", body[m.end():], flags=re.M))
        if back:
            yield body[m.end():m.end() + back[-1].end()]


# tiles from lists; operand B scaled per (row, K tile), whose epilogue has no column scales
@pytest.mark.parametrize("name, variants", [("gemm_i8_chain_listed_kernel", 8), ("gemm_i8_chain_lane_kernel", 4)])
def test_other_forms_of_the_chain_kernel_wait_like_it(tmp_path, name, variants):
    """As above: 16 stores of 16 bytes per variant of the epilogue in one piece, waits for 16 and 20, no scratch, two waves per SIMD."""
    (body,) = kernel_bodies("gemm_chain.hip", tmp_path, name).values()
    assert re.search(r"\.amdhsa_private_segment_fixed_size 0\b", body)
    assert int(re.search(r"\.amdhsa_next_free_vgpr (\d+)", body).group(1)) <= 256
    stores = re.findall(r"^\s*(global_store_\w+|buffer_store_\w+|flat_store_\w+|scratch_store_\w+)", body, flags=re.M)
    assert stores == ["global_store_dwordx4"] * (variants * 16)
    for block in re.split(r"^\.LBB\S+:|^\s*s_cbranch\w+|^\s*s_branch", body, flags=re.M):
        assert len(re.findall(r"^\s*global_store_dwordx4", block, flags=re.M)) in (0, 16)
    waits = {int(w) for w in re.findall(r"s_waitcnt vmcnt\((\d+)\)", body)}
    assert {16, 20} <= waits and max(waits) == 20


def test_few_tokens_kernel_waits_match_its_stores(tmp_path):
    """The walk over dW's tiles waits with vmcnt(8) for the next K tile while the stores of the tile before may be in flight: safe while
    a wave issues exactly 8 memory instructions behind that K tile's loads, its stores of 16 bytes, with nothing branching between."""
    src = open(os.path.join(PKG, "csrc", "gemm_skinny.hip")).read()
    assert re.search(r"THIN_STORES = 8;", src)
    for name, body in kernel_bodies("gemm_skinny.hip", tmp_path, "gemm_i8_few_kernel").items():
        walks = 2 if "ILb0E" in name else 1         # operand A of dW scaled by blocks or by rows; int32 sums: by rows
        assert re.search(r"\.amdhsa_private_segment_fixed_size 0\b", body), name
        blocks = [re.findall(r"^\s*" + VMEM, b, flags=re.M) for b in re.split(r"^\.LBB\S+:|^\s*s_cbranch\w+|^\s*s_branch", body, flags=re.M)]
        stores = [b for b in blocks if "global_store_dwordx4" in b]
        assert stores == [["global_store_dwordx4"] * 8] * walks, (name, stores)
        assert len(re.findall(r"s_waitcnt vmcnt\(8\) lgkmcnt\(0\)", body)) == walks, name
        # the eight loads of a K tile, in front of the walk and in it, also in one piece
        tiles = [b for b in blocks if b == ["global_load_lds_dwordx4"] * 8]
        assert len(tiles) >= 2 * walks, name
    for name, body in kernel_bodies("gemm_skinny.hip", tmp_path, "gemm_i8_raw_weight_kernel").items():      # the same walk, beside other GEMMs
        assert re.search(r"\.amdhsa_private_segment_fixed_size 0\b", body), name
        blocks = [re.findall(r"^\s*" + VMEM, b, flags=re.M) for b in re.split(r"^\.LBB\S+:|^\s*s_cbranch\w+|^\s*s_branch", body, flags=re.M)]
        assert sum(b == ["global_store_dwordx4"] * 8 for b in blocks) == 1 and len(re.findall(r"s_waitcnt vmcnt\(8\) lgkmcnt\(0\)", body)) >= 1, name


def test_attention_kernels_wait_for_what_they_issue(tmp_path):
    """Every step of the attention's backward waits with vmcnt(n) for its own tile while the next one's n loads may be in flight: it has
    to issue exactly n loads, all of them to LDS, and nothing else by the wait's barrier.  The kernels keep out of scratch memory in their loops
    (dK and dV on four waves have one register too many, a store before and a load between them)."""
    for name, body in kernel_bodies("attention.hip", tmp_path, "attention_d").items():
        steps = re.findall(r"s_waitcnt vmcnt\((\d+)\) lgkmcnt\(0\)(.*?)(?=^\.LBB|^\s*s_c?branch|\Z)", body, flags=re.S | re.M)
        assert len(steps) == 2, name            # with and without the mask
        for n, step in steps:
            assert re.match(r"[^\n]*\n(?:\s*;[^\n]*\n|\s*\n)*\s*s_barrier\b", step), (name, step[:200])
            issued = re.findall(r"^\s*" + VMEM + r"([^\n]*)", step, flags=re.M)
            assert len(issued) == int(n) and all(rest.rstrip().endswith("lds") for _, rest in issued), (name, n, issued)
        ahead = body[:body.index("s_barrier")]
        assert len(re.findall(r"^\s*buffer_load_\w+[^\n]* lds\s*$", ahead, flags=re.M)) >= 2 * int(steps[0][0]), name
        scratch = int(re.search(r"\.amdhsa_private_segment_fixed_size (\d+)", body).group(1))
        assert scratch <= (8 if "dkdv_kernelILi128ELi4E" in name else 0), (name, scratch)
        inside = [loop for loop in loops(body) if "mfma" in loop]
        assert len(inside) >= 2 and not any("scratch_" in loop for loop in inside), name
