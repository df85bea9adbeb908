"""The built kernel library loads on a CPU host (dlopen resolves every symbol: a launcher
declared in kernels.h but left undefined fails here, not on the GPU box) and registers
the ops the Python layer calls."""
import os
import re
import subprocess

import pytest
import torch

from hipserve import _build
from hipserve.ops import _SEQ_LIBS, library_path, load_kernel_library


@pytest.mark.skipif(not os.path.exists(library_path()), reason="hipserve/_C.so not built")
def test_library_loads_and_registers_ops():
    from hipserve.ops import load_library

    load_library()
    for op in ("decode_gemm_partial", "gguf_gemm_parts", "fp8_untile", "gguf_dequant_tiled", "paged_decode",
               "splitk_add_rmsnorm", "prefill_gemm_packed", "fp8_decode_gemm"):
        assert hasattr(torch.ops.hipserve, op), op


@pytest.mark.skipif(not os.path.exists(_build.HIPCC), reason="no hipcc")
@pytest.mark.parametrize("hist", ["", ", p"])
def test_the_alignment_asks_for_its_scratch(hist, tmp_path):
    """From 4097 pairs on many workgroups write counts there: a call without it does not compile."""
    src = tmp_path / "k.cpp"
    src.write_text('#include "hipserve/kernels.h"\n'
                   f"void f(int* p, hipStream_t s) {{ hipserve::launch_moe_align(p, 5000, 8, 32, p, 6000, p, 200, p, p, nullptr, s{hist}); }}\n")
    r = subprocess.run(["g++", "-std=c++17", "-fsyntax-only", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(_build.ROCM, "include"),
                        "-I", os.path.join(_build.CSRC, "include"), src], capture_output=True, text=True)
    assert (r.returncode == 0) == bool(hist), r.stderr


@pytest.mark.skipif(not os.path.exists(_build.HIPCC), reason="no hipcc")
@pytest.mark.parametrize("name", ["window_attention_dma", "latent_attention_dma", "skinny_linear", "expert_ffn", "mingru", "latent_attention_prompt"])
def test_copies_into_lds_keep_their_wait_states(name, tmp_path):
    """The copies of lds_copy.h are inline assembly, which the compiler's hazard pass does not look into: between the scalar write of
    m0 (the place in LDS) and the copy lies another instruction, and the vector unit has not written the base address just before."""
    asm = tmp_path / "k.s"
    subprocess.run([_build.HIPCC, *_build.HIP_FLAGS, "-I", os.path.join(_build.CSRC, "include"), "-S", "--cuda-device-only",
                    os.path.join(_build.CSRC, "kernels", "seq", name + ".hip"), "-o", asm], check=True, capture_output=True)
    lines = [ln.strip() for ln in asm.read_text().splitlines()]
    code = [ln for ln in lines if ln and ln[0] not in ".;/" and not ln.endswith(":")]
    copies = [i for i, ln in enumerate(code) if ln.startswith("global_load_lds")]
    assert copies
    for i in copies:
        assert not re.match(r"s_\w+ m0\b", code[i - 1]), code[i - 1:i + 1]
        base = re.search(r", s\[(\d+):(\d+)\]", code[i])
        for ln in code[i - 5:i] if base else ():
            wrote = re.match(r"v_(?:readfirstlane|readlane|cmp)\w* s\[?(\d+)(?::(\d+))?", ln)
            assert not wrote or int(wrote[2] or wrote[1]) < int(base[1]) or int(wrote[1]) > int(base[2]), (ln, code[i])


@pytest.mark.skipif(not os.path.exists(_build.HIPCC), reason="no hipcc")
def test_sequences_of_a_product_come_through_the_scalar_unit(tmp_path):
    """minGRU's product asks for its rows' sequences behind its copies into LDS: the vector unit's loads would be waited for with these. Its own are the biases, the
    states and what the experts beside it need."""
    asm = tmp_path / "k.s"
    subprocess.run([_build.HIPCC, *_build.HIP_FLAGS, "-I", os.path.join(_build.CSRC, "include"), "-S", "--cuda-device-only",
                    os.path.join(_build.CSRC, "kernels", "seq", "mingru.hip"), "-o", asm], check=True, capture_output=True)
    kernels = re.findall(r"\n(_ZN8hipserve\S*mingru_product\S*):\s.*?\n(.*?)s_endpgm", asm.read_text(), re.S)
    assert len(kernels) >= 12
    for name, code in kernels:
        assert len(re.findall(r"global_load_(?!lds)", code)) <= 8 and len(re.findall(r"s_load", code)) >= 24, name


@pytest.mark.skipif(not os.path.exists(_build.HIPCC), reason="no hipcc")
def test_a_carried_state_is_asked_for_at_once(tmp_path):
    """The chunked gated rule's scan loads its 16 numbers per lane with no wait between them."""
    asm = tmp_path / "k.s"
    subprocess.run([_build.HIPCC, *_build.HIP_FLAGS, "-I", os.path.join(_build.CSRC, "include"), "-S", "--cuda-device-only",
                    os.path.join(_build.CSRC, "kernels", "seq", "delta_chunk.hip"), "-o", asm], check=True, capture_output=True)
    code = re.split(r"^_ZN\S*delta_chunk_scan_kernelILi2ELi4ELi2E\S*:", asm.read_text(), maxsplit=1, flags=re.M)[1].split("s_endpgm")[0].split("v_mfma")[0]
    between = code.split("global_load_dword ")   # the operands are loaded sixteen bytes at a time, P alone by single numbers
    assert max(len(run) for run in "".join("w" if "s_waitcnt" in x else "l" for x in between[1:-1]).split("w")) >= 15


@pytest.mark.skipif(not os.path.exists(_build.HIPCC), reason="no hipcc")
def test_decode_window_attention_knows_its_keys_are_global(tmp_path):
    """No flat loads, which wait for each other and for LDS."""
    asm = tmp_path / "k.s"
    subprocess.run([_build.HIPCC, *_build.HIP_FLAGS, "-I", os.path.join(_build.CSRC, "include"), "-S", "--cuda-device-only",
                    os.path.join(_build.CSRC, "kernels", "seq", "window_attention_decode.hip"), "-o", asm], check=True, capture_output=True)
    text = asm.read_text()
    assert "global_load_dwordx4" in text and "flat_load" not in text


@pytest.mark.skipif(not os.path.exists(_build.HIPCC), reason="no hipcc")
def test_short_prompts_of_mingru_leave_room_for_twice_the_waves(tmp_path):
    """Sequences of one block of rows: no registers for a next block's, and no loads of it."""
    asm = tmp_path / "k.s"
    subprocess.run([_build.HIPCC, *_build.HIP_FLAGS, "-I", os.path.join(_build.CSRC, "include"), "-S", "--cuda-device-only",
                    os.path.join(_build.CSRC, "kernels", "seq", "mingru.hip"), "-o", asm], check=True, capture_output=True)
    text = asm.read_text()
    for t, load in (("f", "buffer_load_dword "), ("t", "buffer_load_ushort ")):
        code = re.split(rf"^_ZN\S*mingru_scan_kernelI{t}Lb0E\S*:", text, maxsplit=1, flags=re.M)[1].split("s_endpgm")[0]
        regs = re.search(rf"\.name:\s+_ZN\S*mingru_scan_kernelI{t}Lb0E.*?\.vgpr_count:\s+(\d+)", text, flags=re.S)
        assert int(regs[1]) <= 64 and code.count(load) == 3 * 16


@pytest.mark.skipif(not os.path.exists(_build.HIPCC), reason="no hipcc")
def test_scans_of_wide_heads_leave_room_for_three_waves(tmp_path):
    """Token by token: no second set of a token's vectors at 8 and 16 channels per lane."""
    asm = tmp_path / "k.s"
    subprocess.run([_build.HIPCC, *_build.HIP_FLAGS, "-I", os.path.join(_build.CSRC, "include"), "-S", "--cuda-device-only",
                    os.path.join(_build.CSRC, "kernels", "seq", "delta_scan.hip"), "-o", asm], check=True, capture_output=True)
    regs = {}
    for entry in asm.read_text().split(".name: ")[1:]:
        scan = re.match(r"\s+_ZN\S*?\d(gated_delta|delta_rule)_scan_kernelI([ft]?)Li(\d+)(\S*?)EEE?v", entry)
        if scan: regs[scan.groups()] = int(re.search(r"\.vgpr_count:\s+(\d+)", entry)[1])
    assert len(regs) == 20 and all(n <= (168 if int(ds) == 16 else 128) for (_, _, ds, _), n in regs.items()), regs


@pytest.mark.skipif(not os.path.exists(_build.HIPCC), reason="no hipcc")
def test_a_gate_is_asked_for_beside_the_weights_of_the_runs(tmp_path):
    """The merge of latent decode runs waits for the weights and the gate while the runs' rows are on their way."""
    asm = tmp_path / "k.s"
    subprocess.run([_build.HIPCC, *_build.HIP_FLAGS, "-I", os.path.join(_build.CSRC, "include"), "-S", "--cuda-device-only",
                    os.path.join(_build.CSRC, "kernels", "seq", "latent_attention_mfma.hip"), "-o", asm], check=True, capture_output=True)
    for rows in (4, 8, 12, 16):
        code = re.split(rf"^_ZN\S*latent_attention_reduce_kernelILi{rows}E\S*:", asm.read_text(), maxsplit=1, flags=re.M)[1].split("s_endpgm")[0]
        before, after = code.split("s_waitcnt vmcnt", 1)
        assert after.startswith(f"({rows})") and before.count("global_load_ushort") == 1 and before.count("global_load_dwordx4") == rows, rows


@pytest.mark.skipif(not os.path.exists(_SEQ_LIBS["seq"]), reason="hipserve/_C_seq.so not built")
def test_half_tiles_of_32_bits_copy_no_further_ahead_than_whole_ones():
    """The kernels that the library brings: groups of 8 rows, pieces ahead. 3 groups have one and two, by the weights' size."""
    with open(_SEQ_LIBS["seq"], "rb") as f:
        names = set(re.findall(rb"skinny_linear_kernelILi(\d)ELi1ELi(\d)ELb0EfLb1ELi0ELb1E", f.read()))
    assert {(int(g), int(d)) for g, d in names} == {(1, 2), (2, 2), (3, 1), (3, 2), (4, 1), (6, 1), (8, 1)}


@pytest.mark.skipif(not os.path.exists(_SEQ_LIBS["seq"]), reason="hipserve/_C_seq.so not built")
@pytest.mark.parametrize("cols,k,tiles_and_pairs", [   # measured: whether the kernel for few rows per tile is at least 10 % faster, or slower
    (2048, 1024, {(1, 1): True, (17, 32): True, (143, 4080): True}), (512, 512, {(1, 1): True, (64, 64): True, (36, 1020): True}),
    (2048, 704, {(4, 4): True, (66, 128): True, (572, 16320): True}), (1024, 640, {(16, 16): True, (132, 256): True}), (4096, 1024, {(64, 64): True, (1144, 32640): True}),
    (512, 1024, {(33, 64): True, (286, 8160): True}), (2048, 768, {(16, 16): True, (125, 1): False, (125, 16): False}), (4096, 640, {(16, 16): True, (63, 4): False}),
    (2048, 512, {(16, 16): True, (249, 16): False, (264, 512): False, (2288, 65280): False}), (1000, 520, {(39, 256): True, (159, 4096): False, (286, 8160): False}),
    (2048, 2048, {(249, 4): False})])
def test_choice_of_the_expert_kernels(cols, k, tiles_and_pairs):
    load_kernel_library("seq")
    for (tiles, pairs), rows in tiles_and_pairs.items():
        assert torch.ops.hipserve_seq.expert_rows_pay(tiles, pairs, cols, k) == rows, (tiles, pairs)


@pytest.mark.skipif(not os.path.exists(_SEQ_LIBS["seq"]), reason="hipserve/_C_seq.so not built")
@pytest.mark.parametrize("cols,per_tile", [(16, 1), (17, 2), (2048, 128)])
def test_choice_of_the_expert_kernels_at_its_edges(cols, per_tile):
    load_kernel_library("seq")
    pay, most = torch.ops.hipserve_seq.expert_rows_pay, 8192 // per_tile
    assert pay(most, 10 * most, cols, 512) and not pay(most + 1, 10 * most, cols, 512) and not pay(most + 1, 10 * most, cols, 639) and pay(most + 1, 10 * most, cols, 640)
    assert pay(most + 5, 5, cols, 4096) and not pay(most + 6, 5, cols, 4096)


@pytest.mark.skipif(not os.path.exists(_SEQ_LIBS["seq"]), reason="hipserve/_C_seq.so not built")
def test_an_update_takes_the_columns_that_its_product_would():
    from hipserve.ops import KernelOps
    load_kernel_library("seq")
    half = torch.ops.hipserve_seq.skinny_half
    for rows in (1, 8, 9, 32):
        for cols in (64, 1024, 1088, 2048, 2112, 4096):
            for k in (512, 520, 1024, 1032, 2048, 2056, 4096, 4104):
                for f32 in (False, True):
                    assert (KernelOps._update_cols(rows, cols, k, f32) == 8) == half(rows, cols, k, f32), (rows, cols, k, f32)


@pytest.mark.skipif(not os.path.exists(_SEQ_LIBS["seq"]), reason="hipserve/_C_seq.so not built")
@pytest.mark.parametrize("k,half", [(1024, False), (1792, False), (1984, False), (2048, True), (2112, False), (2304, False), (2560, False), (4096, False), (6144, False),
                                    (8192, True), (12288, False), (16384, True)])
def test_half_tiles_of_wide_products(k, half):
    """By the distance of the weights' rows, as measured: a class of them, not one, and neither their neighbours nor more rows, 32 bits or fewer workgroups."""
    load_kernel_library("seq")
    wide = torch.ops.hipserve_seq.skinny_wide
    for cols in (5648, 6160, 8192, 32000):
        whole = [3 if k >= 2048 and (cols > 6144 if k % 2048 == 0 else k >= 2560 and cols > 8192) else 0, False]
        for rows in (1, 4):
            assert wide(rows, cols, k, False) == ([2 if k <= 4096 else 3, True] if half else whole), (rows, cols)
            assert wide(rows, cols, k, False, True) == whole   # rows without their norm's factor: squares would be summed for half the columns
        assert wide(5, cols, k, False) == whole and wide(9, cols, k, False) == [0, False]
        assert wide(1, cols, k // 2, True) == [3 if whole[0] and k % 2048 == 0 else 0, False]
    assert wide(1, 5632, k, False) == [0, False]


@pytest.mark.skipif(not os.path.exists(_SEQ_LIBS["seq"]), reason="hipserve/_C_seq.so not built")
@pytest.mark.parametrize("rows,cols,k,faster", [
    (9, 11264, 6144, False), (12, 10752, 6144, False), (10, 11264, 4096, False), (13, 11264, 6144, False), (9, 28672, 3072, False), (11, 27648, 3328, False), (9, 10240, 6144, False),
    (16, 6144, 2048, True), (9, 6144, 2048, True), (9, 8704, 3072, True), (12, 10304, 3584, True), (13, 11264, 3072, True), (16, 28672, 3072, True), (16, 8704, 6144, True),
    (33, 8704, 3328, True), (24, 12288, 4096, True), (48, 13376, 3072, True), (24, 20480, 2048, True), (48, 20480, 2048, False), (16, 8200, 2048, False), (16, 4104, 1024, False)])
def test_columns_of_a_workgroup_by_whole_rounds(rows, cols, k, faster):
    """Sizes at which 24 - 56 columns per workgroup were measured to take at least 3 % less than whole tiles (``faster``), or no less."""
    load_kernel_library("seq")
    assert (torch.ops.hipserve_seq.skinny_cols(rows, cols, k) > 0) == faster


@pytest.mark.skipif(not os.path.exists(_SEQ_LIBS["seq"]), reason="hipserve/_C_seq.so not built")
@pytest.mark.parametrize("rows,cols,k,f32,glu,pays", [
    (1, 2048, 2048, False, False, True), (48, 2048, 2048, False, False, True), (64, 6144, 1024, False, False, True), (16, 32000, 1024, True, False, True),
    (48, 512, 8192, False, False, False), (40, 576, 12288, False, False, False), (64, 32768, 128, False, False, False), (64, 65536, 512, False, False, False),
    (56, 12288, 2048, True, False, False), (64, 12288, 512, True, False, False), (48, 576, 2048, True, False, False),
    (16, 2048, 6144, True, True, False), (16, 4096, 12288, False, True, False), (1, 12288, 2048, False, True, True),
    (40, 25600, 3072, False, False, False), (40, 65536, 2560, False, False, False), (40, 25600, 3584, False, False, False), (48, 32000, 2048, False, False, True),
    (32, 65536, 2048, False, False, True), (24, 50000, 2048, False, False, True), (32, 49152, 4096, False, True, True)])
def test_products_of_a_few_rows_take_the_faster_kernel(rows, cols, k, f32, glu, pays):
    """Sizes at which one of the two was measured to be at least 10 % faster (the weight-streaming kernel where ``pays``), among them few columns
    of many k, many columns of few k, matrix products that are bound by their 32-bit arithmetic and weights whose rows lie a multiple of 4096 bytes apart."""
    from hipserve.ops import KernelOps

    assert KernelOps().skinny_pays(rows, cols, k, glu, f32) == pays


@pytest.mark.skipif(not os.path.exists(_SEQ_LIBS["seq"]), reason="hipserve/_C_seq.so not built")
@pytest.mark.parametrize("rows,width,k,f32,pays", [(1, 4096, 2048, False, True), (48, 4096, 2048, False, True), (17, 6000, 1024, False, True),
                                                   (33, 512, 4096, True, False), (64, 256, 3072, True, False)])
def test_mingru_product_where_it_is_faster(rows, width, k, f32, pays):
    from hipserve.ops import KernelOps

    assert KernelOps().mingru_pays(rows, width, k, f32) == pays
