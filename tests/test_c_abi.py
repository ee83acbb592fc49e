"""The C ABI library loads without a GPU, exports every function include/alpha_moe_hip.h declares, and its host-only
entry points (argument validation, workspace sizing, status strings) behave as documented."""
import ctypes
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "alpha_moe_hip.h")
LIB = os.path.join(ROOT, "alpha-moe_amd", "alpha_moe", "libalpha_moe_hip.so")


@pytest.fixture(scope="module")
def lib():
    if not os.path.exists(LIB):
        pytest.fail(f"{LIB} is not built: run `python alpha-moe_amd/build.py`")
    L = ctypes.CDLL(LIB)
    L.alpha_moe_validate.restype = ctypes.c_int
    L.alpha_moe_validate.argtypes = [ctypes.c_int] * 10
    L.alpha_moe_workspace_bytes.restype = ctypes.c_size_t
    L.alpha_moe_workspace_bytes.argtypes = [ctypes.c_int] * 7
    L.alpha_moe_status_string.restype = ctypes.c_char_p
    L.alpha_moe_status_string.argtypes = [ctypes.c_int]
    L.alpha_moe_version.restype = ctypes.c_char_p
    L.alpha_moe_fused_moe_w8a8_up_down.restype = ctypes.c_int
    L.alpha_moe_fused_moe_w8a8_up_down.argtypes = (
        [ctypes.c_void_p] * 11 + [ctypes.c_int] * 10 + [ctypes.c_float, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_void_p])
    return L


def declared_functions():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(alpha_moe_\w+)\s*\(", text)))


def test_every_declared_symbol_is_exported(lib):
    names = declared_functions()
    assert "alpha_moe_fused_moe_w8a8_up_down" in names and len(names) >= 5
    for name in names:
        assert getattr(lib, name) is not None, name


def test_status_codes_match_header(lib):
    text = open(HEADER).read()
    codes = dict((k, int(v)) for k, v in re.findall(r"(ALPHA_MOE_\w+)\s*=\s*(\d+)", text))
    assert codes["ALPHA_MOE_OK"] == 0 and len(set(codes.values())) == len(codes)
    for name, code in codes.items():
        msg = lib.alpha_moe_status_string(code).decode()
        assert msg and msg != "unknown status", name
    assert lib.alpha_moe_status_string(999).decode() == "unknown status"
    assert re.fullmatch(r"\d+\.\d+", lib.alpha_moe_version().decode())


def test_validate_accepts_the_reference_knob_space_and_rejects_the_rest(lib):
    ok = dict(top_k=9, M=64, K=7168, N=512, E=257, sorted_num=4431, block_m=16, block_n=64, warp_n=4, stages=3)

    def v(**kw):
        a = dict(ok, **kw)
        return lib.alpha_moe_validate(a["top_k"], a["M"], a["K"], a["N"], a["E"], a["sorted_num"], a["block_m"],
                                      a["block_n"], a["warp_n"], a["stages"])
    # csrc/torch_interface.cpp:62-64 of the reference: block_m 8..128 step 8, (64,4)|(32,8), stages 1..5
    for bm in range(8, 129, 8):
        for bn, wn in ((64, 4), (32, 8)):
            for st in range(1, 6):
                assert v(block_m=bm, block_n=bn, warp_n=wn, stages=st) == 0
    assert v(block_m=12) == 3 and v(block_m=0) == 3 and v(block_m=136) == 3
    assert v(block_n=64, warp_n=8) == 4 and v(block_n=128, warp_n=2) == 4
    assert v(stages=0) == 5 and v(stages=6) == 5
    assert v(K=7168 + 64) == 2 and v(N=384) == 2 and v(M=0) == 2 and v(top_k=0) == 2
    assert v(K=7168 + 128) == 0                       # K % 256 == 128 is supported (the reference drops columns there)


def test_null_pointers_and_small_workspace_are_refused_without_touching_a_device(lib):
    args = [None] * 11 + [9, 64, 7168, 512, 257, 4431, 16, 64, 4, 3, 2.5, None, 0, None]
    assert lib.alpha_moe_fused_moe_w8a8_up_down(*args) == 1
    fake = [ctypes.c_void_p(4096)] * 11
    assert lib.alpha_moe_fused_moe_w8a8_up_down(*fake, 9, 64, 7168, 512, 257, 4431, 16, 64, 4, 3, 2.5, None, 0, None) == 7
    assert lib.alpha_moe_fused_moe_w8a8_up_down(*fake, 9, 64, 7168, 512, 257, 4431, 16, 64, 4, 3, 2.5,
                                                ctypes.c_void_p(4096), 1024, None) == 7
    assert lib.alpha_moe_fused_moe_w8a8_up_down(*fake, 9, 64, 7168, 512, 257, 4431, 12, 64, 4, 3, 2.5,
                                                ctypes.c_void_p(4096), 1 << 40, None) == 3
    # the store variant runs the same checks
    lib.alpha_moe_fused_moe_w8a8_up_down_store.restype = ctypes.c_int
    lib.alpha_moe_fused_moe_w8a8_up_down_store.argtypes = lib.alpha_moe_fused_moe_w8a8_up_down.argtypes
    assert lib.alpha_moe_fused_moe_w8a8_up_down_store(*args) == 1
    assert lib.alpha_moe_fused_moe_w8a8_up_down_store(*fake, 9, 64, 7168, 512, 257, 4431, 16, 64, 4, 3, 2.5, None, 0,
                                                      None) == 7
    assert lib.alpha_moe_fused_moe_w8a8_up_down_store(*fake, 9, 64, 7168, 512, 257, 4431, 12, 64, 4, 3, 2.5,
                                                      ctypes.c_void_p(4096), 1 << 40, None) == 3


def test_workspace_check_refuses_a_null_workspace(lib):
    lib.alpha_moe_workspace_check.restype = ctypes.c_int
    lib.alpha_moe_workspace_check.argtypes = [ctypes.c_void_p, ctypes.c_void_p]
    assert lib.alpha_moe_workspace_check(None, None) == 1


def test_zeroed_prefix_is_small_and_inside_every_workspace(lib):
    lib.alpha_moe_workspace_zero_bytes.restype = ctypes.c_size_t
    lib.alpha_moe_workspace_zero_bytes.argtypes = []
    z = lib.alpha_moe_workspace_zero_bytes()
    assert z > 0 and z % 256 == 0 and z <= 4 << 20
    assert z <= lib.alpha_moe_workspace_bytes(2, 1, 128, 256, 1, 16, 16)


def test_workspace_bytes_is_monotone_and_covers_both_kernel_families(lib):
    small = lib.alpha_moe_workspace_bytes(9, 1, 7168, 512, 257, 9 + 257 * 15, 16)
    big = lib.alpha_moe_workspace_bytes(9, 64, 7168, 512, 257, 576 + 257 * 15, 16)
    assert 0 < small < big < (1 << 31)
    direct = lib.alpha_moe_workspace_bytes(9, 64, 7168, 512, 257, 576 + 257 * 127, 128)
    assert direct >= 64 * 7168 * 4
    assert lib.alpha_moe_workspace_bytes(9, 0, 7168, 512, 257, 100, 16) == 0


def test_prep_entry_points_refuse_bad_arguments_without_touching_a_device(lib):
    lib.alpha_moe_per_token_group_quant_fp8.restype = ctypes.c_int
    lib.alpha_moe_per_token_group_quant_fp8.argtypes = (
        [ctypes.c_void_p, ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int, ctypes.c_int, ctypes.c_void_p])
    lib.alpha_moe_align_workspace_bytes.restype = ctypes.c_size_t
    lib.alpha_moe_align_workspace_bytes.argtypes = [ctypes.c_int] * 2
    lib.alpha_moe_moe_align_block_size.restype = ctypes.c_int
    lib.alpha_moe_moe_align_block_size.argtypes = (
        [ctypes.c_void_p] + [ctypes.c_int] * 3 + [ctypes.c_void_p, ctypes.c_int, ctypes.c_void_p, ctypes.c_int,
                                                  ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_void_p])
    assert lib.alpha_moe_per_token_group_quant_fp8(None, 0, None, None, 4, 128, None) == 1      # null pointer
    assert lib.alpha_moe_per_token_group_quant_fp8(8, 0, 8, 8, 4, 130, None) == 2               # K % 128
    assert lib.alpha_moe_align_workspace_bytes(0, 8) == 0
    assert lib.alpha_moe_align_workspace_bytes(1024, 8) == 8 * 4
    assert lib.alpha_moe_align_workspace_bytes(1025, 8) == 2 * 8 * 4
    assert lib.alpha_moe_moe_align_block_size(None, 32, 8, 16, None, 0, None, 0, None, None, 0, None) == 1
    # sorted_num must be numel + E * (block - 1), n_blocks its ceiling quotient
    assert lib.alpha_moe_moe_align_block_size(8, 32, 8, 16, 8, 100, 8, 7, 8, None, 0, None) == 2
    assert lib.alpha_moe_moe_align_block_size(8, 32, 5000, 16, 8, 32 + 5000 * 15, 8, 4690, 8, None, 0, None) == 2
    # more than 4096 slots need the scratch buffer
    assert lib.alpha_moe_moe_align_block_size(8, 5000, 8, 16, 8, 5120, 8, 320, 8, None, 0, None) == 7


def test_layer_call_pays_by_token_groups_times_blocks_and_by_weights(lib):
    """groups of four tokens times K blocks of a wavefront (1, 2, 4 or 7): both sides of every border; at 3 x 7 the weights of the
    experts there can be decide; a call that is not taken does not pay"""
    pays, supported = lib.alpha_moe_layer_call_pays, lib.alpha_moe_layer_call_supported
    pays.restype = supported.restype = ctypes.c_int
    pays.argtypes = supported.argtypes = [ctypes.c_int] * 9
    knobs = (16, 32, 8, 4)
    for K, few, many in ((128, 16, 16), (1024, 16, 16), (1152, 16, 16), (2048, 16, 16), (2176, 16, 16), (4096, 16, 16),
                         (4224, 8, 12), (5120, 8, 12), (7168, 8, 12)):
        for M in range(1, 17):
            assert supported(1, M, K, 256, 8, *knobs) == 1
            assert pays(1, M, K, 256, 8, *knobs) == (M <= few), (M, K)
            if K >= 2496:
                assert pays(9, M, K, 512, 257, *knobs) == (M <= many), (M, K)
    # at most rows, at most experts; 80 MiB of both weights: 15.2 experts of K = 7168, I = 256
    assert [pays(1, 10, 7168, 2 * I, 64, *knobs) for I in (256, 384, 512)] == [0, 0, 1]
    assert [pays(8, 10, 7168, 512, E, *knobs) for E in (15, 16)] == [0, 1]
    assert pays(4, 17, 4096, 512, 8, *knobs) == 0 and pays(4, 8, 4096, 512, 8, 64, 32, 8, 4) == 0
    for M, K in ((0, 128), (-4, 128), (4, 0), (4, -128), (4, 7296), (4, 130)):
        assert pays(1, M, K, 256, 8, *knobs) == 0


def test_static_scratch_holds_every_batch_up_to_the_documented_sizes(lib):
    """With the shipped tables the entry point without a workspace takes every batch up to these sizes, also where a table
    keeps the streaming kernel and its fp32 rows (Qwen3-Next shard, 752 .. 768 tokens: 65.4 MiB)."""
    from alpha_moe_python.utils import get_best_config
    limit = int(re.search(r"ALPHA_MOE_STATIC_SCRATCH_BYTES \(\(size_t\)(\d+) << 20\)", open(HEADER).read()).group(1)) << 20
    for E, N, K, top_k, upto in ((257, 512, 7168, 9, 250), (512, 512, 2048, 10, 1355), (128, 1536, 2048, 8, 1565)):
        table = os.path.join(ROOT, "alpha-moe_amd", "configs", f"moe_jit_{E}_{N}_{K}.json")
        for M in range(1, upto + 2):
            bm = get_best_config(table, M)["block_m"]
            need = lib.alpha_moe_workspace_bytes(top_k, M, K, N, E, M * top_k + E * (bm - 1), bm)
            assert (need <= limit) == (M <= upto), (E, M, need)


def test_group_kernel_slab_fits_its_scale_table(lib):
    """Every (K, slices, row block, stages, slab override) the group kernel takes: the scales of the widest slab of output columns are
    at most what the variant's LDS table holds.  (A slab has at least four column groups, so beyond 256 slices - 512 at
    K = 128 - the smallest variant's table would be overrun.)"""
    lib.alpha_moe_group_plan.restype = ctypes.c_int
    lib.alpha_moe_group_plan.argtypes = [ctypes.c_int] * 8 + [ctypes.POINTER(ctypes.c_int)]
    lib.alpha_moe_set_tunable.argtypes = [ctypes.c_char_p, ctypes.c_int, ctypes.c_int]
    plan = (ctypes.c_int * 4)()
    seen = set()
    try:
        for gps in (None, 1, 8, 13, 64, 1 << 30):
            assert lib.alpha_moe_set_tunable(b"ALPHA_MOE_TILE_GPS", gps or 0, gps is not None) == 0
            for kb in [*range(1, 18), 31, 33, 56, 63, 64, 100, 128]:
                most = 1024 // kb
                for n_ib in sorted({*range(1, min(most, 12) + 1), *range(13, most + 1, 37), 255, 256, 257, 300, 341, 342, 511, 512, 513, most}):
                    for block_m in (40, 64, 72, 96, 104, 128):
                        for stages in range(1, 6):
                            rc = lib.alpha_moe_group_plan(1, 50, 128 * kb, 256 * n_ib, 1, 50 + block_m - 1, block_m, stages, plan)
                            assert rc == (0 if n_ib <= most else 2), (kb, n_ib, rc)
                            if rc:
                                continue
                            nt, per, slabs, table = plan
                            groups = 2 * kb
                            assert 16 * nt >= block_m and per % 4 == 0 and per > 0 and slabs == -(-groups // per)
                            scales = max((min((c + 1) * per, groups) - c * per + 1) // 2 * n_ib for c in range(slabs))
                            assert scales <= table, (kb, n_ib, block_m, stages, gps, tuple(plan), scales)
                            seen.add((nt, block_m <= 64))
    finally:
        lib.alpha_moe_set_tunable(b"ALPHA_MOE_TILE_GPS", 0, 0)
    assert seen == {(4, True), (6, True), (6, False), (8, False)}


def test_small_row_blocks_beyond_the_streaming_kernel_take_the_group_kernel(lib):
    """Row blocks of at most 32 rows whose fp32 result rows are more than 1 GiB, or with more than 64 experts to a token, are not the
    streaming kernel's: the group kernel has them (and their scratch holds its bf16 rows) up to eight slices of the intermediate.
    One row less, and the call and its scratch are the streaming kernel's."""
    lib.alpha_moe_group_plan.restype = ctypes.c_int
    lib.alpha_moe_group_plan.argtypes = [ctypes.c_int] * 8 + [ctypes.POINTER(ctypes.c_int)]
    plan = (ctypes.c_int * 4)()

    def grouped(top_k, M, K, N, E, bm):
        return lib.alpha_moe_group_plan(top_k, M, K, N, E, M * top_k + E * (bm - 1), bm, 2, plan) == 0

    def need(top_k, M, K, N, E, bm):
        return lib.alpha_moe_workspace_bytes(top_k, M, K, N, E, M * top_k + E * (bm - 1), bm)
    for bm in (8, 16, 24, 32):
        assert not grouped(9, 4161, 7168, 512, 257, bm) and grouped(9, 4162, 7168, 512, 257, bm)
        assert need(9, 4161, 7168, 512, 257, bm) > 4161 * 9 * 7168 * 4 > need(9, 4162, 7168, 512, 257, bm) > 4162 * 9 * 7168 * 2
        assert not grouped(64, 40, 256, 256, 80, bm) and grouped(65, 40, 256, 256, 80, bm)
        assert grouped(9, 5000, 7168, 256 * 8, 16, bm) and not grouped(9, 5000, 7168, 256 * 9, 16, bm)
        assert not grouped(9, 5000, 128 * 128, 256 * 5, 16, bm) and grouped(9, 5000, 128 * 128, 256 * 4, 16, bm)
    assert grouped(9, 64, 7168, 512, 257, 40)


def test_no_kernel_loads_in_inline_assembly():
    """The compiler takes the output register of inline assembly as written when the instruction is issued: it may copy or reuse it
    while a load is still on its way.  Loads are the compiler's own."""
    csrc = os.path.join(ROOT, "alpha-moe_amd", "csrc")
    load = re.compile(r'asm\b[^;]*?"[^"]*\b(ds_read|ds_load|global_load|buffer_load|flat_load|scratch_load|s_load|s_buffer_load)', re.S)
    for name in sorted(os.listdir(csrc)):
        text = open(os.path.join(csrc, name)).read()
        assert not load.search(text), (name, load.search(text).group(0))


def test_kernel_choice_by_the_names_of_kernels_that_are_gone():
    """ALPHA_MOE_PATH=tile and =wide chose kernels whose successor is the group kernel: like =group they keep the small kernels out of the
    way, and their tunables are taken without effect."""
    import subprocess
    import sys
    code = ("import ctypes, sys; L = ctypes.CDLL(sys.argv[1]); "
            "print(L.alpha_moe_layer_call_supported(2, 4, 2048, 512, 8, 16, 32, 8, 4), "
            "[L.alpha_moe_set_tunable(n, 1, 1) for n in (b'ALPHA_MOE_TILE_LAG', b'ALPHA_MOE_TILE_GRID', b'ALPHA_MOE_WIDE_PP', b'ALPHA_MOE_X')])")
    for path, layer in (("", 1), ("group", 0), ("tile", 0), ("wide", 0), ("small", 1)):
        out = subprocess.run([sys.executable, "-c", code, LIB], env=dict(os.environ, ALPHA_MOE_PATH=path), capture_output=True, text=True)
        assert out.stdout.strip() == f"{layer} [0, 0, 0, 2]", (path, out.stdout, out.stderr)
