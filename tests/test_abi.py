"""The C-ABI library loads on a machine without a GPU and exports exactly what include/ksq.h declares."""
import os
import re

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def declared_functions():
    text = open(os.path.join(ROOT, "include", "ksq.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(ksq_[a-z0-9_]+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    from ksanallm_amd import lib as L
    lib = L.load()
    names = declared_functions()
    assert len(names) >= 20
    for n in names:
        assert hasattr(lib, n), n
    assert sorted(L.SIGNATURES) == names
    assert lib.ksq_version() == 1
    assert lib.ksq_last_error_string() is not None


def test_size_queries_and_tile_selection_are_host_only():
    from ksanallm_amd import lib as L
    lib = L.load()
    assert lib.ksq_w4a16_packed_weight_bytes(1, 4096, 4096) == 4096 * 4096 // 2
    assert lib.ksq_w4a16_packed_scales_bytes(1, 4096, 4096, 128, L.F16) == 32 * 4096 * 2
    assert lib.ksq_w4a16_packed_zeros_bytes(1, 4096, 14336, 128) == 32 * 14336
    assert lib.ksq_moe_align_capacity(64, 256, 16) == 64 + 256 * 15
    d = L.select_tile(L.KIND_W4A16, 1, 4096, 4096, L.F16)
    assert d["kernel"] == 0 and d["grid"] >= 256
    # deterministic: same answer every time, no timing involved
    assert d == L.select_tile(L.KIND_W4A16, 1, 4096, 4096, L.F16)
    import pytest
    with pytest.raises(L.KsqError):
        L.select_tile(99, 1, 16, 128, 0)
    # W4A8: packed size, and a workspace that covers every token count up to the maximum it was asked for
    assert lib.ksq_w4a8_packed_weight_bytes(5120, 5120) == 5120 * 5120 // 2
    assert lib.ksq_w4a8_workspace_size(32, 5120, 5120) == 0        # the streaming kernel needs none
    need = lib.ksq_w4a8_workspace_size(4096, 256, 8192)
    assert need > 0
    for m in (33, 64, 100, 128, 129, 700, 4096):
        assert lib.ksq_w4a8_workspace_size(m, 256, 8192) <= need
    assert lib.ksq_w4a8_workspace_size(64, 256, 100) == 0          # k not a multiple of 128: no kernel, no scratch


def test_small_problem_rule_and_its_switch():
    """Above 32 rows the tile kernels, but for small problems; the switch sends those to the tile kernels too, the
    descriptor follows it, and the workspace query covers both settings."""
    from ksanallm_amd import lib as L
    lib = L.load()
    small, large = (128, 4096, 4096), (160, 14336, 4096)  # ceil(m/32) * n * k = 2^26 and 5 * 14336 * 4096 > 2^28
    assert L.select_tile(L.KIND_W4A16, *small, L.BF16)["kernel"] == 0
    assert L.select_tile(L.KIND_W4A16, *large, L.BF16)["kernel"] == 1
    assert L.select_tile(L.KIND_W4A16, 513, 256, 256, L.BF16)["kernel"] == 1      # never beyond 512 rows
    assert L.select_tile(L.KIND_W4A16, 64, 25600, 5120, L.F16)["kernel"] == 0      # 2 * n * k < 2^28
    assert L.select_tile(L.KIND_W4A16, 64, 5120, 25600, L.F16)["kernel"] == 1      # K the long side by 4x: 2^27
    assert L.select_tile(L.KIND_FP8_BLOCKWISE, 64, 4608, 7168, L.BF16)["kernel"] == 0
    assert L.select_tile(L.KIND_FP8_BLOCKWISE, 64, 24576, 1536, L.BF16)["kernel"] == 1  # n > 4 k
    assert L.select_tile(L.KIND_FP8_BLOCKWISE, 96, 7168, 7168, L.BF16)["kernel"] == 1   # 3 * n * k > 5 * 2^24
    assert L.select_tile(L.KIND_FP8_BLOCKWISE, 128, 4096, 4096, L.BF16)["kernel"] == 0
    assert L.select_tile(L.KIND_FP8_BLOCKWISE, 64, 7168, 7168, L.BF16)["kernel"] == 1
    assert L.select_tile(L.KIND_W4A8, 96, 5120, 5120, L.BF16)["kernel"] == 0
    assert L.select_tile(L.KIND_W4A8, 256, 5120, 5120, L.BF16)["kernel"] == 1
    ws_on = lib.ksq_w4a16_workspace_size(128, 4096, 14336, 128, L.BF16)
    assert L.set_small_problem_rule(False) is True
    try:
        assert L.select_tile(L.KIND_W4A16, *small, L.BF16)["kernel"] == 1
        assert L.select_tile(L.KIND_FP8_BLOCKWISE, 128, 4096, 4096, L.BF16)["kernel"] == 1
        assert L.select_tile(L.KIND_W4A8, 96, 5120, 5120, L.BF16)["kernel"] == 1
        d = L.select_tile(L.KIND_W4A16, 128, 4096, 14336, L.BF16)
        assert d["kernel"] == 1 and d["split_k"] > 1
        assert lib.ksq_w4a16_workspace_size(128, 4096, 14336, 128, L.BF16) == ws_on >= d["split_k"] * 128 * 4096 * 4
    finally:
        assert L.set_small_problem_rule(True) is False
    assert L.select_tile(L.KIND_W4A16, *small, L.BF16)["kernel"] == 0


def test_w4a8_64_token_tiles_serve_whole_tiles_and_long_parts():
    """Up to 64 tokens: 64-token tiles while K is whole or its parts have 32 k-blocks, 128-token tiles over shorter parts."""
    from ksanallm_amd import lib as L
    L.set_small_problem_rule(False)
    try:
        for m, n, k, bm, cut in ((64, 28672, 1024, 64, 1), (33, 8192, 1536, 64, 1), (64, 25600, 3072, 64, 1), (64, 25600, 8192, 64, 2),
                                 (48, 25600, 7936, 128, 2), (40, 16224, 3968, 128, 4), (64, 8192, 14336, 128, 8),
                                 (33, 4352, 20480, 128, 15), (65, 28672, 1024, 128, 1)):
            d = L.select_tile(L.KIND_W4A8, m, n, k, L.BF16)
            assert (d["kernel"], d["block_m"], d["split_k"]) == (1, bm, cut), (m, n, k, d)
            need = L.load().ksq_w4a8_workspace_size(m, n, k)
            assert need >= (d["grid"] * bm * 256 * 4 if cut > 1 else 0)
    finally:
        L.set_small_problem_rule(True)


def test_block_fp8_expert_blocks_follow_the_rounds_of_workgroups():
    """The block size from 16 slots per expert on, for both tile kernels.  Below 104 and from 128 on: the rule of unknown sizes.  Between: 256-slot blocks where the experts that
    need a second 128-slot block start another round of 256 workgroups in either GEMM."""
    from ksanallm_amd import lib as L
    lib = L.load()
    for per in (0, 1, 2, 15, 16, 103, 128, 400):
        for E, hidden, inter in ((1, 7168, 2048), (16, 1152, 512), (256, 7168, 2048)):
            numel = per * E + E // 2
            assert lib.ksq_moe_fp8_block_m_sized(numel, E, hidden, inter) == lib.ksq_moe_fp8_block_m(numel, E)
    assert lib.ksq_moe_fp8_block_m_sized(100, 0, 1024, 512) == 16
    for E, hidden, inter, per, bm in ((32, 2048, 1024, 104, 256), (64, 1024, 512, 120, 256), (256, 7168, 2048, 104, 256),
                                      (16, 7168, 2048, 112, 256), (24, 2048, 1024, 120, 128), (24, 2048, 1024, 127, 256),
                                      (32, 1024, 512, 127, 128), (16, 1152, 512, 120, 128), (8, 7168, 2048, 112, 128),
                                      (8, 7168, 2048, 127, 256), (1, 7168, 2048, 120, 128)):
        assert lib.ksq_moe_fp8_block_m_sized(per * E, E, hidden, inter) == bm, (E, hidden, inter, per)


def test_block_fp8_expert_row_blocks():
    """From 4 to 15 slots per expert the row blocks of the streaming tile kernel where 16 experts or more make 128 tiles of 256
    columns in both GEMMs, the decode form's where they do not; otherwise the lines of the tile kernel."""
    from ksanallm_amd import lib as L
    lib = L.load()
    sizes = ((256, 7168, 2048, True), (32, 1024, 512, True), (32, 2048, 384, False), (31, 1024, 512, False), (16, 7168, 2048, True),
             (15, 7168, 2048, False), (8, 7168, 2048, False))
    for per, many, few in ((0, 16, 16), (1, 16, 16), (2, 32, 32), (3, 32, 32), (4, 128, 32), (15, 128, 32), (16, 128, 128),
                           (63, 128, 128), (64, 128, 128), (103, 128, 128), (128, 256, 256), (1000, 256, 256)):
        for E, hidden, inter, enough in sizes:
            assert lib.ksq_moe_fp8_row_block(per * E + E // 2, E, hidden, inter) == (many if enough else few), (per, E, hidden, inter)
    for per in range(16, 140):
        for E, hidden, inter, _ in sizes:
            assert lib.ksq_moe_fp8_row_block(per * E, E, hidden, inter) == lib.ksq_moe_fp8_block_m_sized(per * E, E, hidden, inter)
    assert lib.ksq_moe_fp8_row_block(100, 0, 1024, 512) == 16
    # what the 128-slot launch refuses (activations of 4 GiB, K whose weight scales do not fit the LDS) stays with the decode form
    for per, E, hidden, inter, bm in ((8, 1024, 524160, 128, 128), (8, 1024, 524416, 128, 32), (15, 256, 1048576, 128, 128),
                                      (15, 256, 1048704, 128, 32), (4, 16, 1572864, 2048, 32), (4, 1024, 256, 1048576, 32)):
        assert lib.ksq_moe_fp8_row_block(per * E, E, hidden, inter) == bm, (per, E, hidden, inter)
        if bm == 128:
            assert per * E * max(hidden, inter) <= 0xffffffff


def test_block_fp8_streaming_launch_serves_means_of_up_to_15_sixteenths_of_a_block():
    from ksanallm_amd import lib as L
    served = L.load().ksq_moe_fp8_fused_quant
    for bm in (128, 256):
        for E in (1, 3, 8, 256):
            most = bm // 16 * 15 * E
            assert (served(most, E, 512, 1024, bm), served(most + 1, E, 512, 1024, bm)) == (1, 0), (bm, E)
    # (more of them where the tile kernel's stages and the weight scales of K do not fit the LDS)
    for bm, k in ((128, 212992), (256, 491520)):
        assert [served(bm * 8, 8, 512, kk, bm) for kk in (k, k + 128, 1000064, 2000000)] == [0, 1, 1, 0], bm
    assert [served(100, 8, n, k, bm) for n, k, bm in ((512, 1024, 32), (384, 1024, 128), (512, 1000, 128))] == [0, 0, 0]


def test_block_fp8_streaming_tile_kernel_serves_one_block_of_129_to_240_rows():
    """From 20 column tiles and six k-blocks per workgroup on."""
    from ksanallm_amd import lib as L

    def kernel(m, n, k):
        return L.select_tile(L.KIND_FP8_BLOCKWISE, m, n, k, L.BF16)["kernel"]
    stream, tile, decode = L.KERNEL_STREAM_TILE, L.KERNEL_MFMA_TILE, L.KERNEL_SPLITK_WAVE
    assert [kernel(m, 18432, 7168) for m in (32, 33, 128, 129, 240, 241, 256, 400)] == [decode, tile, tile, stream, stream, tile, tile, tile]
    assert [kernel(200, n, 20480) for n in (4864, 4880, 5120)] == [tile, stream, stream]        # 19 and 20 column tiles
    assert [kernel(200, 8704, k) for k in (640, 768)] == [tile, stream]                          # whole tiles of five and six k-blocks
    assert [kernel(200, n, k) for n, k in ((66064, 2048), (80656, 3072))] == [tile, stream]      # whole tiles beside parts of four, of eight
    assert [kernel(200, n, 4096) for n in (4096, 8192, 8208)] == [tile, tile, stream]            # 128-row tiles up to 32 column tiles


def test_descriptor_of_the_grouped_streaming_launch():
    """KSQ_KIND_MOE_W4A16 describes the grouped streaming launch, which never cuts K over workgroups: its K slices are its
    wavefronts, four of them while fewer than 32 slots are routed, and then, through LDS, as many as that form has."""
    from ksanallm_amd import lib as L
    for m, n, k in ((1, 4096, 14336), (20, 4096, 14336), (31, 1024, 16384), (16, 14336, 4096)):
        d = L.select_tile(L.KIND_MOE_W4A16, m, n, k, L.BF16)
        assert (d["kernel"], d["waves"], d["split_k"], d["x_chunk"]) == (0, 4, 4, 0)
        assert d["block_m"] == (16 if m <= 16 else 32) and d["grid"] == n // d["block_n"]
    for m, n, k, waves, chunk in ((32, 14336, 4096, 8, 8), (32, 57344, 8192, 4, 4), (64, 4096, 14336, 4, 0)):
        d = L.select_tile(L.KIND_MOE_W4A16, m, n, k, L.BF16)
        assert (d["block_m"], d["waves"], d["split_k"], d["x_chunk"]) == (32, waves, waves, chunk)
        assert d["grid"] == n // d["block_n"] * (m // 32)


def test_decode_with_k_cut_over_workgroups_takes_x_through_lds_where_that_pays():
    """x goes through LDS (one workgroup of eight wavefronts per CU) where every workgroup is resident at once, but for parts
    of 9..11 k-tiles below 32 rows; with more workgroups than CUs only from 32 rows and 16 k-tiles per part on."""
    from ksanallm_amd import lib as L
    for m, n, k, waves, chunk in ((20, 2048, 17024, 8, 8), (20, 2112, 17024, 4, 0), (31, 4160, 9600, 4, 0), (32, 4160, 9600, 8, 8),
                                  (90, 1600, 5760, 4, 0), (90, 2624, 8192, 8, 8), (160, 2432, 9600, 8, 8), (24, 1024, 4096, 8, 8), (24, 1024, 4608, 4, 0),
                                  (24, 1024, 5632, 4, 0), (24, 1024, 6144, 8, 8), (32, 1024, 4608, 8, 8)):
        d = L.select_tile(L.KIND_W4A16, m, n, k, L.BF16)
        assert d["kernel"] == 0 and d["split_k"] > d["waves"]
        assert (d["waves"], d["x_chunk"]) == (waves, chunk), (m, n, k)


def test_align_scratch_covers_every_smaller_call():
    """A caller sizes the alignment's scratch for its largest call: never less than what a smaller one needs, whose chunks of whole
    256 ids may be more (98304 ids are 128 chunks, 98305 are 97), a row of E counts each."""
    from ksanallm_amd import lib as L
    lib = L.load()
    for E in (1, 256):
        sizes = [lib.ksq_moe_align_scratch_bytes(n, E) for n in (0, 1, 256, 257, 32768, 32769, 65536, 65537, 98304, 98305, 131072, 131073)]
        assert sizes == sorted(sizes) and sizes[0] > 0
        assert lib.ksq_moe_align_scratch_bytes(98305, E) >= 128 * E * 4


def test_grouped_int4_launches_of_the_streaming_kernel():
    """32-slot blocks from 192 workgroups of 256 columns on, but for more than one and up to five quarters of a round of the 256 CUs
    (as even routing is expected to fill the blocks) where the decode kernel has eight strips to a workgroup and k is 4096 or more."""
    from ksanallm_amd import lib as L
    kernel = L.load().ksq_moe_w4a16_kernel
    stream, tile, decode = L.KERNEL_STREAM_TILE, L.KERNEL_MFMA_TILE, L.KERNEL_SPLITK_WAVE
    assert [kernel(4096, 256, 4096, 7168, bm) for bm in (16, 32, 128, 256)] == [decode, stream, tile, tile]
    assert [kernel(numel, 32, 1024, 3328, 32) for numel in (991, 992)] == [decode, stream]
    assert [kernel(128, 8, n, 4096, 32) for n in (8192, 8320, 8448, 10240, 10368)] == [stream, decode, decode, decode, stream]   # 32 .. 41 tiles
    assert [kernel(128, 8, n, 4096, 32) for n in (8256, 8512)] == [stream, stream]                   # n not a multiple of 128
    assert [kernel(128, 8, 9216, k, 32) for k in (3968, 4096, 7168)] == [stream, decode, decode]
    assert [kernel(per * 16, 16, 4096, 4096, 32) for per in (16, 20, 28, 32)] == [stream, stream, decode, stream]   # 16, 16, 19 and 23 expected blocks
    assert kernel(256, 1, 8192, 4096, 32) == stream and kernel(256, 1, 9216, 4096, 32) == decode     # one expert: exactly 8 blocks
    assert kernel(4096, 256, 1 << 20, 1 << 16, 32) == stream and kernel(4096, 256, 1 << 20, (1 << 16) + 128, 32) == decode


def test_int4_expert_row_blocks():
    """One value on each side of every line of the sizes-unknown rule, and where the sizes move them: up to 8 experts with 1024
    workgroups of 256 columns in the first GEMM have the line of 16 experts."""
    from ksanallm_amd import lib as L
    lib = L.load()
    for E, small, large in ((1, 16, 129), (8, 16, 129), (9, 16, 72), (16, 16, 72), (17, 16, 56), (31, 16, 56), (32, 10, 56), (33, 10, 44),
                            (127, 10, 44), (128, 7, 44), (256, 7, 44)):
        blocks = [lib.ksq_moe_block_m(per * E + E // 2, E) for per in (small - 1, small, large - 1, large)]
        assert blocks == [16, 32, 32, 256], (E, blocks)
        for per in (small - 1, small, large - 1, large):
            assert lib.ksq_moe_w4a16_row_block(per * E, E, 2048, 1408) == lib.ksq_moe_block_m(per * E, E)
    assert lib.ksq_moe_block_m(100, 0) == 16 and lib.ksq_moe_w4a16_row_block(100, 0, 2048, 1408) == 16
    for E, hidden, inter, line in ((8, 6144, 16384, 72), (8, 4096, 28672, 72), (8, 6144, 16256, 129), (4, 8192, 32768, 72), (4, 8192, 28672, 129)):
        rule = [lib.ksq_moe_w4a16_row_block(per * E, E, hidden, inter) for per in (15, 16, line - 1, line)]
        assert rule == [16, 32, 32, 256], (E, hidden, inter, rule)
    # hidden a multiple of 4096 and inter from 4096 on: 32-row blocks from 11 rows on
    for E, hidden, inter, line in ((128, 4096, 4096, 11), (32, 8192, 14336, 11), (128, 4096, 3968, 7), (128, 4224, 4096, 7), (32, 4096, 2048, 10),
                                   (8, 4096, 14336, 16)):
        rule = [lib.ksq_moe_w4a16_row_block(per * E + E // 2, E, hidden, inter) for per in (line - 1, line)]
        assert rule == [16, 32], (E, hidden, inter, rule)


def test_int4_expert_row_blocks_of_more_activations_than_32_row_blocks_take():
    """The launches of 16- and 32-row blocks refuse activations of 1 GiB.  From 40 rows per expert on the rule gives such a call the tile
    kernel's blocks, whatever its other lines say; below it never did."""
    from ksanallm_amd import lib as L
    rule = L.load().ksq_moe_w4a16_row_block
    numel = 43 * 1024
    most = 0x3fffffff // 2 // numel
    assert L.load().ksq_moe_block_m(numel, 1024) == 32
    for hidden, inter in ((1024, most), (most, 1024), (1024, most + 1), (most + 1, 1024)):
        fits = max(hidden, inter) * numel * 2 < 1 << 30
        assert rule(numel, 1024, hidden, inter) == (32 if fits else 256), (hidden, inter)
    assert rule(39 * 1024, 1024, 1024, 2 * most) == 32 and rule(40 * 1024, 1024, 1024, 2 * most) == 256


def test_w4a8_streaming_tile_kernel_serves_one_row_block():
    """33 to 128 tokens: up to 64 in workgroups of 128 columns that are one round of the 256 CUs, or in 256 columns with parts of 20
    k-blocks and more; above, parts of any length up to 112 tokens and of 10 up to 128, but for short parts of a K of 16384 and its
    multiples from 97 tokens on."""
    from ksanallm_amd import lib as L
    lib = L.load()
    stream, tile, decode = L.KERNEL_STREAM_TILE, L.KERNEL_MFMA_TILE, L.KERNEL_SPLITK_WAVE

    def form(m, n, k):
        d = L.select_tile(L.KIND_W4A8, m, n, k, L.BF16)
        return lib.ksq_w4a8_kernel(m, n, k), d["block_n"], d["split_k"]
    assert [form(m, 25600, 5120)[0] for m in (32, 33, 64, 65, 128, 129)] == [decode, stream, stream, stream, stream, tile]
    assert [form(m, 25600, 5120)[1:] for m in (64, 65)] == [(128, 1), (256, 2)]
    assert form(64, 32768, 1024) == (stream, 128, 1) and form(64, 32784, 1024) == (tile, 256, 1)      # 256 and 258 workgroups
    assert form(64, 40960, 2432) == (tile, 256, 1) and form(64, 40960, 2560) == (stream, 256, 1)      # 19 and 20 k-blocks
    assert form(64, 14336, 8192) == (tile, 256, 4) and form(64, 20480, 8192) == (stream, 256, 3)      # parts of 16 and of 22
    assert [lib.ksq_w4a8_kernel(m, 4096, 16384) for m in (96, 97, 112)] == [stream, tile, tile]       # parts of 8
    assert [lib.ksq_w4a8_kernel(m, 8192, 16384) for m in (96, 97, 128)] == [stream, tile, tile]       # of 16
    assert [lib.ksq_w4a8_kernel(128, n, k) for n, k in ((12288, 16384), (8192, 16256))] == [stream, stream]


def test_w4a8_workspace_of_a_form_that_writes_none():
    """Up to 64 tokens in workgroups of 128 columns over all of K, also where the plan cuts it: no partial tiles and no workspace; a
    buffer sized for more tokens still covers every smaller call."""
    from ksanallm_amd import lib as L
    size = L.load().ksq_w4a8_workspace_size
    for n, k in ((25600, 5120), (24336, 4736)):
        assert L.select_tile(L.KIND_W4A8, 64, n, k, L.BF16)["block_n"] == 128 and L.select_tile(L.KIND_W4A8, 65, n, k, L.BF16)["split_k"] == 2
        assert [size(m, n, k) for m in (1, 32, 33, 64)] == [0, 0, 0, 0], (n, k)
        assert size(128, n, k) >= size(65, n, k) >= -(-n // 256) * 2 * 128 * 256 * 4
    for m, n, k in ((33, 20480, 8192), (64, 14336, 8192)):          # K cut at 64 tokens and below
        assert size(m, n, k) >= L.select_tile(L.KIND_W4A8, m, n, k, L.BF16)["grid"] * 128 * 256 * 4


def test_block_fp8_decode_strips():
    """Up to 32 rows: one strip of 16 columns per workgroup up to 256 strips; above, two with more than 8 rows or a K longer than n, else by
    rows in one round of the CUs and by how full the last round is in several.  Above 32 rows in row blocks: four where every other CU
    still gets a workgroup.  Always as many as divide n."""
    from ksanallm_amd import lib as L

    def strips(m, n, k):
        d = L.select_tile(L.KIND_FP8_BLOCKWISE, m, n, k, L.BF16)
        assert d["kernel"] == L.KERNEL_SPLITK_WAVE and d["grid"] == n // d["block_n"] * -(-m // 32)
        return d["block_n"] // 16
    assert [strips(m, 4096, 14336) for m in (1, 8, 16, 32)] == [1, 1, 1, 1]
    assert [strips(m, 4128, 14336) for m in (1, 8, 16, 32)] == [2, 2, 2, 2] and strips(16, 4112, 4096) == 1      # (257 strips)
    assert [strips(m, 8192, 4096) for m in (1, 4, 5, 8, 9, 32)] == [1, 1, 2, 2, 2, 2]                            # one round of pairs
    assert [strips(8, n, 4096) for n in (12800, 13088, 13120, 16384)] == [1, 1, 2, 2]                            # 409 and 410 of 512
    assert [strips(8, n, 1536) for n in (18432, 22112, 22144, 24576)] == [1, 1, 2, 2]                            # 691 and 692 of 768
    assert [strips(33, n, 4096) for n in (2048, 4096)] == [2, 4]
