"""Launch arithmetic checked on the CPU: the grid a launcher asks for must be exactly what its kernel's decode of the
workgroup index assumes.  libsthip.so computes both with the same functions the GPU path uses (no device is touched)."""
import itertools
import time

import pytest

from spiraltorch_amd import hip


def test_row_blocks_of_a_large_lhs_are_never_empty():
    # An A of 2 GiB or more is cut into row blocks of at least 256 rows whose bytes stay below 2^31; where 256 rows
    # do not fit, the answer is 0 and the product keeps the 64-bit-addressed kernels (a block of 0 rows once made the
    # host loop forever: f32 k = 2088961..2097151, bf16 k = 4177921..4194303).
    for elem in (4, 2):
        limit = (1 << 31) // (256 * elem)
        ks = list(range(1, 64)) + [511, 512, 4096, 50257, 1 << 20, limit - 8192, limit - 1, limit, limit + 1,
                                   2 * limit, (1 << 31) // elem, (1 << 31) // elem + 1]
        ks += list(range(limit - 8200, limit + 3, 97))
        for k in ks:
            block = hip.gemm_row_block(k, elem)
            if 256 * k * elem < (1 << 31):
                assert block >= 256 and block % 256 == 0, (k, elem, block)
                assert block * k * elem < (1 << 31)
                assert (block + 256) * k * elem >= (1 << 31)  # the largest such block
            else:
                assert block == 0, (k, elem, block)
    assert hip.gemm_row_block(2090000, 4) == 256  # the shape of the report: 300 x 128 x 2090000
    assert hip.gemm_row_block(0, 4) == 0


CONTEXTS = (1, 2, 3, 7, 8, 12, 16, 64, 128, 256, 257)
SEQUENCES = (1, 63, 64, 65, 127, 128, 129, 255, 256, 257, 300, 511, 512, 1000, 1024, 2048, 2049, 4096)


@pytest.mark.parametrize("causal,biased", [(False, False), (True, False), (False, True), (True, True)])
def test_attention_grid_decodes_to_every_item_once_and_to_nothing_else(causal, biased):
    for contexts, seq, dim in itertools.product(CONTEXTS, SEQUENCES, (32, 64, 128)):
        plan = hip.attention_f32_launch_plan(contexts, seq, dim, causal, biased)
        where = (contexts, seq, dim, causal, biased, plan)
        assert plan["kernel"] in ("general", "fast", "fast_biased", "tiny"), where
        assert plan["consistent"] == 1, where
        assert plan["out_of_range"] == 0 and plan["duplicates"] == 0, where
        assert plan["items"] == plan["items_expected"], where
        if plan["key_splits"] > 1:
            assert plan["keys_per_split"] % 64 == 0 and plan["keys_per_split"] >= 128, where


def test_the_shape_that_once_read_past_its_operands_keeps_the_pairing():
    # 256 contexts of 256 keys, causal: a split would give every tile one chunk, so the launch keeps tile pairs
    plan = hip.attention_f32_launch_plan(256, 256, 64, True, False)
    assert plan["kernel"] == "fast" and plan["key_splits"] == 1 and plan["workgroups"] == 256
    assert plan["out_of_range"] == 0 and plan["items"] == plan["items_expected"] == 512
    # few contexts, long sequence: (tile, chunk) items
    plan = hip.attention_f32_launch_plan(8, 2048, 128, True, False)
    assert plan["key_splits"] > 1 and plan["items"] == plan["items_expected"] == plan["workgroups"]
    # the reference's caller: one context with a bias matrix, keys split over workgroups
    plan = hip.attention_f32_launch_plan(1, 2048, 64, False, True)
    assert plan["kernel"] == "fast_biased" and plan["key_splits"] > 1 and plan["workgroups"] == 16 * plan["key_splits"]


def test_the_attention_plan_knows_the_scale():
    plan = lambda *shape, **options: hip.attention_f32_launch_plan(*shape, **options)
    # 256-row tiles belong to the split kernel alone
    assert plan(128, 2048, 64, True, scale=0.125)["kernel"] == "split" and plan(128, 2048, 64, True, scale=0.125)["workgroups"] == 128 * 4
    assert plan(128, 2048, 64, True, scale=0.6)["kernel"] == "fast" and plan(128, 2048, 64, True, scale=0.6)["workgroups"] == 128 * 8
    assert plan(128, 2048, 62, True)["kernel"] == "general" and plan(128, 2048, 62, True)["workgroups"] == 128 * 16
    # biases: rows the f32 kernel cannot read 16 bytes at a time, larger heads
    assert plan(2, 777, 64, False, True, scale=0.6)["kernel"] == "general" and plan(2, 776, 64, False, True, scale=0.6)["kernel"] == "fast_biased"
    assert plan(2, 777, 64, False, True, scale=-0.5)["kernel"] == "split" and plan(2, 776, 80, False, True, scale=0.6)["kernel"] == "general"
    for seq, dim in itertools.product((33, 500, 700, 768, 769, 776, 800, 832, 833, 900, 2000), (68, 80, 96, 100, 128)):  # one kernel for all lengths
        assert plan(2, seq, dim, False, True, scale=0.1)["kernel"] == "split", (seq, dim)
    assert plan(300, 64, 64, True, scale=0.6)["kernel"] == "tiny" and plan(300, 64, 64, True, scale=0.125)["kernel"] == "tiny"
    for contexts, seq, dim, causal, biased in itertools.product(CONTEXTS, SEQUENCES, (32, 64, 128), (False, True), (False, True)):
        got = plan(contexts, seq, dim, causal, biased, scale=0.9)
        assert got["consistent"] == 1 and got["out_of_range"] == 0 and got["duplicates"] == 0, (contexts, seq, dim, causal, biased, got)
        assert got["items"] == got["items_expected"], (contexts, seq, dim, causal, biased, got)


@pytest.mark.parametrize("causal,biased", [(False, False), (True, False), (False, True), (True, True)])
def test_shared_keys_are_dealt_out_completely(causal, biased):
    # a workgroup 32 queries of a context and one run of keys: at most one for each of the 256 compute units, every one its own item
    cut = set()
    for contexts, seq, dim in itertools.product((1, 2, 3, 7, 8, 31, 32, 64, 128), SEQUENCES + (33, 96, 250, 333, 777), (32, 48, 64)):
        plan = hip.attention_f32_launch_plan(contexts, seq, dim, causal, biased, scale=dim ** -0.5)
        where = (contexts, seq, dim, causal, biased, plan)
        assert plan["consistent"] == 1 and plan["out_of_range"] == 0 and plan["duplicates"] == 0, where
        assert plan["items"] == plan["items_expected"], where
        if plan["kernel"] == "split" and plan["workgroups"] == contexts * -(-seq // 32) * plan["key_splits"]:
            assert plan["workgroups"] <= 256, where
            assert plan["key_splits"] * plan["keys_per_split"] >= seq > (plan["key_splits"] - 1) * plan["keys_per_split"], where
            cut.add(plan["key_splits"])
    assert {1, 4, 8} <= cut, cut


@pytest.mark.parametrize("causal,biased", [(False, False), (True, False), (False, True), (True, True)])
def test_wide_heads_are_dealt_out_completely(causal, biased):
    kernels = set()
    for contexts, seq, dim in itertools.product((1, 2, 7, 8, 31, 64, 128), SEQUENCES + (33, 96, 250, 333, 768, 769), (68, 96, 100, 128)):
        plan = hip.attention_f32_launch_plan(contexts, seq, dim, causal, biased, scale=dim ** -0.5)
        where = (contexts, seq, dim, causal, biased, plan)
        assert plan["out_of_range"] == 0 and plan["duplicates"] == 0 and plan["items"] == plan["items_expected"], where
        assert plan["kernel"] != "split" or plan["consistent"] == 1, where
        kernels.add(plan["kernel"])
    assert "split" in kernels


def test_key_chunks_of_large_heads():
    # chunks of 128 keys, the last one shorter, where every workgroup has a compute unit to itself; otherwise as many keys as
    # two workgroups a unit leave each, 128 and more
    cut = lambda contexts, seq: [hip.attention_f32_launch_plan(contexts, seq, 128)[name] for name in ("key_splits", "keys_per_split")]
    assert cut(1, 300) == [3, 128] and cut(3, 777) == [7, 128] and cut(8, 500) == [4, 128]
    assert cut(3, 1180) == [7, 192] and cut(8, 777) == [5, 192] and cut(8, 2000) == [4, 512]


def test_long_causal_sequences_are_planned_quickly():
    # 508 query tiles: the number of (tile, chunk) items was once counted tile by tile for every chunk size, 1 to 2 ms a call
    times = []
    for _ in range(20):
        start = time.perf_counter()
        hip.attention_f32_launch_plan(1, 65000, 64, True, False)
        times.append(time.perf_counter() - start)
    assert min(times) < 3e-4


def test_bf16_tile_grids_decode_to_every_split_and_tile_once():
    # few tiles under a long k are split over workgroups: every (k-split, tile) the grid decodes to must exist, have
    # k-tiles to walk, and be decoded exactly once — also where the XCD remap reorders the workgroups
    ms = (1, 33, 64, 65, 100, 255, 256, 257, 300, 512, 1000, 1024, 2048, 4096, 16384)
    ns = (128, 256, 384, 512, 1000, 1536, 2048, 4096, 50257)
    ks = (64, 128, 512, 576, 1024, 2048, 4096, 8192, 65536)
    for m, n, k in itertools.product(ms, ns, ks):
        plan = hip.gemm_bf16_tile_plan(m, n, k)
        where = (m, n, k, plan)
        assert plan["consistent"] == 1, where
        assert plan["out_of_range"] == 0 and plan["duplicates"] == 0, where
        assert plan["items"] == plan["workgroups"] == plan["tiles_m"] * plan["tiles_n"] * plan["k_splits"], where
        assert plan["k_splits"] * plan["k_tiles_per_split"] >= k // 64 > (plan["k_splits"] - 1) * plan["k_tiles_per_split"], where
    assert hip.gemm_bf16_tile_plan(100, 4096, 4096)["k_splits"] > 1       # a batch of 100 rows against a large weight
    assert hip.gemm_bf16_tile_plan(4096, 4096, 4096)["k_splits"] == 1     # 256 tiles of 256×256
    with pytest.raises(hip.HipErr):
        hip.gemm_bf16_tile_plan(128, 128, 100)                            # k not a multiple of 64: another kernel family


# Ragged sizes of every tile shape: rows and columns one short of, on and one past the tiles and the 32-row blocks, long and
# short reductions; the last three are products whose tiles once read 27 MB, 2 MB and 126 KB past the split operands.
SPLIT_SIZES = (33, 64, 65, 97, 129, 161, 257, 425, 770, 1000, 1024, 1121, 1399, 1601, 2049, 3841, 4097)
SPLIT_KNOWN = [(1024, 800, 50257), (4096, 800, 4096), (65, 4097, 1001)]


def test_split_products_stay_inside_their_operands():
    tiles = set()
    shapes = list(itertools.product(SPLIT_SIZES, SPLIT_SIZES, (97, 515, 769, 2100, 4099))) + SPLIT_KNOWN
    for (m, n, k), (transposed, packed) in itertools.product(shapes, ((False, False), (True, False), (False, True))):
        plan = hip.gemm_f32_split_plan(m, n, k, transposed, packed)
        where = (m, n, k, transposed, packed, plan)
        if not plan["served"]:
            continue
        tiles.add((plan["tile_rows"], plan["tile_cols"], plan["k_splits"] > 1))
        steps = (k + 31) // 32 * 2
        assert plan["a_bytes"] == (m + 31) // 32 * steps * 3072 and plan["b_bytes"] == (n + 31) // 32 * steps * 3072, where
        assert plan["a_reach"] == plan["a_bytes"] and plan["b_reach"] == plan["b_bytes"], where
        assert plan["a_bytes"] + plan["b_bytes"] < 1 << 31, where
        assert plan["tiles_m"] * plan["tile_rows"] >= m and plan["tiles_n"] * plan["tile_cols"] >= n, where
        assert plan["steps_per_split"] % 2 == 0, where
        assert plan["k_splits"] * plan["steps_per_split"] >= steps > (plan["k_splits"] - 1) * plan["steps_per_split"], where
    for shape in SPLIT_KNOWN:
        assert hip.gemm_f32_split_plan(*shape)["served"], shape
    assert {t[0] for t in tiles} == {64, 96, 128, 160, 256} and {t[2] for t in tiles} == {False, True}, tiles


def test_split_convolutions_stay_inside_their_operands():
    served = 0
    geometries = [((1, 1), (1, 1), (0, 0), (1, 1)), ((3, 3), (1, 1), (1, 1), (1, 1)), ((3, 3), (2, 2), (1, 1), (1, 1)), ((5, 3), (2, 1), (2, 0), (1, 1)),
                  ((3, 3), (1, 1), (2, 2), (2, 2)), ((3, 3), (1, 1), (4, 3), (1, 1)), ((7, 7), (1, 1), (3, 3), (1, 1))]
    for batch, c_in, side, c_out in itertools.product((1, 2, 31, 32), (16, 33, 64, 250, 512), (7, 14, 29, 56), (31, 64, 129, 512)):
        for kernel, stride, padding, dilation in geometries:
            for direction in ("forward", "grad_input"):
                if side + 2 * padding[0] < (kernel[0] - 1) * dilation[0] + 1:
                    continue
                shape = (batch, c_in, side, side + 1, c_out, kernel, stride, padding, dilation)
                plan = hip.conv2d_f32_split_plan(*shape, direction=direction)
                where = (shape, direction, plan)
                if not plan["served"]:
                    continue
                served += 1
                channels, rows = (c_in, c_out) if direction == "forward" else (c_out, c_in)
                steps = ((channels + 15) // 16 * kernel[0] * kernel[1] + 1) // 2 * 2
                assert plan["weight_bytes"] == (rows + 31) // 32 * steps * 3072, where
                assert plan["image_reach"] <= plan["image_bytes"] and plan["weight_reach"] == plan["weight_bytes"], where
                assert plan["image_bytes"] + plan["weight_bytes"] < 1 << 31, where
                assert plan["steps_per_split"] % 2 == 0, where
                assert plan["k_splits"] * plan["steps_per_split"] >= steps > (plan["k_splits"] - 1) * plan["steps_per_split"], where
    assert served > 100
    # a strip kernel's grad_input for an image is the same bits whatever the batch: such layers stay on it
    layer = (32, 64, 56, 56, 128, (3, 3), (1, 1), (1, 1), (1, 1))
    assert hip.conv2d_f32_split_plan(*layer)["served"] == 1
    assert hip.conv2d_planned_kernel(*layer, direction="grad_input") == "strip9"
    assert hip.conv2d_f32_split_plan(*layer, direction="grad_input")["served"] == 0
    assert hip.conv2d_f32_split_plan(2, 8, 9, 9, 4, (3, 3), (1, 1), (1, 1), (1, 1))["served"] == 0


def test_bf16_convolution_grids_decode_to_every_run_and_tile_once():
    tiles, cut = set(), set()
    geometries = [((1, 1), (1, 1), (0, 0), (1, 1)), ((3, 3), (1, 1), (1, 1), (1, 1)), ((3, 3), (2, 2), (1, 1), (1, 1)), ((7, 7), (2, 2), (3, 3), (1, 1))]
    for batch, c_in, side, c_out, geometry in itertools.product((1, 2, 13, 32), (3, 16, 65, 512), (7, 14, 29, 56), (1, 33, 64, 129, 288, 512), geometries):
        plan = hip.conv2d_bf16_launch_plan(batch, c_in, side, side + 1, c_out, *geometry)
        where = (batch, c_in, side, c_out, geometry, plan)
        assert plan["consistent"] == 1 and plan["out_of_range"] == 0 and plan["duplicates"] == 0, where
        assert plan["items"] == plan["workgroups"], where
        k_tiles = -(-(-(-c_in // 8) * geometry[0][0] * geometry[0][1]) // 8)
        assert plan["k_splits"] * plan["k_tiles_per_split"] >= k_tiles > (plan["k_splits"] - 1) * plan["k_tiles_per_split"], where
        tiles.add((plan["tile_channels"], plan["tile_pixels"]))
        cut.add(plan["k_splits"])
    assert tiles == {(64, 64), (128, 64), (64, 128), (128, 128), (256, 128), (128, 256)} and len(cut) > 3, (tiles, cut)
    # a layer whose operands' copies are too large for the kernels' offsets
    assert hip.conv2d_bf16_launch_plan(64, 2048, 128, 128, 64, (1, 1), (1, 1), (0, 0), (1, 1))["workgroups"] == 0
