"""The one table that says which kernel multiplies how many rows by which matrix
(``ops.choose_product``): the shapes of the three Llama sizes land where they were measured to
be fastest, and a kernel whose operands do not fit is never chosen."""

from __future__ import annotations

import pytest
import torch

from kvcore_amd.ops.library import choose_product


def test_row_counts_and_sizes_choose_the_kernel():
    qkv_8b, down_8b, head, down_70b, o_1b = (6144, 4096), (4096, 14336), (128256, 4096), (8192, 28672), (2048, 2048)
    for N, K in (qkv_8b, down_8b, head, down_70b, o_1b):
        for M in (1, 2, 8):
            assert choose_product(M, N, K) == "few rows"
        for M in (65, 512, 2048):
            assert choose_product(M, N, K) == "vendor"
    assert choose_product(12, *head) == "few rows" and choose_product(13, *head) == "vendor"
    assert choose_product(16, *head) == "vendor"
    assert choose_product(17, *head) == "shared rows" and choose_product(64, *head) == "shared rows"
    assert choose_product(16, *qkv_8b) == "few rows" and choose_product(17, *qkv_8b) == "vendor"
    assert choose_product(9, *down_8b) == "vendor" and choose_product(9, *down_70b) == "vendor"
    assert choose_product(32, *o_1b) == "few rows" and choose_product(33, *o_1b) == "vendor"


def test_a_kernel_that_cannot_take_the_operands_is_not_chosen():
    assert choose_product(4, 4096, 4096, few_rows_ok=False) == "vendor"
    assert choose_product(40, 128256, 4096, shared_rows_ok=False) == "vendor"
    assert choose_product(40, 128256, 4096, few_rows_ok=False) == "shared rows"


@pytest.mark.parametrize("limit", [1, 3, 6, 8, 11, 16, 20, 64, 100, 200, 1024])
def test_decode_graph_sizes(limit):
    """The batch sizes at which steps of single tokens are captured: rising, ending at the
    engine's limit, every size from 8 to 16 (a padded row costs the few-row products what a
    live one does), and never more than twice the live requests beyond one."""
    from kvcore_amd.engine.runner import _decode_buckets

    sizes = _decode_buckets(limit)
    assert sizes == sorted(set(sizes)) and sizes[0] == 1 and sizes[-1] == limit
    assert all(b in sizes for b in range(8, min(limit, 16) + 1))
    for live in range(1, limit + 1):
        padded = next(b for b in sizes if b >= live)
        assert padded <= limit and padded < 2 * live + (live == 1)
        if live > 16:
            assert padded - live < 32


@pytest.mark.parametrize("experts,H,I,rows", [
    (32, 2048, 2048, {1: 16, 4: 16, 16: 64, 40: 64, 64: 128, 128: 64, 192: 128, 512: 128}),
    (8, 512, 512, {3: 16, 16: 16, 48: 16, 96: 64, 192: 64, 512: 64}),
    (8, 2048, 512, {4: 16, 24: 16, 96: 64, 384: 64}),
    (4, 1024, 2048, {3: 16, 32: 16, 96: 64, 256: 64}),
    (4, 256, 320, {4: 16, 48: 16, 256: 64}),
    (128, 1024, 384, {3: 16, 6: 16, 16: 64, 64: 128, 128: 64}),
    (64, 4096, 1408, {2: 16, 8: 64, 32: 64, 96: 128}),
    (16, 512, 2048, {4: 16, 8: 16, 32: 16, 48: 64, 192: 64})])  # 32 rows: 40 us in tiles of 16, 44 of 64
def test_rows_a_tile_of_the_experts_products_holds(experts, H, I, rows):
    """Experts of small matrices keep tiles of 16 until their rows fill larger ones, and none gets tiles of 128 whose
    blocks would leave the chip idle: within a few percent of the fastest measured of the three."""
    from kvcore_amd.ops import library as ops

    x = torch.empty(1, H, dtype=torch.bfloat16)
    for each, tile in rows.items():
        assert ops.moe_tile_rows(each * experts, experts, x, (H, I)) == tile, each
    assert ops.moe_tile_rows(512 * experts, experts, x.float(), (H, I)) == 16
    assert ops.moe_tile_rows(512 * experts, experts, x, (H, I + 8)) == 16
    assert ops.moe_max_tiles(0, experts, 64) == 0 and ops.moe_tile_rows(0, experts, x, (H, I)) == 16


def test_rows_a_tile_of_few_rows_and_without_a_gate():
    """No step of as many pairs as experts or fewer leaves tiles of 16, whose estimate and that of larger tiles lie close
    there; without a gate a product has half the columns of weights a block, and larger tiles pay from fewer rows on."""
    from kvcore_amd.ops import library as ops

    x = torch.empty(1, 8, dtype=torch.bfloat16)
    for E, H, I in ((128, 2048, 768), (64, 2048, 1408), (64, 4096, 1408), (32, 2048, 2048), (8, 4096, 4096), (4, 256, 320)):
        for gated in (True, False):
            assert {ops.moe_tile_rows(p, E, x, (H, I), gated) for p in range(1, E + 1)} == {16}, (E, H, I, gated)
    for (E, H, I), rows in {(32, 2048, 2048): {1: 16, 4: 64, 6: 64, 16: 64}, (128, 2048, 768): {2: 16, 6: 64, 8: 64},
                            (64, 4096, 1408): {2: 16, 8: 64}, (16, 2048, 2048): {8: 16, 12: 16, 24: 64}}.items():
        for each, tile in rows.items():
            assert ops.moe_tile_rows(each * E, E, x, (H, I), False) == tile, (E, H, I, each)


def test_tiles_of_384_rows_need_rows_and_blocks_for_every_unit():
    from kvcore_amd.ops import library as ops

    x = torch.empty(1, 8, dtype=torch.bfloat16)
    for (E, H, I), rows in {(32, 2048, 2048): {64: 0, 103: 0, 104: 384, 256: 384, 512: 384},
                            # one block a unit: rows enough for uneven experts not to be waited for, and a long K
                            (16, 2048, 2048): {130: 0, 229: 0, 230: 384, 500: 384}, (64, 1024, 512): {130: 0, 256: 0, 500: 384},
                            (128, 1024, 384): {130: 0, 256: 0, 500: 384}, (64, 1024, 1024): {256: 0, 500: 384},
                            (64, 2048, 1024): {103: 0, 104: 384}, (16, 1024, 1024): {256: 0, 400: 0, 500: 0},
                            (8, 2048, 1024): {256: 0, 500: 0}, (32, 2048, 2016): {256: 0}}.items():
        for each, tile in rows.items():
            assert ops.moe_wide_tile_rows(each * E, E, x, (H, I)) == tile, (E, H, I, each)
    assert ops.moe_wide_tile_rows(256 * 32, 32, x.float(), (2048, 2048)) == 0
    assert ops.moe_wide_tile_rows(0, 32, x, (2048, 2048)) == 0


def test_tiles_of_384_rows_for_experts_in_one_tile_need_blocks_for_every_unit():
    from kvcore_amd.ops import library as ops

    x = torch.empty(1, 8, dtype=torch.bfloat16)
    for (E, H, I, gated), rows in {(32, 2048, 2048, True): {47: 0, 48: 384, 103: 384, 104: 0}, (64, 2048, 1024, True): {47: 0, 48: 384},
                                   (32, 2048, 2048, False): {100: 0}, (64, 2048, 2048, False): {47: 0, 48: 384},
                                   (31, 2048, 2048, True): {100: 0}, (64, 1024, 1024, True): {100: 0},
                                   (32, 2048, 2016, True): {100: 0}}.items():
        for each, tile in rows.items():
            assert ops.moe_one_tile_rows(each * E, E, x, (H, I), gated) == tile, (E, H, I, gated, each)
    assert ops.moe_one_tile_rows(100 * 32, 32, x.float(), (2048, 2048)) == 0
    assert ops.moe_one_tile_rows(0, 32, x, (2048, 2048)) == 0


@pytest.mark.parametrize("E,top,H,I,wanted", [
    (32, 4, 2048, 2048, {1: 16, 32: 16, 64: 16, 72: 16, 96: 0, 128: 0, 180: 0, 300: 64, 500: 0, 800: 0, 831: 0, 1962: 0}),
    (24, 4, 3072, 3072, {1: 16, 64: 16, 96: 64, 128: 64, 300: 384, 800: 384}),
    (16, 2, 2048, 8192, {1: 16, 32: 16, 40: 0, 48: 0, 96: 0}),
    (16, 2, 4096, 4096, {1: 16, 48: 16, 64: 0, 96: 0, 128: 0}),
    (64, 4, 2048, 2048, {1: 16, 64: 16, 128: 16, 160: 0}),
    (64, 4, 4096, 2048, {1: 16, 96: 16, 128: 0}),
    (256, 8, 2048, 512, {1: 16, 128: 16, 129: 0})])
def test_when_an_expert_of_every_token_joins_the_others(E, top, H, I, wanted):
    """In tiles of 16 up to some hundred tokens, fewer where its own tiles would read large matrices again and again; in larger tiles where
    no unit gets one block more; never where it does.  Asked as a step on one stream asks."""
    from kvcore_amd.ops import library as ops

    x = torch.empty(1, 8, dtype=torch.bfloat16)
    for T, want in wanted.items():
        sizes = (T * top, E, x, (H, I))
        alone = ops.moe_wide_tile_rows(*sizes) or ops.moe_one_tile_rows(*sizes) or ops.moe_tile_rows(*sizes)
        assert ops.moe_shared_tile_rows(T * top, E, (H, I), True, T, alone) == want, T


def test_which_matrix_of_an_expert_of_every_token_fits_the_others():
    """Of their type, size and order of storage, contiguous and 16-byte aligned: what is not stays with products of its own."""
    from kvcore_amd.ops import library as ops

    w = torch.zeros(4 * 32, 64, dtype=torch.bfloat16)
    shared = torch.zeros(32, 64, dtype=torch.bfloat16)
    assert ops.moe_shared_fits(w, shared, 4)
    assert not ops.moe_shared_fits(w, shared.float(), 4) and not ops.moe_shared_fits(w.float(), shared, 4)
    assert not ops.moe_shared_fits(w, shared[:16], 4) and not ops.moe_shared_fits(w, shared, 5)
    assert not ops.moe_shared_fits(w, torch.zeros(64, 32, dtype=torch.bfloat16).t(), 4)
    assert not ops.moe_shared_fits(w, torch.zeros(32, 128, dtype=torch.bfloat16)[:, :64], 4)
    assert not ops.moe_shared_fits(w, torch.zeros(32 * 64 + 1, dtype=torch.bfloat16)[1:].view(32, 64), 4)
    packed = shared.clone()
    packed.kvc_packed = shared
    assert not ops.moe_shared_fits(w, packed, 4)


def test_tiles_of_16_for_an_expert_of_every_token():
    from kvcore_amd.ops import library as ops

    assert ops.moe_shared_tile_rows(0, 32, (2048, 2048), True, 0, 16) == 0
    assert ops.moe_shared_tile_rows(129 * 2, 64, (2048, 2048), True, 129, 16) == 0
    # two tiles of any matrix cost less than products of its own, eight tiles of 100 MB do not
    assert ops.moe_shared_tile_rows(32, 128, (4096, 4096), True, 32, 16) == 16
    assert ops.moe_shared_tile_rows(128, 128, (4096, 4096), True, 128, 16) == 0


@pytest.mark.parametrize("E,top,H,I,wanted", [
    (32, 4, 2048, 2048, {1: 16, 64: 16, 96: 64, 180: 64, 500: 128, 831: 128, 1000: 384, 2048: 384}),
    (128, 8, 2048, 1024, {130: 64, 160: 64, 640: 128, 2048: 384}),
    (16, 2, 4096, 4096, {48: 16, 64: 64, 511: 128, 800: 0, 1024: 0, 1500: 0}),
    (256, 8, 2048, 512, {129: 16, 150: 16, 180: 64}),
    (512, 1, 4096, 4096, {32: 16, 40: 0, 129: 0, 200: 0})])
def test_when_an_expert_of_every_token_joins_beside_another_branch(E, top, H, I, wanted):
    """More often than on one stream, but not in tiles of 16 that read its matrices again and again, nor large matrices over many tokens."""
    from types import SimpleNamespace

    from kvcore_amd.ops import library as ops
    from kvcore_amd.parts.moe import RoutedExperts

    part = RoutedExperts(hidden_size=H, experts=E, top=top, expert_size=I, limit=None, shared_size=I)
    x = torch.empty(1, 8, dtype=torch.bfloat16)
    for T, want in wanted.items():
        ctx = SimpleNamespace(num_tokens=T, scratch={}, buffers=SimpleNamespace(token_capacity=4096))
        tile_rows, joined, max_tiles, most_tiles, *_ = part._plan(x, ctx, True, True)
        assert (tile_rows if joined else 0) == want, T
        assert max_tiles == ops.moe_max_tiles(T * top, E, tile_rows, T if joined else 0) <= most_tiles
        alone = part._plan(x, ctx, False, True)
        assert not alone[1] and alone[3] == ops.moe_max_tiles(4096 * top, E, 16, 0)
        assert part._plan(x, ctx, True, True) is ctx.scratch[("routed_experts", E, H, I, top, True, True, True)]


def _mixers():
    from kvcore_amd.parts.linear_attention import GatedLinearAttention, MaxGatedMatrixMemory
    from kvcore_amd.parts.recurrent import StateSpaceMixer

    return {
        "space": StateSpaceMixer(hidden_size=64, heads=64, head_dim=64, state_size=128, groups=8, conv=4, eps=1e-5,
                                 norm_groups=8),
        "narrow": StateSpaceMixer(hidden_size=64, heads=80, head_dim=32, state_size=64, groups=1, conv=4, eps=1e-5,
                                  norm_groups=1),
        "channel": GatedLinearAttention(hidden_size=64, heads=16, dim=64, vdim=128, tau=8.0, decay_rank=8, eps=1e-5),
        "wide": GatedLinearAttention(hidden_size=64, heads=16, dim=128, vdim=128, tau=8.0, decay_rank=8, eps=1e-5),
        "memory": MaxGatedMatrixMemory(hidden_size=64, heads=16, dim=64, vdim=128, gate_cap=15.0, eps=1e-5)}


@pytest.mark.parametrize("kind,lengths,cut", [
    ("space", [199], 0), ("space", [256], 160), ("space", [2048], 160),                 # one request
    ("space", [192] * 3, 0), ("space", [256] * 3, 160), ("space", [160] * 4, 160),      # until each unit has a block
    ("space", [256] * 8, 160), ("space", [512] * 12, 0), ("space", [256] * 16, 160), ("space", [256] * 32, 0),
    ("space", [100, 320], 0), ("space", [100, 384], 160), ("space", [1, 208], 0),       # the scan of the rest follows
    ("space", [1] * 8 + [192], 160), ("space", [1] * 60 + [160] * 2, 160), ("space", [1] * 64, 0),
    # heads of fewer columns than a tile of the scan: chunks cost as much a head, the scan less
    ("narrow", [160], 0), ("narrow", [256], 160), ("narrow", [200] * 4, 0), ("narrow", [160] * 8, 0), ("narrow", [256] * 8, 0),
    ("narrow", [2048] * 2, 160), ("narrow", [1] * 8 + [160], 0),
    ("channel", [191], 0), ("channel", [192], 160), ("channel", [160] * 4, 0), ("channel", [160] * 8, 160),
    ("channel", [100, 256], 0), ("channel", [100, 300], 160), ("channel", [100] * 8 + [180], 0),
    ("channel", [100] * 8 + [256], 160), ("wide", [152], 0), ("wide", [160], 160),
    ("memory", [151], 0), ("memory", [152], 128), ("memory", [128] * 4, 0), ("memory", [128] * 6, 128),
    ("memory", [1] * 30 + [128], 128), ("memory", [127] * 30, 0)])
def test_which_requests_are_cut_into_chunks(kind, lengths, cut):
    """By the tokens of the requests, by how far they are ahead of those that stay with the scan, and by how full of
    scans the chip is: the side that was measured to be the faster."""
    assert _mixers()[kind].chunk_start(lengths) == cut


def test_a_scan_s_blocks_leave_units_to_another_stream():
    """Up to half as many blocks as units: one a unit; up to as many: two; they never ask for more than a unit has."""
    from kvcore_amd.ops import library as ops

    unit = 160 * 1024
    for blocks, each in {1: 1, 128: 1, 129: 2, 256: 2}.items():
        assert unit // ops.load().kvc_linear_state_scan_lds(blocks) == each, blocks
    assert ops.load().kvc_linear_state_scan_lds(257) == 0 and ops.load().kvc_linear_state_scan_lds(1 << 40) == 0
