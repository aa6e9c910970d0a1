"""How the weight-streaming product deals rows of the weight and steps of K to waves: for every size the plan must
name a kernel that exists and sizes that the kernel accepts (no GPU needed)."""
import random

import pytest
import torch

from atoma_infer_amd.kernels import gemm_bf16

# (rows of 16 per wave, waves that split K) that csrc/kernels/gemm_bf16.hip instantiates, per entry point
PLAIN = {(1, 1), (2, 1), (4, 1), (1, 4), (2, 4), (4, 4), (1, 8), (2, 8)}
SWIGLU = {(2, 1), (4, 1), (2, 4), (4, 4), (2, 8)}
ROPE = {(1, 1), (2, 1), (1, 4), (2, 4), (1, 8), (2, 8)}


def shapes():
    rnd = random.Random(7)
    fixed = [(n, k) for n in (16, 48, 2048, 3072, 5120, 6144, 16384, 28672, 128256) for k in (32, 96, 2048, 3072, 8192, 14336)]
    return fixed + [(rnd.randrange(1, 40000), 32 * rnd.randrange(1, 500)) for _ in range(300)]


@pytest.mark.parametrize("m", [1, 8, 16, 17, 33, 48, 49, 64])
def test_plans_name_kernels_that_exist(m):
    for n, k in shapes():
        for allow in (False, True):
            rt, wk, slices = gemm_bf16._plan(m, n, k, allow)
            assert (rt, wk) in PLAIN, (m, n, k, allow)
            assert slices >= 1 and (allow or slices == 1)
            assert k % (32 * wk * slices) == 0, (m, n, k, rt, wk, slices)
            if slices > 1:
                assert k // (wk * slices) >= 128          # a wave's share of K stays worth its launch
                groups = -(-(-(-n // 16)) // ((4 if wk == 1 else 1) * rt))
                assert groups * slices <= 1024
        # the fused epilogues adjust the plan to their own kernels
        rt, wk, _ = gemm_bf16._plan(m, n, k, False)
        r2 = rt if rt % 2 == 0 else 2
        if (r2, wk) in SWIGLU:
            assert (r2, wk) != (2, 8) or m <= 48          # eight waves of four row tiles do not exist
        assert (min(rt, 2), wk) in ROPE
        assert (min(rt, 2), wk) != (2, 8) or m <= 48


def test_few_rows_keep_their_two_planes():
    # sizes of Llama-3.2-1B: o and down projections of a decode step
    assert gemm_bf16._plan(8, 2048, 2048, True) == (1, 4, 2)
    assert gemm_bf16._plan(8, 2048, 8192, True) == (1, 4, 2)
    # more rows: about 256 workgroups
    rt, wk, slices = gemm_bf16._plan(64, 2048, 8192, True)
    assert -(-128 // rt) * slices == 256


def test_library_thresholds():
    import torch
    wins = gemm_bf16._library_wins
    assert not wins(64, 3072, 2048, torch.bfloat16) and wins(65, 3072, 2048, torch.bfloat16)
    assert wins(33, 16384, 2048, torch.bfloat16) and not wins(32, 16384, 2048, torch.bfloat16)
    assert wins(17, 128256, 2048, torch.float32) == gemm_bf16._MM_OUT_DTYPE and not wins(16, 128256, 2048, torch.float32)
    # the head: eight waves splitting K up to 8 rows, then 64 rows of W a wave and four waves splitting K
    assert [gemm_bf16._plan(m, 128256, 2048, False) for m in (8, 9, 16)] == [(2, 8, 1), (4, 4, 1), (4, 4, 1)]


# (tiles, waves splitting K, steps a batch of loads, half tiles) of the residual product in csrc/kernels/gemm_bf16.hip
RESID = {(1, 4, 4, 0), (1, 8, 4, 0), (1, 8, 2, 0), (1, 8, 8, 0), (1, 1, 4, 0),
         (1, 4, 4, 1), (1, 4, 8, 1), (1, 8, 4, 1), (1, 8, 8, 1), (1, 8, 2, 1), (1, 1, 4, 1)}


def test_residual_products_name_kernels_that_exist():
    for n, k in shapes():
        for m in (1, 8, 16):
            rt, wk, depth, half = gemm_bf16.resid_plan(m, n, k)
            assert (rt, wk, depth, half) in RESID, (m, n, k)
            assert k % (32 * wk) == 0
            if half:            # a step of half tiles covers 64 values of K, and N is small
                assert k % (64 * wk) == 0 and n <= 2048
    # Llama 1B: 8 rows of the weight a wave; 3B and 8B: whole tiles, and as many steps a batch as K allows
    assert gemm_bf16.resid_plan(8, 2048, 2048) == (1, 8, 4, 1) and gemm_bf16.resid_plan(8, 2048, 8192) == (1, 8, 4, 1)
    assert gemm_bf16.resid_plan(8, 3072, 8192) == (1, 8, 8, 0) and gemm_bf16.resid_plan(8, 4096, 14336) == (1, 8, 8, 0)
    assert gemm_bf16.resid_plan(8, 3072, 3072) == (1, 8, 4, 0)


# -- the tile kernel for many rows ---------------------------------------------------------------------------------------
T_F32, T_RESID, T_SILU, T_ROPE = gemm_bf16.TILE_F32, gemm_bf16.TILE_RESID, gemm_bf16.TILE_SILU, gemm_bf16.TILE_ROPE


def test_tile_plans_fit_the_kernel():
    rnd = random.Random(5)
    for _ in range(3000):
        m, n, k = int(65 * 1.07 ** rnd.uniform(0, 80)), 32 * rnd.randrange(1, 2000), 64 * rnd.randrange(1, 300)
        for kind in (T_F32, T_RESID, T_SILU, T_ROPE):
            planes = kind in (T_F32, T_RESID)
            tile, slices, us = gemm_bf16.tile_plan(m, n, k, kind, planes)
            assert us > 0 and k % (64 * slices) == 0
            assert 1 <= slices <= (gemm_bf16.TILE_MAX_SLICES if planes else 1)
            # (what the kernel's `pick` takes for the result)
            assert tile in {T_F32: (0, 1, 2, 3, 4, 5, 6, 7), T_RESID: (0, 1, 2, 3, 4, 5), T_SILU: (0, 1, 2, 3, 6), T_ROPE: (1, 2, 3, 4, 5, 8)}[kind]
            assert tile in {T_F32: gemm_bf16.TILES_SUMS, T_RESID: gemm_bf16.TILES_SUMS, T_SILU: gemm_bf16.TILES_SILU, T_ROPE: gemm_bf16.TILES_ROPE}[kind]


# measured on MI355X with the weights not in any cache, each with what follows it: (kind, rows, N, K, library us, tiles us)
LIBRARY_QUICKER = [(T_RESID, 65, 5120, 5120, 35.2, 48.1), (T_RESID, 80, 8192, 8192, 61.5, 81.3), (T_F32, 100, 8192, 8192, 67.6, 81.4),
                   (T_RESID, 640, 8192, 28672, 298.6, 394.1), (T_RESID, 1536, 8192, 8192, 185.2, 257.3),
                   (T_RESID, 3000, 4096, 14336, 291.1, 355.3), (T_RESID, 4096, 3072, 3072, 85.3, 105.3),
                   (T_SILU, 1300, 27648, 5120, 337.9, 382.5), (T_ROPE, 65, 2048, 1536, 13.1, 14.8), (T_SILU, 640, 16384, 3072, 70.5, 77.5),
                   (T_ROPE, 160, 3072, 2048, 15.9, 17.2), (T_RESID, 3333, 3584, 18944, 372.7, 459.4),
                   (T_SILU, 512, 28672, 8192, 187.3, 197.4), (T_SILU, 3072, 16384, 8192, 556.6, 585.8), (T_SILU, 3072, 4096, 5120, 103.0, 107.4),
                   (T_RESID, 2048, 6144, 2048, 76.2, 82.2), (T_RESID, 4096, 6144, 11008, 453.2, 519.4), (T_F32, 640, 8192, 3072, 68.4, 71.8),
                   (T_F32, 4096, 3072, 1792, 68.4, 73.0)]
TILES_QUICKER = [(T_SILU, 2048, 16384, 2048, 127.5, 114.8), (T_SILU, 200, 16384, 2048, 33.9, 24.9), (T_ROPE, 2048, 3072, 2048, 38.1, 32.8),
                 (T_RESID, 128, 4096, 14336, 80.9, 37.8), (T_RESID, 200, 3072, 8192, 42.6, 29.5), (T_F32, 128, 4096, 4096, 30.3, 18.4),
                 (T_SILU, 2600, 16384, 4096, 410.4, 276.0), (T_RESID, 2048, 3584, 18944, 365.7, 222.8), (T_F32, 2048, 4096, 11008, 178.9, 158.1),
                 (T_RESID, 2048, 4096, 14336, 217.5, 195.9), (T_SILU, 1368, 16384, 3072, 137.4, 128.9), (T_SILU, 2594, 8192, 2560, 146.6, 108.2)]


def test_tile_rule_where_one_side_is_much_the_quicker():
    for kind, m, n, k, lib, tiles in LIBRARY_QUICKER + TILES_QUICKER:
        assert gemm_bf16._tile_wins(m, n, k, kind) == (tiles < lib), (kind, m, n, k)


# the same, us by the tiles of 256 x 256 and by others: (kind, rows, N, K, their slices, the others' tile and slices)
@pytest.mark.parametrize("kind, m, n, k, wide_us, slices, other, other_us", [
    (T_F32, 836, 8192, 4096, 92.5, 2, (1, 1), 85.3), (T_RESID, 1024, 8192, 8192, 143.4, 2, (1, 1), 136.3),
    (T_RESID, 160, 8192, 28672, 179.1, 8, (1, 4), 163.4), (T_RESID, 2048, 4096, 14336, 195.9, 2, (1, 1), 200.2),
    (T_F32, 2048, 3584, 18944, 222.8, 2, (1, 1), 280.4)])
def test_tiles_of_256_by_256_where_they_are_the_quicker_ones(kind, m, n, k, wide_us, slices, other, other_us):
    assert gemm_bf16.tile_plan(m, n, k, kind, True)[:2] == ((0, slices) if wide_us < other_us else other)


# us of both products of ``tokens`` rows for each of ``top`` of ``experts`` chosen at random, by the plan and by the one in its place
@pytest.mark.parametrize("tokens, experts, top, width, inter, plan, us, other, other_us", [
    (196, 8, 4, 6144, 3072, (128, 2, 2), 315.4, (128, 3, 3), 405.8), (767, 4, 1, 2560, 3072, (128, 2, 2), 68.0, (128, 3, 2), 81.4),
    (976, 4, 1, 4096, 2560, (128, 2, 2), 136.1, (128, 3, 2), 160.4), (1296, 4, 1, 4096, 14336, (256, 0, 1), 732.0, (128, 2, 3), 905.6),
    (382, 16, 4, 3072, 1536, (128, 2, 2), 173.2, (128, 3, 3), 206.6), (679, 16, 8, 5120, 8192, (256, 0, 1), 1904.4, (128, 2, 2), 2225.6)])
def test_experts_plans_count_rounds_as_their_tiles_take_them(tokens, experts, top, width, inter, plan, us, other, other_us):
    assert us < other_us and gemm_bf16.tile_groups_plan(tokens * top, experts, 2 * inter, width, width, inter) == plan != other


def test_few_rows_plans_count_what_their_reader_pays_for_a_plane():
    """41 to 64 rows: sizes where more planes were measured slower than fewer, or than the streaming kernel's (None), and sizes where
    they are the quicker ones; beyond 64 rows no slice of more than 1,536 values of K."""
    plan = gemm_bf16._few_rows_plan
    for (m, n, k), slices in {(48, 2048, 2048): 4, (41, 1024, 1024): 2, (48, 512, 1024): 4, (56, 1536, 1536): 4, (41, 4096, 1024): 2,
                              (64, 2048, 8192): 8, (48, 1024, 4096): 4}.items():
        assert plan(m, n, k) == (6, slices), (m, n, k)
    for m, n, k in ((48, 5120, 3072), (41, 6144, 4096), (64, 4096, 8192), (40, 2048, 2048), (65, 2048, 2048)):
        assert plan(m, n, k) is None, (m, n, k)
    assert plan(41, 5120, 3072, True) == (7, 4) and plan(64, 3072, 2048, True) == (6, 4) and plan(48, 6144, 4096, True) == (7, 4)
    assert plan(41, 768, 512, True) is None and plan(64, 768, 512, True) is not None and plan(64, 8192, 8192, True) is None
    for m, n, k in ((320, 1024, 8192), (200, 2048, 4096), (160, 1536, 6144), (1000, 512, 11008)):
        assert gemm_bf16._small_product_slices(m, n, k) == 0, (m, n, k)
    for (m, n, k), slices in {(200, 2048, 2048): 2, (65, 2048, 4096): 4, (128, 1024, 4096): 8, (160, 1024, 4096): 4, (128, 3072, 3072): 2}.items():
        assert gemm_bf16._small_product_slices(m, n, k) == slices, (m, n, k)


@pytest.mark.parametrize("n, k, made", [(3072, 2048, False), (5120, 3072, False), (6144, 4096, False), (7168, 5120, False), (768, 512, True)])
def test_the_planes_copy_of_q_k_v_is_made_only_where_it_is_read(n, k, made, monkeypatch):
    """Llama 1B, 3B, 8B and larger: 41 to 64 rows all go to the tile kernel or the library; very small ones to the kernel that reads it."""
    monkeypatch.setattr(gemm_bf16, "tile_weight_rope", lambda w: "few")
    monkeypatch.setattr(gemm_bf16, "tile_weight_planes", lambda w: "many")
    w = torch.empty(n, k, dtype=torch.bfloat16, device="meta")
    assert gemm_bf16.tile_copies_rope(w).many == ("many" if made else None)
    left = [m for m in range(41, 65) if gemm_bf16._few_rows_plan(m, n, k, True) is None
            and not gemm_bf16._library_wins(m, n, k, torch.bfloat16)]
    assert bool(left) == made


def test_products_that_small_tiles_and_planes_were_measured_slower_at():
    """What three rules leave to the kernels and the library that were there before them, and neighbours that they take."""
    for m, n, k in ((64, 28672, 5120), (40, 16384, 8192), (64, 22016, 5120)):
        assert not gemm_bf16._few_rows_swiglu(m, n, k), (m, n, k)
    for m, n, k in ((64, 28672, 4096), (40, 16384, 5120), (64, 16384, 2048), (33, 16384, 3072)):
        assert gemm_bf16._few_rows_swiglu(m, n, k), (m, n, k)
    for m, n, k in ((65, 2048, 4096), (96, 2048, 5120), (128, 2048, 5120), (256, 2048, 8192)):
        assert not gemm_bf16._small_swiglu(m, n, k), (m, n, k)
    for m, n, k in ((200, 2048, 4096), (128, 8192, 1024), (65, 4096, 512), (200, 4096, 8192)):
        assert gemm_bf16._small_swiglu(m, n, k), (m, n, k)
    for m, n, k in ((160, 6144, 2048), (320, 5120, 3072), (200, 12288, 4096), (320, 10240, 8192)):
        assert gemm_bf16._rope_planes_plan(m, n, k) is None, (m, n, k)
    for m, n, k in ((200, 3072, 2048), (128, 5120, 3072), (65, 6144, 4096), (400, 1536, 1024)):
        assert gemm_bf16._rope_planes_plan(m, n, k) is not None, (m, n, k)
