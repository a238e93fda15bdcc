"""Host logic of the prompt GEMM's launch geometry (prima_cpp_amd/csrc/mmq_pf.hip pm_gemm_pf_plan, through the C ABI - no GPU, no kernel launch): tile size by
batch, the uniform K split of launches with few tiles, and the tail-only split of launches that are full rounds of workgroups + a short tail. The shapes are
the layer shapes of BASELINE.json's models on a 256-CU device in 8 XCDs; every workgroup id of the planned grid must map to exactly one (tile, K slice)."""
import ctypes as C

import pytest

from prima_cpp_amd import lib as L

CUS = 256


def plan(tiles, K, T, mixed=1, cus=CUS):
    lib = L.load()
    lib.pm355_gemm_plan.restype = C.c_int
    lib.pm355_gemm_plan.argtypes = [C.c_int64, C.c_int64, C.c_int64, C.c_int, C.c_int, C.c_void_p]
    out = (C.c_int32 * 5)()
    assert lib.pm355_gemm_plan(tiles, K, T, cus, mixed, out) == 0
    return dict(tile_tokens=out[0], nt_t=out[1], S=out[2], full=out[3], grid=out[4])


def coverage(tiles, p):
    """The kernel's block id -> (row tile, token tile, K slice) mapping (gemm_pf_kernel), restated: returns {(tile_n, tile_t): sorted slices}."""
    seen = {}
    for bid in range(p["grid"]):
        x, q = bid & 7, bid >> 3
        if q < p["full"]:
            S, ks, slot = 1, 0, q
        else:
            S, ks, slot = p["S"], (q - p["full"]) % p["S"], p["full"] + (q - p["full"]) // p["S"]
        per_x = (tiles + 7 - x) >> 3
        if slot >= per_x * p["nt_t"]:
            continue
        key = (x + 8 * (slot // p["nt_t"]), slot % p["nt_t"])
        seen.setdefault(key, []).append((ks, S))
    return seen


@pytest.mark.parametrize("tiles,K,T", [(40, 8192, 2048), (231, 8192, 2048), (112, 8192, 2048), (224, 8192, 2048), (32, 8192, 2048), (32, 28672, 2048),
                                       (40, 8192, 512), (32, 8192, 512), (224, 8192, 512), (32, 28672, 512), (112, 8192, 64), (32, 8192, 40), (5, 1024, 300),
                                       (33, 4096, 2048), (17, 2048, 4096), (1, 512, 1)])
def test_every_tile_and_slice_is_covered_exactly_once(tiles, K, T):
    for mixed in (1, 0):
        p = plan(tiles, K, T, mixed)
        assert p["tile_tokens"] == (64 if T <= 64 else 128 if T <= 128 else 256)
        assert p["nt_t"] == -(-T // p["tile_tokens"])
        cov = coverage(tiles, p)
        assert len(cov) == tiles * p["nt_t"]
        for key, sl in cov.items():
            S = sl[0][1]
            assert sorted(sl) == [(k, S) for k in range(S)], (key, sl)
        if not mixed:
            assert p["full"] == 0
        if p["S"] > 1:
            assert (K + 255) // 256 // p["S"] >= 4                  # at least four super-blocks per slice


def test_layer_shapes_of_the_baseline_models():
    # Llama-3-70B, 2048-token prompt: wq | wk | wv = 40 row tiles x 8 token tiles = 320 workgroups on 256 CUs: one full round of whole tiles (32 slots per
    # XCD), the 64 tiles behind them in four K slices each (8 slots x 4 = the XCD's 32 CUs)
    assert plan(40, 8192, 2048) == dict(tile_tokens=256, nt_t=8, S=4, full=32, grid=8 * (32 + 8 * 4))
    # ... the uniform split it replaces: three slices of every tile
    assert plan(40, 8192, 2048, mixed=0)["S"] == 3 and plan(40, 8192, 2048, mixed=0)["full"] == 0
    # ffn_gate | ffn_up as pair tiles: 224 x 8 = exactly 7 rounds, nothing to split; wo / ffn_down: exactly one round
    assert plan(224, 8192, 2048) == dict(tile_tokens=256, nt_t=8, S=1, full=0, grid=8 * 224)
    assert plan(32, 8192, 2048)["S"] == 1 and plan(32, 28672, 2048)["S"] == 1
    # Qwen2.5-72B's pair launch: 231 tiles x 8 = 7 rounds + 56 tiles: XCDs 0..6 own 29 row tiles (232 slots), XCD 7 owns 28 - 224 whole-tile slots, the rest x 4
    assert plan(231, 8192, 2048) == dict(tile_tokens=256, nt_t=8, S=4, full=224, grid=8 * (224 + 8 * 4))
    # the reference's default micro-batch (n_ubatch 512, common/common.h:178): 64-80 tiles for 256 CUs - every tile split
    assert plan(32, 8192, 512)["S"] == 4 and plan(32, 8192, 512)["full"] == 0
    assert plan(32, 28672, 512)["S"] == 4
    assert plan(40, 8192, 512)["S"] == 3
    # 33..64-token batches: 64-token tiles, one token tile
    p = plan(32, 8192, 64)
    assert p["tile_tokens"] == 64 and p["nt_t"] == 1 and p["S"] == 8


@pytest.mark.parametrize("rows,K,T,S", [((4096, 1024, 1024), 4096, 101, 4), ((4096,), 4096, 101, 4), ((4096,), 14336, 101, 8), ((14336, 14336), 4096, 101, 1), ((8192,), 8192, 64, 4), ((132,), 512, 33, 1)])
def test_launches_of_128_row_tiles(rows, K, T, S):
    """Up to 128 tokens, launches with at most one 128-row tile per CU are planned on those tiles (of every matrix of the launch; a pair launch: 64 rows of each): Llama-3-8B's at 101 tokens"""
    tiles = -(-rows[0] // 64) if rows == (14336, 14336) else sum(-(-n // 128) for n in rows)
    assert tiles <= CUS
    p = plan(tiles, K, T)
    assert p["tile_tokens"] == (64 if T <= 64 else 128) and p["nt_t"] == 1 and p["S"] == S and p["full"] == 0
    cov = coverage(tiles, p)
    assert len(cov) == tiles and all(sorted(sl) == [(k, S) for k in range(S)] for sl in cov.values())


def test_bad_arguments_are_refused():
    lib = L.load()
    lib.pm355_gemm_plan.restype = C.c_int
    lib.pm355_gemm_plan.argtypes = [C.c_int64, C.c_int64, C.c_int64, C.c_int, C.c_int, C.c_void_p]
    out = (C.c_int32 * 5)()
    assert lib.pm355_gemm_plan(0, 8192, 512, CUS, 1, out) != 0
    assert lib.pm355_gemm_plan(4, 8192, 512, CUS, 1, None) != 0
    assert lib.pm355_gemm_plan(4, 128, 512, CUS, 1, out) != 0


ROWS_256, ROWS_128, WIDE_Q4_K, WIDE = 2, 4, 8, 16


def every_slice_once(tiles, p):
    cov = coverage(tiles, p)
    return len(cov) == tiles * p["nt_t"] and all(sorted(sl) == [(k, sl[0][1]) for k in range(sl[0][1])] for sl in cov.values())


@pytest.mark.parametrize("tiles,K,T,tile", [
    (112, 4096, 129, 192), (112, 4096, 192, 192), (112, 4096, 193, 256), (112, 4096, 300, 192), (112, 4096, 384, 192), (112, 4096, 385, 256), (112, 4096, 512, 256),      # ffn_gate | ffn_up of the 8B shape
    (112, 4096, 128, 128), (112, 4096, 64, 64), (112, 4096, 6001, 256), (224, 8192, 513, 192), (224, 8192, 576, 192), (224, 8192, 577, 256),
    (224, 8192, 256, 256), (224, 8192, 257, 192), (224, 8192, 384, 192), (224, 8192, 385, 256), (231, 8192, 300, 192), (501, 4096, 320, 192), (501, 4096, 1300, 256), (108, 5120, 1344, 256), (32, 29568, 513, 192),
    (24, 4096, 150, 192), (24, 4096, 1500, 192), (24, 4096, 6001, 192), (16, 4096, 3000, 192), (16, 4096, 6001, 192), (16, 14336, 380, 192), (17, 2048, 4096, 256), (5, 1024, 300, 192),
    (4, 8192, 777, 256), (4, 8192, 1100, 192), (9, 4096, 4096, 256), (9, 4096, 300, 192), (17, 4096, 2100, 256), (25, 4096, 777, 256), (50, 8192, 777, 256), (8, 8192, 777, 256)])
def test_tiles_of_256_rows_as_launched(tiles, K, T, tile):
    """tiles of 192 tokens beside those of 256, on either side of where they change; the K split stays that of 256 tokens, a split of the last tiles only goes; no tile or slice is left out. Where row
    tiles do not divide by eight, the XCDs that own one more decide"""
    p, by_tokens = plan(tiles, K, T, ROWS_256), plan(tiles, K, T)
    assert p["tile_tokens"] == tile and p["nt_t"] == -(-T // tile) and every_slice_once(tiles, p)
    if tile != 192:
        assert p == by_tokens
    else:
        assert p["full"] == 0 and p["S"] == (1 if by_tokens["full"] else by_tokens["S"])


def test_tiles_of_192_tokens_over_many_sizes():
    """every plan covers its tiles, and one of 192 tokens has fewer or as many sub-tiles of 32 tokens in its rounds of workgroups"""
    taken = 0
    for tiles in (1, 7, 16, 24, 40, 64, 112, 128, 200, 224, 255, 501):
        for K in (512, 1024, 4096, 14336):
            for T in (129, 191, 192, 193, 256, 257, 320, 384, 385, 448, 449, 512, 513, 576, 577, 700, 1000, 1345, 2049, 4000):
                p, q = plan(tiles, K, T, ROWS_256), plan(tiles, K, T)
                assert every_slice_once(tiles, p), (tiles, K, T, p)
                if p["tile_tokens"] == 256:
                    assert p == q
                    continue
                taken += 1
                rounds = lambda x, tile: -(-(-(-tiles // 8)) * x["nt_t"] * x["S"] // (CUS // 8)) * (tile // 32 + 1)  # noqa: E731      (of the XCD with the most row tiles)
                assert p["tile_tokens"] == 192 and (q["full"] or rounds(p, 192) < rounds(q, 256)), (tiles, K, T, p, q)
    assert taken > 100


@pytest.mark.parametrize("tiles,K,T,flags,tile", [(32, 4096, 64, ROWS_128, 64), (32, 4096, 65, ROWS_128, 96), (32, 14336, 96, ROWS_128, 96), (32, 4096, 97, ROWS_128, 128), (224, 4096, 128, ROWS_128, 128),
                                                  (32, 4096, 40, WIDE_Q4_K, 64), (224, 4096, 79, WIDE_Q4_K, 96), (224, 4096, 147, WIDE_Q4_K, 96), (224, 4096, 128, WIDE_Q4_K, 128), (32, 4096, 500, WIDE_Q4_K, 128),
                                                  (83, 2048, 231, WIDE_Q4_K, 128), (18, 4096, 231, WIDE_Q4_K, 128), (99, 8192, 385, WIDE_Q4_K, 128), (84, 8192, 300, WIDE_Q4_K, 96), (11, 4096, 459, WIDE_Q4_K, 128),
                                                  (32, 14336, 40, WIDE, 64), (32, 14336, 147, WIDE, 64), (1, 512, 512, WIDE, 64)])
def test_tiles_of_128_rows_as_launched(tiles, K, T, flags, tile):
    """up to 128 tokens 64, 96 or 128 a tile; of 8-bit activations 96 beside 128 by rounds of workgroups (of the XCD with the most row tiles), 64 with other types than Q4_K"""
    p = plan(tiles, K, T, flags)
    assert p["tile_tokens"] == tile and p["nt_t"] == -(-T // tile) and every_slice_once(tiles, p), p


def test_forms_that_have_no_launch_are_refused():
    lib, out = L.load(), (C.c_int32 * 5)()
    lib.pm355_gemm_plan.argtypes = [C.c_int64, C.c_int64, C.c_int64, C.c_int, C.c_int, C.c_void_p]
    assert lib.pm355_gemm_plan(4, 512, 129, CUS, ROWS_128, out) != 0 and lib.pm355_gemm_plan(4, 512, 513, CUS, WIDE, out) != 0 and lib.pm355_gemm_plan(4, 512, 513, CUS, WIDE_Q4_K, out) != 0
