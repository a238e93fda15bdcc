"""GPU parity tests (run with -m gpu on an MI355X): every op goes through the C ABI of
libprima_mi355.so and is compared with the CPU oracle on the same seeded inputs.
Integer / byte results: bit-exact. Float results: tolerance stated per test."""
import ctypes as C
import os

import numpy as np
import pytest

from _bind import Q4_K, Q5_K, Q6_K, Q8_0, Q8_K, QUANT_TYPES, TYPE_NAMES, rand_blocks, row_size, vec_dot_type

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def P():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("GPU tests need a HIP device")
    import prima_cpp_amd.ops as ops
    ops.torch = torch
    return ops


def _dev(P, a):
    return P.torch.from_numpy(np.ascontiguousarray(a)).to("cuda")


def _acts(rng, k, kind):
    if kind == "normal":
        return rng.normal(0, 1, k).astype(np.float32)
    if kind == "cos":
        return (0.1 + 2 * np.cos(np.arange(k, dtype=np.float32))).astype(np.float32)
    if kind == "zeros":
        return np.zeros(k, dtype=np.float32)
    if kind == "ties":
        x = rng.normal(0, 0.1, k).astype(np.float32)
        x[5::256] = -3.0
        x[9::256] = 3.0
        if k > 300:
            x[300] = 3.0      # second block: positive one comes first
            x[261] = 0.0
        return x
    if kind == "halfway":
        return ((np.arange(k) % 255 - 127).astype(np.float32) * 0.5).astype(np.float32)
    if kind == "sparse":
        x = np.zeros(k, dtype=np.float32)
        x[::97] = rng.normal(0, 5, x[::97].size)
        return x
    raise ValueError(kind)


@pytest.mark.parametrize("kind", ["normal", "cos", "zeros", "ties", "halfway", "sparse"])
@pytest.mark.parametrize("K", [256, 2048, 8192])
def test_quantize_q8_K_bitexact(P, oracle, kind, K):
    rng = np.random.default_rng(21)
    x = np.stack([_acts(rng, K, kind), _acts(rng, K, "normal"), _acts(rng, K, kind)])
    yq = P.quantize_act(_dev(P, x), Q8_K)
    got = P.act_to_ggml_blocks(yq, Q8_K, K, 3).reshape(3, -1)
    for r in range(3):
        want = oracle.quantize_row_q8_K(x[r])
        assert np.array_equal(got[r], want), (kind, K, r)


@pytest.mark.parametrize("kind", ["normal", "cos", "zeros", "halfway", "sparse"])
def test_quantize_q8_0_bitexact(P, oracle, kind):
    rng = np.random.default_rng(22)
    K = 4096
    x = np.stack([_acts(rng, K, kind), _acts(rng, K, "normal")])
    yq = P.quantize_act(_dev(P, x), Q8_0)
    got = P.act_to_ggml_blocks(yq, Q8_0, K, 2).reshape(2, -1)
    for r in range(2):
        assert np.array_equal(got[r], oracle.quantize_row_q8_0(x[r]))


@pytest.mark.parametrize("K,rows", [(32, 1), (32, 1025), (96, 77), (256, 1), (256, 4099), (480, 501), (512, 130), (2080, 9)])
def test_quantizers_of_short_rows_bitexact(P, oracle, K, rows):
    """one index over rows and blocks (less than 512 values), rows x groups (the others): first, last and odd rows against the oracle"""
    x = np.random.default_rng(K + rows).normal(0, 1, (rows, K)).astype(np.float32)
    for t, row in ((Q8_0, oracle.quantize_row_q8_0), (Q8_K, oracle.quantize_row_q8_K)):
        if t == Q8_K and K % 256:
            continue
        got = P.act_to_ggml_blocks(P.quantize_act(_dev(P, x), t), t, K, rows).reshape(rows, -1)
        for r in sorted({*range(min(rows, 40)), *range(max(rows - 9, 0), rows), *range(0, rows, 97)}):
            assert np.array_equal(got[r], row(x[r])), (t, r)


@pytest.mark.parametrize("t", QUANT_TYPES)
@pytest.mark.parametrize("K", [2048, 768])
def test_repack_roundtrip_bitexact(P, t, K):
    rng = np.random.default_rng(23)
    N = 19
    blocks = rand_blocks(t, N, K, rng)
    w = P.upload_weight(t, blocks, K, N)
    assert np.array_equal(P.download_weight(w), blocks)
    if t in (Q4_K, Q6_K, Q8_0):  # and the HBM image is the documented row-SoA permutation (rows 16-B aligned):
        # one stream per 16-byte piece a lane loads (repack.hip)
        stride = P.L.load().pm355_row_stride(t, K)
        assert stride % 16 == 0 and 0 <= stride - row_size(t, K) < 16
        img = w.data.cpu().numpy().reshape(N, stride)[:, :row_size(t, K)]
        src = blocks.reshape(N, -1)
        if t == Q6_K:
            nb = K // 256
            b = src.reshape(N, nb, 210)
            ql = b[:, :, :128].reshape(N, nb, 2, 2, 2, 16)          # [block][half hh][second][v][16]
            la = ql[:, :, :, 0].reshape(N, -1)                       # unit order (b, hh, v)
            lb = ql[:, :, :, 1].reshape(N, -1)
            if P.L.load().pm355_q6k_tail_grouped():                  # round 5: per group of <= 8 blocks scales[r][16] | d[r]
                tail = [np.concatenate([b[:, g0:g0 + 8, 192:208].reshape(N, -1), b[:, g0:g0 + 8, 208:].reshape(N, -1)], axis=1) for g0 in range(0, nb, 8)]
            else:
                tail = [b[:, :, 192:208].reshape(N, -1), b[:, :, 208:].reshape(N, -1)]
            want = np.concatenate([la, lb, b[:, :, 128:192].reshape(N, -1)] + tail, axis=1)
        elif t == Q4_K:
            nb = K // 256
            b = src.reshape(N, nb, 144)
            qs = b[:, :, 16:].reshape(N, nb, 4, 2, 16)               # [block][j][second][16]
            want = np.concatenate([qs[:, :, :, 0].reshape(N, -1), qs[:, :, :, 1].reshape(N, -1),
                                   b[:, :, :16].reshape(N, -1)], axis=1)
        else:
            nb = K // 32
            b = src.reshape(N, nb, 34)
            qs = b[:, :, 2:].reshape(N, nb, 2, 16)
            want = np.concatenate([qs[:, :, 0].reshape(N, -1), qs[:, :, 1].reshape(N, -1), b[:, :, :2].reshape(N, -1)], axis=1)
        assert np.array_equal(img, want)


@pytest.mark.parametrize("threads", [0, 3])
def test_async_uploader_matches_synchronous_set_tensor(P, threads):
    """upload.hip (pinned ring + copier threads + private stream + repack per chunk) leaves exactly the HBM image of the synchronous
    H2D + repack path, for chunks smaller than a tensor (rows split over many chunks), ragged tails, and plain byte tensors."""
    import ctypes as C
    import torch
    lib = P.L.load()
    rng = np.random.default_rng(231)
    up = lib.pm355_uploader_new(1 << 20, threads)                      # 1-MiB chunks: every tensor below spans several
    assert up
    try:
        total = 0
        for t, K, N in ((Q4_K, 4096, 1500), (Q6_K, 2304, 1111), (Q8_0, 1056, 4099), (Q5_K, 2048, 999)):
            blocks = rand_blocks(t, N, K, rng)
            want = P.upload_weight(t, blocks, K, N)
            host = np.ascontiguousarray(blocks, dtype=np.uint8).reshape(-1)
            dst = torch.zeros_like(want.data)
            assert lib.pm355_upload(up, t, K, host.ctypes.data, dst.data_ptr(), host.size, 1) == 0
            host[:] = 0                                               # the source may be reused as soon as the call returns
            assert lib.pm355_uploader_sync(up) == 0
            assert torch.equal(dst, want.data)
            total += host.size
        raw = rng.integers(0, 256, (3 << 20) + 12345, dtype=np.uint8)
        dst = torch.zeros(raw.size, dtype=torch.uint8, device="cuda")
        assert lib.pm355_upload(up, -1, 0, raw.ctypes.data, dst.data_ptr(), raw.size, 0) == 0
        assert lib.pm355_uploader_sync(up) == 0
        assert np.array_equal(dst.cpu().numpy(), raw)
        assert lib.pm355_uploader_bytes(up) == total + raw.size
        # a row that does not fit a chunk is refused, never truncated
        big = rand_blocks(Q4_K, 1, 2 << 20, rng).reshape(-1)
        d2 = torch.zeros(big.size, dtype=torch.uint8, device="cuda")
        assert lib.pm355_upload(up, Q4_K, 2 << 20, big.ctypes.data, d2.data_ptr(), big.size, 1) != 0
    finally:
        lib.pm355_uploader_free(up)


@pytest.mark.parametrize("t", QUANT_TYPES)
@pytest.mark.parametrize("K,N", [(256, 3), (768, 5), (2048, 5), (4096, 37), (5120, 4), (8192, 64), (14336, 9), (28672, 6)])
def test_gemv_integer_partials_bitexact_and_float_close(P, oracle, t, K, N):
    rng = np.random.default_rng(24)
    blocks = rand_blocks(t, N, K, rng)
    x = rng.normal(0, 1, K).astype(np.float32)
    w = P.upload_weight(t, blocks, K, N)
    xq = P.quantize_act(_dev(P, x[None]), vec_dot_type(t))
    y, ip = P.mul_mat_vec_dbg(w, xq)
    y, ip = y.cpu().numpy(), ip.cpu().numpy().astype(np.int64)
    a = oracle.quantize_act(t, x)
    rs = row_size(t, K)
    upb = ip.shape[1] // (K // (32 if t == Q8_0 else 256))      # units per activation block
    for r in range(N):
        wr = blocks[r * rs:(r + 1) * rs]
        isum, msum = oracle.int_partials(t, K, wr, a)
        got_i = ip[r, :, 0].reshape(-1, upb).sum(1)
        got_m = ip[r, :, 1].reshape(-1, upb).sum(1)
        assert np.array_equal(got_i, isum.astype(np.int64)), (TYPE_NAMES[t], K, r)
        assert np.array_equal(got_m, msum.astype(np.int64)), (TYPE_NAMES[t], K, r)
        want = oracle.vec_dot(t, K, wr, a)
        mag = float(np.abs(oracle.dequantize_row(t, wr, K)) @ np.abs(x))
        # identical integer terms; only the f32 summation order differs (K/256 <= 112 terms)
        assert abs(y[r] - want) <= 4e-6 * mag + 1e-30, (TYPE_NAMES[t], K, r, y[r], want)


@pytest.mark.parametrize("t", [Q4_K, Q6_K, Q8_0])
def test_gemv_rows_whatever_the_slices(P, t):
    """A row's product is the same bits whatever the number of rows, i.e. the slice that it is in: fewer rows than workgroups, whole slices, slices of unequal length, more rows than 256 workgroups
    take (one matrix, and pairs)."""
    K, most, rng = 256, 131077, np.random.default_rng(55)
    b = rand_blocks(t, 4099, K, rng).reshape(4099, -1)
    blocks = np.concatenate([b] * (most // 4099 + 1))[:most]
    x = _dev(P, rng.normal(0, 1, (1, K)).astype(np.float32))
    w = lambda n, at=0: P.upload_weight(t, np.ascontiguousarray(blocks[at:at + n]).reshape(-1), K, n)
    y, pair = P.mul_mat_vec(w(most), x=x), P.mul_mat_vec(w(most), x=x, w2=w(most))
    assert P.torch.equal(y[:, 4099:2 * 4099], y[:, :4099]) and P.torch.equal(y[:, 31 * 4099:], y[:, :most - 31 * 4099])
    for n in (1, 3, 255, 256, 257, 511, 1000, 4098):
        assert P.torch.equal(P.mul_mat_vec(w(n, 77), x=x), y[:, 77:77 + n]), n
        assert P.torch.equal(P.mul_mat_vec(w(n, 77), x=x, w2=w(n, 77)), pair[:, 77:77 + n]), n


def test_gemv_of_more_rows_than_a_launch_takes(P):
    """34 million rows, launched in pieces: the bits of the same rows in a small matrix - with a bias, as a pair, several columns, and beside another matrix"""
    K, part, N, rng, torch = 32, 10007, 34000001, np.random.default_rng(56), P.torch
    small = P.upload_weight(Q8_0, rand_blocks(Q8_0, part, K, rng).reshape(-1), K, part)
    stretch = lambda v: v.repeat((N + part - 1) // part, *[1] * (v.ndim - 1))[:N]
    large = P.QWeight(Q8_0, K, N, stretch(small.data.view(part, -1)).reshape(-1))
    b = _dev(P, rng.normal(0, 1, part).astype(np.float32))
    x = _dev(P, rng.normal(0, 1, (8, K)).astype(np.float32))
    same = lambda got, want: all(torch.equal(g, stretch(w)) for g, w in zip(got, want))
    for n in (1, 3, 8):
        assert same(P.mul_mat_vec(large, x=x[:n], bias=stretch(b)), P.mul_mat_vec(small, x=x[:n], bias=b)), n
    assert same(P.mul_mat_vec(large, x=x[:1], w2=large), P.mul_mat_vec(small, x=x[:1], w2=small))
    got, beside = P.mul_mat_vec_fused([large, small], x[0])
    want = P.mul_mat_vec_fused([small], x[0])[0]
    assert torch.equal(got, stretch(want)) and torch.equal(beside, want)


@pytest.mark.parametrize("C", [2, 3, 4, 5, 7, 8])       # column slots per launch group (mmvq_cols.hip): 2, 4 (one idle), 4, 4+1, 4+4 (one idle), 8; pairs: 2 per launch
@pytest.mark.parametrize("t", QUANT_TYPES)
def test_gemv_epilogues_and_columns(P, oracle, t, C):
    rng = np.random.default_rng(25)
    K, N = 4096, 70
    b1, b2 = rand_blocks(t, N, K, rng), rand_blocks(t, N, K, rng)
    x = rng.normal(0, 1, (C, K)).astype(np.float32)
    bias = rng.normal(0, 1, N).astype(np.float32)
    resid = rng.normal(0, 1, (C, N)).astype(np.float32)
    w1, w2 = P.upload_weight(t, b1, K, N), P.upload_weight(t, b2, K, N)
    want1 = oracle.mul_mat(t, b1, K, N, x)
    want2 = oracle.mul_mat(t, b2, K, N, x)
    tol = dict(rtol=2e-5, atol=2e-5)
    y = P.mul_mat_vec(w1, x=_dev(P, x)).cpu().numpy()
    assert np.allclose(y, want1, **tol)
    y = P.mul_mat_vec(w1, x=_dev(P, x), bias=_dev(P, bias), resid=_dev(P, resid)).cpu().numpy()
    assert np.allclose(y, want1 + bias[None] + resid, **tol)
    y = P.mul_mat_vec(w1, x=_dev(P, x), w2=w2).cpu().numpy()
    assert np.allclose(y, oracle.silu_mul(want1, want2), rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("T", [1, 3, 8, 9, 16, 17, 33, 64])
def test_small_batch_matmul_q8_0_blocks(P, oracle, T):
    """mmq_i8.hip, Q8_0 weights x Q8_0 activations (ggml_vec_dot_q8_0_q8_0: integer block sums times d_w * d_a, f32): one 32-k matrix instruction per
    block. Shapes: K not a multiple of 128 or 256 (Qwen2.5-72B's ffn_down fallback, K = 29568 = 924 blocks: the last step holds 4 of 8 blocks), ragged rows,
    several row groups; passes of 16 tokens over 32-slot tables (T = 17, 33: second half / second table)."""
    rng = np.random.default_rng(4000 + T)
    for K, N in ((4096, 70), (608, 600), (1184, 9000), (29568, 40)):
        if (N == 9000 or K == 29568) and T not in (3, 17, 64): continue
        b = rand_blocks(Q8_0, N, K, rng)
        x = rng.normal(0, 1, (T, K)).astype(np.float32)
        bias = rng.normal(0, 1, N).astype(np.float32)
        resid = rng.normal(0, 1, (T, N)).astype(np.float32)
        w = P.upload_weight(Q8_0, b, K, N)
        want = oracle.mul_mat(Q8_0, b, K, N, x)
        tol = dict(rtol=2e-5, atol=2e-5 * np.sqrt(K / 4096))
        y = P.mul_mat_small(w, x=_dev(P, x)).cpu().numpy()
        assert np.isfinite(y).all()
        assert np.allclose(y, want, **tol), (K, N, np.abs(y - want).max())
        xq = P.quantize_act(_dev(P, x), P.vec_dot_act_type(Q8_0))
        y2 = P.mul_mat_small(w, xq=xq, n_tokens=T, bias=_dev(P, bias), resid=_dev(P, resid)).cpu().numpy()
        assert np.allclose(y2, want + bias[None] + resid, **tol)
        if T <= 8:
            y1 = P.mul_mat_vec(w, xq=xq, ncols=T).cpu().numpy()
            assert np.allclose(y, y1, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("T", [1, 2, 5, 8, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("t", [Q4_K, Q5_K, Q6_K])
def test_small_batch_matmul_on_integer_matrix_cores(P, oracle, t, T):
    """mmq_i8.hip: same integer block sums as the mat-vec (vec_dot_q4_K_q8_K / vec_dot_q6_K_q8_K), f32 super-block terms added in a
    different order -> oracle.mul_mat within the mat-vec's tolerance. Shapes: ragged row slices (N = 70: clamped rows), several row
    groups per workgroup (N = 600 on <= 256 workgroups is 1 group; N = 20000 gives 3), odd super-block count (K = 768)."""
    rng = np.random.default_rng(100 * t + T)
    for K, N in ((4096, 70), (768, 600), (1024, 20000)):
        if N == 20000 and T not in (5, 32, 64): continue
        b = rand_blocks(t, N, K, rng)
        x = rng.normal(0, 1, (T, K)).astype(np.float32)
        bias = rng.normal(0, 1, N).astype(np.float32)
        resid = rng.normal(0, 1, (T, N)).astype(np.float32)
        w = P.upload_weight(t, b, K, N)
        want = oracle.mul_mat(t, b, K, N, x)
        tol = dict(rtol=2e-5, atol=2e-5 * np.sqrt(K / 4096))
        y = P.mul_mat_small(w, x=_dev(P, x)).cpu().numpy()
        assert np.allclose(y, want, **tol), (K, N, np.abs(y - want).max())
        xq = P.quantize_act(_dev(P, x), P.vec_dot_act_type(t))
        y2 = P.mul_mat_small(w, xq=xq, n_tokens=T, bias=_dev(P, bias), resid=_dev(P, resid)).cpu().numpy()
        assert np.allclose(y2, want + bias[None] + resid, **tol)
        # against the mat-vec itself: identical integers, f32 sums of <= K/256 terms in another order
        if T <= 8:
            y1 = P.mul_mat_vec(w, xq=xq, ncols=T).cpu().numpy()
            assert np.allclose(y, y1, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("t", [Q4_K, Q6_K])
def test_prompt_matmul_on_integer_matrix_cores(P, oracle, t):
    """mmq_big.hip: prompt-sized batches with the CPU reference's integer arithmetic (Q8_K activations, exact int32 sub-block sums, one f32
    multiply-add per super-block, super-blocks in k order) -> oracle.mul_mat within f32 summation order, where the F16 GEMM sits at 1e-3.
    Shapes: ragged token and row tiles (T = 130 / 200, N = 70 / 300: clamped rows and tokens, tables of a partial 32-token pass), several
    tiles per XCD (N = 4100), many super-blocks (K = 8192), bias + residual epilogue; and the mat-vec's own result for the same rows."""
    rng = np.random.default_rng(900 + t)
    for K, N, T in ((1024, 70, 130), (2048, 300, 200), (8192, 520, 128), (1024, 4100, 257)):
        b = rand_blocks(t, N, K, rng)
        x = rng.normal(0, 1, (T, K)).astype(np.float32)
        bias = rng.normal(0, 1, N).astype(np.float32)
        resid = rng.normal(0, 1, (T, N)).astype(np.float32)
        w = P.upload_weight(t, b, K, N)
        want = oracle.mul_mat(t, b, K, N, x)
        tol = dict(rtol=2e-5, atol=2e-5 * np.sqrt(K / 4096))
        y = P.mul_mat_i8(w, _dev(P, x)).cpu().numpy()
        assert np.isfinite(y).all()
        assert np.allclose(y, want, **tol), (K, N, T, np.abs(y - want).max(), np.argwhere(~np.isclose(y, want, **tol))[:8])
        y2 = P.mul_mat_i8(w, _dev(P, x), bias=_dev(P, bias), resid=_dev(P, resid)).cpu().numpy()
        assert np.allclose(y2, want + bias[None] + resid, **tol)
        xq = P.quantize_act(_dev(P, x[:4]), P.vec_dot_act_type(t))
        y1 = P.mul_mat_vec(w, xq=xq, ncols=4).cpu().numpy()
        assert np.allclose(y[:4], y1, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("t", [Q4_K, Q5_K, Q6_K])
def test_wide_batch_matmul_with_8_bit_activations(P, oracle, t):
    """The prompt GEMM's 8-bit form: whole-number sums of every half super-block in the F16 matrix cores -> oracle.mul_mat (integers) within the tolerance of the integer kernels. Edges: rows and
    tokens of partial tiles, either tile size (33 / 64, 65 / 128 tokens), an odd number of super-blocks, K split over workgroups (32 super-blocks), matrices of two types, pair tiles. Quants and
    scales at their limits: weights of all-ones bytes (Q6_K: the largest quants with scales of -1, Q4_K / Q5_K the largest quants, scales and minima) and scales of -128 (Q6_K: products of 4096)."""
    rng = np.random.default_rng(700 + t)
    for K, N, T in ((768, 132, 33), (4096, 72, 64), (1024, 600, 65), (8192, 260, 128), (512, 4, 1), (1024, 132, 129), (512, 260, 512)):
        b, b2 = rand_blocks(t, N, K, rng), rand_blocks(Q4_K if t == Q6_K else Q6_K, 64, K, rng)
        x = rng.normal(0, 1, (T, K)).astype(np.float32)
        x[0] = 0
        bias, resid = rng.normal(0, 1, N).astype(np.float32), rng.normal(0, 1, (T, N)).astype(np.float32)
        w, w2 = P.upload_weight(t, b, K, N), P.upload_weight(Q4_K if t == Q6_K else Q6_K, b2, K, 64)
        want, want2 = oracle.mul_mat(t, b, K, N, x), oracle.mul_mat(w2.type, b2, K, 64, x)
        tol = dict(rtol=2e-5, atol=2e-5 * np.sqrt(K / 4096))
        y, y2 = P.mul_mat_wide([w, w2], _dev(P, x), biases=[_dev(P, bias), None], resids=[_dev(P, resid), None])
        assert np.allclose(y.cpu().numpy(), want + bias[None] + resid, **tol), (K, N, T, np.abs(y.cpu().numpy() - want - bias[None] - resid).max())
        assert np.allclose(y2.cpu().numpy(), want2, **tol)
        g = P.mul_mat_wide([w, w], _dev(P, x / 8), pair=True)[0].cpu().numpy()
        p = oracle.mul_mat(t, b, K, N, x / 8).astype(np.float64)
        err = (2 + np.abs(p)) * 2e-5 * (np.abs(p) + np.sqrt(K / 4096))          # |d(silu(p) p) / dp| < 2 |p| + 0.2, times the error of p
        assert (np.abs(g - p / (1 + np.exp(-p)) * p) <= err + 1e-6).all()
    K, N, T = 1024, 64, 40
    b = np.full(rand_blocks(t, N, K, rng).shape, 0xFF, np.uint8).reshape(N, K // 256, -1)
    if t == Q6_K:
        b[:, :, :192] = np.where(rng.random((N, K // 256, 192)) < 0.5, 0, 255)
        b[:, :, 192:208] = np.where(rng.random((N, K // 256, 16)) < 0.5, 0x80, 0x7F)
        b[:, :, 208:] = np.frombuffer(np.float16(0.01).tobytes(), np.uint8)
    else:
        b[:, :, :4] = np.frombuffer(np.float16([0.01, 0.02]).tobytes(), np.uint8)
    b = b.reshape(-1)
    for x in (np.ones((T, K), np.float32), rng.choice([-1.0, 1.0], (T, K)).astype(np.float32), rng.normal(0, 1, (T, K)).astype(np.float32)):
        want = oracle.mul_mat(t, b, K, N, x)
        y = P.mul_mat_wide([P.upload_weight(t, b, K, N)], _dev(P, x))[0].cpu().numpy()
        # (the sums cancel: three f32 roundings of each half super-block's sum and one of every sum so far, 2^-24 of at most sum |w x| each, here and in the oracle)
        lim = (3 + 2 * (K // 256)) * 2 * 2.0 ** -24 * K * {Q4_K: 945, Q5_K: 1953, Q6_K: 4096}[t] * 0.01 * np.abs(x).max()
        assert np.allclose(y, want, rtol=2e-5, atol=2e-5 + lim), np.abs(y - want).max()


@pytest.mark.parametrize("T", [40, 130])
@pytest.mark.parametrize("t", [Q4_K, Q5_K, Q6_K])
def test_wide_batch_matmul_adds_whole_numbers_exactly(P, oracle, t, T):
    """Quants and scales at their largest (Q6_K: 31 x 127, odd), values of 126 and 127 that change sign between the 128-k halves of a super-block: partial sums of up to 64 x 3937 x 127 = 2^24.9 on
    the way to a few ten thousand. Whole numbers of that size are not all in f32's 24 bits: the sums of a super-block have to be exact, as in the integer kernels. Bound: three roundings of each
    half super-block's sum and one of every sum so far, 2^-24 of what they round, here and in the oracle."""
    rng = np.random.default_rng(900 + t + T)
    K, N = 1024, 64
    nb = K // 256
    b = np.full(rand_blocks(t, N, K, rng).shape, 0xFF, np.uint8).reshape(N, nb, -1)
    if t == Q6_K:
        b[:, :, 192:208], b[:, :, 208:] = 0x7F, np.frombuffer(np.float16(0.01).tobytes(), np.uint8)
    else:
        b[:, :, :4] = np.frombuffer(np.float16([0.01, 0.0]).tobytes(), np.uint8)
    b = b.reshape(-1)
    v = rng.integers(126, 128, (T, nb, 2, 128))
    v[:, :, 0, 0] = 127
    v[:, :, 1] *= -1
    x = (v / 127.0).astype(np.float32).reshape(T, K)
    half = np.abs(v.reshape(T, nb, 2, 2, 64).sum((2, 4))).sum((1, 2)) * {Q4_K: 15 * 63, Q5_K: 31 * 63, Q6_K: 31 * 127}[t] * float(np.float16(0.01)) / 127
    want = oracle.mul_mat(t, b, K, N, x)
    y = P.mul_mat_wide([P.upload_weight(t, b, K, N)], _dev(P, x))[0].cpu().numpy()
    err = np.abs(y.astype(np.float64) - want)
    assert (err <= (half * (3 + 2 * nb) * 2 * 2.0 ** -24)[:, None]).all(), (err.max(), half.max())


@pytest.mark.parametrize("t", [Q4_K, Q6_K])
def test_small_batch_matmul_multi_job_launch(P, oracle, t):
    """wq | wk | wv and ffn_gate | ffn_up as ONE launch over a virtual row space: every job equals its own single-job launch (same integers; the
    K split over waves may differ) and the oracle; row groups straddle the job boundaries (N not a multiple of 32)."""
    rng = np.random.default_rng(300 + t)
    for K, Ns, T in ((1024, (300, 70, 75), 5), (768, (2100, 2100), 16), (4096, (515, 40), 9), (1024, (300, 70, 75), 20), (2048, (2100, 2100), 32), (1024, (300, 70), 45), (768, (600, 600, 90), 64)):
        blocks = [rand_blocks(t, N, K, rng) for N in Ns]
        ws = [P.upload_weight(t, b, K, N) for b, N in zip(blocks, Ns)]
        x = rng.normal(0, 1, (T, K)).astype(np.float32)
        biases = [rng.normal(0, 1, N).astype(np.float32) for N in Ns]
        xq = P.quantize_act(_dev(P, x), P.vec_dot_act_type(t))
        ys = P.mul_mat_small_multi(ws, xq, T, biases=[_dev(P, b) for b in biases])
        for w, b, bias, y in zip(ws, blocks, biases, ys):
            want = oracle.mul_mat(t, b, K, w.N, x) + bias[None]
            got = y.cpu().numpy()
            assert np.allclose(got, want, rtol=2e-5, atol=2e-5 * np.sqrt(K / 4096)), (K, w.N, np.abs(got - want).max())
            one = P.mul_mat_small(w, xq=xq, n_tokens=T, bias=_dev(P, bias)).cpu().numpy()
            assert np.allclose(got, one, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("tv", [Q6_K, Q5_K])
def test_small_batch_matmul_wv_of_another_type_in_the_same_grid(P, oracle, tv):
    """wq | wk (Q4_K) and wv (Q6_K / Q5_K: the Q4_K_M files' use_more_bits layers, src/llama.cpp:19447) as ONE grid - the device's workgroups divided by
    weight bytes, every part with its own row split: each job equals its own single launch (same integers; the K split over waves may differ) and the oracle."""
    rng = np.random.default_rng(330 + tv)
    for K, Ns, T in ((1024, (300, 70, 75), 5), (8192, (1024, 128, 128), 8), (2048, (2100, 260, 300), 16), (4096, (515, 40, 33), 9)) + (((1024, (600, 64, 90), 32), (8192, (520, 130, 100), 24)) if tv == Q6_K else ()):
        types = (Q4_K, Q4_K, tv)
        blocks = [rand_blocks(t, N, K, rng) for t, N in zip(types, Ns)]
        ws = [P.upload_weight(t, b, K, N) for t, b, N in zip(types, blocks, Ns)]
        x = rng.normal(0, 1, (T, K)).astype(np.float32)
        biases = [rng.normal(0, 1, N).astype(np.float32) for N in Ns]
        xq = P.quantize_act(_dev(P, x), P.vec_dot_act_type(Q4_K))
        ys = P.mul_mat_small_mixed(ws, xq, T, biases=[_dev(P, b) for b in biases])
        for w, t, b, bias, y in zip(ws, types, blocks, biases, ys):
            want = oracle.mul_mat(t, b, K, w.N, x) + bias[None]
            got = y.cpu().numpy()
            assert np.allclose(got, want, rtol=2e-5, atol=2e-5 * np.sqrt(K / 4096)), (K, w.N, np.abs(got - want).max())
            one = P.mul_mat_small(w, xq=xq, n_tokens=T, bias=_dev(P, bias)).cpu().numpy()
            assert np.allclose(got, one, rtol=1e-5, atol=1e-5)
    # what the single grid does not serve is refused, not approximated
    ws = [P.upload_weight(t, rand_blocks(t, 64, 1024, rng), 1024, 64) for t in (Q4_K, Q4_K, tv)]
    xq = P.quantize_act(_dev(P, rng.normal(0, 1, (40, 1024)).astype(np.float32)), P.vec_dot_act_type(Q4_K))
    with pytest.raises(Exception):
        P.mul_mat_small_mixed(ws, xq, 40)


@pytest.mark.parametrize("K,Ns,T", [(512, (8192, 1024, 1024), 12), (768, (8192, 1024, 1024), 16), (512, (8160, 1020, 1028), 9), (2304, (8192, 1024, 1030), 3)])
def test_last_matrix_of_two_types_in_slices_of_whole_row_groups(P, oracle, K, Ns, T):
    """wv of Q5_K whose share of the workgroups would make slices a row or two longer than 32 (the first matrix gives it some of its own), short rows of one and two steps: the bound of the other
    mixed launches"""
    rng = np.random.default_rng(K + T)
    types = (Q4_K, Q4_K, Q5_K)
    blocks = [rand_blocks(t, N, K, rng) for t, N in zip(types, Ns)]
    x = rng.normal(0, 1, (T, K)).astype(np.float32)
    xq = P.quantize_act(_dev(P, x), P.vec_dot_act_type(Q4_K))
    ys = P.mul_mat_small_mixed([P.upload_weight(t, b, K, N) for t, b, N in zip(types, blocks, Ns)], xq, T)
    for t, b, N, y in zip(types, blocks, Ns, ys):
        assert np.allclose(y.cpu().numpy(), oracle.mul_mat(t, b, K, N, x), rtol=2e-5, atol=2e-5 * np.sqrt(K / 4096)), (t, N)


def test_rms_norm_matches_oracle(P, oracle):
    rng = np.random.default_rng(26)
    for K, eps in ((4096, 1e-5), (8192, 1e-6)):
        x = rng.normal(0, 2, (3, K)).astype(np.float32)
        w = (1 + rng.normal(0, 0.02, K)).astype(np.float32)
        y, yq = P.rms_norm(_dev(P, x), _dev(P, w), eps, want_f32=True, want_q8=True)
        want = oracle.rms_norm(x, w, eps)
        got = y.cpu().numpy()
        # f64 sum of f32 squares in a different order: the f32 mean is the same except on rare rounding
        # boundaries -> allow 1 ulp
        ulp = np.abs(got.view(np.int32).astype(np.int64) - want.view(np.int32).astype(np.int64)).max()
        assert ulp <= 1, ulp
        blocks = P.act_to_ggml_blocks(yq, Q8_K, K, 3).reshape(3, -1)
        for r in range(3):
            assert np.array_equal(blocks[r], oracle.quantize_row_q8_K(got[r]))
        y2 = P.rms_norm(_dev(P, x), None, eps).cpu().numpy()
        assert np.abs(y2.view(np.int32).astype(np.int64) - oracle.rms_norm(x, None, eps).view(np.int32).astype(np.int64)).max() <= 1


@pytest.mark.parametrize("K", [4352, 5120, 8192])
def test_rms_norm_rows_of_two_workgroups(P, K):
    """Rows of 17 .. 32 blocks, two workgroups each up to 128 of them and one beyond: the same bits, f32 and Q8_K."""
    rng = np.random.default_rng(K)
    x, w = _dev(P, rng.normal(0, 2, (129, K)).astype(np.float32)), _dev(P, (1 + rng.normal(0, 0.02, K)).astype(np.float32))
    y, yq = P.rms_norm(x, w, 1e-5, want_q8=True)
    for rows in (1, 128):
        a, aq = P.rms_norm(x[:rows], w, 1e-5, want_q8=True)
        assert P.torch.equal(a, y[:rows]) and P.torch.equal(aq, yq[:aq.numel()]), rows


@pytest.mark.parametrize("K", [4096, 4352, 8192, 8448])
def test_rms_norm_in_place(P, K):
    """y_f32 == x: the same bits as into memory of its own, for rows that two workgroups take otherwise and for their neighbours"""
    import ctypes as C
    from prima_cpp_amd import lib as L
    rng = np.random.default_rng(K)
    f = L.declare("pm355_rms_norm", C.c_int, [C.c_void_p] * 4 + [C.c_int64, C.c_int64, C.c_float, C.c_void_p])
    for rows in (1, 8, 128):
        x, w = _dev(P, rng.normal(0, 2, (rows, K)).astype(np.float32)), _dev(P, (1 + rng.normal(0, 0.02, K)).astype(np.float32))
        want, want_q = P.rms_norm(x, w, 1e-5, want_q8=True)
        q = P.torch.empty_like(want_q)
        L.check(f(L.ptr(x), L.ptr(w), L.ptr(x), L.ptr(q), K, rows, 1e-5, L.stream_ptr()), "rms_norm")
        assert P.torch.equal(x, want) and P.torch.equal(q, want_q), rows


def test_gemv_full_size_linearity(P):
    """BASELINE-size property test (no oracle at this size): W.(a) + W.(b) == W.(a+b) is NOT exact after
    activation quantization, so instead check y(W, x) against dequantize-free structure: scaling x by 2
    (exact in fp) must scale y by exactly 2, and permuting rows of W permutes y."""
    torch = P.torch
    rng = np.random.default_rng(27)
    K, N = 8192, 8192
    blocks = rand_blocks(Q4_K, N, K, rng)
    w = P.upload_weight(Q4_K, blocks, K, N)
    x = torch.from_numpy(rng.normal(0, 1, (1, K)).astype(np.float32)).cuda()
    y1 = P.mul_mat_vec(w, x=x)
    y2 = P.mul_mat_vec(w, x=2 * x)
    assert torch.equal(y2, 2 * y1)
    perm = torch.from_numpy(rng.permutation(N)).cuda()
    wp = P.QWeight(Q4_K, K, N, w.data.view(N, -1)[perm].contiguous().view(-1))
    assert torch.equal(P.mul_mat_vec(wp, x=x), y1[:, perm])
    assert torch.isfinite(y1).all()


def _f16bits(P, a):
    return P.torch.from_numpy(np.ascontiguousarray(a).view(np.int16)).cuda()


@pytest.mark.parametrize("mode", [0, 2])
@pytest.mark.parametrize("with_ff", [False, True])
def test_rope_kv_store_vs_oracle(P, oracle, mode, with_ff):
    torch = P.torch
    rng = np.random.default_rng(41)
    T, H, Hkv, dh, n_ctx, pos0 = 3, 8, 2, 128, 64, 37
    q = rng.normal(0, 1, (T, H * dh)).astype(np.float32)
    k = rng.normal(0, 1, (T, Hkv * dh)).astype(np.float32)
    v = rng.normal(0, 1, (T, Hkv * dh)).astype(np.float32)
    ff = (1 + rng.uniform(0, 7, dh // 2)).astype(np.float32) if with_ff else None
    kc = torch.zeros(n_ctx * Hkv * dh, dtype=torch.int16, device="cuda")
    vc = torch.zeros(n_ctx * Hkv * dh, dtype=torch.int16, device="cuda")
    qr, kr = P.rope_kv_store(_dev(P, q), _dev(P, k), _dev(P, v), kc, vc, pos0, H, Hkv, dh, n_ctx,
                             freq_factors=None if ff is None else _dev(P, ff), mode=mode, freq_base=500000.0)
    pos = np.arange(pos0, pos0 + T, dtype=np.int32)
    q_ref = oracle.rope(q.reshape(T, H, dh), pos, freq_factors=ff, mode=mode, freq_base=500000.0).reshape(T, -1)
    k_ref = oracle.rope(k.reshape(T, Hkv, dh), pos, freq_factors=ff, mode=mode, freq_base=500000.0).reshape(T, -1)
    # identical f32 op sequence except device cosf/sinf (<= 2 ulp): |err| <= 4 ulp of the operand magnitude
    for got, want, src in ((qr.cpu().numpy(), q_ref, q), (kr.cpu().numpy(), k_ref, k)):
        assert np.abs(got - want).max() <= 1e-6 * np.abs(src).max() * 4
    # KV cache contents: K rows = f16(rope(k)) at positions pos0.., V transposed = f16(v); everything else zero
    kc_h = kc.cpu().numpy().view(np.uint16).reshape(n_ctx, Hkv * dh)
    vc_h = vc.cpu().numpy().view(np.uint16).reshape(Hkv * dh, n_ctx)
    assert np.array_equal(kc_h[pos0:pos0 + T], kr.cpu().numpy().astype(np.float16).view(np.uint16))
    assert np.array_equal(vc_h[:, pos0:pos0 + T], v.T.astype(np.float16).view(np.uint16))
    assert not kc_h[:pos0].any() and not kc_h[pos0 + T:].any() and not vc_h[:, :pos0].any() and not vc_h[:, pos0 + T:].any()


@pytest.mark.parametrize("T,H,Hkv,dh,n_dims,mode,ff", [(256, 8, 2, 128, 128, 0, True), (257, 3, 1, 64, 64, 2, False), (300, 5, 5, 96, 64, 0, False), (319, 4, 2, 256, 128, 2, True)])
def test_rope_kv_store_of_a_prompt_equals_small_batches(P, T, H, Hkv, dh, n_dims, mode, ff):
    """256 tokens and more take a workgroup per token and turned tiles of V: the same bits as batches of fewer, and nothing written beside them"""
    torch = P.torch
    g = torch.Generator(device="cuda").manual_seed(T)
    q, k, v = (torch.randn(T, n * dh, generator=g, device="cuda") for n in (H, Hkv, Hkv))
    f = 1 + torch.rand(dh // 2, generator=g, device="cuda") if ff else None
    kw = dict(freq_factors=f, mode=mode, freq_base=500000.0, n_dims=n_dims)
    n_ctx, pos0 = 384, 37
    one, many = ([torch.zeros(n_ctx * Hkv * dh, dtype=torch.int16, device="cuda") for _ in range(2)] for _ in range(2))
    got = P.rope_kv_store(q, k, v, *one, pos0, H, Hkv, dh, n_ctx, **kw)
    parts = [P.rope_kv_store(q[i:i + 160], k[i:i + 160], v[i:i + 160], *many, pos0 + i, H, Hkv, dh, n_ctx, **kw) for i in range(0, T, 160)]
    assert all(torch.equal(a, torch.cat(b)) for a, b in zip(got, zip(*parts)))
    assert all(torch.equal(a, b) for a, b in zip(one, many))


@pytest.mark.parametrize("n_past,T", [(0, 1), (5, 1), (63, 1), (200, 3), (0, 4)])
def test_attn_decode_vs_oracle(P, oracle, n_past, T):
    """Same rounding points as the reference (q and p rounded to F16, F16 K/V): compare with an exact numpy
    restatement of llm_build_kqv in float64 on the SAME f16-rounded inputs."""
    torch = P.torch
    rng = np.random.default_rng(42)
    H, Hkv, dh, n_ctx = 8, 2, 128, 256
    n_kv = n_past + T
    q = rng.normal(0, 1, (T, H, dh)).astype(np.float32)
    K = rng.normal(0, 1, (n_ctx, Hkv, dh)).astype(np.float16)
    V = rng.normal(0, 1, (Hkv, dh, n_ctx)).astype(np.float16)
    K[n_kv:] = 0; V[:, :, n_kv:] = 0
    out = P.attn_decode(_dev(P, q.reshape(T, -1)), _f16bits(P, K), _f16bits(P, V), n_past, H, Hkv, dh, n_ctx,
                        1.0 / np.sqrt(dh)).cpu().numpy().reshape(T, H, dh)
    qh = q.astype(np.float16).astype(np.float64)
    for t in range(T):
        nk = n_past + t + 1
        for h in range(H):
            hk = h // (H // Hkv)
            s = (K[:nk, hk].astype(np.float64) @ qh[t, h]).astype(np.float32) * np.float32(1.0 / np.sqrt(dh))
            e = np.exp((s - s.max()).astype(np.float32)).astype(np.float32)
            p = (e * np.float32(1.0 / e.astype(np.float64).sum())).astype(np.float16).astype(np.float64)
            want = V[hk, :, :nk].astype(np.float64) @ p
            assert np.abs(out[t, h] - want).max() <= 2e-3 * np.abs(want).max() + 1e-4, (t, h)


@pytest.mark.parametrize("dh", [64, 128])
@pytest.mark.parametrize("n_past,T", [(0, 1), (0, 16), (0, 37), (5, 128), (40, 200), (96, 160)])
def test_attn_prefill_mfma_vs_exact(P, oracle, n_past, T, dh):
    """MFMA prefill attention: same rounding points as the reference (q, p -> F16; F16 K/V; f32 accumulate), compared with
    the float64 restatement of llm_build_kqv on the same f16-rounded inputs AND with the per-token kernel."""
    torch = P.torch
    rng = np.random.default_rng(43)
    H, Hkv, n_ctx = 8, 2, 256
    n_kv = n_past + T
    q = rng.normal(0, 1, (T, H, dh)).astype(np.float32)
    K = rng.normal(0, 1, (n_ctx, Hkv, dh)).astype(np.float16)
    V = rng.normal(0, 1, (Hkv, dh, n_ctx)).astype(np.float16)
    K[n_kv:] = 0; V[:, :, n_kv:] = 0
    args = (_dev(P, q.reshape(T, -1)), _f16bits(P, K), _f16bits(P, V), n_past, H, Hkv, dh, n_ctx, 1.0 / np.sqrt(dh))
    out = P.attn_prefill(*args).cpu().numpy().reshape(T, H, dh)
    ref = P.attn_decode(*args).cpu().numpy().reshape(T, H, dh)
    assert np.abs(out - ref).max() <= 2e-3 * np.abs(ref).max()
    qh = q.astype(np.float16).astype(np.float64)
    for t in sorted({0, T // 2, T - 1}):
        nk = n_past + t + 1
        for h in range(H):
            hk = h // (H // Hkv)
            s = (K[:nk, hk].astype(np.float64) @ qh[t, h]).astype(np.float32) * np.float32(1.0 / np.sqrt(dh))
            e = np.exp((s - s.max()).astype(np.float32)).astype(np.float32)
            p = (e * np.float32(1.0 / e.astype(np.float64).sum())).astype(np.float16).astype(np.float64)
            want = V[hk, :, :nk].astype(np.float64) @ p
            assert np.abs(out[t, h] - want).max() <= 2e-3 * np.abs(want).max() + 1e-4, (t, h)


@pytest.mark.parametrize("H,Hkv,n,rowmajor", [(65538, 32769, 36, False), (65537, 65537, 5, False), (131074, 65537, 40, True), (70000, 7, 300, False)])
def test_cached_attention_of_more_heads_than_16_bits(P, H, Hkv, n, rowmajor):
    """the bits of the same heads in calls of fewer"""
    torch, dh, n_ctx, R = P.torch, 64, 320 if n > 64 else 64, H // Hkv
    g = torch.Generator(device="cuda").manual_seed(H)
    q = torch.randn((H, dh), generator=g, device="cuda").half().float()
    K = torch.randn((n_ctx, Hkv, dh), generator=g, device="cuda").half()
    V = torch.randn((n_ctx, Hkv, dh) if rowmajor else (Hkv, dh, n_ctx), generator=g, device="cuda").half()
    pos = torch.tensor([n - 1], dtype=torch.int32, device="cuda")
    go = lambda q, K, V, H, Hkv: P.attn_cached(q.contiguous(), K.contiguous(), V.contiguous(), pos, H, Hkv, dh, n_ctx, dh ** -0.5, flags=1 if rowmajor else 0)
    out = go(q, K, V, H, Hkv)
    c = Hkv // 3
    for a, b in ((0, c), (c, 2 * c), (2 * c, Hkv)):
        assert (b - a) * R <= 65535
        want = go(q[a * R:b * R], K[:, a:b], V[:, a:b] if rowmajor else V[a:b], (b - a) * R, b - a)
        assert torch.equal(out[a * R:b * R], want), (a, b)


@pytest.mark.parametrize("H,Hkv,dh,T,past,mask", [
    (8, 2, 128, 1, 0, None), (8, 2, 64, 31, 1, None), (6, 3, 128, 33, 95, None), (8, 8, 64, 65, 127, None), (8, 1, 128, 130, 30, None),      # 64 queries per workgroup
    (64, 8, 128, 500, 12, None), (256, 32, 64, 128, 1, None),                                                                           # 128
    (128, 8, 64, 1000, 23, None), (128, 8, 128, 1021, 0, None),                                                                          # 256
    (8, 2, 128, 40, 60, "f32"), (8, 2, 64, 40, 60, "f16"), (64, 8, 128, 500, 12, "f16"), (128, 8, 64, 1000, 24, "f32")])
def test_attn_prefill_tiles_against_float64(P, H, Hkv, dh, T, past, mask):
    """Every tile choice of the one-pass kernel (64 / 128 / 256 queries per workgroup), tokens and keys around the tile edges, caches that end on half a stage, both mask types.
    Bound: every probability is rounded to F16 once (2^-11 of itself at most), so an output is off by 2^-11 sum p |v|; a tenth of it again for the f32 scores and sums."""
    import ctypes as C
    from prima_cpp_amd import lib as L
    torch = P.torch
    n = past + T
    n_ctx = -(-n // 32) * 32
    g = torch.Generator(device="cuda").manual_seed(n + dh)
    q = torch.randn((T, H, dh), generator=g, device="cuda") * 2
    K = torch.randn((n_ctx, Hkv, dh), generator=g, device="cuda").half()
    V = torch.randn((Hkv, dh, n_ctx), generator=g, device="cuda").half()
    sc = 1.0 / np.sqrt(dh)
    seen = torch.arange(n, device="cuda")[None] <= torch.arange(T, device="cuda")[:, None] + past
    if mask is None:
        out = P.attn_prefill(q.view(T, -1), K, V, past, H, Hkv, dh, n_ctx, sc).view(T, H, dh)
    else:                                                  # cells at random, the query's own always; n_kv a multiple of 4 as the graphs have it
        seen &= torch.rand((T, n), generator=g, device="cuda") < 0.7
        seen[torch.arange(T), torch.arange(T) + past] = True
        n_kv = -(-n // 4) * 4
        m = torch.full((T, n_kv), -np.inf, device="cuda", dtype=torch.float32 if mask == "f32" else torch.float16)
        m[:, :n][seen] = 0
        out = torch.empty((T, H, dh), device="cuda")
        f = L.declare("pm355_attn_prefill_masked_ex", C.c_int, [C.c_void_p] * 4 + [C.c_int64, C.c_void_p] + [C.c_int] * 6 + [C.c_float, C.c_int, C.c_void_p])
        L.check(f(L.ptr(q), L.ptr(K), L.ptr(V), L.ptr(m), n_kv, L.ptr(out), T, H, Hkv, dh, n_ctx, n_kv, float(sc), 0 if mask == "f32" else 2, L.stream_ptr()), "masked")
    for h in range(0, H, max(1, H // 8)):
        k, v = K[:n, h * Hkv // H].double(), V[h * Hkv // H, :, :n].double()
        p = ((q[:, h].half().double() @ k.T) * sc).masked_fill(~seen, -np.inf).softmax(-1)
        off = (out[:, h].double() - p @ v.T).abs()
        bound = 1.1 * 2.0 ** -11 * (p @ v.abs().T) + 1e-6
        assert bool((off <= bound).all()), (h, float((off / bound).max()))


@pytest.mark.parametrize("H,Hkv,T,past,mask", [(40, 8, 400, 33, None), (64, 8, 800, 5, None), (48, 8, 400, 101, "f32"), (96, 8, 200, 0, "f16")])
def test_attn_prefill_of_64_wide_heads_two_workgroups_to_a_cu(P, H, Hkv, T, past, mask):
    """more workgroups than CUs: the form whose waves request for themselves, 64 and 128 queries (256: 128 heads x 1000 above)"""
    test_attn_prefill_tiles_against_float64(P, H, Hkv, 64, T, past, mask)


def _masked_attention(P, q, K, V, m, n_kv, H, Hkv, dh, n_ctx, sc):
    import ctypes as C
    from prima_cpp_amd import lib as L
    out = P.torch.empty((q.shape[0], H, dh), device="cuda")
    f = L.declare("pm355_attn_prefill_masked_ex", C.c_int, [C.c_void_p] * 4 + [C.c_int64, C.c_void_p] + [C.c_int] * 6 + [C.c_float, C.c_int, C.c_void_p])
    L.check(f(L.ptr(q), L.ptr(K), L.ptr(V), L.ptr(m), m.shape[1], L.ptr(out), q.shape[0], H, Hkv, dh, n_ctx, n_kv, float(sc), 0 if m.dtype == P.torch.float32 else 2, L.stream_ptr()), "masked")
    return out


@pytest.mark.parametrize("junk", [float("nan"), float("inf")])
@pytest.mark.parametrize("H,Hkv,dh,T,past,n_kv", [
    (8, 2, 128, 40, 3, None), (8, 2, 64, 70, 30, None), (64, 8, 128, 512, 33, None), (128, 8, 64, 1000, 29, None), (128, 8, 128, 1021, 0, None),
    (8, 2, 128, 40, 0, 60), (8, 2, 64, 33, 0, 96), (64, 8, 128, 512, 32, 544), (64, 8, 64, 512, 32, 548), (128, 8, 128, 1000, 0, 1012)])
def test_attn_prefill_does_not_look_behind_the_attended_cells(P, H, Hkv, dh, T, past, n_kv, junk):
    """Cells behind the last attended one - of the causal form, and of n_kv with a mask - may hold anything: the same bits as with zeros there. Every tile, counts that end inside a stage of
    keys, inside 32 and inside 8 of them"""
    torch = P.torch
    n = n_kv or past + T
    n_ctx = -(-n // 32) * 32 + 64
    g = torch.Generator(device="cuda").manual_seed(n + dh)
    q = torch.randn((T, H * dh), generator=g, device="cuda")
    outs = []
    for fill in (0.0, junk):
        g.manual_seed(n)
        K = torch.randn((n_ctx, Hkv, dh), generator=g, device="cuda").half()
        V = torch.randn((Hkv, dh, n_ctx), generator=g, device="cuda").half()
        K[n:], V[:, :, n:] = fill, fill
        if n_kv is None:
            outs.append(P.attn_prefill(q, K, V, past, H, Hkv, dh, n_ctx, dh ** -0.5))
            continue
        hidden = torch.arange(n_kv, device="cuda")[None] > torch.arange(T, device="cuda")[:, None] + past
        for dt in (torch.float32, torch.float16):
            outs.append(_masked_attention(P, q, K, V, torch.zeros((T, n_kv), device="cuda", dtype=dt).masked_fill_(hidden, -np.inf), n_kv, H, Hkv, dh, n_ctx, dh ** -0.5))
    assert all(bool(o.isfinite().all()) for o in outs)
    assert all(torch.equal(o, w) for o, w in zip(outs[len(outs) // 2:], outs))


@pytest.mark.parametrize("off", [1, 4])
@pytest.mark.parametrize("H,Hkv,dh,T,past,mask", [(8, 2, 128, 40, 60, False), (8, 4, 64, 70, 130, False), (8, 2, 64, 33, 0, True), (8, 2, 128, 130, 0, True),
                                                    (48, 8, 64, 350, 20, False), (48, 8, 64, 350, 0, True)])
def test_attn_prefill_of_caches_that_do_not_start_on_16_bytes(P, H, Hkv, dh, T, past, mask, off):
    """views that begin 2 or 8 bytes into a buffer: the same bits as caches that start on 16"""
    torch = P.torch
    n = past + T
    n_ctx = -(-n // 32) * 32
    g = torch.Generator(device="cuda").manual_seed(n)
    q = torch.randn((T, H * dh), generator=g, device="cuda")
    K, V = (torch.randn(n_ctx * Hkv * dh, generator=g, device="cuda").half() for _ in range(2))
    outs = []
    for o in (0, off):
        k, v = (torch.cat([torch.zeros(o, device="cuda").half(), x])[o:] for x in (K, V))
        assert k.data_ptr() % 16 == 2 * o
        if not mask:
            outs.append(P.attn_prefill(q, k, v, past, H, Hkv, dh, n_ctx, dh ** -0.5))
            continue
        n_kv = -(-n // 4) * 4
        hidden = torch.arange(n_kv, device="cuda")[None] > torch.arange(T, device="cuda")[:, None]
        outs.append(_masked_attention(P, q, k, v, torch.zeros((T, n_kv), device="cuda").masked_fill_(hidden, -np.inf), n_kv, H, Hkv, dh, n_ctx, dh ** -0.5))
    assert bool(outs[0].isfinite().all()) and torch.equal(*outs)


@pytest.mark.parametrize("scale", [-0.09, 0.0])
@pytest.mark.parametrize("H,Hkv,dh,T,past", [(8, 2, 128, 40, 60), (64, 8, 64, 300, 12)])
def test_attn_prefill_scales_that_are_not_positive(P, H, Hkv, dh, T, past, scale):
    """hidden cells stay hidden whatever the sign of the scale; the bound of test_attn_prefill_tiles_against_float64"""
    torch = P.torch
    n = past + T
    n_ctx = -(-n // 32) * 32
    g = torch.Generator(device="cuda").manual_seed(n)
    q = torch.randn((T, H, dh), generator=g, device="cuda")
    K = torch.randn((n_ctx, Hkv, dh), generator=g, device="cuda").half()
    V = torch.randn((Hkv, dh, n_ctx), generator=g, device="cuda").half()
    out = P.attn_prefill(q.view(T, -1), K, V, past, H, Hkv, dh, n_ctx, scale).view(T, H, dh)
    hidden = torch.arange(n, device="cuda")[None] > torch.arange(T, device="cuda")[:, None] + past
    for h in range(H):
        k, v = K[:n, h * Hkv // H].double(), V[h * Hkv // H, :, :n].double()
        p = ((q[:, h].half().double() @ k.T) * scale).masked_fill(hidden, -np.inf).softmax(-1)
        assert bool(((out[:, h].double() - p @ v.T).abs() <= 1.1 * 2.0 ** -11 * (p @ v.abs().T) + 1e-6).all()), h


@pytest.mark.parametrize("H,Hkv,dh,T,n_kv", [(8, 2, 128, 40, 100), (64, 8, 128, 500, 512), (128, 8, 64, 1000, 1024)])
@pytest.mark.parametrize("lowest", [float(np.finfo(np.float32).min), -1e32, float(np.finfo(np.float16).min)])
def test_attn_prefill_masks_of_the_lowest_value(P, H, Hkv, dh, T, n_kv, lowest):
    """Masks that hide with the lowest finite value of their type: cells beside visible ones weigh nothing, and a row of which every cell is hidden that way attends all of them like the sum of
    score and mask says (the f32 sums are all the same number where the mask's step is larger than the scores; the F16 one leaves steps of 2^-8, so 2^-9 of every weight more in the bound)"""
    torch = P.torch
    f16 = lowest > -1e5
    g = torch.Generator(device="cuda").manual_seed(n_kv)
    q = torch.randn((T, H, dh), generator=g, device="cuda")
    K = torch.randn((n_kv + 28, Hkv, dh), generator=g, device="cuda").half()[:-(-n_kv // 32) * 32].contiguous()
    n_ctx = K.shape[0]
    V = torch.randn((Hkv, dh, n_ctx), generator=g, device="cuda").half()
    m = torch.zeros((T, n_kv), device="cuda").masked_fill_(torch.rand((T, n_kv), generator=g, device="cuda") < 0.3, lowest)
    m[::3] = lowest
    m = m.half() if f16 else m
    sc = dh ** -0.5
    out = _masked_attention(P, q.view(T, -1), K, V, m, n_kv, H, Hkv, dh, n_ctx, sc)
    for h in range(0, H, max(1, H // 8)):
        k, v = K[:n_kv, h * Hkv // H].double(), V[h * Hkv // H, :, :n_kv].double()
        s = ((q[:, h].half().double() @ k.T) * sc + m.double()).float() if not f16 else (q[:, h].half().double() @ k.T) * sc + m.double()
        p = s.double().softmax(-1)
        bound = (1.1 * 2.0 ** -11 + (2.0 * 2.0 ** -9 if f16 else 0.0)) * (p @ v.abs().T) + 1e-6
        off = (out[:, h].double() - p @ v.T).abs()
        assert bool((off <= bound).all()), (h, float((off / bound).nan_to_num(1e9).max()))


@pytest.mark.parametrize("dh", [64, 128])
@pytest.mark.parametrize("n_past", [0, 5, 255, 256, 700, 1023])
def test_attn_decode_split_equals_single_workgroup_kernel(P, n_past, dh):
    """Long-context path (keys split over workgroups, attn_split.hip) against the per-head kernel: same rounding points,
    only the summation order differs."""
    rng = np.random.default_rng(44)
    H, Hkv, n_ctx = 16, 2, 1024
    n_kv = n_past + 1
    q = rng.normal(0, 1, (1, H, dh)).astype(np.float32)
    K = rng.normal(0, 1, (n_ctx, Hkv, dh)).astype(np.float16)
    V = rng.normal(0, 1, (Hkv, dh, n_ctx)).astype(np.float16)
    K[n_kv:] = 0; V[:, :, n_kv:] = 0
    args = (_dev(P, q.reshape(1, -1)), _f16bits(P, K), _f16bits(P, V), n_past, H, Hkv, dh, n_ctx, 1.0 / np.sqrt(dh))
    ref = P.attn_decode(*args).cpu().numpy()
    out = P.attn_decode_split(*args).cpu().numpy()
    # p is rounded to F16 in both kernels; a sum of exponentials assembled per chunk can move 1/sum by an ulp and with it a
    # few p values by one F16 ulp (2^-11 relative): bound = a handful of such flips
    assert np.abs(out - ref).max() <= 2e-4 * np.abs(ref).max() + 1e-6


def test_argmax_first_maximum(P):
    torch = P.torch
    x = torch.randn(128256, device="cuda")
    x[777] = 50.0; x[90000] = 50.0
    assert int(P.argmax(x).item()) == 777
    x[3] = 60.0
    assert int(P.argmax(x).item()) == 3


@pytest.mark.parametrize("t", QUANT_TYPES)
def test_get_rows_bitexact(P, oracle, t):
    torch = P.torch
    rng = np.random.default_rng(43)
    K, N = 768, 50
    blocks = rand_blocks(t, N, K, rng, scale=1.0)
    w = P.upload_weight(t, blocks, K, N)
    toks = np.array([0, 49, 7, 7, 23], dtype=np.int32)
    got = P.get_rows(w, _dev(P, toks)).cpu().numpy()
    rs = row_size(t, K)
    for i, tk in enumerate(toks):
        want = oracle.dequantize_row(t, blocks[tk * rs:(tk + 1) * rs], K)
        assert np.array_equal(got[i].view(np.uint32), want.view(np.uint32)), (t, i)


@pytest.mark.parametrize("mode,dh", [(0, 128), (2, 128), (0, 64)])
@pytest.mark.parametrize("n_past", [0, 1, 7, 8, 9, 63, 300])
def test_attn_rope_fused_equals_two_kernel_path(P, mode, dh, n_past):
    """The fused single-token kernel must agree with rope_kv_store + attn_decode (same rounding points) and must
    leave the caches in exactly the same state."""
    torch = P.torch
    rng = np.random.default_rng(44)
    H, Hkv, n_ctx = 8, 2, 512
    K0 = rng.normal(0, 1, (n_ctx, Hkv * dh)).astype(np.float16)
    V0 = rng.normal(0, 1, (Hkv * dh, n_ctx)).astype(np.float16)
    K0[n_past:] = 0; V0[:, n_past:] = 0
    q = rng.normal(0, 1, (1, H * dh)).astype(np.float32)
    k = rng.normal(0, 1, (1, Hkv * dh)).astype(np.float32)
    v = rng.normal(0, 1, (1, Hkv * dh)).astype(np.float32)
    ff = (1 + rng.uniform(0, 7, dh // 2)).astype(np.float32)
    kw = dict(freq_factors=_dev(P, ff), mode=mode, freq_base=500000.0)
    kc1, vc1 = _f16bits(P, K0), _f16bits(P, V0)
    qr, _ = P.rope_kv_store(_dev(P, q), _dev(P, k), _dev(P, v), kc1, vc1, n_past, H, Hkv, dh, n_ctx, **kw)
    want = P.attn_decode(qr, kc1, vc1, n_past, H, Hkv, dh, n_ctx, 1.0 / np.sqrt(dh))
    kc2, vc2 = _f16bits(P, K0), _f16bits(P, V0)
    got = P.attn_rope_fused(_dev(P, q), _dev(P, k), _dev(P, v), kc2, vc2, n_past, H, Hkv, dh, n_ctx, 1.0 / np.sqrt(dh), **kw)
    assert torch.equal(kc1, kc2) and torch.equal(vc1, vc2)
    w, g = want.cpu().numpy(), got.cpu().numpy()
    assert np.abs(w - g).max() <= 2e-6 * max(1.0, np.abs(w).max())      # summation order only


@pytest.mark.parametrize("t", QUANT_TYPES)
@pytest.mark.parametrize("K", [256, 4096, 8192, 14336, 28672])
@pytest.mark.parametrize("norm", [False, True])
def test_fused_prologue_equals_separate_kernels_bitexact(P, t, K, norm):
    """f32 -> (rms_norm) -> quantize inside the GEMV prologue must give EXACTLY what the stand-alone rms_norm /
    quantize kernels + pre-quantized GEMV give (same integers, same float order)."""
    torch = P.torch
    rng = np.random.default_rng(51)
    N = 33
    w = P.upload_weight(t, rand_blocks(t, N, K, rng), K, N)
    x = torch.from_numpy(rng.normal(0, 1.5, (1, K)).astype(np.float32)).cuda()
    x[0, 3] = 7.5; x[0, 5] = -7.5                    # tie on |max| inside the first block
    nw = torch.from_numpy((1 + rng.normal(0, 0.05, K)).astype(np.float32)).cuda() if norm else None
    resid = torch.from_numpy(rng.normal(0, 1, N).astype(np.float32)).cuda()
    xn = P.rms_norm(x, nw, 1e-5) if norm else x
    want = P.mul_mat_vec(w, x=xn, resid=resid.view(1, -1))[0]
    got = P.mul_mat_vec_fused([w], x, norm_w=nw, eps=1e-5, resids=[resid])[0]
    assert torch.equal(got, want), (got - want).abs().max()


@pytest.mark.experiments
@pytest.mark.parametrize("t", [Q4_K, Q6_K, Q8_0])
@pytest.mark.parametrize("K_in,E", [(4096, 4096), (28672, 8192), (1024, 768)])
def test_producer_side_sum_of_squares_gives_the_same_q8_K_blocks(P, oracle, t, K_in, E):
    """Round 5: the wo / ffn_down launch leaves per-workgroup f64 partials of sum (f32 x^2) of the row it writes (+ residual); the next launch's
    rms_norm prologue adds them instead of reducing the row (ggml_compute_forward_rms_norm_f32, ggml.c:11975-11980). Acceptance: the consumer's
    outputs - i.e. its Q8_K / Q8_0 activation blocks and everything after them - are bit-identical to the plain form, and the partials add up to
    the f64 sum of the f32-rounded squares."""
    torch = P.torch
    rng = np.random.default_rng(505 + K_in + E)
    wp = P.upload_weight(Q4_K, rand_blocks(Q4_K, E, K_in, rng), K_in, E)                 # producer: E rows (wo / ffn_down), + residual
    a = torch.from_numpy(rng.normal(0, 1.0, (1, K_in)).astype(np.float32)).cuda()
    resid = torch.from_numpy(rng.normal(0, 2.0, E).astype(np.float32)).cuda()
    (y_ss,), ss = P.mul_mat_vec_fused_ss([wp], a, resids=[resid], want_sumsq=True)
    y_plain = P.mul_mat_vec_fused([wp], a, resids=[resid])[0]
    assert torch.equal(y_ss, y_plain)                                                       # the producer's output itself is untouched
    y64 = (y_ss.cpu().numpy().astype(np.float32) ** 2).astype(np.float32).astype(np.float64)   # f32-rounded squares, then widened
    assert abs(float(ss.sum().cpu()) - y64.sum()) <= 1e-12 * y64.sum()
    # per-workgroup slices: workgroup b owns rows [E b / G, E (b + 1) / G)
    G = ss.numel()
    for b in (0, G // 2, G - 1):
        r0, r1 = E * b // G, E * (b + 1) // G
        assert abs(float(ss[b].cpu()) - y64[r0:r1].sum()) <= 1e-12 * max(1.0, y64[r0:r1].sum())
    # consumer: rms_norm(y) * w -> quantize -> mat-vec, with and without the partials
    Nc = 70
    wc = P.upload_weight(t, rand_blocks(t, Nc, E, rng), E, Nc)
    nw = torch.from_numpy((1 + rng.normal(0, 0.05, E)).astype(np.float32)).cuda()
    want = P.mul_mat_vec_fused([wc], y_ss.view(1, -1), norm_w=nw, eps=1e-5)[0]
    got = P.mul_mat_vec_fused_ss([wc], y_ss.view(1, -1), norm_w=nw, eps=1e-5, sumsq_in=ss)[0]
    assert torch.equal(got, want), (got - want).abs().max()
    # and a pair launch (ffn_gate | ffn_up) as consumer is covered by the engine test (PM355_SS=0 vs default: identical logits)


def test_fused_qkv_mixed_types_one_launch(P, oracle):
    """wq/wk (Q4_K) + wv (Q6_K or Q5_K) in one launch == three separate mat-vecs, and == the oracle's mul_mat."""
    torch = P.torch
    rng = np.random.default_rng(52)
    K = 4096
    for tv in (Q6_K, Q5_K, Q4_K):
        blocks = [rand_blocks(Q4_K, 96, K, rng), rand_blocks(Q4_K, 40, K, rng), rand_blocks(tv, 40, K, rng)]
        ws = [P.upload_weight(Q4_K, blocks[0], K, 96), P.upload_weight(Q4_K, blocks[1], K, 40), P.upload_weight(tv, blocks[2], K, 40)]
        x = rng.normal(0, 1, (1, K)).astype(np.float32)
        nw = (1 + rng.normal(0, 0.05, K)).astype(np.float32)
        bias = [torch.from_numpy(rng.normal(0, 1, w.N).astype(np.float32)).cuda() for w in ws]
        ys = P.mul_mat_vec_fused(ws, _dev(P, x), norm_w=_dev(P, nw), eps=1e-6, biases=bias)
        xn = oracle.rms_norm(x, nw, 1e-6)
        for w, b, y, bl in zip(ws, bias, ys, blocks):
            sep = P.mul_mat_vec_fused([w], _dev(P, x), norm_w=_dev(P, nw), eps=1e-6, biases=[b])[0]
            assert torch.equal(y, sep)
            want = oracle.mul_mat(w.type, bl, K, w.N, xn)[0] + b.cpu().numpy()
            assert np.allclose(y.cpu().numpy(), want, rtol=2e-5, atol=2e-5)


@pytest.mark.parametrize("t", QUANT_TYPES)
@pytest.mark.parametrize("K,N,T", [(256, 132, 17), (1024, 256, 128), (768, 64, 200), (2048, 516, 300), (1536, 260, 129), (6144, 64, 96), (8192, 260, 33), (4096, 516, 64)])
def test_mfma_prefill_gemm_vs_oracle(P, oracle, t, K, N, T):
    """MFMA batched GEMM (F16 tiles, f32 accumulate, activations not re-quantized) against the reference arithmetic
    (activations quantized to Q8_K/Q8_0): the reference's own backend tolerance is NMSE <= 5e-4
    (tests/test-backend-ops.cpp:1660); also against an exact f64 product of the dequantized weights."""
    rng = np.random.default_rng(71)
    if t == Q8_0 and K == 1536:
        K = 1152                                           # 4.5 super-blocks of 256: Q8_0 rows may end on half of one (Qwen2.5-72B's ffn_down, K = 29568)
    blocks = rand_blocks(t, N, K, rng, scale=1.0)
    w = P.upload_weight(t, blocks, K, N)
    x = rng.normal(0, 1, (T, K)).astype(np.float32)
    bias = rng.normal(0, 1, N).astype(np.float32)
    resid = rng.normal(0, 1, (T, N)).astype(np.float32)
    got = P.mul_mat_mfma(w, _dev(P, x), bias=_dev(P, bias), resid=_dev(P, resid)).cpu().numpy()
    rs = row_size(t, K)
    Wf = np.stack([oracle.dequantize_row(t, blocks[r * rs:(r + 1) * rs], K) for r in range(N)]).astype(np.float64)
    exact = x.astype(np.float64) @ Wf.T + bias + resid
    nm_exact = ((got - exact) ** 2).sum() / (exact ** 2).sum()
    assert nm_exact < 1e-6, nm_exact                       # f16 rounding of operands only
    ref = oracle.mul_mat(t, blocks, K, N, x) + bias + resid
    nm_ref = ((got - ref) ** 2).sum() / (ref ** 2).sum()
    assert nm_ref < 5e-4, nm_ref


@pytest.mark.parametrize("t", [Q4_K, Q6_K])
def test_prompt_gemm_tail_tiles_split_along_k(P, oracle, t):
    """A launch of full rounds of workgroups + a short tail (17 row tiles x 16 token tiles: 32 whole-tile slots per XCD, then 16 slots on one XCD): only the
    tail's tiles are split along K (two slices each, slabs summed in slice order by the last arriver) - against the exact f64 product of the dequantized
    weights, whole tiles and split tiles separately, and bit-identical between two launches."""
    torch = P.torch
    rng = np.random.default_rng(91 + t)
    K, N, T = 2048, 4352, 4096
    blocks = rand_blocks(t, N, K, rng, scale=1.0)
    w = P.upload_weight(t, blocks, K, N)
    x = rng.normal(0, 1, (T, K)).astype(np.float32)
    bias = rng.normal(0, 1, N).astype(np.float32)
    xd, bd = _dev(P, x), _dev(P, bias)
    got = P.mul_mat_mfma(w, xd, bias=bd)
    again = P.mul_mat_mfma(w, xd, bias=bd)
    assert torch.equal(got, again)
    rs = row_size(t, K)
    Wf = np.stack([oracle.dequantize_row(t, blocks[r * rs:(r + 1) * rs], K) for r in range(N)]).astype(np.float64)
    exact = x.astype(np.float64) @ Wf.T + bias
    g = got.cpu().numpy()
    for lo, hi in ((0, 4096), (4096, N)):             # whole tiles | the split tail (row tile 16 = XCD 0's third)
        nm = ((g[:, lo:hi] - exact[:, lo:hi]) ** 2).sum() / (exact[:, lo:hi] ** 2).sum()
        assert nm < 1e-6, (lo, nm)


@pytest.mark.parametrize("types", [(Q4_K, Q4_K, Q6_K), (Q4_K, Q4_K, Q5_K), (Q6_K, Q6_K, Q6_K), (Q5_K, Q6_K), (Q4_K,)])
@pytest.mark.parametrize("T", [77, 300])
def test_prompt_gemm_jobs_one_launch(P, oracle, types, T):
    """wq | wk | wv of a prompt batch as jobs of ONE launch (mmq_pf.hip), each with its own quant type, bias and row count (incl. a ragged last tile):
    every job's output is bit-identical to its own single launch, and equals the f64 product of the dequantized weights to F16 operand rounding."""
    torch = P.torch
    rng = np.random.default_rng(81)
    K = 1024
    Ns = [520, 132, 256][:len(types)]
    blocks = [rand_blocks(t, n, K, rng, scale=1.0) for t, n in zip(types, Ns)]
    ws = [P.upload_weight(t, b, K, n) for t, b, n in zip(types, blocks, Ns)]
    x = rng.normal(0, 1, (T, K)).astype(np.float32)
    biases = [torch.from_numpy(rng.normal(0, 1, n).astype(np.float32)).cuda() for n in Ns]
    xd = _dev(P, x)
    ys = P.mul_mat_mfma_multi(ws, xd, biases=biases)
    for w, t, b, bl, y in zip(ws, types, biases, blocks, ys):
        single = P.mul_mat_mfma(w, xd, bias=b)
        assert torch.equal(y, single)
        rs = row_size(t, K)
        Wf = np.stack([oracle.dequantize_row(t, bl[r * rs:(r + 1) * rs], K) for r in range(w.N)]).astype(np.float64)
        exact = x.astype(np.float64) @ Wf.T + b.cpu().numpy()
        nm = ((y.cpu().numpy() - exact) ** 2).sum() / (exact ** 2).sum()
        assert nm < 1e-6, (t, nm)


# token tiles of 64 and 128 tokens, rows that end inside a 128-row tile and inside a wave's 32, fewer steps of K than are requested ahead, K slices (8 super-blocks and more), for Q8_0 a last
# step that is half a super-block (in a slice and without one); 256 tiles, the last launch of one round, and 258, which the 256-row tiles take, as they take the first counts beyond 128 tokens
# (129 and 257: the general tiles against themselves, other slices of K)
@pytest.mark.parametrize("t", QUANT_TYPES)
@pytest.mark.parametrize("K,N,T", [(512, 132, 33), (768, 260, 64), (512, 4, 65), (4096, 388, 128), (2304, 128, 129), (1024, 1028, 257), (512, 32768, 40), (512, 33024, 40)])
def test_prompt_gemm_tiles_of_128_rows(P, oracle, t, K, N, T):
    """Against the general tiles (the same rows in a launch of more than 256 tiles): the operands are the same F16 numbers, so the results differ by the order of f32 sums only - at most
    2 K 2^-24 sum |w x| between two orders; and against the exact f64 product of the dequantized weights."""
    torch = P.torch
    rng = np.random.default_rng(K + N + T)
    if t == Q8_0:
        K = {512: 640, 768: 896, 2304: 2176, 4096: 4224}.get(K, K)
    uniq = min(N, 516)
    blocks = rand_blocks(t, uniq, K, rng, scale=1.0).reshape(uniq, -1)
    rows = lambda n: np.concatenate([blocks] * (n // uniq + 1))[:n].reshape(-1)
    x = rng.normal(0, 1, (T, K)).astype(np.float32)
    xd = _dev(P, x)
    w, big = P.upload_weight(t, rows(N), K, N), P.upload_weight(t, rows(33024), K, 33024)
    got = P.mul_mat_mfma(w, xd)
    assert torch.equal(got, P.mul_mat_mfma(w, xd))
    Wf = torch.from_numpy(np.stack([oracle.dequantize_row(t, b, K) for b in blocks]).astype(np.float64)).cuda()
    xx = xd.double()
    bound = 2 * K * 2.0 ** -24 * (xx.abs() @ Wf.abs().T)
    assert ((P.mul_mat_mfma(big, xd)[:, :uniq].double() - got[:, :uniq].double()).abs() <= bound).all()
    exact = xx @ Wf.T
    for at in range(0, N - uniq + 1, uniq):
        nm = ((got[:, at:at + uniq].double() - exact) ** 2).sum() / (exact ** 2).sum()
        assert nm < 1e-6, (at, float(nm))


@pytest.mark.parametrize("t", QUANT_TYPES)
@pytest.mark.parametrize("K,N", [(512, 132), (4096, 260), (768, 4100)])
def test_prompt_tiles_of_192_tokens(P, t, K, N):
    """Tiles of 192 tokens beside those of 256, at the first and last counts of either: a token's sums are the same bits in a batch of another tile. Slices of K (4096) and none, rows that end
    inside a wave's, several matrices and pairs."""
    rng = np.random.default_rng(K + N + t)
    if t == Q8_0:
        K += 128
    w = P.upload_weight(t, rand_blocks(t, N, K, rng, scale=1.0), K, N)
    v = P.upload_weight(t, rand_blocks(t, N, K, rng, scale=1.0), K, N)
    x = _dev(P, rng.normal(0, 1, (600, K)).astype(np.float32))
    runs = [lambda a: [P.mul_mat_mfma(w, a)], lambda a: P.mul_mat_mfma_multi([w, v], a), lambda a: [P.mul_mat_mfma_pair(w, v, a)]]
    for run in runs:
        for counts in ((129, 192, 193, 256), (257, 384, 385, 448, 449, 512), (513, 576, 577, 600)):      # (as many tiles of 256 tokens, one split of K; the last one cut to 128 or 192, or whole)
            full = run(x[:counts[-1]].contiguous())
            for T in counts[:-1]:
                for a, b in zip(run(x[:T].contiguous()), full):
                    assert P.torch.equal(a, b[:T]), (T, counts)


@pytest.mark.parametrize("t", QUANT_TYPES)
@pytest.mark.parametrize("K,N", [(512, 132), (4096, 260)])
def test_prompt_tiles_of_96_tokens(P, t, K, N):
    """Tiles of 96 tokens (65..96 tokens; of 8-bit activations also several side by side) beside those of 64 and 128: a token's sums are the same bits in each. Slices of K (4096) and none, rows that
    end inside a wave's, several matrices and pairs; the first and last counts of a tile."""
    rng = np.random.default_rng(K + N + t)
    if t == Q8_0:
        K += 128
    w, w2 = (P.upload_weight(t, rand_blocks(t, N, K, rng), K, N) for _ in range(2))
    x = _dev(P, rng.normal(0, 0.1, (512, K)).astype(np.float32))
    full, multi = P.mul_mat_mfma(w, x[:128]), P.mul_mat_mfma_multi([w, w2], x[:128])
    pair = P.mul_mat_mfma_pair(w, w2, x[:128]) if t != Q8_0 else None
    for T in (64, 65, 95, 96, 97):
        assert P.torch.equal(P.mul_mat_mfma(w, x[:T]), full[:T]), T
        assert all(P.torch.equal(a, b[:T]) for a, b in zip(P.mul_mat_mfma_multi([w, w2], x[:T]), multi)), T
        assert pair is None or P.torch.equal(P.mul_mat_mfma_pair(w, w2, x[:T]), pair[:T]), T
    if t == Q8_0:
        return
    full, pair = P.mul_mat_wide([w], x)[0], P.mul_mat_wide([w, w2], x, pair=True)[0]
    for T in (65, 96, 97, 128, 129, 192, 193, 288, 289, 480, 481):
        assert P.torch.equal(P.mul_mat_wide([w], x[:T])[0], full[:T]), T
        assert P.torch.equal(P.mul_mat_wide([w, w2], x[:T], pair=True)[0], pair[:T]), T


@pytest.mark.parametrize("K", [512, 640, 1664])
def test_prompt_products_of_few_q8_0_rows(P, oracle, K):
    """up to 64 tokens and less than 128 workgroups of 128 rows: the kernel without loaders, the bits of the one with them (129 workgroups; no K split at these K, rows that end on half a
    super-block among them), and the oracle's products of the F16 activations"""
    N, rng = 129 * 128, np.random.default_rng(K)
    b = rand_blocks(Q8_0, N, K, rng)
    x = rng.normal(0, 1, (64, K)).astype(np.float16).astype(np.float32)
    few, many = b.reshape(N, -1), P.upload_weight(Q8_0, b, K, N)
    for T in (33, 64):
        xd = _dev(P, x[:T])
        want = P.mul_mat_mfma(many, xd)
        for n in (4, 132, 1024, 127 * 128):
            got = P.mul_mat_mfma(P.upload_weight(Q8_0, np.ascontiguousarray(few[:n]).reshape(-1), K, n), xd)
            assert P.torch.equal(got, want[:, :n]), (T, n)
    w = np.stack([oracle.dequantize_row(Q8_0, np.ascontiguousarray(r), K) for r in few[:132]]).astype(np.float64)
    y = want[:, :132].cpu().numpy().astype(np.float64)
    exact = x.astype(np.float64) @ w.T
    assert np.linalg.norm(y - exact) < 1e-3 * np.linalg.norm(exact)      # (a weight is rounded to F16 once: 2^-11 at most)


@pytest.mark.parametrize("types", [(Q4_K, Q6_K), (Q4_K, Q5_K), (Q5_K, Q6_K), (Q4_K,), (Q5_K,), (Q6_K,)])
def test_prompt_products_of_four_steps(P, types):
    """K = 512, 97..128 tokens: the kernel without loaders, the bits of the one with them (the first 96 tokens, tiles of 96), one type and two in a launch; one row tile, several, and the most"""
    K, rng = 512, np.random.default_rng(sum(types))
    x = _dev(P, rng.normal(0, 1, (128, K)).astype(np.float32))
    for N in (4, 132, 16384):
        ws = [P.upload_weight(t, rand_blocks(t, N, K, rng), K, N) for t in types]
        run = lambda a: P.mul_mat_mfma_multi(ws, a) if len(ws) > 1 else [P.mul_mat_mfma(ws[0], a)]
        want = run(x[:96].contiguous())
        late = run(x[32:].contiguous())
        for T in (97, 128):
            for a, b, c in zip(run(x[:T].contiguous()), want, late):
                assert P.torch.equal(a[:96], b) and P.torch.equal(a[32:], c[:T - 32]), (N, T)


@pytest.mark.parametrize("t", [Q4_K, Q5_K, Q6_K])
@pytest.mark.parametrize("K,N,T", [(1024, 384, 200), (2048, 132, 64), (512, 256, 257), (8192, 132, 200)])
def test_prompt_gemm_pair_tiles_silu_gate_times_up(P, oracle, t, K, N, T):
    """ffn_gate | ffn_up as one launch of pair tiles: silu(gate) * up formed inside the workgroup == the two separate launches followed by the product
    (the reference's MUL_MAT, MUL_MAT, SILU, MUL: llm_build_ffn, src/llama.cpp:9804)."""
    torch = P.torch
    rng = np.random.default_rng(83)
    wg = P.upload_weight(t, rand_blocks(t, N, K, rng, scale=1.0), K, N)
    wu = P.upload_weight(t, rand_blocks(t, N, K, rng, scale=1.0), K, N)
    x = _dev(P, rng.normal(0, 1, (T, K)).astype(np.float32))
    got = P.mul_mat_mfma_pair(wg, wu, x)
    g, u = P.mul_mat_mfma(wg, x), P.mul_mat_mfma(wu, x)
    want = (g.double() / (1.0 + torch.exp(-g.double()))) * u.double()
    err = (got.double() - want).abs().max().item()
    assert err <= 2e-6 * want.abs().max().item(), err


@pytest.mark.parametrize("mode", [0, 2])
@pytest.mark.parametrize("tv", [Q6_K, Q5_K, Q4_K])
@pytest.mark.parametrize("dh,H,Hkv", [(128, 8, 4), (64, 16, 8)])
def test_qkv_epilogue_and_cached_attention_equal_the_fused_attention_path(P, oracle, tv, dh, H, Hkv, mode):
    """Round-3 decode form - RoPE + F16 KV store in the EPILOGUE of the wq | wk | wv launch (per-token cos / sin table, wk / wv dealt out
    step by step over all waves), attention over cached cells only (one-barrier kernel up to 64 cells, per-head body beyond) - against
    the round-2 form (plain mat-vecs, rope + store inside the fused attention kernel) on a run of tokens that crosses the 64-cell
    boundary; the mat-vec outputs against the oracle's mul_mat. mode 2 = NEOX rope (build_qwen2: pairs (i, i + n_rot / 2); every workgroup's
    slice of wq / wk is two runs of rows n_rot / 2 apart, GemvJob::nx_s)."""
    torch = P.torch
    rng = np.random.default_rng(61)
    if tv != Q4_K and mode == 2 and dh == 64:
        pytest.skip("one attn_v type per NEOX shape is enough")
    K, n_ctx = 1024, 128
    Nq, Nkv = H * dh, Hkv * dh
    assert Nq % 512 == 0 and Nkv % 512 == 0
    blocks = [rand_blocks(Q4_K, Nq, K, rng), rand_blocks(Q4_K, Nkv, K, rng), rand_blocks(tv, Nkv, K, rng)]
    ws = [P.upload_weight(Q4_K, blocks[0], K, Nq), P.upload_weight(Q4_K, blocks[1], K, Nkv), P.upload_weight(tv, blocks[2], K, Nkv)]
    nw = _dev(P, (1 + rng.normal(0, 0.05, K)).astype(np.float32))
    bias = [_dev(P, rng.normal(0, 0.3, n).astype(np.float32)) for n in (Nq, Nkv, Nkv)]
    ff = _dev(P, (1 + rng.uniform(0, 7, dh // 2)).astype(np.float32))
    kcA = torch.zeros(n_ctx * Nkv, dtype=torch.int16, device="cuda"); vcA = torch.zeros_like(kcA)
    kcB = torch.zeros_like(kcA); vcB = torch.zeros_like(kcA)
    kcC = torch.zeros_like(kcA); vcC = torch.zeros_like(kcA)          # ggml-graph mode of the same launches (cell / cells attended + mask)
    mask0 = torch.zeros(n_ctx, dtype=torch.float32, device="cuda")
    scale = 1.0 / np.sqrt(dh)
    worst = 0.0
    for pos in list(range(0, 6)) + [31, 32, 62, 63, 64, 65, 90]:
        x = rng.normal(0, 1, (1, K)).astype(np.float32)
        xd = _dev(P, x)
        qA, kA, vA = P.mul_mat_vec_fused(ws, xd, norm_w=nw, eps=1e-5, biases=bias)
        outA = P.attn_rope_fused(qA, kA, vA, kcA, vcA, pos, H, Hkv, dh, n_ctx, scale, freq_factors=ff, freq_base=500000.0, mode=mode)
        pd = torch.tensor([pos], dtype=torch.int32, device="cuda")
        tab = P.rope_table(pd, dh, freq_factors=ff, freq_base=500000.0, mode=mode)
        qB = P.mul_mat_vec_qkv(ws, xd, tab, pd, kcB, vcB, Hkv, dh, n_ctx, norm_w=nw, eps=1e-5, biases=bias, neox=mode == 2)
        outB = P.attn_cached(qB, kcB, vcB, pd, H, Hkv, dh, n_ctx, scale)
        dyn = torch.tensor([pos, pos + 1], dtype=torch.int32, device="cuda")
        qC = P.mul_mat_vec_qkv(ws, xd, tab, None, kcC, vcC, Hkv, dh, n_ctx, norm_w=nw, eps=1e-5, biases=bias, cell_nkv=dyn, neox=mode == 2)
        outC = P.attn_cached(qC, kcC, vcC, None, H, Hkv, dh, n_ctx, scale, cell_nkv=dyn, mask=mask0, max_keys=n_ctx)
        torch.cuda.synchronize()
        assert torch.equal(qC, qB) and torch.equal(outC, outB) and torch.equal(kcC, kcB) and torch.equal(vcC, vcB), pos
        # the K row / V column of this cell: the same F16 values up to the summation order of the split wk / wv rows (<= 1 F16 ulp, rarely)
        a = kcA.cpu().numpy().view(np.float16).astype(np.float32).reshape(n_ctx, Nkv)[pos]
        b = kcB.cpu().numpy().view(np.float16).astype(np.float32).reshape(n_ctx, Nkv)[pos]
        assert np.abs(a - b).max() <= 2e-3 * max(1.0, np.abs(a).max()) and (a != b).mean() < 0.02, (pos, np.abs(a - b).max(), (a != b).mean())
        va = vcA.cpu().numpy().view(np.float16).astype(np.float32).reshape(Nkv, n_ctx)[:, pos]
        vb = vcB.cpu().numpy().view(np.float16).astype(np.float32).reshape(Nkv, n_ctx)[:, pos]
        assert np.abs(va - vb).max() <= 2e-3 * max(1.0, np.abs(va).max()) and (va != vb).mean() < 0.02
        # q: rotated + F16-rounded == F16 rounding of the oracle's rope of the round-2 q
        q_ref = oracle.rope(qA.cpu().numpy().reshape(1, H, dh), np.array([pos], dtype=np.int32), freq_factors=ff.cpu().numpy(), freq_base=500000.0, mode=mode)
        q_ref = q_ref.astype(np.float16).astype(np.float32).reshape(-1)
        qb = qB.cpu().numpy()
        assert np.abs(qb - q_ref).max() <= 2e-3 * max(1.0, np.abs(q_ref).max()) and (qb != q_ref).mean() < 0.02
        # from here on both caches must hold the SAME bytes, or later cells would compare different histories
        kcB.copy_(kcA); vcB.copy_(vcA); kcC.copy_(kcA); vcC.copy_(vcA)
        wa, wb = outA.cpu().numpy(), outB.cpu().numpy()
        worst = max(worst, float(np.abs(wa - wb).max() / max(1.0, np.abs(wa).max())))
        assert np.abs(wa - wb).max() <= 3e-3 * max(1.0, np.abs(wa).max()), (pos, np.abs(wa - wb).max())
        # cells in between: identical random history for both paths
        if pos >= 5:
            nxt = {5: 31, 31: 32, 32: 62, 62: 63, 63: 64, 64: 65, 65: 90}.get(pos)
            if nxt:
                fill_k = rng.normal(0, 1, (nxt - pos - 1, Nkv)).astype(np.float16).view(np.int16)
                fill_v = rng.normal(0, 1, (Nkv, nxt - pos - 1)).astype(np.float16).view(np.int16)
                if fill_k.size:
                    kcA.view(n_ctx, Nkv)[pos + 1:nxt] = torch.from_numpy(fill_k).cuda()
                    vcA.view(Nkv, n_ctx)[:, pos + 1:nxt] = torch.from_numpy(fill_v).cuda()
                    kcB.copy_(kcA); vcB.copy_(vcA); kcC.copy_(kcA); vcC.copy_(vcA)
    print(f"\n[qkv epilogue + cached attention, dh {dh}, attn_v type {tv}] max |d out| / max |out| = {worst:.2e}")
    # and the epilogue's mat-vecs against the oracle (q before rope is not observable: check k / v through the cache at one more cell)
    x = rng.normal(0, 1, (1, K)).astype(np.float32)
    pd = torch.tensor([100], dtype=torch.int32, device="cuda")
    tab = P.rope_table(pd, dh, freq_factors=ff, freq_base=500000.0, mode=mode)
    P.mul_mat_vec_qkv(ws, _dev(P, x), tab, pd, kcB, vcB, Hkv, dh, n_ctx, norm_w=nw, eps=1e-5, biases=bias, neox=mode == 2)
    xn = oracle.rms_norm(x, nw.cpu().numpy(), 1e-5)
    v_ref = oracle.mul_mat(tv, blocks[2], K, Nkv, xn)[0] + bias[2].cpu().numpy()
    v_got = vcB.cpu().numpy().view(np.float16).astype(np.float32).reshape(Nkv, n_ctx)[:, 100]
    assert np.allclose(v_got, v_ref.astype(np.float16).astype(np.float32), rtol=2e-3, atol=2e-3)
    k_ref = oracle.mul_mat(Q4_K, blocks[1], K, Nkv, xn)[0] + bias[1].cpu().numpy()
    k_ref = oracle.rope(k_ref.reshape(1, Hkv, dh), np.array([100], dtype=np.int32), freq_factors=ff.cpu().numpy(), freq_base=500000.0, mode=mode).reshape(-1)
    k_got = kcB.cpu().numpy().view(np.float16).astype(np.float32).reshape(n_ctx, Nkv)[100]
    assert np.allclose(k_got, k_ref.astype(np.float16).astype(np.float32), rtol=2e-3, atol=2e-3)


@pytest.mark.parametrize("dh,H,Hkv", [(128, 8, 1), (128, 8, 2), (64, 8, 4), (64, 4, 4), (64, 16, 1)])
def test_long_context_matrix_core_attention_over_cached_cells(P, dh, H, Hkv):
    """attn_flash_mfma.hip: scores and P.V of a GQA group on v_mfma_f32_16x16x32_f16 with permuted key rows, per-wave online softmax, spans
    merged in the launch - against softmax(K q * scale + mask) V in float64 on the same F16 cache values, over cells-attended that
    exercise: one partial tile, one span, several spans with a ragged tail, the doubled span (> 8k cells), with and without a mask that
    hides cells (-inf), position given as d_pos and as {cell, cells attended}."""
    torch = P.torch
    rng = np.random.default_rng(77 + dh + H)
    n_ctx = 16640
    Nkv = Hkv * dh
    R = H // Hkv
    kc = rng.normal(0, 1, (n_ctx, Nkv)).astype(np.float16)
    vt = rng.normal(0, 1, (Nkv, n_ctx)).astype(np.float16)
    kcd = torch.from_numpy(kc.view(np.int16)).cuda().reshape(-1)
    vcd = torch.from_numpy(vt.view(np.int16)).cuda().reshape(-1)
    scratch = P.attn_split_scratch(H, dh, n_ctx)
    scale = 1.0 / np.sqrt(dh)
    worst = 0.0
    for n_kv, use_mask, dyn_mode in [(1, False, False), (33, False, True), (700, True, True), (2000, False, False), (2049, True, True),
                                     (5000, False, True), (8192, False, False), (16300, True, True)]:
        q = (rng.normal(0, 1, (H, dh)) * 1.5).astype(np.float16).astype(np.float32)      # (the epilogue hands over F16-rounded values)
        qd = torch.from_numpy(q.reshape(1, -1)).cuda()
        mask = None
        mnp = np.zeros(n_kv, dtype=np.float64)
        if use_mask:
            m32 = np.zeros(n_ctx, dtype=np.float32)
            hide = rng.random(n_kv) < 0.3
            hide[n_kv - 1] = False
            m32[:n_kv][hide] = -np.inf
            m32[n_kv:] = -np.inf
            mask = torch.from_numpy(m32).cuda()
            mnp = m32[:n_kv].astype(np.float64)
        cells = 1024
        while cells < n_kv: cells *= 2
        cells = min(cells, n_ctx)
        if dyn_mode:
            dyn = torch.tensor([n_kv - 1, n_kv], dtype=torch.int32, device="cuda")
            out = P.attn_cached(qd, kcd, vcd, None, H, Hkv, dh, n_ctx, scale, cell_nkv=dyn, mask=mask, max_keys=cells, scratch=scratch)
        else:
            pd = torch.tensor([n_kv - 1], dtype=torch.int32, device="cuda")
            out = P.attn_cached(qd, kcd, vcd, pd, H, Hkv, dh, n_ctx, scale, mask=mask, max_keys=0, scratch=scratch)
        torch.cuda.synchronize()
        got = out.cpu().numpy().reshape(H, dh)
        for h in range(H):
            g = h // R
            Kh = kc[:n_kv, g * dh:(g + 1) * dh].astype(np.float64)
            Vh = vt[g * dh:(g + 1) * dh, :n_kv].astype(np.float64)
            s = Kh @ q[h].astype(np.float64) * scale + mnp
            pr = np.exp(s - s.max()); pr /= pr.sum()
            ref = Vh @ pr
            err = np.abs(got[h] - ref).max() / max(1e-3, np.abs(ref).max())
            worst = max(worst, float(err))
            assert err < 2e-3, (n_kv, h, err)
    print(f"\n[matrix-core long-context attention dh {dh} H {H} Hkv {Hkv}] worst max|d| / max|ref| = {worst:.2e}")


def _attn_refs(kc, vt, q, n_kv, H, Hkv, dh, scale):
    """float64 attention over F16 cache values, and the reference graph's rounding points (MUL_MAT(k, q) -> SOFT_MAX_EXT -> MUL_MAT(v, kq), ggml.c:12445-12473:
    the NORMALISED probabilities are rounded to F16 as src1 of the V^T.p product, accumulation in f32): [H][dh] each."""
    R = H // Hkv
    ref64 = np.empty((H, dh)); ref16 = np.empty((H, dh))
    for g in range(Hkv):
        Kh = kc[:n_kv, g * dh:(g + 1) * dh].astype(np.float32)
        Vh = vt[g * dh:(g + 1) * dh, :n_kv].astype(np.float32)
        for h in range(g * R, (g + 1) * R):
            s = (Kh.astype(np.float64) @ q[h].astype(np.float64)) * scale
            pr = np.exp(s - s.max()); pr /= pr.sum()
            ref64[h] = Vh.astype(np.float64) @ pr
            s32 = (Kh @ q[h]).astype(np.float32) * np.float32(scale)
            e32 = np.exp(s32 - s32.max()).astype(np.float32)
            p16 = (e32 / np.float32(e32.astype(np.float64).sum())).astype(np.float16).astype(np.float32)
            ref16[h] = (Vh.astype(np.float64) @ p16.astype(np.float64))
    return ref64, ref16


@pytest.mark.parametrize("dh,H,Hkv", [(128, 64, 8), (64, 12, 4)])
@pytest.mark.parametrize("n_kv", [700, 8192])
def test_long_context_attention_on_a_row_major_v_cache(P, n_kv, dh, H, Hkv):
    """--flash-attn layout (V cache [cell][n_head_kv * head_dim], F16 mask; llm_build_kv, src/llama.cpp:9705, :10075-10095) on the matrix-core kernel: the wave's
    V rows go through its LDS image and come back as operands through the transposing LDS read. Same cache VALUES as the transposed layout -> the two layouts'
    results must be bitwise equal; and both against float64. A sparse F16 mask (-inf on every 7th cell) checks the masked path on the way."""
    torch = P.torch
    ATTN_V_ROWMAJOR, ATTN_MASK_F16 = 1, 2                                    # include/prima_mi355.h: PM355_ATTN_V_ROWMAJOR, PM355_ATTN_MASK_F16
    rng = np.random.default_rng(7000 + n_kv + dh)
    n_ctx = 8192 + 256
    Nkv = Hkv * dh
    kc = rng.normal(0, 1, (n_ctx, Nkv)).astype(np.float16)
    vt = rng.normal(0, 1, (Nkv, n_ctx)).astype(np.float16)
    vrow = np.ascontiguousarray(vt.T)                                        # [cell][Hkv * dh]
    kcd = torch.from_numpy(kc.view(np.int16)).cuda().reshape(-1)
    vtd = torch.from_numpy(vt.view(np.int16)).cuda().reshape(-1)
    vrd = torch.from_numpy(vrow.view(np.int16)).cuda().reshape(-1)
    scale = 1.0 / np.sqrt(dh)
    q = (rng.normal(0, 1, (H, dh)) * 1.5).astype(np.float16).astype(np.float32)
    qd = torch.from_numpy(q.reshape(1, -1)).cuda()
    pd = torch.tensor([n_kv - 1], dtype=torch.int32, device="cuda")
    mnp = np.zeros(n_ctx, dtype=np.float16); mnp[::7] = -np.inf
    md = torch.from_numpy(mnp.view(np.int16)).cuda()
    cells = 1024
    while cells < n_kv: cells *= 2
    cells = min(cells, n_ctx)
    for mask, flags in ((None, 0), (md, ATTN_MASK_F16)):
        s_t, s_r = P.attn_split_scratch(H, dh, n_ctx), P.attn_split_scratch(H, dh, n_ctx)
        out_t = P.attn_cached(qd, kcd, vtd, pd, H, Hkv, dh, n_ctx, scale, mask=mask, max_keys=cells, flags=flags, scratch=s_t).cpu().numpy().reshape(H, dh)
        out_r = P.attn_cached(qd, kcd, vrd, pd, H, Hkv, dh, n_ctx, scale, mask=mask, max_keys=cells, flags=flags | ATTN_V_ROWMAJOR, scratch=s_r).cpu().numpy().reshape(H, dh)
        assert np.isfinite(out_r).all()
        assert np.array_equal(out_t, out_r), np.abs(out_t - out_r).max()
        R = H // Hkv
        for h in range(H):
            g = h // R
            Kh = kc[:n_kv, g * dh:(g + 1) * dh].astype(np.float64)
            Vh = vt[g * dh:(g + 1) * dh, :n_kv].astype(np.float64)
            sc = Kh @ q[h].astype(np.float64) * scale + (mnp[:n_kv].astype(np.float64) if mask is not None else 0.0)
            pr = np.exp(sc - sc.max()); pr /= pr.sum()
            ref = Vh @ pr
            assert np.abs(out_r[h] - ref).max() / max(1e-3, np.abs(ref).max()) < 2e-3, (n_kv, h)


@pytest.mark.parametrize("n_kv", [8192, 32700])
def test_long_context_attention_at_the_70b_head_shape(P, n_kv):
    """The shape the long-context numbers are quoted on - 64 query heads, 8 KV heads, head_dim 128, 8k and 32.7k cells (grid = 8 x 32 spans: every
    resident slot of the chip) - against float64 AND against the reference graph's own rounding points (p rounded to F16 AFTER the normalisation;
    the kernel rounds exp(s - m) before it, attn_flash_mfma.hip): both differences are measured and bounded."""
    torch = P.torch
    H, Hkv, dh = 64, 8, 128
    rng = np.random.default_rng(1000 + n_kv)
    n_ctx = 32768 + 256
    Nkv = Hkv * dh
    kc = rng.normal(0, 1, (n_ctx, Nkv)).astype(np.float16)
    vt = rng.normal(0, 1, (Nkv, n_ctx)).astype(np.float16)
    kcd = torch.from_numpy(kc.view(np.int16)).cuda().reshape(-1)
    vcd = torch.from_numpy(vt.view(np.int16)).cuda().reshape(-1)
    scratch = P.attn_split_scratch(H, dh, n_ctx)
    scale = 1.0 / np.sqrt(dh)
    q = (rng.normal(0, 1, (H, dh)) * 1.5).astype(np.float16).astype(np.float32)
    qd = torch.from_numpy(q.reshape(1, -1)).cuda()
    pd = torch.tensor([n_kv - 1], dtype=torch.int32, device="cuda")
    cells = 1024
    while cells < n_kv: cells *= 2
    cells = min(cells, n_ctx)
    outs = [P.attn_cached(qd, kcd, vcd, pd, H, Hkv, dh, n_ctx, scale, max_keys=cells, scratch=scratch).cpu().numpy().reshape(H, dh) for _ in range(3)]
    assert all(np.array_equal(outs[0], o) for o in outs[1:])              # launch to launch: bitwise (fixed merge order)
    got = outs[0]
    ref64, ref16 = _attn_refs(kc, vt, q, n_kv, H, Hkv, dh, scale)
    den = np.maximum(1e-3, np.abs(ref64).max(axis=1))
    e64 = (np.abs(got - ref64).max(axis=1) / den).max()
    e16 = (np.abs(got - ref16).max(axis=1) / den).max()
    r1664 = (np.abs(ref16 - ref64).max(axis=1) / den).max()
    print(f"\n[matrix-core attention, H 64 / Hkv 8 / dh 128, {n_kv} cells] max|d| / max|ref|: kernel vs float64 {e64:.2e}, kernel vs F16-rounded-p reference {e16:.2e}, "
          f"that reference vs float64 {r1664:.2e}")
    assert np.isfinite(got).all()
    assert e64 < 2e-3 and e16 < 2e-3 + r1664


@pytest.mark.parametrize("H, Hkv, cells", [
    (2, 1, [1]), (8, 4, [1, 63, 64, 2, 33]), (8, 8, [64, 65, 128, 127, 1]), (16, 2, [129, 256, 255, 8, 64, 200]), (32, 8, list(range(9, 41))),                  # rows: each its own sequence
    (2, 1, (0, 1)), (4, 2, (0, 32)), (8, 2, (63, 3)), (32, 8, (100, 17)), (16, 2, (480, 32)),                                                             # (first position, consecutive tokens)
])
def test_attention_leaves_the_blocks_its_quantizer_would(P, H, Hkv, cells):
    """A small batch's attention that writes wo's 8-bit activations itself, against the attention stored as f32 rows and quantized by a launch of its own: every byte of the rows and of the tables."""
    torch = P.torch
    f = P.L.load_probe().pm355_probe_attn_blocks
    f.restype, f.argtypes = C.c_int, [C.c_void_p] * 5 + [C.c_int64] + [C.c_int] * 3 + [C.c_float] + [C.c_int] * 3 + [C.c_void_p] * 8
    rows = isinstance(cells, list)
    T, dh, n_ctx = (len(cells) if rows else cells[1]), 128, (256 if rows else 512)
    K, n_seq = H * dh, (T if rows else 1)
    rng = np.random.default_rng(1000 * H + T)
    half = lambda a: torch.from_numpy(a.astype(np.float16).view(np.int16)).cuda()
    kc, vc = (half(rng.normal(0, 1, n_seq * n_ctx * Hkv * dh)) for _ in range(2))
    q = torch.from_numpy((rng.normal(0, 1.5, (T, K))).astype(np.float16).astype(np.float32)).cuda()
    pos = torch.tensor([c - 1 for c in cells] if rows else [cells[0] + t for t in range(T)], dtype=torch.int32, device="cuda")
    seq = torch.tensor(list(range(T))[::-1] if rows else [0] * T, dtype=torch.int32, device="cuda")
    row = K + K // 256 * 4 + K // 16 * 2
    out = [[torch.full((n,), 0x5a, dtype=torch.uint8, device="cuda") for n in (T * row + 64, K // 256 * 1152, K // 256 * 8192)] for _ in range(2)]
    y32 = torch.zeros((T, K), dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()
    args = [q, kc, vc, pos, seq, n_ctx * Hkv * dh, H, Hkv, n_ctx, 1.0 / np.sqrt(dh), int(rows), max(cells) if rows else 0, T, *out[0], y32, *out[1]]
    rc = f(*[a.data_ptr() if isinstance(a, torch.Tensor) else a for a in args], None)
    torch.cuda.synchronize()
    assert rc == 0 and bool(torch.isfinite(y32).all()) and bool((y32 != 0).any(dim=1).all())
    for name, a, b in zip(("rows", "sums", "values"), *out):
        assert bool((b != 0x5a).any()) and bool((a == b).all()), f"{name}: {int((a != b).sum())} of {a.numel()} bytes differ"


def test_long_context_attention_merge_survives_a_starved_chip(P):
    """The in-launch merge of attn_flash_mfma.hip lets the last arrivals of a KV head spin (bounded) for workgroups still behind them. Provoked here:
    a co-running stream-read kernel holds every CU's wave slots while the 8 x 32 attention grid is launched on another stream, so its workgroups
    trickle in as slots free up. Required: the launch ENDS (no hang) and the result is either correct or the fail-loud NaN - never a wrong number."""
    import ctypes as C
    torch = P.torch
    plib = P.L.load_probe()
    plib.pm355_probe_stream_read.restype = C.c_int
    plib.pm355_probe_stream_read.argtypes = [C.c_void_p, C.c_size_t, C.c_int, C.c_int, C.c_void_p, C.c_void_p]
    H, Hkv, dh, n_kv = 64, 8, 128, 16384
    rng = np.random.default_rng(4242)
    n_ctx = 16384 + 256
    Nkv = Hkv * dh
    kc = rng.normal(0, 1, (n_ctx, Nkv)).astype(np.float16)
    vt = rng.normal(0, 1, (Nkv, n_ctx)).astype(np.float16)
    kcd = torch.from_numpy(kc.view(np.int16)).cuda().reshape(-1)
    vcd = torch.from_numpy(vt.view(np.int16)).cuda().reshape(-1)
    scratch = P.attn_split_scratch(H, dh, n_ctx)
    scale = 1.0 / np.sqrt(dh)
    q = (rng.normal(0, 1, (H, dh)) * 1.5).astype(np.float16).astype(np.float32)
    qd = torch.from_numpy(q.reshape(1, -1)).cuda()
    pd = torch.tensor([n_kv - 1], dtype=torch.int32, device="cuda")
    ref64, _ = _attn_refs(kc, vt, q, n_kv, H, Hkv, dh, scale)
    hog_src = torch.empty(1 << 30, dtype=torch.uint8, device="cuda")
    sink = torch.zeros(4, dtype=torch.int32, device="cuda")
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    n_nan = n_ok = 0
    for trial in range(6):
        # two 1024-thread workgroups per CU (every wave slot of the chip), several passes queued back to back on the side stream
        for _ in range(3):
            assert plib.pm355_probe_stream_read(hog_src.data_ptr(), hog_src.numel(), 2, 8, sink.data_ptr(), side.cuda_stream) == 0
        out = P.attn_cached(qd, kcd, vcd, pd, H, Hkv, dh, n_ctx, scale, max_keys=16384, scratch=scratch)
        torch.cuda.synchronize()
        got = out.cpu().numpy().reshape(H, dh)
        if np.isnan(got).any():
            n_nan += 1                                    # fail-loud path: a whole KV head's outputs are NaN
            bad = np.isnan(got).any(axis=1)
            assert all(bad[g * 8:(g + 1) * 8].all() or not bad[g * 8:(g + 1) * 8].any() for g in range(Hkv))
            good = ~bad
        else:
            n_ok += 1
            good = np.ones(H, dtype=bool)
        err = np.abs(got[good] - ref64[good]).max(axis=1) / np.maximum(1e-3, np.abs(ref64[good]).max(axis=1)) if good.any() else np.zeros(1)
        assert err.max() < 2e-3, (trial, err.max())
    print(f"\n[starved merge] {n_ok} launches correct, {n_nan} launches took the fail-loud NaN path; none hung, none wrong")
    # and an undisturbed launch afterwards is clean (the arrival counters are never reset: a timed-out launch must not poison the next)
    out = P.attn_cached(qd, kcd, vcd, pd, H, Hkv, dh, n_ctx, scale, max_keys=16384, scratch=scratch).cpu().numpy().reshape(H, dh)
    assert np.isfinite(out).all() and (np.abs(out - ref64).max(axis=1) / np.maximum(1e-3, np.abs(ref64).max(axis=1))).max() < 2e-3


def _pm_tensor(C, t, type_, ne, nb):
    class PMT(C.Structure):
        _fields_ = [("data", C.c_void_p), ("type", C.c_int32), ("pad_", C.c_int32), ("ne", C.c_int64 * 4), ("nb", C.c_size_t * 4)]
    x = PMT()
    x.data, x.type, x.pad_ = t.data_ptr(), type_, 0
    for i in range(4):
        x.ne[i] = ne[i] if i < len(ne) else 1
        x.nb[i] = nb[i] if i < len(nb) else nb[len(nb) - 1] * (ne[len(nb) - 1] if len(nb) == len(ne) else 1)
    return x


def test_native_q8_0_cache_view_matmul_and_dequantizing_copy(P, oracle):
    """The two node-equivalent ops a `-ctk q8_0` cache needs outside flash attention, on a strided view of native 34-byte blocks shaped like
    llm_build_kqv's k view [head_dim, n_kv, n_head_kv] (row stride = a whole cache row): MUL_MAT(k, q) = quantize_row_q8_0(q) +
    ggml_vec_dot_q8_0_q8_0, against the oracle's mul_mat per head; and CPY -> F32 (K-shift graphs) = dequantize_row_q8_0."""
    import ctypes as C
    torch = P.torch
    lib = P.L.load()
    rng = np.random.default_rng(77)
    dh, Hkv, H, n_kv, n_ctx, T = 128, 2, 4, 40, 64, 3
    Ekv = dh * Hkv
    kf = rng.normal(0, 1, (n_ctx, Ekv)).astype(np.float32)
    blocks = np.concatenate([oracle.quantize_row_q8_0(kf[i]) for i in range(n_ctx)])          # cache rows in native block order
    kc = torch.from_numpy(blocks).cuda()
    row_b, head_b = Ekv // 32 * 34, dh // 32 * 34
    q = rng.normal(0, 1, (H, T, dh)).astype(np.float32)
    qd = torch.from_numpy(q).cuda()
    out = torch.zeros((H, T, n_kv), dtype=torch.float32, device="cuda")
    a = _pm_tensor(C, kc, Q8_0, [dh, n_kv, Hkv, 1], [34, row_b, head_b, n_ctx * row_b])
    b = _pm_tensor(C, qd, 0, [dh, T, H, 1], [4, dh * 4, T * dh * 4, H * T * dh * 4])
    d = _pm_tensor(C, out, 0, [n_kv, T, H, 1], [4, n_kv * 4, T * n_kv * 4, H * T * n_kv * 4])
    lib.pm355_op_mul_mat_f.restype = C.c_int
    lib.pm355_op_mul_mat_f.argtypes = [C.c_void_p] * 4
    assert lib.pm355_op_mul_mat_f(C.addressof(a), C.addressof(b), C.addressof(d), P.stream_ptr()) == 0
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    kb = blocks.reshape(n_ctx, Hkv, head_b)
    for h in range(H):
        hk = h // (H // Hkv)
        w = np.ascontiguousarray(kb[:n_kv, hk]).reshape(-1)
        want = oracle.mul_mat(Q8_0, w, dh, n_kv, q[h])                                           # [T, n_kv]
        assert np.allclose(got[h], want, rtol=1e-5, atol=1e-5), (h, np.abs(got[h] - want).max())
    # dequantizing copy of the view [dh, Hkv, n_ctx] -> contiguous f32
    deq = torch.zeros((n_ctx, Hkv, dh), dtype=torch.float32, device="cuda")
    s = _pm_tensor(C, kc, Q8_0, [dh, Hkv, n_ctx, 1], [34, head_b, row_b, n_ctx * row_b])
    t = _pm_tensor(C, deq, 0, [dh, Hkv, n_ctx, 1], [4, dh * 4, Hkv * dh * 4, n_ctx * Hkv * dh * 4])
    lib.pm355_op_cpy.restype = C.c_int
    lib.pm355_op_cpy.argtypes = [C.c_void_p] * 3
    assert lib.pm355_op_cpy(C.addressof(s), C.addressof(t), P.stream_ptr()) == 0
    torch.cuda.synchronize()
    want = np.stack([oracle.dequantize_row(Q8_0, blocks[i * row_b:(i + 1) * row_b], Ekv) for i in range(n_ctx)]).reshape(n_ctx, Hkv, dh)
    assert np.array_equal(deq.cpu().numpy(), want)


@pytest.mark.experiments
@pytest.mark.parametrize("t", [Q4_K, Q6_K])
@pytest.mark.parametrize("K,N", [(1024, 512), (8192, 8192), (4096, 1024), (5120, 2560)])
def test_engine_matvec_phase_is_bit_identical_to_the_launch(P, t, K, N):
    """Persistent decode engine, one mat-vec phase (+ residual, + producer-side partials) against pm355_mul_mat_vec_fused_ss on the same operands: the same
    row loops (the leading steps of a wave's first rows come out of its LDS prefetch slot instead of registers: same consume() calls in the same order)
    -> the same bits; then a two-phase list (wo-like phase -> rms_norm + ffn_gate | ffn_up pair phase fed through the in-launch seam; the pair is Q4_K,
    the only pair type compiled into the engine)."""
    torch = P.torch
    rng = np.random.default_rng(900 + K + N)
    w = P.upload_weight(t, rand_blocks(t, N, K, rng), K, N)
    x = torch.from_numpy(rng.normal(0, 1.0, (1, K)).astype(np.float32)).cuda()
    resid = torch.from_numpy(rng.normal(0, 2.0, N).astype(np.float32)).cuda()
    (want,), ss_want = P.mul_mat_vec_fused_ss([w], x, resids=[resid], want_sumsq=True)
    e = P.EngineRun()
    (got,), ss = e.matvec([w], x, resids=[resid], want_sumsq=True)
    e.run()
    assert torch.equal(got, want), (got - want).abs().max()
    assert torch.equal(ss[:ss_want.numel()], ss_want)
    if N % 256:
        return
    # two phases: y = W x + resid, then h = silu(G n(y)) * (U n(y)) with the sum of squares handed over inside the launch
    F = 768
    g = P.upload_weight(Q4_K, rand_blocks(Q4_K, F, N, rng), N, F)
    u = P.upload_weight(Q4_K, rand_blocks(Q4_K, F, N, rng), N, F)
    nw = torch.from_numpy((1 + rng.normal(0, 0.05, N)).astype(np.float32)).cuda()
    want_h = P.mul_mat_vec_fused([g], want.view(1, -1), norm_w=nw, eps=1e-5, w2s=[u])[0]
    e = P.EngineRun()
    (y1,), ss1 = e.matvec([w], x, resids=[resid], want_sumsq=True)
    (h,) = e.matvec([g], y1, norm_w=nw, eps=1e-5, w2s=[u], sumsq_in=ss1[:ss_want.numel()])
    e.run()
    assert torch.equal(y1, want)
    assert torch.equal(h, want_h), (h - want_h).abs().max()


@pytest.mark.experiments
@pytest.mark.parametrize("t", [Q4_K, Q6_K])
def test_engine_long_rows_continue_from_the_prefetched_steps(P, oracle, t):
    """ffn_down-sized rows (K = 28672: seven steps per row) do not fit a wave's prefetch slot: the first two or three steps of a wave's first row come out
    of LDS, the per-lane partial sums are handed to the register row loop (Item::run_job's c_start / acc0) - same accumulation chain, same bits as the launch."""
    torch = P.torch
    rng = np.random.default_rng(77)
    K, N = 28672, 8192
    blocks = rand_blocks(t, N, K, rng)
    w = P.upload_weight(t, blocks, K, N)
    x = torch.from_numpy(rng.normal(0, 1.0, (1, K)).astype(np.float32)).cuda()
    resid = torch.from_numpy(rng.normal(0, 2.0, N).astype(np.float32)).cuda()
    want = P.mul_mat_vec_fused([w], x, resids=[resid])[0]
    e = P.EngineRun()
    (got,) = e.matvec([w], x, resids=[resid])
    e.run()
    assert torch.equal(got, want), (got - want).abs().max().item()


@pytest.mark.experiments
@pytest.mark.parametrize("tv", [Q6_K, Q5_K, Q4_K])
@pytest.mark.parametrize("mode", [0, 2])
@pytest.mark.parametrize("n_past", [0, 5, 63, 64, 200])
def test_engine_qkv_and_attention_phases_equal_the_launches(P, mode, n_past, tv):
    """wq | wk | wv + RoPE + KV store, then attention over the cached cells, as two phases of one engine launch (q and the token's cell cross the
    in-launch seam) against pm355_mul_mat_vec_qkv + pm355_attn_cached: same bits in q, in the caches and in the attention output, below and above the
    64-cell short path."""
    torch = P.torch
    rng = np.random.default_rng(31 + n_past + mode)
    E_, H, Hkv, dh, n_ctx = 2048, 16, 4, 128, 256
    ws = [P.upload_weight(Q4_K, rand_blocks(Q4_K, H * dh, E_, rng), E_, H * dh), P.upload_weight(Q4_K, rand_blocks(Q4_K, Hkv * dh, E_, rng), E_, Hkv * dh),
          P.upload_weight(tv, rand_blocks(tv, Hkv * dh, E_, rng), E_, Hkv * dh)]
    x = torch.from_numpy(rng.normal(0, 1.0, (1, E_)).astype(np.float32)).cuda()
    nw = torch.from_numpy((1 + rng.normal(0, 0.05, E_)).astype(np.float32)).cuda()
    pos = torch.tensor([n_past], dtype=torch.int32, device="cuda")
    tab = P.rope_table(pos, dh, mode=mode, freq_base=500000.0)
    kc0 = torch.from_numpy(rng.normal(0, 1, (n_ctx, Hkv * dh)).astype(np.float16)).cuda()
    vc0 = torch.from_numpy(rng.normal(0, 1, (Hkv * dh, n_ctx)).astype(np.float16)).cuda()
    scale = 1.0 / np.sqrt(dh)
    ssx = (x.double() ** 2).float().double().sum().view(1)          # one-partial sum of squares of the input row (f32-rounded squares)
    # launches
    kc1, vc1 = kc0.clone(), vc0.clone()
    q1 = P.mul_mat_vec_qkv(ws, x, tab, pos, kc1, vc1, Hkv, dh, n_ctx, norm_w=nw, eps=1e-5, neox=bool(mode & 2))
    a1 = P.attn_cached(q1, kc1, vc1, pos, H, Hkv, dh, n_ctx, scale)
    # engine
    kc2, vc2 = kc0.clone(), vc0.clone()
    e = P.EngineRun()
    ys = e.matvec(ws, x, norm_w=nw, eps=1e-5, sumsq_in=ssx,
                  qkv=dict(tab=tab, pos=pos, k_cache=kc2, v_cache=vc2, n_head_kv=Hkv, head_dim=dh, n_ctx=n_ctx, neox=bool(mode & 2)))
    a2 = e.attention(ys[0], kc2, vc2, pos, H, Hkv, dh, n_ctx, scale)
    e.run()
    assert torch.equal(ys[0], q1), (ys[0] - q1).abs().max()
    assert torch.equal(kc2, kc1) and torch.equal(vc2, vc1)
    assert torch.equal(a2, a1), (a2 - a1).abs().max()


@pytest.mark.experiments
@pytest.mark.parametrize("shape", [(8192, 64, 8, 128), (4096, 32, 8, 128), (2048, 16, 4, 128), (1024, 16, 8, 64)])
@pytest.mark.parametrize("tv", [Q6_K, Q4_K])
@pytest.mark.parametrize("mode", [0, 2])
def test_attention_in_the_qkv_launch_tail_equals_the_two_launches(P, shape, tv, mode):
    """Round 5: pm355_mul_mat_vec_qkv_attn - the attention over the cached cells computed in the TAIL of the wq | wk | wv launch by
    the last workgroups of each KV-head group (per-group ticket; q and the token's cell are read back through write-through stores / cache-bypassing
    loads) - against pm355_mul_mat_vec_qkv followed by pm355_attn_cached: the same bits in q, in both caches and in the attention output, at the
    Llama-3-70B / 8B head shapes and two small ones, on both sides of the 64-cell short path, the launch repeated on one set of ticket counters
    (they are monotonic across launches), NORM and NEOX rope."""
    torch = P.torch
    E_, H, Hkv, dh = shape
    n_ctx = 1024
    rng = np.random.default_rng(77 + E_ + mode)
    ws = [P.upload_weight(Q4_K, rand_blocks(Q4_K, H * dh, E_, rng), E_, H * dh), P.upload_weight(Q4_K, rand_blocks(Q4_K, Hkv * dh, E_, rng), E_, Hkv * dh),
          P.upload_weight(tv, rand_blocks(tv, Hkv * dh, E_, rng), E_, Hkv * dh)]
    nw = torch.from_numpy((1 + rng.normal(0, 0.05, E_)).astype(np.float32)).cuda()
    kc0 = torch.from_numpy(rng.normal(0, 1, (n_ctx, Hkv * dh)).astype(np.float16)).cuda()
    vc0 = torch.from_numpy(rng.normal(0, 1, (Hkv * dh, n_ctx)).astype(np.float16)).cuda()
    scale = 1.0 / np.sqrt(dh)
    ticket = torch.zeros(Hkv, dtype=torch.int32, device="cuda")
    dog = torch.zeros(1, dtype=torch.int32, device="cuda")
    kc1, vc1, kc2, vc2 = kc0.clone(), vc0.clone(), kc0.clone(), vc0.clone()
    for n_past in (0, 1, 17, 63, 64, 65, 200, 639):
        x = torch.from_numpy(rng.normal(0, 1.0, (1, E_)).astype(np.float32)).cuda()
        pos = torch.tensor([n_past], dtype=torch.int32, device="cuda")
        tab = P.rope_table(pos, dh, mode=mode, freq_base=500000.0)
        q1 = P.mul_mat_vec_qkv(ws, x, tab, pos, kc1, vc1, Hkv, dh, n_ctx, norm_w=nw, eps=1e-5, neox=bool(mode & 2))
        a1 = P.attn_cached(q1, kc1, vc1, pos, H, Hkv, dh, n_ctx, scale, max_keys=648)
        q2, a2 = P.mul_mat_vec_qkv_attn(ws, x, tab, pos, kc2, vc2, H, Hkv, dh, n_ctx, scale, ticket, norm_w=nw, eps=1e-5, neox=bool(mode & 2), max_keys=648, watchdog=dog)
        torch.cuda.synchronize()
        assert int(dog.item()) == 0
        assert torch.equal(q2, q1), (n_past, (q2 - q1).abs().max())
        assert torch.equal(kc2, kc1) and torch.equal(vc2, vc1), n_past
        assert torch.equal(a2, a1), (n_past, (a2 - a1).abs().max())


def _q8_cache(oracle, rng, n_ctx, Ekv):
    f = rng.normal(0, 1, (n_ctx, Ekv)).astype(np.float32)
    blocks = np.concatenate([oracle.quantize_row_q8_0(f[i]) for i in range(n_ctx)])
    deq = np.stack([oracle.dequantize_row(Q8_0, blocks[i * (Ekv // 32 * 34):(i + 1) * (Ekv // 32 * 34)], Ekv) for i in range(n_ctx)])
    return blocks, deq


@pytest.mark.parametrize("kq8,vq8", [(True, True), (True, False), (False, True)])
@pytest.mark.parametrize("shape", [(64, 8, 128), (32, 8, 128), (16, 4, 64)])
@pytest.mark.parametrize("n_kv", [700, 2500, 8200])
def test_long_context_attention_over_q8_0_caches_on_the_matrix_cores(P, oracle, kq8, vq8, shape, n_kv):
    """Round 5: attn_flash_mfma.hip over Q8_0 K and / or V caches (native 34-byte blocks, row-major V: `-fa -ctk q8_0 -ctv q8_0`,
    src/llama.cpp:3531-3560, :10075-10095) - the dequantizing operand fetch (q_i * d rounded to F16 per value) against float64 attention over the
    dequantized cache values (dequantize_row_q8_0 / F16), 2e-3 of max |out| as for the F16 caches (probabilities are rounded to F16 as MFMA
    operands), at the Llama-3-70B / 8B head shapes and a head_dim-64 one, 700 .. 8200 cells."""
    torch = P.torch
    H, Hkv, dh = shape
    Ekv = Hkv * dh
    n_ctx = ((n_kv + 300) // 256) * 256
    rng = np.random.default_rng(n_kv + H + 2 * kq8 + vq8)
    if kq8:
        kb, kd = _q8_cache(oracle, rng, n_ctx, Ekv)
        kc = torch.from_numpy(kb).cuda()
    else:
        kd = rng.normal(0, 1, (n_ctx, Ekv)).astype(np.float16).astype(np.float32)
        kc = torch.from_numpy(kd.astype(np.float16)).cuda()
    if vq8:
        vb, vd = _q8_cache(oracle, rng, n_ctx, Ekv)
        vc = torch.from_numpy(vb).cuda()
    else:
        vd = rng.normal(0, 1, (n_ctx, Ekv)).astype(np.float16).astype(np.float32)
        vc = torch.from_numpy(vd.astype(np.float16)).cuda()
    q = rng.normal(0, 1, (H, dh)).astype(np.float16).astype(np.float32)
    scale = 1.0 / np.sqrt(dh)
    dyn = torch.tensor([n_kv - 1, n_kv], dtype=torch.int32, device="cuda")
    scratch = P.attn_split_scratch(H, dh, n_ctx)
    grid = 1024
    while grid < n_kv:
        grid *= 2
    flags = P.ATTN_V_ROWMAJOR | (P.ATTN_K_Q8_0 if kq8 else 0) | (P.ATTN_V_Q8_0 if vq8 else 0)
    out = P.attn_cached(torch.from_numpy(q.reshape(1, -1)).cuda(), kc, vc, None, H, Hkv, dh, n_ctx, scale, cell_nkv=dyn, max_keys=min(grid, n_ctx), flags=flags, scratch=scratch)
    got = out.cpu().numpy().reshape(H, dh)
    want = np.zeros((H, dh))
    for h in range(H):
        hk = h // (H // Hkv)
        K = kd[:n_kv, hk * dh:(hk + 1) * dh].astype(np.float64)
        V = vd[:n_kv, hk * dh:(hk + 1) * dh].astype(np.float64)
        s = K @ q[h].astype(np.float64) * scale
        p = np.exp(s - s.max())
        want[h] = (p / p.sum()) @ V
    err = np.abs(got - want).max()
    assert err <= 2e-3 * np.abs(want).max(), (err, np.abs(want).max())


@pytest.mark.parametrize("kq8,vq8", [(True, True), (True, False), (False, True)])
@pytest.mark.parametrize("mode", [0, 2])
def test_long_context_q8_0_token_step_matches_the_one_workgroup_per_head_kernel(P, oracle, kq8, vq8, mode):
    """pm355_attn_token with Q8_0 caches beyond the long-context threshold: rope + quantizing KV store (attn_q8.hip q8_token_prep_kernel) + the matrix-core
    kernel over the cached cells, against the one-workgroup-per-head kernel that serves short contexts (attn_q8_token_kernel: the reference's
    block-wise integer K.q, f32 P.V): the same bytes in both caches (quantize_row_q8_0_ref of the rotated k / of v), outputs within the F16-operand
    tier of each other and of float64."""
    torch = P.torch
    H, Hkv, dh, n_kv = 32, 8, 128, 1500
    Ekv, n_ctx = Hkv * dh, 2048
    rng = np.random.default_rng(500 + 2 * kq8 + vq8 + mode)
    def cache(q8):
        if q8:
            b, _ = _q8_cache(oracle, rng, n_ctx, Ekv)
            return torch.from_numpy(b).cuda()
        return torch.from_numpy(rng.normal(0, 1, (n_ctx, Ekv)).astype(np.float16)).cuda()
    kc0, vc0 = cache(kq8), cache(vq8)
    q = torch.from_numpy(rng.normal(0, 1, (1, H * dh)).astype(np.float32)).cuda()
    k = torch.from_numpy(rng.normal(0, 1, (1, Ekv)).astype(np.float32)).cuda()
    v = torch.from_numpy(rng.normal(0, 1, (1, Ekv)).astype(np.float32)).cuda()
    pos = torch.tensor([n_kv - 1], dtype=torch.int32, device="cuda")
    dyn = torch.tensor([n_kv - 1, n_kv], dtype=torch.int32, device="cuda")
    flags = P.ATTN_V_ROWMAJOR | (P.ATTN_K_Q8_0 if kq8 else 0) | (P.ATTN_V_Q8_0 if vq8 else 0)
    scale = 1.0 / np.sqrt(dh)
    kc1, vc1, kc2, vc2 = kc0.clone(), vc0.clone(), kc0.clone(), vc0.clone()
    a1 = P.attn_token(q, k, v, kc1, vc1, pos, dyn, H, Hkv, dh, n_ctx, scale, flags=flags, mode=mode, freq_base=500000.0)
    scratch = P.attn_split_scratch(H, dh, n_ctx)
    a2 = P.attn_token(q, k, v, kc2, vc2, pos, dyn, H, Hkv, dh, n_ctx, scale, flags=flags, mode=mode, freq_base=500000.0, scratch=scratch, max_keys=2048)
    torch.cuda.synchronize()
    assert torch.equal(kc1, kc2) and torch.equal(vc1, vc2)
    d = (a2 - a1).abs().max().item()
    assert d <= 2e-3 * a1.abs().max().item(), (d, a1.abs().max().item())
    nm = float(((a2 - a1).double() ** 2).sum() / (a1.double() ** 2).sum())
    assert nm < 1e-5, nm


def test_small_batch_attention_fallback_is_indifferent_to_the_pre_rounded_query(P):
    """small batches store q F16-rounded (rope + KV store with round_q) for pm355_attn_cached; when that kernel refuses a shape the older
    pm355_attn_decode consumes the same rows. It rounds q to F16 itself (MUL_MAT's src1 conversion, ggml.c:12445-12473), so an already rounded q gives
    the same bits as the raw one - shown here at head_dim 96, a shape attn_cached does not serve."""
    torch = P.torch
    rng = np.random.default_rng(9)
    T, H, Hkv, dh, n_ctx, pos0 = 3, 8, 4, 96, 64, 20
    q = torch.from_numpy(rng.normal(0, 1, (T, H * dh)).astype(np.float32)).cuda()
    kc = torch.from_numpy(rng.normal(0, 1, (n_ctx, Hkv * dh)).astype(np.float16)).cuda().view(torch.int16)
    vc = torch.from_numpy(rng.normal(0, 1, (Hkv * dh, n_ctx)).astype(np.float16)).cuda().view(torch.int16)
    scale = 1.0 / np.sqrt(dh)
    raw = P.attn_decode(q, kc, vc, pos0, H, Hkv, dh, n_ctx, scale)
    rounded = P.attn_decode(q.half().float(), kc, vc, pos0, H, Hkv, dh, n_ctx, scale)
    assert torch.equal(raw, rounded)


@pytest.mark.parametrize("t", [Q4_K, Q5_K, Q6_K, Q8_0])
def test_small_batch_rows_kernel_at_its_edges(P, oracle, t):
    """mmq_rows.hip: one and two super-blocks more than a step of eight pairs holds, odd and even counts, a single pair, blocks of 32 that end inside a pair; rows below, at and above
    the 16 of a row group, one to three groups in one pass and several passes of 64 (activations in LDS where they fit, passes of 48 where they do not); every token count. Against the oracle:
    the same integers, <= K / 256 (Q8_0: K / 32) f32 terms in another order - the bound of the other small-batch products."""
    rng = np.random.default_rng(7100 + t)
    tail = 32 if t == Q8_0 else 256
    for K, N, T in ((512, 1, 8), (512, 15, 1), (768, 16, 2), (2048, 17, 3), (4096, 33, 4), (4096 + tail, 100, 5), (4352, 4096, 7), (4608, 4097, 8), (8192 + tail, 8192 + 31, 6), (1024, 12300, 8), (768, 28700, 3),
                    (8192, 12290, 2), (12288, 16390, 8),
                    (512, 16, 17), (768, 4096, 16), (4096 + tail, 33, 9), (4608, 100, 24), (14336, 4095, 23),      # (up to 24 tokens where a workgroup has one group of rows)
                    (512, 40, 25), (4096 + tail, 4096, 32), (768, 17, 61), (4352, 8191, 17), (512, 4097, 24), (8192 + tail, 8230, 23),      # (Q5_K, Q8_0: up to 32, and 17..24 with two and more)
                    (4096, 4999, 7), (4096, 10243, 8), (8192 + tail, 10243, 3), (8192, 20491, 5), (12288, 20487, 8), (3072, 9001, 2)):      # (two and three groups, 64-row and 48-row passes of the
                                                                                                                                            # types that have them: test_host_launches.py)
        b = rand_blocks(t, N, K, rng)
        x = rng.normal(0, 1, (T, K)).astype(np.float32)
        bias, resid = rng.normal(0, 1, N).astype(np.float32), rng.normal(0, 1, (T, N)).astype(np.float32)
        w = P.upload_weight(t, b, K, N)
        rows = np.unique(np.concatenate([np.arange(min(N, 70)), np.arange(max(N - 70, 0), N), rng.integers(0, N, 150)]))   # (the oracle is a scalar program)
        bytes_per_row = b.size // N
        want = oracle.mul_mat(t, b.reshape(N, bytes_per_row)[rows].copy(), K, len(rows), x)
        tol = dict(rtol=2e-5, atol=2e-5 * np.sqrt(max(K, 4096) / 4096))
        y = P.mul_mat_small(w, x=_dev(P, x)).cpu().numpy()
        assert np.isfinite(y).all(), (K, N, T)
        assert np.allclose(y[:, rows], want, **tol), (K, N, T, np.abs(y[:, rows] - want).max())
        xq = P.quantize_act(_dev(P, x), P.vec_dot_act_type(t))
        y2 = P.mul_mat_small(w, xq=xq, n_tokens=T, bias=_dev(P, bias), resid=_dev(P, resid)).cpu().numpy()
        assert np.array_equal(y2, (y + bias[None]) + resid), (K, N, T)
        # a token's sums do not depend on the tokens beside it, where those do not turn the pass over to the other kernel (pm_mmq_rows_takes)
        if T <= 8 or N <= 4096 and (t == Q5_K or t == Q8_0 and T > 16 and K >= 1024 or t in (Q4_K, Q6_K) and T <= 24 and K >= 3072):
            one = P.mul_mat_small(w, x=_dev(P, x[T - 1:])).cpu().numpy()
            assert np.array_equal(one[0], y[T - 1]), (K, N, T)


@pytest.mark.parametrize("t", [Q4_K, Q6_K, Q8_0])
def test_small_batch_activations_staged_behind_weight_requests(P, oracle, t):
    """mmq_rows.hip with activations in LDS: 32 super-blocks (all asked for in front of the weights), one more and 36 (the rest by loops behind them), a single pair; the bound of the test above."""
    rng = np.random.default_rng(7200 + t)
    tail = 32 if t == Q8_0 else 256
    for K, N, T in ((8192, 16390, 8), (8192 + tail, 16401, 5), (9216, 33000, 7), (1536 + tail, 50001, 1)):
        b = rand_blocks(t, N, K, rng)
        x = rng.normal(0, 1, (T, K)).astype(np.float32)
        w = P.upload_weight(t, b, K, N)
        rows = np.unique(np.concatenate([np.arange(70), np.arange(N - 70, N), rng.integers(0, N, 100)]))
        want = oracle.mul_mat(t, b.reshape(N, b.size // N)[rows].copy(), K, len(rows), x)
        y = P.mul_mat_small(w, x=_dev(P, x)).cpu().numpy()
        assert np.isfinite(y).all(), (K, N, T)
        assert np.allclose(y[:, rows], want, rtol=2e-5, atol=2e-5 * np.sqrt(max(K, 4096) / 4096)), (K, N, T, np.abs(y[:, rows] - want).max())


@pytest.mark.parametrize("rows,K", [(65, 4096), (256, 8192), (257, 4096), (256, 12288), (2, 256)])
def test_rms_norm_of_many_rows(P, oracle, rows, K):
    """16 waves per row up to 256 rows, 4 beyond; rows that fit the registers of either form and rows that do not. The bound of the test of few rows: one unit in the last place (the f64 sum's
    order), and the quantized rows are those of the values returned."""
    rng = np.random.default_rng(rows + K)
    x, w = rng.normal(0, 2, (rows, K)).astype(np.float32), (1 + rng.normal(0, 0.02, K)).astype(np.float32)
    y, yq = P.rms_norm(_dev(P, x), _dev(P, w), 1e-5, want_f32=True, want_q8=True)
    got = y.cpu().numpy()
    at = [0, rows // 2, rows - 1]
    want = oracle.rms_norm(x[at], w, 1e-5)
    assert np.abs(got[at].view(np.int32).astype(np.int64) - want.view(np.int32).astype(np.int64)).max() <= 1
    assert np.array_equal(P.act_to_ggml_blocks(yq, Q8_K, K, rows), P.act_to_ggml_blocks(P.quantize_act(y, Q8_K), Q8_K, K, rows))


SHORT_ATTENTION = [(dh, n_ctx, n_kv, mask) for dh, n_ctx, n_kvs in ((64, 256, (1, 36, 64, 65, 100, 128, 129, 204, 256)), (128, 320, (1, 36, 64, 65, 100, 128, 129, 204, 256)), (256, 64, (7, 64)),
                                                                     (128, 32, (9, 32)), (64, 96, (64, 80)), (128, 200, (128, 199)), (256, 256, (65, 200)))
                   for n_kv in n_kvs for mask in ([None] if n_kv not in (36, 204) else [None, "f32", "f16"])]


def short_attention_inputs(dh, n_ctx, n_kv, mask):
    """q (as the wq launch leaves it: F16 values), caches of two KV heads, three query heads each, random behind the attended cells too, a mask that hides every fifth cell"""
    rng = np.random.default_rng(dh * 1000003 + n_ctx * 1009 + n_kv)
    H, Hkv = 6, 2
    q = rng.normal(0, 1, (H, dh)).astype(np.float16).astype(np.float32)
    kc, vc = rng.normal(0, 1, (n_ctx, Hkv, dh)).astype(np.float16), rng.normal(0, 1, (Hkv, dh, n_ctx)).astype(np.float16)
    m = None if mask is None else np.where(np.arange(n_ctx) % 5 == 3, -np.inf, rng.normal(0, 1, n_ctx).astype(np.float16)).astype(np.float32 if mask == "f32" else np.float16)
    return q, kc, vc, m


@pytest.mark.parametrize("dh,n_ctx,n_kv,mask", SHORT_ATTENTION)
def test_single_token_attention_over_few_cells_keeps_its_sums(P, dh, n_ctx, n_kv, mask):
    """Up to 256 cells: every rounding of a decoded token is what it is with a lane per key and a lane per dimension, whatever the loads look like - the 8-bit roundings behind it carry one other
    bit to 3 % of an eight-layer model's logits. Bit for bit against outputs recorded with that form (golden/attn_short.npz: edges of the 64 / 128 / 256-cell forms, caches too small for a form,
    masks), and against float64: probabilities rounded to F16 (2^-11 of each) and f32 sums of at most 256 terms."""
    torch = P.torch
    q, kc, vc, m = short_attention_inputs(dh, n_ctx, n_kv, mask)
    H, Hkv = q.shape[0], kc.shape[1]
    scale = dh ** -0.5
    dyn = torch.tensor([n_kv - 1, n_kv], dtype=torch.int32, device="cuda")
    run = lambda: P.attn_cached(_dev(P, q.reshape(1, -1)), _dev(P, kc.view(np.int16)), _dev(P, vc.view(np.int16)), None, H, Hkv, dh, n_ctx, scale, cell_nkv=dyn,  # noqa: E731
                                mask=None if m is None else _dev(P, m.view(np.int16) if mask == "f16" else m), max_keys=n_ctx, flags=P.ATTN_MASK_F16 if mask == "f16" else 0).cpu().numpy().reshape(H, dh)
    out = run()
    k, v = kc[:n_kv].astype(np.float64), vc[:, :, :n_kv].astype(np.float64)
    for h in range(H):
        s = k[:, h // 3] @ q[h].astype(np.float64) * np.float32(scale) + (0 if m is None else m[:n_kv].astype(np.float64))
        p = np.exp(s - s.max())
        p /= p.sum()
        assert np.abs(out[h] - v[h // 3] @ p).max() <= (2.0 ** -11 + 1e-5) * (np.abs(v[h // 3]) @ p).max() + 2.0 ** -25 * n_kv * np.abs(v).max()
    want = np.load(os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "attn_short.npz"))[f"{dh}_{n_ctx}_{n_kv}_{mask}"]
    assert np.array_equal(out.view(np.uint32), want.view(np.uint32)), np.abs(out - want).max()


@pytest.mark.parametrize("t", [Q4_K, Q5_K, Q6_K, Q8_0])
def test_small_batch_cells_at_their_edges(P, oracle, t):
    """mmq_mid.hip: one step per round and several, pairs that do not divide among the cells, odd super-blocks, blocks of 32 that end inside a pair; up to 32, 33..64 and more rows per workgroup
    (one, two and four row groups at a time), a group of one row, a cell without rows, several rounds, blocks of scales that reach into the next round; 8, 16, 24 and 32 tokens and one more.
    Against the oracle: the same integers, <= K / 256 (Q8_0: K / 32) f32 terms in another order - the bound of the other small-batch products."""
    rng = np.random.default_rng(8100 + t)
    tail = 32 if t == Q8_0 else 256
    for K, N, T in ((4352, 4097, 17), (4608, 8193, 20), (8192 + tail, 8230, 25), (5120, 16385, 24), (4096 + tail, 16500, 32), (5120 + tail, 20000, 17), (512, 33000, 9), (1024, 40000, 25), (2560, 41000, 20), (4608, 33100, 28),
                    (2048, 70, 25), (768, 5000, 12), (12288 + tail, 4200, 18), (5120, 50000, 16), (4864, 33000, 8)):
        b = rand_blocks(t, N, K, rng)
        x = rng.normal(0, 1, (T, K)).astype(np.float32)
        bias, resid = rng.normal(0, 1, N).astype(np.float32), rng.normal(0, 1, (T, N)).astype(np.float32)
        w = P.upload_weight(t, b, K, N)
        rows = np.unique(np.concatenate([np.arange(min(N, 40)), np.arange(max(N - 40, 0), N), rng.integers(0, N, 120)]))   # (the oracle is a scalar program)
        want = oracle.mul_mat(t, b.reshape(N, b.size // N)[rows].copy(), K, len(rows), x)
        tol = dict(rtol=2e-5, atol=2e-5 * np.sqrt(max(K, 4096) / 4096))
        y = P.mul_mat_small(w, x=_dev(P, x)).cpu().numpy()
        assert np.isfinite(y).all(), (K, N, T)
        assert np.allclose(y[:, rows], want, **tol), (K, N, T, np.abs(y[:, rows] - want).max())
        xq = P.quantize_act(_dev(P, x), P.vec_dot_act_type(t))
        y2 = P.mul_mat_small(w, xq=xq, n_tokens=T, bias=_dev(P, bias), resid=_dev(P, resid)).cpu().numpy()
        assert np.array_equal(y2, (y + bias[None]) + resid), (K, N, T)
        if t in (Q4_K, Q6_K) and N > 5000:                         # two matrices share the workgroups
            n0 = N // 2 + 13
            rb = b.size // N
            ws = [P.upload_weight(t, b.reshape(N, rb)[:n0], K, n0), P.upload_weight(t, b.reshape(N, rb)[n0:], K, N - n0)]
            y3 = np.concatenate([v.cpu().numpy() for v in P.mul_mat_small_multi(ws, xq, T)], axis=1)
            assert np.allclose(y3[:, rows], want, **tol), (K, N, T, np.abs(y3[:, rows] - want).max())


@pytest.mark.parametrize("t", [Q4_K, Q6_K])
@pytest.mark.parametrize("K,N,T", [(4352, 16500, 8), (5120, 24500, 5), (9472, 17000, 2), (512, 36000, 3), (768, 33024, 8), (5120, 45000, 8), (4608, 37001, 16), (2304, 49100, 24), (1792, 33100, 32)])
def test_small_batch_cells_in_rounds(P, oracle, K, N, T, t):
    """mmq_mid.hip: three, five and six row groups a workgroup, one or two at a time; the last round full, with one group, with a group of a few rows. The bound of the others"""
    rng = np.random.default_rng(K + N + T)
    b = rand_blocks(t, N, K, rng)
    x = rng.normal(0, 1, (T, K)).astype(np.float32)
    rows = np.unique(np.concatenate([np.arange(200), np.arange(N - 200, N), rng.integers(0, N, 200)]))                     # (the oracle is a scalar program)
    want = oracle.mul_mat(t, b.reshape(N, b.size // N)[rows].copy(), K, len(rows), x)
    y = P.mul_mat_small(P.upload_weight(t, b, K, N), x=_dev(P, x)).cpu().numpy()
    assert np.isfinite(y).all() and np.allclose(y[:, rows], want, rtol=2e-5, atol=2e-5 * np.sqrt(max(K, 4096) / 4096)), np.abs(y[:, rows] - want).max()


@pytest.mark.parametrize("t", [Q4_K, Q5_K, Q6_K, Q8_0])
def test_small_batches_of_more_than_one_pass(P, oracle, t):
    """33..64 tokens of one matrix: passes of 32 and of 16, and a last pass of any width, on each of the three kernels (which, by rows, K and tokens: test_host_launches.py). Every token against the
    oracle, inside the bound of the other small-batch products; rows the oracle has not seen: written."""
    rng = np.random.default_rng(8200 + t)
    for K, N, Ts in ((768 if t != Q8_0 else 896, 12288, (33, 48, 49, 52, 56, 57, 64)), (512, 9000, (50, 41)), (2048, 12300, (52, 36)), (4096, 4096, (52, 63)), (4608, 9000, (49, 64)), (1024, 16384, (56, 40))):
        b = rand_blocks(t, N, K, rng)
        w = P.upload_weight(t, b, K, N)
        rows = np.unique(np.concatenate([np.arange(20), np.arange(N - 20, N), rng.integers(0, N, 40)]))                    # (the oracle is a scalar program)
        x = rng.normal(0, 1, (64, K)).astype(np.float32)
        want = oracle.mul_mat(t, b.reshape(N, b.size // N)[rows].copy(), K, len(rows), x)
        for T in Ts:
            xd, y = _dev(P, x[:T]), _dev(P, np.full((T, N), np.nan, np.float32))
            f = P.L.load().pm355_mul_mat_q_small
            f.restype, f.argtypes = C.c_int, [C.c_int, C.c_void_p, C.c_int64, C.c_int64, C.c_void_p, C.c_void_p, C.c_int64, C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p]
            assert f(w.type, w.data.data_ptr(), K, N, None, xd.data_ptr(), T, y.data_ptr(), None, None, P.stream_ptr()) == 0
            y = y.cpu().numpy()
            assert np.isfinite(y).all(), (K, N, T, np.flatnonzero(~np.isfinite(y).all(1)))
            assert np.allclose(y[:, rows], want[:T], rtol=2e-5, atol=2e-5 * np.sqrt(max(K, 4096) / 4096)), (K, N, T, np.abs(y[:, rows] - want[:T]).max())
