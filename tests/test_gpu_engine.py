"""GPU parity of the engine (resident layer window) against the CPU oracle on tiny Llama / Qwen2
shaped models: prefill + decode, KV cache contents, window hand-off, graph replay, greedy loop."""
import numpy as np
import pytest

from _bind import Q4_K, Q6_K, Q8_0, tiny_model

pytestmark = pytest.mark.gpu


def _nmse(a, b):
    a = np.asarray(a, dtype=np.float64).ravel()
    b = np.asarray(b, dtype=np.float64).ravel()
    return float(((a - b) ** 2).sum() / max((b ** 2).sum(), 1e-30))


def _hp(d):
    return dict(arch=d.arch, n_layer=d.n_layer, n_embd=d.n_embd, n_head=d.n_head, n_head_kv=d.n_head_kv,
                head_dim=d.head_dim, n_ff=d.n_ff, n_vocab=d.n_vocab, rms_eps=d.rms_eps, rope_freq_base=d.rope_freq_base)


@pytest.fixture(scope="module")
def E():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("needs a HIP device")
    import prima_cpp_amd.engine as eng
    eng.torch = torch
    return eng


def _quantizer():
    from _bind import Ref, have_ref
    return Ref("scalar").quantize_weights if have_ref("scalar") else None


@pytest.mark.parametrize("arch", [0, 1])
def test_window_prefill_and_decode_vs_oracle(E, oracle, arch):
    torch = E.torch
    rng = np.random.default_rng(31 + arch)
    d = tiny_model(rng, arch=arch, n_layer=2, n_embd=256, n_head=4, n_head_kv=2, n_ff=512, n_vocab=320, n_ctx=64,
                   rope_freqs=(arch == 0), quantize=_quantizer())
    w = E.Window(_hp(d), n_ctx=64)
    w.load_desc(d)
    w.finalize(max_tokens=8)
    ho = oracle.model_new(d)
    toks = rng.integers(0, d.n_vocab, 9).astype(np.int32)
    steps = [(toks[:5], 0), (toks[5:6], 5), (toks[6:7], 6), (toks[7:9], 7)]
    for tk, p0 in steps:
        hid, lg, am = w.decode(tokens=torch.from_numpy(tk).cuda(), pos0=p0, want_argmax=True)
        h_ref, l_ref = oracle.model_eval(ho, d, tokens=tk, pos0=p0)
        # north_star: logits within 1e-3 relative; whole-stack metric = NMSE (reference: test-backend-ops)
        assert _nmse(hid.cpu().numpy(), h_ref) < 1e-3
        assert _nmse(lg.cpu().numpy(), l_ref) < 1e-3
        assert int(am.item()) == int(np.argmax(lg.cpu().numpy()))
    # layer-0 KV cache: K rows are rope(f32)->f16, V rows plain f16: compare as floats (cos/sin <= 2 ulp apart)
    for which in (0, 1):
        a = w.kv(0, which).view(np.float16).astype(np.float32)
        b = oracle.model_kv(ho, d, 0, which).view(np.float16).astype(np.float32)
        assert _nmse(a, b) < 1e-6
        if which == 1:
            assert np.array_equal(w.kv(0, 1), oracle.model_kv(ho, d, 0, 1))     # V path has no transcendental: bit-exact
    oracle.model_free(ho)
    w.close()


def test_two_windows_hand_off_equals_single_window(E):
    """Piped-ring split: window A = layers [0,1) + embd, window B = layers [1,2) + head. The activation
    handed from A to B must reproduce the single-window result exactly (same kernels, same order)."""
    torch = E.torch
    rng = np.random.default_rng(33)
    d = tiny_model(rng, arch=0, n_layer=2, n_embd=256, n_head=4, n_head_kv=2, n_ff=512, n_vocab=320, n_ctx=64, rope_freqs=True)
    full = E.Window(_hp(d), n_ctx=64)
    full.load_desc(d); full.finalize(4)
    a = E.Window(_hp(d), lo=0, hi=1, flags=E.HAS_EMBD, n_ctx=64)
    a.load_desc(d); a.finalize(4)
    b = E.Window(_hp(d), lo=1, hi=2, flags=E.HAS_HEAD, n_ctx=64)
    b.load_desc(d); b.finalize(4)
    toks = torch.from_numpy(rng.integers(0, d.n_vocab, 4).astype(np.int32)).cuda()
    for tk, p0 in ((toks[:3], 0), (toks[3:4], 3)):
        hf, lf, _ = full.decode(tokens=tk, pos0=p0)
        ha, _, _ = a.decode(tokens=tk, pos0=p0, want_logits=False)
        hb, lb, _ = b.decode(x_in=ha, pos0=p0)
        assert torch.equal(hf, hb) and torch.equal(lf, lb)
    for w in (full, a, b):
        w.close()


def test_graph_replay_and_device_greedy_loop(E, oracle):
    torch = E.torch
    rng = np.random.default_rng(34)
    d = tiny_model(rng, arch=0, n_layer=2, n_embd=256, n_head=4, n_head_kv=2, n_ff=512, n_vocab=320, n_ctx=64, rope_freqs=True)
    w = E.Window(_hp(d), n_ctx=64)
    w.load_desc(d); w.finalize(4)
    n = 12
    first = int(rng.integers(0, d.n_vocab))
    outs = []
    for use_graph in (False, True):
        w.kv_clear()
        io = torch.zeros(n + 1, dtype=torch.int32, device="cuda")
        io[0] = first
        w.generate(io, 0, n, use_graph=use_graph)
        torch.cuda.synchronize()
        outs.append(io.cpu().numpy())
    assert np.array_equal(outs[0], outs[1])               # graph replay == eager launches, token for token
    # greedy parity with the CPU oracle; a flat synthetic logit distribution may flip near-ties, so
    # follow the oracle only while its top-1/top-2 margin is above the observed logit noise
    ho = oracle.model_new(d)
    tok = first
    for i in range(n):
        _, lg = oracle.model_eval(ho, d, tokens=np.array([tok], dtype=np.int32), pos0=i)
        top2 = np.sort(lg)[-2:]
        if top2[1] - top2[0] < 1e-2 * max(1.0, abs(top2[1])):
            break
        assert outs[0][i + 1] == int(np.argmax(lg)), (i, outs[0][: i + 2])
        tok = int(np.argmax(lg))
    oracle.model_free(ho)
    w.close()


def test_step_with_external_activation_buffers(E):
    """pm355_model_step: position in device memory, x_in/x_out owned by the caller (ring transport buffers)."""
    torch = E.torch
    rng = np.random.default_rng(35)
    d = tiny_model(rng, arch=1, n_layer=2, n_embd=256, n_head=4, n_head_kv=2, n_ff=512, n_vocab=320, n_ctx=64)
    w = E.Window(_hp(d), lo=0, hi=2, flags=0, n_ctx=64)
    w.load_desc(d); w.finalize(1)
    x = torch.randn(5, 1, d.n_embd, device="cuda")
    ref = []
    for i in range(5):
        h, _, _ = w.decode(x_in=x[i], pos0=i, want_logits=False)
        ref.append(h.clone())
    w.kv_clear()
    xin = torch.empty(1, d.n_embd, device="cuda"); xout = torch.empty(1, d.n_embd, device="cuda")
    w.set_pos(0)
    for i in range(5):
        xin.copy_(x[i])
        w.step(x_in=xin, x_out=xout, advance=1, use_graph=True)
        assert torch.equal(xout, ref[i])
    w.close()


@pytest.mark.parametrize("name", ["llama", "qwen2"])
def test_golden_greedy_decode_vs_reference(E, name):
    """The committed golden run of the REFERENCE CPU backend (tests/golden/tiny_*_decode.npz): same GGUF-order weights,
    same prompt; logits NMSE < 1e-3 per step (teacher-forced) and greedy-token parity wherever the reference's own
    top-1/top-2 margin is above the logit noise."""
    import os
    from _bind import desc_from_arrays
    torch = E.torch
    z = np.load(os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", f"tiny_{name}_decode.npz"))
    d = desc_from_arrays(z)
    w = E.Window(_hp(d), n_ctx=int(d.n_ctx))
    w.load_desc(d)
    w.finalize(max_tokens=8)
    prompt, toks, logits = z["prompt"], z["tokens"], z["logits"]
    _, lg, _ = w.decode(tokens=torch.from_numpy(prompt).cuda(), pos0=0)
    got, nm = [int(lg.argmax().item())], [_nmse(lg.cpu().numpy(), logits[0])]
    for i in range(len(toks) - 1):
        _, lg, am = w.decode(tokens=torch.tensor([int(toks[i])], dtype=torch.int32, device="cuda"), pos0=len(prompt) + i, want_argmax=True)
        got.append(int(am.item()))
        nm.append(_nmse(lg.cpu().numpy(), logits[i + 1]))
    w.close()
    assert max(nm) < 1e-3, nm
    for i, (a, b) in enumerate(zip(got, toks)):
        top2 = np.sort(logits[i])[-2:]
        if top2[1] - top2[0] > 2e-2 * max(1.0, abs(float(top2[1]))):
            assert a == int(b), (i, got, toks.tolist())


@pytest.mark.parametrize("arch", [0, 1])
def test_prefill_mfma_path_vs_oracle(E, oracle, arch):
    """n_tokens >= 16 goes through the MFMA GEMMs (f16 tiles, activations not re-quantized): logits NMSE vs the reference
    arithmetic stays within the reference's whole-layer backend tolerance (2e-3, tests/test-backend-ops.cpp:3000), and a
    following single-token decode step continues from the KV cache the prefill wrote."""
    torch = E.torch
    rng = np.random.default_rng(81 + arch)
    d = tiny_model(rng, arch=arch, n_layer=2, n_embd=256, n_head=4, n_head_kv=2, n_ff=512, n_vocab=320, n_ctx=64,
                   rope_freqs=(arch == 0), quantize=_quantizer())
    w = E.Window(_hp(d), n_ctx=64)
    w.load_desc(d)
    w.finalize(max_tokens=32)
    ho = oracle.model_new(d)
    toks = rng.integers(0, d.n_vocab, 25).astype(np.int32)
    hid, lg, _ = w.decode(tokens=torch.from_numpy(toks[:24]).cuda(), pos0=0)
    h_ref, l_ref = oracle.model_eval(ho, d, tokens=toks[:24], pos0=0)
    assert _nmse(hid.cpu().numpy(), h_ref) < 2e-3
    assert _nmse(lg.cpu().numpy(), l_ref) < 2e-3
    hid, lg, _ = w.decode(tokens=torch.from_numpy(toks[24:25]).cuda(), pos0=24)
    h_ref, l_ref = oracle.model_eval(ho, d, tokens=toks[24:25], pos0=24)
    assert _nmse(lg.cpu().numpy(), l_ref) < 2e-3
    oracle.model_free(ho)
    w.close()


@pytest.mark.parametrize("T,n_embd", [(72, 2048), (130, 2048)])
def test_prompt_with_norms_behind_split_products(E, oracle, T, n_embd):
    """K slices of wo and ffn_down are added up by the launch that also forms the next RMS norm, those of wq | wk | wv by one that rotates and stores (128-row tiles up to 128 tokens, 256-row
    tiles beyond): hidden rows against the oracle."""
    torch = E.torch
    rng = np.random.default_rng(T)
    d = tiny_model(rng, n_layer=2, n_embd=n_embd, n_head=n_embd // 128, n_head_kv=2, n_ff=4096, n_vocab=320, n_ctx=192, rope_freqs=True, quantize=_quantizer())
    w = E.Window(_hp(d), n_ctx=192)
    w.load_desc(d)
    w.finalize(max_tokens=T)
    ho = oracle.model_new(d)
    toks = rng.integers(0, d.n_vocab, T).astype(np.int32)
    hid, lg, _ = w.decode(tokens=torch.from_numpy(toks).cuda(), pos0=0)
    h_ref, l_ref = oracle.model_eval(ho, d, tokens=toks, pos0=0)
    assert _nmse(hid.cpu().numpy(), h_ref) < 2e-3
    assert _nmse(lg.cpu().numpy(), l_ref) < 2e-3
    oracle.model_free(ho)
    w.close()


def _filled_window(E, n_embd, n_head, n_head_kv, n_ff, n_ctx, bias, flags=0):
    """two layers of random weights made on the device (n_vocab 320 where the window has its ends); ffn_down is Q6_K, with biases wv too (a launch of two types, tiles of 64 tokens in a wide pass)"""
    w = E.Window(dict(arch=0, n_layer=2, n_embd=n_embd, n_head=n_head, n_head_kv=n_head_kv, head_dim=128, n_ff=n_ff, n_vocab=320, rms_eps=1e-5, rope_freq_base=10000.0), flags=flags, n_ctx=n_ctx)
    for il in range(2):
        for i, kind in enumerate((E.T_ATTN_NORM, E.T_FFN_NORM)):
            w.fill_tensor(kind, il, E.F32, 100 * il + 1 + i, 0.0)
        for i, kind in enumerate((E.T_WQ, E.T_WK, E.T_WV, E.T_WO, E.T_FFN_GATE, E.T_FFN_UP, E.T_FFN_DOWN)):
            w.fill_tensor(kind, il, Q6_K if kind == E.T_FFN_DOWN or bias and kind == E.T_WV else Q4_K, 100 * il + 10 + i, 2.0 / np.sqrt(n_ff if kind == E.T_FFN_DOWN else n_embd))
        for i, kind in enumerate((E.T_BQ, E.T_BK, E.T_BV) if bias else ()):
            w.fill_tensor(kind, il, E.F32, 100 * il + 20 + i, 0.5)
    if flags:
        w.fill_tensor(E.T_OUT_NORM, -1, E.F32, 300, 0.0)
        w.fill_tensor(E.T_OUTPUT, -1, Q6_K, 301, 2.0 / np.sqrt(n_embd))
        w.fill_tensor(E.T_TOK_EMBD, -1, Q4_K, 302, 1.0)
    return w


# rows of a norm beyond 4096 and of wq | wk | wv beyond 4096 and 8192 (a wave's second and third column), K in five to eight slices and in fewer, tiles of 128 and of 256 rows
# (test_host_launches.py holds which shape reaches which form)
SLICED = [(4352, 32, 8, 14336), (8192, 64, 8, 28672), (8192, 16, 4, 4096)]


@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("n_embd,n_head,n_head_kv,n_ff", SLICED)
def test_prompts_with_slices_added_up_in_the_norm_and_the_rope(E, n_embd, n_head, n_head_kv, n_ff, bias):
    """560 tokens in one pass - slices, norms, rope and cache stores are launches of their own at that size - against passes of 72 (128-row tiles), 130, 200 and 158 tokens, whose slices are added
    up by the launches that form the norm and that rotate and store, and of 512 and 48 (norm only). The same sums in slices of other lengths: f32 rounding, which turns F16 roundings of the
    activations (2^-11 of one) here and there; a wrong row, column, position or slice is another value altogether."""
    torch = E.torch
    T = 560
    w = _filled_window(E, n_embd, n_head, n_head_kv, n_ff, 576, bias)
    w.finalize(max_tokens=T)
    x = torch.randn((T, n_embd), generator=torch.Generator(device="cuda").manual_seed(n_embd + n_head), device="cuda")
    one = torch.randn((3, n_embd), generator=torch.Generator(device="cuda").manual_seed(1), device="cuda")
    want = w.decode(x_in=x, pos0=0)[0].double()
    behind = [w.decode(x_in=one[i:i + 1], pos0=T + i)[0].double() for i in range(3)]
    for lens in ((72, 130, 200, 158), (512, 48)):
        w.kv_clear()
        at = 0
        for n in lens:
            got = w.decode(x_in=x[at:at + n].contiguous(), pos0=at)[0].double()
            err = (got - want[at:at + n]).norm(dim=1) / want[at:at + n].norm(dim=1)
            assert err.max() < 2e-3, (lens, at, err.max().item(), err.argmax().item())
            at += n
        for i in range(3):                                      # single tokens read the cache that the passes left
            got = w.decode(x_in=one[i:i + 1], pos0=T + i)[0].double()
            assert (got - behind[i]).norm() < 2e-2 * behind[i].norm(), ((got - behind[i]).norm() / behind[i].norm()).item()
    w.close()


@pytest.mark.parametrize("n_embd,n_head,n_head_kv,n_ff,lens", [(2048, 16, 4, 4096, [7, 31, 2, 19, 1, 12]), (2048, 16, 4, 4096, [30] * 9), (2048, 16, 4, 4096, [30, 29] * 3 + [23]), (8192, 16, 4, 4096, [5, 27, 14, 1])])
@pytest.mark.parametrize("bias", [False, True])
def test_wide_passes_with_split_products_equal_the_portions_alone(E, n_embd, n_head, n_head_kv, n_ff, lens, bias):
    """Wide passes whose K is split: wq | wk | wv ends with the rope and the cache stores of every row's own sequence and position (up to 255 rows; 270 in a launch of its own), q rounded as the
    small passes round it. Three rounds, so that positions differ and the stored cells are read back. Against the same portions alone, which small passes take."""
    torch = E.torch
    rng = np.random.default_rng(len(lens) + n_embd)
    ws = []
    for _ in range(2):
        w = _filled_window(E, n_embd, n_head, n_head_kv, n_ff, 96, bias, flags=E.HAS_EMBD | E.HAS_HEAD)
        w.finalize_pool(512, len(lens), len(lens) * 96)
        ws.append((w, [w.seq_new() for _ in lens]))
    (w, seqs), (w1, seqs1) = ws
    for k in range(3):
        part = [rng.integers(0, 320, 1 if k == 2 else n if k == 0 else max(1, n // 2) + 9).astype(np.int32) for n in lens]
        lg, lg1 = torch.full((len(lens), 320), float("nan"), device="cuda"), torch.empty((len(lens), 320), device="cuda")
        w.batch([(q, t, [len(t) - 1]) for q, t in zip(seqs, part)], logits=lg)
        for i, t in enumerate(part):
            w1.batch([(seqs1[i], t, [len(t) - 1])], logits=lg1[i:i + 1])
        a, b = lg.double(), lg1.double()
        err = ((a - b) ** 2).sum(-1) / (b ** 2).sum(-1)
        assert (err < 1e-3).all(), (k, err.max().item())
    w.close()
    w1.close()


@pytest.mark.parametrize("flash,n_head,n_embd,n_head_kv", [("1", 8, 512, 2), ("1", 4, 512, 2), ("0", 8, 512, 2), ("1", 8, 1024, 4), ("1", 16, 1024, 8)])
def test_long_context_split_attention_path(E, monkeypatch, flash, n_head, n_embd, n_head_kv):
    """Beyond PM355_ATTN_SPLIT_MIN positions the engine switches from the one-workgroup-per-head attention kernel to the
    keys-split-over-workgroups path - one launch of flash-decoding with an in-launch merge (attn_flash.hip; head_dim 64 and 128, up to
    three spans merged here), or with PM355_ATTN_FLASH=0 the three-launch form (attn_split.hip) - in another captured graph: hidden
    state and logits agree at every position, through graph replay and through plain decode(). The n_embd 1024 shapes have wk / wv row
    slices that take the QKV epilogue (rope + KV store there), so their long-context regime is the matrix-core kernel over cached cells
    (attn_flash_mfma.hip, head_dim 128 and 64)."""
    torch = E.torch
    rng = np.random.default_rng(78)
    monkeypatch.setenv("PM355_ATTN_FLASH", flash)
    d = tiny_model(rng, arch=0, n_layer=2, n_embd=n_embd, n_head=n_head, n_head_kv=n_head_kv, n_ff=1024, n_vocab=320, n_ctx=320, rope_freqs=True)
    toks = rng.integers(0, d.n_vocab, 300).astype(np.int32)
    res = []
    for split_min in ("100000", "40"):
        monkeypatch.setenv("PM355_ATTN_SPLIT_MIN", split_min)
        w = E.Window(_hp(d), n_ctx=320)
        w.load_desc(d); w.finalize(4)
        out = []
        x_out = torch.empty((1, d.n_embd), dtype=torch.float32, device="cuda")
        lg = torch.empty(d.n_vocab, dtype=torch.float32, device="cuda")
        tok = torch.zeros(1, dtype=torch.int32, device="cuda")
        w.set_pos(0)
        for i, t in enumerate(toks):
            tok[0] = int(t)
            if i % 2 == 0:
                w.step(token=tok, x_out=x_out, logits=lg, advance=1, use_graph=True)       # device-side position, graph replay
            else:
                h, l, _ = w.decode(tokens=tok, pos0=i)                                     # host-given position, eager launches
                x_out.copy_(h); lg.copy_(l)
                w.set_pos(i + 1)
            if i in (0, 39, 40, 41, 100, 255, 256, 257, 299):
                torch.cuda.synchronize()
                out.append((x_out.cpu().numpy().copy(), lg.cpu().numpy().copy()))
        res.append(out)
        w.close()
    for (h0, l0), (h1, l1) in zip(*res):
        # not bit-identical: a different f32 summation order can flip an F16 / int8 re-quantization downstream, and the KV
        # caches of the two runs then differ by that much for all later tokens (same effect as between the reference's own builds)
        assert _nmse(h1, h0) < 1e-4 and _nmse(l1, l0) < 1e-3        # the whole-stack bound used against the reference itself


def test_step_refuses_to_write_past_the_kv_slab(E):
    """pm355_model_step_ex / set_seq_pos must bound the position by n_ctx (llama_decode returns an error when no KV
    cell is left, src/llama.cpp:18445); a failed step must not move the host mirror of the device counters."""
    import prima_cpp_amd.lib as L
    torch = E.torch
    rng = np.random.default_rng(3)
    d = tiny_model(rng, arch=0, n_layer=1, n_embd=256, n_head=4, n_head_kv=2, n_ff=512, n_vocab=320, n_ctx=32, rope_freqs=True)
    w = E.Window(_hp(d), n_ctx=32)
    w.load_desc(d)
    w.finalize(max_tokens=1, n_seq=2)
    tok = torch.zeros(1, dtype=torch.int32, device="cuda")
    am = torch.zeros(1, dtype=torch.int32, device="cuda")
    w.set_pos(31)
    w.step(token=tok, argmax=am)                       # position 31 = last cell: fine
    torch.cuda.synchronize()
    for use_graph in (True, False):
        with pytest.raises(L.PM355Error):
            w.step(token=tok, argmax=am, use_graph=use_graph)    # position 32 == n_ctx: refused, nothing launched
    with pytest.raises(L.PM355Error):
        w.set_seq_pos(1, 33)
    with pytest.raises(L.PM355Error):
        w.set_seq_pos(1, -1)
    torch.cuda.synchronize()
    w.set_pos(5)
    w.step(token=tok, argmax=am)                       # still usable after the refusals
    torch.cuda.synchronize()
    w.close()


@pytest.mark.parametrize("n_slots", [1, 2, 3, 4])
def test_window_streaming_matches_resident(E, n_slots):
    """pm355_model_set_streaming: layer tensors parked in pinned host memory and cycled through n_slots device slots by the copy
    stream (the GPU-side form of prima.cpp's layer-window prefetch, src/llama.cpp:18152-18218) must give bit-identical results to the
    fully resident window: 20-token MFMA prefill, a short multi-token batch, and single-token steps wrapping around the slot ring."""
    torch = E.torch
    rng = np.random.default_rng(99)
    d = tiny_model(rng, arch=0, n_layer=4, n_embd=256, n_head=4, n_head_kv=2, n_ff=512, n_vocab=320, n_ctx=64, rope_freqs=True)
    toks = rng.integers(0, d.n_vocab, 30).astype(np.int32)
    outs = []
    for slots in (0, n_slots):
        w = E.Window(_hp(d), n_ctx=64)
        if slots:
            w.set_streaming(slots)
        w.load_desc(d)
        w.finalize(max_tokens=20)
        res = []
        h, lg, _ = w.decode(tokens=torch.from_numpy(toks[:20]).cuda(), pos0=0)
        res.append((h.cpu().numpy(), lg.cpu().numpy()))
        h, lg, _ = w.decode(tokens=torch.from_numpy(toks[20:23]).cuda(), pos0=20)
        res.append((h.cpu().numpy(), lg.cpu().numpy()))
        w.set_pos(23)
        x_out = torch.empty((1, d.n_embd), dtype=torch.float32, device="cuda")
        lgt = torch.empty(d.n_vocab, dtype=torch.float32, device="cuda")
        tok = torch.zeros(1, dtype=torch.int32, device="cuda")
        for t in toks[23:]:
            tok[0] = int(t)
            w.step(token=tok, x_out=x_out, logits=lgt, advance=1)
            torch.cuda.synchronize()
            res.append((x_out.cpu().numpy().copy(), lgt.cpu().numpy().copy()))
        if slots:
            assert w.streamed_bytes() > 0
        outs.append(res)
        w.close()
    for (h0, l0), (h1, l1) in zip(*outs):
        assert np.array_equal(h0, h1) and np.array_equal(l0, l1)


def test_qkv_epilogue_decode_form_matches_round2_form(E, oracle, monkeypatch):
    """PM355_QKV_EPI=0 (rope + KV store inside the attention kernel, the round-2 launch sequence) against the default (RoPE + KV store in
    the epilogue of the wq | wk | wv launch, attention over cached cells) through graph replay, on a window whose projections give every
    workgroup whole rotation pairs (N % 512 == 0), across the 64-cell boundary of the short attention kernel; both against the oracle."""
    torch = E.torch
    rng = np.random.default_rng(123)
    d = tiny_model(rng, arch=0, n_layer=2, n_embd=1024, n_head=8, n_head_kv=4, n_ff=2048, n_vocab=320, n_ctx=128, rope_freqs=True)
    assert d.head_dim == 128
    toks = rng.integers(0, d.n_vocab, 80).astype(np.int32)
    outs = []
    for flag in ("0", "1"):
        monkeypatch.setenv("PM355_QKV_EPI", flag)
        w = E.Window(_hp(d), n_ctx=128)
        w.load_desc(d)
        w.finalize(max_tokens=1)
        w.set_pos(0)
        x_out = torch.empty((1, d.n_embd), dtype=torch.float32, device="cuda")
        lg = torch.empty(d.n_vocab, dtype=torch.float32, device="cuda")
        tok = torch.zeros(1, dtype=torch.int32, device="cuda")
        res = []
        for t in toks:
            tok[0] = int(t)
            w.step(token=tok, x_out=x_out, logits=lg, advance=1, use_graph=True)
            torch.cuda.synchronize()
            res.append((x_out.cpu().numpy().copy(), lg.cpu().numpy().copy()))
        assert w.check() == 0
        outs.append(res)
        kv = [(w.kv(il, 0).copy(), w.kv(il, 1).copy()) for il in range(d.n_layer)]
        outs.append(kv)
        w.close()
    (r0, kv0, r1, kv1) = outs
    per = [_nmse(l1, l0) for (_, l0), (_, l1) in zip(r0, r1)]
    nm = max(per)
    print(f"\n[QKV epilogue form vs round-2 form] worst per-step logits NMSE {nm:.2e}; steps above 1e-9: {[(i, float(f'{v:.1e}')) for i, v in enumerate(per) if v > 1e-9]}")
    # summation order only (1e-13) - until a value that sits on an int8 / F16 rounding boundary tips the other way in one of the two runs:
    # that token differs by ~1e-4 and, through its K / V cache rows, every later token by ~1e-5 (observed: identical up to step 24 of 80).
    # The per-op comparison is tests/test_gpu_ops.py::test_qkv_epilogue_and_cached_attention_equal_the_fused_attention_path.
    assert nm < 1e-3 and max(per[:10]) < 1e-9, (nm, per[:10])
    # layer-0 caches (their inputs are identical in both runs): the same F16 bits except where the split wk / wv rows round differently
    for which in (0, 1):
        a, b = kv0[0][which], kv1[0][which]
        assert (a != b).mean() < 0.01
    # and against the oracle (teacher-forced)
    ho = oracle.model_new(d)
    worst = 0.0
    for i, t in enumerate(toks[:70]):
        _, l_ref = oracle.model_eval(ho, d, tokens=np.array([t], dtype=np.int32), pos0=i)
        worst = max(worst, _nmse(r1[i][1], l_ref))
    oracle.model_free(ho)
    print(f"[QKV epilogue form vs oracle] worst per-step logits NMSE {worst:.2e}")
    assert worst < 1e-3, worst


@pytest.mark.experiments
@pytest.mark.parametrize("arch", [0, 1])
def test_producer_side_sum_of_squares_decode_is_bit_identical(E, monkeypatch, arch):
    """PM355_SS=0 (every rms_norm prologue reduces its own row: the round-4 form) against the default (wo / ffn_down leave per-workgroup
    partials, the wq | wk | wv, ffn_gate | ffn_up and lm_head launches add them): hidden rows and logits of 40 graph-replayed tokens must be
    the same bits - the partial sums are exact in f64 for these magnitudes, and where they are not the f32 rounding of the mean hides it."""
    torch = E.torch
    rng = np.random.default_rng(321)
    d = tiny_model(rng, arch=arch, n_layer=3, n_embd=1024, n_head=8, n_head_kv=4, n_ff=2048, n_vocab=320, n_ctx=128, rope_freqs=(arch == 0))
    toks = rng.integers(0, d.n_vocab, 40).astype(np.int32)
    outs = []
    for flag in ("0", "1"):
        monkeypatch.setenv("PM355_SS", flag)
        w = E.Window(_hp(d), n_ctx=128)
        w.load_desc(d)
        w.finalize(max_tokens=1)
        w.set_pos(0)
        x_out = torch.empty((1, d.n_embd), dtype=torch.float32, device="cuda")
        lg = torch.empty(d.n_vocab, dtype=torch.float32, device="cuda")
        tok = torch.zeros(1, dtype=torch.int32, device="cuda")
        res = []
        for t in toks:
            tok[0] = int(t)
            w.step(token=tok, x_out=x_out, logits=lg, advance=1, use_graph=True)
            torch.cuda.synchronize()
            res.append((x_out.cpu().numpy().copy(), lg.cpu().numpy().copy()))
        assert w.check() == 0
        outs.append(res)
        w.close()
    for i, ((h0, l0), (h1, l1)) in enumerate(zip(*outs)):
        assert np.array_equal(h0, h1) and np.array_equal(l0, l1), i


@pytest.mark.experiments
@pytest.mark.parametrize("arch,n_tok", [(0, 90), (1, 70)])
def test_persistent_decode_engine_matches_the_five_launch_path(E, oracle, monkeypatch, arch, n_tok):
    """Round 5: csrc/decode_engine.hip (opt-in, PM355_ENGINE=1) - every phase of every layer of a single-token step as ONE persistent launch, device-wide
    barriers in place of kernel boundaries - against the default five launches per layer. The same row loops, prologue and epilogue code run in both:
    hidden rows and logits must be the same BITS, across the 64-cell boundary of the short attention path, NORM and NEOX rope, with the engine's
    watchdog clean (a stale hand-off between workgroups showed as 1e-4 while the engine was being built). Then against the oracle, teacher-forced."""
    torch = E.torch
    rng = np.random.default_rng(4321 + arch)
    d = tiny_model(rng, arch=arch, n_layer=3, n_embd=1024, n_head=8, n_head_kv=4, n_ff=2048, n_vocab=320, n_ctx=128, rope_freqs=(arch == 0))
    toks = rng.integers(0, d.n_vocab, n_tok).astype(np.int32)
    outs = []
    for flag in ("0", "1"):
        monkeypatch.setenv("PM355_ENGINE", flag)
        monkeypatch.setenv("PM355_ENGINE_VERBOSE", "1")
        w = E.Window(_hp(d), n_ctx=128)
        w.load_desc(d)
        w.finalize(max_tokens=1)
        w.set_pos(0)
        x_out = torch.empty((1, d.n_embd), dtype=torch.float32, device="cuda")
        lg = torch.empty(d.n_vocab, dtype=torch.float32, device="cuda")
        tok = torch.zeros(1, dtype=torch.int32, device="cuda")
        res = []
        for t in toks:
            tok[0] = int(t)
            w.step(token=tok, x_out=x_out, logits=lg, advance=1, use_graph=True)
            torch.cuda.synchronize()
            res.append((x_out.cpu().numpy().copy(), lg.cpu().numpy().copy()))
        assert w.check() == 0
        outs.append(res)
        w.close()
    per = [max(_nmse(h1, h0), _nmse(l1, l0)) for (h0, l0), (h1, l1) in zip(*outs)]
    print(f"\n[engine vs five launches, arch {arch}] worst per-step NMSE {max(per):.2e}; bit-identical steps {sum(int(np.array_equal(a[1], b[1])) for a, b in zip(*outs))}/{n_tok}")
    assert max(per) == 0.0, per
    ho = oracle.model_new(d)
    worst = 0.0
    for i, t in enumerate(toks[:40]):
        _, l_ref = oracle.model_eval(ho, d, tokens=np.array([t], dtype=np.int32), pos0=i)
        worst = max(worst, _nmse(outs[1][i][1], l_ref))
    oracle.model_free(ho)
    assert worst < 1e-3, worst


@pytest.mark.experiments
@pytest.mark.parametrize("arch", [0, 1])
def test_attention_tail_decode_is_bit_identical(E, monkeypatch, arch):
    """Round 5: PM355_ATTN_TAIL=1 - the attention computed in the tail of the wq | wk | wv launch by the last workgroups of each
    KV-head group (four launches per layer) - against the default five launches: the same hidden rows and logits, bit for bit, across the 64-cell
    boundary of the short attention path, NORM and NEOX rope, with the tail's watchdog clean."""
    torch = E.torch
    rng = np.random.default_rng(977 + arch)
    d = tiny_model(rng, arch=arch, n_layer=3, n_embd=1024, n_head=16, n_head_kv=8, n_ff=2048, n_vocab=320, n_ctx=128, rope_freqs=(arch == 0))
    toks = rng.integers(0, d.n_vocab, 80).astype(np.int32)
    outs = []
    for flag in ("0", "1"):
        monkeypatch.setenv("PM355_ATTN_TAIL", flag)
        w = E.Window(_hp(d), n_ctx=128)
        w.load_desc(d)
        w.finalize(max_tokens=1)
        w.set_pos(0)
        x_out = torch.empty((1, d.n_embd), dtype=torch.float32, device="cuda")
        lg = torch.empty(d.n_vocab, dtype=torch.float32, device="cuda")
        tok = torch.zeros(1, dtype=torch.int32, device="cuda")
        res = []
        for t in toks:
            tok[0] = int(t)
            w.step(token=tok, x_out=x_out, logits=lg, advance=1, use_graph=True)
            torch.cuda.synchronize()
            res.append((x_out.cpu().numpy().copy(), lg.cpu().numpy().copy()))
        assert w.check() == 0
        outs.append(res)
        w.close()
    for i, ((h0, l0), (h1, l1)) in enumerate(zip(*outs)):
        assert np.array_equal(h0, h1) and np.array_equal(l0, l1), i


@pytest.mark.parametrize("arch,max_tokens,n_ctx", [(0, 64, 96), (1, 64, 96), (0, 7, 64), (0, 40, 288), (0, 2, 64), (0, 64, 72)])
def test_batches_of_several_sequences_equal_one_sequence_at_a_time(E, arch, max_tokens, n_ctx):
    """pm355_model_batch over several sequences runs their rows in common passes: prompts of unequal length (single tokens, odd ones, longer than 32 - the 16-bit arithmetic -, cut by
    max_tokens), decoded tokens taken on the device, rows wanted out of order, twice or not at all; behind 192 cells the attention changes kernels; n_ctx = 72 takes the sequences one by
    one. Against the same portions given alone: the same arithmetic with other summation orders, so 8-bit roundings may turn (the bound of the oracle comparisons above)."""
    torch = E.torch
    rng = np.random.default_rng(7 + max_tokens)
    d = tiny_model(rng, arch=arch, n_layer=2, n_embd=256, n_head=4, n_head_kv=2, n_ff=512, n_vocab=320, n_ctx=n_ctx, rope_freqs=arch == 0)
    lens = [1, 3, 17, 38, 5] if n_ctx < 200 else [200, 3, 17, 38, 190]
    ws = []
    for _ in range(2):
        w = E.Window(_hp(d), n_ctx=n_ctx)
        w.load_desc(d)
        w.finalize_pool(max_tokens, len(lens), len(lens) * n_ctx)
        ws.append((w, [w.seq_new() for _ in lens]))
    (w, seqs), (w1, seqs1) = ws
    toks = [rng.integers(0, 320, n + 8).astype(np.int32) for n in lens]
    steps = [[(i, toks[i][:n], [n - 1] if i != 2 else [n - 1, 0, n - 1]) for i, n in enumerate(lens)],
             [(4, None, [0]), (0, toks[0][lens[0]:lens[0] + 2], []), (3, None, [0]), (1, toks[1][3:4], [0])],
             [(2, None, [0]), (4, None, [0])],
             [(0, toks[0][:1], [0]), (1, None, [0]), (2, toks[2][:1], [0]), (3, toks[3][:1], [0])],
             [(3, None, [0])]]
    last = {}
    for entries in steps:
        rows = sum(len(x[2]) for x in entries)
        lg, am = torch.full((rows, 320), float("nan"), device="cuda"), torch.full((rows,), -1, dtype=torch.int32, device="cuda")
        w.batch([(seqs[i], t, want) for i, t, want in entries], logits=lg, argmax=am)
        lg1, at = torch.empty((rows, 320), device="cuda"), 0
        for i, t, want in entries:
            w1.batch([(seqs1[i], np.array([last[i]], dtype=np.int32) if t is None else t, want)], logits=lg1[at:at + len(want)], argmax=None)
            at += len(want)
            if want:
                last[i] = int(am[at - 1])
        a, b = lg.double().cpu().numpy(), lg1.double().cpu().numpy()
        assert (am.cpu().numpy() == a.argmax(-1)).all()
        for r in range(rows):
            assert ((a[r] - b[r]) ** 2).sum() < 1e-3 * (b[r] ** 2).sum(), (r, ((a[r] - b[r]) ** 2).sum() / (b[r] ** 2).sum())
        assert [w.seq_len(s) for s in seqs] == [w1.seq_len(s) for s in seqs1]
    # the device's own counters are where the sequences are: a single step behind the batches
    tok, out, out1 = torch.tensor([5], dtype=torch.int32, device="cuda"), torch.empty(320, device="cuda"), torch.empty(320, device="cuda")
    for m, s, o in ((w, seqs, out), (w1, seqs1, out1)):
        m.set_seq(s[1])
        m.step(token=tok, logits=o)
    a, b = out.double().cpu().numpy(), out1.double().cpu().numpy()
    assert ((a - b) ** 2).sum() < 1e-3 * (b ** 2).sum()
    w.close()
    w1.close()


@pytest.mark.parametrize("arch,lens,max_tokens", [(0, [20, 17, 31, 3, 1], 64), (1, [30] * 5, 256), (0, [32, 31, 30, 9] * 2, 100), (0, [1] * 40, 64), (0, [13, 20], 33)])
def test_batches_of_short_portions_in_wide_passes(E, arch, lens, max_tokens):
    """More rows of short portions than one small pass takes go through the prompt GEMM with 8-bit activations, portions cut where passes end; then a token of every sequence. Against the same
    portions one at a time: the same arithmetic with other summation orders (the bound of the comparisons above)."""
    torch = E.torch
    rng = np.random.default_rng(len(lens))
    d = tiny_model(rng, arch=arch, n_layer=2, n_embd=512, n_head=4, n_head_kv=2, n_ff=1024, n_vocab=320, n_ctx=64, rope_freqs=arch == 0)
    ws = []
    for _ in range(2):
        w = E.Window(_hp(d), n_ctx=64)
        w.load_desc(d)
        w.finalize_pool(max_tokens, len(lens), len(lens) * 64)
        ws.append((w, [w.seq_new() for _ in lens]))
    (w, seqs), (w1, seqs1) = ws
    for k in range(2):
        part = [rng.integers(0, 320, n if k == 0 else 1).astype(np.int32) for n in lens]
        lg, lg1 = torch.full((len(lens), 320), float("nan"), device="cuda"), torch.empty((len(lens), 320), device="cuda")
        w.batch([(q, t, [len(t) - 1]) for q, t in zip(seqs, part)], logits=lg)
        for i, t in enumerate(part):
            w1.batch([(seqs1[i], t, [len(t) - 1])], logits=lg1[i:i + 1])
        a, b = lg.double().cpu().numpy(), lg1.double().cpu().numpy()
        err = ((a - b) ** 2).sum(-1) / (b ** 2).sum(-1)
        assert (err < 1e-3).all(), (k, err.max())
    w.close()
    w1.close()


def _heads_of_128(E, n_ctx, n_seq, n_head, windows=2):
    """windows over one model of heads of 128 (two heads are a block of the wo product's activations), with sequences"""
    d = tiny_model(np.random.default_rng(n_ctx), n_layer=2, n_embd=128 * n_head, n_head=n_head, n_head_kv=2, n_ff=512, n_vocab=320, n_ctx=n_ctx, rope_freqs=True)
    ws = []
    for _ in range(windows):
        w = E.Window(_hp(d), n_ctx=n_ctx)
        w.load_desc(d)
        w.finalize_pool(64, n_seq, n_seq * n_ctx)
        ws.append((w, [w.seq_new() for _ in range(n_seq)]))
    return ws


@pytest.mark.parametrize("lens,n_ctx", [([1, 62, 63, 64, 2, 30], 72), ([63, 126, 127, 128, 1, 64], 136), ([150, 128, 3, 64, 127, 63], 256), ([129, 7], 200)])
def test_rows_beside_others_keep_their_attention(E, lens, n_ctx):
    """single tokens of several sequences, heads of 128 quantized where they are made: rows on both sides of 64 and 128 cells, caches of fewer cells than a form takes. The same
    in whatever company, but for the order of the head's sums."""
    torch = E.torch
    (w, s), (w1, s1) = _heads_of_128(E, n_ctx, len(lens), 4)
    rng = np.random.default_rng(sum(lens))
    for i, n in enumerate(lens):
        t = rng.integers(0, 320, n).astype(np.int32)
        for m, q in ((w, s), (w1, s1)):
            m.batch([(q[i], t, [n - 1])], logits=torch.empty((1, 320), device="cuda"))
    for _ in range(2):
        toks = rng.integers(0, 320, len(lens)).astype(np.int32)
        lg, lg1 = torch.full((len(lens), 320), float("nan"), device="cuda"), torch.empty((len(lens), 320), device="cuda")
        w.batch([(q, toks[i:i + 1], [0]) for i, q in enumerate(s)], logits=lg)
        for i in range(0, len(lens), 2):
            w1.batch([(s1[j], toks[j:j + 1], [0]) for j in (i, i + 1)], logits=lg1[i:i + 2])
        assert torch.isfinite(lg).all() and (lg - lg1).abs().max() <= 512 * 2.0 ** -24 * lg1.abs().max()      # (n_embd f32 sums of the head; a turned 8-bit rounding is 1 / 127 of a value)
    w.close()
    w1.close()


@pytest.mark.parametrize("n_head", [2, 4, 8])
@pytest.mark.parametrize("past,T", [(200, 2), (191, 5), (130, 31), (255, 32), (250, 33)])
def test_small_portions_behind_histories_of_heads_of_128(E, past, T, n_head):
    """a portion of up to 32 tokens on the matrix cores, two heads of a KV head per workgroup (n_head 2: a head each, the launch that quantizes); against the tokens one after the other: the same
    arithmetic with other summation orders (the bound of the comparisons above)"""
    torch = E.torch
    (w, s), (w1, s1) = _heads_of_128(E, 320, 1, n_head)
    rng = np.random.default_rng(past + T)
    t, more = rng.integers(0, 320, past).astype(np.int32), rng.integers(0, 320, T).astype(np.int32)
    lg, lg1 = torch.full((T, 320), float("nan"), device="cuda"), torch.empty((T, 320), device="cuda")
    for m, q in ((w, s), (w1, s1)):
        m.batch([(q[0], t, [past - 1])], logits=torch.empty((1, 320), device="cuda"))
    w.batch([(s[0], more, list(range(T)))], logits=lg)
    for i in range(T):
        w1.batch([(s1[0], more[i:i + 1], [0])], logits=lg1[i:i + 1])
    a, b = lg.double().cpu().numpy(), lg1.double().cpu().numpy()
    assert (((a - b) ** 2).sum(-1) < 1e-3 * (b ** 2).sum(-1)).all()
    w.close()
    w1.close()


@pytest.mark.parametrize("n_vocab", [320, 4097, 20011, 140001])
def test_greedy_token_is_the_first_of_equal_maxima_over_many_workgroups(E, n_vocab):
    """result_norm + lm_head + argmax: rows of the vocabulary are shared by up to 32 workgroups; equal rows of the head (equal logits to the bit) in several of their parts - the first one
    wins; a token that ends a step also moves the position counter."""
    torch = E.torch
    rng = np.random.default_rng(n_vocab)
    d = tiny_model(rng, n_layer=1, n_vocab=320, n_ctx=32, rope_freqs=True)
    w = E.Window(dict(_hp(d), n_vocab=n_vocab), n_ctx=32)
    from _bind import rand_blocks, row_size
    for name, kind in (("attn_norm", E.T_ATTN_NORM), ("wq", E.T_WQ), ("wk", E.T_WK), ("wv", E.T_WV), ("wo", E.T_WO), ("ffn_norm", E.T_FFN_NORM), ("ffn_gate", E.T_FFN_GATE),
                       ("ffn_up", E.T_FFN_UP), ("ffn_down", E.T_FFN_DOWN)):
        t = getattr(d, name)[0]
        k, n = dict(attn_norm=(256, 1), wq=(256, 256), wk=(256, 128), wv=(256, 128), wo=(256, 256), ffn_norm=(256, 1), ffn_gate=(256, 512), ffn_up=(256, 512), ffn_down=(512, 256))[name]
        w._chk(w.lib.pm355_model_set_tensor(w.h, kind, 0, t.type, t.data, E.L.row_size(t.type, k) * n), name)
    rs = row_size(Q4_K, 256)
    emb, head = rand_blocks(Q4_K, 512, 256, rng), rand_blocks(Q4_K, n_vocab, 256, rng).reshape(n_vocab, rs)
    w.set_tensor(E.T_TOK_EMBD, -1, Q4_K, np.resize(emb, n_vocab * rs))
    w.set_tensor(E.T_OUT_NORM, -1, E.F32, np.ones(256, dtype=np.float32))
    w.set_tensor(E.T_OUTPUT, -1, Q4_K, head)
    w.finalize(max_tokens=1)
    lg, am = torch.empty(n_vocab, device="cuda"), torch.empty(1, dtype=torch.int32, device="cuda")
    x = torch.randn((1, 256), generator=torch.Generator(device="cuda").manual_seed(1), device="cuda")
    w.head(x, logits=lg, argmax=am)
    assert int(am) == int((lg == lg.max()).nonzero()[0])
    best = int(am)
    for at in sorted({0, n_vocab // 3, 2 * n_vocab // 3, n_vocab - 1} - {best}, reverse=True):       # the same row again, each time further in front or behind
        head[at] = head[best]
        w.set_tensor(E.T_OUTPUT, -1, Q4_K, head)
        torch.cuda.synchronize()                           # (the uploader's stream)
        w.head(x, logits=lg, argmax=am)
        top = (lg == lg.max()).nonzero()[:, 0]
        assert at in top.tolist() and best in top.tolist() and int(am) == int(top[0])
    tok = torch.zeros(1, dtype=torch.int32, device="cuda")
    w.set_pos(0)
    outs = []
    for i in range(3):                                     # captured once, replayed: the position moves on its own
        tok.fill_(3 + i)
        w.step(token=tok, logits=lg, argmax=am)
        torch.cuda.synchronize()
        outs.append(lg.clone())
        assert int(am) == int((lg == lg.max()).nonzero()[0])
    for pos in (1, 0):                                     # without the argmax: the same token behind the same single one, and behind none
        w.set_pos(pos)
        tok.fill_(4)
        w.step(token=tok, logits=lg)
        torch.cuda.synchronize()
        assert torch.equal(lg, outs[1]) == (pos == 1)
    w.close()


def _pool_window(E, d, n_ctx, max_tokens, n_seq, n_vocab=None):
    w = E.Window(dict(_hp(d), n_vocab=n_vocab or d.n_vocab), n_ctx=n_ctx)
    w.load_desc(d)
    w.finalize_pool(max_tokens, n_seq, n_seq * n_ctx)
    return w


def _batch(E, w, entries, argmax=False):
    """logits of the wanted rows (and greedy tokens) of one batch"""
    rows = sum(len(e[2]) for e in entries)
    lg, am = E.torch.full((rows, w.n_vocab), float("nan"), device="cuda"), E.torch.full((rows,), -1, dtype=E.torch.int32, device="cuda")
    w.batch(entries, logits=lg, argmax=am if argmax else None)
    return (lg, am) if argmax else lg


def test_heads_on_two_streams(E):
    """the head on the caller's own logits and index shares nothing between calls: two streams at once, a vocabulary of many workgroups"""
    torch = E.torch
    rng = np.random.default_rng(14)
    n_vocab = 131072
    d = tiny_model(rng, n_layer=1, n_vocab=320, n_ctx=32)
    w = E.Window(dict(_hp(d), n_vocab=n_vocab), lo=0, hi=0, flags=E.HAS_HEAD, n_ctx=32)
    w._chk(w.lib.pm355_model_set_tensor(w.h, E.T_OUT_NORM, -1, d.out_norm.type, d.out_norm.data, 256 * 4), "out_norm")
    w.fill_tensor(E.T_OUTPUT, -1, Q4_K, 5, 1.0)
    w.finalize(max_tokens=1)
    x = torch.randn((2, 256), generator=torch.Generator(device="cuda").manual_seed(2), device="cuda")
    want = []
    for r in range(2):
        lg = torch.empty(n_vocab, device="cuda")
        w.head(x[r:r + 1], logits=lg)
        want.append(int((lg == lg.max()).nonzero()[0]))
    assert want[0] != want[1]
    n, streams, graphs = 100, [torch.cuda.Stream() for _ in range(2)], []
    lg, am = torch.empty((2, n_vocab), device="cuda"), torch.full((2, n), -1, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    for r, st in enumerate(streams):                       # (captured: back to back on the device)
        graphs.append(torch.cuda.CUDAGraph())
        with torch.cuda.graph(graphs[r], stream=st):
            for i in range(n):
                w.head(x[r:r + 1], logits=lg[r], argmax=am[r, i:])
    for _ in range(5):
        am.fill_(-1)
        torch.cuda.synchronize()
        for g, st in zip(graphs, streams):
            with torch.cuda.stream(st):
                g.replay()
        torch.cuda.synchronize()
        assert [int(am[r].ne(want[r]).sum()) for r in range(2)] == [0, 0]
    w.close()


def test_a_refused_batch_leaves_the_positions(E):
    """the head is refused (the window has none yet): the sequences stay where they were, on the host and on the device"""
    torch = E.torch
    rng = np.random.default_rng(13)
    d = tiny_model(rng, n_layer=1, n_embd=256, n_head=4, n_head_kv=2, n_ff=512, n_vocab=320, n_ctx=64)
    toks = rng.integers(0, 320, (2, 6)).astype(np.int32)
    outs = []
    for head in (True, False):
        w = E.Window(_hp(d), n_ctx=64)
        w.flags = E.HAS_EMBD | (E.HAS_HEAD if head else 0)  # (the wrapper's: what it loads)
        w.load_desc(d)
        w.finalize_pool(16, 2, 128)
        s = [w.seq_new() for _ in range(2)]
        if not head:
            with pytest.raises(E.L.PM355Error, match="head"):
                _batch(E, w, [(q, t, (5,)) for q, t in zip(s, toks)])
            assert [w.seq_len(q) for q in s] == [0, 0]
            w._chk(w.lib.pm355_model_set_tensor(w.h, E.T_OUT_NORM, -1, d.out_norm.type, d.out_norm.data, 256 * 4), "out_norm")
            w._chk(w.lib.pm355_model_set_tensor(w.h, E.T_OUTPUT, -1, d.output.type, d.output.data, E.L.row_size(d.output.type, 256) * 320), "output")
            torch.cuda.synchronize()
        lg = torch.empty(320, device="cuda")
        for q in s:
            w.set_seq(q)
            w.step(token=torch.from_numpy(toks[q][:1]).cuda(), logits=lg, use_graph=False)
            outs.append(lg.clone())
        w.close()
    assert torch.equal(outs[0], outs[2]) and torch.equal(outs[1], outs[3])


@pytest.mark.parametrize("n_vocab", [320, 4099])
def test_positions_behind_a_portion_cut_into_passes(E, n_vocab):
    """20 tokens with scratch for 8: pieces of one sequence that meet in a pass; a step behind them continues where the sequence ends (the device's counter), and so does the next portion"""
    torch = E.torch
    rng = np.random.default_rng(15)
    d = tiny_model(rng, n_layer=2, n_embd=512, n_head=8, n_head_kv=2, n_ff=1024, n_vocab=n_vocab, n_ctx=64, rope_freqs=True)
    toks = rng.integers(0, n_vocab, (3, 21)).astype(np.int32)
    outs = []
    for together in (True, False):
        w = _pool_window(E, d, 64, 8, 3)
        s = [w.seq_new() for _ in range(3)]
        entries = [(q, t[:n], ()) for q, t, n in zip(s, toks, (20, 20, 13))]
        for e in [entries] if together else [[x] for x in entries]:
            w.batch(e)
        lg = torch.empty((3, n_vocab), device="cuda")
        for i, q in enumerate(s):
            w.set_seq(q)
            w.step(token=torch.from_numpy(toks[i][-1:]).cuda(), logits=lg[i], use_graph=False)
        outs.append(lg.double().cpu().numpy())
        w.close()
    for a, b in zip(*outs):
        assert ((a - b) ** 2).sum() < 1e-3 * (b ** 2).sum()


@pytest.mark.parametrize("lens", [(3, 40), (40, 3), (3, 4), (1, 1)])
def test_the_last_portion_of_a_batch_is_the_current_sequence(E, lens):
    """whichever pass it ran in"""
    torch = E.torch
    rng = np.random.default_rng(16)
    d = tiny_model(rng, n_layer=1, n_embd=256, n_head=4, n_head_kv=2, n_ff=512, n_vocab=320, n_ctx=64)
    w = _pool_window(E, d, 64, 64, 3)
    s = [w.seq_new() for _ in lens]
    w.batch([(q, rng.integers(0, 320, n), ()) for q, n in zip(s, lens)])
    a, b = torch.empty(320, device="cuda"), torch.empty(320, device="cuda")
    w.step(token=torch.tensor([7], dtype=torch.int32, device="cuda"), logits=a, use_graph=False)
    assert [w.seq_len(q) for q in s] == [lens[0], lens[1] + 1]
    w.set_seq_pos(s[1], lens[1])
    w.set_seq(s[1])
    w.step(token=torch.tensor([7], dtype=torch.int32, device="cuda"), logits=b, use_graph=False)
    assert torch.equal(a, b)
    w.close()


def test_portions_keep_their_tier_where_only_some_layers_have_an_8_bit_path(E):
    """ffn_down of 65536 columns, Q6_K in the first layer and Q4_K in the second: Q4_K has the integer small-batch product, Q6_K has none. Portions of 16..32 tokens then run one layer on 16-bit and one on 8-bit activations; two of them in
    one step do as well, in passes of their size: the same bits as alone."""
    rng = np.random.default_rng(12)
    d = tiny_model(rng, n_layer=2, n_embd=512, n_head=8, n_head_kv=2, n_ff=65536, n_vocab=320, n_ctx=256, types=dict(attn_v=Q4_K))
    toks = rng.integers(0, 320, (2, 220)).astype(np.int32)
    w = _pool_window(E, d, 256, 64, 4)
    s = [w.seq_new() for _ in range(4)]
    for i, q in enumerate(s):
        w.batch([(q, toks[i % 2, 20:], ())])
    toks = toks[:, :20]
    alone = [_batch(E, w, [(s[i], toks[i], (19,))]) for i in range(2)]
    both = _batch(E, w, [(s[2 + i], toks[i], (19,)) for i in range(2)])
    assert E.torch.equal(both, E.torch.cat(alone))
    w.close()


@pytest.mark.parametrize("arch", [0, 1])
def test_a_portion_does_not_depend_on_the_histories_beside_it(E, arch):
    """A sequence's rows next to short and to long histories: the pass has the same rows, so the same products, and the attention of a row is chosen by its own sequence - equal bits"""
    rng = np.random.default_rng(3 + arch)
    d = tiny_model(rng, arch=arch, n_layer=2, n_embd=512, n_head=8, n_head_kv=2, n_ff=1024, n_vocab=320, n_ctx=448, types=dict(attn_v=Q6_K))
    toks = rng.integers(0, 320, 448).astype(np.int32)
    got = {}
    for other in (5, 250, 420):                            # cells of the sequence beside them
        w = _pool_window(E, d, 448, 64, 4)
        a, b, c = (w.seq_new() for _ in range(3))
        w.batch([(a, toks[:10], ())])
        w.batch([(b, toks[:other], ())])
        got[other] = [_batch(E, w, [(a, toks[i:i + 1], (0,)), (b, toks[i:i + 1], (0,))])[0] for i in range(10, 14)]
        got[other].append(_batch(E, w, [(c, toks[:20], (19,)), (b, toks[:1], ())]))
        w.close()
    for other in (250, 420):
        assert all(E.torch.equal(x, y) for x, y in zip(got[other], got[5])), other


def test_single_tokens_behind_long_histories_share_a_pass(E):
    """Decoded tokens behind 3, 350, 1500 and 2900 cells in one pass: a workgroup per head, tiles of the matrix-core kernel and the key-split kernel side by side, wanted rows out of order.
    Against the same tokens one sequence at a time (the same arithmetic, other summation orders: the bound of the comparisons above), step by step."""
    torch = E.torch
    rng = np.random.default_rng(17)
    lens = [2900, 3, 1500, 350, 2870]
    d = tiny_model(rng, n_layer=2, n_embd=512, n_head=8, n_head_kv=2, n_ff=1024, n_vocab=320, n_ctx=2944, rope_freqs=True)
    toks = rng.integers(0, 320, (len(lens), 2944)).astype(np.int32)
    ws = []
    for _ in range(2):
        w = _pool_window(E, d, 2944, 512, len(lens))
        s = [w.seq_new() for _ in lens]
        for i, n in enumerate(lens):
            w.batch([(s[i], toks[i, :n], ())])
        ws.append((w, s))
    for step in range(4):
        (w, s), (w1, s1) = ws
        some = [i for i in range(len(lens)) if not (step == 2 and i == 1)]
        a = _batch(E, w, [(s[i], toks[i, lens[i] + step:lens[i] + step + 1], (0,)) for i in some]).double()
        b = torch.cat([_batch(E, w1, [(s1[i], toks[i, lens[i] + step:lens[i] + step + 1], (0,))]) for i in some]).double()
        off = (a - b).square().sum(-1) / b.square().sum(-1)
        assert bool((off < 1e-3).all()), (step, off.tolist())
    for w, _ in ws:
        w.close()


def test_large_batches_of_several_sequences(E):
    """Portions of up to 600 tokens in passes of 512 rows: tables of more than one launch's arguments, rope + store by token with a position and a sequence per row, tiles of 64 and 128
    queries, argmax over rows that several workgroups share (odd vocabulary: rows that do not start on 16 bytes). Against one sequence at a time; then the same captured on a stream and
    replayed after the host's arrays are gone."""
    torch = E.torch
    rng = np.random.default_rng(18)
    lens, V, n_ctx = [600, 33, 290, 431, 50], 4099, 640
    d = tiny_model(rng, n_layer=2, n_embd=1024, n_head=16, n_head_kv=4, n_ff=1024, n_vocab=V, n_ctx=n_ctx, rope_freqs=True)
    toks = [rng.integers(0, V, n).astype(np.int32) for n in lens]
    st = torch.cuda.Stream()
    with torch.cuda.stream(st):
        w, w1 = (_pool_window(E, d, n_ctx, 512, len(lens)) for _ in range(2))
        s, s1 = ([m.seq_new() for _ in lens] for m in (w, w1))
        lg, am = _batch(E, w, [(q, t, (len(t) - 1, len(t) - 7)) for q, t in zip(s, toks)], argmax=True)
        lg1 = torch.cat([_batch(E, w1, [(q, t, (len(t) - 1, len(t) - 7))]) for q, t in zip(s1, toks)])
        assert torch.equal(am.long(), lg.argmax(-1))
        off = (lg - lg1).double().square().sum(-1) / lg1.double().square().sum(-1)
        assert bool((off < 1e-3).all()), off.tolist()
        assert [w.seq_len(q) for q in s] == lens
        for q in s:
            w.seq_free(q)
        s = [w.seq_new() for _ in lens]
        out = torch.zeros((2 * len(lens), V), device="cuda")
        g = torch.cuda.CUDAGraph()
        torch.cuda.synchronize()
        with torch.cuda.graph(g, stream=st, capture_error_mode="relaxed"):
            w.batch([(q, t.copy(), (len(t) - 1, len(t) - 7)) for q, t in zip(s, toks)], logits=out)
        junk = [np.full(1 << 16, 0x7f7f7f7f, dtype=np.int32) for _ in range(64)]      # (what the call allocated is someone else's by now)
        for _ in range(3):
            out.zero_()
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, lg)
            torch.cuda.synchronize()
        del junk
    w.close()
    w1.close()


@pytest.mark.parametrize("arch,types,n_vocab", [(0, dict(attn_v=Q4_K), 320), (0, dict(attn_v=Q6_K), 4099), (0, {}, 320), (1, dict(attn_v=Q6_K), 4099), (0, dict(attn_v=Q4_K, output=Q4_K), 8197)])
def test_shared_passes_on_the_integer_products(E, arch, types, n_vocab):
    """Matrices of 512 columns and more take the integer small-batch products, with rope and KV store in the epilogue of wq | wk | wv (one launch for three matrices of a type, two parts for
    another wv, NEOX in a launch of its own), and the head the same for neighbouring rows: passes of 3, 8, 9, 17, 26 and 32 rows of several sequences against one sequence at a time."""
    torch = E.torch
    rng = np.random.default_rng(19 + arch)
    d = tiny_model(rng, arch=arch, n_layer=2, n_embd=1024, n_head=8, n_head_kv=2, n_ff=1536, n_vocab=n_vocab, n_ctx=224, types=types, rope_freqs=arch == 0)
    w, w1 = (_pool_window(E, d, 224, 64, 4) for _ in range(2))
    s, s1 = ([m.seq_new() for _ in range(4)] for m in (w, w1))
    for ns in ((1, 2, 0, 0), (3, 2, 1, 2), (1, 4, 3, 1), (5, 1, 9, 2), (8, 8, 2, 8), (14, 1, 16, 1), (32, 20, 12, 32), (31, 3, 40, 1), (1, 1, 1, 1), (1, 0, 1, 1)):
        entries = [(i, rng.integers(0, n_vocab, n).astype(np.int32), range(n - 1, max(n - 5, -1), -1) if i % 2 else (n - 1,)) for i, n in enumerate(ns) if n]
        a, am = _batch(E, w, [(s[i], t, want) for i, t, want in entries], argmax=True)
        b = torch.cat([_batch(E, w1, [(s1[i], t, want)]) for i, t, want in entries]).double()
        off = (a - b).square().sum(-1) / b.square().sum(-1)
        assert bool((off < 1e-3).all()), (ns, off.tolist())
        assert torch.equal(am.long(), a.argmax(-1))
    # equal rows of the head in several workgroups' parts: the first one wins in every row
    if n_vocab > 4096:
        best, k = int(am[0]), E.L.row_size(d.output.type, 1024)
        head = np.ctypeslib.as_array((np.ctypeslib.ctypes.c_uint8 * (k * n_vocab)).from_address(d.output.data)).reshape(n_vocab, k)
        head[[7, n_vocab - 1]] = head[best]
        w._chk(w.lib.pm355_model_set_tensor(w.h, E.T_OUTPUT, -1, d.output.type, d.output.data, k * n_vocab), "output")
        torch.cuda.synchronize()
        a, am = _batch(E, w, [(s[i], t, want) for i, t, want in entries], argmax=True)
        assert torch.equal(a[:, 7], a[:, -1]) and am.tolist() == a.cpu().numpy().argmax(-1).tolist() and 7 in am.tolist()
    w.close()
    w1.close()
