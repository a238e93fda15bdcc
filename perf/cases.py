"""What this framework is measured on: passes through engine.Window (quantized Llama / Qwen2 layer windows) and engine.Stack (layer-described models with dense weights) as a
program that serves them makes them. Layer shapes are the configurations of prima_cpp_amd/engine.py, bench_design.py and bench_keranex.py with fewer layers; weights are normal
values, quantized here; every sequence is random tokens.

kind "step": one decoded token on a filled cache (set_pos + step, replayed from the window's graph); "batch": one decode() call over `tokens` tokens behind `past` cached ones - a
speculative batch, a short prompt, a micro-batch of a long one; "serve": sequences through the batch interface - every prompt, then decoded tokens of all sequences, step by step
(the tokens come from the host, as from a sampler); "prompts": the sequences' prompts alone."""
import math

import numpy as np
import torch

from prima_cpp_amd import engine as E
from prima_cpp_amd import keranex, kudirax
from prima_cpp_amd.lib import BF16, F32, Q4_K, Q5_K, Q6_K, Q8_0

# the last one: the window of the engine tests
WINDOWS = {"8b": dict(E.LLAMA3_8B), "70b": dict(E.LLAMA3_70B), "72b": dict(E.QWEN25_72B),
           "toy": dict(arch=0, n_layer=2, n_embd=256, n_head=4, n_head_kv=2, head_dim=64, n_ff=512, n_vocab=320, rms_eps=1e-5, rope_freq_base=10000.0)}
DENSE = {"1b": dict(W=2048, H=32, G=8, d=64, F=8192, vocab=32000), "4b": dict(W=4096, H=32, G=8, d=128, F=14336, vocab=32000)}
LATENT = {"1b": dict(W=2048, H=32, d=64, rot=32, qr=768, kr=512, inner=4096, state=16, dt=128, E=32, top=4, ff=2048, vocab=32000),
          "4b": dict(W=4096, H=32, d=128, rot=64, qr=1536, kr=512, inner=8192, state=16, dt=256, E=32, top=4, ff=3584, vocab=32000)}


def listed():
    return [
        # the smallest model there is: a token is all launches and no work
        dict(name="toy_step", kind="step", model="toy", mix="q4_k_m", layers=2, head=True, past=20),
        # chat with the 8B file type that most people download: one token, short history
        dict(name="8b_step", kind="step", model="8b", mix="q4_k_m", layers=8, head=True, past=203),
        # a rank of the ring on the headline model: its layers only, activations in and out
        dict(name="70b_step", kind="step", model="70b", mix="q4_k_m", layers=3, head=False, past=611),
        # a long document in the cache, the other file type and architecture (rope pairs apart, biases, Q8_0 ffn_down)
        dict(name="72b_step_long", kind="step", model="72b", mix="q6_k", layers=2, head=False, past=8203),
        # speculative decoding: eight drafted tokens verified at once
        dict(name="70b_batch_8", kind="batch", model="70b", mix="q4_k_m", layers=3, head=False, tokens=8, past=403),
        # a short question: all of it in one small batch, odd size
        dict(name="72b_batch_23", kind="batch", model="72b", mix="q6_k", layers=2, head=False, tokens=23, past=0),
        # an ordinary chat message behind a system prompt
        dict(name="8b_batch_101", kind="batch", model="8b", mix="q4_k_m", layers=4, head=True, tokens=101, past=300),
        # a micro-batch of 512 tokens in the middle of a prompt, on a rank of the ring
        dict(name="70b_batch_512", kind="batch", model="70b", mix="q4_k_m", layers=3, head=False, tokens=512, past=1024),
        # a long document read in one pass
        dict(name="8b_batch_6001", kind="batch", model="8b", mix="q4_k_m", layers=4, head=True, tokens=6001, past=0),
        # eight users of the 8B model at once
        dict(name="8b_serve_8", kind="serve", model="8b", mix="q4_k_m", layers=8, seqs=8, prompt=24, steps=12),
        # six users of the dense design: prompts of unequal length, then their tokens
        dict(name="kudirax_serve_6", kind="serve", model="kudirax_4b", mix="bf16", layers=3, seqs=6, prompt=180, steps=12),
        # the same for latent attention, scans and experts
        dict(name="keranex_serve_5", kind="serve", model="keranex_1b", mix="bf16", layers=4, seqs=5, prompt=150, steps=12),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "step", "batch", "batch", "batch", "serve", "dense", "dense"])
    if kind == "dense":
        model = rng.choice(["kudirax_1b", "kudirax_4b", "keranex_1b"])
        mix = rng.choice(["bf16", "bf16", "bf16", "f32"]) if model == "kudirax_1b" else "bf16"
        if rng.random() < 0.4:
            return dict(kind="prompts", model=model, mix=mix, layers=rng.choice([2, 3]), seqs=rng.choice([1, 1, 2]), prompt=_log_uniform(rng, 70, 2048 if mix == "bf16" else 300))
        return dict(kind="serve", model=model, mix=mix, layers=rng.choice([2, 3]), seqs=_log_uniform(rng, 1, 20), prompt=_log_uniform(rng, 5, 200), steps=rng.randint(6, 12))
    if kind == "serve":
        return dict(kind="serve", model=rng.choice(["toy", "8b", "8b"]), mix=rng.choice(["q4_k_m", "q6_k", "q8_0"]), layers=2, seqs=_log_uniform(rng, 2, 24), prompt=_log_uniform(rng, 3, 70),
                    steps=rng.randint(5, 8))
    model = rng.choice(["8b", "8b", "70b", "72b"])
    c = dict(kind=kind, model=model, mix=rng.choice(["q4_k_m", "q6_k"] + (["q8_0"] if model == "8b" else [])), layers=rng.choice([1, 2]), head=rng.random() < 0.3)
    if kind == "step":
        return dict(c, past=_log_uniform(rng, 8, 12000))
    tokens = _log_uniform(rng, 2, 6000 if model == "8b" else 1200)
    return dict(c, tokens=tokens, past=rng.choice([0, _log_uniform(rng, 16, 2000)]))


# ---- quantized blocks: the GGUF formats, written from normal weights and read back in 64 bits ---------------------------------------------------------------------------------
def _mixture(hp, mix, il):
    """types of a layer's matrices: (wq, wk, wo, gate, up), wv, down - the file types as their quantizer mixes them"""
    n = hp["n_layer"]
    if mix == "q4_k_m":
        more = il < n // 8 or il >= 7 * n // 8 or (il - n // 8) % 3 == 2
        big = n == 80 and hp["n_head"] // hp["n_head_kv"] == 8
        t = (Q4_K, Q6_K if more else (Q5_K if big else Q4_K), Q6_K if more else Q4_K)
    else:
        t = (Q6_K,) * 3 if mix == "q6_k" else (Q8_0,) * 3
    return t if hp["n_ff"] % 256 == 0 else (t[0], t[1], Q8_0)


def _f16(x):
    return x.to(torch.float16)


def _bytes(x):
    return x.contiguous().view(torch.uint8)


def _pack_6bit(sc, mn):
    """scales and minima of 8 sub-blocks, 6 bits each -> 12 bytes"""
    lo = torch.cat([sc[..., :4] | (sc[..., 4:] >> 4 << 6), mn[..., :4] | (mn[..., 4:] >> 4 << 6)], -1)
    return torch.cat([lo, (sc[..., 4:] & 15) | ((mn[..., 4:] & 15) << 4)], -1)


def _unpack_6bit(b):
    sc = torch.cat([b[..., :4] & 63, (b[..., 8:] & 15) | (b[..., :4] >> 6 << 4)], -1)
    return sc, torch.cat([b[..., 4:8] & 63, (b[..., 8:] >> 4) | (b[..., 4:8] >> 6 << 4)], -1)


def _quantize(t, w):
    """f32 [N, K] -> the bytes of its rows in blocks of type t"""
    N, K = w.shape
    if t == Q8_0:
        b = w.view(N, -1, 32)
        d = _f16(b.abs().amax(-1, keepdim=True) / 127)
        q = (b / d.float()).round_().clamp_(-127, 127).to(torch.int8)
        return torch.cat([_bytes(d).view(N, -1, 2), _bytes(q).view(N, -1, 32)], -1).view(N, -1)
    if t == Q6_K:
        b = w.view(N, -1, 16, 16)
        s = b.abs().amax(-1) / 31
        d = _f16(s.amax(-1, keepdim=True) / 127)
        sc = (s / d.float()).round_().clamp_(1, 127)
        q = ((b / (sc * d.float()).unsqueeze(-1)).round_().clamp_(-32, 31) + 32).to(torch.uint8).view(N, -1, 2, 4, 32)
        ql = torch.stack([(q[..., 0, :] & 15) | ((q[..., 2, :] & 15) << 4), (q[..., 1, :] & 15) | ((q[..., 3, :] & 15) << 4)], -2)
        qh = (q[..., 0, :] >> 4) | (q[..., 1, :] >> 4 << 2) | (q[..., 2, :] >> 4 << 4) | (q[..., 3, :] >> 4 << 6)
        return torch.cat([ql.reshape(N, -1, 128), qh.reshape(N, -1, 64), _bytes(sc.to(torch.int8)).view(N, -1, 16), _bytes(d).view(N, -1, 2)], -1).view(N, -1)
    top = 15 if t == Q4_K else 31
    b = w.view(N, -1, 8, 32)
    lo = b.amin(-1).clamp_(max=0).neg_()
    s = (b.amax(-1) + lo) / top
    d, dm = _f16(s.amax(-1, keepdim=True) / 63), _f16(lo.amax(-1, keepdim=True) / 63)
    sc, mn = (s / d.float()).round_().clamp_(1, 63), (lo / dm.float()).round_().clamp_(0, 63)
    q = ((b + (mn * dm.float()).unsqueeze(-1)) / (sc * d.float()).unsqueeze(-1)).round_().clamp_(0, top).to(torch.uint8).view(N, -1, 4, 2, 32)
    parts = [_bytes(d).view(N, -1, 2), _bytes(dm).view(N, -1, 2), _pack_6bit(sc.to(torch.uint8), mn.to(torch.uint8))]
    if t == Q5_K:
        bit = torch.arange(8, dtype=torch.uint8, device=w.device).view(4, 2, 1)
        parts.append((q >> 4 << bit).sum((-3, -2), dtype=torch.uint8))
    parts.append(((q[..., 0, :] & 15) | ((q[..., 1, :] & 15) << 4)).reshape(N, -1, 128))
    return torch.cat(parts, -1).view(N, -1)


BLOCK_BYTES = {Q4_K: 144, Q5_K: 176, Q6_K: 210, Q8_0: 34}


def _row_bytes(t, K):
    return K // (32 if t == Q8_0 else 256) * BLOCK_BYTES[t]


def _dequantize(t, rows):
    """the values of such rows, f64 [N, K]"""
    N = rows.shape[0]
    b = rows.view(N, -1, BLOCK_BYTES[t])
    f16 = lambda x: x.contiguous().view(torch.float16).double()  # noqa: E731
    if t == Q8_0:
        return (f16(b[..., :2]) * b[..., 2:].contiguous().view(torch.int8).double()).view(N, -1)
    if t == Q6_K:
        ql, qh = b[..., :128].reshape(N, -1, 2, 2, 32), b[..., 128:192].reshape(N, -1, 2, 32)
        q = torch.stack([(ql[..., 0, :] & 15) | ((qh & 3) << 4), (ql[..., 1, :] & 15) | ((qh >> 2 & 3) << 4), (ql[..., 0, :] >> 4) | ((qh >> 4 & 3) << 4),
                         (ql[..., 1, :] >> 4) | (qh >> 6 << 4)], -2).reshape(N, -1, 16, 16)
        s = b[..., 192:208].contiguous().view(torch.int8).double() * f16(b[..., 208:])
        return ((q.double() - 32) * s.unsqueeze(-1)).view(N, -1)
    sc, mn = _unpack_6bit(b[..., 4:16])
    qs = b[..., -128:].reshape(N, -1, 4, 1, 32)
    q = torch.cat([qs & 15, qs >> 4], -2)
    if t == Q5_K:
        bit = torch.arange(8, dtype=torch.uint8, device=rows.device).view(4, 2, 1)
        q = q | ((b[..., 16:48].reshape(N, -1, 1, 1, 32) >> bit & 1) << 4)
    v = q.reshape(N, -1, 8, 32).double() * (sc.double() * f16(b[..., :2])).unsqueeze(-1)
    return (v - (mn.double() * f16(b[..., 2:4])).unsqueeze(-1)).view(N, -1)


# ---- inputs, from the seed alone ---------------------------------------------------------------------------------------------------------------------------------------------
def _gen(seed, *what):
    k = seed
    for x in what:
        k = (k * 1000003 + x + 1) % (1 << 61)
    return torch.Generator(device="cuda").manual_seed(k)


def _normal(seed, what, shape, std=1.0, mean=0.0):
    return torch.randn(shape, generator=_gen(seed, *what), device="cuda") * std + mean


def _tokens(seed, what, n, vocab):
    return torch.randint(0, vocab, (n,), generator=_gen(seed, 77, what), device="cuda", dtype=torch.int32)


def _lengths(case, seed):
    """prompt lengths of a serving case: unequal, around case["prompt"]; the first is the longest that any seed has"""
    r = np.random.RandomState(seed % (1 << 31))
    n = case["prompt"]
    return [n] + [int(r.randint(max(1, n // 2), n + 1)) for _ in range(case["seqs"] - 1)]


def _hp(case):
    return WINDOWS[case["model"]]


def _layers(case):
    """which layers of the model: behind the first eighth, so that both kinds of layer of a mixture are among any three"""
    n = _hp(case)["n_layer"]
    lo = n // 8 + 1 if n > 8 else 0
    return range(lo, lo + case["layers"])


def _matrices(case, il):
    """(kind, type, N, K) of a layer's matrices"""
    hp = _hp(case)
    W, Eq, Ekv, F = hp["n_embd"], hp["n_head"] * hp["head_dim"], hp["n_head_kv"] * hp["head_dim"], hp["n_ff"]
    t, tv, td = _mixture(hp, case["mix"], il)
    return [(E.T_WQ, t, Eq, W), (E.T_WK, t, Ekv, W), (E.T_WV, tv, Ekv, W), (E.T_WO, t, W, Eq), (E.T_FFN_GATE, t, F, W), (E.T_FFN_UP, t, F, W), (E.T_FFN_DOWN, td, W, F)]


def _ends(case):
    """the embedding and the head"""
    hp = _hp(case)
    t = Q8_0 if case["mix"] == "q8_0" else Q6_K
    return [(E.T_TOK_EMBD, Q4_K if case["mix"] == "q4_k_m" else t, hp["n_vocab"], hp["n_embd"]), (E.T_OUTPUT, t, hp["n_vocab"], hp["n_embd"])]


def _matrix(seed, kind, il, t, N, K):
    return _quantize(t, _normal(seed, (kind, il), (N, K), 1.0 if kind == E.T_TOK_EMBD else K ** -0.5))


def _vectors(case, il):
    """(kind, size, mean, spread): norms, and the biases of the second architecture"""
    hp = _hp(case)
    v = [(E.T_ATTN_NORM, hp["n_embd"], 1.0, 0.1), (E.T_FFN_NORM, hp["n_embd"], 1.0, 0.1)]
    if hp["arch"] == 1:
        v += [(E.T_BQ, hp["n_head"] * hp["head_dim"], 0.0, 0.1), (E.T_BK, hp["n_head_kv"] * hp["head_dim"], 0.0, 0.1), (E.T_BV, hp["n_head_kv"] * hp["head_dim"], 0.0, 0.1)]
    return v


def _rope_factors(case, seed):
    hp = _hp(case)
    return 1 + 6 * torch.rand(hp["head_dim"] // 2, generator=_gen(seed, E.T_ROPE_FREQS), device="cuda") if hp["arch"] == 0 else None


def _design(case):
    """configuration of a layer-described model"""
    name, size = case["model"].split("_")
    if name == "kudirax":
        z = DENSE[size]
        mixer = dict(heads=z["H"], kv_heads=z["G"], dim=z["d"], vdim=z["d"], mask={"size": 8192}, scale=12.0 / z["d"], softcap=50.0, v_mix=True)
        return dict(architecture="Kudirax", width=z["W"], vocab=z["vocab"], norm={"eps": 1e-5},
                    layers=[dict(type="attention", mixer=mixer, mlp=dict(kind="dense", ff=z["F"]))] * case["layers"])
    z = LATENT[size]
    moe = {"kind": "moe", "expert": {"ff": z["ff"]}, "router": {"experts": z["E"], "top": z["top"], "groups": {"count": 4, "keep": 2}}}
    lat = dict(heads=z["H"], dim=z["d"], rot_dim=z["rot"], vdim=z["d"], q_rank=z["qr"], kv_rank=z["kr"], mask={"size": 4096}, rot={"base": 10000.0, "dims": z["rot"]},
               scale=(z["d"] + z["rot"]) ** -0.5)
    ssm = dict(inner=z["inner"], state=z["state"], dt_rank=z["dt"], conv=4)
    layers = [dict(type="mamba1", mixer=ssm, mlp=moe) if i % 2 else dict(type="latent_attention", mixer=dict(lat, kv_from=i - 2) if i % 4 else lat, mlp=moe) for i in range(case["layers"])]
    return dict(architecture="Keranex", width=z["W"], vocab=z["vocab"], norm={"eps": 1e-5}, embedding={"bigram": {"buckets": 50021, "mul_prev": 1009, "mul_cur": 31}}, layers=layers)


CODE = 8  # entries of the residual stream of a model with experts that say which kind of token this is: the routers read them, the sublayers leave them alone


def _design_tensors(config):
    """(engine kind, layer, part, name, shape) of every tensor"""
    mod = kudirax if config["architecture"] == "Kudirax" else keranex
    for row in mod.tensors(config):
        yield row if len(row) == 5 else (row[0], row[1], 0, row[2], row[3])


def _design_tensor(config, seed, kind, il, part, name, shape):
    """f32 values of a tensor: matrices keep a row's size, and a trained router decides clearly"""
    what, leaf = (kind, il, part), name.split(".", 1)[-1]
    code = slice(0, CODE) if config["architecture"] == "Keranex" else slice(0, 0)
    W = config["width"]
    if leaf == "mlp.router":
        w = _normal(seed, what, shape, 0.02 * W ** -0.5)
        order = torch.rand((CODE, shape[0]), generator=_gen(seed, 5, *what), device="cuda").argsort(-1).float()
        w[:, code] = ((order / (shape[0] - 1) * 2 - 1) * (0.5 * shape[0] * W ** -0.5)).T
        return w
    if leaf == "mix.A_log":
        return (0.3 + 5.7 * torch.rand(shape, generator=_gen(seed, *what), device="cuda")).log()
    std, mean = 0.2, 0.0
    if name.endswith(("norm1", "norm2", "norm1b", "norm2b", "final.norm", "dq.norm", "dkv.norm")) or leaf in ("mix.D", "mix.vmix", "mix.sink"):
        mean = 0.5 if leaf == "mix.vmix" else 1.0
    elif leaf == "mix.dt.b":
        std, mean = 1.0, -2.5
    elif leaf == "mix.conv":
        std = 0.6
    elif name in ("embed", "bigram"):
        std = 1.0 if name == "embed" else 0.7
    elif len(shape) == 2:
        std = shape[1] ** -0.5
    w = _normal(seed, what, shape, std, mean)
    if config["architecture"] == "Keranex":
        if name in ("embed", "bigram", "head"):
            w[:, code] = 0.0
        if name == "embed":
            at = torch.arange(shape[0], device="cuda")
            w[at, at % CODE] = 0.5 * W ** 0.5
        if name.endswith(("norm1b", "norm2b")):
            w[code] = 0.0
        elif name.endswith((".dq", ".dkv", "mix.in", ".up")):
            w[:, code] = 0.0
    return w


# ---- the program's side ------------------------------------------------------------------------------------------------------------------------------------------------------
def _host(t):
    h = torch.empty(t.shape, dtype=t.dtype, pin_memory=True)
    h.copy_(t)
    return h.numpy()


def _prepare_design(case, seed):
    config = _design(case)
    dtype = {"bf16": "bfloat16", "f32": "float32"}[case["mix"]]
    m = (kudirax if config["architecture"] == "Kudirax" else keranex).build(config, dtype)
    for kind, il, part, name, shape in _design_tensors(config):
        w = _design_tensor(config, seed, kind, il, part, name, shape).to(torch.bfloat16)
        if w.dim() < 2 or dtype == "float32" or w.numel() < 4096:
            m.set_tensor(kind, il, F32, _host(w.float()), part)
        else:
            m.set_tensor(kind, il, BF16, _host(w.view(torch.int16)), part)
    return m


def _prepare_window(case, seed, n_ctx):
    hp, lay = _hp(case), _layers(case)
    ends = case["kind"] in ("serve", "prompts") or case["head"]
    m = E.Window(dict(hp), lay.start, lay.stop, (E.HAS_EMBD | E.HAS_HEAD) if ends else 0, n_ctx=n_ctx)
    for il in lay:
        for kind, t, N, K in _matrices(case, il):
            m.set_tensor(kind, il, t, _host(_matrix(seed, kind, il, t, N, K)))
        for kind, n, mean, amp in _vectors(case, il):
            m.set_tensor(kind, il, F32, _host(_normal(seed, (kind, il), (n,), amp, mean)))
    if ends:
        for kind, t, N, K in _ends(case):
            m.set_tensor(kind, -1, t, _host(_matrix(seed, kind, -1, t, N, K)))
        m.set_tensor(E.T_OUT_NORM, -1, F32, _host(_normal(seed, (E.T_OUT_NORM, -1), (hp["n_embd"],), 0.1, 1.0)))
    ff = _rope_factors(case, seed)
    if ff is not None:
        m.set_tensor(E.T_ROPE_FREQS, -1, F32, _host(ff))
    return m


def _is_design(case):
    return case["model"].startswith(("kudirax", "keranex"))


def _prepare_serve(case, seed):
    lens, steps = _lengths(case, seed), case.get("steps", 0)
    n_ctx = -(-(case["prompt"] + steps + 1) // 64) * 64
    if _is_design(case):
        m, vocab = _prepare_design(case, seed), _design(case)["vocab"]
        m.finalize_pool(2048, case["seqs"], case["seqs"] * n_ctx)
    else:
        m, vocab = _prepare_window(case, seed, n_ctx), _hp(case)["n_vocab"]
        m.finalize_pool(512, case["seqs"], case["seqs"] * n_ctx)
    toks = [_tokens(seed, i, n + steps, vocab).cpu().numpy() for i, n in enumerate(lens)]
    prompts = [(t[:n], (n - 1,)) for t, n in zip(toks, lens)]
    forced = [[(t[n + k:n + k + 1], (0,)) for t, n in zip(toks, lens)] for k in range(steps)]
    logits = torch.zeros((steps + 1, case["seqs"], vocab), device="cuda")
    return dict(kind="serve", m=m, rounds=[prompts] + forced, logits=logits)


def prepare(case, seed):
    torch.cuda.init()
    if case["kind"] in ("serve", "prompts"):
        return _prepare_serve(case, seed)
    hp, past = _hp(case), case["past"]
    n = case.get("tokens", 1)
    n_ctx = -(-(past + n + 1) // 64) * 64
    m = _prepare_window(case, seed, n_ctx)
    portion = min(past, 2048)
    m.finalize(max_tokens=max(n, portion, 1))
    # the whole sequence: tokens, or the activations that another rank hands on
    seq = _sequence(case, seed)
    for at in range(0, past, max(portion, 1)):  # the history is in the cache
        part = seq[at:min(at + portion, past)]
        m.decode(**{"tokens" if case["head"] else "x_in": part}, pos0=at, want_hidden=False, want_logits=False)
    s = dict(kind=case["kind"], m=m, head=case["head"], past=past, x=seq[past:].contiguous())
    if case["kind"] == "step":
        s["logits"] = torch.zeros(hp["n_vocab"], device="cuda") if case["head"] else None
        s["argmax"] = torch.zeros(1, dtype=torch.int32, device="cuda") if case["head"] else None
        s["out"] = torch.zeros((1, hp["n_embd"]), device="cuda")
    torch.cuda.synchronize()
    return s


def _sequence(case, seed):
    n = case["past"] + case.get("tokens", 1)
    hp = _hp(case)
    return _tokens(seed, 0, n, hp["n_vocab"]) if case["head"] else _normal(seed, (78,), (n, hp["n_embd"]))


def run(s):
    m = s["m"]
    if s["kind"] == "serve":
        seqs = [m.seq_new() for _ in s["rounds"][0]]
        for k, entries in enumerate(s["rounds"]):
            m.batch([(q, t, want) for q, (t, want) in zip(seqs, entries)], logits=s["logits"][k])
        for q in seqs:
            m.seq_free(q)
        return s["logits"]
    if s["kind"] == "step":
        m.set_pos(s["past"])
        m.step(**{"token" if s["head"] else "x_in": s["x"]}, x_out=s["out"], logits=s["logits"], argmax=s["argmax"])
        return [s["out"]] + ([s["logits"]] if s["head"] else [])  # (the greedy token follows from the logits; the two largest of random ones may lie within rounding)
    hidden, logits, _ = m.decode(**{"tokens" if s["head"] else "x_in": s["x"]}, pos0=s["past"])
    return [hidden] + ([logits] if s["head"] else [])


# ---- what a pass cannot do without --------------------------------------------------------------------------------------------------------------------------------------------
def work(case):
    """weights once per call of the model (of the experts: as many as the call's tokens can choose), the cached keys and values once, inputs and outputs; products and attention"""
    if case["kind"] in ("serve", "prompts"):
        rounds = [[(0, n) for n in _lengths(case, 1)]] + [[(n + k, 1) for n in _lengths(case, 1)] for k in range(case.get("steps", 0))]
    else:
        rounds = [[(case["past"], case.get("tokens", 1))]]
    flops = byts = 0
    for entries in rounds:
        T = sum(n for _, n in entries)
        pairs = sum(n * p + n * (n + 1) // 2 for p, n in entries)
        keys = sum(p + n for p, n in entries)
        if _is_design(case):
            config, size = _design(case), 2 if case["mix"] == "bf16" else 4
            W, V = config["width"], config["vocab"]
            byts += T * W * size + V * W * size + len(entries) * V * 4
            flops += 2 * len(entries) * V * W
            for layer in config["layers"]:
                x, ff = layer["mixer"], layer.get("mlp")
                if layer["type"] == "attention":
                    params = W * (2 * x["heads"] * x["dim"] + 2 * x["kv_heads"] * x["dim"] + x["heads"] * x["vdim"])
                    byts += keys * x["kv_heads"] * (x["dim"] + x["vdim"]) * size
                    flops += 2 * pairs * x["heads"] * (x["dim"] + x["vdim"])
                elif layer["type"] == "latent_attention":
                    params = W * x["q_rank"] + x["q_rank"] * x["heads"] * (x["dim"] + x["rot_dim"]) + x["kv_rank"] * x["heads"] * 2 * x["dim"] + W * x["heads"] * x["vdim"]
                    params += W * (x["kv_rank"] + x["rot_dim"]) if x.get("kv_from") is None else 0
                    byts += keys * (x["kv_rank"] + x["rot_dim"]) * size
                    flops += 2 * pairs * x["heads"] * (2 * x["dim"] + x["rot_dim"])
                else:
                    params = 3 * W * x["inner"] + x["inner"] * (2 * x["dt_rank"] + 2 * x["state"])
                    byts += 2 * len(entries) * x["inner"] * x["state"] * 4
                    flops += 7 * T * x["inner"] * x["state"]
                byts, flops = byts + params * size, flops + 2 * T * params
                if ff["kind"] == "dense":
                    byts, flops = byts + 2 * W * ff["ff"] * size, flops + 4 * T * W * ff["ff"]
                else:
                    n, top, F = ff["router"]["experts"], ff["router"]["top"], ff["expert"]["ff"]
                    byts += (W * n + 2 * W * F * min(n, CODE * top, T * top)) * size
                    flops += 2 * T * W * n + 4 * T * top * W * F
            continue
        hp = _hp(case)
        kv = hp["n_head_kv"] * hp["head_dim"]
        ends = case["kind"] in ("serve", "prompts") or case["head"]
        for il in _layers(case):
            for _, t, N, K in _matrices(case, il):
                byts, flops = byts + N * _row_bytes(t, K), flops + 2 * T * N * K
            byts += keys * kv * 2 * 2
            flops += 4 * pairs * hp["n_head"] * hp["head_dim"]
        if ends:
            (_, te, V, W), (_, to, _, _) = _ends(case)
            byts += T * _row_bytes(te, W) + V * _row_bytes(to, W) + len(entries) * V * 4
            flops += 2 * len(entries) * V * W
        else:
            byts += T * hp["n_embd"] * 4
        if case["kind"] not in ("serve", "prompts"):
            byts += T * hp["n_embd"] * 4
    return {"bytes": byts, "flops": flops}


def tolerance(case):
    """The quantized windows round every activation to 8 bits (up to 32 tokens at once, and in front of the head) or to 16: a correct implementation that sums in another order turns
    some of these roundings around. Measured against exact(): 8-bit passes 0.7-2.7 %, 16-bit ones 0.11-0.14 %, dense bf16 models 0.3-0.8 %, 32-bit ones 8e-7."""
    if case["mix"] == "f32":
        return {"rel": 4e-6, "max": 1e-4}
    if case["kind"] == "batch" and case["tokens"] > 32 and not case["head"]:
        return {"rel": 0.006, "max": 0.2}
    return {"rel": 0.03, "max": 0.8}


# ---- the same in 64 bits --------------------------------------------------------------------------------------------------------------------------------------------------------
def _rms(x, w, eps):
    return x / (x.square().mean(-1, keepdim=True) + eps).sqrt() * w


def _rotate(x, pos, base, factors, neox):
    """x [n, heads, d] turned by position: pairs (2 i, 2 i + 1), or (i, i + d / 2)"""
    d = x.shape[-1]
    a = pos.double()[:, None] * base ** (-torch.arange(0, d, 2, device="cuda").double() / d)
    a = (a / factors if factors is not None else a)[:, None, :]
    u, v = (x[..., :d // 2], x[..., d // 2:]) if neox else (x[..., 0::2], x[..., 1::2])
    p, q = u * a.cos() - v * a.sin(), v * a.cos() + u * a.sin()
    return torch.cat([p, q], -1) if neox else torch.stack([p, q], -1).flatten(-2)


def _attend(q, k, v, parts, scale, weights=None):
    """causal attention inside every sequence: q [n, H, d], k / v [n, G, d]; weights(scores, head) -> probabilities"""
    out = torch.empty(q.shape[:2] + v.shape[2:], dtype=torch.float64, device="cuda")
    for a, b in parts:
        for h in range(q.shape[1]):
            g = h * k.shape[1] // q.shape[1]
            s = (q[a:b, h] @ k[a:b, g].T).mul_(scale)
            hidden = torch.ones_like(s, dtype=torch.bool).triu_(1)
            p = s.masked_fill_(hidden, -math.inf).softmax(-1) if weights is None else weights(s, hidden, h)
            out[a:b, h] = p @ v[a:b, g]
    return out.flatten(1)


def _exact_window(case, seed, x, tokens, parts):
    """hidden rows of all tokens of the sequences `parts` (ranges of rows); x: activations, or tokens"""
    hp = _hp(case)
    H, G, d, eps = hp["n_head"], hp["n_head_kv"], hp["head_dim"], hp["rms_eps"]
    vec = lambda kind, il, n, mean, amp: _normal(seed, (kind, il), (n,), amp, mean).double()  # noqa: E731
    if tokens is not None:
        kind, t, N, K = _ends(case)[0]
        x = _dequantize(t, _matrix(seed, kind, -1, t, N, K)[tokens.long()])
    x, ff = x.double(), _rope_factors(case, seed)
    ff = None if ff is None else ff.double()
    pos = torch.cat([torch.arange(b - a, device="cuda") for a, b in parts])
    for il in _layers(case):
        v = {kind: vec(kind, il, n, mean, amp) for kind, n, mean, amp in _vectors(case, il)}
        mats = {kind: (t, N, K) for kind, t, N, K in _matrices(case, il)}
        mul = lambda y, kind: y @ _dequantize(mats[kind][0], _matrix(seed, kind, il, *mats[kind])).T  # noqa: E731,B023
        h = _rms(x, v[E.T_ATTN_NORM], eps)
        q, k, w = (mul(h, kind) + v.get(b, 0.0) for kind, b in ((E.T_WQ, E.T_BQ), (E.T_WK, E.T_BK), (E.T_WV, E.T_BV)))
        q, k = (_rotate(y.view(len(x), -1, d), pos, hp["rope_freq_base"], ff, hp["arch"] == 1) for y in (q, k))
        x = x + mul(_attend(q, k, w.view(-1, G, d), parts, d ** -0.5), E.T_WO)
        h = _rms(x, v[E.T_FFN_NORM], eps)
        gate = mul(h, E.T_FFN_GATE)
        x = x + mul(gate * torch.sigmoid(gate) * mul(h, E.T_FFN_UP), E.T_FFN_DOWN)
    return x


def _exact_logits(case, seed, rows):
    hp = _hp(case)
    kind, t, N, K = _ends(case)[1]
    return _rms(rows, _normal(seed, (E.T_OUT_NORM, -1), (K,), 0.1, 1.0).double(), hp["rms_eps"]) @ _dequantize(t, _matrix(seed, kind, -1, t, N, K)).T


def _exact_kudirax(config, w, tokens, parts):
    eps = config["norm"]["eps"]

    def norm(x, name):
        c = x - x.mean(-1, keepdim=True)
        return c / (c.square().mean(-1, keepdim=True) + eps).sqrt() * w(name) + w(name + ".b")
    x, first = w("embed")[tokens.long()], None
    for i, layer in enumerate(config["layers"]):
        m, p = layer["mixer"], "l%d." % i
        q, k = ((x @ w(p + "mix." + n).T).view(len(x), -1, m["dim"]) for n in "qk")
        q, k = (y / (y.square().mean(-1, keepdim=True) + eps).sqrt() for y in (q, k))
        v = (x @ w(p + "mix.v").T).view(len(x), -1, m["vdim"])
        lam = w(p + "mix.vmix")
        first = v if first is None else first
        v = (1 - lam) * v + lam * first
        sink = w(p + "mix.sink")

        def weights(s, hidden, h):
            s = (m["softcap"] * torch.tanh(s / m["softcap"])).masked_fill_(hidden, -math.inf)  # noqa: B023
            return torch.cat([s, sink[h].expand(len(s), 1)], -1).softmax(-1)[:, :-1]  # noqa: B023
        y = _attend(q, k, v, parts, m["scale"], weights) * torch.sigmoid(x @ w(p + "mix.g").T)
        x = x + norm(y @ w(p + "mix.o").T, p + "norm1")
        y = torch.relu(x @ w(p + "mlp.up").T + w(p + "mlp.up.b")).square() @ w(p + "mlp.down").T + w(p + "mlp.down.b")
        x = x + norm(y, p + "norm2")
    return norm(x, "final.norm")


def _exact_scan(h, w, p, m, parts):
    I, r, S = m["inner"], m["dt_rank"], m["state"]
    xz = h @ w(p + "in").T
    taps, A, out = w(p + "conv"), -torch.exp(w(p + "A_log")), torch.empty((len(h), I), dtype=torch.float64, device="cuda")
    for a, b in parts:
        pad = torch.cat([torch.zeros((3, I), dtype=torch.float64, device="cuda"), xz[a:b, :I]])
        x = torch.nn.functional.silu(w(p + "conv.b") + sum(pad[j:j + b - a] * taps[:, j] for j in range(4)))
        f = x @ w(p + "x").T
        dt = torch.nn.functional.softplus(f[:, :r] @ w(p + "dt").T + w(p + "dt.b"))
        state = torch.zeros((I, S), dtype=torch.float64, device="cuda")
        for t in range(b - a):
            state = torch.exp(dt[t][:, None] * A) * state + (dt[t] * x[t])[:, None] * f[t, r:r + S]
            out[a + t] = state @ f[t, r + S:] + w(p + "D") * x[t]
    return out * torch.nn.functional.silu(xz[:, I:])


def _exact_keranex(config, w, tokens, parts):
    eps, bg = config["norm"]["eps"], config["embedding"]["bigram"]
    t = tokens.long()
    row = (t.roll(1) * bg["mul_prev"] + t * bg["mul_cur"]) % bg["buckets"]
    row[[a for a, _ in parts]] = bg["buckets"]
    x, pos, caches = w("embed")[t] + w("bigram")[row], torch.cat([torch.arange(b - a, device="cuda") for a, b in parts]), {}
    for i, layer in enumerate(config["layers"]):
        m, p, ff = layer["mixer"], "l%d." % i, layer["mlp"]
        h = _rms(x, w(p + "norm1"), eps)
        if layer["type"] == "latent_attention":
            H, dn, kr = m["heads"], m["dim"], m["kv_rank"]
            src = i if m.get("kv_from") is None else m["kv_from"]
            if src == i:
                y = h @ w(p + "mix.dkv").T
                caches[i] = _rms(y[:, :kr], w(p + "mix.dkv.norm"), eps), _rotate(y[:, None, kr:], pos, m["rot"]["base"], None, True)
            c, k_rot = caches[src]
            q = (_rms(h @ w(p + "mix.dq").T, w(p + "mix.dq.norm"), eps) @ w(p + "mix.uq").T).view(len(x), H, -1)
            q = torch.cat([q[..., :dn], _rotate(q[..., dn:], pos, m["rot"]["base"], None, True)], -1)
            k = torch.cat([(c @ w(p + "mix.uk").T).view(len(x), H, dn), k_rot.expand(-1, H, -1)], -1)
            y = _attend(q, k, (c @ w(p + "mix.uv").T).view(len(x), H, -1), parts, m["scale"])
        else:
            y = _exact_scan(h, w, p + "mix.", m, parts)
        x = x + _rms(y @ w(p + "mix.o").T, w(p + "norm1b"), eps)
        h, r = _rms(x, w(p + "norm2"), eps), ff["router"]
        s = (h @ w(p + "mlp.router").T).softmax(-1)
        groups = s.view(len(s), r["groups"]["count"], -1)
        keep = torch.zeros(groups.shape[:2], device="cuda").scatter_(1, groups.amax(-1).topk(r["groups"]["keep"]).indices, 1.0)
        ids = (groups * keep[..., None]).flatten(1).topk(r["top"]).indices
        y = torch.zeros_like(h)
        for e in ids.unique().tolist():
            at = (ids == e).any(-1).nonzero()[:, 0]
            y[at] += s[at, e, None] * (torch.relu(h[at] @ w("%smlp.e%d.up" % (p, e)).T).square() @ w("%smlp.e%d.down" % (p, e)).T)
        x = x + _rms(y, w(p + "norm2b"), eps)
    return _rms(x, w("final.norm"), eps)


def exact(case, seed):
    if case["kind"] not in ("serve", "prompts"):
        n, seq = case["past"] + case.get("tokens", 1), _sequence(case, seed)
        x = _exact_window(case, seed, None if case["head"] else seq, seq if case["head"] else None, [(0, n)])[case["past"]:]
        if not case["head"]:
            return [x]
        return [x, _exact_logits(case, seed, x[-1])]
    lens, steps = _lengths(case, seed), case.get("steps", 0)
    vocab = _design(case)["vocab"] if _is_design(case) else _hp(case)["n_vocab"]
    tokens = torch.cat([_tokens(seed, i, n + steps, vocab) for i, n in enumerate(lens)])
    ends = np.cumsum([n + steps for n in lens])
    parts = [(int(e) - n - steps, int(e)) for e, n in zip(ends, lens)]
    want = torch.tensor([[e - steps - 1 + k for _, e in parts] for k in range(steps + 1)], device="cuda")
    if not _is_design(case):
        return _exact_logits(case, seed, _exact_window(case, seed, None, tokens, parts)[want])
    config = _design(case)
    rows = {name: (kind, il, part, name, shape) for kind, il, part, name, shape in _design_tensors(config)}
    w = lambda name: _design_tensor(config, seed, *rows[name]).to(torch.bfloat16).double()  # noqa: E731
    x = (_exact_kudirax if config["architecture"] == "Kudirax" else _exact_keranex)(config, w, tokens, parts)
    return x[want] @ w("head").T
