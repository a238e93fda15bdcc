"""What the library's host code launches, and in what order, on the CPU: in a process of its own, in front of a HIP runtime that runs nothing (hip_shim.cpp)."""
import os
import re
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
LIB = os.path.join(ROOT, "prima_cpp_amd", "libprima_mi355.so")

COMMON = r"""
import ctypes as C, re, sys, threading
shim = C.CDLL(sys.argv[1])
shim.shim_launches.restype, shim.shim_held.restype = C.c_long, C.c_size_t
shim.shim_refuse.argtypes = [C.c_size_t]
def launches():
    out, name, r = (C.c_int * 4)(), C.create_string_buffer(500), []
    for i in range(shim.shim_launches()):
        shim.shim_launch(C.c_long(i), out, name, C.c_long(500))
        n = name.value.decode().replace("(anonymous namespace)::", "")
        r.append((out[0], re.sub(r"^_Z.*?([a-z]\w*_kernel)ILi(\d+)EE.*", r"\1<\2>", n), tuple(out[1:])))     # (names with _Float16 in them stay mangled)
    return r
"""
WINDOW = COMMON + r"""
import numpy as np, torch
torch.cuda.current_device = lambda: 0
import prima_cpp_amd.engine as E
E.stream_ptr = lambda: 1
Q4_K, Q6_K = 12, 14
def window(n_ctx=64, down=Q4_K, max_tokens=64, seqs=8, **hp):
    hp = dict(dict(arch=0, n_layer=1, n_embd=2048, n_head=16, n_head_kv=4, head_dim=128, n_ff=4096, n_vocab=320, rms_eps=1e-5, rope_freq_base=10000.0), **hp)
    w = E.Window(hp, n_ctx=n_ctx)
    for il in range(hp["n_layer"]):
        for k in (E.T_ATTN_NORM, E.T_FFN_NORM):
            w.fill_tensor(k, il, 0, 1, 1.0)
        for k in (E.T_WQ, E.T_WK, E.T_WV, E.T_WO, E.T_FFN_GATE, E.T_FFN_UP, E.T_FFN_DOWN):
            w.fill_tensor(k, il, down if k == E.T_FFN_DOWN else Q4_K, 1, 1.0)
    w.fill_tensor(E.T_OUT_NORM, -1, 0, 1, 1.0); w.fill_tensor(E.T_OUTPUT, -1, Q6_K, 1, 1.0); w.fill_tensor(E.T_TOK_EMBD, -1, Q4_K, 1, 1.0)
    w.finalize_pool(max_tokens, seqs, seqs * n_ctx)
    return w
def decode(w, n):
    x = torch.zeros(n, w.hp.n_embd)
    shim.shim_forget()
    assert w.lib.pm355_model_decode(w.h, None, x.data_ptr(), n, 0, x.data_ptr(), None, None, 1) == 0
    return [name for _, name, _ in launches()]
def batch(w, lens):
    qs = [w.seq_new() for _ in lens]
    shim.shim_forget()
    w.batch([(q, np.zeros(n, np.int32), (n - 1,)) for q, n in zip(qs, lens)], logits=torch.zeros(len(lens), 320))
    return [name for _, name, _ in launches()]
def wide(names):
    return sum("gemm_pf_kernel" in n and "true, 0, true>" in n for n in names)
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    if not os.path.exists(LIB):
        pytest.skip("library not built")
    shim = str(tmp_path_factory.mktemp("shim") / "hip_shim.so")
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", os.path.join(HERE, "hip_shim.cpp"), "-o", shim, "-lpthread"], check=True)

    def go(program):
        env = dict(os.environ, LD_PRELOAD=shim, PYTHONPATH=ROOT)
        r = subprocess.run([sys.executable, "-c", program, shim, LIB], env=env, capture_output=True, text=True, timeout=300)
        assert r.returncode == 0 and r.stdout.strip().endswith("ok"), r.stdout + r.stderr
    return go


def test_slices_of_a_product_are_added_up_before_another_product_of_the_stream(run):
    """The slices of a product that is split along K wait in scratch memory of the (device, stream) for the launch that adds them up: no other thread's launch of the same kind comes between."""
    run(COMMON + r"""
lib = C.CDLL(sys.argv[2])
f = lib.pm355_mul_mat_q_wide
f.argtypes = [C.c_void_p, C.c_int] + [C.c_void_p] * 6 + [C.c_int64, C.c_int64, C.c_int, C.c_void_p, C.c_void_p]
K, N, T, CALLS = 8192, 256, 40, 20                     # 32 super-blocks over two row tiles: split along K
at = C.addressof(C.create_string_buffer(256))
shim.shim_pause(300)
bad = []
def work(i):
    shim.shim_thread(i)
    ty, W, y, n = (C.c_int * 1)(12), (C.c_void_p * 1)(at), (C.c_void_p * 1)(at), (C.c_int64 * 1)(N)
    for _ in range(CALLS):
        rc = f(ty, 1, W, n, y, None, None, at, K, T, 0, at, 1)
        if rc: bad.append(rc)
ts = [threading.Thread(target=work, args=(i,)) for i in range(2)]
[t.start() for t in ts]; [t.join() for t in ts]
assert not bad, bad
log = launches()
assert len(log) == 2 * CALLS * 3, len(log)              # quantizer, product, its slices added up
both = [e for e in log if "quantize" not in e[1]]       # (the quantizer writes memory of the call's own)
for i in range(0, len(both), 2):
    a, b = both[i:i + 2]
    assert a[0] == b[0] and "gemm_pf_kernel" in a[1] and "pf_reduce" in b[1], (i, both[max(i - 2, 0):i + 4])
assert sum(log[i][0] != log[i + 1][0] for i in range(len(log) - 1)) > 4     # (the threads did meet)
print("ok")
""")


def test_a_pool_without_memory_for_wide_passes_serves_small_ones(run):
    """Activations of wide passes: as many rows as a pass may have, and where the device does not have them the pool is there all the same."""
    run(WINDOW + r"""
rows = lambda n, K: n * (2 * K + K // 256 * 36)         # values as F16, 16 sums as F16 and a scale per super-block
for n, m in ((33, 64), (64, 64), (100, 128), (300, 384), (512, 512)):
    h = shim.shim_held(); w = window(max_tokens=n); full = shim.shim_held() - h
    assert wide(batch(w, [7] * 8)) == (4 if n > 33 else 0)
    w.close()
    shim.shim_refuse(rows(m, 4096))                     # (n_ff is the longest row)
    h = shim.shim_held(); w = window(max_tokens=n); less = shim.shim_held() - h
    assert full - less == rows(m, 4096), (n, full - less)
    assert wide(batch(w, [7] * 8)) == 0 and shim.shim_last() == 0
    w.close()
    shim.shim_refuse(0)
print("ok")
""")


def test_which_portions_meet_in_wide_passes(run):
    """More rows of short portions than one small pass takes: wide passes, whose wq | wk | wv ends with the rope and the cache stores at up to 255 rows, plain beyond."""
    run(WINDOW + r"""
w = window(max_tokens=512, seqs=24)
names = batch(w, [7] * 8)
assert wide(names) == 4 and sum("pf_reduce_rope_kernel" in n for n in names) == 1 and not any("rope_kv" in n for n in names), names
w = window(max_tokens=512, seqs=24)
names = batch(w, [30] * 10)                             # 300 rows
assert wide(names) == 4 and not any("pf_reduce_rope_kernel" in n for n in names) and any("rope_kv" in n for n in names), names
w = window(max_tokens=512, seqs=24)
assert wide(batch(w, [4] * 8)) == 0                     # 32 rows: one small pass
w = window(max_tokens=33, seqs=24)
assert wide(batch(w, [4] * 9)) == 0                     # two passes of 18: small ones
w = window(max_tokens=512, seqs=24)
assert wide(batch(w, [40, 50])) == 0                    # longer portions: 16-bit activations
print("ok")
""")


def test_which_forms_add_up_the_slices_of_a_prompt(run):
    """The shapes of test_gpu_engine.py's SLICED: norms with up to four slices and with more, rows beyond one and two columns of a wave, 128-row tiles up to 128 tokens; nothing rides along from 256
    (rope) and 513 tokens (norm) on."""
    run(WINDOW + r"""
def forms(n_embd, n_head, n_head_kv, n_ff, tokens):
    w = window(n_ctx=576, down=Q6_K, max_tokens=560, seqs=1, n_layer=2, n_embd=n_embd, n_head=n_head, n_head_kv=n_head_kv, n_ff=n_ff)
    out = []
    for n in tokens:
        names = decode(w, n)
        mid = any(re.search(r"gemm_pf_kernel<1., 1., ., true", x) for x in names)
        out.append((mid, sorted(m.group(1) for x in names for m in [re.search(r"pf_reduce_((?:norm|rope)_kernel<.>)", x)] if m), any("rope_kv" in x for x in names)))
    w.close()
    return out
N4, N8, R4, R8 = "norm_kernel<4>", "norm_kernel<8>", "rope_kernel<4>", "rope_kernel<8>"
# (the second layer's ffn_down has no norm behind it)
got = forms(4352, 32, 8, 14336, (72, 130, 512, 560))
assert got[0] == (True, [N4, N4, N8, R4, R4], False), got[0]
assert got[1][1].count(N4) + got[1][1].count(N8) == 3 and not got[1][2], got[1]
assert got[2][2] and len(got[2][1]) == 3 and all("norm" in x for x in got[2][1]), got[2]
assert got[3] == (False, [], True), got[3]
got = forms(8192, 64, 8, 28672, (72, 130, 200))
assert got[0][0] and got[1] == got[2] == (False, [N8, N8, N8, R8, R8], False), got
got = forms(8192, 16, 4, 4096, (72,))
assert got[0][0] and got[0][1].count(R8) == 2, got
print("ok")
""")


def test_which_products_of_few_tokens_take_16_row_operands(run):
    """mmq_rows.hip where it is the faster form - one group of 16 rows per CU, or steps and passes that are full -, mmq_mid.hip elsewhere, for one matrix, several, and two types; one matrix of Q5_K
    or Q8_0 over up to 16 tokens: mmq_i8.hip."""
    run(COMMON + r"""
lib = C.CDLL(sys.argv[2])
lib.pm355_mul_mat_q_small.argtypes = [C.c_int, C.c_void_p, C.c_int64, C.c_int64, C.c_void_p, C.c_void_p, C.c_int64, C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p]
at = C.addressof(C.create_string_buffer(256))
Q4, Q5, Q6, Q8 = 12, 13, 14, 8
def forms():
    return [m.groups() for _, n, _ in launches() for m in [re.search(r"mmq_(rows|mid|i8)_kernel<(.*?)>", n)] if m]
def one(t, N, K, T):
    shim.shim_forget()
    rc = lib.pm355_mul_mat_q_small(t, at, K, N, at, None, T, at, None, None, 1)
    assert rc == 0, (t, N, K, T, rc)
    return [f for f, _ in forms()]
def several(types, Ns, K, T):
    n = len(types)
    arr = lambda v, ty: (ty * n)(*v)
    shim.shim_forget()
    W, y, N64 = arr([at] * n, C.c_void_p), arr([at] * n, C.c_void_p), arr(Ns, C.c_int64)
    if len(set(types)) == 1:
        f = lib.pm355_mul_mat_q_small_multi
        f.argtypes = [C.c_int, C.c_int] + [C.c_void_p] * 5 + [C.c_int64, C.c_int64, C.c_void_p]
        rc = f(types[0], n, W, N64, y, None, at, K, T, 1)
    else:
        f = lib.pm355_mul_mat_q_small_mixed
        f.argtypes = [C.c_void_p, C.c_int] + [C.c_void_p] * 5 + [C.c_int64, C.c_int64, C.c_void_p]
        rc = f(arr(types, C.c_int), n, W, N64, y, None, at, K, T, 1)
    assert rc == 0, (types, Ns, K, T, rc)
    return [f for f, _ in forms()]
R, M, S = ["rows"], ["mid"], ["i8"]
for T in (1, 2, 5, 8):
    for t in (Q4, Q5, Q6, Q8):
        for K in (1024, 2048, 4096, 14336):
            assert one(t, 4096, K, T) == R and one(t, 17, K, T) == R, (t, K, T)
        for K in (512, 1024, 1536, 2048):
            for N in (8192, 16384, 32000):
                assert one(t, N, K, T) == (M if t in (Q4, Q6) else S), (t, N, K, T)
    for t in (Q4, Q6):
        assert one(t, 128256, 4096, T) == one(t, 36864, 8192, T) == one(t, 10240, 4096, T) == one(t, 8001, 3072, T) == R
        assert one(t, 27648, 5120, T) == one(t, 5120, 5120, T) == one(t, 14336, 14336, T) == one(t, 16384, 3072, T) == M
        assert several([t] * 2, [14336] * 2, 4096, T) == several([t] * 3, [4096, 1024, 1024], 4096, T) == several([t] * 3, [3072, 1024, 1024], 3072, T) == R
        assert several([t] * 2, [8192] * 2, 2048, T) == several([t] * 3, [5120] * 3, 5120, T) == M
    for tb in (Q5, Q6):
        assert several([Q4, Q4, tb], [4096, 1024, 1024], 4096, T) == several([Q4, Q4, tb], [8192, 1024, 1024], 8192, T) == several([Q4, Q4, tb], [2048, 512, 512], 2048, T) == R
        assert several([Q4, Q4, tb], [5120] * 3, 5120, T) == several([Q4, Q4, tb], [8192, 1024, 1024], 2048, T) == M
    assert one(Q5, 5000, 4096, T) == R and one(Q5, 128256, 4096, T) == one(Q5, 8192, 8192, T) == S
    assert one(Q8, 10240, 8192, T) == one(Q8, 49152, 2048, T) == R and one(Q8, 8192, 8192, T) == one(Q8, 4096, 512, T) == S
for t, T, K, N, want in ((Q4, 12, 2048, 4096, M), (Q4, 12, 3072, 4096, R), (Q4, 24, 8192, 4096, R), (Q4, 25, 8192, 4096, M), (Q4, 12, 8192, 4097, M), (Q6, 20, 2048, 4096, R), (Q6, 20, 1024, 4096, M),
                         (Q5, 9, 512, 4096, R), (Q5, 32, 8192, 4096, R), (Q5, 33, 8192, 4096, R + R), (Q5, 20, 2048, 32000, S + S), (Q5, 20, 4096, 32000, R), (Q5, 16, 4096, 32000, S), (Q5, 25, 4096, 32000, S + S),
                         (Q8, 12, 4096, 4096, S), (Q8, 12, 8192, 4096, R), (Q8, 17, 512, 4096, R), (Q8, 20, 512, 16384, S + S), (Q8, 20, 1024, 16384, R), (Q8, 32, 4096, 8192, S + S), (Q4, 40, 8192, 4096, M + R),
                         (Q5, 17, 4352, 8192, M), (Q5, 40, 8192, 32000, M + S), (Q8, 20, 2048, 8192, M), (Q8, 25, 1024, 16384, M), (Q8, 52, 896, 12288, M + S + S), (Q8, 60, 896, 12288, M + M)):
    assert one(t, N, K, T) == want, (t, T, K, N, one(t, N, K, T))
print("ok")
""")


def test_forms_of_one_dense_matrix(run):
    """the shapes of test_gpu_kudirax.py's test_dense_mul_mat_forms take the forms that they are there for, of either type of results; every form is among them"""
    from test_gpu_kudirax import DENSE_FORMS
    assert len(set(DENSE_FORMS.values())) == 7
    run(COMMON + "want = " + repr(DENSE_FORMS) + r"""
lib = C.CDLL(sys.argv[2])
f = lib.pm355_dense_mul_mat
f.argtypes = [C.c_int, C.c_void_p, C.c_int64, C.c_int64, C.c_void_p, C.c_int64, C.c_int, C.c_void_p, C.c_int64, C.c_int, C.c_int64, C.c_void_p, C.c_int, C.c_void_p]
at = (C.addressof(C.create_string_buffer(512)) + 255) // 256 * 256
for (T, K, n, pad), form in want.items():
    N = (n + 63) // 64 * 64
    for y_type in (0, 30):
        shim.shim_forget()
        assert f(30, at, K, N, at, K, T, at, N + pad, y_type, n, None, 0, 1) == 0
        names = [name.replace(" ", "") for _, name, _ in launches()]
        assert len(names) == 1 and "dense_" + form in names[0], (T, K, n, names)
print("ok")
""")


def test_a_dense_model_without_room_for_all_k_ranges_splits_less(run):
    """59 MB for the sums of k ranges where the device has them, 17 where it does not: prompts are served all the same"""
    run(COMMON + r"""
import os
sys.path.insert(0, os.path.join(os.environ["PYTHONPATH"], "tests"))
import numpy as np, torch
torch.cuda.current_device = lambda: 0
import prima_cpp_amd.engine as E
E.stream_ptr = lambda: 1
from prima_cpp_amd import kudirax
from test_gpu_kudirax import P, config, layer
c = config(layer(heads=4, kv=1, dim=64, vdim=64, size=400, mix=False, ff=4096), width=2048, vocab=90)
w = P.random_model(c, 1)
MOST, LEAST = 256 * 224 * 256 * 4, 256 * 128 * 128 * 4
def pool(refused):
    m = kudirax.load_arrays(c, w, "bfloat16")
    h = shim.shim_held()
    shim.shim_refuse(refused)
    try:
        m.finalize_pool(max_tokens=900, n_seq=1, pool_tokens=1024)
    finally:
        shim.shim_refuse(0)
    return m, shim.shim_held() - h
def tiles(m, T):                                        # workgroups of a prompt's products
    s = m.seq_new()
    shim.shim_forget()
    m.batch([(s, np.zeros(T, np.int32), (T - 1,))], logits=torch.zeros(1, 90))
    m.seq_free(s)
    return [g[0] for _, name, g in launches() if "dense_tile" in name or "dense_gemm" in name]
m, full = pool(0)
a = tiles(m, 900); m.close()
m, less = pool(MOST)
assert full - less == MOST - LEAST and shim.shim_last() == 0, (full, less)
b = tiles(m, 900); m.close()
assert len(a) == len(b) == 4, (a, b)
print("ok")
""")


def test_passes_of_a_product_hold_all_tokens(run):
    """1..64 tokens, one matrix: the launched kernels have room for every token (their tiles' tokens are in the names), and only the last pass is not full"""
    run(COMMON + r"""
lib = C.CDLL(sys.argv[2])
f = lib.pm355_mul_mat_q_small
f.argtypes = [C.c_int, C.c_void_p, C.c_int64, C.c_int64, C.c_void_p, C.c_void_p, C.c_int64, C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p]
at = C.addressof(C.create_string_buffer(256))
def room(name):
    m = re.search(r"mmq_(rows|mid|i8)_kernel<(.*?)>", name)
    if not m: return 0
    a = m.group(2).split(", ")
    return 8 * int(a[2]) if m.group(1) == "rows" else 2 * int(a[2] if m.group(1) == "mid" else a[1])     # groups of 8 tokens; result registers of 2
short = []
for t in (12, 13, 14, 8):
    for N in (17, 4096, 4097, 8192, 8193, 12288, 16384, 32000, 57344, 151936):
        for K in (512, 768, 1024, 1536, 2048, 3072, 4096, 7168, 14336) + ((544, 896, 992) if t == 8 else ()):
            for T in range(1, 65):
                shim.shim_forget()
                assert f(t, at, K, N, at, None, T, at, None, None, 1) == 0
                r = [x for x in map(room, (n for _, n, _ in launches())) if x]
                if sum(r) < T or sum(r[:-1]) >= T or any(x not in (16, 32) for x in r[:-1]): short.append((t, N, K, T, r))
assert not short, (len(short), short[:20])
print("ok")
""")


def test_a_norm_whose_results_lie_on_its_input_has_one_workgroup_to_a_row(run):
    """pm355_rms_norm in place (y_f32 == x), or with the Q8_K blocks on the row: of two workgroups to a row (17..32 blocks, up to half the CUs' rows) one could store its half before the other has
    read the row"""
    run(COMMON + r"""
lib = C.CDLL(sys.argv[2])
f = lib.pm355_rms_norm
f.argtypes = [C.c_void_p] * 4 + [C.c_int64, C.c_int64, C.c_float, C.c_void_p]
at = C.addressof(C.create_string_buffer(256)) // 16 * 16 + 16
def grid(K, rows, y, yq):
    shim.shim_forget()
    assert f(at, None, y, yq, K, rows, 1e-5, 1) == 0
    (_, _, g), = launches()
    return g[:2]
for K in (4352, 8192):
    for rows in (1, 8, 128):
        n, q = rows * K * 4, rows * (K + K // 256 * 4 + K // 16 * 2)
        assert grid(K, rows, at + n, None) == grid(K, rows, at - n, None) == grid(K, rows, None, at + n) == grid(K, rows, None, at - q) == grid(K, rows, at + n, at - q) == (rows, 2), (K, rows)
        assert grid(K, rows, at, None) == grid(K, rows, None, at) == grid(K, rows, at, at + n) == grid(K, rows, at + n, at + n - 16) == grid(K, rows, at - 16, None) == (rows, 1), (K, rows)
assert grid(4096, 8, at, None) == grid(4096, 8, at + (1 << 20), None) == (8, 1) and grid(8192, 129, at + (1 << 30), None) == (129, 1)
print("ok")
""")


def test_a_tile_that_there_is_no_kernel_for_is_not_forced(run):
    """PM355_GEMM_PF_NT names the 256-row tiles' sub-tiles of 32 tokens, 2, 4, 6 or 8: with another value a prompt product has the tiles that its tokens ask for (3: grids of 96 tokens in front of the
    64-token kernel, a third of the tokens never written)"""
    run(COMMON + r"""
import os
def products(nt):
    r, w = os.pipe()
    if os.fork() == 0:
        os.environ["PM355_GEMM_PF_NT"] = nt
        lib = C.CDLL(sys.argv[2])
        f = lib.pm355_mul_mat_q_mfma
        f.argtypes = [C.c_int, C.c_void_p, C.c_int64, C.c_int64, C.c_void_p, C.c_int64, C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p]
        at = C.addressof(C.create_string_buffer(256))
        out = []
        for t, K, N, T in ((12, 4096, 4096, 300), (14, 14336, 4096, 101), (8, 896, 512, 40), (12, 4096, 28672, 1500)):
            shim.shim_forget()
            assert f(t, at, K, N, at, T, at, None, None, 1) == 0, (t, K, N, T)
            out.append([(n, g) for _, n, g in launches() if "gemm_pf" in n or "pf_reduce" in n])
        os.write(w, repr(out).encode()); os._exit(0)
    os.close(w)
    return eval(b"".join(iter(lambda: os.read(r, 65536), b"")).decode())
plain, three = products("1"), products("3")
assert len(plain) == 4 and all(len(x) in (1, 2) for x in plain), plain
assert products("") == products("5") == products("9") == plain
assert three == plain, three
assert products("4") != plain and all(re.search(r"gemm_pf_kernel<\d+, \d+, 4,", x[0][0]) for x in products("4")), products("4")
print("ok")
""")


CACHED = COMMON + r"""
lib = C.CDLL(sys.argv[2])
f = lib.pm355_attn_cached
f.argtypes = [C.c_void_p] * 7 + [C.c_int] * 4 + [C.c_float, C.c_int, C.c_int, C.c_void_p]
at = C.addressof(C.create_string_buffer(256))
def cached(H, Hkv, dh=64, n_ctx=64):
    shim.shim_forget()
    return f(at, at, at, at, None, None, at, H, Hkv, dh, n_ctx, 0.125, 0, 0, 1), [(n, g) for _, n, g in launches()]
"""


def test_cached_attention_of_heads_that_share_nothing_is_refused(run):
    """no KV heads, or more of them than heads: an error code, no launch, no division by zero on the host"""
    run(CACHED + r"""
for H, Hkv in ((8, 0), (8, -1), (4, 8), (0, 0), (0, 8)):
    for dh in (64, 128, 256):
        rc, seen = cached(H, Hkv, dh)
        assert rc and not seen, (H, Hkv, dh, rc, seen)
for H, Hkv in ((8, 8), (8, 1), (6, 2)):
    rc, seen = cached(H, Hkv)
    assert rc == 0 and len(seen) == 1, (H, Hkv, rc, seen)
print("ok")
""")


def test_cached_attention_of_more_heads_than_16_bits(run):
    run(CACHED + r"""
for H, Hkv in ((65535, 65535), (65536, 1), (65536, 65536), (1 << 20, 1 << 10)):
    for dh in (64, 128, 256):
        rc, seen = cached(H, Hkv, dh)
        assert rc == 0 and [g for _, g in seen] == [(H, 1, 1)] and ("true" in seen[0][0]) == (H > 65535), (H, Hkv, dh, rc, seen)
print("ok")
""")


def test_quantizers_of_short_rows_fill_their_workgroups(run):
    """rows of less than 512 values, and more rows than a grid of rows has room for, by one index"""
    run(COMMON + r"""
lib = C.CDLL(sys.argv[2])
at = C.addressof(C.create_string_buffer(256))
def grid(name, K, rows):
    f = getattr(lib, name)
    f.argtypes = [C.c_void_p] * 2 + [C.c_int64, C.c_int64, C.c_void_p]
    shim.shim_forget()
    assert f(at, at, K, rows, 1) == 0
    (_, _, g), = launches()
    return g
for rows in (1, 7, 200000, 16777215, 16777216, 20000000):
    for K in (32, 64, 96, 256, 480):
        assert grid("pm355_quantize_q8_0", K, rows) == (-(-rows * K // 1024), 1, 1), (K, rows)
    assert grid("pm355_quantize_q8_K", 256, rows) == (-(-rows // 4), 1, 1), rows
    for K in (512, 768):
        many = rows >= 1 << 24
        assert grid("pm355_quantize_q8_0", K, rows) == ((-(-rows * K // 1024), 1, 1) if many else (rows, 1, 1)), (K, rows)
        assert grid("pm355_quantize_q8_K", K, rows) == ((-(-rows * K // 1024), 1, 1) if many else (rows, 1, 1)), (K, rows)
assert grid("pm355_quantize_q8_0", 2080, 9) == (9, 3, 1) and grid("pm355_quantize_q8_K", 1280, 9) == (9, 2, 1)
print("ok")
""")


PROMPT_ATTENTION = COMMON + r"""
lib = C.CDLL(sys.argv[2])
at = C.addressof(C.create_string_buffer(256)) // 16 * 16 + 16
f, fm = lib.pm355_attn_prefill, lib.pm355_attn_prefill_masked_ex
f.argtypes = [C.c_void_p] * 5 + [C.c_int] * 5 + [C.c_float, C.c_void_p]
fm.argtypes = [C.c_void_p] * 4 + [C.c_int64, C.c_void_p] + [C.c_int] * 6 + [C.c_float, C.c_int, C.c_void_p]
def form(H, dh, T, mask=False, off=0):
    "(query waves, its waves request themselves, workgroups)"
    shim.shim_forget()
    k = at + off
    rc = fm(at, k, k, at, 4096, at, T, H, 8, dh, 4096, 4096, 0.1, 0, 1) if mask else f(at, k, k, at, at, T, H, 8, dh, 4096, 0.1, 1)
    assert rc == 0
    (_, n, g), = launches()
    a = re.search(r"attn_prompt_kernel<(.*)>", n).group(1).split(", ")
    assert a[0] == str(dh) and a[3] == str(mask).lower() and a[4] == str(bool(off)).lower() and g[1:] == (1, 1), n
    return int(a[1]), a[6] == "true", g[0]
"""


def test_heads_of_64_leave_room_for_two_workgroups_where_there_are_more_than_cus(run):
    run(PROMPT_ATTENTION + r"""
for H in (8, 24, 40, 48, 64, 96):
    for T in (40, 400, 640, 1000, 2048, 4000):
        for off in (0, 8):
            q, own, n = form(H, 64, T, off=off)
            assert q == (2 if off else 8 if -(-T // 256) * H >= 512 else 4 if -(-T // 128) * H >= 256 else 2) and n == -(-T // (32 * q)) * H
            assert own == (n > 256), (H, T, off, q, n)
            q, own, n = form(H, 64, T, True, off)
            assert own == (n > 256 and q == 2), (H, T, off, q, n)
            assert not form(H, 128, T, off=off)[1]
            q, own, n = form(H, 128, T, True, off)      # (with a mask, tiles of 128 and 256 queries: registers)
            assert own == (q > 2), (H, T, off, q, n)
print("ok")
""")


def test_prompt_attention_keeps_its_registers(tmp_path):
    """no kernel of it has registers spilled: what the compiler wrote beside the kernels of the library built here"""
    readelf = "/opt/rocm/llvm/bin/llvm-readelf"
    if not os.path.exists(LIB) or not os.path.exists(readelf):
        pytest.skip("library not built, or no tool to read it")
    blob, seen = open(LIB, "rb").read(), {}
    at = blob.find(b"__CLANG_OFFLOAD_BUNDLE__")
    while at >= 0:                                          # magic, number of entries, then (offset, size, length of the name, name) of each
        n, p = int.from_bytes(blob[at + 24:at + 32], "little"), at + 32
        for _ in range(n):
            off, size, k = (int.from_bytes(blob[p + 8 * i:p + 8 * i + 8], "little") for i in range(3))
            name, p = blob[p + 24:p + 24 + k], p + 24 + k
            obj = blob[at + off:at + off + size]
            if b"gfx950" in name and b"attn_prompt_kernel" in obj:
                f = tmp_path / "device.o"
                f.write_bytes(obj)
                notes = subprocess.run([readelf, "--notes", str(f)], capture_output=True, text=True, check=True).stdout
                for kernel in notes.split(".agpr_count")[1:]:
                    field = lambda key: re.search(key + r":\s+(\S+)", kernel).group(1)  # noqa: E731
                    seen[field(r"\.name")] = int(field(r"\.vgpr_spill_count")), int(field(r"\.private_segment_fixed_size"))
        at = blob.find(b"__CLANG_OFFLOAD_BUNDLE__", at + 24)
    seen = {k: v for k, v in seen.items() if "attn_prompt_kernel" in k}
    assert len(seen) >= 16, len(seen)
    assert not any(a or b for a, b in seen.values()), {k: v for k, v in seen.items() if v != (0, 0)}


def test_products_of_few_tokens_take_as_many_rows_as_memory_holds(run):
    """a workgroup of more than 2^22 rows: a small matrix beside one of 220 GB, the longest that the device holds"""
    run(COMMON + r"""
lib = C.CDLL(sys.argv[2])
at = C.addressof(C.create_string_buffer(256))
one, several = lib.pm355_mul_mat_q_small, lib.pm355_mul_mat_q_small_multi
one.argtypes = [C.c_int, C.c_void_p, C.c_int64, C.c_int64, C.c_void_p, C.c_void_p, C.c_int64, C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p]
several.argtypes = [C.c_int, C.c_int] + [C.c_void_p] * 5 + [C.c_int64, C.c_int64, C.c_void_p]
def products():
    return [g for _, n, g in launches() if re.search(r"mmq_(rows|mid)_kernel", n)]
for T in (2, 8, 30):
    shim.shim_forget()
    rc = one(12, at, 512, (1 << 30) - 1, at, None, T, at, None, None, 1)
    assert rc == 0 and products() == [(256, 1, 1)], (T, rc)
arr = lambda v, ty: (ty * len(v))(*v)
for Ns in ([760000000, 4250000], [380000000, 380000000, 4250000], [1 << 20, 4250000]):
    shim.shim_forget()
    rc = several(12, len(Ns), arr([at] * len(Ns), C.c_void_p), arr(Ns, C.c_int64), arr([at] * len(Ns), C.c_void_p), None, at, 512, 4, 1)
    assert rc == 0 and products() == [(256, 1, 1)], (Ns, rc)
print("ok")
""")


def test_a_mat_vec_of_rows_beyond_lds_says_so(run):
    """K a multiple of the block size, however large: PM355_E_RANGE ("K too large"), not the error of a K that is no multiple"""
    run(COMMON + r"""
lib = C.CDLL(sys.argv[2])
f = lib.pm355_mul_mat_vec_q
f.argtypes = [C.c_int, C.c_void_p, C.c_void_p, C.c_int64, C.c_int64, C.c_void_p, C.c_int, C.c_void_p, C.c_int64, C.c_void_p, C.c_void_p, C.c_void_p]
at = C.addressof(C.create_string_buffer(256))
go = lambda t, K: f(t, at, None, K, 64, at, 1, at, 64, None, None, 1)
for t in (12, 13, 14, 8):
    assert go(t, 4096) == 0
    want = go(t, 1 << 20)
    assert want not in (0, go(t, 4097)) and all(go(t, K) == want for K in (1 << 24, 1 << 28, (1 << 28) + 256, 1 << 30)), (t, want, [go(t, K) for K in (1 << 24, 1 << 28, 1 << 30)])
print("ok")
""")


def test_prompt_products_are_launched_as_planned(run):
    """what pm355_gemm_plan answers is the grid that is launched, and its tile the kernel's: tiles of 256 and of 128 rows, one matrix, several and pairs, and 8-bit activations"""
    run(COMMON + r"""
lib = C.CDLL(sys.argv[2])
at = C.addressof(C.create_string_buffer(256)) // 16 * 16 + 16
lib.pm355_gemm_plan.argtypes = [C.c_int64, C.c_int64, C.c_int64, C.c_int, C.c_int, C.c_void_p]
lib.pm355_mul_mat_q_mfma.argtypes = [C.c_int, C.c_void_p, C.c_int64, C.c_int64, C.c_void_p, C.c_int64, C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p]
lib.pm355_mul_mat_q_mfma_pair.argtypes = [C.c_int, C.c_void_p, C.c_void_p, C.c_int64, C.c_int64, C.c_void_p, C.c_int64, C.c_void_p, C.c_void_p]
lib.pm355_mul_mat_q_wide.argtypes = [C.c_void_p, C.c_int] + [C.c_void_p] * 6 + [C.c_int64, C.c_int64, C.c_int, C.c_void_p, C.c_void_p]
def plan(tiles, K, T, flags):
    out = (C.c_int32 * 5)()
    assert lib.pm355_gemm_plan(tiles, K, T, 256, flags, out) == 0
    global split
    split = out[2], out[3]
    return out[0] // 32, out[4]
def launched():
    (n, g), = [(n, g) for _, n, g in launches() if "gemm_pf_kernel" in n]
    a = re.search(r"gemm_pf_kernel<(.*?)>", n).group(1).split(", ")
    return (int(a[2]), g[0]), a[3] == "true"
seen = set()
for t in (12, 13, 14, 8):
    for K in (512, 4096, 14336):
        for N in (132, 1024, 4096, 14336, 40960):
            for T in (33, 65, 96, 97, 128, 129, 192, 193, 300, 384, 385, 513, 576, 700, 1500, 2049):
                for pair in (False, True):
                    if pair and t == 8: continue
                    shim.shim_forget()
                    rc = lib.pm355_mul_mat_q_mfma_pair(t, at, at, K, N, at, T, at, 1) if pair else lib.pm355_mul_mat_q_mfma(t, at, K, N, at, T, at, None, None, 1)
                    assert rc == 0, (t, K, N, T, pair, rc)
                    got, mid = launched()
                    small, large = (-(-N // 64), -(-N // 128)) if pair else (-(-N // 128), -(-N // 256))
                    assert mid == (T <= 128 and small <= 256), (t, K, N, T, pair)
                    assert got == plan(small if mid else large, K, T, 4 if mid else 2), (t, K, N, T, pair, got)
                    own = mid and (T <= 64 and got[1] < 128 if t == 8 else K == 512 and T > 96)    # (few workgroups of Q8_0, four steps: no loaders)
                    assert any("gemm_pf_kernel" in n and ", 512, " in n for _, n, _ in launches()) == own, (t, K, N, T, pair)
                    tiles, left = -(-T // 256), (T - 1) % 256 + 1            # (the last tile of 256 tokens: the kernel that multiplies what is left of it, where that is enough or every tile is split)
                    saved = 4 if left <= 128 else 2 if left <= 192 else 0
                    cut = got[0] == 8 and saved > 0 and ((split[0] > 1 and not split[1]) or saved * K > 215 * 9 * tiles)
                    seen.add((got[0], cut))
                    assert any("gemm_pf_kernel" in n and ", 256, " in n for _, n, _ in launches()) == cut, (t, K, N, T, pair)
assert seen >= {(8, False), (8, True), (6, False)}
arr = lambda v, ty: (ty * len(v))(*v)
for types, Ns, K in (([12], [4096], 4096), ([12, 12], [1024, 14336], 4096), ([12, 14], [4096, 1024], 4096), ([14], [4096], 14336), ([13], [132], 512)):
    for T in (33, 64, 65, 96, 97, 128, 129, 147, 192, 231, 288, 289, 512):
        shim.shim_forget()
        n = len(types)
        assert lib.pm355_mul_mat_q_wide(arr(types, C.c_int), n, arr([at] * n, C.c_void_p), arr(Ns, C.c_int64), arr([at] * n, C.c_void_p), None, None, at, K, T, 0, at, 1) == 0
        got, mid = launched()
        assert mid and got == plan(sum(-(-N // 128) for N in Ns), K, T, 8 if set(types) == {12} else 16), (types, Ns, K, T, got)
print("ok")
""")


def test_which_experts_products_are_one_sequence_of_load_groups(run):
    """the shapes of test_gpu_keranex.py's test of dense_experts_kernel reach it: both products of the experts, up to 71 blocks of 64 values; the hidden one of 72 does not"""
    run(COMMON + r"""
import os
sys.path.insert(0, os.path.join(os.environ["PYTHONPATH"], "tests"))
import numpy as np, torch
torch.cuda.current_device = lambda: 0
import prima_cpp_amd.engine as E
E.stream_ptr = lambda: 1
from prima_cpp_amd import keranex
from test_gpu_keranex import moe, one, scan, silent, weights_for
for (n, top, ff, width), want in (((6, 4, 4160, 260), 2), ((64, 4, 520, 600), 2), ((33, 1, 64, 2000), 2), ((2, 2, 4544, 130), 2), ((2, 2, 4600, 130), 1)):
    c = one(scan(inner=64, mlp=moe(n, top, 1, 1, ff)), width=width, vocab=120)
    m = keranex.load_arrays(c, silent(weights_for(c, "bfloat16", 9), 0), "bfloat16")
    m.finalize_pool(max_tokens=64, n_seq=2, pool_tokens=128)
    for T in (5, 8, 9, 23, 64):
        s = m.seq_new()
        shim.shim_forget()
        m.batch([(s, np.zeros(T, np.int32), (T - 1,))], logits=torch.zeros(1, 120))
        m.seq_free(s)
        got = sum("dense_experts_kernel" in name for _, name, _ in launches())
        assert got == want, (n, top, ff, width, T, got, [name for _, name, _ in launches()])
    m.close()
print("ok")
""")


def test_grids_of_small_mat_vecs(run):
    """a matrix of less than four rows per CU and 512 KB: workgroups of four rows for one, two and four columns, one workgroup per CU for eight and for what is larger"""
    run(COMMON + r"""
lib = C.CDLL(sys.argv[2])
f = lib.pm355_mul_mat_vec_q
f.argtypes = [C.c_int, C.c_void_p, C.c_void_p, C.c_int64, C.c_int64, C.c_void_p, C.c_int, C.c_void_p, C.c_int64, C.c_void_p, C.c_void_p, C.c_void_p]
at = C.addressof(C.create_string_buffer(256))
def grids(K, N, cols):
    shim.shim_forget()
    assert f(12, at, None, K, N, at, cols, at, N, None, None, 1) == 0
    return [g[0] for _, _, g in launches()]
for K, N in ((256, 16), (1024, 333), (8192, 64), (4096, 200)):
    assert grids(K, N, 1) == grids(K, N, 2) == grids(K, N, 3) == grids(K, N, 4) == [(N + 3) // 4], (K, N)
    assert grids(K, N, 8) == [256] and grids(K, N, 5) == [(N + 3) // 4] * 2, (K, N)
for cols in (1, 2, 4, 8):
    assert grids(4096, 1024, cols) == grids(8192, 4096, cols) == [256]
print("ok")
""")


def test_mat_vecs_of_many_rows_are_launched_in_pieces(run):
    """33 million rows and more: a launch of more than 65536 workgroups would find its slices with more than 32 bits. One matrix, one column and several, and a fused launch"""
    run(COMMON + r"""
lib = C.CDLL(sys.argv[2])
f = lib.pm355_mul_mat_vec_q
f.argtypes = [C.c_int, C.c_void_p, C.c_void_p, C.c_int64, C.c_int64, C.c_void_p, C.c_int, C.c_void_p, C.c_int64, C.c_void_p, C.c_void_p, C.c_void_p]
at = C.addressof(C.create_string_buffer(256))
grids = lambda: [g for _, _, g in launches()]
for N, pieces in ((33357824, 1), (33357825, 2), (34000001, 3), ((1 << 31) - 1, 128)):
    for cols in (1, 2, 4, 8):
        shim.shim_forget()
        rc = f(8, at, None, 32, N, at, cols, at, N, at, None, 1)
        got = grids()
        assert rc == 0 and len(got) == pieces and all(g[0] <= 65536 for g in got), (N, cols, rc, len(got), got[:4])
class Job(C.Structure):
    _fields_ = [("type", C.c_int32), ("pad", C.c_int32), ("N", C.c_int64), ("W", C.c_void_p), ("W2", C.c_void_p), ("y", C.c_void_p), ("bias", C.c_void_p), ("resid", C.c_void_p)]
jobs = (Job * 2)(Job(12, 0, 34000001, at, None, at, None, None), Job(12, 0, 77, at, None, at, None, None))
shim.shim_forget()
assert lib.pm355_mul_mat_vec_fused(jobs, 2, C.c_int64(256), C.c_void_p(at), None, C.c_float(0), C.c_void_p(1)) == 0
assert len(grids()) == 4 and all(g[0] <= 65536 for g in grids()), grids()
print("ok")
""")
