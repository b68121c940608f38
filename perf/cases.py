"""The measured workloads of the packed-trit fabric.

Each case is work that a user of the framework has it do, through the public
entry points of ter_amd.fabric and the decoders, over the sizes of this
repository's own configurations (the BitNet-b1.58-2B and Llama-3.2-1B shapes
of bench.py) and ragged ones beside them.  listed() names twelve, draw() takes
more from the same ranges:

  gemv     one M = 1 GEMV of any activation kind, one call (the reference's
           mm_packed_dispatch, or the fused prologues)
  mm_row   the host route of the reference's own forward: int32 row in host
           memory in, fp32 row in host memory out, synchronous
  sweep    a work list of every projection of a model, one launch (M = 1)
  layer    one BitNet layer of a decode step over a filled KV cache, from a
           HIP graph: embedding, Q/K/V, attention, O, gate/up, down
  decode   one whole token of the packed Llama forward from a HIP graph
  gemm     one batched projection (M = 2-256), int8 rows or a fused row prologue
  ffn      the three batched projections of a BitNet FFN with their prologues
  msweep   a work list of every projection of a model at M rows, one launch
  tail     final RMSNorm, fp16 lm_head over the vocabulary, argmax
  convert  a projection from a file format (GGUF i2_s or v11 bytes) into the
           device layout, and exported as v11 bytes
"""
import math

import numpy as np
import torch

from ter_amd import fabric as F
from ter_amd import llama

EPS = 1e-5
BITNET = dict(H=2560, F=6912, nh=20, nkv=5, hd=128)
LLAMA = dict(H=2048, F=8192, nh=32, nkv=8, hd=64)
VOCAB = 128256


def listed():
    return [
        # the smallest call of a decode step: one K or V projection, int8 row in hand
        dict(name="gemv_kv_i8", kind="gemv", K=2560, N=640, act="i8", out="y"),
        # the reference host forward's own call: a 9-trit row through an FFN projection
        dict(name="mm_row_9trit", kind="mm_row", K=2560, N=6912, xmax=9841),
        # every projection of Llama-3.2-1B at M = 1: the headline sweep
        dict(name="sweep_llama_i8", kind="sweep", L=16, act="i8", **LLAMA),
        # one BitNet layer of a decode step at a full 2048-position context
        dict(name="layer_bitnet_2048", kind="layer", smax=2048, pos=2047, **BITNET),
        # one token of the packed Llama forward, early in a generation
        dict(name="decode_llama", kind="decode", L=16, V=VOCAB, smax=512, pos=40, **LLAMA),
        # a small serving batch through one attention projection
        dict(name="gemm_m8_i8", kind="gemm", M=8, K=2560, N=2560, act="i8", out="y"),
        # a serving batch of 64 through a BitNet FFN
        dict(name="ffn_bitnet_m64", kind="ffn", M=64, H=2560, F=6912),
        # a prefill chunk of the largest size through an FFN projection, fp32 rows
        dict(name="gemm_m256_f32", kind="gemm", M=256, K=2560, N=6912, act="f32", out="y"),
        # every projection of BitNet-2B for a batch of 32 sequences
        dict(name="msweep_bitnet_m32", kind="msweep", M=32, L=30, **BITNET),
        # a generic matrix whose rows are not 16-byte aligned
        dict(name="gemm_ragged_m77", kind="gemm", M=77, K=1003, N=1236, act="f32", out="y"),
        # the end of every BitNet token: the 657 MB tied fp16 table
        dict(name="tail_bitnet", kind="tail", H=2560, V=VOCAB),
        # loading a BitNet projection from a GGUF file and writing the packed format
        dict(name="convert_i2s", kind="convert", K=6912, N=2560, src="i2s"),
    ]


def _logi(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _dim(rng, lo, hi, step=4):
    """A size in [lo, hi], log-uniform: half the time a multiple of 256 (a
    model's), else any multiple of `step`."""
    v = _logi(rng, lo, hi)
    if rng.random() < 0.5 and v >= 256:
        return max(lo, v // 256 * 256)
    return max(lo, v // step * step)


def _shape(rng):
    hd = rng.choice([64, 128])
    nkv = rng.randint(1, 8)
    nh = nkv * rng.randint(1, 4)
    while nh * hd > 2560:
        nkv = max(1, nkv - 1)
        nh = nkv * rng.randint(1, 4)
    H = max(256, nh * hd)
    return dict(H=H, F=_dim(rng, 512, 8192, 16), nh=nh, nkv=nkv, hd=hd)


def draw(rng):
    kind = rng.choice(["gemv", "gemv", "mm_row", "sweep", "layer", "decode", "gemm", "gemm", "gemm", "ffn",
                       "msweep", "tail", "convert"])
    if kind == "gemv":
        act = rng.choice(["i8", "f32", "f32rms", "f16rms", "relu2", "f16", "silu"])
        # (rows of any length; the packed file format needs N a multiple of 4)
        return dict(kind=kind, K=_dim(rng, 256, 8192, 1), N=_dim(rng, 64, 16384), act=act,
                    out=rng.choice(["y", "y16"]))
    if kind == "mm_row":
        return dict(kind=kind, K=_dim(rng, 256, 8192, 1), N=_dim(rng, 64, 8192), xmax=rng.choice([121, 9841]))
    if kind == "sweep":
        return dict(kind=kind, L=rng.randint(1, 16), act=rng.choice(["i8", "f32"]), **_shape(rng))
    if kind == "layer":
        smax = _logi(rng, 64, 4096)
        return dict(kind=kind, smax=smax, pos=rng.randint(0, smax - 1), **_shape(rng))
    if kind == "decode":
        s = _shape(rng)
        s["H"] = s["nh"] * s["hd"]
        smax = _logi(rng, 64, 2048)
        return dict(kind=kind, L=rng.randint(1, 12), V=_dim(rng, 1024, VOCAB), smax=smax,
                    pos=rng.randint(0, smax - 1), **s)
    if kind == "gemm":
        ragged = rng.random() < 0.25
        M = _logi(rng, 2, 256)
        K = _logi(rng, 256, 2048) | 1 if ragged else _dim(rng, 256, 8192, 16)
        N = _dim(rng, 64, 2048 if ragged else 8192)
        return dict(kind=kind, M=M, K=K, N=N, act=rng.choice(["i8", "f32", "f32rms", "f16rms", "relu2"]),
                    out=rng.choice(["y", "y", "y16"]))
    if kind == "ffn":
        return dict(kind=kind, M=_logi(rng, 2, 256), H=_dim(rng, 256, 4096, 16), F=_dim(rng, 512, 8192, 16))
    if kind == "msweep":
        s, M = _shape(rng), _logi(rng, 2, 256)
        per = 2 * M * sum(K * N for K, N in _proj(s))
        return dict(kind=kind, M=M, L=max(1, min(rng.randint(1, 30), int(1.2e11 // per))), **s)
    if kind == "tail":
        return dict(kind=kind, H=_dim(rng, 256, 2560, 2), V=_logi(rng, 1000, VOCAB))
    # whole 128-element blocks of i2_s: N * K a multiple of 128
    return dict(kind=kind, K=_dim(rng, 256, 8192, 16), N=_dim(rng, 64, 8192, 8), src=rng.choice(["i2s", "v11"]))


def _proj(c):
    """(K, N) of a layer's projections Q, K, V, O, gate, up, down."""
    hq, hkv = c["nh"] * c["hd"], c["nkv"] * c["hd"]
    return [(c["H"], hq), (c["H"], hkv), (c["H"], hkv), (hq, c["H"]), (c["H"], c["F"]), (c["H"], c["F"]),
            (c["F"], c["H"])]


# ---- inputs, from the seed alone -------------------------------------------

def _gen(seed, i):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 1_000_003 + i)
    return g


def _trits(seed, i, K, N):
    """int8 [K][N] in {-1, 0, +1}, 40% zeros (BitNet's density)."""
    u = torch.randint(0, 10, (K, N), generator=_gen(seed, 7 * i + 1), device="cuda", dtype=torch.int8)
    return (u >= 4).to(torch.int8) - 2 * (u >= 7).to(torch.int8)


def _v11(t):
    """v11 bytes of trits [K][N]: byte [N/4][K], column 4 j + s at bits 2 s, codes 0, 01 = +1, 10 = -1."""
    K, N = t.shape
    c = (t == 1).to(torch.uint8) + 2 * (t == -1).to(torch.uint8)
    c = c.view(K, N // 4, 4)
    b = c[:, :, 0] | (c[:, :, 1] << 2) | (c[:, :, 2] << 4) | (c[:, :, 3] << 6)
    return b.t().contiguous().view(-1)


def _i2s(t):
    """i2_s codes of trits [K][N]: the (N, K) tensor in blocks of 128 elements, 32 bytes each."""
    u = (t + 1).to(torch.uint8).t().contiguous().view(-1, 4, 32)
    return ((u[:, 0] << 6) | (u[:, 1] << 4) | (u[:, 2] << 2) | u[:, 3]).contiguous().view(-1)


def _wscale(seed, i, K):
    """A per-tensor scale that keeps a unit-variance row's outputs near unit variance, as trained weights do."""
    u = (((seed * 1009 + i) * 2654435761) % 2 ** 32) / 2 ** 32
    return (0.7 + 0.6 * u) / math.sqrt(0.6 * K)


def _weight(seed, i, K, N):
    return F.PackedTrits.from_v11(_v11(_trits(seed, i, K, N)), K, N, _wscale(seed, i, K))


def _randn(seed, i, *shape):
    return torch.randn(*shape, generator=_gen(seed, i), device="cuda")


def _norm(seed, i, n):
    return (torch.rand(n, generator=_gen(seed, i), device="cuda") + 0.5).to(torch.float16)


def _act(seed, act, M, K):
    """The activation operand of kind `act` as keyword arguments (x, ...)."""
    sh = (K,) if M == 0 else (M, K)
    if act == "i8":
        x = (_randn(seed, 901, *sh) * 36).round().clamp(-127, 127).to(torch.int8)
        s = torch.rand(max(M, 1), generator=_gen(seed, 902), device="cuda") * 0.03 + 0.01
        return dict(x=x, x_scale_dev=s)
    x = _randn(seed, 901, *sh)
    if act in ("f32", "f32rms"):
        a = dict(x=x)
    else:
        a = dict(x=x.to(torch.float16))
    if act in ("relu2", "silu"):
        a["up"] = _randn(seed, 903, *sh).to(torch.float16)
    if act in ("f32rms", "f16rms", "relu2"):
        a["gamma"] = _norm(seed, 904, K)
    return a


def _host_row(c, seed):
    """A one-row TritTensor payload of integers within +-xmax."""
    x = np.random.default_rng(seed).standard_normal((1, c["K"])) * (c["xmax"] / 4)
    return np.rint(x).clip(-c["xmax"], c["xmax"]).astype(np.int32)


def _slots(M, ns):
    """One fp32 buffer for the [M][N] outputs of a list's items, each on a
    256-byte line as an allocation of its own would be: (buffer, views)."""
    size = [(M * n + 63) // 64 * 64 for n in ns]
    buf = torch.zeros(sum(size), dtype=torch.float32, device="cuda")
    return buf, [b[:M * n].view(M, n) for b, n in zip(buf.split(size), ns)]


def _capture(fn):
    """`fn`'s launches as a HIP graph (run once before, as a warm-up)."""
    fn()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        fn()
    torch.cuda.synchronize()
    return g


def _prep_layer(c, seed):
    H, hq, hkv = c["H"], c["nh"] * c["hd"], c["nkv"] * c["hd"]
    W = F.group_contiguous([_weight(seed, i, K, N) for i, (K, N) in enumerate(_proj(c))])
    f16, f32 = torch.float16, torch.float32
    z = lambda n, dt=f16: torch.zeros(n, dtype=dt, device="cuda")
    hidden, q, k, v, o, gate, up = z(H, f32), z(hq), z(hkv), z(hkv), z(hq), z(c["F"]), z(c["F"])
    emb = _randn(seed, 910, 64, H).to(f16)
    token = torch.full((1,), seed % 64, dtype=torch.int32, device="cuda")
    pos = torch.full((1,), c["pos"], dtype=torch.int32, device="cuda")
    kc = _randn(seed, 911, c["smax"], c["nkv"], c["hd"]).to(f16)
    vc = _randn(seed, 912, c["smax"], c["nkv"], c["hd"]).to(f16)
    n1, n2, n3, n4 = _norm(seed, 913, H), _norm(seed, 914, hq), _norm(seed, 915, H), _norm(seed, 916, c["F"])
    attn = F.Attention(c["nh"], c["nkv"], c["hd"], c["smax"], 500000.0, neox=True)
    plans = [F.Plan([dict(w=W[0], x=hidden, gamma=n1, eps=EPS, y16=q), dict(w=W[1], x=hidden, gamma=n1, eps=EPS, y16=k),
                     dict(w=W[2], x=hidden, gamma=n1, eps=EPS, y16=v)]),
             F.Plan([dict(w=W[3], x=o, gamma=n2, eps=EPS, resid=hidden)]),
             F.Plan([dict(w=W[4], x=hidden, gamma=n3, eps=EPS, y16=gate),
                     dict(w=W[5], x=hidden, gamma=n3, eps=EPS, y16=up)]),
             F.Plan([dict(w=W[6], x=gate, up=up, gamma=n4, eps=EPS, resid=hidden)])]

    def step():
        F.embed_f16(emb, token, hidden)
        plans[0].launch()
        attn.decode(q, k, v, kc, vc, pos, o)
        for p in plans[1:]:
            p.launch()
    keep = (W, q, k, v, emb, token, pos, n1, n2, n3, n4, attn, plans)
    return dict(graph=_capture(step), out=[hidden, o, gate, up, kc, vc], keep=keep)


def _llama_shape(c):
    return llama.Shape(H=c["H"], F=c["F"], Nl=c["L"], Nh=c["nh"], Nkv=c["nkv"], Hd=c["hd"], V=c["V"], eps=EPS,
                       rope_theta=500000.0)


def _prep_decode(c, seed):
    names = llama.PROJ
    layers = []
    for l in range(c["L"]):
        W = {nm: _weight(seed, 10 * l + i, *_proj(c)[i]) for i, nm in enumerate(names)}
        layers.append(llama.Layer(W, _norm(seed, 3000 + 2 * l, c["H"]), _norm(seed, 3001 + 2 * l, c["H"])))
    emb = (_randn(seed, 920, 64, c["H"]) * 2.0).to(torch.float16)  # (the lookup reads one row)
    emb = emb.repeat((c["V"] + 63) // 64, 1)[:c["V"]].contiguous()
    m = llama.Model(_llama_shape(c), layers, emb, _norm(seed, 921, c["H"]), _weight(seed, 5000, c["H"], c["V"]))
    d = llama.Decoder(m, c["smax"])
    d.K.copy_(_randn(seed, 922, *d.K.shape).to(torch.float16))
    d.V.copy_(_randn(seed, 923, *d.V.shape).to(torch.float16))

    def step():
        d.token.fill_(seed % 64)
        d.pos.fill_(c["pos"])
        d.step()
    return dict(graph=_capture(step), out=[d.logits, d.token, d.hidden, d.K, d.V], keep=d)


def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind == "gemv":
        s = dict(c=c, W=_weight(seed, 0, c["K"], c["N"]), a=_act(seed, c["act"], 0, c["K"]))
        dt = torch.float32 if c["out"] == "y" else torch.float16
        s["y"] = torch.empty(c["N"], dtype=dt, device="cuda")
        return s
    if kind == "mm_row":
        return dict(c=c, W=_weight(seed, 0, c["K"], c["N"]), x=_host_row(c, seed))
    if kind == "sweep":
        items = []
        out, ys = _slots(1, [N for _, N in _proj(c)] * c["L"])
        for i in range(7 * c["L"]):
            K, N = _proj(c)[i % 7]
            items.append(dict(w=_weight(seed, i, K, N), y=ys[i], **_act(seed + 17 * i, c["act"], 0, K)))
        return dict(c=c, plan=F.Plan(items), out=out)
    if kind == "layer":
        return dict(c=c, **_prep_layer(c, seed))
    if kind == "decode":
        return dict(c=c, **_prep_decode(c, seed))
    if kind == "gemm":
        return dict(c=c, W=_weight(seed, 0, c["K"], c["N"]), a=_act(seed, c["act"], c["M"], c["K"]))
    if kind == "ffn":
        a = _act(seed, "f32rms", c["M"], c["H"])
        return dict(c=c, W=[_weight(seed, 0, c["H"], c["F"]), _weight(seed, 1, c["H"], c["F"]),
                            _weight(seed, 2, c["F"], c["H"])], x=a["x"], gamma=a["gamma"],
                    gamma2=_norm(seed, 905, c["F"]))
    if kind == "msweep":
        items = []
        out, ys = _slots(c["M"], [N for _, N in _proj(c)] * c["L"])
        for i in range(7 * c["L"]):
            K, N = _proj(c)[i % 7]
            if i % 7 in (0, 3, 4, 6):  # Q, K, V and gate, up read one activation matrix
                a = _act(seed + 17 * i, "i8", c["M"], K)
            items.append(dict(w=_weight(seed, i, K, N), x=a["x"], x_scale_dev=a["x_scale_dev"], y=ys[i]))
        return dict(c=c, plan=F.GemmPlan(items), out=out)
    if kind == "tail":
        emb = (_randn(seed, 930, c["V"], c["H"]) * 0.03).to(torch.float16)
        return dict(c=c, emb=emb, x=_randn(seed, 931, c["H"]), gamma=_norm(seed, 932, c["H"]),
                    token=torch.zeros(1, dtype=torch.int32, device="cuda"), state=F.ArgmaxState(),
                    logits=torch.empty(c["V"], dtype=torch.float16, device="cuda"))
    t = _trits(seed, 0, c["K"], c["N"])
    return dict(c=c, raw=_i2s(t) if c["src"] == "i2s" else _v11(t), scale=_wscale(seed, 0, c["K"]))


def run(s):
    c = s["c"]
    kind = c["kind"]
    if kind == "gemv":
        if c["act"] == "i8" and c["out"] == "y":
            return F.mm_packed_dispatch(s["a"]["x"], s["a"]["x_scale_dev"], s["W"], s["y"], c["K"], c["N"])
        if c["act"] == "i8":
            return F.mm_packed_dispatch_f16(s["a"]["x"], s["a"]["x_scale_dev"], s["W"], s["y"], c["K"], c["N"])
        F.gemv(s["W"], eps=EPS, **s["a"], **{c["out"]: s["y"]})
        return s["y"]
    if kind == "mm_row":
        return F.mm_row(s["x"], 0, 0.0123, s["W"], c["K"], c["N"])
    if kind in ("sweep", "msweep"):
        s["plan"].launch()
        return s["out"]
    if kind in ("layer", "decode"):
        s["graph"].replay()
        return s["out"]
    if kind == "gemm":
        a = dict(s["a"])
        x = a.pop("x")
        if c["out"] == "y":
            return F.mm_batched(s["W"], x, eps=EPS, **a)[0]
        y16 = torch.empty((c["M"], c["N"]), dtype=torch.float16, device="cuda")
        F.mm_batched(s["W"], x, eps=EPS, y16=y16, **a)
        return y16
    if kind == "ffn":
        M, W = c["M"], s["W"]
        gate = torch.empty((M, c["F"]), dtype=torch.float16, device="cuda")
        up = torch.empty_like(gate)
        q, qs = F.rmsnorm_quant(s["x"], s["gamma"], EPS)
        F.mm_batched(W[0], q, x_scale_dev=qs, y16=gate)
        F.mm_batched(W[1], q, x_scale_dev=qs, y16=up)
        y, _ = F.mm_batched(W[2], gate, up=up, gamma=s["gamma2"], eps=EPS)
        return [gate, up, y]
    if kind == "tail":
        F.lm_head_argmax(s["x"], s["gamma"], s["emb"], EPS, token_out=s["token"], state=s["state"],
                         logits_out=s["logits"])
        return [s["logits"], s["token"]]
    load = F.PackedTrits.from_i2s if c["src"] == "i2s" else F.PackedTrits.from_v11
    return load(s["raw"], c["K"], c["N"], s["scale"]).to_v11()


def work(case):
    c, kind = case, case["kind"]
    el = {"i8": 1, "f32": 4, "f32rms": 4, "f16rms": 2, "relu2": 4, "f16": 2, "silu": 4}
    if kind in ("gemv", "mm_row", "gemm"):
        M, K, N = c.get("M", 1), c["K"], c["N"]
        if kind == "mm_row":
            return {"bytes": K * N // 4 + 2 * K + 4 * N, "flops": 2 * K * N}
        ob = 4 if c["out"] == "y" else 2
        return {"bytes": K * N // 4 + M * K * el[c["act"]] + M * N * ob, "flops": 2 * M * K * N}
    if kind == "ffn":
        M, H, Fd = c["M"], c["H"], c["F"]
        return {"bytes": 3 * H * Fd // 4 + M * H * 4 + 2 * M * Fd * 2 + M * H * 4, "flops": 6 * M * H * Fd}
    if kind in ("sweep", "msweep"):
        M = c.get("M", 1)
        P = _proj(c)
        xin = sum(P[i][0] for i in ((0, 3, 4, 6) if M > 1 else range(7)))
        xb = el[c["act"]] if kind == "sweep" else 1
        return {"bytes": c["L"] * (sum(K * N for K, N in P) // 4 + M * xin * xb + 4 * M * sum(N for _, N in P)),
                "flops": 2 * M * c["L"] * sum(K * N for K, N in P)}
    if kind in ("layer", "decode"):
        P, L = _proj(c), c.get("L", 1)
        n = sum(K * N for K, N in P)
        kv = 2 * (c["pos"] + 1) * c["nkv"] * c["hd"]
        b = L * (n // 4 + 2 * kv + 4 * c["H"])
        f = L * (2 * n + 2 * kv * (c["nh"] // c["nkv"]))
        if kind == "decode":
            b += c["H"] * c["V"] // 4 + 2 * c["V"]
            f += 2 * c["H"] * c["V"]
        return {"bytes": b, "flops": f}
    if kind == "tail":
        return {"bytes": 2 * c["V"] * c["H"] + 6 * c["H"] + 2 * c["V"], "flops": 2 * c["V"] * c["H"]}
    return {"bytes": 3 * c["K"] * c["N"] // 4, "flops": 0}


def tolerance(case):
    """About four times the largest difference from exact() measured over the
    listed and drawn cases of the kind; the integer sums are exact, so with
    int8 rows only the two fp32 multiplications of the scales round."""
    c, kind = case, case["kind"]
    if kind == "convert":
        return "exact"
    if c.get("out") == "y16":
        return {"rel": 1e-3}
    if kind == "mm_row" or c.get("act") == "i8" or kind == "msweep":
        return {"rel": 4e-7}
    if kind in ("gemv", "gemm", "sweep"):
        return {"rel": 1e-3}
    return {"rel": {"ffn": 1e-2, "layer": 5e-2, "tail": 1.2e-3, "decode": 1e-1}[kind]}


# ---- the same results in 64 bits --------------------------------------------

def _d(t):
    return t.to(torch.float64)


def _h(x):
    """Rounded to fp16 where the path stores a vector as fp16 between two steps
    (left out, the int8 codes behind it flip and every later layer moves)."""
    return x.to(torch.float16).to(torch.float64)


def _rms(x, gamma):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * _d(gamma)


def _quant(x):
    """int8 codes (as float64) and step of each row: the activation quantizer."""
    s = 127.0 / (x.abs().amax(-1, keepdim=True) + 1e-9)
    return torch.clamp(torch.round(x * s), -128, 127), 1.0 / s


def _mm(q, step, seed, i, K, N):
    ws = float(np.float32(_wscale(seed, i, K)))
    y = torch.empty((q.shape[0], N), dtype=torch.float64, device="cuda")
    t = _trits(seed, i, K, N)
    for n in range(0, N, 16384):  # (columns in pieces: the wide vocabulary matrices)
        y[:, n:n + 16384] = q @ _d(t[:, n:n + 16384])
    return y * step * ws


def _act64(seed, act, M, K):
    a = _act(seed, act, M, K)
    x = _d(a["x"]).reshape(-1, K)
    if act == "i8":
        return x, _d(a["x_scale_dev"]).reshape(-1, 1)
    if act == "relu2":
        x = torch.relu(x) ** 2 * _d(a["up"]).reshape(-1, K)
    if act == "silu":
        x = x * torch.sigmoid(x) * _d(a["up"]).reshape(-1, K)
    if "gamma" in a:
        x = _rms(x, a["gamma"])
    return _quant(x)


def _rope(x, pos, hd, neox):
    k = torch.arange(hd // 2, device="cuda", dtype=torch.float64)
    ang = pos * 500000.0 ** (-2.0 * k / hd)
    cs, sn = torch.cos(ang), torch.sin(ang)
    x = x.reshape(-1, hd)
    a, b = (x[:, :hd // 2], x[:, hd // 2:]) if neox else (x[:, 0::2], x[:, 1::2])
    ra, rb = a * cs - b * sn, a * sn + b * cs
    return torch.cat([ra, rb], -1) if neox else torch.stack([ra, rb], -1).reshape(x.shape)


def _attend(c, q, k, v, kc, vc, neox):
    """Attention of one position; returns the output and writes the caches."""
    p, nh, nkv, hd = c["pos"], c["nh"], c["nkv"], c["hd"]
    kc[p] = _h(_rope(k, p, hd, neox))
    vc[p] = v.reshape(nkv, hd)
    qr = _h(_rope(q, p, hd, neox)).reshape(nkv, nh // nkv, hd)
    sc = torch.einsum("gqd,sgd->gqs", qr, kc[:p + 1]) / math.sqrt(hd)
    return torch.einsum("gqs,sgd->gqd", torch.softmax(sc, -1), vc[:p + 1]).reshape(1, nh * hd)


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "gemv":
        q, s = _act64(seed, c["act"], 0, c["K"])
        return _mm(q, s, seed, 0, c["K"], c["N"])[0]
    if kind == "mm_row":
        x = torch.from_numpy(_host_row(c, seed)).cuda()
        return _mm(_d(x), float(np.float32(0.0123)), seed, 0, c["K"], c["N"])[0].cpu().numpy()
    if kind in ("sweep", "msweep"):
        out = []
        for i in range(7 * c["L"]):
            K, N = _proj(c)[i % 7]
            if kind == "sweep" or i % 7 in (0, 3, 4, 6):
                q, s = _act64(seed + 17 * i, c.get("act", "i8"), c.get("M", 0), K)
            y = _mm(q, s, seed, i, K, N).reshape(-1)
            out.append(torch.nn.functional.pad(y, (0, -y.numel() % 64)))
        return torch.cat(out)
    if kind == "gemm":
        q, s = _act64(seed, c["act"], c["M"], c["K"])
        return _mm(q, s, seed, 0, c["K"], c["N"])
    if kind == "ffn":
        q, s = _act64(seed, "f32rms", c["M"], c["H"])
        gate, up = _mm(q, s, seed, 0, c["H"], c["F"]), _mm(q, s, seed, 1, c["H"], c["F"])
        q, s = _quant(_rms(torch.relu(_h(gate)) ** 2 * _h(up), _norm(seed, 905, c["F"])))
        return [gate, up, _mm(q, s, seed, 2, c["F"], c["H"])]
    if kind == "layer":
        P, H = _proj(c), c["H"]
        h = _d(_randn(seed, 910, 64, H).to(torch.float16)[seed % 64]).reshape(1, H)
        kc = _d(_randn(seed, 911, c["smax"], c["nkv"], c["hd"]).to(torch.float16))
        vc = _d(_randn(seed, 912, c["smax"], c["nkv"], c["hd"]).to(torch.float16))
        qs = _quant(_rms(h, _norm(seed, 913, H)))
        o = _attend(c, *[_h(_mm(*qs, seed, i, *P[i])) for i in range(3)], kc, vc, True)
        h = h + _h(_mm(*_quant(_rms(_h(o), _norm(seed, 914, c["nh"] * c["hd"]))), seed, 3, *P[3]))
        qs = _quant(_rms(h, _norm(seed, 915, H)))
        gate, up = _mm(*qs, seed, 4, *P[4]), _mm(*qs, seed, 5, *P[5])
        f = _rms(torch.relu(_h(gate)) ** 2 * _h(up), _norm(seed, 916, c["F"]))
        h = h + _h(_mm(*_quant(f), seed, 6, *P[6]))
        return [h[0], o[0], gate[0], up[0], kc, vc]
    if kind == "decode":
        P, H = _proj(c), c["H"]
        h = _d((_randn(seed, 920, 64, H) * 2.0).to(torch.float16)[seed % 64]).reshape(1, H)
        cs = (c["L"], c["smax"], c["nkv"], c["hd"])
        kc, vc = (_d(_randn(seed, i, *cs).to(torch.float16)) for i in (922, 923))
        for l in range(c["L"]):
            w = lambda i, qs: _h(_mm(*qs, seed, 10 * l + i, *P[i]))
            qs = _quant(_rms(h, _norm(seed, 3000 + 2 * l, H)))
            o = _attend(c, w(0, qs), w(1, qs), w(2, qs), kc[l], vc[l], False)
            h = _h(h + w(3, _quant(_h(o))))
            qs = _quant(_rms(h, _norm(seed, 3001 + 2 * l, H)))
            gate = w(4, qs)
            h = _h(h + w(6, _quant(gate * torch.sigmoid(gate) * w(5, qs))))
        logits = _mm(*_quant(_rms(h, _norm(seed, 921, H))), seed, 5000, H, c["V"])[0]
        return [logits, None, h[0], kc, vc]
    if kind == "tail":
        emb = (_randn(seed, 930, c["V"], c["H"]) * 0.03).to(torch.float16)
        x = _rms(_d(_randn(seed, 931, c["H"])), _norm(seed, 932, c["H"]))
        y = torch.empty(c["V"], dtype=torch.float64, device="cuda")
        for r in range(0, c["V"], 16384):
            y[r:r + 16384] = _d(emb[r:r + 16384]) @ x
        return [y, None]
    return _v11(_trits(seed, 0, c["K"], c["N"]))
