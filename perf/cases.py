"""Performance cases of the quantized-matmul backend: the calls a GGUF inference program makes, through the C ABI.

Four kinds of case, told apart by `kind`:

  host    one synchronous matmul with host A and C against an uploaded weight (`ggq_mul_mat`)
  layer   the matmuls of one or more transformer layers, one call per dependency level (q/k/v, o, gate/up, down), with
          `M` activation rows: decode (M = 1), a batch of sequences, or a prompt; optionally the vocabulary projection
          with the greedy token at the end.  `act` is the activation treatment (fp32, per-row int8, per-32-block int8)
  block   a decode token's layer with its neighbours: RMSNorm, SwiGLU and the residual adds fused into the matmuls, and
          attention over the layer's KV cache
  moe     one mixture-of-experts FFN layer: routing, SwiGLU experts, weighted combine, shared expert

Weights are blocks of N(0, 0.02) values (real codes and scales), activations N(0, 1), as in the benchmark.
"""
import ctypes
import functools

import numpy as np
import torch

import ggnpu_amd.lib as gl

F32, Q8_ROW, Q8_BLOCK32 = 0, 1, 2
TYPES = {t.name: int(t) for t in gl.GgmlType}
BLOCK = {int(t): b for t, b in gl.BLOCK.items()}  # type -> (values, bytes) of a block


# ---------------------------------------------------------------- the cases

def _layer(name, M, act, H, F, NQ, NKV, types, layers=1, vocab=0, ragged=0):
    return dict(name=name, kind="layer", M=M, act=act, H=H, F=F, NQ=NQ, NKV=NKV, types=types, layers=layers,
                vocab=vocab, ragged=ragged)


# types of q, k, v, o, gate, up, down (and the vocabulary projection)
Q4_K_M = "Q4_K,Q4_K,Q6_K,Q4_K,Q4_K,Q4_K,Q6_K,Q4_K"
ALL_Q8_0 = ",".join(["Q8_0"] * 8)
IQ4_MIX = "IQ4_NL,IQ4_XS,Q5_K,IQ4_NL,IQ4_XS,Q5_K,IQ4_NL,IQ4_XS"


def listed():
    return [
        # a host program's single call, as the backend interface issues it: launch and PCIe latency
        dict(name="host_gemv_q4k", kind="host", type="Q4_K", N=2048, K=2048, M=1, act=F32),
        # one token of a small model: the smallest launches
        _layer("decode_iq4_0.6b", 1, F32, 1024, 3072, 2048, 1024, IQ4_MIX),
        # eight sequences of the same model decoded together
        _layer("decode_iq4_0.6b_b8", 8, F32, 1024, 3072, 2048, 1024, IQ4_MIX),
        # the whole matmul work of one token of a 1B model with the logits and the greedy token
        _layer("decode_step_1b", 1, F32, 2048, 8192, 2048, 512, Q4_K_M, layers=16, vocab=128256),
        # one layer of the same model as a decoder runs it, at a long context
        dict(name="decode_block_1b", kind="block", H=2048, F=8192, heads=32, kv_heads=8, head_dim=64, ctx=6000,
             types=Q4_K_M),
        # a server's batch of 32 sequences
        _layer("decode_1b_b32", 32, F32, 2048, 8192, 2048, 512, Q4_K_M),
        # a prompt with fp32 activations (the reference's CPU semantics), ragged length
        _layer("prefill_1b_f32", 500, F32, 2048, 8192, 2048, 512, Q4_K_M),
        # a prompt with per-row int8 activations (the reference's NPU semantics): Q8_0 and the K-quant mix
        _layer("prefill_1.5b_q8_0", 512, Q8_ROW, 1536, 8960, 1536, 256, ALL_Q8_0),
        _layer("prefill_1b_q8row", 1023, Q8_ROW, 2048, 8192, 2048, 512, Q4_K_M),
        # MoE: one token, a batch of sequences, a prompt
        dict(name="moe_1", kind="moe", T=1, H=2048, F=512, E=256, top_k=8, shared=True, act=F32, types="Q4_K,Q4_K,Q6_K"),
        dict(name="moe_64", kind="moe", T=64, H=2048, F=512, E=256, top_k=8, shared=True, act=F32,
             types="Q4_K,Q4_K,Q6_K"),
        dict(name="moe_512_q8row", kind="moe", T=512, H=2048, F=512, E=256, top_k=8, shared=True, act=Q8_ROW,
             types="Q4_K,Q4_K,Q6_K"),
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def _types(rng, n):
    if rng.random() < 0.4:
        return ",".join([rng.choice(sorted(TYPES))] * n)
    if rng.random() < 0.4:
        return ",".join(Q4_K_M.split(",")[:n]) if n == 8 else "Q4_K,Q4_K,Q6_K"
    return ",".join(rng.choice(sorted(TYPES)) for _ in range(n))


def _draw(rng):
    kind = rng.choice(["host", "layer", "layer", "layer", "layer", "block", "moe", "moe"])
    if kind == "host":
        return dict(kind=kind, type=rng.choice(sorted(TYPES)), N=_log(rng, 200, 9000), K=256 * _log(rng, 2, 32),
                    M=rng.choice([1, 1, 2, 5, 17]), act=rng.choice([F32, F32, Q8_ROW]))
    if kind == "layer":
        H = 256 * rng.randint(4, 8)
        M = rng.choice([1, 1, _log(rng, 2, 64), _log(rng, 65, 1023), _log(rng, 65, 1023)])
        act = rng.choice([F32, F32, Q8_ROW, Q8_ROW, Q8_BLOCK32])
        c = _layer("", M, act, H, 256 * _log(rng, 12, 35), H, 128 * rng.randint(1, 8), _types(rng, 8),
                   layers=rng.choice([1, 2]), vocab=rng.choice([0, 0, _log(rng, 8000, 128256)]) if M == 1 else 0,
                   ragged=rng.choice([0, 0, rng.randint(1, 40)]))
        del c["name"]
        return c
    if kind == "block":
        hd = rng.choice([64, 128])
        kv = rng.choice([2, 4, 8])
        heads = kv * rng.choice([1, 2, 4])
        return dict(kind=kind, H=256 * rng.randint(4, 8), F=256 * _log(rng, 12, 32), heads=max(heads, 256 // hd),
                    kv_heads=kv, head_dim=hd, ctx=_log(rng, 100, 16384), types=_types(rng, 8))
    E = rng.choice([32, 64, 128, 256])
    return dict(kind=kind, T=rng.choice([1, 1, _log(rng, 2, 64), _log(rng, 64, 512)]), H=256 * rng.randint(4, 8),
                F=256 * rng.randint(1, 3), E=E, top_k=rng.choice([2, 4, 6, 8]), shared=rng.random() < 0.7,
                act=rng.choice([F32, F32, Q8_ROW]), types=_types(rng, 3))


@functools.lru_cache(maxsize=1)
def _most():
    w = [work(c) for c in listed()]
    return {k: max(v[k] for v in w) for k in ("bytes", "flops")}


def draw(rng):
    most = _most()
    while True:
        c = _draw(rng)
        w = work(c)
        if w["bytes"] <= most["bytes"] and w["flops"] <= most["flops"]:
            return c


# ------------------------------------------------------------------- shapes

def _names(case):
    return [TYPES[t] for t in case["types"].split(",")]


def _levels(case):
    """The dependency levels of one layer: lists of (type, N, K) that share an input."""
    tq, tk, tv, to, tg, tu, td = _names(case)[:7]
    H, F, r = case["H"], case["F"], case.get("ragged", 0)
    nq, nkv = case["NQ"], case["NKV"]
    return [[(tq, nq + r, H), (tk, nkv + r, H), (tv, nkv + r, H)], [(to, H + r, nq)],
            [(tg, F + r, H), (tu, F + r, H)], [(td, H + r, F)]]


def _block_case(case):
    return dict(case, NQ=case["heads"] * case["head_dim"], NKV=case["kv_heads"] * case["head_dim"])


def _experts_hit(case):
    """Experts that T tokens with independent top-k choices hit, on average."""
    return case["E"] * (1.0 - (1.0 - case["top_k"] / case["E"]) ** case["T"])


def work(case):
    def mm(t, N, K, M):
        return gl.row_bytes(t, K) * N, 2 * M * N * K

    b = f = 0
    if case["kind"] == "host":
        M, N, K = case["M"], case["N"], case["K"]
        b, f = mm(TYPES[case["type"]], N, K, M)
        b += 4 * M * (N + K)
    elif case["kind"] == "layer":
        M = case["M"]
        for lv in _levels(case):
            b += 4 * M * lv[0][2]
            for t, N, K in lv:
                wb, wf = mm(t, N, K, M)
                b, f = b + wb + 4 * M * N, f + wf
        b, f = b * case["layers"], f * case["layers"]
        if case["vocab"]:
            wb, wf = mm(_names(case)[7], case["vocab"], case["H"], M)
            b, f = b + wb + 4 * (case["vocab"] + case["H"]), f + wf
    elif case["kind"] == "block":
        for lv in _levels(_block_case(case)):
            for t, N, K in lv:
                wb, wf = mm(t, N, K, 1)
                b, f = b + wb, f + wf
        kv = case["kv_heads"] * case["head_dim"] * case["ctx"]
        b += 2 * 4 * kv + 4 * (2 * case["H"] + 2 * case["H"])
        f += 4 * case["heads"] * case["head_dim"] * case["ctx"]
    else:
        T, H, F, k = case["T"], case["H"], case["F"], case["top_k"]
        tg, tu, td = _names(case)
        per = [mm(tg, F, H, 1), mm(tu, F, H, 1), mm(td, H, F, 1)]
        one = sum(p[0] for p in per)
        b = one * (_experts_hit(case) + (1 if case["shared"] else 0)) + 4 * T * (2 * H + case["E"])
        f = sum(p[1] for p in per) * T * (k + (1 if case["shared"] else 0))
    return {"bytes": int(b), "flops": int(f)}


def tolerance(case):
    # fp32 sums of exact products: about four times the error against exact() (2e-8 ... 6e-7 over the ranges)
    if case["kind"] == "moe":
        # per-row int8: an int8 code of a SwiGLU row changes where the value lies within fp32 rounding of a half-integer
        return {"rel": 1e-3} if case["act"] == Q8_ROW else {"rel": 3e-6}
    return {"rel": 3e-6}


# -------------------------------------------------------------------- inputs

@functools.lru_cache(maxsize=8)
def _pool(t, seed):
    """Blocks of N(0, 0.02) values, encoded once on the host."""
    be, bb = BLOCK[t]
    n = 2048 * 256
    x = np.random.default_rng([seed, t]).standard_normal((n // 2048, 2048), dtype=np.float32) * np.float32(0.02)
    return torch.from_numpy(gl.encode(t, x).reshape(n // be, bb))


class _Source:
    def __init__(self, seed):
        self.seed = seed
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(seed)
        self.pools = {}

    def weight(self, t, rows, K):
        """Raw blocks of a [rows][K] matrix on the GPU, 256 bytes of padding after them."""
        be, bb = BLOCK[t]
        if t not in self.pools:
            self.pools[t] = _pool(t, self.seed).cuda()
        pool = self.pools[t]
        idx = torch.randint(0, pool.shape[0], (rows * (K // be),), generator=self.gen, device="cuda")
        w = torch.zeros(idx.numel() * bb + 256, dtype=torch.uint8, device="cuda")
        torch.index_select(pool, 0, idx, out=w[: idx.numel() * bb].view(-1, bb))
        return w

    def normal(self, *shape):
        return torch.randn(shape, generator=self.gen, device="cuda")


def _empty(*shape):
    return torch.empty(shape, dtype=torch.float32, device="cuda")


def _stream():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


def prepare(case, seed):
    ctx = gl.Context(0)
    return {"case": case, "ctx": ctx, **globals()["_prepare_" + case["kind"]](case, _Source(seed), ctx)}


def run(state):
    return globals()["_run_" + state["case"]["kind"]](state)


def exact(case, seed):
    return globals()["_exact_" + case["kind"]](case, _Source(seed))


# ---------------------------------------------------------------------- host

def _host_inputs(case, src):
    w = src.weight(TYPES[case["type"]], case["N"], case["K"])
    return w, src.normal(case["M"], case["K"])


def _prepare_host(case, src, ctx):
    w, a = _host_inputs(case, src)
    raw = w[:-256].cpu().numpy()
    h = ctypes.c_void_p()
    ctx.check(ctx.lib.ggq_weight_upload(ctx.h, raw.ctypes.data, TYPES[case["type"]], case["N"], case["K"],
                                        ctypes.byref(h)), "weight_upload")
    return {"w": h, "A": a.cpu().numpy(), "C": np.empty((case["M"], case["N"]), np.float32)}


def _run_host(s):
    c, ctx = s["case"], s["ctx"]
    ctx.check(ctx.lib.ggq_mul_mat(ctx.h, s["w"], s["A"].ctypes.data, c["K"], s["C"].ctypes.data, c["N"], c["M"],
                                  c["act"]), "mul_mat")
    return s["C"]


def _exact_host(case, src):
    w, a = _host_inputs(case, src)
    return _matmul(a, case["act"], w, TYPES[case["type"]], case["N"], case["K"]).cpu().numpy()


# --------------------------------------------------------------------- layer

def _layer_inputs(case, src):
    """[(A, [(type, N, K, W)])] of every dependency level, and the vocabulary projection's."""
    levels = [(src.normal(case["M"], lv[0][2]), [(t, N, K, src.weight(t, N, K)) for t, N, K in lv])
              for _ in range(case["layers"]) for lv in _levels(case)]
    vocab = None
    if case["vocab"]:
        t, N, K = _names(case)[7], case["vocab"], case["H"]
        vocab = (src.normal(1, K), (t, N, K, src.weight(t, N, K)))
    return levels, vocab


def _out_places(case, levels):
    """Where each matrix's output [M][N] starts (in floats) in its layer's output buffer, and the buffers' sizes."""
    places, sizes = [], [0] * case["layers"]
    for i, (_, mats) in enumerate(levels):
        layer = i * case["layers"] // len(levels)
        for _, N, _, _ in mats:
            places.append((layer, sizes[layer]))
            sizes[layer] += (case["M"] * N + 63) // 64 * 64
    return places, sizes


def _prepare_layer(case, src, ctx):
    M, act = case["M"], case["act"]
    levels, vocab = _layer_inputs(case, src)
    plan, keep = [], [levels]
    places, sizes = _out_places(case, levels)
    outs = [torch.zeros(n, dtype=torch.float32, device="cuda") for n in sizes]
    place = iter(places)
    for A, mats in levels:
        C = [outs[layer][at:] for _, (layer, at) in zip(mats, place)]
        K = mats[0][2]
        if act == Q8_ROW and M > 8:
            # a prompt: the level's input quantized once, weights of one type in one launch
            q, sa = torch.empty((M, K), dtype=torch.int8, device="cuda"), _empty(M)
            keep.append((q, sa))
            groups = []
            for t in dict.fromkeys(m[0] for m in mats):
                same = [(m, c) for m, c in zip(mats, C) if m[0] == t]
                d = (gl.GemmDesc * len(same))()
                for i, (m, c) in enumerate(same):
                    d[i].W, d[i].N, d[i].C, d[i].ldc = m[3].data_ptr(), m[1], c.data_ptr(), m[1]
                groups.append((t, d, len(same)))
            plan.append(("q8", A.data_ptr(), K, q.data_ptr(), sa.data_ptr(), groups))
        elif M <= 64 and (len(mats) > 1 or act != F32):
            d = (gl.GemvDesc * len(mats))()
            for i, (m, c) in enumerate(zip(mats, C)):
                d[i].W, d[i].type, d[i].N, d[i].K = m[3].data_ptr(), m[0], m[1], m[2]
                d[i].A, d[i].C = A.data_ptr(), c.data_ptr()
            plan.append(("batch", d, len(mats)))
        else:
            plan += [("one", m[3].data_ptr(), m[0], m[1], m[2], A.data_ptr(), c.data_ptr()) for m, c in zip(mats, C)]
    state = {"plan": plan, "outs": outs, "keep": keep, "vocab": None}
    if vocab:
        A, (t, N, K, w) = vocab
        logits, token, value = _empty(1, N), torch.zeros(1, dtype=torch.int32, device="cuda"), _empty(1)
        keep.append((A, w))
        state["vocab"] = (w.data_ptr(), t, N, K, A.data_ptr(), logits.data_ptr(), token.data_ptr(), value.data_ptr())
        state["outs"] = outs + [logits, token, value]
    return state


def _run_layer(s):
    c, ctx, stream = s["case"], s["ctx"], _stream()
    M, act, lib, h = c["M"], c["act"], ctx.lib, ctx.h
    for p in s["plan"]:
        if p[0] == "batch":
            ctx.check(lib.ggq_mul_mat_batch_act_dev(h, p[1], p[2], M, act, stream), "batch")
        elif p[0] == "one":
            _, w, t, N, K, A, C = p
            ctx.check(lib.ggq_mul_mat_dev(h, w, t, N, K, A, K, C, N, M, act, stream), "mul_mat")
        else:
            _, A, K, q, sa, groups = p
            ctx.check(lib.ggq_quantize_act_dev(h, A, K, M, K, act, q, sa, stream), "quantize")
            for t, d, n in groups:
                ctx.check(lib.ggq_mul_mat_q8_batch_dev(h, d, n, t, K, q, sa, M, stream), "q8 batch")
    if s["vocab"]:
        w, t, N, K, A, logits, token, value = s["vocab"]
        ctx.check(lib.ggq_logits_argmax_dev(h, w, t, N, K, A, M, act, logits, token, value, stream), "logits")
    return s["outs"]


def _exact_layer(case, src):
    levels, vocab = _layer_inputs(case, src)
    places, sizes = _out_places(case, levels)
    outs = [torch.zeros(n, dtype=torch.float64, device="cuda") for n in sizes]
    place = iter(places)
    for A, mats in levels:
        for (t, N, K, w), (layer, at) in zip(mats, place):
            outs[layer][at:at + case["M"] * N] = _matmul(A, case["act"], w, t, N, K).view(-1)
    if vocab:
        A, (t, N, K, w) = vocab
        logits = _matmul(A, case["act"], w, t, N, K)
        outs += [logits, None, logits.max(dim=1).values]
    return outs


# --------------------------------------------------------------------- block

def _block_inputs(case, src):
    c = _block_case(case)
    H, hd, ctx_len = c["H"], c["head_dim"], c["ctx"]
    mats = [[(t, N, K, src.weight(t, N, K)) for t, N, K in lv] for lv in _levels(c)]
    x = src.normal(1, H)
    norms = [1.0 + 0.1 * src.normal(H) for _ in range(2)]
    cache = [src.normal(ctx_len, c["kv_heads"] * hd) for _ in range(2)]
    return mats, x, norms, cache


def _prepare_block(case, src, ctx):
    mats, x, norms, (kc, vc) = _block_inputs(case, src)
    (q, k, v), (o,), (g, u), (dn,) = mats
    pos = case["ctx"] - 1
    bufs = {n: _empty(1, N) for n, N in (("q", q[1]), ("att", q[1]), ("x1", o[1]), ("g", g[1]), ("u", u[1]), ("x2", dn[1]))}

    def desc(m, A, C, rms=None, res=None, up=None, silu=0):
        d = gl.GemvFusedDesc()
        d.W, d.type, d.N, d.K, d.A, d.C = m[3].data_ptr(), m[0], m[1], m[2], A.data_ptr(), C.data_ptr()
        d.silu = silu
        if rms is not None:
            d.rms_norm, d.rms_eps, d.rms_w = 1, 1e-5, rms.data_ptr()
        if res is not None:
            d.residual = res.data_ptr()
        if up is not None:
            d.A_up = up.data_ptr()
        return d

    b = bufs
    levels = [[desc(q, x, b["q"], rms=norms[0]), desc(k, x, kc[pos], rms=norms[0]), desc(v, x, vc[pos], rms=norms[0])],
              [desc(o, b["att"], b["x1"], res=x)],
              [desc(g, b["x1"], b["g"], rms=norms[1], silu=1), desc(u, b["x1"], b["u"], rms=norms[1])],
              [desc(dn, b["g"], b["x2"], up=b["u"], res=b["x1"])]]
    plan = [((gl.GemvFusedDesc * len(lv))(*lv), len(lv)) for lv in levels]
    return {"plan": plan, "bufs": bufs, "kc": kc, "vc": vc, "keep": (mats, x, norms), "pos": pos}


def _run_block(s):
    c, ctx, stream, b = s["case"], s["ctx"], _stream(), s["bufs"]
    lib, h = ctx.lib, ctx.h
    for i, (d, n) in enumerate(s["plan"]):
        ctx.check(lib.ggq_mul_mat_fused_dev(h, d, n, 1, stream), "fused")
        if i == 0:
            ctx.check(lib.ggq_attention_decode_dev(h, b["q"].data_ptr(), s["kc"].data_ptr(), s["vc"].data_ptr(), 1,
                                                   c["heads"], c["kv_heads"], c["head_dim"], c["ctx"], s["pos"],
                                                   b["att"].data_ptr(), stream), "attention")
    return [b["q"], s["kc"][s["pos"]], s["vc"][s["pos"]], b["att"], b["x1"], b["g"], b["u"], b["x2"]]


def _exact_block(case, src):
    mats, x, norms, (kc, vc) = _block_inputs(case, src)
    (q, k, v), (o,), (g, u), (dn,) = mats
    hd, heads, kvh = case["head_dim"], case["heads"], case["kv_heads"]

    def mm(a, m):
        return a @ _dequant(m[3], m[0], m[1], m[2]).T

    def norm(a, w):
        return a / torch.sqrt((a * a).mean(dim=1, keepdim=True) + 1e-5) * w.double()

    def silu(a):
        return a / (1.0 + torch.exp(-a))

    x = x.double()
    n0 = norm(x, norms[0])
    qo, ko, vo = mm(n0, q), mm(n0, k), mm(n0, v)
    kc, vc = kc.double(), vc.double()
    kc[-1], vc[-1] = ko[0], vo[0]
    att = []
    for i in range(heads):
        j = i // (heads // kvh)
        s = kc[:, j * hd:(j + 1) * hd] @ qo[0, i * hd:(i + 1) * hd] / hd ** 0.5
        att.append(torch.softmax(s, 0) @ vc[:, j * hd:(j + 1) * hd])
    att = torch.cat(att).view(1, -1)
    x1 = x + mm(att, o)
    n1 = norm(x1, norms[1])
    go, uo = silu(mm(n1, g)), mm(n1, u)
    return [qo, ko[0], vo[0], att, x1, go, uo, x1 + mm(go * uo, dn)]


# ----------------------------------------------------------------------- moe

def _moe_inputs(case, src):
    T, H, F, E = case["T"], case["H"], case["F"], case["E"]
    shapes = list(zip(_names(case), ((F, H), (F, H), (H, F))))
    experts = [src.weight(t, E * n, k) for t, (n, k) in shapes]
    shared = [src.weight(t, n, k) for t, (n, k) in shapes] if case["shared"] else None
    return src.normal(T, H), src.normal(T, E), experts, shared, torch.sigmoid(src.normal(T))


def _prepare_moe(case, src, ctx):
    T, H, F, E, k = (case[n] for n in ("T", "H", "F", "E", "top_k"))
    x, logits, experts, shared, sw = _moe_inputs(case, src)
    out, wsel = _empty(T, H), _empty(T, k)
    sel = torch.empty((T, k), dtype=torch.int32, device="cuda")
    p = gl.MoeParams()
    p.T, p.H, p.F, p.E, p.top_k = T, H, F, E, k
    p.x, p.router_logits = x.data_ptr(), logits.data_ptr()
    p.gate_type, p.up_type, p.down_type = _names(case)
    p.gate_exps, p.up_exps, p.down_exps = (w.data_ptr() for w in experts)
    if shared:
        p.gate_shexp, p.up_shexp, p.down_shexp = (w.data_ptr() for w in shared)
        p.shared_w = sw.data_ptr()
    p.out, p.sel_experts, p.sel_weights = out.data_ptr(), sel.data_ptr(), wsel.data_ptr()
    return {"p": p, "outs": [out, sel, wsel], "keep": (x, logits, experts, shared, sw)}


def _run_moe(s):
    ctx = s["ctx"]
    ctx.check(ctx.lib.ggq_moe_ffn_act_dev(ctx.h, ctypes.byref(s["p"]), s["case"]["act"], _stream()), "moe")
    return s["outs"]


def _exact_moe(case, src):
    T, H, F, E, k = (case[n] for n in ("T", "H", "F", "E", "top_k"))
    x, logits, experts, shared, sw = _moe_inputs(case, src)
    shapes = list(zip(_names(case), ((F, H), (F, H), (H, F))))
    top, sel = torch.sort(logits, dim=1, descending=True, stable=True)
    sel, wsel = sel[:, :k], torch.softmax(top[:, :k].double(), dim=1)

    def ffn(rows, weights):
        a = _treat(rows, case["act"])
        g, u, d = (_dequant(w, t, n, kk) for w, (t, (n, kk)) in zip(weights, shapes))
        go, uo = a @ g.T, a @ u.T
        hid = go / (1.0 + torch.exp(-go)) * uo
        return (_treat(hid.float(), case["act"]) if case["act"] != F32 else hid) @ d.T

    out = torch.zeros((T, H), dtype=torch.float64, device="cuda")
    size = [n * gl.row_bytes(t, kk) for t, (n, kk) in shapes]
    for e in range(E):
        tok, slot = torch.nonzero(sel == e, as_tuple=True)
        if tok.numel():
            w = [ws[e * b:(e + 1) * b] for ws, b in zip(experts, size)]
            out.index_add_(0, tok, ffn(x[tok], w) * wsel[tok, slot].view(-1, 1))
    if shared:
        out += ffn(x, shared) * sw.double().view(-1, 1)
    return [out, None, wsel]


# ----------------------------------------- 64-bit values of blocks and inputs

def _treat(a, act):
    """Activations as the matmul sees them, in 64 bits: fp32 rows, or their int8 codes times their scales."""
    if act == F32:
        return a.double()
    v = a.view(a.shape[0], -1, 32) if act == Q8_BLOCK32 else a.view(a.shape[0], 1, -1)
    amax = v.abs().amax(dim=2, keepdim=True)
    s = torch.where(amax > 0, amax / torch.full_like(amax, 127.0), torch.ones_like(amax))
    q = torch.clamp(torch.round(v * (torch.ones_like(s) / s)), -128, 127)
    return (q.double() * s.double()).view(a.shape)


_IQ4 = [-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113]


def _dequant(w, t, rows, K):
    """The float64 matrix [rows][K] of raw GGUF blocks."""
    be, bb = BLOCK[t]
    b = w[: rows * (K // be) * bb].view(-1, bb)
    n = b.shape[0]

    def half(i):
        return b[:, i:i + 2].contiguous().view(torch.float16).double()

    def nibbles(x):  # [n, chunks, 32] bytes -> values in order: 32 low nibbles, 32 high nibbles of each chunk
        return torch.stack((x & 15, x >> 4), dim=2)

    if t == TYPES["Q8_0"]:
        out = b[:, 2:].view(torch.int8).double() * half(0)
    elif t in (TYPES["IQ4_NL"], TYPES["IQ4_XS"]):
        lut = torch.tensor(_IQ4, dtype=torch.float64, device=w.device)
        if t == TYPES["IQ4_NL"]:
            out = lut[nibbles(b[:, 2:].reshape(n, 1, 16)).long()].reshape(n, -1) * half(0)
        else:
            sh = b[:, 2].int() | (b[:, 3].int() << 8)
            ib = torch.arange(8, device=w.device)
            lo = (b[:, 4:8].int().repeat_interleave(2, dim=1) >> (4 * (ib & 1))) & 15
            ls = lo | (((sh.view(-1, 1) >> (2 * ib)) & 3) << 4)
            kv = lut[nibbles(b[:, 8:].reshape(n, 8, 16)).long()].reshape(n, 8, 32)
            out = kv * ((ls - 32).double() * half(0)).view(n, 8, 1)
    elif t == TYPES["Q6_K"]:
        ql, qh = b[:, :128].int().view(n, 2, 2, 32), b[:, 128:192].int().view(n, 2, 32)
        q = torch.stack([(ql[:, :, i & 1] >> (4 * (i >> 1)) & 15) | ((qh >> (2 * i) & 3) << 4) for i in range(4)], dim=2)
        sc = b[:, 192:208].contiguous().view(torch.int8).double() * half(208)
        out = (q - 32).double().view(n, 16, 16) * sc.view(n, 16, 1)
    else:
        s = b[:, 4:16].int()
        sc = torch.cat((s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)), dim=1).double() * half(0)
        mn = torch.cat((s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)), dim=1).double() * half(2)
        q = nibbles(b[:, bb - 128:].int().view(n, 4, 32)).view(n, 8, 32)
        if t == TYPES["Q5_K"]:
            bit = torch.arange(8, device=w.device).view(1, 8, 1)
            q = q + ((b[:, 16:48].int().view(n, 1, 32) >> bit & 1) << 4)
        out = q.double() * sc.view(n, 8, 1) - mn.view(n, 8, 1)
    return out.reshape(rows, K)


def _matmul(a, act, w, t, N, K):
    x = _treat(a, act)
    rb = gl.row_bytes(t, K)
    step = max(1, (1 << 26) // K)
    return torch.cat([x @ _dequant(w[i * rb:min(N, i + step) * rb], t, min(N, i + step) - i, K).T
                      for i in range(0, N, step)], dim=1)
