"""Performance cases of libnn-hip.so: the work that a program using this library has it do, through the
Python binding of the C ABI (neuralnet.cpp_amd/__init__.py) and the decoder over it (decoder.py).

A case is a dict of plain values with a "kind":

  linear        one BitLinear W1.58A8 layer on X (K, M): [RMSNorm ->] absmax -> int8, then the
                ternary x int8 product (+ bias)
  stack         the decode GEMVs of a whole layer stack in one grouped launch
  ffn           a decoder block's gated feed-forward half: RMSNorm -> int8 -> fc1 -> activation ->
                [SubLN ->] int8 -> fc2, plus the residual
  float_linear  one BitLinear layer with activation quantization off (the default branch): the
                ternary x float product
  train_linear  one training step's work in that layer: absmean and packing of the latent weights,
                forward, and the input gradient
  decode_attn   one layer's attention of a decode step over a KV cache, with RoPE and the append
  prefill_attn  one layer's cache fill and causal attention of a prompt
  decode_step   a whole decode step of a decoder (captured once in a graph, replayed per token)
  prompt        a whole prompt through a decoder, to the logits of each sequence's last token

The shapes are the BitNet-2B-class ones of bench.py (d 2560, 20 heads, 5 KV heads of 128, FFN 6912,
30 layers), the 4096 / 11008 GEMM shapes and 1024 x 1024 of its first configuration, and generic
odd sizes. Weights are random-init N(0, 0.02), ternarized per row by absmean, the decoder's o and
fc2 (which write to the residual stream) smaller by sqrt(2 x 30 layers) as decoders initialize
them; activations N(0, 1) with a share of large channels, as residual streams have them.
"""
import importlib.util
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
DEV = "cuda"
EPS = 1e-5


def _pkg():
    """The repository's package (its folder name holds a dot, so it is loaded by path)."""
    name = "nnhip_py"
    if name not in sys.modules:
        path = os.path.join(ROOT, "neuralnet.cpp_amd")
        spec = importlib.util.spec_from_file_location(name, os.path.join(path, "__init__.py"),
                                                      submodule_search_locations=[path])
        mod = importlib.util.module_from_spec(spec)
        sys.modules[name] = mod
        spec.loader.exec_module(mod)
    return sys.modules[name]


# ------------------------------------------------------------------------------------------ cases

def listed():
    return [
        # the smallest call: one token through a key / value projection
        dict(name="linear_1_token", kind="linear", K=2560, N=640, M=1, norm=True, bias=False),
        # a serving batch a little past the decode GEMV's 16 tokens, through the gate projection
        dict(name="linear_40_tokens", kind="linear", K=2560, N=6912, M=40, norm=True, bias=False),
        # a long prompt through one large projection, with a bias
        dict(name="linear_prompt", kind="linear", K=4096, N=11008, M=2048, norm=False, bias=True),
        # one token through the 210 projections of the 30-layer stack: the headline decode GEMV sweep
        dict(name="stack_1_token", kind="stack", layers=30, M=1),
        # the feed-forward half of a block over 2048 prompt tokens
        dict(name="ffn_prompt", kind="ffn", d=2560, F=6912, M=2048, act=0, subln=True),
        # one token through the down projection with float activations
        dict(name="float_linear_1_token", kind="float_linear", K=6912, N=2560, M=1, f16=False),
        # a training step's work in the gate projection, 2048 tokens in f32
        dict(name="train_linear", kind="train_linear", K=2560, N=6912, M=2048, f16=False),
        # 16 sequences around position 2112, f32 caches
        dict(name="decode_attn", kind="decode_attn", B=16, H=20, Hkv=5, dk=128, lo=1920, hi=2176, f16=False),
        # a prompt of 4 x 2048 tokens over f16 caches (compute = F16)
        dict(name="prefill_attn_f16", kind="prefill_attn", B=4, T=2048, H=20, Hkv=5, dk=128, pos0=0, f16=True),
        # the second chunk of a prompt, odd lengths, f32 caches
        dict(name="prefill_attn_chunk", kind="prefill_attn", B=3, T=1111, H=20, Hkv=5, dk=128, pos0=517, f16=False),
        # one token for each of 16 sequences through 8 of the decoder's layers at context 2048 (weights
        # and caches past the 256 MiB memory-side cache, as in the whole model)
        dict(name="decode_step", kind="decode_step", layers=8, B=16, ctx=2048, f16=True),
        # 8 prompts of 1024 tokens through two of the decoder's layers
        dict(name="prompt", kind="prompt", layers=2, B=8, T=1024, f16=False),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _dim(rng, lo, hi):
    """A feature count: one of the model shapes' more often than not, else any (odd ones too)."""
    known = [k for k in (640, 1024, 2560, 4096, 6912, 11008) if lo <= k <= hi]
    return rng.choice(known) if rng.random() < 0.6 else _log(rng, lo, hi)


def _heads(rng, long_dk):
    H, Hkv = rng.choice([(20, 5), (20, 5), (16, 16), (16, 2), (8, 4), (32, 8)])
    return H, Hkv, rng.choice([64, 128, 128] if not long_dk else [64, 128, 128, 256])


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "stack", "ffn", "ffn", "float_linear", "train_linear",
                       "decode_attn", "prefill_attn", "prefill_attn", "decode_step", "prompt"])
    if kind == "linear":
        return dict(kind=kind, K=_dim(rng, 256, 6912), N=_dim(rng, 256, 11008), M=_log(rng, 1, 2400),
                    norm=rng.random() < 0.5, bias=rng.random() < 0.3)
    if kind == "stack":
        return dict(kind=kind, layers=rng.randint(2, 30), M=_log(rng, 1, 16))
    if kind == "ffn":
        return dict(kind=kind, d=_dim(rng, 512, 2560), F=_dim(rng, 512, 6912), M=_log(rng, 1, 2048),
                    act=rng.randint(0, 1), subln=rng.random() < 0.7)
    if kind == "float_linear":
        return dict(kind=kind, K=_dim(rng, 256, 6912), N=_dim(rng, 256, 6912), M=_log(rng, 1, 1024),
                    f16=rng.random() < 0.3)
    if kind == "train_linear":
        return dict(kind=kind, K=_dim(rng, 256, 4096), N=_dim(rng, 256, 6912), M=_log(rng, 64, 2048),
                    f16=rng.random() < 0.3)
    if kind == "decode_attn":
        H, Hkv, dk = _heads(rng, True)
        hi = _log(rng, 16, 2300)
        return dict(kind=kind, B=rng.randint(1, 16), H=H, Hkv=Hkv, dk=dk, lo=rng.randint(0, hi - 1), hi=hi,
                    f16=rng.random() < 0.5)
    if kind == "prefill_attn":
        H, Hkv, dk = _heads(rng, False)
        T = _log(rng, 32, 2048)
        return dict(kind=kind, B=max(1, min(rng.randint(1, 8), 8192 // T)), T=T, H=H, Hkv=Hkv, dk=dk,
                    pos0=0 if rng.random() < 0.6 else rng.randint(1, 1024), f16=rng.random() < 0.5)
    if kind == "decode_step":
        return dict(kind=kind, layers=rng.randint(1, 8), B=rng.randint(1, 16), ctx=_log(rng, 64, 2048),
                    f16=rng.random() < 0.5)
    T = _log(rng, 24, 1024)
    return dict(kind=kind, layers=rng.randint(1, 2), B=rng.randint(1, 8), T=T, f16=rng.random() < 0.5)


# ----------------------------------------------------------------------------------------- inputs

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _weights(g, N, K, std=0.02):
    """N(0, std). The few values within 1e-5 of the ternary threshold, half their row's absmean, move a
    little past it: on which side of it 32-bit rounding puts them is no property of an implementation."""
    W = torch.randn((N, K), generator=g, device=DEV) * std
    t = 0.5 * W.abs().mean(1, keepdim=True, dtype=torch.float64).float()
    return torch.where((W.abs() - t).abs() < 1e-5 * t, W * 1.0001, W)


def _acts(g, K, M):
    """(K, M) activations: N(0, 1) with one channel in 128 eight times as large."""
    x = torch.randn((K, M), generator=g, device=DEV)
    big = torch.rand((K, 1), generator=g, device=DEV) < 1.0 / 128
    return torch.where(big, 8.0 * x, x).contiguous()


def _gamma(g, K):
    return 1.0 + 0.1 * torch.randn((K,), generator=g, device=DEV)


def _keys(g, rows, dk):
    """(rows, dk) attention inputs: N(0, 1) under a per-channel spread of scales."""
    return torch.randn((rows, dk), generator=g, device=DEV) * torch.exp(0.4 * torch.randn((1, dk), generator=g, device=DEV))


def _rope(dk, max_len):
    """cos, sin (max_len, dk / 2), the plan an attention caller keeps."""
    th = np.arange(max_len)[:, None] / np.power(10000.0, 2.0 * np.arange(dk // 2) / dk)[None, :]
    return [torch.from_numpy(f(th).astype(np.float32)).to(DEV) for f in (np.cos, np.sin)]


def _packed(ctx, W):
    """The layer's plan: per-row scale and repacked ternary words of W (N, K)."""
    tau = ctx.row_absmean(W)
    return ctx.repack(ctx.trit_pack(W, tau), W.shape[1]), tau


D, KV, FF, HEADS, KVH, DK, VOCAB = 2560, 640, 6912, 20, 5, 128, 10000
STACK = [(D, D), (D, KV), (D, KV), (D, D), (D, FF), (D, FF), (FF, D)]   # (K, N): q k v o gate up down
BLOCK = [("q", D, D), ("k", KV, D), ("v", KV, D), ("o", D, D), ("fc1", 2 * FF, D), ("fc2", D, FF)]   # name, N, K
RESIDUAL_STD = 0.02 / math.sqrt(2 * 30)


def _stack_weights(g, c):
    for _ in range(c["layers"]):
        for K, N in STACK:
            yield _weights(g, N, K), K, N


def _linear_inputs(c, seed):
    g = _gen(seed)
    W, X = _weights(g, c["N"], c["K"]), _acts(g, c["K"], c["M"])
    gamma = _gamma(g, c["K"]) if c.get("norm") else None
    bias = torch.randn((c["N"],), generator=g, device=DEV) if c.get("bias") else None
    return W, X, gamma, bias


def _ffn_inputs(c, seed):
    g = _gen(seed)
    d, F, M = c["d"], c["F"], c["M"]
    W1, W2, X = _weights(g, 2 * F, d), _weights(g, d, F), _acts(g, d, M)
    return W1, W2, X, _gamma(g, d), _gamma(g, F) if c["subln"] else None


def _float_inputs(c, seed):
    g = _gen(seed)
    dt = torch.float16 if c["f16"] else torch.float32
    W, X = _weights(g, c["N"], c["K"]), _acts(g, c["K"], c["M"]).to(dt)
    dY = (torch.randn((c["N"], c["M"]), generator=g, device=DEV) * 1e-3).to(dt) if c["kind"] == "train_linear" else None
    return W, X, dY


def _attn_inputs(c, seed):
    """q (M, H, dk), k, v (M, Hkv, dk) of the new tokens, the caches with their history, positions."""
    g = _gen(seed)
    B, H, Hkv, dk = c["B"], c["H"], c["Hkv"], c["dk"]
    cdt = torch.float16 if c["f16"] else torch.float32
    if c["kind"] == "decode_attn":
        M, max_len = B, c["hi"] + 1
        pos = torch.randint(c["lo"], c["hi"] + 1, (B,), generator=g, device=DEV, dtype=torch.int32)
        pos[0] = c["hi"]
    else:
        M, max_len = B * c["T"], c["pos0"] + c["T"] + 5
        pos = None
    q = _keys(g, M * H, dk).view(M, H, dk)
    k = _keys(g, M * Hkv, dk).view(M, Hkv, dk)
    v = torch.randn((M, Hkv, dk), generator=g, device=DEV)
    kc = _keys(g, B * max_len * Hkv, dk).view(B, max_len, Hkv * dk).to(cdt)
    vc = torch.randn((B, max_len, Hkv * dk), generator=g, device=DEV).to(cdt)
    return q, k, v, kc, vc, pos, max_len


def _cols(t):
    """(M, heads, dk) -> (heads * dk, M)."""
    return t.flatten(1).t().contiguous()


def _model_weights(g, c):
    """The decoder's tensors, block by block: (name, W) of each projection, then the norms."""
    for _ in range(c["layers"]):
        blk = {name: _weights(g, N, K, RESIDUAL_STD if name in ("o", "fc2") else 0.02) for name, N, K in BLOCK}
        for name, n in (("g1", D), ("g2", D), ("ga", D), ("gf", FF)):
            blk[name] = _gamma(g, n)
        yield blk


def _model_rest(g, c):
    head, emb, gf = _weights(g, VOCAB, D), torch.randn((VOCAB, D), generator=g, device=DEV), _gamma(g, D)
    T = c["T"] if c["kind"] == "prompt" else 1
    ids = torch.randint(0, VOCAB, (c["B"] * T,), generator=g, device=DEV, dtype=torch.int32)
    return head, emb, gf, ids


def _model_caches(g, c):
    """Every layer's caches, ctx positions filled (decode_step)."""
    cdt = torch.float16 if c["f16"] else torch.float32
    shape = (c["B"], c["ctx"] + 8, KV)
    return [tuple(torch.randn(shape, generator=g, device=DEV).to(cdt) for _ in range(2)) for _ in range(c["layers"])]


def _decoder(nn, ctx, c, seed):
    from nnhip_py import decoder as dm
    g = _gen(seed)
    blocks = []
    for w in _model_weights(g, c):
        lin = {}
        for name, N, K in BLOCK:
            if name == "fc1":
                t = ctx.row_absmean(w["fc1"])
                wo, to, _ = ctx.glu_interleave(ctx.trit_pack(w["fc1"], t), t, None, FF, D)
                lin["fc1"] = dm.Linear(ctx.repack(wo, D), to, None, nn.glu_rows(FF), D)
            else:
                rp, tau = _packed(ctx, w[name])
                lin[name] = dm.Linear(rp, tau, None, N, K)
        blocks.append(dm.Block(g1=w["g1"], q=lin["q"], k=lin["k"], v=lin["v"], o=lin["o"], g2=w["g2"],
                               fc1=lin["fc1"], fc2=lin["fc2"], g_attn_sub=w["ga"], g_ffn_sub=w["gf"]))
    head, emb, gf, ids = _model_rest(g, c)
    rp, tau = _packed(ctx, head)
    decode = c["kind"] == "decode_step"
    cfg = dm.Config(d=D, H=HEADS, Hkv=KVH, F=FF, vocab=VOCAB, max_len=c["ctx"] + 8 if decode else c["T"] + 8, act=0,
                    eps=EPS, cache_f16=c["f16"])
    dec = dm.Decoder(ctx, cfg, blocks, emb, gf, dm.Linear(rp, tau, None, VOCAB, D), c["B"],
                     caches=_model_caches(g, c) if decode else None)
    return dec, ids


def prepare(case, seed):
    nn = _pkg()
    ctx = nn.Context(0)
    c, kind = case, case["kind"]
    st = dict(case=c, ctx=ctx, nn=nn)
    if kind == "linear":
        W, X, gamma, bias = _linear_inputs(c, seed)
        rp, tau = _packed(ctx, W)
        st.update(rp=rp, tau=tau, X=X, gamma=gamma, bias=bias, acts=ctx._act_out(c["K"], c["M"]))
    elif kind == "stack":
        g = _gen(seed)
        acts = {K: ctx.act_quant_i8(_acts(g, K, c["M"])) for K in (D, FF)}
        probs, y, at = [], torch.empty((c["layers"] * sum(N for _, N in STACK), c["M"]), device=DEV), 0
        for W, K, N in _stack_weights(g, c):
            rp, tau = _packed(ctx, W)
            xi, s, rs = acts[K]
            probs.append(dict(rp=rp, tau=tau, xi=xi, s=s, rowsum=rs, bias=None, N=N, K=K, M=c["M"], y=y[at:at + N]))
            at += N
        st.update(probs=probs, y=y, group=ctx.group_create(probs))
    elif kind == "ffn":
        W1, W2, X, gamma, gsub = _ffn_inputs(c, seed)
        t1 = ctx.row_absmean(W1)
        wo, to, _ = ctx.glu_interleave(ctx.trit_pack(W1, t1), t1, None, c["F"], c["d"])
        rp2, t2 = _packed(ctx, W2)
        st.update(rp1=ctx.repack(wo, c["d"]), t1=to, rp2=rp2, t2=t2, X=X, gamma=gamma, gsub=gsub)
    elif kind == "float_linear":
        W, X, _ = _float_inputs(c, seed)
        rp, tau = _packed(ctx, W)
        st.update(rp=rp, tau=tau, X=X)
    elif kind == "train_linear":
        W, X, dY = _float_inputs(c, seed)
        st.update(W=W, X=X, dY=dY)
    elif kind in ("decode_attn", "prefill_attn"):
        q, k, v, kc, vc, pos, max_len = _attn_inputs(c, seed)
        cos, sin = _rope(c["dk"], max_len)
        if kind == "prefill_attn":
            q, k, v = _cols(q), _cols(k), _cols(v)
        else:
            q, k, v = (t.flatten(1).contiguous() for t in (q, k, v))
        st.update(q=q, k=k, v=v, kc=kc, vc=vc, pos=pos, max_len=max_len, cos=cos, sin=sin,
                  scale=float(np.float32(1.0) / np.float32(math.sqrt(c["dk"]))))
    elif kind == "decode_step":
        dec, ids = _decoder(nn, ctx, c, seed)
        pos = torch.full((c["B"],), c["ctx"], device=DEV, dtype=torch.int32)
        dec.step(ids, pos, c["ctx"] + 8)   # the scratch is allocated here, outside the capture
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            outs = dec.step(ids, pos, c["ctx"] + 8)
        st.update(dec=dec, ids=ids, pos=pos, graph=graph, outs=outs)
    else:
        dec, ids = _decoder(nn, ctx, c, seed)
        st.update(dec=dec, ids=ids)
    torch.cuda.synchronize()
    return st


def run(state):
    st, ctx, c = state, state["ctx"], state["case"]
    kind = c["kind"]
    if kind == "linear":
        if st["gamma"] is None:
            xi, s, rs = ctx.act_quant_i8(st["X"], outs=st["acts"])
        else:
            xi, s, rs = ctx.rmsnorm_quant_i8(st["X"], st["gamma"], EPS, outs=st["acts"])
        return ctx.ternary_matmul(st["rp"], st["tau"], xi, s, rs, c["N"], c["K"], c["M"], bias=st["bias"])
    if kind == "stack":
        ctx.group_run(st["group"])
        return st["y"]
    if kind == "ffn":
        return ctx.ffn_glu_i8_add(st["X"], st["gamma"], EPS, c["F"], st["rp1"], st["t1"], None, st["rp2"], st["t2"], None,
                                  st["X"], c["act"], gamma_sub=st["gsub"], eps_sub=EPS)
    if kind == "float_linear":
        return ctx.ternary_matmul_f(st["rp"], st["tau"], st["X"], c["N"], c["K"], out_f16=c["f16"])
    if kind == "train_linear":
        tau = ctx.row_absmean(st["W"])
        wq = ctx.trit_pack(st["W"], tau)
        Y = ctx.ternary_matmul_f(ctx.repack(wq, c["K"]), tau, st["X"], c["N"], c["K"], out_f16=c["f16"])
        rpT = ctx.repack(ctx.trit_transpose(wq, c["K"]), c["N"])
        dX = ctx.ternary_matmul_t_f(rpT, tau, st["dY"], c["K"], out_f16=c["f16"])
        return {"tau": tau, "Y": Y, "dX": dX}
    if kind == "decode_attn":
        out = ctx.attention_decode(st["q"], st["k"], st["v"], c["H"], c["Hkv"], c["dk"], st["pos"], st["max_len"], st["kc"],
                                   st["vc"], st["scale"], st["cos"], st["sin"], tokens=True)
        return {"out": out, "k_cache": st["kc"], "v_cache": st["vc"]}
    if kind == "prefill_attn":
        B, T, H, Hkv, dk, pos0 = (c[x] for x in ("B", "T", "H", "Hkv", "dk", "pos0"))
        ctx.kv_cache_fill(st["k"], st["v"], B, T, Hkv, dk, pos0, st["kc"], st["vc"], st["cos"], st["sin"])
        out = ctx.attention_prefill(st["q"], st["kc"], st["vc"], B, T, H, Hkv, dk, pos0, st["scale"], st["cos"], st["sin"])
        return {"out": out, "k_cache": st["kc"], "v_cache": st["vc"]}
    if kind == "decode_step":
        st["graph"].replay()
        logits = st["outs"][0]
    else:
        logits = st["dec"].prefill(st["ids"], c["T"])[0]
    # the greedy ids are these logits' argmax, which a last-place change of two near ones can move
    return {"logits": logits, "caches": [t for kv in st["dec"].caches for t in kv]}


# ------------------------------------------------------------------------------------------- work

def work(case):
    """Each input read once, each output written once; ternary weights at 2 bits, int8 products as
    two operations per multiply-add."""
    c, kind = case, case["kind"]
    if kind in ("linear", "float_linear"):
        N, K, M = c["N"], c["K"], c["M"]
        e = 2 if c.get("f16") else 4
        return dict(bytes=e * K * M + N * K // 4 + 4 * N + e * N * M, flops=2 * N * K * M)
    if kind == "stack":
        M = c["M"]
        b = sum(N * K // 4 + 4 * N + 4 * N * M for K, N in STACK) * c["layers"] + (D + FF) * M
        return dict(bytes=b, flops=2 * M * sum(N * K for K, N in STACK) * c["layers"])
    if kind == "ffn":
        d, F, M = c["d"], c["F"], c["M"]
        return dict(bytes=8 * d * M + 3 * F * d // 4 + 4 * (2 * F + d), flops=6 * M * F * d)
    if kind == "train_linear":
        N, K, M = c["N"], c["K"], c["M"]
        e = 2 if c["f16"] else 4
        return dict(bytes=4 * N * K + 2 * e * K * M + 2 * e * N * M + 4 * N, flops=4 * N * K * M)
    if kind in ("decode_attn", "prefill_attn"):
        B, H, Hkv, dk = (c[x] for x in ("B", "H", "Hkv", "dk"))
        e = 2 if c["f16"] else 4
        if kind == "decode_attn":
            rows = B * ((c["lo"] + c["hi"]) // 2 + 1)
            return dict(bytes=2 * e * rows * Hkv * dk + 8 * B * H * dk + 8 * B * Hkv * dk, flops=4 * rows * H * dk)
        T, pos0 = c["T"], c["pos0"]
        pairs = B * (T * pos0 + T * (T + 1) // 2)
        return dict(bytes=2 * e * B * (pos0 + T) * Hkv * dk + 8 * B * T * H * dk + 8 * B * T * Hkv * dk,
                    flops=4 * pairs * H * dk)
    weights = c["layers"] * sum(N * K for _, N, K in BLOCK)
    if kind == "decode_step":
        e = 2 if c["f16"] else 4
        cached = 2 * e * c["layers"] * c["B"] * (c["ctx"] + 1) * KV
        return dict(bytes=weights // 4 + VOCAB * D // 4 + cached + 4 * VOCAB * c["B"],
                    flops=2 * c["B"] * (weights + VOCAB * D) + 4 * c["layers"] * c["B"] * (c["ctx"] + 1) * HEADS * DK)
    M = c["B"] * c["T"]
    pairs = c["B"] * c["T"] * (c["T"] + 1) // 2
    return dict(bytes=weights // 4 + VOCAB * D // 4 + 4 * M * D + (4 if c["f16"] else 8) * c["layers"] * M * KV,
                flops=2 * M * weights + 4 * c["layers"] * pairs * HEADS * DK + 2 * c["B"] * VOCAB * D)


def tolerance(case):
    """About four times what was measured against exact(). A quantized path also differs where a code
    sits on a rounding tie: one int8 step in a small share of the codes (5.7e-5 of the result's norm
    after one quantization, 4.5e-4 after the feed-forward block's two, 9e-3 after a model's nine)."""
    kind = case["kind"]
    if kind == "linear":
        return {"rel": 3e-4, "max": 0.1}
    if kind == "ffn":
        return {"rel": 2e-3, "max": 0.3}
    if kind in ("float_linear", "train_linear"):
        return {"rel": 1e-3 if case["f16"] else 1e-5}
    if kind in ("stack", "decode_attn"):
        return {"rel": 1e-5}
    if kind == "prefill_attn":
        # f16 caches: a cached value on a rounding tie is one f16 step apart (4.4e-6)
        return {"rel": 2e-5 if case["f16"] else 1e-5}
    return {"rel": 3e-2}


# --------------------------------------------------------------------------- the same in 64 bits

def _t64(W):
    """tau (N, 1) and tau * trit of W in 64 bits."""
    w = W.double()
    tau = w.abs().mean(1, keepdim=True)
    trit = (w > 0.5 * tau).double() - (w < -0.5 * tau).double()
    return tau, trit


def _q64(x):
    """Per-column absmax int8 codes and scales of x (K, M)."""
    s = x.abs().amax(0, keepdim=True) * float(np.float32(1.0) / np.float32(127.0))
    y = torch.where(s > 0, x / torch.where(s > 0, s, torch.ones_like(s)), torch.zeros_like(x)).clamp(-127, 127)
    return torch.sign(y) * torch.floor(y.abs() + 0.5), s


def _norm64(x, gamma):
    return x / torch.sqrt((x * x).mean(0, keepdim=True) + EPS) * gamma.double()[:, None]


def _lin64(W, x):
    """BitLinear W1.58A8 of x (K, M)."""
    tau, trit = _t64(W)
    q, s = _q64(x)
    return tau * s * (trit @ q)


def _glu64(y, F, act):
    gate, up = y[:F], y[F:]
    return (gate * torch.sigmoid(gate) if act == 0 else torch.relu(gate) ** 2) * up


def _rot64(x, cos, sin):
    """x (M, heads, dk) rotated at its token's row of cos / sin (M, dk / 2)."""
    h = x.shape[-1] // 2
    x0, x1, c, s = x[..., :h], x[..., h:], cos[:, None, :].double(), sin[:, None, :].double()
    return torch.cat([x0 * c - x1 * s, x1 * c + x0 * s], -1)


def _attend64(q, kc, vc, limit, scale):
    """q (T, H, dk) over kc / vc (L, Hkv, dk): query t sees rows [0, limit[t]]. -> (T, H, dk)"""
    T, H, dk = q.shape
    R = H // kc.shape[1]
    mask = torch.arange(kc.shape[0], device=DEV)[None, :] > limit[:, None]
    out = torch.empty_like(q)
    for h in range(H):
        s = (q[:, h] @ kc[:, h // R].t()) * scale
        out[:, h] = torch.softmax(s.masked_fill(mask, float("-inf")), -1) @ vc[:, h // R]
    return out


def _as_cache(t, f16):
    """What a cache of this element type holds of t: f32 or f16 is the storage format."""
    return t.to(torch.float16 if f16 else torch.float32).double()


def _table32(dk, n):
    """The decoder's RoPE table, whose angles are 32-bit by definition."""
    th = np.arange(n, dtype=np.float32)[:, None] / np.power(
        np.float32(10000.0), (2 * np.arange(dk // 2)).astype(np.float32) / np.float32(dk))[None, :]
    return [torch.from_numpy(f(th.astype(np.float32))).to(DEV) for f in (np.cos, np.sin)]


def _model64(c, seed):
    g = _gen(seed)
    decode = c["kind"] == "decode_step"
    # the generator makes the blocks, then the head, embedding and ids, then the caches: walk it once
    # for the tensors that come after the blocks
    for _ in _model_weights(g, c):
        pass
    head, emb, gfin, ids = _model_rest(g, c)
    caches = _model_caches(g, c) if decode else None
    B = c["B"]
    T = 1 if decode else c["T"]
    p0 = c["ctx"] if decode else 0
    cos, sin = (t[p0:p0 + T].repeat(B, 1) for t in _table32(DK, p0 + T))
    scale = 1.0 / math.sqrt(DK)
    limit = p0 + torch.arange(T, device=DEV)
    x = emb[ids.long()].double().t()
    kept = []
    for i, w in enumerate(_model_weights(_gen(seed), c)):
        a = _norm64(x, w["g1"])
        q, k, v = (_lin64(w[n], a).t().reshape(B * T, -1, DK) for n in ("q", "k", "v"))
        q, k = _rot64(q, cos, sin), _rot64(k, cos, sin)
        att = torch.empty((B * T, HEADS, DK), dtype=torch.float64, device=DEV)
        both = [caches[i][j].double() if decode else torch.zeros((B, T + 8, KV), dtype=torch.float64, device=DEV)
                for j in range(2)]
        for t, new in zip(both, (k, v)):
            t[:, p0:p0 + T] = _as_cache(new, c["f16"]).reshape(B, T, KV)
        for b in range(B):
            kb, vb = (t[b, :p0 + T].view(p0 + T, KVH, DK) for t in both)
            att[b * T:(b + 1) * T] = _attend64(q[b * T:(b + 1) * T], kb, vb, limit, scale)
        kept += both
        x = x + _lin64(w["o"], _norm64(att.flatten(1).t(), w["ga"]))
        h = _glu64(_lin64(w["fc1"], _norm64(x, w["g2"])), FF, 0)
        x = x + _lin64(w["fc2"], _norm64(h, w["gf"]))
    x = x[:, T - 1::T]
    logits = _lin64(head, _norm64(x, gfin))
    return {"logits": logits, "caches": kept}


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "linear":
        W, X, gamma, bias = _linear_inputs(c, seed)
        x = X.double()
        y = _lin64(W, x if gamma is None else _norm64(x, gamma))
        return y if bias is None else y + bias.double()[:, None]
    if kind == "stack":
        g = _gen(seed)
        acts = {K: _q64(_acts(g, K, c["M"]).double()) for K in (D, FF)}
        out = []
        for W, K, N in _stack_weights(g, c):
            tau, trit = _t64(W)
            out.append(tau * acts[K][1] * (trit @ acts[K][0]))
        return torch.cat(out)
    if kind == "ffn":
        W1, W2, X, gamma, gsub = _ffn_inputs(c, seed)
        x = X.double()
        h = _glu64(_lin64(W1, _norm64(x, gamma)), c["F"], c["act"])
        return x + _lin64(W2, h if gsub is None else _norm64(h, gsub))
    if kind == "float_linear":
        W, X, _ = _float_inputs(c, seed)
        tau, trit = _t64(W)
        return tau * (trit @ X.double())
    if kind == "train_linear":
        W, X, dY = _float_inputs(c, seed)
        tau, trit = _t64(W)
        return {"tau": tau[:, 0], "Y": tau * (trit @ X.double()), "dX": trit.t() @ (tau * dY.double())}
    if kind in ("decode_attn", "prefill_attn"):
        q, k, v, kc, vc, pos, max_len = _attn_inputs(c, seed)
        cos, sin = _rope(c["dk"], max_len)
        B, Hkv, dk = c["B"], c["Hkv"], c["dk"]
        T = c.get("T", 1)
        where = pos[:, None].long() if pos is not None else c["pos0"] + torch.arange(T, device=DEV).repeat(B, 1)
        flat = where.reshape(-1)
        q, k, v = _rot64(q.double(), cos[flat], sin[flat]), _rot64(k.double(), cos[flat], sin[flat]), v.double()
        kc, vc = (t.double().view(B, max_len, Hkv, dk) for t in (kc, vc))
        out = torch.empty((B * T, c["H"], dk), dtype=torch.float64, device=DEV)
        for b in range(B):
            rows = slice(b * T, (b + 1) * T)
            kc[b, where[b]], vc[b, where[b]] = _as_cache(k[rows], c["f16"]), _as_cache(v[rows], c["f16"])
            n = int(where[b].max()) + 1
            out[rows] = _attend64(q[rows], kc[b, :n], vc[b, :n], where[b], 1.0 / math.sqrt(dk))
        out = out.flatten(1)
        return {"out": out if pos is not None else out.t(), "k_cache": kc.flatten(2), "v_cache": vc.flatten(2)}
    return _model64(c, seed)
