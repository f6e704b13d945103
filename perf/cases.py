"""Performance cases: the work that programs on top of libne have it do.

Two kinds of program use the library.  One composes its own training step from the kernel-level
entry points (ne_k_*): the cases `mlp_*`, `attn_*`, `layer`, `head` and `adam` are the blocks of
such a step, each a short sequence of calls on device buffers that the program keeps (weights,
saved activations, gradients).  The other drives a whole model through the context API: `train`
is its training loop, `decode` its token loop.  Shapes are those of the model headers (tiny,
Stories110M, Qwen3-0.6B) and of the benchmark (256 tokens; 8 sequences of 2048 tokens; the token
loop at batch 1 and 32), or other multiples of 64, the unit of the entry points' sizes.

`exact` is the same mathematics in float64 on plain torch, from the same 16-bit inputs.
"""
import ctypes as C
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "neural-engine_amd"))
import ne  # noqa: E402

DEV = "cuda"
TDT = {"fp16": torch.float16, "bf16": torch.bfloat16}
NDT = {"fp16": ne.NE_FP16, "bf16": ne.NE_BF16}
EPS = 1e-5
DLOGITS_SCALE = 256.0  # the 16-bit backward's gradient scale

# Model families of the repository: width, FFN width, heads, KV heads, head size, QK-norm, RoPE base
FAMILY = {
    "tiny": dict(D=128, H=256, NH=4, NKV=2, HD=64, qk_norm=False, theta=1e4),
    "stories110m": dict(D=768, H=2048, NH=12, NKV=12, HD=64, qk_norm=False, theta=1e4),
    "qwen3": dict(D=1024, H=3072, NH=16, NKV=8, HD=128, qk_norm=True, theta=1e6),
    "wide": dict(D=2048, H=2816, NH=16, NKV=4, HD=128, qk_norm=True, theta=1e6),
    "odd": dict(D=832, H=1728, NH=10, NKV=5, HD=64, qk_norm=True, theta=1e4),
}


def listed():
    s, q = FAMILY["stories110m"], FAMILY["qwen3"]
    return [
        # the smallest block: one FFN forward of a Stories110M step of 256 tokens (three launches)
        dict(name="mlp-fwd-256", op="mlp_fwd", dtype="fp16", B=1, S=256, **s),
        # a Qwen3 FFN's backward at an ordinary micro-batch (2048 tokens), with its weight gradients
        dict(name="mlp-bwd-2048", op="mlp_bwd", dtype="bf16", B=1, S=2048, **q),
        # attention block forward of the Stories110M step: multi-head, 64-wide heads, short
        dict(name="attn-fwd-256", op="attn_fwd", dtype="fp16", B=1, S=256, **s),
        # attention block forward of the large batch: 8 sequences of 2048, grouped-query, QK-norm
        dict(name="attn-fwd-8x2048", op="attn_fwd", dtype="bf16", B=8, S=2048, **q),
        # attention block backward at a ragged length (17 tiles of 64 positions), 3 sequences
        dict(name="attn-bwd-3x1088", op="attn_bwd", dtype="fp16", B=3, S=1088, **q),
        # attention block backward of the 256-token Qwen3 step (latency-bound)
        dict(name="attn-bwd-256", op="attn_bwd", dtype="fp16", B=1, S=256, **q),
        # one whole Qwen3 layer, forward and backward, of the 16,384-token step
        dict(name="layer-8x2048", op="layer", dtype="fp16", B=8, S=2048, **q),
        # LM head, loss and their gradients: Qwen3's 151,936-token vocabulary (not a multiple of 256)
        dict(name="head-4096", op="head", dtype="bf16", T=4096, D=1024, V=151936),
        # gradient norm, clip and AdamW over Stories110M's parameters
        dict(name="adam-110m", op="adam", dtype="fp16", n=109529856, n_gain=19200),
        # the training loop: consecutive Qwen3-0.6B steps of 256 tokens (step + optimizer step)
        dict(name="train-256", op="train", dtype="fp16", B=1, S=256, L=28, V=151936, steps=8, **q),
        # generation as the command line does it by default: one sequence, fp16, temperature, top-p
        dict(name="decode-b1", op="decode", dtype="fp16", B=1, P=32, n_new=64, temp=0.8, top_p=0.9, L=28, V=151936, **q),
        # batched greedy generation, 32 sequences, bf16 weights
        dict(name="decode-b32", op="decode", dtype="bf16", B=32, P=32, n_new=64, temp=0.0, top_p=1.0, L=28, V=151936, **q),
    ]


def _log(rng, lo, hi, unit):
    return max(lo, min(hi, int(math.exp(rng.uniform(math.log(lo), math.log(hi + unit - 1))) // unit * unit)))


def draw(rng):
    op = rng.choice(["mlp_fwd", "mlp_bwd", "attn_fwd", "attn_bwd", "layer", "head", "adam", "train", "decode",
                     "mlp_bwd", "attn_fwd", "attn_bwd", "head"])
    dtype = rng.choice(["fp16", "bf16"])
    if op == "head":
        T = _log(rng, 64, 4096, 64)
        V = _log(rng, 512, min(151936, max(4096, 4096 * 151936 // T)), 64)
        return dict(op=op, dtype=dtype, T=T, D=rng.choice([128, 768, 832, 1024]), V=V)
    if op == "adam":
        n_gain = 4 * rng.randint(16, 20000)
        return dict(op=op, dtype=dtype, n=n_gain + 4 * _log(rng, 4096, 27000000, 1), n_gain=n_gain)
    fam = FAMILY[rng.choice(["stories110m", "qwen3", "wide", "odd", "tiny"])]
    if op == "train":
        fam = FAMILY[rng.choice(["stories110m", "qwen3", "tiny", "odd"])]
        S = 64 * rng.randint(1, 16)
        return dict(op=op, dtype=dtype, B=rng.randint(1, 3), S=S, L=rng.randint(1, 6), V=_log(rng, 512, 32000, 64),
                    steps=rng.randint(2, 6), **fam)
    if op == "decode":
        fam = FAMILY[rng.choice(["stories110m", "qwen3", "tiny"])]
        greedy = rng.random() < 0.5
        return dict(op=op, dtype=dtype, B=rng.choice([1, 1, 2, 3, 4, 5, 8, 13, 16, 24, 32]), P=rng.randint(1, 48),
                    n_new=rng.randint(16, 64), temp=0.0 if greedy else round(rng.uniform(0.5, 1.0), 2),
                    top_p=1.0 if greedy else rng.choice([1.0, 0.9, 0.95]), L=rng.randint(2, 8),
                    V=_log(rng, 512, 65536, 64), **fam)
    S = _log(rng, 64, 2048, 64)
    B = rng.randint(1, max(1, min(8, 16384 // S)))
    return dict(op=op, dtype=dtype, B=B, S=S, **fam)


# ------------------------------------------------------------------------------ inputs ----


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _randn(g, shape, std=1.0, dtype=torch.float32):
    return (torch.randn(shape, generator=g, device=DEV, dtype=torch.float32) * std).to(dtype)


def _alpha(c):
    return 0.25  # residual branch scale of a block (1/sqrt(2 L) at 8 layers)


def _rope(S, HD, theta):
    i = torch.arange(HD // 2, dtype=torch.float64, device=DEV)
    ang = torch.arange(S, dtype=torch.float64, device=DEV)[:, None] * (float(theta) ** (-2.0 * i / HD))[None]
    return torch.cos(ang), torch.sin(ang)


def _block_inputs(c, seed):
    """Residual stream, upstream gradient and the weights of one layer.  Weights N(0, 0.02) as the
    benchmark's, gains around 1, activations and gradients of unit scale."""
    g, t = _gen(seed), TDT[c["dtype"]]
    D, H, Q, KV = c["D"], c["H"], c["NH"] * c["HD"], c["NKV"] * c["HD"]
    T = c["B"] * c["S"]
    i = dict(x=_randn(g, (T, D)), g_att=1 + _randn(g, (D,), 0.1), g_ffn=1 + _randn(g, (D,), 0.1))
    if c["op"] in ("mlp_bwd", "attn_bwd", "layer"):
        i["dy"] = _randn(g, (T, D))
    if c["op"] in ("mlp_fwd", "mlp_bwd", "layer"):
        i.update(w13=_randn(g, (2 * H, D), 0.02, t), w2=_randn(g, (D, H), 0.02, t))
    if c["op"] in ("attn_fwd", "attn_bwd", "layer"):
        i.update(wqkv=_randn(g, (Q + 2 * KV, D), 0.02, t), wo=_randn(g, (D, Q), 0.02, t))
        i["gq"] = 1 + _randn(g, (c["HD"],), 0.1) if c["qk_norm"] else None
        i["gk"] = 1 + _randn(g, (c["HD"],), 0.1) if c["qk_norm"] else None
    return i


def prepare(case, seed):
    c = dict(case)
    return _PREPARE[c["op"]](c, seed)


def _buf(*shape, dtype=torch.float32):
    return torch.empty(shape, dtype=dtype, device=DEV)


def _prepare_block(c, seed):
    t = TDT[c["dtype"]]
    D, H, NH, NKV, HD = c["D"], c["H"], c["NH"], c["NKV"], c["HD"]
    Q, KV, T, a = NH * HD, NKV * HD, c["B"] * c["S"], _alpha(c)
    s = dict(c=c, T=T, Q=Q, KV=KV, QKV=Q + 2 * KV, dt=NDT[c["dtype"]], alpha=a, scale=1.0 / math.sqrt(HD))
    s.update(_block_inputs(c, seed))
    mlp, att = c["op"] in ("mlp_fwd", "mlp_bwd", "layer"), c["op"] in ("attn_fwd", "attn_bwd", "layer")
    if att:
        cs, sn = _rope(c["S"], HD, c["theta"])
        s.update(cos=cs.float().contiguous(), sin=sn.float().contiguous())
        s.update(xn=_buf(T, D, dtype=t), r1=_buf(T), qkv=_buf(T, Q + 2 * KV, dtype=t), qr=_buf(T, Q, dtype=t),
                 kr=_buf(T, KV, dtype=t), rq=_buf(T, NH), rk=_buf(T, NKV), att=_buf(T, Q, dtype=t), lse=_buf(T, NH),
                 x2=_buf(T, D))
    if mlp:
        s.update(x2n=_buf(T, D, dtype=t), r2=_buf(T), h13=_buf(T, 2 * H, dtype=t), gate=_buf(T, H, dtype=t),
                 out=_buf(T, D))
    if "dy" in s:
        s.update(db=(s["dy"] * a).to(t), dtmp=_buf(T, D), dxb=_buf(T, D, dtype=t))
        if mlp:
            s.update(dh13=_buf(T, 2 * H, dtype=t), dw13=_buf(2 * H, D), dw2=_buf(D, H), dg_ffn=_buf(D), dx2=_buf(T, D))
        if att:
            s.update(dattn=_buf(T, Q, dtype=t), delta=_buf(T, NH), dq=_buf(T, Q), dk=_buf(T, KV),
                     dqkv=_buf(T, Q + 2 * KV, dtype=t), dwqkv=_buf(Q + 2 * KV, D), dwo=_buf(D, Q), dg_att=_buf(D),
                     dgq=_buf(HD), dgk=_buf(HD), dx=_buf(T, D))
    # saved activations of the backward blocks: the forward in float32, rounded where the step
    # holds 16 bits
    if c["op"] == "mlp_bwd":
        x2n, s["r2"] = _norm(s["x"], s["g_ffn"])
        s["r2"] = s["r2"].reshape(T).contiguous()
        s["x2n"] = x2n.to(t)
        s["h13"] = (s["x2n"].float() @ s["w13"].float().t()).to(t)
        h = s["h13"].float()
        s["gate"] = (torch.nn.functional.silu(h[:, :H]) * h[:, H:]).to(t)
    if c["op"] == "attn_bwd":
        xn, r1 = _norm(s["x"], s["g_att"])
        s["xn"], s["r1"] = xn.to(t), r1.reshape(T).contiguous()
        s["qkv"] = (s["xn"].float() @ s["wqkv"].float().t()).to(t)
        q, k, v, rq, rk = _qk(c, s["qkv"].float(), s["gq"], s["gk"], s["cos"], s["sin"])
        s["qr"], s["kr"] = q.reshape(T, Q).to(t), k.reshape(T, KV).to(t)
        if rq is not None:
            s["rq"], s["rk"] = rq.reshape(T, NH).contiguous(), rk.reshape(T, NKV).contiguous()
        o, lse = _sdpa(c, s["qr"].float().view(T, NH, HD), s["kr"].float().view(T, NKV, HD), v)
        s["att"], s["lse"] = o.reshape(T, Q).to(t), lse.contiguous()
    return s


def _prepare_head(c, seed):
    g, t = _gen(seed), TDT[c["dtype"]]
    T, D, V = c["T"], c["D"], c["V"]
    return dict(c=c, dt=NDT[c["dtype"]], x=_randn(g, (T, D), 1.0, t), E=_randn(g, (V, D), 0.02, t),
                tgt=torch.randint(0, V, (T,), generator=g, device=DEV, dtype=torch.int32), part=_buf(T * (V // 64) * 2),
                tl=_buf(T), lse=_buf(T), rows=_buf(T), loss=_buf(1), dlogits=_buf(T, V, dtype=t), dx=_buf(T, D),
                dE=_buf(V, D))


def _prepare_adam(c, seed):
    g, n = _gen(seed), c["n"]
    return dict(c=c, dt=NDT[c["dtype"]], p=_randn(g, (n,), 0.02), g=_randn(g, (n,), 1e-3), m=_randn(g, (n,), 1e-4),
                v=_randn(g, (n,), 1e-3).square_(), pb=_buf(n, dtype=TDT[c["dtype"]]),
                partials=_buf(1024, dtype=torch.float64), gscale=_buf(1), gnorm=_buf(1))


def _model_params(c, seed):
    """(name, tensor) of a whole model: N(0, 0.02) matrices, gains 1 (the final gain of a token
    loop 12, for logits as peaked as a trained model's)."""
    g = _gen(seed)
    D, H, Q, KV = c["D"], c["H"], c["NH"] * c["HD"], c["NKV"] * c["HD"]
    shape = {"Wq": (Q, D), "Wk": (KV, D), "Wv": (KV, D), "Wo": (D, Q), "W1": (H, D), "W2": (D, H), "W3": (H, D)}
    for l in range(c["L"]):
        for n, sh in shape.items():
            yield f"layers.{l}.{n}", _randn(g, sh, 0.02)
    yield "embed", _randn(g, (c["V"], D), 0.02)
    if c["op"] == "decode":
        yield "rms_final", torch.full((D,), 12.0, device=DEV)


_STAGE = {}


def _make_model(c, seed, **kw):
    m = ne.Model(c["D"], c["H"], c["NH"], c["NKV"], c["HD"], c["L"], c["V"], qk_norm=c["qk_norm"],
                 rope_theta=c["theta"], dtype=NDT[c["dtype"]], **kw)
    for name, w in _model_params(c, seed):  # through pinned memory, one tensor at a time
        n = w.numel()
        if _STAGE.get("n", 0) < n:
            _STAGE.update(n=n, t=torch.empty(n, dtype=torch.float32, pin_memory=True))
        h = _STAGE["t"][:n]
        h.copy_(w.reshape(-1))
        m.set(name, h.numpy())
    return m


def _tokens(c, seed, *shape):
    return np.random.default_rng(int(seed)).integers(0, c["V"], size=shape).astype(np.int32)


def _train_alpha(c):
    return float(np.float32(1.0) / np.sqrt(np.float32(2.0 * c["L"])))


def _prepare_train(c, seed):
    return dict(c=c, m=_make_model(c, seed, seq=c["S"], batch=c["B"], res_alpha=_train_alpha(c)),
                tokens=list(_tokens(c, seed, c["steps"], c["B"], c["S"] + 1)))


def _prepare_decode(c, seed):
    m = _make_model(c, seed, seq=64, res_alpha=1.0, decode_batch=c["B"], decode_ctx=c["P"] + c["n_new"])
    u = np.random.default_rng(int(seed) + 1).random((c["B"], c["n_new"])) if c["temp"] > 0 else None
    return dict(c=c, m=m, prompt=_tokens(c, seed, c["B"], c["P"]), u=u)


# --------------------------------------------------------------------------------- run ----


def run(state):
    return _RUN[state["c"]["op"]](state)


def _ok(rc):
    if rc != 0:
        raise ne.NEError(f"{rc}: {ne.lib().ne_last_error().decode()}")


def _p(t):
    return t.data_ptr() if t is not None else None


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _gemm(s, layout, epi, M, N, K, A, lda, B, ldb, Cm, ldc, R=None, ldr=0, alpha=1.0):
    _ok(ne.lib().ne_k_gemm(s["dt"], layout, epi, M, N, K, _p(A), lda, _p(B), ldb, _p(Cm), ldc, _p(R), ldr, alpha,
                           _stream()))


def _attn_fwd(s):
    L, c, st = ne.lib(), s["c"], _stream()
    T, D, Q, KV, QKV, NH, NKV, HD, S = s["T"], c["D"], s["Q"], s["KV"], s["QKV"], c["NH"], c["NKV"], c["HD"], c["S"]
    _ok(L.ne_k_rmsnorm_fwd(s["dt"], _p(s["x"]), _p(s["g_att"]), _p(s["xn"]), _p(s["r1"]), T, D, EPS, st))
    _gemm(s, 0, 0, T, QKV, D, s["xn"], D, s["wqkv"], D, s["qkv"], QKV)
    _ok(L.ne_k_qk_prep_fwd(s["dt"], _p(s["qkv"]), QKV, _p(s["cos"]), _p(s["sin"]), _p(s["gq"]), _p(s["gk"]),
                           _p(s["qr"]), _p(s["kr"]), _p(s["rq"]), _p(s["rk"]), T, S, NH, NKV, HD, EPS, st))
    _ok(L.ne_k_attn_fwd(s["dt"], _p(s["qr"]), Q, _p(s["kr"]), KV, _p(s["qkv"][:, Q + KV:]), QKV, _p(s["att"]), Q,
                        _p(s["lse"]), c["B"], S, NH, NKV, HD, s["scale"], st))
    _gemm(s, 0, 3, T, D, Q, s["att"], Q, s["wo"], Q, s["x2"], D, s["x"], D, s["alpha"])


def _mlp_fwd(s, x):
    L, c, st = ne.lib(), s["c"], _stream()
    T, D, H = s["T"], c["D"], c["H"]
    _ok(L.ne_k_rmsnorm_fwd(s["dt"], _p(x), _p(s["g_ffn"]), _p(s["x2n"]), _p(s["r2"]), T, D, EPS, st))
    if T <= 2048:  # the gate in the GEMM's epilogue, as the library's own step does on short steps
        _gemm(s, 0, 7, T, 2 * H, D, s["x2n"], D, s["w13"], D, s["h13"], 2 * H, s["gate"], H)
    else:
        _gemm(s, 0, 0, T, 2 * H, D, s["x2n"], D, s["w13"], D, s["h13"], 2 * H)
        _ok(L.ne_k_swiglu_fwd(s["dt"], _p(s["h13"]), _p(s["gate"]), T, H, st))
    _gemm(s, 0, 3, T, D, H, s["gate"], H, s["w2"], H, s["out"], D, x, D, s["alpha"])


def _wgrads(s, problems):
    """Weight gradients dW[M, N] = dY[T, M]^T X[T, N]: the grouped launch where it is for them."""
    T, n = s["T"], len(problems)
    tiles = sum((M // 256) * (N // 256) for M, N, *_ in problems)
    if n > 1 and T >= 8192 and tiles >= 192 and all(M % 256 == 0 and N % 256 == 0 for M, N, *_ in problems):
        arr = lambda ct, v: (ct * n)(*v)  # noqa: E731
        _ok(ne.lib().ne_k_gemm_wgrad_group(
            s["dt"], n, arr(C.c_int, [p[0] for p in problems]), arr(C.c_int, [p[1] for p in problems]), T,
            arr(C.c_void_p, [p[2].data_ptr() for p in problems]), arr(C.c_int64, [p[0] for p in problems]),
            arr(C.c_void_p, [p[3].data_ptr() for p in problems]), arr(C.c_int64, [p[1] for p in problems]),
            arr(C.c_void_p, [p[4].data_ptr() for p in problems]), 0, 1.0, _stream()))
        return
    for M, N, dY, X, dW in problems:
        _gemm(s, 3, 1, M, N, T, dY, M, X, N, dW, N)


def _mlp_bwd(s, x, dx, db, dxo, dxb, queue=None):
    L, c, st = ne.lib(), s["c"], _stream()
    T, D, H = s["T"], c["D"], c["H"]
    _gemm(s, 2, 4, T, H, D, db, D, s["w2"], H, s["dh13"], 2 * H, s["h13"], 2 * H)
    w = [(D, H, db, s["gate"], s["dw2"]), (2 * H, D, s["dh13"], s["x2n"], s["dw13"])]
    if queue is None:
        _wgrads(s, w)
    else:
        queue += w
    _gemm(s, 2, 1, T, D, 2 * H, s["dh13"], 2 * H, s["w13"], D, s["dtmp"], D)
    s["dg_ffn"].zero_()
    _ok(L.ne_k_rmsnorm_bwd(s["dt"], _p(s["dtmp"]), _p(x), _p(s["g_ffn"]), _p(s["r2"]), _p(dx), _p(dxo), _p(dxb),
                           s["alpha"], _p(s["dg_ffn"]), 1.0, T, D, st))


def _attn_bwd(s, x, dx, db, dxo, queue=None):
    L, c, st = ne.lib(), s["c"], _stream()
    T, D, Q, KV, QKV, NH, NKV, HD, S = s["T"], c["D"], s["Q"], s["KV"], s["QKV"], c["NH"], c["NKV"], c["HD"], c["S"]
    v, dv = s["qkv"][:, Q + KV:], s["dqkv"][:, Q + KV:]
    _gemm(s, 2, 0, T, Q, D, db, D, s["wo"], Q, s["dattn"], Q)
    _ok(L.ne_k_attn_bwd(s["dt"], _p(s["qr"]), Q, _p(s["kr"]), KV, _p(v), QKV, _p(s["att"]), Q, _p(s["lse"]),
                        _p(s["dattn"]), Q, _p(s["delta"]), _p(s["dq"]), Q, _p(s["dk"]), KV, _p(dv), QKV, c["B"], S, NH,
                        NKV, HD, s["scale"], st))
    if c["qk_norm"]:
        s["dgq"].zero_()
        s["dgk"].zero_()
    _ok(L.ne_k_qk_prep_bwd(s["dt"], _p(s["dq"]), _p(s["dk"]), _p(s["qkv"]), QKV, _p(s["cos"]), _p(s["sin"]),
                           _p(s["gq"]), _p(s["gk"]), _p(s["rq"]), _p(s["rk"]), _p(s["dqkv"]), _p(s["dgq"]),
                           _p(s["dgk"]), 1.0, T, S, NH, NKV, HD, st))
    w = [(D, Q, db, s["att"], s["dwo"]), (QKV, D, s["dqkv"], s["xn"], s["dwqkv"])]
    _wgrads(s, w if queue is None else queue + w)
    _gemm(s, 2, 1, T, D, QKV, s["dqkv"], QKV, s["wqkv"], D, s["dtmp"], D)
    s["dg_att"].zero_()
    _ok(L.ne_k_rmsnorm_bwd(s["dt"], _p(s["dtmp"]), _p(x), _p(s["g_att"]), _p(s["r1"]), _p(dx), _p(dxo), None, 1.0,
                           _p(s["dg_att"]), 1.0, T, D, st))


def _run_mlp_fwd(s):
    _mlp_fwd(s, s["x"])
    return {k: s[k] for k in ("out", "h13", "gate", "r2")}


def _run_attn_fwd(s):
    _attn_fwd(s)
    return {k: s[k] for k in ("x2", "qkv", "att", "lse")}


def _mlp_grads(s):
    return {k: s[k] for k in ("dw13", "dw2", "dg_ffn")}


def _attn_grads(s):
    out = {k: s[k] for k in ("dwqkv", "dwo", "dg_att")}
    if s["c"]["qk_norm"]:
        out.update(dgq=s["dgq"], dgk=s["dgk"])
    return out


def _run_mlp_bwd(s):
    _mlp_bwd(s, s["x"], s["dy"], s["db"], s["dx2"], s["dxb"])
    return dict(dx=s["dx2"], dxb=s["dxb"], **_mlp_grads(s))


def _run_attn_bwd(s):
    _attn_bwd(s, s["x"], s["dy"], s["db"], s["dx"])
    return dict(dx=s["dx"], **_attn_grads(s))


def _run_layer(s):
    q = []
    _attn_fwd(s)
    _mlp_fwd(s, s["x2"])
    _mlp_bwd(s, s["x2"], s["dy"], s["db"], s["dx2"], s["dxb"], q)
    _attn_bwd(s, s["x"], s["dx2"], s["dxb"], s["dx"], q)
    return dict(out=s["out"], dx=s["dx"], **_mlp_grads(s), **_attn_grads(s))


def _run_head(s):
    c = s["c"]
    T, D, V = c["T"], c["D"], c["V"]
    _ok(ne.lib().ne_k_ce_fwd_grad(s["dt"], _p(s["x"]), _p(s["E"]), _p(s["tgt"]), T, D, V, _p(s["part"]), _p(s["tl"]),
                                  _p(s["lse"]), _p(s["rows"]), _p(s["loss"]), DLOGITS_SCALE, _p(s["dlogits"]),
                                  _stream()))
    _gemm(s, 2, 1, T, D, V, s["dlogits"], V, s["E"], D, s["dx"], D)
    _gemm(s, 3, 1, V, D, T, s["dlogits"], V, s["x"], D, s["dE"], D, alpha=1.0 / (DLOGITS_SCALE * T))
    return {k: s[k] for k in ("loss", "lse", "dlogits", "dx", "dE")}


ADAM = dict(lr=3e-4, b1=0.9, b2=0.95, eps=1e-8, wd=0.1)


def _run_adam(s):
    L, c, st, k = ne.lib(), s["c"], _stream(), ADAM
    n = c["n"]
    _ok(L.ne_k_grad_norm(_p(s["g"]), n, 1.0, 1.0, _p(s["partials"]), _p(s["gscale"]), _p(s["gnorm"]), st))
    _ok(L.ne_k_adam(s["dt"], _p(s["p"]), _p(s["g"]), _p(s["m"]), _p(s["v"]), _p(s["pb"]), n, n - c["n_gain"], k["lr"],
                    k["b1"], k["b2"], k["eps"], k["wd"], 10, _p(s["gscale"]), 0, st))
    return {k: s[k] for k in ("p", "m", "v", "pb", "gnorm")}


TRAIN_READ = ("layers.0.Wk", "layers.0.Wo", "layers.0.rms_att", "rms_final")


def _run_train(s):
    m, k = s["m"], ADAM
    losses = []
    for tok in s["tokens"]:
        losses.append(m.train_step(tok))  # the loss is read each step, as the command line prints it
        m.optimizer_step(k["lr"], k["b1"], k["b2"], k["eps"], k["wd"])
    out = {n: m.get(n) for n in TRAIN_READ}  # updated weights: a few whole tensors of the model
    out["loss"] = np.array(losses, np.float64)
    return out


def _run_decode(s):
    c = s["c"]
    # the token loop's entry points give tokens only
    return s["m"].decode(s["prompt"], c["n_new"], c["temp"], c["top_p"], s["u"])


# -------------------------------------------------------------------------------- work ----


def work(case):
    c = dict(case)
    op = c["op"]
    if op == "head":
        T, D, V = c["T"], c["D"], c["V"]
        return dict(flops=6.0 * T * V * D, bytes=2.0 * T * D + 2.0 * V * D + 4 * T + 2.0 * T * V + 4.0 * T * D + 4.0 * V * D)
    if op == "adam":
        return dict(flops=15.0 * c["n"], bytes=30.0 * c["n"])
    D, H, Q, KV = c["D"], c["H"], c["NH"] * c["HD"], c["NKV"] * c["HD"]
    QKV = Q + 2 * KV
    wa, wm = D * QKV + D * Q, 3 * D * H
    if op == "decode":
        pos = c["P"] + c["n_new"] - 1
        wts = 2.0 * c["L"] * (wa + wm)
        head = 2.0 * c["V"] * D
        kv = 4.0 * 2 * c["L"] * KV * c["B"]  # one position's K and V rows
        return dict(flops=c["B"] * (pos * wts + c["n_new"] * head + pos * (pos + 1) / 2 * 4.0 * c["L"] * Q),
                    bytes=pos * wts + c["n_new"] * head + kv * (pos * (pos + 1) / 2 + pos))
    T = c["B"] * c["S"]
    sd = 2.0 * c["S"] * T * Q  # causal QK^T and PV
    if op == "train":
        n = c["L"] * (wa + wm) + c["V"] * D
        return dict(flops=c["steps"] * (3.0 * (2.0 * T * n + c["L"] * sd) + 15.0 * n),
                    bytes=c["steps"] * (30.0 + 2.0 + 2.0 + 4.0) * n)
    fa, fm = 2.0 * T * wa + sd, 2.0 * T * wm
    # each input read once and each output written once
    in_x, w_a, w_m = 4.0 * T * D, 2.0 * wa, 2.0 * wm
    if op == "mlp_fwd":
        return dict(flops=fm, bytes=in_x + w_m + 4.0 * T * D + 6.0 * T * H + 4 * T)
    if op == "attn_fwd":
        return dict(flops=fa, bytes=in_x + w_a + 4.0 * T * D + 2.0 * T * QKV + 2.0 * T * Q + 4.0 * T * c["NH"])
    if op == "mlp_bwd":
        return dict(flops=2 * fm, bytes=in_x + 6.0 * T * D + 2.0 * T * D + 6.0 * T * H + w_m + 6.0 * T * D + 2 * w_m)
    if op == "attn_bwd":
        return dict(flops=4.0 * T * wa + 2.5 * sd,
                    bytes=in_x + 6.0 * T * D + 2.0 * T * D + 2.0 * T * QKV + 2.0 * T * (2 * Q + KV) + w_a + 4.0 * T * D + 2 * w_a)
    return dict(flops=3 * (2.0 * T * (wa + wm)) + 3.5 * sd,
                bytes=2 * in_x + w_a + w_m + 2 * 4.0 * T * D + 2 * (w_a + w_m))  # layer: forward + backward


def tolerance(case):
    """About four times the distance from `exact` that the 16-bit roundings inside each block give
    (measured: forward blocks 4.8e-4 fp16, 4.6e-3 bf16; backward blocks 1.0e-3, 4.2e-3; training
    7e-4 on updated weights in fp16)."""
    op, b = case["op"], case["dtype"] == "bf16"
    if op == "adam":  # fp32 to a few ulp; the 16-bit copy of a value an ulp away may round the other way
        return {"rel": 1e-4 if b else 2e-5, "max": 0.01}
    if op == "decode":
        return {"differ": 0.01}
    if op == "train":  # AdamW's first steps turn a sign change of a small gradient into a whole update
        return {"rel": 1.2e-2 if b else 3e-3, "max": 0.6}
    if op == "head":  # the rounding of (p - 1) * scale at the targets, on small vocabularies
        return {"rel": 6e-3 if b else 8e-4, "max": 0.1}
    if op in ("mlp_fwd", "attn_fwd"):
        return {"rel": 1.5e-2 if b else 2e-3, "max": 0.2}
    return {"rel": 1.6e-2 if b else 4e-3, "max": 0.5}


# ------------------------------------------------------------------------------- exact ----


def _norm(x, g):
    r = torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS)
    return x * r * g, r


def _rot(x, cos, sin):
    """Interleaved RoPE of x [B, S, heads, HD] with tables [S, HD/2]."""
    c, s = cos[None, :, None, :], sin[None, :, None, :]
    x0, x1 = x[..., 0::2], x[..., 1::2]
    return torch.stack((x0 * c - x1 * s, x0 * s + x1 * c), -1).flatten(-2)


def _qk(c, qkv, gq, gk, cos, sin):
    B, S, NH, NKV, HD = c["B"], c["S"], c["NH"], c["NKV"], c["HD"]
    q, k, v = qkv.split((NH * HD, NKV * HD, NKV * HD), -1)
    q, k, v = q.reshape(B, S, NH, HD), k.reshape(B, S, NKV, HD), v.reshape(B * S, NKV, HD)
    rq = rk = None
    if gq is not None:
        q, rq = _norm(q, gq)
        k, rk = _norm(k, gk)
    return _rot(q, cos, sin).reshape(B * S, NH, HD), _rot(k, cos, sin).reshape(B * S, NKV, HD), v, rq, rk


def _sdpa(c, q, k, v):
    """Causal GQA attention, one (sequence, head) at a time; also the rows' log-sum-exp."""
    B, S, NH, NKV, HD = c["B"], c["S"], c["NH"], c["NKV"], c["HD"]
    mask = torch.ones(S, S, dtype=torch.bool, device=q.device).triu(1)
    o, lse = [], []
    for b in range(B):
        ob, lb = [], []
        for h in range(NH):
            r = slice(b * S, (b + 1) * S)
            kv = h // (NH // NKV)
            s = (q[r, h] @ k[r, kv].t()) * (1.0 / math.sqrt(HD))
            s = s.masked_fill(mask, float("-inf"))
            l = torch.logsumexp(s, -1)
            ob.append(torch.exp(s - l[:, None]) @ v[r, kv])
            lb.append(l)
        o.append(torch.stack(ob, 1))
        lse.append(torch.stack(lb, 1))
    return torch.cat(o), torch.cat(lse)


def _ref_attn(c, x, w, cos, sin, alpha):
    T = c["B"] * c["S"]
    xn, _ = _norm(x, w["g_att"])
    qkv = xn @ w["wqkv"].t()
    q, k, v, _, _ = _qk(c, qkv, w["gq"], w["gk"], cos, sin)
    o, lse = _sdpa(c, q, k, v)
    att = o.reshape(T, -1)
    return x + alpha * (att @ w["wo"].t()), qkv, att, lse


def _ref_mlp(c, x, w, alpha):
    H = c["H"]
    xn, r = _norm(x, w["g_ffn"])
    h13 = xn @ w["w13"].t()
    gate = torch.nn.functional.silu(h13[:, :H]) * h13[:, H:]
    return x + alpha * (gate @ w["w2"].t()), h13, gate, r


def exact(case, seed):
    c = dict(case)
    if c["op"] in ("mlp_fwd", "mlp_bwd", "attn_fwd", "attn_bwd", "layer"):
        return _exact_block(c, seed)
    if c["op"] == "head":
        return _exact_head(c, seed)
    if c["op"] == "adam":
        return _exact_adam(c, seed)
    if c["op"] == "train":
        return _exact_train(c, seed)
    return None  # tokens


def _exact_block(c, seed):
    i = {k: v.double() if v is not None else None for k, v in _block_inputs(c, seed).items()}
    a, op = _alpha(c), c["op"]
    cos, sin = _rope(c["S"], c["HD"], c["theta"])
    back = op in ("mlp_bwd", "attn_bwd", "layer")
    leaves = [k for k in i if k != "dy" and i[k] is not None]
    if back:
        for k in leaves:
            i[k].requires_grad_(True)
    x = i["x"]
    out = {}
    if op in ("attn_fwd", "attn_bwd", "layer"):
        x, qkv, att, lse = _ref_attn(c, x, i, cos, sin, a)
        out.update(x2=x, qkv=qkv, att=att, lse=lse)
    if op in ("mlp_fwd", "mlp_bwd", "layer"):
        x, h13, gate, r = _ref_mlp(c, x, i, a)
        out.update(out=x, h13=h13, gate=gate, r2=r.reshape(-1))
    if not back:
        return {k: out[k] for k in (("out", "h13", "gate", "r2") if op == "mlp_fwd" else ("x2", "qkv", "att", "lse"))}
    used = [k for k in leaves if not (op == "mlp_bwd" and k == "g_att") and not (op == "attn_bwd" and k == "g_ffn")]
    gr = dict(zip(used, torch.autograd.grad(x, [i[k] for k in used], i["dy"])))
    res = dict(dx=gr["x"])
    if op == "layer":
        res["out"] = x.detach()
    if op == "mlp_bwd":
        res["dxb"] = a * gr["x"]
    if "w13" in gr:
        res.update(dw13=gr["w13"], dw2=gr["w2"], dg_ffn=gr["g_ffn"])
    if "wqkv" in gr:
        res.update(dwqkv=gr["wqkv"], dwo=gr["wo"], dg_att=gr["g_att"])
        if c["qk_norm"]:
            res.update(dgq=gr["gq"], dgk=gr["gk"])
    return res


def _exact_head(c, seed):
    s = _prepare_head(c, seed)
    x, E, t = s["x"].double(), s["E"].double(), s["tgt"].long()
    T, D = x.shape
    lse, loss = torch.empty(T, dtype=torch.float64, device=DEV), 0.0
    dl = torch.empty(s["dlogits"].shape, dtype=torch.float32, device=DEV)
    dx, dE = torch.empty_like(x), torch.zeros_like(E)
    for r0 in range(0, T, 1024):
        r = slice(r0, min(T, r0 + 1024))
        lg = x[r] @ E.t()
        lse[r] = torch.logsumexp(lg, -1)
        p = torch.exp(lg - lse[r, None])
        pt = p.gather(1, t[r, None])
        loss = loss - torch.log(pt + 1e-10).sum()
        p.scatter_add_(1, t[r, None], torch.full_like(pt, -1.0))
        dl[r] = p * DLOGITS_SCALE
        dx[r] = DLOGITS_SCALE * (p @ E)
        dE += p.t() @ x[r] / T
    return dict(loss=(loss / T).reshape(1), lse=lse, dlogits=dl, dx=dx, dE=dE)


def _adamw(p, g, m, v, t, wd):
    k = ADAM
    m = k["b1"] * m + (1 - k["b1"]) * g
    v = k["b2"] * v + (1 - k["b2"]) * g * g
    u = (m / (1 - k["b1"] ** t)) / (torch.sqrt(v / (1 - k["b2"] ** t)) + k["eps"])
    return p - k["lr"] * (u + wd * p), m, v


def _exact_adam(c, seed):
    s = _prepare_adam(c, seed)
    p, g, m, v = (s[k].double() for k in "pgmv")
    norm = g.norm()
    g = g * min(1.0, 1.0 / float(norm))
    wd = torch.full_like(p, ADAM["wd"])
    wd[c["n"] - c["n_gain"]:] = 0
    p, m, v = _adamw(p, g, m, v, 10, wd)
    return dict(p=p, m=m, v=v, pb=p, gnorm=norm.reshape(1))


def _exact_train(c, seed):
    D, L = c["D"], c["L"]
    raw = dict(_model_params(c, seed))
    P = {}
    for l in range(L):
        w = {n: raw.pop(f"layers.{l}.{n}").double() for n in ("Wq", "Wk", "Wv", "Wo", "W1", "W2", "W3")}
        P[f"wqkv.{l}"] = torch.cat((w["Wq"], w["Wk"], w["Wv"]))
        P[f"wo.{l}"], P[f"w2.{l}"] = w["Wo"], w["W2"]
        P[f"w13.{l}"] = torch.cat((w["W1"], w["W3"]))
        for n, k in (("g_att", D), ("g_ffn", D)) + ((("gq", c["HD"]), ("gk", c["HD"])) if c["qk_norm"] else ()):
            P[f"{n}.{l}"] = torch.ones(k, dtype=torch.float64, device=DEV)
    P["embed"] = raw.pop("embed").double()
    P["rms_final"] = torch.ones(D, dtype=torch.float64, device=DEV)
    M = {k: torch.zeros_like(v) for k, v in P.items()}
    V = {k: torch.zeros_like(v) for k, v in P.items()}
    cos, sin = _rope(c["S"], c["HD"], c["theta"])
    a, T = _train_alpha(c), c["B"] * c["S"]
    losses = []
    for step, tok in enumerate(_tokens(c, seed, c["steps"], c["B"], c["S"] + 1)):
        tk = torch.from_numpy(tok).to(DEV).long()
        for v in P.values():
            v.requires_grad_(True)
        x = P["embed"][tk[:, :-1].reshape(-1)]
        for l in range(L):
            w = {n: P.get(f"{n}.{l}") for n in ("wqkv", "wo", "w13", "w2", "g_att", "g_ffn", "gq", "gk")}
            x = _ref_attn(c, x, w, cos, sin, a)[0]
            x = _ref_mlp(c, x, w, a)[0]
        xf, _ = _norm(x, P["rms_final"])
        pt = torch.exp((torch.log_softmax(xf @ P["embed"].t(), -1)).gather(1, tk[:, 1:].reshape(T, 1)))
        loss = -torch.log(pt + 1e-10).mean()
        losses.append(float(loss.detach()))
        g = torch.autograd.grad(loss, list(P.values()))
        f = min(1.0, 1.0 / float(sum(x.square().sum() for x in g).sqrt()))
        for (k, p), gk in zip(list(P.items()), g):
            wd = 0.0 if p.dim() == 1 else ADAM["wd"]
            P[k], M[k], V[k] = _adamw(p.detach(), gk * f, M[k], V[k], step + 1, wd)
    Q, KV = c["NH"] * c["HD"], c["NKV"] * c["HD"]
    return {"layers.0.Wk": P["wqkv.0"][Q:Q + KV].reshape(-1), "layers.0.Wo": P["wo.0"].reshape(-1),
            "layers.0.rms_att": P["g_att.0"], "rms_final": P["rms_final"], "loss": np.array(losses, np.float64)}


_PREPARE = dict(mlp_fwd=_prepare_block, mlp_bwd=_prepare_block, attn_fwd=_prepare_block, attn_bwd=_prepare_block,
                layer=_prepare_block, head=_prepare_head, adam=_prepare_adam, train=_prepare_train, decode=_prepare_decode)
_RUN = dict(mlp_fwd=_run_mlp_fwd, mlp_bwd=_run_mlp_bwd, attn_fwd=_run_attn_fwd, attn_bwd=_run_attn_bwd, layer=_run_layer,
            head=_run_head, adam=_run_adam, train=_run_train, decode=_run_decode)
