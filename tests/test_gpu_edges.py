"""Kernel entry points at the sizes where their launch rules change: remainders of blocks, the
smallest and largest of a range, row pitches that are not multiples of a wide access.  Against
float64 numpy; tolerances from the fp32 sums (a sum of n terms in any order: about sqrt(n) * 2^-24
of its terms' norm) and one 16-bit rounding of the outputs."""
import numpy as np
import pytest

from gpu_util import FMT, _release_device_tensors, call, dev, host, need_gpu, ptr, rel_l2, torch, zeros  # noqa: F401
import ne
from oracle import model as om

pytestmark = pytest.mark.gpu
L = None


@pytest.fixture(autouse=True)
def _gpu():
    need_gpu()
    global L
    L = ne.lib()


# 4 row groups a block, at most 256 blocks: one row, a partial group, one row past a block, the last
# block partly empty, several rows a group; D below, at and above one float4 per thread
@pytest.mark.parametrize("T,D", [(1, 64), (3, 768), (5, 2048), (1024, 832), (1025, 1028), (2051, 128)])
def test_rmsnorm_bwd_gain_sums(T, D):
    dt, tdt, _, u = FMT["fp16"]
    rng = np.random.default_rng(T + D)
    x, dy, res = (rng.standard_normal((T, D)).astype(np.float32) for _ in range(3))
    g = (1 + 0.2 * rng.standard_normal(D)).astype(np.float32)
    r = (1.0 / np.sqrt((x.astype(np.float64) ** 2).mean(1) + 1e-5)).astype(np.float32)
    dx, dxb = zeros((T + 1, D)), zeros((T + 1, D), tdt)
    dg = dev(np.ones(D, np.float32))  # accumulates
    call(L.ne_k_rmsnorm_bwd, dt, ptr(dev(dy)), ptr(dev(x)), ptr(dev(g)), ptr(dev(r)), ptr(dev(res)), ptr(dx),
         ptr(dxb), 0.5, ptr(dg), 2.0, T, D, None)
    X, DY, R = x.astype(np.float64), dy.astype(np.float64), r.astype(np.float64)[:, None]
    ref = R * g * DY - X * R ** 3 * (DY * X * g).sum(1, keepdims=True) / D + res
    got = host(dx)
    assert rel_l2(got[:T], ref) < 1e-6 and not got[T].any() and not host(dxb)[T].any()
    assert rel_l2(host(dxb)[:T], 0.5 * ref) < u
    assert rel_l2(host(dg), 1 + 2 * (DY * X * R).sum(0)) < 1e-5


# tokens a block: 2 on short steps, ceil(T / 512) above; a last block with one token; heads whose slots
# leave lanes of the last pass idle; a pitch of 2 elements more than a row (4-byte aligned rows)
@pytest.mark.parametrize("fmt", ["fp16", "bf16"])
@pytest.mark.parametrize("T,S,NH,NKV,HD,pad,qk", [(64, 64, 2, 1, 64, 0, True), (192, 64, 3, 3, 128, 2, True),
                                                  (1088, 1088, 10, 5, 64, 0, True), (1088, 64, 5, 1, 128, 2, True),
                                                  (192, 192, 5, 5, 64, 2, False)])
def test_qk_prep_bwd_edges(fmt, T, S, NH, NKV, HD, pad, qk):
    dt, tdt, rnd, u = FMT[fmt]
    Q, KV = NH * HD, NKV * HD
    QKV = Q + 2 * KV
    ld = QKV + pad
    rng = np.random.default_rng(T + HD + pad)
    qkv = rnd(rng.standard_normal((T, ld)).astype(np.float32))
    gq, gk = ((1 + 0.3 * rng.standard_normal(HD)).astype(np.float32) for _ in range(2))
    cos, sin = om.rope_tables(S, HD, 1e4)
    dq, dk = rng.standard_normal((T, Q)).astype(np.float32), rng.standard_normal((T, KV)).astype(np.float32)
    B = T // S
    q, k = qkv[:, :Q].reshape(B, S, NH, HD), qkv[:, Q:Q + KV].reshape(B, S, NKV, HD)
    dqn, dkn = om.rope_bwd(dq.reshape(B, S, NH, HD), cos, sin), om.rope_bwd(dk.reshape(B, S, NKV, HD), cos, sin)
    rq = rk = None
    if qk:
        rq, rk = om.rmsnorm(q, gq, 1e-5)[1], om.rmsnorm(k, gk, 1e-5)[1]
        (dqn, dgqr), (dkn, dgkr) = om.rmsnorm_bwd(dqn, q, gq, rq), om.rmsnorm_bwd(dkn, k, gk, rk)
    dqkv = zeros((T, ld), tdt)
    o = np.ones(HD, np.float32)
    dgq, dgk = (dev(o), dev(o)) if qk else (None, None)
    P = lambda a: ptr(dev(a)) if a is not None else None  # noqa: E731
    call(L.ne_k_qk_prep_bwd, dt, P(dq), P(dk), ptr(dev(qkv, tdt)), ld,
         P(cos.astype(np.float32)), P(sin.astype(np.float32)), P(gq) if qk else None, P(gk) if qk else None,
         P(rq.reshape(T, NH)) if qk else None, P(rk.reshape(T, NKV)) if qk else None, ptr(dqkv), ptr(dgq), ptr(dgk),
         2.0, T, S, NH, NKV, HD, None)
    got = host(dqkv)
    assert rel_l2(got[:, :Q], dqn.reshape(T, Q)) < u
    assert rel_l2(got[:, Q:Q + KV], dkn.reshape(T, KV)) < u
    assert not got[:, Q + KV:].any()  # the v columns and the padding are not this call's
    if qk:
        assert rel_l2(host(dgq), 1 + 2 * dgqr) < 1e-4 and rel_l2(host(dgk), 1 + 2 * dgkr) < 1e-4


# The sums behind dqkv have one order, whichever form runs (the wide one, on 16-byte rows or on a pitch or a base
# that is not; one head a block for few tokens without gains, which the training step uses too): a head's
# products by pairs, the pairs in a butterfly of strides 1, 2, 4 ..., fused multiply-adds where written here.  Restated in numpy (a float64
# product of two float32 values is exact), so every element has the same bits; the two forms' borders
# (191 / 192 tokens without gains), one token, and an empty last pass.
@pytest.mark.parametrize("fmt", ["fp16", "bf16"])
@pytest.mark.parametrize("T,NH,NKV,HD,qk", [(512, 16, 8, 128, True), (1, 16, 8, 128, True), (512, 10, 5, 64, True),
                                            (191, 12, 12, 64, False), (192, 12, 12, 64, False), (1025, 16, 8, 128, False)])
def test_qk_prep_bwd_bits(fmt, T, NH, NKV, HD, qk):
    dt, tdt, rnd, _ = FMT[fmt]
    f32 = np.float32
    Q, KV, N = NH * HD, NKV * HD, NH + NKV
    rng = np.random.default_rng(T + HD)
    qkv = rnd(rng.standard_normal((T, Q + 2 * KV)).astype(f32))
    gq, gk = ((1 + 0.3 * rng.standard_normal(HD)).astype(f32) for _ in range(2))
    rq, rk = (rng.uniform(0.5, 2, (T, n)).astype(f32) for n in (NH, NKV))
    cos, sin = (t.astype(f32) for t in om.rope_tables(T, HD, 1e4))
    dq, dk = rng.standard_normal((T, Q)).astype(f32), rng.standard_normal((T, KV)).astype(f32)

    def fma64(a, b, c):
        return a.astype(np.float64) * b.astype(np.float64) + c.astype(np.float64)

    y = np.concatenate([dq, dk], 1).reshape(T, N, HD // 2, 2)
    c, s = cos[:, None], sin[:, None]
    rot = np.stack([fma64(y[..., 0], c, y[..., 1] * s), fma64(y[..., 1], c, -(y[..., 0] * s))], -1)
    if qk:
        d, x = rot.astype(f32), qkv[:, :Q + KV].reshape(T, N, HD // 2, 2)
        g = np.concatenate([np.tile(gq, (NH, 1)), np.tile(gk, (NKV, 1))]).reshape(N, HD // 2, 2)
        r = np.concatenate([rq, rk], 1)[..., None]
        dx = d * x
        dot = fma64(dx[..., 0], g[..., 0], dx[..., 1] * g[..., 1]).astype(f32)
        while dot.shape[-1] > 1:
            dot = dot[..., 0::2] + dot[..., 1::2]
        cc = (r * r * r * dot / f32(HD))[..., None]
        ref = rnd(fma64(r[..., None] * g, d, -(x * cc)).astype(f32))
    else:  # fp16: the rotation is rounded once
        ref = rot.astype(np.float16).astype(f32) if fmt == "fp16" else rnd(rot.astype(f32))
    ref = ref.reshape(T, Q + KV)
    P = lambda a: ptr(dev(a)) if qk else None  # noqa: E731
    for pitch, base in ((0, 0), (8, 0), (2, 0), (8, 2)):  # elements beyond a row; of the arrays' start
        ld = Q + 2 * KV + pitch
        buf, out = zeros(T * ld + base, tdt), zeros(T * ld + base, tdt)
        buf[base:].view(T, ld)[:, :Q + 2 * KV] = dev(qkv, tdt)
        dgq, dgk = (dev(np.ones(HD, f32)) for _ in range(2))
        call(L.ne_k_qk_prep_bwd, dt, ptr(dev(dq)), ptr(dev(dk)), ptr(buf[base:]), ld, ptr(dev(cos)), ptr(dev(sin)),
             P(gq), P(gk), P(rq), P(rk), ptr(out[base:]), ptr(dgq) if qk else None, ptr(dgk) if qk else None, 2.0, T, T,
             NH, NKV, HD, None)
        got = host(out)[base:].reshape(T, ld)
        assert np.array_equal(got[:, :Q + KV], ref), (pitch, base, int((got[:, :Q + KV] != ref).sum()))
        assert not got[:, Q + KV:].any()
        if qk:
            a = dx.astype(np.float64) * r[..., None]
            for got_g, h in ((dgq, slice(0, NH)), (dgk, slice(NH, N))):
                assert rel_l2(host(got_g), 1 + 2 * a[:, h].sum((0, 1)).reshape(HD)) < 1e-4


# Sampling runs a row of logits in chunks of at least 1024 columns: one chunk, two, a last chunk shorter
# than the others, and without the mask up to 2048 columns in one block; peaked (gain 8) and flat (gain 1) distributions, with and without the top-p mask.
# A pick may differ from the oracle's only where its uniform lies within 1e-5 of the boundary between
# the two in cumulative probability (the fp32 logits and their softmax, 32k terms of rounding 6e-8).
@pytest.mark.parametrize("V,B,gain,top_p", [(512, 1, 8.0, 0.9), (1024, 3, 1.0, 1.0), (2112, 5, 8.0, 0.95),
                                            (2112, 2, 1.0, 0.5), (2048, 2, 1.0, 1.0), (2112, 3, 1.0, 1.0),
                                            (32064, 1, 8.0, 0.9), (32064, 6, 1.0, 1.0)])
def test_decode_sampling_chunks(V, B, gain, top_p):
    cfg = om.tiny(vocab=V)
    P = {k: om.round_bf16(v) for k, v in om.init_params(cfg, seed=V).items()}
    P["rms_final"] = np.full_like(P["rms_final"], gain)
    n, temp = 12, 0.8
    m = ne.Model.from_oracle(cfg, decode_batch=B, decode_ctx=4 + n, dtype=ne.NE_BF16)
    m.set_params(P)
    rng = np.random.default_rng(V + B)
    prompt, u = rng.integers(0, V, (B, 4)).astype(np.int32), rng.random((B, n))
    got = m.decode(prompt, n, temp, top_p, u)
    np.testing.assert_array_equal(m.decode(prompt, n, temp, top_p, u), got)
    picks, dist = om.decode(cfg, P, prompt, n, temperature=temp, top_p=top_p, uniforms=u, forced=got)
    assert np.abs(dist).max() < 1e-5, (np.argwhere(picks != got), np.abs(dist).max())
    # the first uniform picks the first kept token, the last one the last; no finite logit: token 0
    lo = m.decode(prompt, 1, temp, 1.0, np.zeros((B, 1)))
    hi = m.decode(prompt, 1, temp, 1.0, np.full((B, 1), 1 - 2.0 ** -53))
    assert (lo == 0).all() and (hi > V - 64).all()
    # a uniform of 1 or more lies past every token: the last one that holds mass
    one = m.decode(prompt, 1, temp, top_p, np.full((B, 1), 1.0))
    np.testing.assert_array_equal(one, m.decode(prompt, 1, temp, top_p, np.full((B, 1), 1 - 2.0 ** -53)))
    np.testing.assert_array_equal(one, m.decode(prompt, 1, temp, top_p, np.full((B, 1), 7.0)))
    m.set("rms_final", np.full(cfg.dim, np.nan, np.float32))
    assert (m.decode(prompt, 2, temp, top_p, u[:, :2]) == 0).all()
    m.close()


# A uniform of 0 picks the first token whose probability is above 0, however small (numpy: the first index
# with cdf > 0): logits spread so that probabilities run down to the smallest normal float32.
@pytest.mark.parametrize("top_p", [1.0, 0.9])
def test_decode_sampling_tiny_probabilities(top_p):
    B, V = 4, 2112
    cfg = om.tiny(vocab=V)
    P = {k: om.round_bf16(v) for k, v in om.init_params(cfg, seed=3).items()}
    P["rms_final"] = np.full_like(P["rms_final"], 60.0)
    rng = np.random.default_rng(5)
    prompt, u = rng.integers(0, V, (B, 4)).astype(np.int32), np.zeros((B, 1))
    want, _, logits = om.decode(cfg, P, prompt, 1, return_logits=True)
    first = np.exp(np.float64(logits[0][:, 0]) - np.float64(logits[0]).max(1))
    assert ((first > 2.0 ** -110) & (first < 2.0 ** -64)).any()  # token 0, far from 1 and above 0
    m = ne.Model.from_oracle(cfg, decode_batch=B, decode_ctx=8, dtype=ne.NE_BF16)
    m.set_params(P)
    got = m.decode(prompt, 1, 1.0, top_p, u)
    np.testing.assert_array_equal(got, om.decode(cfg, P, prompt, 1, temperature=1.0, top_p=top_p, uniforms=u))
    m.close()


# The prompt before its last position runs in chunks of up to 256 rows (sequence x position): rows below 16
# and 32 and at several 32s, chunk borders, the last chunk with one position, batches of both K-cache
# layouts, and the one or two positions that a small batch takes one at a time.  Picks as in
# test_decode_sampling_chunks.
@pytest.mark.parametrize("B,P,fmt,kw", [(1, 2, "bf16", {}), (1, 3, "bf16", {}), (1, 4, "fp16", {}), (2, 40, "bf16", dict(qk_norm=True)),
                                        (3, 87, "fp16", dict(head_dim=128, qk_norm=True)), (4, 66, "bf16", {}),
                                        (5, 53, "bf16", dict(head_dim=128, n_heads=2, qk_norm=True)),
                                        (5, 2, "fp16", {}), (17, 17, "fp16", dict(n_heads=8)),
                                        (32, 18, "bf16", dict(dim=256, hidden=384))])
def test_decode_prompt_chunks(B, P, fmt, kw):
    cfg = om.tiny(**kw)
    dt, _, rnd, _ = FMT[fmt]
    W = {k: rnd(v) for k, v in om.init_params(cfg, seed=P).items()}
    W["rms_final"] = np.full_like(W["rms_final"], 8.0)
    n = 6
    m = ne.Model.from_oracle(cfg, decode_batch=B, decode_ctx=P + n, dtype=dt)
    m.set_params(W)
    rng = np.random.default_rng(P + B)
    prompt, u = rng.integers(0, cfg.vocab, (B, P)).astype(np.int32), rng.random((B, n))
    got = m.decode(prompt, n, 0.8, 1.0, u)
    m.use_graphs(False)
    np.testing.assert_array_equal(m.decode(prompt, n, 0.8, 1.0, u), got)
    picks, dist = om.decode(cfg, W, prompt, n, temperature=0.8, top_p=1.0, uniforms=u, forced=got)
    assert np.abs(dist).max() < 1e-5, (np.argwhere(picks != got), np.abs(dist).max())
    m.close()


# The entry point's GEMM at the sizes where its tile changes.  Two edges of the ragged 8-wave 128x128 tile (M, N
# odd multiples of 64: the last tile overlaps the one before it), 64x64 on 64-deep steps, ragged 128x64 for the
# epilogues that read, and the K-divided tiles of 64x64, 64x32 and 32x32, with fewer K steps than waves
# (K = 64, 192) and an uneven share of them (K = 576, 1088).  Then 256x256, 256x128 (also at the SwiGLU backward's
# 256 tiles, and below it, where that epilogue takes 128x128 on 4 waves), 128x128 on 4 waves (289 and exactly 256
# tiles) and on 8 (143 tiles), 64x64 for 289 ragged tiles and 8 waves again with a long K, 128x64 for a ragged
# residual of 575 tiles, 128x64 with K = 448, and the K-divided 64x32 at 80 tiles and 64x64 for the SwiGLU backward.
# Last 841 ragged 64x64 tiles for an accumulation of both operands K-contiguous, 8 waves for the others.
# C has rows and columns of its own around it.  fp32 sums of K products: 1e-5 of the largest.
@pytest.mark.parametrize("M,N,K", [(3136, 4160, 128), (3136, 2112, 64), (1856, 1472, 192), (1088, 1024, 64),
                                   (2496, 832, 128), (576, 1024, 2112), (384, 1024, 1088), (320, 768, 576),
                                   (64, 64, 64), (64, 1024, 192),
                                   (3072, 4096, 128), (2048, 4224, 64), (2048, 3200, 64), (2176, 2176, 128),
                                   (2048, 2048, 192), (1408, 1600, 128), (2112, 2112, 128), (2112, 2112, 2112),
                                   (3136, 2880, 64), (1088, 1024, 448), (320, 1024, 576), (576, 1024, 4160),
                                   (1856, 1856, 192)])
@pytest.mark.parametrize("layout,epi,fmt", [(0, 0, "bf16"), (0, 2, "fp16"), (0, 3, "fp16"), (1, 1, "fp16"), (2, 1, "fp16"),
                                            (2, 2, "bf16"), (2, 4, "fp16"), (3, 1, "bf16"), (3, 2, "fp16"),
                                            (2, 0, "fp16"), (2, 0, "bf16"), (2, 4, "bf16")])
def test_gemm_tiles(M, N, K, layout, epi, fmt):
    dt, tdt, _, u = FMT[fmt]
    g = torch.Generator(device="cuda").manual_seed(M + N + K + layout)
    rnd = lambda *sh: torch.randn(sh, generator=g, device="cuda")  # noqa: E731
    A, B = rnd(M, K).to(tdt), rnd(K, N).to(tdt)
    ref = 0.5 * (A.double() @ B.double())
    a = A.t().contiguous() if layout & 1 else A
    b = B if layout & 2 else B.t().contiguous()
    ld = 2 * N + 8 if epi == 4 else N + 8
    half = epi in (0, 4)
    c = torch.full((M + 1, ld), 3.0, device="cuda", dtype=tdt if half else torch.float32)
    R = rnd(M, 2 * N).to(tdt) if epi == 4 else rnd(M, N) if epi == 3 else None
    if epi == 2:
        ref = ref + 3.0
    elif epi == 3:
        ref = ref + R.double()
    elif epi == 4:
        h1, h3 = R.double()[:, :N], R.double()[:, N:]
        sg = torch.sigmoid(h1)
        ref = torch.cat([ref * h3 * sg * (1 + h1 * (1 - sg)), ref * h1 * sg], 1)
    call(L.ne_k_gemm, dt, layout, epi, M, N, K, ptr(a), a.shape[1], ptr(b), b.shape[1], ptr(c), ld, ptr(R),
         R.shape[1] if R is not None else 0, 0.5, None)
    W = ref.shape[1]
    assert (c[M] == 3.0).all() and (c[:, W:] == 3.0).all()
    d = c[:M, :W].double() - ref
    if half:
        assert float(d.norm() / ref.norm()) < u
    else:
        assert float(d.abs().max() / ref.abs().max()) < 1e-5


# dQ blocks of 128 queries: S a multiple of 64 only, so that the block with the first queries is half
# outside; dK / dV blocks of two head groups (short sequences, 2 or 4 query heads per KV head, up to
# 256 blocks in all and one more; exactly 256, 240 in rows that the XCDs share unevenly); bf16 heads of 64 with
# 352 and 570 blocks (two and three waves per SIMD); against float64 autograd.  P and dS are rounded to 16 bits: a few roundings deep.
@pytest.mark.parametrize("B,S,NH,NKV,HD", [(8, 192, 16, 4, 64), (8, 192, 16, 8, 128), (2, 576, 26, 13, 128),
                                           (8, 256, 16, 16, 64), (1, 64, 2, 1, 128), (1, 128, 8, 2, 64),
                                           (2, 192, 6, 3, 128), (1, 512, 16, 8, 128), (1, 576, 16, 8, 64),
                                           (32, 64, 4, 2, 64), (2, 256, 16, 8, 128), (10, 64, 16, 4, 64),
                                           (6, 576, 10, 5, 64)])
@pytest.mark.parametrize("fmt", ["fp16", "bf16"])
def test_attn_bwd_two_groups(fmt, B, S, NH, NKV, HD):
    dt, tdt, _, u = FMT[fmt]
    g = torch.Generator(device="cuda").manual_seed(S + HD)
    T, Q, KV = B * S, NH * HD, NKV * HD
    q, k, v, do = (torch.randn((T, n), generator=g, device="cuda").to(tdt) for n in (Q, KV, KV, Q))
    qd, kd, vd = (t.double().view(B, S, -1, HD).transpose(1, 2).contiguous().requires_grad_() for t in (q, k, v))
    rep = lambda t: t.repeat_interleave(NH // NKV, 1)  # noqa: E731
    s = torch.matmul(qd, rep(kd).transpose(2, 3).contiguous()) * HD ** -0.5
    s = s.masked_fill(torch.ones(S, S, dtype=torch.bool, device="cuda").triu(1), float("-inf"))
    o = torch.matmul(s.softmax(-1), rep(vd))
    o.backward(do.double().view(B, S, NH, HD).transpose(1, 2))
    flat = lambda t: t.detach().transpose(1, 2).reshape(T, -1)  # noqa: E731
    lse = s.detach().logsumexp(-1).transpose(1, 2).reshape(T, NH).float().contiguous()
    od = flat(o).to(tdt)
    delta, dq, dk, dv = zeros((T, NH)), zeros((T, Q)), zeros((T, KV)), zeros((T, KV), tdt)
    call(L.ne_k_attn_bwd, dt, ptr(q), Q, ptr(k), KV, ptr(v), KV, ptr(od), Q, ptr(lse), ptr(do), Q,
         ptr(delta), ptr(dq), Q, ptr(dk), KV, ptr(dv), KV, B, S, NH, NKV, HD, HD ** -0.5, None)
    for got, ref in ((dq, qd), (dk, kd), (dv, vd)):
        assert rel_l2(host(got), flat(ref.grad).cpu().numpy()) < 4 * u
