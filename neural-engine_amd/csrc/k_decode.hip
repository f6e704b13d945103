// KV-cached token loop: the MI355X form of generate() in TD/tools/generate.py:113-228.
//
// Per position every layer runs: RMSNorm -> fused QKV GEMV -> (QK-norm) RoPE + KV-cache
// append -> GQA attention over the cache -> Wo GEMV + residual -> RMSNorm -> W1|W3 GEMV ->
// SwiGLU -> W2 GEMV + residual; then the final norm, the tied LM-head GEMV and greedy /
// temperature / top-p sampling on the device.  Weights are the 16-bit shadow; activations,
// the KV cache and all accumulation are fp32.
//
// Every kernel reads the position from device memory (DecState), so the launch sequence of
// one position does not depend on it: it is captured once as a HIP graph (one for prompt
// positions, one for generated ones) and replayed per position.  A longer prompt's positions before
// the last run in chunks of up to 256 rows (sequence x position) through the batch 5..32 GEMVs
// (enqueue_prompt).
//
// GEMVs are HBM-bound (each weight byte is read once per position whatever the batch):
//  * batch <= 4: VALU kernel.  The block stages its input rows in LDS (fusing the RMSNorm or
//    the SwiGLU gate into that prologue), each wave streams 1-4 weight rows with 16-byte
//    loads (8 weights per lane, two chunks of 512 in flight), wave reductions.  The LM-head
//    launch also writes per-block (max, first index) partials for greedy argmax.
//  * batch 5..32: v_mfma_f32_16x16x4_f32, 16 weight rows x 16 sequences per MFMA tile,
//    K split over the 4 waves of a block and over grid.y (fp32 partials, ordered reduction).
#include <math.h>
#include <type_traits>

#include "common.h"
#include "ne_ctx.h"

namespace {

struct DecState {
  int pos;      // position being processed
  int P;        // prompt length
  float temp;   // < 1e-6: greedy
  float top_p;
};

// How a position's token is chosen: not at all (a prompt position before the last), the first maximum, or
// sampled without or with a top-p mask.
enum { PICK_NONE = -1, PICK_GREEDY = 0, PICK_SAMPLE = 1, PICK_TOPP = 2 };

constexpr int VB = 4;            // largest batch of the VALU GEMV path
constexpr int PROMPT_ROWS = 256; // most rows of a prompt chunk
constexpr int BIG_ARGMAX = 256;  // argmax partials per sequence on the MFMA path

struct Dec {
  int Bmax;               // decode_batch
  int Bp;                 // MFMA path: batch padded to 16 or 32
  int Rp;                 // rows (sequence x position) of a prompt chunk: >= Bp, a multiple of 16
  int ctx;                // max positions
  float *kc, *vc;         // [L][Bmax][NKV] of V [ctx][HD] and K [ctx][HD] (batch <= 4: [HD/4][ctx] float4 pieces)
  float *x, *xn, *att;    // [Rp, *]
  float *qkv, *logits;    // [Bp, *]
  float *ws;              // MFMA split-K partials
  long ws_elems;
  float *gate;            // [Rp, H] SwiGLU gate (MFMA path)
  h16_t *xn3, *att3, *gate3;  // bf16 weights, MFMA path: the bf16 parts (part_at) of xn, att, gate
  float *amv;             // argmax partials [Bmax][nblk]
  int32_t *ami;
  int lm_nblk;
  int32_t *tok;           // [Bp] current token
  int32_t *out;           // [Bp, ctx] generated tokens
  int32_t *prompt;        // [Bp, ctx]
  double *unif;           // [Bp, ctx]
  int sg, schunk;         // sampling: chunks per row of logits, columns per chunk
  float *spmax;           // sampling partials (SampArgs)
  double *spsum;
  unsigned long long *shist, *smass, *sabove;
  uint32_t *spre;
  float *cosb, *sinb;     // [ctx, HD/2]
  DecState *st;
  void *arena;
  struct Graph { int B, mode; hipGraphExec_t exec; };  // mode: PICK_*
  std::vector<Graph> graphs;
};

// x = hi + mid + lo, three bf16 values obtained by truncation: hi keeps the top 8 significant
// bits of x, mid the next 8 of the remainder x - hi, lo what is left, so the sum is exact and
// each product of a bf16 weight with a part is exact in fp32.
__device__ __forceinline__ void split3(float x, uint16_t &hi, uint16_t &mid, uint16_t &lo) {
  const uint32_t u = __float_as_uint(x) & 0xFFFF0000u;
  const float r1 = x - __uint_as_float(u);
  const uint32_t u1 = __float_as_uint(r1) & 0xFFFF0000u;
  const float r2 = r1 - __uint_as_float(u1);
  hi = (uint16_t)(u >> 16);
  mid = (uint16_t)(u1 >> 16);
  lo = (uint16_t)(__float_as_uint(r2) >> 16);
}

// The parts of a row-major [rows, K] matrix as gemv_bf3_kernel reads them: for each tile of 16 rows and
// step of 32 columns three 1 KB fragments (hi, mid, lo) in lane order (16 (k / 8 % 4) + row % 16, 8
// columns each), so that a fragment is one contiguous read.  As row-major planes each load of a wave
// touched 16 rows a power of two apart.
__device__ __forceinline__ long part_at(long K, long row, long k) {
  return ((row >> 4) * (K >> 5) + (k >> 5)) * 1536 + (((k >> 3) & 3) * 16 + (row & 15)) * 8 + (k & 7);
}
// The three parts of element (row, k), or of 4 from k on (a multiple of 4); p may be null.
__device__ __forceinline__ void put3(h16_t *p, long K, long row, long k, float v) {
  if (!p) return;
  uint16_t h, m, l;
  split3(v, h, m, l);
  h16_t *q = p + part_at(K, row, k);
  q[0] = h;
  q[512] = m;
  q[1024] = l;
}
__device__ __forceinline__ void put3(h16_t *p, long K, long row, long k, const float4 &v) {
  if (!p) return;
  const float f[4] = {v.x, v.y, v.z, v.w};
  u16x4 h, m, l;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    uint16_t a, b, c;
    split3(f[i], a, b, c);
    h[i] = a; m[i] = b; l[i] = c;
  }
  h16_t *q = p + part_at(K, row, k);
  *(u16x4 *)q = h;
  *(u16x4 *)(q + 512) = m;
  *(u16x4 *)(q + 1024) = l;
}

// ------------------------------------------------------------------ GEMV, batch <= 4 ----

enum { PRO_NONE = 0, PRO_RMSNORM = 1, PRO_SWIGLU = 2 };

// out[b, n] = alpha * sum_k W[n, k] * in'(b, k) + (resid ? resid[b, n] : 0), rows n of this
// block = (blockIdx.x * 4 + wave) * RPW + r.  in' = in (PRO_NONE), in / rms(in) * g
// (PRO_RMSNORM, generate.py:81-84) or silu(h1) * h3 with in = [h1 | h3] rows of 2K
// (PRO_SWIGLU).  resid may alias out (each element is read, then written, by one lane).
// AMX: also write the block's (max, first row) of each sequence to amv/ami [b][blockIdx.x].
// Every global load (input rows, gains, residual, then the wave's weights: KC chunks of 512
// per row, K <= 512*KC) is issued before the first wait, so the block pays one HBM latency,
// not one per load: with loads behind branches or in a load-store loop each waited for the
// one before, which doubled the time of a batch-1 GEMV.
// GATE (W1|W3 rows [2*gate_n, K]): the wave's rows are j..j+RPW/2-1 of W1 and the same j of
// W3 (rows gate_n + j), and it writes gate[b, j] = silu(h1) * h3 (generate.py:190) instead of h1, h3.
template <typename HT, int NB, int RPW, int KC, int PRO, bool AMX, bool GATE>
__global__ __launch_bounds__(256) void gemv_valu_kernel(const h16_t *__restrict__ W, int K,
                                                        const float *__restrict__ in, long ldi,
                                                        const float *__restrict__ g, float eps, float *out, long ldo,
                                                        const float *resid, float alpha, int B, float *amv,
                                                        int32_t *ami, int nblk, long gate_n) {
  extern __shared__ float xs[];  // [NB][K]
  __shared__ float red[4][NB];
  __shared__ float bmv[NB][4 * RPW];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  constexpr int HALF = GATE ? RPW / 2 : RPW;
  const long row0 = ((long)blockIdx.x * 4 + w) * HALF;
  auto wrow = [&](int r) -> long { return GATE && r >= HALF ? gate_n + row0 + (r - HALF) : row0 + r; };
  // Every global load of the block is issued before the first wait: the input rows (16 bytes
  // per lane, XI per row), the gains, the residual and then the weights.  Addresses past the
  // end of a row are clamped into it (no branches around loads, so none waits for another);
  // the values they bring are not used.
  constexpr int XI = (KC + 1) / 2;  // 1024 * XI >= 512 * KC >= K
  float4 xa[NB][XI], xb[PRO == PRO_SWIGLU ? NB : 1][XI], gv[XI];
#pragma unroll
  for (int i = 0; i < XI; i++) {
    const int k = (i * 256 + tid) * 4, kc = k < K ? k : K - 4;
#pragma unroll
    for (int b = 0; b < NB; b++) {
      const float *src = in + (long)(b < B ? b : B - 1) * ldi;
      xa[b][i] = *(const float4 *)(src + kc);
      if (PRO == PRO_SWIGLU) xb[b][i] = *(const float4 *)(src + K + kc);
    }
    if (PRO == PRO_RMSNORM) gv[i] = *(const float4 *)(g + kc);
  }
  // residual of this lane's output (written by the same lane below; resid may alias out)
  const int rl = lane < RPW * NB ? lane / NB : 0, bl = lane < RPW * NB ? lane % NB : 0;
  const float res_v = !GATE && resid && lane < RPW * NB && bl < B ? resid[(long)bl * ldo + row0 + rl] : 0.f;
  u16x8 wv[RPW][KC];
#pragma unroll
  for (int c = 0; c < KC; c++) {
    const int k = c * 512 + lane * 8, kc = k < K ? k : K - 8;
#pragma unroll
    for (int r = 0; r < RPW; r++) wv[r][c] = __builtin_nontemporal_load((const u16x8 *)(W + wrow(r) * K + kc));
  }
  float rms[NB];
  if (PRO == PRO_RMSNORM) {
    float ss[NB];
#pragma unroll
    for (int b = 0; b < NB; b++) {
      ss[b] = 0.f;
#pragma unroll
      for (int i = 0; i < XI; i++)
        if ((i * 256 + tid) * 4 < K) {
          const float4 v = xa[b][i];
          ss[b] += v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w;
        }
      ss[b] = wave_sum(ss[b]);
    }
    if (lane == 0)
#pragma unroll
      for (int b = 0; b < NB; b++) red[w][b] = ss[b];
    __syncthreads();
#pragma unroll
    for (int b = 0; b < NB; b++) rms[b] = sqrtf((red[0][b] + red[1][b] + red[2][b] + red[3][b]) / (float)K + eps);
  }
#pragma unroll
  for (int i = 0; i < XI; i++) {
    const int k = (i * 256 + tid) * 4;
    if (k < K) {
#pragma unroll
      for (int b = 0; b < NB; b++) {
        float4 v = xa[b][i];
        if (PRO == PRO_SWIGLU) {
          const float4 h3 = xb[b][i];
          v.x = v.x * (1.f / (1.f + expf(-v.x))) * h3.x;
          v.y = v.y * (1.f / (1.f + expf(-v.y))) * h3.y;
          v.z = v.z * (1.f / (1.f + expf(-v.z))) * h3.z;
          v.w = v.w * (1.f / (1.f + expf(-v.w))) * h3.w;
        } else if (PRO == PRO_RMSNORM) {
          v.x = v.x / rms[b] * gv[i].x;
          v.y = v.y / rms[b] * gv[i].y;
          v.z = v.z / rms[b] * gv[i].z;
          v.w = v.w / rms[b] * gv[i].w;
        }
        if (b >= B) v = make_float4(0.f, 0.f, 0.f, 0.f);
        *(float4 *)(xs + b * K + k) = v;
      }
    }
  }
  __syncthreads();

  float acc[RPW][NB];
#pragma unroll
  for (int r = 0; r < RPW; r++)
#pragma unroll
    for (int b = 0; b < NB; b++) acc[r][b] = 0.f;
#pragma unroll
  for (int c = 0; c < KC; c++) {
    const int k = c * 512 + lane * 8;
    if (k < K) {
#pragma unroll
      for (int b = 0; b < NB; b++) {
        const float4 x0 = *(const float4 *)(xs + b * K + k), x1 = *(const float4 *)(xs + b * K + k + 4);
        const float xv[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
#pragma unroll
        for (int r = 0; r < RPW; r++)
#pragma unroll
          for (int j = 0; j < 8; j++) acc[r][b] = fmaf(HT::f(wv[r][c][j]), xv[j], acc[r][b]);
      }
    }
  }
#pragma unroll
  for (int r = 0; r < RPW; r++)
#pragma unroll
    for (int b = 0; b < NB; b++) acc[r][b] = wave_sum(acc[r][b]);
  if (GATE) {
    if (lane < HALF * NB) {
      const int r = lane / NB, b = lane % NB;
      float h1 = 0.f, h3 = 0.f;
#pragma unroll
      for (int rr = 0; rr < HALF; rr++)
#pragma unroll
        for (int bb = 0; bb < NB; bb++)
          if (rr == r && bb == b) {
            h1 = acc[rr][bb];
            h3 = acc[rr + HALF][bb];
          }
      if (b < B) out[(long)b * ldo + row0 + r] = h1 * (1.f / (1.f + expf(-h1))) * h3;
    }
    return;
  }
  if (lane < RPW * NB) {
    const int r = lane / NB, b = lane % NB;
    float v = 0.f;
#pragma unroll
    for (int rr = 0; rr < RPW; rr++)
#pragma unroll
      for (int bb = 0; bb < NB; bb++)
        if (rr == r && bb == b) v = acc[rr][bb];
    if (b < B) {
      const long n = row0 + r;
      float o = alpha * v;
      if (resid) o += res_v;
      out[(long)b * ldo + n] = o;
      if (AMX) bmv[b][w * RPW + r] = o;
    }
  }
  if (AMX) {
    __syncthreads();
    if (tid < NB && tid < B) {
      float best = bmv[tid][0];
      int bi = 0;
      for (int i = 1; i < 4 * RPW; i++)
        if (bmv[tid][i] > best) { best = bmv[tid][i]; bi = i; }  // first maximum
      amv[(long)tid * nblk + blockIdx.x] = best;
      ami[(long)tid * nblk + blockIdx.x] = (int32_t)(blockIdx.x * 4 * RPW + bi);
    }
  }
}

// ------------------------------------------------------------------ GEMV, batch 5..32 ----

__device__ __forceinline__ f32x4 mfma_f32(float a, float b, const f32x4 &c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Products of 16 weight rows (blockIdx.x) with x rows [Bp, K] (fp32, row stride ldx) over the
// K range of split blockIdx.y, for NT tiles of 16 sequences; the 4 waves split that range.
// With a workspace ws, split z's products go to slice z of ws [ksplit][Bp, N] (one split's
// slice is laid out as the output rows); without (one split), out = alpha * products + resid.
// blockIdx.z takes the rows NT * 16 * z .. of x (a prompt chunk has more than NT * 16).
// GATE (one split; W = [W1; W3], gate_n rows each): the block's rows are j0..j0+7 of W1 and
// the same of W3 (j0 = 8 * blockIdx.x), and it writes out[b, j] = silu(h1) * h3
// (generate.py:190).  WV waves per block split the K range (a multiple of 32 each).
template <typename HT, int NT, bool GATE, int WV = 4>
__global__ __launch_bounds__(WV * 64) void gemv_mfma_kernel(const h16_t *__restrict__ W, long ldw,
                                                        const float *__restrict__ x, long ldx, int K, int ksplit,
                                                        float *out, long ldo, const float *resid, float alpha,
                                                        float *ws, int N, int B, int Bp, long gate_n,
                                                        h16_t *out3) {
  __shared__ f32x4 red[WV][NT][64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int g = lane >> 4, r = lane & 15;
  const long row = GATE ? (r < 8 ? (long)blockIdx.x * 8 + r : gate_n + (long)blockIdx.x * 8 + r - 8)
                        : (long)blockIdx.x * 16 + r;
  const int kc = K / ksplit, ks = kc / WV;
  const int kbeg = blockIdx.y * kc + w * ks, kend = kbeg + ks;
  f32x4 acc[NT];
#pragma unroll
  for (int t = 0; t < NT; t++) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  const h16_t *wr = W + row * ldw;
  // G chunks of 32: the weights and the x rows all loaded before the first MFMA (the barrier keeps
  // them there), no load behind another's use.
  auto group = [&](int base, auto gc) {
    constexpr int G = decltype(gc)::value;
    u16x8 wv[G];
    float4 xa[G][NT][2];
#pragma unroll
    for (int i = 0; i < G; i++) wv[i] = __builtin_nontemporal_load((const u16x8 *)(wr + base + i * 32 + g * 8));
#pragma unroll
    for (int i = 0; i < G; i++)
#pragma unroll
      for (int t = 0; t < NT; t++) {
        const float *xr = x + (long)((blockIdx.z * NT + t) * 16 + r) * ldx + base + i * 32 + g * 8;
        xa[i][t][0] = *(const float4 *)xr;
        xa[i][t][1] = *(const float4 *)(xr + 4);
      }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < G; i++)
#pragma unroll
      for (int t = 0; t < NT; t++) {
        const float4 a0 = xa[i][t][0], a1 = xa[i][t][1];
        const float xv[8] = {a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w};
#pragma unroll
        for (int j = 0; j < 8; j++) acc[t] = mfma_f32(HT::f(wv[i][j]), xv[j], acc[t]);
      }
  };
  int base = kbeg;
  for (; base + 4 * 32 <= kend; base += 4 * 32) group(base, std::integral_constant<int, 4>{});
  if (base + 2 * 32 <= kend) {
    group(base, std::integral_constant<int, 2>{});
    base += 2 * 32;
  }
  if (base < kend) group(base, std::integral_constant<int, 1>{});
#pragma unroll
  for (int t = 0; t < NT; t++) red[w][t][lane] = acc[t];
  __syncthreads();
  if (w == 0) {
#pragma unroll
    for (int t = 0; t < NT; t++) {
      f32x4 s = red[0][t][lane];
#pragma unroll
      for (int v = 1; v < WV; v++) s += red[v][t][lane];
      // s[i] = sum for sequence b, weight row blockIdx.x*16 + 4g + i
      const int b = (blockIdx.z * NT + t) * 16 + r;
      const long n = (long)blockIdx.x * 16 + g * 4;
      if (GATE) {
        // lanes g = 0, 1 hold h1 of gate outputs j0 + 4g + i; lanes g + 2 hold their h3
        f32x4 h3;
#pragma unroll
        for (int i = 0; i < 4; i++) h3[i] = __shfl(s[i], (lane + 32) & 63, 64);
        if (g < 2 && b < B) {
          float4 o;
          float *op = &o.x;
#pragma unroll
          for (int i = 0; i < 4; i++) op[i] = s[i] * (1.f / (1.f + expf(-s[i]))) * h3[i];
          const long j = (long)blockIdx.x * 8 + g * 4;
          *(float4 *)(out + b * ldo + j) = o;
          put3(out3, gate_n, b, j, o);
        }
      } else if (ws) {
        *(f32x4 *)(ws + ((long)blockIdx.y * Bp + b) * N + n) = s;
      } else if (b < B) {
        float4 o = make_float4(alpha * s[0], alpha * s[1], alpha * s[2], alpha * s[3]);
        if (resid) {
          const float4 q = *(const float4 *)(resid + b * ldo + n);
          o.x += q.x; o.y += q.y; o.z += q.z; o.w += q.w;
        }
        *(float4 *)(out + b * ldo + n) = o;
      }
    }
  }
}

// ------------------------------------------- GEMV, batch 5..32, bf16 weights, exact ----

enum { BF3_WS = 0, BF3_GATE = 1, BF3_PLAIN = 2 };

// Products of bf16 weight rows W [N, K] with fp32 x rows [Bp, K] (row stride ldx) on
// v_mfma_f32_16x16x32_bf16: each x value comes as three bf16 parts (split3) in
// fragment order (part_at), written by the kernel that made the value, and every weight fragment
// meets the three, so the sums are of the exact products (fp32 accumulation,
// as the fp32-MFMA GEMV).  A block has 4 * NTW waves: wave w takes batch tile w / 4 (16
// sequences) and K slice w % 4 of the block's K range (KS steps of 32), holds that slice of x
// as bf16 parts in registers for all its RT row tiles of 16 weight rows, and the four K
// slices are summed in LDS in slice order.  x is read once per block for RT * 16 rows
// (the 16-row fp32-MFMA GEMV reads it once per 16 rows, 4x its weight bytes at batch 32).
//  BF3_WS:    split blockIdx.y's sums to ws slice [blockIdx.y][Bp, N] (every sequence row);
//  BF3_GATE:  W = [W1; W3] (gate_n rows each), one split: row tiles 0..RT/2-1 are W1 rows
//             j0 + 16 rt.., the rest the same rows of W3; writes out[b, j] = silu(h1) * h3
//             (generate.py:190) for b < B;
//  BF3_PLAIN: one split, out[b, n] = sums for b < B (the LM head's logits).
// blockIdx.z takes the x rows 16 * NTW * z .. (a prompt chunk has more than 16 * NTW).
template <int NTW, int RT, int KS, int MODE>
__global__ __launch_bounds__(NTW * 256) void gemv_bf3_kernel(const h16_t *__restrict__ W, long ldw,
                                                             const h16_t *__restrict__ x, int K,
                                                             float *__restrict__ out, long ldo, int N, int B,
                                                             int Bp, long gate_n, h16_t *__restrict__ out3) {
  __shared__ f32x4 red[3][NTW][RT][64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int ksl = w & 3, t = w >> 2;
  const int r16 = lane & 15, g = lane >> 4;
  const int kb = (blockIdx.y * 4 + ksl) * KS * 32 + g * 8;  // this lane's k in step 0
  constexpr int HALF = RT / 2;
  auto wrow = [&](int rt) -> long {
    if constexpr (MODE == BF3_GATE) {
      const long j = (long)blockIdx.x * 16 * HALF + (rt % HALF) * 16 + r16;
      return rt < HALF ? j : gate_n + j;
    } else {
      return (long)blockIdx.x * 16 * RT + rt * 16 + r16;
    }
  };
  // Ordinary loads: a load takes 64 bytes of each of 16 rows, and a non-temporal one did not keep the
  // line for the load of its other half (96 positions at batch 32: 112.3 ms non-temporal, 103.0).
  // The weight stream first: PF row tiles of the wave in flight (all of them up to 16 fragments).
  // The scheduling barriers keep the loads where they are written: left to itself the compiler
  // moved them down to their uses (48 VGPRs for 16 fragments and the x parts).  With the x parts in
  // fragment order: the W1|W3 launch of Qwen3-0.6B at batch 32 9.6 -> 8.6 us at best, 96 positions
  // 115.6 -> 112.2 ms (116.1 without the barriers).
  constexpr int PF = RT * KS <= 16 ? RT : 3;
  u16x8 wf[PF][KS];
  auto wload = [&](int slot, int rt) {
    const h16_t *wr = W + wrow(rt) * ldw + kb;
#pragma unroll
    for (int ks = 0; ks < KS; ks++) wf[slot][ks] = *(const u16x8 *)(wr + ks * 32);
  };
#pragma unroll
  for (int rt = 0; rt < PF; rt++) wload(rt, rt);
  const int b = (blockIdx.z * NTW + t) * 16 + r16;
  u16x8 xh[KS], xm[KS], xl[KS];
  {
    const h16_t *xr = x + ((long)(blockIdx.z * NTW + t) * (K >> 5) + (blockIdx.y * 4 + ksl) * KS) * 1536 + lane * 8;
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
      xh[ks] = *(const u16x8 *)(xr + ks * 1536);
      xm[ks] = *(const u16x8 *)(xr + ks * 1536 + 512);
      xl[ks] = *(const u16x8 *)(xr + ks * 1536 + 1024);
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  f32x4 acc[RT];
#pragma unroll
  for (int rt = 0; rt < RT; rt++) {
    acc[rt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
      const bf16x8 a = H16B::op(wf[rt % PF][ks]);
      acc[rt] = H16B::mfma16(a, H16B::op(xh[ks]), acc[rt]);
      acc[rt] = H16B::mfma16(a, H16B::op(xm[ks]), acc[rt]);
      acc[rt] = H16B::mfma16(a, H16B::op(xl[ks]), acc[rt]);
    }
    if constexpr (PF < RT) {
      if (rt + PF < RT) wload(rt % PF, rt + PF);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  // acc[rt][i] = sum over this K slice for weight row (tile rt) 4g + i, sequence b
  if (ksl > 0) {
#pragma unroll
    for (int rt = 0; rt < RT; rt++) red[ksl - 1][t][rt][lane] = acc[rt];
  }
  __syncthreads();
  if (ksl != 0) return;
#pragma unroll
  for (int rt = 0; rt < RT; rt++) {
#pragma unroll
    for (int q = 0; q < 3; q++) acc[rt] += red[q][t][rt][lane];
  }
  if constexpr (MODE == BF3_WS) {
#pragma unroll
    for (int rt = 0; rt < RT; rt++) {
      const long n = (long)blockIdx.x * 16 * RT + rt * 16 + g * 4;
      *(f32x4 *)(out + ((long)blockIdx.y * Bp + b) * N + n) = acc[rt];
    }
  } else if constexpr (MODE == BF3_GATE) {
    if (b < B) {
#pragma unroll
      for (int rt = 0; rt < HALF; rt++) {
        float4 o;
        float *op = &o.x;
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const float h1 = acc[rt][i], h3 = acc[rt + HALF][i];
          op[i] = h1 * (1.f / (1.f + expf(-h1))) * h3;
        }
        const long j = (long)blockIdx.x * 16 * HALF + rt * 16 + g * 4;
        *(float4 *)(out + (long)b * ldo + j) = o;
        put3(out3, gate_n, b, j, o);
      }
    }
  } else {
    if (b < B) {
#pragma unroll
      for (int rt = 0; rt < RT; rt++)
        *(f32x4 *)(out + (long)b * ldo + (long)blockIdx.x * 16 * RT + rt * 16 + g * 4) = acc[rt];
    }
  }
}

// One block per sequence b: out[b, :] = alpha * (ordered sum of the split-K partials, split 0
// first) + resid[b, :], and (gn != null) xn[b, :] = out[b, :] / rms * gn, the RMSNorm of the
// new row (generate.py:81-84, rms = sqrt(mean(out^2) + eps)) that the next GEMV reads.
// KS > 0 (the split count, rows of at most 1024): every partial and residual load of a thread
// is issued before the first add.
template <int KS>
__global__ __launch_bounds__(256) void gemv_reduce_rows_kernel(const float *__restrict__ ws, int ksplit, int Bp, int N,
                                                               float *out, long ldo, const float *resid, float alpha,
                                                               const float *gn, float *xn, float eps, h16_t *xn3) {
  __shared__ float red[4];
  const int b = blockIdx.x, tid = threadIdx.x;
  float ss = 0.f;
  float rv[4];  // KS path: the thread's residual inputs, then its outputs
  if constexpr (KS > 0) {
    float v[4 * (KS > 0 ? KS : 1)];
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const int n = min(tid + 256 * e, N - 1);  // rows shorter than 1024: clamped, unused
#pragma unroll
      for (int z = 0; z < KS; z++) v[e * KS + z] = ws[((long)z * Bp + b) * N + n];
      rv[e] = resid ? resid[(long)b * ldo + n] : 0.f;
    }
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const int n = tid + 256 * e;
      if (n < N) {
        float s = 0.f;
#pragma unroll
        for (int z = 0; z < KS; z++) s += v[e * KS + z];
        float o = alpha * s;
        if (resid) o += rv[e];
        out[(long)b * ldo + n] = o;
        ss += o * o;
        rv[e] = o;
      }
    }
  } else {
    for (int n = tid; n < N; n += 256) {
      float s = 0.f;
      for (int z = 0; z < ksplit; z++) s += ws[((long)z * Bp + b) * N + n];
      float o = alpha * s;
      if (resid) o += resid[(long)b * ldo + n];
      out[(long)b * ldo + n] = o;
      ss += o * o;
    }
  }
  if (!gn) return;
  ss = wave_sum(ss);
  if ((tid & 63) == 0) red[tid >> 6] = ss;
  __syncthreads();
  const float rms = sqrtf((red[0] + red[1] + red[2] + red[3]) / (float)N + eps);
  if constexpr (KS > 0) {
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const int n = tid + 256 * e;
      if (n < N) {
        const float v = rv[e] / rms * gn[n];
        xn[(long)b * N + n] = v;
        put3(xn3, N, b, n, v);
      }
    }
  } else {  // read back what this thread wrote
    for (int n = tid; n < N; n += 256) {
      const float v = out[(long)b * ldo + n] / rms * gn[n];
      xn[(long)b * N + n] = v;
      put3(xn3, N, b, n, v);
    }
  }
}

// ------------------------------------------------------------- elementwise / attention ----

// Token of this position (prompt id while pos < P, else the last sampled id) and its
// embedding row.  One block per sequence.
template <typename HT>
__global__ void dec_token_kernel(const int32_t *__restrict__ prompt, int ctx, const DecState *__restrict__ st,
                                 int32_t *tok, const h16_t *__restrict__ E, float *x, int D, int B,
                                 const float *__restrict__ gn, float *xn, float eps, h16_t *xn3) {
  __shared__ float red[4];
  const int b = blockIdx.x;
  const int pos = st->pos;
  const int t = pos < st->P ? prompt[(long)b * ctx + pos] : tok[b];
  float ss = 0.f;
  for (int i = threadIdx.x; i < D; i += blockDim.x) {
    const float v = b < B ? HT::f(E[(long)t * D + i]) : 0.f;
    x[(long)b * D + i] = v;
    ss += v * v;
  }
  ss = wave_sum(ss);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
  __syncthreads();
  if (threadIdx.x == 0) tok[b] = t;
  if (gn) {  // the RMSNorm of the row (generate.py:81-84), read by the batch-5..32 QKV GEMV
    const float rms = sqrtf((red[0] + red[1] + red[2] + red[3]) / (float)D + eps);
    for (int i = threadIdx.x; i < D; i += blockDim.x) {
      const float v = x[(long)b * D + i] / rms * gn[i];
      xn[(long)b * D + i] = v;
      put3(xn3, D, b, i, v);
    }
  }
}

// KCOL (batch <= 4, one block per KV head): the K cache holds float4 d4 of position t at
// K4[d4 * ctx + t], so that the score loop's lanes (one position each) read consecutive 16-byte
// pieces; else row-major like V ([ctx][HD]), which measured faster at batch 32.
// PRE: row blockIdx.x of a prompt chunk (sequence row / nc, position p0 + row % nc), whose keys
// and values pre_append_kernel has put into the cache; otherwise row = sequence, the position is
// the state's, and its key and value are appended here.
template <int HD, int RATIO, bool KCOL, bool PRE>
__global__ __launch_bounds__(256) void dec_attn_kernel(const float *__restrict__ qkv, int QKV,
                                                       const float *__restrict__ gq, const float *__restrict__ gk,
                                                       const float *__restrict__ cosb, const float *__restrict__ sinb,
                                                       float *kc, float *vc, float *att, int NH, int NKV, int ctx,
                                                       const DecState *__restrict__ st, float eps, double scale,
                                                       const float *__restrict__ qws, int qnz, int Bp, int p0,
                                                       int nc, h16_t *att3) {
  extern __shared__ float sc[];  // [RATIO][ctx]
  constexpr int C4 = HD / 4, NG = 256 / C4, HALF = HD / 2;
  __shared__ float4 qs[RATIO][C4];
  __shared__ float4 vn[C4];
  __shared__ float4 part[NG][RATIO][C4];
  __shared__ float red[RATIO][8];
  // block y: query heads qh0 .. qh0 + RATIO - 1 of KV head kvh (RATIO may be a part of the
  // model's NH / NKV query heads per KV head: the blocks of one KV head then append the same
  // K and V values)
  const int ri = blockIdx.x, b = PRE ? ri / nc : ri;
  const int qh0 = blockIdx.y * RATIO, kvh = qh0 / (NH / NKV), tid = threadIdx.x;
  const int pos = PRE ? p0 + ri % nc : st->pos, npos = pos + 1;
  float *K = kc + ((long)b * NKV + kvh) * ctx * HD;
  float *V = vc + ((long)b * NKV + kvh) * ctx * HD;
  const float *row = qkv + (long)ri * QKV;
  // element col of this sequence's q|k|v row: the row itself, or (qnz > 1) the ordered sum of
  // the QKV GEMV's split-K partial slices [qnz][Bp, QKV]
  auto qval = [&](int col) -> float {
    if (qnz <= 1) return row[col];
    float s = 0.f;
    for (int z = 0; z < qnz; z++) s += qws[((long)z * Bp + ri) * QKV + col];
    return s;
  };
  // slots 0..RATIO-1: q heads qh0 + slot; RATIO: k head kvh; RATIO+1: v head kvh
  for (int i = tid; i < (PRE ? RATIO : RATIO + 2) * HALF; i += 256) {
    const int slot = i / HALF, p = i % HALF;
    float *q2 = (float *)qs, *v2 = (float *)vn;
    if (slot == RATIO + 1) {
      const int c0 = (NH + NKV) * HD + kvh * HD;
      const float y0 = qval(c0 + 2 * p), y1 = qval(c0 + 2 * p + 1);
      v2[2 * p] = y0; v2[2 * p + 1] = y1;
      V[(long)pos * HD + 2 * p] = y0;
      V[(long)pos * HD + 2 * p + 1] = y1;
      continue;
    }
    const bool isq = slot < RATIO;
    const int c0 = isq ? (qh0 + slot) * HD : NH * HD + kvh * HD;
    float x0 = qval(c0 + 2 * p), x1 = qval(c0 + 2 * p + 1);
    const float *gg = isq ? gq : gk;
    if (gg) {  // uniform per block: every lane of the slot's (half-)wave takes part
      float ss = x0 * x0 + x1 * x1;
      ss = HALF == 64 ? wave_sum(ss) : half_wave_sum(ss);
      const float rms = sqrtf(ss / (float)HD + eps);
      x0 = x0 / rms * gg[2 * p];
      x1 = x1 / rms * gg[2 * p + 1];
    }
    const float c = cosb[pos * HALF + p], s = sinb[pos * HALF + p];
    const float y0 = x0 * c - x1 * s, y1 = x0 * s + x1 * c;
    if (isq) {
      q2[slot * HD + 2 * p] = y0;
      q2[slot * HD + 2 * p + 1] = y1;
    } else {
      if (KCOL) {
        *(float2 *)(K + ((long)(p >> 1) * ctx + pos) * 4 + 2 * (p & 1)) = make_float2(y0, y1);
      } else {
        K[(long)pos * HD + 2 * p] = y0;
        K[(long)pos * HD + 2 * p + 1] = y1;
      }
    }
  }
  __syncthreads();
  float mx[RATIO];
#pragma unroll
  for (int r = 0; r < RATIO; r++) mx[r] = -INFINITY;
  const float4 *K4 = (const float4 *)K;
  for (int t = tid; t < npos; t += 256) {
    // position pos was written by this block above; the barrier made it visible
    float s[RATIO];
#pragma unroll
    for (int r = 0; r < RATIO; r++) s[r] = 0.f;
#pragma unroll 8
    for (int d4 = 0; d4 < C4; d4++) {
      const float4 kv = KCOL ? K4[(long)d4 * ctx + t] : K4[(long)t * C4 + d4];
#pragma unroll
      for (int r = 0; r < RATIO; r++) {
        const float4 qv = qs[r][d4];
        s[r] += qv.x * kv.x + qv.y * kv.y + qv.z * kv.z + qv.w * kv.w;
      }
    }
#pragma unroll
    for (int r = 0; r < RATIO; r++) {
      const float v = (float)((double)s[r] * scale);
      sc[r * ctx + t] = v;
      mx[r] = fmaxf(mx[r], v);
    }
  }
#pragma unroll
  for (int r = 0; r < RATIO; r++) {
    mx[r] = wave_max(mx[r]);
    if ((tid & 63) == 0) red[r][tid >> 6] = mx[r];
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < RATIO; r++) mx[r] = fmaxf(fmaxf(red[r][0], red[r][1]), fmaxf(red[r][2], red[r][3]));
  float sum[RATIO];
#pragma unroll
  for (int r = 0; r < RATIO; r++) sum[r] = 0.f;
  for (int t = tid; t < npos; t += 256)
#pragma unroll
    for (int r = 0; r < RATIO; r++) {
      const float e = __expf(sc[r * ctx + t] - mx[r]);
      sc[r * ctx + t] = e;
      sum[r] += e;
    }
#pragma unroll
  for (int r = 0; r < RATIO; r++) {
    sum[r] = wave_sum(sum[r]);
    if ((tid & 63) == 0) red[r][4 + (tid >> 6)] = sum[r];
  }
  __syncthreads();
  const int c = tid % C4, grp = tid / C4;
  float4 acc[RATIO];
#pragma unroll
  for (int r = 0; r < RATIO; r++) acc[r] = make_float4(0.f, 0.f, 0.f, 0.f);
  // four positions per iteration: their V loads are in flight together
  int t = grp;
  for (; t + 3 * NG < npos; t += 4 * NG) {
    float4 v[4];
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const int tu = t + u * NG;
      v[u] = !PRE && tu == pos ? vn[c] : *(const float4 *)(V + (long)tu * HD + c * 4);
    }
#pragma unroll
    for (int u = 0; u < 4; u++)
#pragma unroll
      for (int r = 0; r < RATIO; r++) {
        const float p = sc[r * ctx + t + u * NG];
        acc[r].x += p * v[u].x; acc[r].y += p * v[u].y; acc[r].z += p * v[u].z; acc[r].w += p * v[u].w;
      }
  }
  for (; t < npos; t += NG) {
    const float4 v = !PRE && t == pos ? vn[c] : *(const float4 *)(V + (long)t * HD + c * 4);
#pragma unroll
    for (int r = 0; r < RATIO; r++) {
      const float p = sc[r * ctx + t];
      acc[r].x += p * v.x; acc[r].y += p * v.y; acc[r].z += p * v.z; acc[r].w += p * v.w;
    }
  }
#pragma unroll
  for (int r = 0; r < RATIO; r++) part[grp][r][c] = acc[r];
  __syncthreads();
  if (grp < RATIO) {
    const int r = grp;
    const float inv = 1.f / (red[r][4] + red[r][5] + red[r][6] + red[r][7]);
    float4 o = part[0][r][c];
    for (int gi = 1; gi < NG; gi++) {
      const float4 p = part[gi][r][c];
      o.x += p.x; o.y += p.y; o.z += p.z; o.w += p.w;
    }
    o.x *= inv; o.y *= inv; o.z *= inv; o.w *= inv;
    const long k = (long)(qh0 + r) * HD + c * 4;
    *(float4 *)(att + (long)ri * NH * HD + k) = o;
    put3(att3, NH * HD, ri, k, o);
  }
}

// Tokens and embedding rows of a prompt chunk (row i: sequence i / nc, position p0 + i % nc),
// and their RMSNorm with the first gain.  One block per row.
template <typename HT>
__global__ __launch_bounds__(256) void pre_token_kernel(const int32_t *__restrict__ prompt, int ctx, int p0, int nc,
                                                        const h16_t *__restrict__ E, float *x, int D,
                                                        const float *__restrict__ gn, float *xn, float eps, h16_t *xn3) {
  __shared__ float red[4];
  const long i = blockIdx.x;
  const int t = prompt[(i / nc) * ctx + p0 + i % nc];
  float ss = 0.f;
  for (int k = threadIdx.x; k < D; k += 256) {
    const float v = HT::f(E[(long)t * D + k]);
    x[i * D + k] = v;
    ss += v * v;
  }
  ss = wave_sum(ss);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
  __syncthreads();
  const float rms = sqrtf((red[0] + red[1] + red[2] + red[3]) / (float)D + eps);
  for (int k = threadIdx.x; k < D; k += 256) {
    const float v = x[i * D + k] / rms * gn[k];
    xn[i * D + k] = v;
    put3(xn3, D, i, k, v);
  }
}

// Keys (QK-norm, RoPE) and values of a prompt chunk into the cache, from the qnz split-K slices
// [Rp, QKV] of the QKV rows.  Block (row, KV head): HD / 2 threads for the key's pairs, as many for
// the value's.
template <int HD, bool KCOL>
__global__ __launch_bounds__(HD) void pre_append_kernel(const float *__restrict__ qws, int qnz, int Rp, int QKV,
                                                        const float *__restrict__ gk, const float *__restrict__ cosb,
                                                        const float *__restrict__ sinb, float *kc, float *vc, int NH,
                                                        int NKV, int ctx, int p0, int nc, float eps) {
  constexpr int HALF = HD / 2;
  const int ri = blockIdx.x, kvh = blockIdx.y, b = ri / nc, pos = p0 + ri % nc;
  const bool isv = threadIdx.x >= HALF;
  const int p = threadIdx.x % HALF, col = (NH + (isv ? NKV : 0) + kvh) * HD + 2 * p;
  const long cache = ((long)b * NKV + kvh) * ctx * HD;
  float x0 = 0.f, x1 = 0.f;
  for (int z = 0; z < qnz; z++) {
    const float2 v = *(const float2 *)(qws + ((long)z * Rp + ri) * QKV + col);
    x0 += v.x;
    x1 += v.y;
  }
  float ss = x0 * x0 + x1 * x1;
  ss = HALF == 64 ? wave_sum(ss) : half_wave_sum(ss);
  if (isv) {
    *(float2 *)(vc + cache + (long)pos * HD + 2 * p) = make_float2(x0, x1);
    return;
  }
  if (gk) {
    const float rms = sqrtf(ss / (float)HD + eps);
    x0 = x0 / rms * gk[2 * p];
    x1 = x1 / rms * gk[2 * p + 1];
  }
  const float c = cosb[pos * HALF + p], s = sinb[pos * HALF + p];
  const float2 y = make_float2(x0 * c - x1 * s, x0 * s + x1 * c);
  if (KCOL) *(float2 *)(kc + cache + ((long)(p >> 1) * ctx + pos) * 4 + 2 * (p & 1)) = y;
  else *(float2 *)(kc + cache + (long)pos * HD + 2 * p) = y;
}

__device__ __forceinline__ int gen_step(const DecState *st) { return st->pos - (st->P - 1); }

// Greedy from per-block partials: first index of the maximum logit (np.argmax).  One block
// (1024 threads) per sequence.
__global__ __launch_bounds__(1024) void dec_argmax_kernel(const float *__restrict__ amv, const int32_t *__restrict__ ami,
                                                          int nblk, const DecState *__restrict__ st, int ctx,
                                                          int32_t *tok, int32_t *out) {
  __shared__ float rv[16];
  __shared__ int ri[16];
  const int b = blockIdx.x, tid = threadIdx.x;
  float best = -INFINITY;
  int bi = 0x7fffffff;
  for (int i = tid; i < nblk; i += 1024) {
    const float v = amv[(long)b * nblk + i];
    const int j = ami[(long)b * nblk + i];
    if (v > best || (v == best && j < bi)) { best = v; bi = j; }
  }
  for (int o = 32; o > 0; o >>= 1) {
    const float ov = __shfl_xor(best, o, 64);
    const int oi = __shfl_xor(bi, o, 64);
    if (ov > best || (ov == best && oi < bi)) { best = ov; bi = oi; }
  }
  if ((tid & 63) == 0) { rv[tid >> 6] = best; ri[tid >> 6] = bi; }
  __syncthreads();
  if (tid == 0) {
    best = rv[0]; bi = ri[0];
    for (int w = 1; w < 16; w++)
      if (rv[w] > best || (rv[w] == best && ri[w] < bi)) { best = rv[w]; bi = ri[w]; }
    // no logit above -inf (all NaN or -inf): token 0, so the next lookup stays in the table
    if (bi == 0x7fffffff) bi = 0;
    tok[b] = bi;
    out[(long)b * ctx + gen_step(st)] = bi;
  }
}

// Greedy over full logits rows (batch > 4): per-block partials of 4096-wide chunks.
__global__ __launch_bounds__(256) void dec_argmax_part_kernel(const float *__restrict__ logits, int V, int nblk,
                                                              float *amv, int32_t *ami) {
  __shared__ float rv[4];
  __shared__ int ri[4];
  const int b = blockIdx.y, tid = threadIdx.x;
  const int chunk = (V + nblk - 1) / nblk;
  const int i0 = blockIdx.x * chunk, i1 = min(V, i0 + chunk);
  float best = -INFINITY;
  int bi = 0x7fffffff;
  for (int i = i0 + tid; i < i1; i += 256) {
    const float v = logits[(long)b * V + i];
    if (v > best) { best = v; bi = i; }
  }
  for (int o = 32; o > 0; o >>= 1) {
    const float ov = __shfl_xor(best, o, 64);
    const int oi = __shfl_xor(bi, o, 64);
    if (ov > best || (ov == best && oi < bi)) { best = ov; bi = oi; }
  }
  if ((tid & 63) == 0) { rv[tid >> 6] = best; ri[tid >> 6] = bi; }
  __syncthreads();
  if (tid == 0) {
    best = rv[0]; bi = ri[0];
    for (int w = 1; w < 4; w++)
      if (rv[w] > best || (rv[w] == best && ri[w] < bi)) { best = rv[w]; bi = ri[w]; }
    amv[(long)b * nblk + blockIdx.x] = best;
    ami[(long)b * nblk + blockIdx.x] = bi;
  }
}

// ------------------------------------------------------------------------- sampling ----
//
// p = softmax(logits / T) in fp32, an optional top-p mask, then the first index whose cumulative
// mass exceeds u * total (np.random.choice: cdf.searchsorted(u, side='right')).  A sequence's
// row of V logits is cut into SampArgs::G contiguous chunks, one block each, and the row passes
// through a chain of kernels over them; what a kernel needs of the whole row (max, sum, masses)
// every block of the next one reduces again from the G partials, in order.  As one block per
// sequence (1024 threads, about 36 passes over the row, 31 of them the bisection for the top-p
// threshold) a sample of 151,936 logits took 747 us at batch 1; the chain takes 34 us (seven launches of 4-6 us: latency).
//
// Masses are sums of fixed-point values, p * 2^62 as an integer (p <= 1; exact for p >= 2^-38,
// smaller ones are off by less than 2^-62 each, and every p above 0 counts at least one unit, so that
// a uniform of 0 picks the first of them): integer sums do not depend on the order of the atomics
// that form them, so the same logits and uniform always give the same token.

struct SampArgs {
  float *logits;              // [B][V]: logits, then exp(x - max), then p
  int V, G, chunk;            // chunk: columns per block (a multiple of 4); G * chunk >= V
  const DecState *st;
  const double *unif;         // [B][ctx]
  int ctx;
  int32_t *tok, *out;
  float *pmax;                // [B][G]
  double *psum;               // [B][G]
  unsigned long long *hist;   // [B][3][SAMP_BINS] mass per bin of p's bit pattern
  unsigned long long *mass;   // [B][G] kept mass per chunk
  uint32_t *pre;              // [B][2] threshold bits found so far (levels 1, 2)
  unsigned long long *above;  // [B][2] mass above that prefix
  bool topp;
};

constexpr int SAMP_NT = 256, SAMP_BINS = 1024;  // 10 bits of the pattern per level
constexpr int SAMP_G = 128;                     // chunks per row at most: half the CUs at batch 1
constexpr int SAMP_SHORT = 2048;                // longest row that one block samples
constexpr double SAMP_ONE = 4611686018427387904.0;  // 2^62
constexpr uint32_t SAMP_P1 = 0x3f800000u;       // the bits of p = 1, the largest

__device__ __forceinline__ unsigned long long samp_mass(float p) {
  if (!(p > 0.f)) return 0ull;  // also NaN
  const unsigned long long m = (unsigned long long)((double)p * SAMP_ONE);
  return m ? m : 1ull;
}

template <typename T>
__device__ __forceinline__ T samp_wave_sum(T v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}
// Sum over the block, the same in every thread, waves in order (red: SAMP_NT / 64 slots).
template <typename T>
__device__ __forceinline__ T samp_block_sum(T v, T *red) {
  v = samp_wave_sum(v);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  T s = red[0];
#pragma unroll
  for (int i = 1; i < SAMP_NT / 64; i++) s += red[i];
  return s;
}

// Inclusive prefix sum over the block's threads; *total receives the block's sum.
__device__ __forceinline__ unsigned long long samp_block_scan(unsigned long long v, unsigned long long *red,
                                                              unsigned long long *total) {
  for (int o = 1; o < 64; o <<= 1) {
    const unsigned long long n = __shfl_up(v, o, 64);
    if ((int)(threadIdx.x & 63) >= o) v += n;
  }
  if ((threadIdx.x & 63) == 63) red[threadIdx.x >> 6] = v;
  __syncthreads();
  unsigned long long before = 0, t = 0;
#pragma unroll
  for (int i = 0; i < SAMP_NT / 64; i++) {
    if (i < (int)(threadIdx.x >> 6)) before += red[i];
    t += red[i];
  }
  *total = t;
  return before + v;
}

// 1. The chunk's max of x = logit / T, and this position's empty histograms.
__device__ __forceinline__ void samp_max(const SampArgs &a, int b, int g) {
  __shared__ float red[SAMP_NT / 64];
  const int tid = threadIdx.x;
  const float *lg = a.logits + (long)b * a.V;
  const int i1 = min(a.V, (g + 1) * a.chunk);
  float mx = -INFINITY;
  const float temp = a.st->temp;
  for (int i = g * a.chunk + tid * 4; i < i1; i += SAMP_NT * 4) {
    const float4 v = *(const float4 *)(lg + i);
    mx = fmaxf(fmaxf(fmaxf(mx, v.x / temp), v.y / temp), fmaxf(v.z / temp, v.w / temp));
  }
  if (a.topp)
    for (int i = g * SAMP_NT + tid; i < 3 * SAMP_BINS; i += gridDim.x * SAMP_NT) a.hist[(long)b * 3 * SAMP_BINS + i] = 0;
  mx = wave_max(mx);
  if ((tid & 63) == 0) red[tid >> 6] = mx;
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < SAMP_NT / 64; w++) mx = fmaxf(mx, red[w]);
    a.pmax[b * a.G + g] = mx;
  }
}
__global__ __launch_bounds__(SAMP_NT) void samp_max_kernel(SampArgs a) { samp_max(a, blockIdx.y, blockIdx.x); }

// 2. exp(x - max) in place, and its fp64 sum over the chunk (generate.py:87-90).
__device__ __forceinline__ void samp_exp(const SampArgs &a, int b, int g) {
  __shared__ float redm[SAMP_NT / 64];
  __shared__ double red[SAMP_NT / 64];
  const int tid = threadIdx.x;
  float *lg = a.logits + (long)b * a.V;
  const int i1 = min(a.V, (g + 1) * a.chunk);
  float mx = -INFINITY;
  for (int i = tid; i < a.G; i += SAMP_NT) mx = fmaxf(mx, a.pmax[b * a.G + i]);
  mx = wave_max(mx);
  if ((tid & 63) == 0) redm[tid >> 6] = mx;
  __syncthreads();
  for (int w = 0; w < SAMP_NT / 64; w++) mx = fmaxf(mx, redm[w]);
  const float temp = a.st->temp;
  double z = 0.0;
  for (int i = g * a.chunk + tid * 4; i < i1; i += SAMP_NT * 4) {
    float4 v = *(const float4 *)(lg + i);
    v.x = expf(v.x / temp - mx); v.y = expf(v.y / temp - mx);
    v.z = expf(v.z / temp - mx); v.w = expf(v.w / temp - mx);
    *(float4 *)(lg + i) = v;
    z += (double)v.x; z += (double)v.y; z += (double)v.z; z += (double)v.w;
  }
  z = samp_block_sum(z, red);
  if (tid == 0) a.psum[b * a.G + g] = z;
}
__global__ __launch_bounds__(SAMP_NT) void samp_exp_kernel(SampArgs a) { samp_exp(a, blockIdx.y, blockIdx.x); }

// The largest bin k whose suffix mass (base + bins k.. of `hist`) reaches top_p, and the suffix mass
// above it; k = 0 when none does.  256 threads, 4 bins each; the same result in every thread.
__device__ __forceinline__ void samp_select(const unsigned long long *hist, unsigned long long base, float top_p,
                                            uint32_t &k, unsigned long long &above) {
  __shared__ unsigned long long red[SAMP_NT / 64], s_above;
  __shared__ uint32_t s_k;
  const int tid = threadIdx.x;
  unsigned long long h[4], own = 0;
#pragma unroll
  for (int e = 0; e < 4; e++) own += h[e] = hist[4 * tid + e];
  if (tid == 0) s_k = 0;
  unsigned long long total;
  const unsigned long long incl = samp_block_scan(own, red, &total);
  unsigned long long up = base + (total - incl);  // mass above this thread's bins
  if (tid == 0) s_above = up + h[3] + h[2] + h[1];
  __syncthreads();
  // suffix masses fall with k: the one bin where the mass first reaches top_p from above
#pragma unroll
  for (int e = 3; e >= 0; e--) {
    const unsigned long long at = up + h[e];
    const bool top = tid == SAMP_NT - 1 && e == 3;
    if ((double)at / SAMP_ONE >= (double)top_p && (top || !((double)up / SAMP_ONE >= (double)top_p))) {
      s_k = 4 * tid + e;
      s_above = up;
    }
    up = at;
  }
  __syncthreads();
  k = s_k;
  above = s_above;
  __syncthreads();
}

// Bin of p at level LV (1: bits 20.., 2: bits 10..19, 3: bits 0..9), or -1 if p's higher bits are not
// the prefix chosen so far.
template <int LV>
__device__ __forceinline__ int samp_bin(float p, uint32_t prefix) {
  const uint32_t u = __float_as_uint(p);
  if (LV == 1) return (int)(u >> 20);
  if (LV == 2) return u >> 20 == prefix ? (int)((u >> 10) & 1023u) : -1;
  return u >> 10 == prefix ? (int)(u & 1023u) : -1;
}

// The block's histogram in LDS, its non-empty bins added to the row's.
template <int LV>
__device__ __forceinline__ void samp_hist_add(unsigned long long *lds, float p, uint32_t prefix) {
  if (!(p > 0.f)) return;
  const int k = samp_bin<LV>(p, prefix);
  if (k >= 0) atomicAdd(&lds[k], samp_mass(p));
}
__device__ __forceinline__ void samp_hist_out(const unsigned long long *lds, unsigned long long *out) {
  __syncthreads();
  for (int i = threadIdx.x; i < SAMP_BINS; i += SAMP_NT)
    if (lds[i]) atomicAdd(out + i, lds[i]);
}

// 3. p = exp / Z in place; with top-p the first histogram level (8 bins per octave), without it the
// chunk's mass.
__device__ __forceinline__ void samp_prob(const SampArgs &a, int b, int g) {
  __shared__ double red[SAMP_NT / 64];
  __shared__ unsigned long long redm[SAMP_NT / 64];
  __shared__ unsigned long long lds[SAMP_BINS];
  const int tid = threadIdx.x;
  float *lg = a.logits + (long)b * a.V;
  const int i1 = min(a.V, (g + 1) * a.chunk);
  double z = 0.0;
  for (int i = tid; i < a.G; i += SAMP_NT) z += a.psum[b * a.G + i];
  if (a.topp)
    for (int i = tid; i < SAMP_BINS; i += SAMP_NT) lds[i] = 0;
  const float Z = (float)samp_block_sum(z, red);
  unsigned long long m = 0;
  for (int i = g * a.chunk + tid * 4; i < i1; i += SAMP_NT * 4) {
    float4 v = *(const float4 *)(lg + i);
    v.x /= Z; v.y /= Z; v.z /= Z; v.w /= Z;
    *(float4 *)(lg + i) = v;
    if (a.topp) {
      samp_hist_add<1>(lds, v.x, 0); samp_hist_add<1>(lds, v.y, 0);
      samp_hist_add<1>(lds, v.z, 0); samp_hist_add<1>(lds, v.w, 0);
    } else {
      m += samp_mass(v.x) + samp_mass(v.y) + samp_mass(v.z) + samp_mass(v.w);
    }
  }
  if (a.topp) {
    samp_hist_out(lds, a.hist + (long)b * 3 * SAMP_BINS);
  } else {
    m = samp_block_sum(m, redm);
    if (tid == 0) a.mass[b * a.G + g] = m;
  }
}
__global__ __launch_bounds__(SAMP_NT) void samp_prob_kernel(SampArgs a) { samp_prob(a, blockIdx.y, blockIdx.x); }

// 4, 5. Histogram level LV (2, 3) among the values in the bin that level LV - 1 selects.
template <int LV>
__global__ __launch_bounds__(SAMP_NT) void samp_hist_kernel(SampArgs a) {
  __shared__ unsigned long long lds[SAMP_BINS];
  const int b = blockIdx.y, g = blockIdx.x, tid = threadIdx.x;
  const float *lg = a.logits + (long)b * a.V;
  const int i1 = min(a.V, (g + 1) * a.chunk);
  for (int i = tid; i < SAMP_BINS; i += SAMP_NT) lds[i] = 0;
  unsigned long long *hist = a.hist + (long)b * 3 * SAMP_BINS;
  uint32_t k;
  unsigned long long above;
  samp_select(hist + (LV - 2) * SAMP_BINS, LV == 2 ? 0ull : a.above[b * 2], a.st->top_p, k, above);
  const uint32_t prefix = LV == 2 ? k : (a.pre[b * 2] << 10) | k;
  if (g == 0 && tid == 0) {
    a.pre[b * 2 + LV - 2] = prefix;
    a.above[b * 2 + LV - 2] = above;
  }
  for (int i = g * a.chunk + tid * 4; i < i1; i += SAMP_NT * 4) {
    const float4 v = *(const float4 *)(lg + i);
    samp_hist_add<LV>(lds, v.x, prefix); samp_hist_add<LV>(lds, v.y, prefix);
    samp_hist_add<LV>(lds, v.z, prefix); samp_hist_add<LV>(lds, v.w, prefix);
  }
  samp_hist_out(lds, hist + (LV - 1) * SAMP_BINS);
}

// The top-p threshold: the largest probability v with mass(p >= v) >= top_p (generate.py:205-213), 0
// when even the whole row's mass stays below it.
__device__ __forceinline__ float samp_threshold(const SampArgs &a, int b) {
  uint32_t k;
  unsigned long long above;
  samp_select(a.hist + ((long)b * 3 + 2) * SAMP_BINS, a.above[b * 2 + 1], a.st->top_p, k, above);
  return __uint_as_float(min((a.pre[b * 2 + 1] << 10) | k, SAMP_P1));
}

// 6 (top-p). The chunk's mass of p >= threshold.
__global__ __launch_bounds__(SAMP_NT) void samp_mass_kernel(SampArgs a) {
  __shared__ unsigned long long red[SAMP_NT / 64];
  const int b = blockIdx.y, g = blockIdx.x, tid = threadIdx.x;
  const float *lg = a.logits + (long)b * a.V;
  const int i1 = min(a.V, (g + 1) * a.chunk);
  const float thr = samp_threshold(a, b);
  unsigned long long m = 0;
  for (int i = g * a.chunk + tid * 4; i < i1; i += SAMP_NT * 4) {
    const float4 v = *(const float4 *)(lg + i);
    m += (v.x >= thr ? samp_mass(v.x) : 0) + (v.y >= thr ? samp_mass(v.y) : 0) + (v.z >= thr ? samp_mass(v.z) : 0) +
         (v.w >= thr ? samp_mass(v.w) : 0);
  }
  m = samp_block_sum(m, red);
  if (tid == 0) a.mass[b * a.G + g] = m;
}

// 7. One block per sequence: the chunk whose cumulative mass passes u * total, then the index in it.
// Token 0 when nothing is kept (no finite probability).
__device__ __forceinline__ void samp_pick(const SampArgs &a, int b) {
  __shared__ unsigned long long red[SAMP_NT / 64], s_before;
  __shared__ int s_chunk, s_pick;
  const int tid = threadIdx.x;
  const float *lg = a.logits + (long)b * a.V;
  const float thr = a.topp ? samp_threshold(a, b) : 0.f;
  const int step = gen_step(a.st);
  static_assert(SAMP_G <= SAMP_NT, "one chunk mass per thread");
  const unsigned long long own = tid < a.G ? a.mass[b * a.G + tid] : 0ull;
  unsigned long long total;
  const unsigned long long incl = samp_block_scan(own, red, &total);
  if (tid == 0) {
    s_chunk = -1;
    s_pick = -1;
  }
  __syncthreads();
  const double u = a.unif[(long)b * a.ctx + step] * (double)total;
  // the first chunk that passes u; a uniform of 1 or more (no draw from [0, 1) rounds up to the total) takes
  // the last one that holds mass
  if (own && (double)incl > u && !((double)(incl - own) > u)) {
    s_chunk = tid;
    s_before = incl - own;
  }
  __syncthreads();
  const bool none = s_chunk < 0;
  __syncthreads();  // every wave has read s_chunk before one writes it again
  if (none && own && incl == total) {
    s_chunk = tid;
    s_before = incl - own;
  }
  __syncthreads();
  if (s_chunk >= 0) {
    const int c0 = s_chunk * a.chunk, c1 = min(a.V, c0 + a.chunk);
    const int per = (a.chunk + SAMP_NT - 1) / SAMP_NT;
    const int i0 = min(c1, c0 + tid * per), i1 = min(c1, i0 + per);
    unsigned long long m = 0, tot;
    for (int i = i0; i < i1; i++) m += lg[i] >= thr ? samp_mass(lg[i]) : 0ull;
    unsigned long long c = s_before + samp_block_scan(m, red, &tot) - m;
    if (m && (none ? c + m == s_before + tot : (double)(c + m) > u && !((double)c > u))) {
      int pick = -1;
      for (int i = i0; i < i1; i++) {
        const unsigned long long q = lg[i] >= thr ? samp_mass(lg[i]) : 0ull;
        if (!q) continue;
        pick = i;
        c += q;
        if (!none && (double)c > u) break;
      }
      s_pick = pick;
    }
  }
  __syncthreads();
  if (tid == 0) {
    const int pick = s_pick < 0 ? 0 : s_pick;
    a.tok[b] = pick;
    a.out[(long)b * a.ctx + step] = pick;
  }
}
__global__ __launch_bounds__(SAMP_NT) void samp_pick_kernel(SampArgs a) { samp_pick(a, blockIdx.x); }

// The same without a top-p mask in one launch, a block per row (one chunk), the same tokens: a short row's four
// launches of 4-6 us cost more than its passes by one block (a two-layer model, batch 1, 100 tokens: 512 columns
// 4.97 -> 4.68 ms, 2048 5.08 -> 4.88, 4096 5.12 and 5.31).
__global__ __launch_bounds__(SAMP_NT) void samp_short_kernel(SampArgs a) {
  const int b = blockIdx.x;
  samp_max(a, b, 0);
  __syncthreads();
  samp_exp(a, b, 0);
  __syncthreads();
  samp_prob(a, b, 0);
  __syncthreads();
  samp_pick(a, b);
}

int launch_sample(const SampArgs &a, int B, hipStream_t s) {
  const dim3 grid(a.G, B), block(SAMP_NT);
  if (!a.topp && a.V <= SAMP_SHORT) {
    SampArgs one = a;
    one.G = 1;
    one.chunk = a.V;
    hipLaunchKernelGGL(samp_short_kernel, dim3(B), block, 0, s, one);
    return ne_hip_status(hipGetLastError(), "decode sampling");
  }
  hipLaunchKernelGGL(samp_max_kernel, grid, block, 0, s, a);
  hipLaunchKernelGGL(samp_exp_kernel, grid, block, 0, s, a);
  hipLaunchKernelGGL(samp_prob_kernel, grid, block, 0, s, a);
  if (a.topp) {
    hipLaunchKernelGGL(samp_hist_kernel<2>, grid, block, 0, s, a);
    hipLaunchKernelGGL(samp_hist_kernel<3>, grid, block, 0, s, a);
    hipLaunchKernelGGL(samp_mass_kernel, grid, block, 0, s, a);
  }
  hipLaunchKernelGGL(samp_pick_kernel, dim3(B), block, 0, s, a);
  return ne_hip_status(hipGetLastError(), "decode sampling");
}

__global__ void dec_advance_kernel(DecState *st) {
  if (threadIdx.x == 0) st->pos += 1;
}

// ----------------------------------------------------------------------- launchers ----

int pick_rpw(int N) {
  for (int rpw : {4, 2}) if (N % (4 * rpw) == 0 && N / (4 * rpw) >= 512) return rpw;
  return 1;
}

template <typename HT, int NB, int RPW, int PRO, bool AMX, bool GATE>
int gemv_valu_kc(const h16_t *W, int N, int K, const float *in, long ldi, const float *g, float eps, float *out,
                 long ldo, const float *resid, float alpha, int B, float *amv, int32_t *ami, hipStream_t s) {
  // GATE: N counts gate outputs, each from two weight rows
  const int nblk = GATE ? N / (4 * RPW / 2) : N / (4 * RPW);
  const size_t sh = (size_t)NB * K * sizeof(float);
  const long gate_n = N;
  if (K <= 1024)
    hipLaunchKernelGGL((gemv_valu_kernel<HT, NB, RPW, 2, PRO, AMX, GATE>), dim3(nblk), dim3(256), sh, s, W, K, in,
                       ldi, g, eps, out, ldo, resid, alpha, B, amv, ami, nblk, gate_n);
  else if (K <= 2048)
    hipLaunchKernelGGL((gemv_valu_kernel<HT, NB, RPW, 4, PRO, AMX, GATE>), dim3(nblk), dim3(256), sh, s, W, K, in,
                       ldi, g, eps, out, ldo, resid, alpha, B, amv, ami, nblk, gate_n);
  else
    hipLaunchKernelGGL((gemv_valu_kernel<HT, NB, RPW, 6, PRO, AMX, GATE>), dim3(nblk), dim3(256), sh, s, W, K, in,
                       ldi, g, eps, out, ldo, resid, alpha, B, amv, ami, nblk, gate_n);
  return ne_hip_status(hipGetLastError(), "decode gemv");
}

template <typename HT, int NB, int PRO, bool AMX, bool GATE = false>
int gemv_valu_nb(const h16_t *W, int N, int K, const float *in, long ldi, const float *g, float eps, float *out,
                 long ldo, const float *resid, float alpha, int B, float *amv, int32_t *ami, hipStream_t s) {
  if (GATE) {  // two weight rows (W1 j, W3 j) per gate output; 2 outputs per wave
    if (N % 8) return ne_fail(NE_ERR_ARG, "decode gate gemv: hidden %d not a multiple of 8", N);
    return gemv_valu_kc<HT, NB, 4, PRO, AMX, true>(W, N, K, in, ldi, g, eps, out, ldo, resid, alpha, B, amv, ami, s);
  }
  const int rpw = pick_rpw(N);
  if (rpw == 4) return gemv_valu_kc<HT, NB, 4, PRO, AMX, false>(W, N, K, in, ldi, g, eps, out, ldo, resid, alpha, B, amv, ami, s);
  if (rpw == 2) return gemv_valu_kc<HT, NB, 2, PRO, AMX, false>(W, N, K, in, ldi, g, eps, out, ldo, resid, alpha, B, amv, ami, s);
  return gemv_valu_kc<HT, NB, 1, PRO, AMX, false>(W, N, K, in, ldi, g, eps, out, ldo, resid, alpha, B, amv, ami, s);
}

template <typename HT, int PRO, bool AMX, bool GATE = false>
int gemv_valu_pro(int B, const h16_t *W, int N, int K, const float *in, long ldi, const float *g, float eps,
                  float *out, long ldo, const float *resid, float alpha, float *amv, int32_t *ami, hipStream_t s) {
  if (B == 1) return gemv_valu_nb<HT, 1, PRO, AMX, GATE>(W, N, K, in, ldi, g, eps, out, ldo, resid, alpha, B, amv, ami, s);
  if (B == 2) return gemv_valu_nb<HT, 2, PRO, AMX, GATE>(W, N, K, in, ldi, g, eps, out, ldo, resid, alpha, B, amv, ami, s);
  return gemv_valu_nb<HT, 4, PRO, AMX, GATE>(W, N, K, in, ldi, g, eps, out, ldo, resid, alpha, B, amv, ami, s);
}

// Batch <= 4: out = alpha * W . pro(in) + resid.  Requires N % 4 == 0, K % 8 == 0.
int gemv_small(ne_ctx *c, int B, int pro, bool amx, const h16_t *W, int N, int K, const float *in, long ldi,
               const float *g, float *out, long ldo, const float *resid, float alpha, bool gate = false) {
  Dec *d = (Dec *)c->dec;
  if (N % 4 || K % 8 || K > 3072)
    return ne_fail(NE_ERR_ARG, "decode gemv: N=%d K=%d (need N%%4, K%%8, K <= 3072)", N, K);
  if ((((uintptr_t)in | (uintptr_t)(g ? g : in)) & 15) || ldi % 4)
    return ne_fail(NE_ERR_ARG, "decode gemv: input rows and gains must be 16-byte aligned");
  const float eps = c->c.norm_eps;
  return DISPATCH_H16(c->dt, [&] {
    if (pro == PRO_RMSNORM && gate)
      return gemv_valu_pro<HT, PRO_RMSNORM, false, true>(B, W, N, K, in, ldi, g, eps, out, ldo, nullptr, 1.f, nullptr, nullptr, c->st);
    if (pro == PRO_RMSNORM) {
      if (amx) return gemv_valu_pro<HT, PRO_RMSNORM, true>(B, W, N, K, in, ldi, g, eps, out, ldo, resid, alpha, d->amv, d->ami, c->st);
      return gemv_valu_pro<HT, PRO_RMSNORM, false>(B, W, N, K, in, ldi, g, eps, out, ldo, resid, alpha, nullptr, nullptr, c->st);
    }
    if (pro == PRO_SWIGLU)
      return gemv_valu_pro<HT, PRO_SWIGLU, false>(B, W, N, K, in, ldi, g, eps, out, ldo, resid, alpha, nullptr, nullptr, c->st);
    return gemv_valu_pro<HT, PRO_NONE, false>(B, W, N, K, in, ldi, g, eps, out, ldo, resid, alpha, nullptr, nullptr, c->st);
  }());
}

// Rows of the MFMA GEMVs' x and outputs: 16, or a multiple of 32 of them (decode: d->Bp).
inline int pad_rows(int rows) { return rows <= 16 ? 16 : (rows + 31) / 32 * 32; }

// Batch 5..32 (or the B rows of a prompt chunk, padded to Bp): the products of W [N, K] with x
// rows [Bp, K] (row stride ldx).  wsp
// (nullable): a workspace of cap floats for the split-K partials.
//  * nz_out != null: the partials stay in wsp for the consumer (*nz_out slices of [Bp, N]);
//  * else, with wsp: out = alpha * (their ordered sum) + resid, one block per sequence, and
//    with gn also xn = RMSNorm(out) * gn (the next GEMV's input);
//  * without wsp: one split, out = alpha * products (+ resid) directly;
//  * gate: W = [W1; W3] (2N rows), out [Bp, N] = silu(W1.x) * (W3.x), one split.
// Requires N % 16 (gate: N % 8), K % 128.
int gemv_big(ne_ctx *c, int B, int Bp, const h16_t *W, int N, int K, const float *x, long ldx, float *wsp, long cap,
             float *out, long ldo, const float *resid, float alpha, int *nz_out, const float *gn = nullptr,
             float *xn = nullptr, bool gate = false) {
  Dec *d = (Dec *)c->dec;
  if ((gate ? N % 8 : N % 16) || K % 128)
    return ne_fail(NE_ERR_ARG, "decode gemv: N=%d K=%d (need N%%16 (gate: %%8), K%%128)", N, K);
  if (gate && wsp) return ne_fail(NE_ERR_ARG, "decode gemv: the gate form has one split");
  int ks = 1;
  if (wsp)
    while ((N / 16) * ks < 512 && K % (128 * ks * 2) == 0 && (long)ks * 2 * Bp * N <= cap) ks *= 2;
  if (wsp && (long)ks * Bp * N > cap) return ne_fail(NE_ERR_ARG, "decode gemv: workspace too small");
  const dim3 grid(gate ? N / 8 : N / 16, ks, Bp <= 16 ? 1 : Bp / 32);
  // the gate form has one split: 8 waves per block shorten each wave's K range instead
  // (K % 256 then; else 4 waves)
  const bool wide = gate && K % 256 == 0;
  NE_CHECK(DISPATCH_H16(c->dt, [&] {
    auto go = [&](auto kernel, int threads) {
      hipLaunchKernelGGL(kernel, grid, dim3(threads), 0, c->st, W, (long)K, x, ldx, K, ks, out, ldo, resid, alpha,
                         wsp, N, B, Bp, (long)N, gate ? d->gate3 : nullptr);
    };
    if (Bp == 16) {
      if (wide) go(gemv_mfma_kernel<HT, 1, true, 8>, 512);
      else if (gate) go(gemv_mfma_kernel<HT, 1, true>, 256);
      else go(gemv_mfma_kernel<HT, 1, false>, 256);
    } else {
      if (wide) go(gemv_mfma_kernel<HT, 2, true, 8>, 512);
      else if (gate) go(gemv_mfma_kernel<HT, 2, true>, 256);
      else go(gemv_mfma_kernel<HT, 2, false>, 256);
    }
    return ne_hip_status(hipGetLastError(), "decode gemv");
  }()));
  if (nz_out) {
    *nz_out = ks;
    return 0;
  }
  if (wsp) {
    auto go = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3(B), dim3(256), 0, c->st, wsp, ks, Bp, N, out, ldo, resid, alpha, gn, xn,
                         c->c.norm_eps, d->xn3);
    };
    if (N > 1024) go(gemv_reduce_rows_kernel<0>);
    else if (ks == 1) go(gemv_reduce_rows_kernel<1>);
    else if (ks == 2) go(gemv_reduce_rows_kernel<2>);
    else if (ks == 4) go(gemv_reduce_rows_kernel<4>);
    else if (ks == 8) go(gemv_reduce_rows_kernel<8>);
    else go(gemv_reduce_rows_kernel<0>);
    NE_HIP(hipGetLastError());
  }
  return 0;
}

// Batch 5..32 with bf16 weights: the GEMV on gemv_bf3_kernel when its shape allows (returns
// 1 after launching; 0: not applicable, nothing launched).  mode BF3_WS: the split-K partials
// go to d->ws and *nz receives the split count; BF3_GATE: W = [W1; W3] (N rows each), gate
// [Bp, N] -> out; BF3_PLAIN: out [Bp, ldo] = products.
int gemv_bf3(ne_ctx *c, int B, int Bp, const h16_t *W, int N, int K, const h16_t *x3, int mode, float *out,
             long ldo, int *nz) {
  Dec *d = (Dec *)c->dec;
  if (c->dt != NE_BF16 || K % 128 || !x3) return 0;
  int ks = 0, rt = 2, ksplit = 1;
  if (mode == BF3_WS) {
    for (int cand : {2, 3, 1})
      if (K % (128 * cand) == 0 && K / (128 * cand) <= 8) {
        ks = cand;
        break;
      }
    if (!ks) return 0;
    ksplit = K / (128 * ks);
    rt = (N % 64 == 0 && (N / 64) * ksplit >= 192) ? 4 : 2;
    if (N % (16 * rt) || (long)ksplit * Bp * N > d->ws_elems) return 0;
  } else {
    ks = K / 128;
    if (ks != 1 && ks != 6 && ks != 8) return 0;
    if (N % (mode == BF3_GATE ? 16 : 32)) return 0;
    // the LM head: 128 rows per block (x read once per 128 rows: 1.61 -> 1.57 ms per batch-32
    // position against 32)
    if (mode == BF3_PLAIN && N % 128 == 0) rt = 8;
  }
  const int ntw = Bp == 16 ? 1 : 2;
  const dim3 grid(mode == BF3_GATE ? N / 16 : N / (16 * rt), ksplit, Bp / (16 * ntw));
  float *dst = mode == BF3_WS ? d->ws : out;
  const long ldd = mode == BF3_WS ? N : ldo;
  bool done = false;
  auto go = [&](auto kernel, int nt) {
    hipLaunchKernelGGL(kernel, grid, dim3(nt * 256), 0, c->st, W, (long)K, x3, K, dst, ldd, N, B, Bp, (long)N,
                       mode == BF3_GATE ? d->gate3 : nullptr);
    done = true;
  };
#define NE_BF3(NTW_)                                                                                 \
  if (mode == BF3_WS) {                                                                              \
    if (rt == 4 && ks == 2) go(gemv_bf3_kernel<NTW_, 4, 2, BF3_WS>, NTW_);                           \
    else if (rt == 4 && ks == 3) go(gemv_bf3_kernel<NTW_, 4, 3, BF3_WS>, NTW_);                      \
    else if (rt == 4 && ks == 1) go(gemv_bf3_kernel<NTW_, 4, 1, BF3_WS>, NTW_);                      \
    else if (rt == 2 && ks == 2) go(gemv_bf3_kernel<NTW_, 2, 2, BF3_WS>, NTW_);                      \
    else if (rt == 2 && ks == 3) go(gemv_bf3_kernel<NTW_, 2, 3, BF3_WS>, NTW_);                      \
    else if (rt == 2 && ks == 1) go(gemv_bf3_kernel<NTW_, 2, 1, BF3_WS>, NTW_);                      \
  } else if (mode == BF3_GATE) {                                                                     \
    if (ks == 8) go(gemv_bf3_kernel<NTW_, 2, 8, BF3_GATE>, NTW_);                                    \
    else if (ks == 6) go(gemv_bf3_kernel<NTW_, 2, 6, BF3_GATE>, NTW_);                               \
    else go(gemv_bf3_kernel<NTW_, 2, 1, BF3_GATE>, NTW_);                                            \
  } else if (rt == 8) {                                                                              \
    if (ks == 8) go(gemv_bf3_kernel<NTW_, 8, 8, BF3_PLAIN>, NTW_);                                   \
    else if (ks == 6) go(gemv_bf3_kernel<NTW_, 8, 6, BF3_PLAIN>, NTW_);                              \
    else go(gemv_bf3_kernel<NTW_, 8, 1, BF3_PLAIN>, NTW_);                                           \
  } else {                                                                                           \
    if (ks == 8) go(gemv_bf3_kernel<NTW_, 2, 8, BF3_PLAIN>, NTW_);                                   \
    else if (ks == 6) go(gemv_bf3_kernel<NTW_, 2, 6, BF3_PLAIN>, NTW_);                              \
    else go(gemv_bf3_kernel<NTW_, 2, 1, BF3_PLAIN>, NTW_);                                           \
  }
  if (ntw == 1) {
    NE_BF3(1)
  } else {
    NE_BF3(2)
  }
#undef NE_BF3
  if (!done) return 0;
  NE_CHECK(ne_hip_status(hipGetLastError(), "decode gemv (bf16 parts)"));
  if (nz) *nz = ksplit;
  return 1;
}

// Wo / W2 on gemv_bf3_kernel with the split-K sum, residual and RMSNorm of gemv_big's
// workspace form (gemv_reduce_rows_kernel); returns 0 when not applicable.
int gemv_bf3_resid(ne_ctx *c, int B, int Bp, const h16_t *W, int N, int K, const h16_t *x3, float *out, long ldo,
                   const float *resid, float alpha, const float *gn, float *xn) {
  Dec *d = (Dec *)c->dec;
  int ks = 0;
  const int rc = gemv_bf3(c, B, Bp, W, N, K, x3, BF3_WS, nullptr, 0, &ks);
  if (rc <= 0) return rc;
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(B), dim3(256), 0, c->st, d->ws, ks, Bp, N, out, ldo, resid, alpha, gn, xn,
                       c->c.norm_eps, d->xn3);
  };
  if (N > 1024) go(gemv_reduce_rows_kernel<0>);
  else if (ks == 1) go(gemv_reduce_rows_kernel<1>);
  else if (ks == 2) go(gemv_reduce_rows_kernel<2>);
  else if (ks == 4) go(gemv_reduce_rows_kernel<4>);
  else if (ks == 8) go(gemv_reduce_rows_kernel<8>);
  else go(gemv_reduce_rows_kernel<0>);
  NE_CHECK(ne_hip_status(hipGetLastError(), "decode gemv reduce"));
  return 1;
}

// qkv: the q|k|v rows [Bp, QKV], or (qnz > 1) qnz split-K partial slices of them.  nc > 0: the
// rows of a prompt chunk of nc positions from p0 on (PRE of dec_attn_kernel).
template <int HD, int R, bool KCOL>
void attn_go(ne_ctx *c, dim3 grid, size_t sh, const float *gq, const float *gk, float *kc, float *vc, const float *qkv,
             int qnz, int Bp, int p0, int nc) {
  Dec *d = (Dec *)c->dec;
  const double scale = 1.0 / sqrt((double)c->HD);
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(256), sh, c->st, qkv, c->QKV, gq, gk, d->cosb, d->sinb, kc, vc, d->att, c->NH,
                       c->NKV, d->ctx, d->st, c->c.norm_eps, scale, qkv, qnz, Bp, p0, nc,
                       KCOL && !nc ? nullptr : d->att3);
  };
  if (nc > 0) go(dec_attn_kernel<HD, R, KCOL, true>);
  else if constexpr (!KCOL || R == 1) go(dec_attn_kernel<HD, R, KCOL, false>);  // launch_attn: one head a block
}

template <int HD, int R>
void attn_kcol(ne_ctx *c, bool kcol, dim3 grid, size_t sh, const float *gq, const float *gk, float *kc, float *vc,
               const float *qkv, int qnz, int Bp, int p0, int nc) {
  if (kcol) attn_go<HD, R, true>(c, grid, sh, gq, gk, kc, vc, qkv, qnz, Bp, p0, nc);
  else attn_go<HD, R, false>(c, grid, sh, gq, gk, kc, vc, qkv, qnz, Bp, p0, nc);
}

int launch_attn(ne_ctx *c, int rows, int Bp, const LayerOff &o, float *kc, float *vc, const float *qkv, int qnz,
                bool kcol, int p0 = 0, int nc = 0) {
  Dec *d = (Dec *)c->dec;
  const int ratio = c->NH / c->NKV;
  // query heads per block: at batch <= 4 one (the blocks of a KV head share its K/V reads
  // through L2, and twice the blocks run), else all of the KV head's.  A prompt chunk has blocks
  // enough: all, unless their scores would not fit the LDS that batch <= 4 gets by with.
  const bool fits = (size_t)ratio * d->ctx * sizeof(float) <= 32768;
  const int qpb = kcol && !(nc && fits) ? 1 : ratio;
  const size_t sh = (size_t)qpb * d->ctx * sizeof(float);
  const float *gq = c->c.qk_norm ? c->P + o.gq : nullptr, *gk = c->c.qk_norm ? c->P + o.gk : nullptr;
  const dim3 grid(rows, c->NH / qpb);
  if (c->HD == 128) {
    if (qpb == 1) attn_kcol<128, 1>(c, kcol, grid, sh, gq, gk, kc, vc, qkv, qnz, Bp, p0, nc);
    else if (qpb == 2) attn_kcol<128, 2>(c, kcol, grid, sh, gq, gk, kc, vc, qkv, qnz, Bp, p0, nc);
    else attn_kcol<128, 4>(c, kcol, grid, sh, gq, gk, kc, vc, qkv, qnz, Bp, p0, nc);
  } else {
    if (qpb == 1) attn_kcol<64, 1>(c, kcol, grid, sh, gq, gk, kc, vc, qkv, qnz, Bp, p0, nc);
    else if (qpb == 2) attn_kcol<64, 2>(c, kcol, grid, sh, gq, gk, kc, vc, qkv, qnz, Bp, p0, nc);
    else attn_kcol<64, 4>(c, kcol, grid, sh, gq, gk, kc, vc, qkv, qnz, Bp, p0, nc);
  }
  return ne_hip_status(hipGetLastError(), "decode attention");
}

// One layer from its Wo on, on the MFMA GEMVs: x += alpha Wo.att, the FFN, and xn = RMSNorm(x)
// with the next gain.  rows of x, padded to Bp.
int big_layer_tail(ne_ctx *c, int rows, int Bp, const LayerOff &o, const float *g_next) {
  Dec *d = (Dec *)c->dec;
  const int D = c->D, H = c->H, Q = c->Q;
  const float alpha = c->c.res_alpha;
  const long cap = d->ws_elems;
  const h16_t *Pb = c->Pb;
  const float *g_ffn = c->P + o.g_ffn;
  int rc = gemv_bf3_resid(c, rows, Bp, Pb + o.wo, D, Q, d->att3, d->x, D, d->x, alpha, g_ffn, d->xn);
  if (rc < 0) return rc;
  if (!rc)
    NE_CHECK(gemv_big(c, rows, Bp, Pb + o.wo, D, Q, d->att, Q, d->ws, cap, d->x, D, d->x, alpha, nullptr, g_ffn, d->xn));
  rc = gemv_bf3(c, rows, Bp, Pb + o.w13, H, D, d->xn3, BF3_GATE, d->gate, H, nullptr);
  if (rc < 0) return rc;
  if (!rc)
    NE_CHECK(gemv_big(c, rows, Bp, Pb + o.w13, H, D, d->xn, D, nullptr, 0, d->gate, H, nullptr, 1.f, nullptr, nullptr,
                      nullptr, true));
  rc = gemv_bf3_resid(c, rows, Bp, Pb + o.w2, D, H, d->gate3, d->x, D, d->x, alpha, g_next, d->xn);
  if (rc < 0) return rc;
  if (!rc)
    NE_CHECK(gemv_big(c, rows, Bp, Pb + o.w2, D, H, d->gate, H, d->ws, cap, d->x, D, d->x, alpha, nullptr, g_next, d->xn));
  return 0;
}

// The QKV products of the rows of xn into d->ws; *qnz receives their split-K slice count.
int big_qkv(ne_ctx *c, int rows, int Bp, const LayerOff &o, int *qnz) {
  Dec *d = (Dec *)c->dec;
  const int rc = gemv_bf3(c, rows, Bp, c->Pb + o.wqkv, c->QKV, c->D, d->xn3, BF3_WS, nullptr, 0, qnz);
  if (rc < 0) return rc;
  if (!rc)
    NE_CHECK(gemv_big(c, rows, Bp, c->Pb + o.wqkv, c->QKV, c->D, d->xn, c->D, d->ws, d->ws_elems, nullptr, 0, nullptr,
                      1.f, qnz));
  return 0;
}

// Prompt positions 0 .. n_pos - 1 of B sequences into the KV cache, in chunks of up to d->Rp rows
// (row = sequence x position): the weights are read once per 32 rows and the chain of a position's
// launches is paid once per chunk.  Position by position that chain bounded the prompt (about
// 0.63 ms a position at batch 1, 1.43 ms at batch 32, Qwen3-0.6B): a 32-token prompt and 64 new
// tokens took 60.6 ms at batch 1 (fp16, sampled), 136.1 at batch 32 (bf16, greedy), now 44.8 and 115.6.
// The last layer's outputs are not needed: it ends with its keys and values.
int enqueue_prompt(ne_ctx *c, int B, int n_pos) {
  Dec *d = (Dec *)c->dec;
  const bool kcol = B <= VB;
  const float eps = c->c.norm_eps;
  const int per = d->Rp / B;  // positions per chunk
  for (int p0 = 0; p0 < n_pos; p0 += per) {
    const int nc = std::min(per, n_pos - p0), rows = B * nc, Bp = pad_rows(rows);
    auto token = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3(rows), dim3(256), 0, c->st, d->prompt, d->ctx, p0, nc, c->Pb + c->off_E, d->x,
                         c->D, c->P + c->lo[0].g_att, d->xn, eps, d->xn3);
    };
    if (c->dt == NE_FP16) token(pre_token_kernel<H16F>);
    else token(pre_token_kernel<H16B>);
    NE_HIP(hipGetLastError());
    for (int l = 0; l < c->L; l++) {
      const LayerOff &o = c->lo[l];
      const size_t kvl = (size_t)l * d->Bmax * c->NKV * d->ctx * c->HD;
      int qnz = 0;
      NE_CHECK(big_qkv(c, rows, Bp, o, &qnz));
      auto append = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(rows, c->NKV), dim3(c->HD), 0, c->st, d->ws, qnz, Bp, c->QKV,
                           c->c.qk_norm ? c->P + o.gk : nullptr, d->cosb, d->sinb, d->kc + kvl, d->vc + kvl, c->NH,
                           c->NKV, d->ctx, p0, nc, eps);
      };
      if (c->HD == 128) kcol ? append(pre_append_kernel<128, true>) : append(pre_append_kernel<128, false>);
      else kcol ? append(pre_append_kernel<64, true>) : append(pre_append_kernel<64, false>);
      NE_HIP(hipGetLastError());
      if (l + 1 == c->L) break;
      NE_CHECK(launch_attn(c, rows, Bp, o, d->kc + kvl, d->vc + kvl, d->ws, qnz, kcol, p0, nc));
      NE_CHECK(big_layer_tail(c, rows, Bp, o, c->P + c->lo[l + 1].g_att));
    }
  }
  return 0;
}

// Enqueue the kernels of one position for B sequences, with the final norm, LM head and token choice
// unless mode is PICK_NONE.  Position-independent (everything position-dependent is read from
// d->st), so it can be captured once and replayed.
int enqueue_position(ne_ctx *c, int B, int mode) {
  const bool gen = mode != PICK_NONE, greedy = mode == PICK_GREEDY;
  Dec *d = (Dec *)c->dec;
  const int D = c->D, H = c->H, Q = c->Q, NKV = c->NKV, HD = c->HD, QKV = c->QKV, V = c->V;
  const float eps = c->c.norm_eps, alpha = c->c.res_alpha;
  const h16_t *Pb = c->Pb;
  const float *Pf = c->P;
  const bool small = B <= VB;
  // batch 5..32: the kernels that write x (the token lookup, the Wo / W2 split-K reductions)
  // also write its RMSNorm with the next gain into xn; the QKV GEMV's partials are summed by
  // the attention kernel
  const float *g0 = small ? nullptr : Pf + c->lo[0].g_att;
  if (c->dt == NE_FP16)
    hipLaunchKernelGGL(dec_token_kernel<H16F>, dim3(B), dim3(256), 0, c->st, d->prompt, d->ctx, d->st, d->tok,
                       Pb + c->off_E, d->x, D, B, g0, d->xn, eps, d->xn3);
  else
    hipLaunchKernelGGL(dec_token_kernel<H16B>, dim3(B), dim3(256), 0, c->st, d->prompt, d->ctx, d->st, d->tok,
                       Pb + c->off_E, d->x, D, B, g0, d->xn, eps, d->xn3);
  NE_HIP(hipGetLastError());
  for (int l = 0; l < c->L; l++) {
    const LayerOff &o = c->lo[l];
    const size_t kvl = (size_t)l * d->Bmax * NKV * d->ctx * HD;
    if (small) {
      NE_CHECK(gemv_small(c, B, PRO_RMSNORM, false, Pb + o.wqkv, QKV, D, d->x, D, Pf + o.g_att, d->qkv, QKV, nullptr, 1.f));
      NE_CHECK(launch_attn(c, B, d->Bp, o, d->kc + kvl, d->vc + kvl, d->qkv, 1, true));
      NE_CHECK(gemv_small(c, B, PRO_NONE, false, Pb + o.wo, D, Q, d->att, Q, nullptr, d->x, D, d->x, alpha));
      // W1|W3 with the SwiGLU gate in its epilogue (gate -> xn), then W2 + residual
      NE_CHECK(gemv_small(c, B, PRO_RMSNORM, false, Pb + o.w13, H, D, d->x, D, Pf + o.g_ffn, d->xn, H, nullptr, 1.f,
                          true));
      NE_CHECK(gemv_small(c, B, PRO_NONE, false, Pb + o.w2, D, H, d->xn, H, nullptr, d->x, D, d->x, alpha));
    } else {
      int qnz = 0;
      NE_CHECK(big_qkv(c, B, d->Bp, o, &qnz));
      NE_CHECK(launch_attn(c, B, d->Bp, o, d->kc + kvl, d->vc + kvl, d->ws, qnz, false));
      NE_CHECK(big_layer_tail(c, B, d->Bp, o, l + 1 < c->L ? Pf + c->lo[l + 1].g_att : Pf + c->off_gfinal));
    }
  }
  if (gen) {
    if (small) {
      NE_CHECK(gemv_small(c, B, PRO_RMSNORM, greedy, Pb + c->off_E, V, D, d->x, D, Pf + c->off_gfinal, d->logits, V,
                          nullptr, 1.f));
      if (greedy)
        hipLaunchKernelGGL(dec_argmax_kernel, dim3(B), dim3(1024), 0, c->st, d->amv, d->ami, V / (4 * pick_rpw(V)),
                           d->st, d->ctx, d->tok, d->out);
    } else {
      const int rc = gemv_bf3(c, B, d->Bp, Pb + c->off_E, V, D, d->xn3, BF3_PLAIN, d->logits, V, nullptr);
      if (rc < 0) return rc;
      if (!rc) NE_CHECK(gemv_big(c, B, d->Bp, Pb + c->off_E, V, D, d->xn, D, nullptr, 0, d->logits, V, nullptr, 1.f, nullptr));
      if (greedy) {
        hipLaunchKernelGGL(dec_argmax_part_kernel, dim3(BIG_ARGMAX, B), dim3(256), 0, c->st, d->logits, V, BIG_ARGMAX,
                           d->amv, d->ami);
        hipLaunchKernelGGL(dec_argmax_kernel, dim3(B), dim3(1024), 0, c->st, d->amv, d->ami, BIG_ARGMAX, d->st, d->ctx,
                           d->tok, d->out);
      }
    }
    if (!greedy)
      NE_CHECK(launch_sample({d->logits, V, d->sg, d->schunk, d->st, d->unif, d->ctx, d->tok, d->out, d->spmax, d->spsum,
                              d->shist, d->smass, d->spre, d->sabove, mode == PICK_TOPP},
                             B, c->st));
  }
  hipLaunchKernelGGL(dec_advance_kernel, dim3(1), dim3(64), 0, c->st, d->st);
  return ne_hip_status(hipGetLastError(), "decode position");
}

int capture(ne_ctx *c, int B, int mode, hipGraphExec_t *exec) {
  hipGraph_t graph = nullptr;
  NE_HIP(hipStreamBeginCapture(c->st, hipStreamCaptureModeThreadLocal));
  const int rc = enqueue_position(c, B, mode);
  const hipError_t ec = hipStreamEndCapture(c->st, &graph);
  if (rc) {
    if (graph) (void)hipGraphDestroy(graph);
    return rc;
  }
  NE_HIP(ec);
  const hipError_t ei = hipGraphInstantiate(exec, graph, nullptr, nullptr, 0);
  (void)hipGraphDestroy(graph);
  NE_HIP(ei);
  return 0;
}

}  // namespace

int decode_alloc(ne_ctx *c) {
  Dec *d = new Dec();
  c->dec = d;
  if (c->c.decode_batch > 32) return ne_fail(NE_ERR_ARG, "decode_batch %d > 32", c->c.decode_batch);
  if (c->NH / c->NKV != 1 && c->NH / c->NKV != 2 && c->NH / c->NKV != 4)
    return ne_fail(NE_ERR_ARG, "decode: %d query heads per KV head (1, 2 or 4)", c->NH / c->NKV);
  if (c->D % 128 || c->H % 128 || c->Q % 128)
    return ne_fail(NE_ERR_ARG, "decode: dim, hidden and q_dim must be multiples of 128");
  d->Bmax = c->c.decode_batch;
  d->Bp = d->Bmax <= 16 ? 16 : 32;
  d->ctx = c->c.decode_ctx;
  d->Rp = std::max(d->Bp, pad_rows((int)std::min<long>(PROMPT_ROWS, (long)d->Bmax * (d->ctx - 1))));
  const size_t Rp = d->Rp, Bp = d->Bp, Bm = d->Bmax, ctx = d->ctx, L = c->L, D = c->D, H = c->H, Q = c->Q, NKV = c->NKV,
               HD = c->HD, V = c->V;
  const size_t kv = L * Bm * NKV * ctx * HD;
  d->lm_nblk = std::max<int>(c->V / (4 * pick_rpw(c->V)), BIG_ARGMAX);
  d->ws_elems = (long)8 * Rp * std::max<size_t>(2 * H, Q + 2 * NKV * HD);
  size_t off = 0;
  auto take = [&](size_t bytes) { size_t o = off; off += (bytes + 255) & ~(size_t)255; return o; };
  const size_t o_kc = take(kv * 4), o_vc = take(kv * 4), o_x = take(Rp * D * 4);
  const size_t o_xn = take(Rp * std::max(D, H) * 4);
  const size_t o_qkv = take(Bp * (Q + 2 * NKV * HD) * 4), o_att = take(Rp * Q * 4);
  const size_t o_lg = take(Bp * V * 4);
  const size_t o_ws = take((size_t)d->ws_elems * 4), o_gate = take(Rp * H * 4);
  const size_t parts = c->dt == NE_BF16 ? 3 * Rp * 2 : 0;  // bytes a column of the bf16-part planes
  const size_t o_xn3 = take(parts * D), o_att3 = take(parts * Q), o_gate3 = take(parts * H);
  const size_t o_amv = take(Bp * (size_t)d->lm_nblk * 4), o_ami = take(Bp * (size_t)d->lm_nblk * 4);
  const size_t o_tok = take(Bp * 4), o_out = take(Bp * ctx * 4), o_pr = take(Bp * ctx * 4), o_u = take(Bp * ctx * 8);
  // row chunks of at least 1024 columns, a multiple of 4 (16-byte accesses)
  d->sg = std::max(1, std::min(SAMP_G, c->V / 1024));
  d->schunk = ((c->V + d->sg - 1) / d->sg + 3) / 4 * 4;
  const size_t o_pm = take(Bp * d->sg * 4), o_ps = take(Bp * d->sg * 8), o_ms = take(Bp * d->sg * 8);
  const size_t o_hi = take(Bp * 3 * SAMP_BINS * 8), o_ab = take(Bp * 2 * 8), o_pf = take(Bp * 2 * 4);
  const size_t o_cos = take(ctx * HD / 2 * 4), o_sin = take(ctx * HD / 2 * 4), o_st = take(sizeof(DecState));
  NE_HIP(hipMalloc(&d->arena, off));
  char *base = (char *)d->arena;
  d->kc = (float *)(base + o_kc); d->vc = (float *)(base + o_vc);
  d->x = (float *)(base + o_x); d->xn = (float *)(base + o_xn);
  d->qkv = (float *)(base + o_qkv); d->att = (float *)(base + o_att);
  d->logits = (float *)(base + o_lg);
  d->ws = (float *)(base + o_ws);
  d->gate = (float *)(base + o_gate);
  if (parts) {
    d->xn3 = (h16_t *)(base + o_xn3);
    d->att3 = (h16_t *)(base + o_att3);
    d->gate3 = (h16_t *)(base + o_gate3);
  }
  d->amv = (float *)(base + o_amv); d->ami = (int32_t *)(base + o_ami);
  d->tok = (int32_t *)(base + o_tok); d->out = (int32_t *)(base + o_out); d->prompt = (int32_t *)(base + o_pr);
  d->unif = (double *)(base + o_u);
  d->spmax = (float *)(base + o_pm); d->spsum = (double *)(base + o_ps);
  d->smass = (unsigned long long *)(base + o_ms); d->shist = (unsigned long long *)(base + o_hi);
  d->sabove = (unsigned long long *)(base + o_ab); d->spre = (uint32_t *)(base + o_pf);
  d->cosb = (float *)(base + o_cos); d->sinb = (float *)(base + o_sin);
  d->st = (DecState *)(base + o_st);
  NE_HIP(hipMemset(d->arena, 0, off));
  // RoPE tables for decode positions: float64 angles rounded to fp32 (generate.py:101-105)
  const int half = c->HD / 2;
  std::vector<float> cs(ctx * half), sn(ctx * half);
  for (size_t p = 0; p < ctx; p++)
    for (int i = 0; i < half; i++) {
      const double ang = (double)p * (1.0 / pow((double)c->c.rope_theta, 2.0 * i / c->HD));
      cs[p * half + i] = (float)cos(ang);
      sn[p * half + i] = (float)sin(ang);
    }
  NE_HIP(hipMemcpy(d->cosb, cs.data(), cs.size() * 4, hipMemcpyHostToDevice));
  NE_HIP(hipMemcpy(d->sinb, sn.data(), sn.size() * 4, hipMemcpyHostToDevice));
  return 0;
}

void decode_free(ne_ctx *c) {
  Dec *d = (Dec *)c->dec;
  if (!d) return;
  for (auto &g : d->graphs) {
    if (g.exec) hipGraphExecDestroy(g.exec);
  }
  if (d->arena) hipFree(d->arena);
  delete d;
  c->dec = nullptr;
}

namespace {
int positions(ne_ctx *c, int B, int n, int mode);
}

int decode_run(ne_ctx *c, const int32_t *prompt, int B, int P, int n_new, float temp, float top_p,
               const double *uniforms, int32_t *out) {
  Dec *d = (Dec *)c->dec;
  if (!d) return ne_fail(NE_ERR_STATE, "context created without decode buffers (decode_batch/decode_ctx)");
  if (B <= 0 || B > c->c.decode_batch || P <= 0 || n_new <= 0 || P + n_new > d->ctx)
    return ne_fail(NE_ERR_ARG, "decode: B=%d P=%d n_new=%d exceed decode_batch=%d / decode_ctx=%d", B, P, n_new,
                   c->c.decode_batch, d->ctx);
  const bool greedy = temp < 1e-6f;
  const int mode = greedy ? PICK_GREEDY : top_p < 1.f ? PICK_TOPP : PICK_SAMPLE;
  if (!greedy && !uniforms) return ne_fail(NE_ERR_ARG, "decode: sampling needs uniforms");
  for (long i = 0; i < (long)B * P; i++)
    if (prompt[i] < 0 || prompt[i] >= c->V) return ne_fail(NE_ERR_ARG, "decode: prompt id out of range");
  // Every call runs its prompt from position 0 and rebuilds the KV cache, so the cache layout
  // may follow this call's batch size (K column-major at B <= 4, row-major above,
  // dec_attn_kernel); a cache kept across calls would have to keep one layout for both.
  // per-call inputs: prompt rows, uniforms, state (outside the captured graphs)
  std::vector<int32_t> pr((size_t)d->Bp * d->ctx, 0);
  for (int b = 0; b < B; b++)
    for (int j = 0; j < P; j++) pr[(size_t)b * d->ctx + j] = prompt[(size_t)b * P + j];
  NE_HIP(hipMemcpyAsync(d->prompt, pr.data(), pr.size() * 4, hipMemcpyHostToDevice, c->st));
  std::vector<double> u;
  if (!greedy) {
    u.assign((size_t)d->Bp * d->ctx, 0.0);
    for (int b = 0; b < B; b++)
      for (int j = 0; j < n_new; j++) u[(size_t)b * d->ctx + j] = uniforms[(size_t)b * n_new + j];
    NE_HIP(hipMemcpyAsync(d->unif, u.data(), u.size() * 8, hipMemcpyHostToDevice, c->st));
  }
  // Prompt positions before the last: in chunks, except the one or two of a small batch (a chunk
  // takes about as long as two positions of the VALU GEMVs).
  const bool by_chunk = P - 1 > (B <= VB ? 2 : 1);
  const DecState s0 = {by_chunk ? P - 1 : 0, P, temp, top_p};
  NE_HIP(hipMemcpyAsync(d->st, &s0, sizeof s0, hipMemcpyHostToDevice, c->st));
  NE_HIP(hipStreamSynchronize(c->st));  // host staging vectors are released at return

  if (by_chunk) NE_CHECK(enqueue_prompt(c, B, P - 1));
  else NE_CHECK(positions(c, B, P - 1, PICK_NONE));
  NE_CHECK(positions(c, B, n_new, mode));
  std::vector<int32_t> o((size_t)d->Bp * d->ctx);
  NE_HIP(hipMemcpyAsync(o.data(), d->out, o.size() * 4, hipMemcpyDeviceToHost, c->st));
  NE_HIP(hipStreamSynchronize(c->st));
  for (int b = 0; b < B; b++)
    for (int j = 0; j < n_new; j++) out[(size_t)b * n_new + j] = o[(size_t)b * d->ctx + j];
  return 0;
}

namespace {

// The next n positions: the captured graph of one (captured on first use per batch size and mode) replayed
// n times, or eager launches where graphs are off (tracers that do not follow graph launches).  The one or
// two prompt positions of a short prompt replay theirs too: eagerly their 140 launches each took longer than
// their kernels (batch 1, Qwen3-0.6B, a prompt of 3 tokens and 1 new: 1.75 ms replayed, 1.81-1.88 eager).
int positions(ne_ctx *c, int B, int n, int mode) {
  Dec *d = (Dec *)c->dec;
  if (!c->use_graphs) {
    for (int j = 0; j < n; j++) NE_CHECK(enqueue_position(c, B, mode));
    return 0;
  }
  if (n <= 0) return 0;
  Dec::Graph *gr = nullptr;
  for (auto &g : d->graphs)
    if (g.B == B && g.mode == mode) gr = &g;
  if (!gr) {
    Dec::Graph g = {B, mode, nullptr};
    NE_CHECK(capture(c, B, mode, &g.exec));
    d->graphs.push_back(g);
    gr = &d->graphs.back();
  }
  for (int j = 0; j < n; j++) NE_HIP(hipGraphLaunch(gr->exec, c->st));
  return 0;
}

}  // namespace
