// north-mini-code resident preprocessing and attention bank (gfx950): the steps either side of the MoE block.
//   int64 matrices                  nmc_qk_cuda.cu:1068 `qk_register_i64` (qk_cuda.py:285-303)
//   RMSNorm + router + top-k        nmc_qk_cuda.cu:1116 `qk_rmsnorm_router` (qk_cuda.py:331-372); semantics
//                                   cohere2.py:162-188 (router = exact linear >> fw, lowest-index top-k, sigmoid
//                                   gates without the 2^62 / log2e cap, nmc/_bonsai/fixedpoint.py:148)
//   attention bank                  nmc_qk_cuda.cu:877-1040, :1363-1780 (qk_cuda.py:476-715): per-request K/V
//                                   per layer, M = 1 decode: Q/K/V -> interleaved RoPE (cohere2.py:125-133,
//                                   nmc/_bonsai/rope.py:79-100) -> K/V append -> GQA fixed-point attention over
//                                   the window (cohere2.py:136-161) -> O; MoE layer begin / continue with the
//                                   parallel residual x + Attn(n(x)) + MoE(n(x)) (cohere2.py:191-199)
// Guards follow the reference producer: a RoPE / attention / router / RMSNorm envelope miss returns 3 and
// poisons the bank layer (its K/V length does not advance).
#include "imie_common.h"
#include "imie_kernels.h"
#include <string.h>
#include <climits>

int imie_qk_info(int64_t h, int64_t* out_f, int64_t* nb, int* qtype, const uint8_t** p);
int64_t imie_qk_register_i64(const int64_t* W, int64_t rows, int64_t cols);
int imie_qk_linear_dev(int64_t h, const int64_t* x, int64_t T, int fw, int64_t* out, int* status, hipStream_t st);
int imie_qk_linears_dev(const int64_t* hs, int cnt, const int64_t* x, int fw, int64_t* const* outs, int* status,
                        hipStream_t st);
int imie_qk_moe_dev(const long long* gate_h, const long long* up_h, const long long* down_h, int k,
                    const int64_t* h_dev, const int64_t* gates_dev, int64_t d_model, int64_t e_ffn, int fa, int fw,
                    const int64_t* res, const int64_t* ao, int64_t* moe, int64_t* out_dev, int* status_dev,
                    hipStream_t st);

namespace {

typedef __int128 i128;
typedef unsigned __int128 u128;
constexpr int kGuard = 8;                             // bank status bit: an exact envelope guard fired

__device__ inline uint64_t nb_uabs(int64_t v) { return v < 0 ? 0 - (uint64_t)v : (uint64_t)v; }

__device__ inline int64_t nb_exp2_neg(int64_t u, int fa) {     // fixedpoint.py:74-96
  const int64_t fp = (int64_t)1 << fa;
  const int64_t k = u >> fa, f = u & (fp - 1);
  const int sh = 16 - fa;
  int64_t c0, c1, c2, c3;
  if (sh >= 0) { c0 = 65536 >> sh; c1 = 45426 >> sh; c2 = 15743 >> sh; c3 = 3638 >> sh; }
  else { c0 = (int64_t)65536 << -sh; c1 = (int64_t)45426 << -sh; c2 = (int64_t)15743 << -sh; c3 = (int64_t)3638 << -sh; }
  const int64_t f2 = (int64_t)((uint64_t)f * (uint64_t)f) >> fa;
  const int64_t f3 = (int64_t)((uint64_t)f2 * (uint64_t)f) >> fa;
  int64_t poly = c0 - ((int64_t)((uint64_t)c1 * (uint64_t)f) >> fa) + ((int64_t)((uint64_t)c2 * (uint64_t)f2) >> fa) -
                 ((int64_t)((uint64_t)c3 * (uint64_t)f3) >> fa);
  if (poly < 0) poly = 0;
  if (k < 0) return 0;
  return poly >> (k < 63 ? k : 63);
}

__device__ inline int64_t nb_log2e(int fa) {
  const int sh = 16 - fa;
  return sh >= 0 ? (94548 >> sh) : ((int64_t)94548 << -sh);
}

// gate sigmoid (the nmc variant: d_clip without the 2^62 / log2e cap)
__device__ inline int64_t nb_sigmoid(int64_t x, int fa) {
  const int64_t l = nb_log2e(fa), dclip = ((int64_t)(fa + 2) << (2 * fa)) / l;
  const int64_t m = x > 0 ? x : 0;
  int64_t d0 = m, d1 = (int64_t)((uint64_t)m - (uint64_t)x);
  if (d0 > dclip) d0 = dclip;
  if (d1 > dclip) d1 = dclip;
  const int64_t e0 = nb_exp2_neg((int64_t)((uint64_t)d0 * (uint64_t)l) >> fa, fa);
  const int64_t e1 = nb_exp2_neg((int64_t)((uint64_t)d1 * (uint64_t)l) >> fa, fa);
  const int64_t z = e0 + e1;
  return z == 0 ? 0 : (int64_t)(((u128)(uint64_t)e1 << fa) / (u128)(uint64_t)z);
}

// block max of u64 (256 threads); result in every thread
__device__ inline uint64_t nb_block_max(uint64_t v) {
  __shared__ uint64_t s[4];
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    const uint64_t u = (uint64_t)__shfl_xor((long long)v, o, 64);
    v = u > v ? u : v;
  }
  __syncthreads();
  if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = v;
  __syncthreads();
  uint64_t m = 0;
  for (int k = 0; k < (int)(blockDim.x >> 6); ++k) m = s[k] > m ? s[k] : m;
  return m;
}

// router: logits[r, e] = (sum_i h[r, i] * W[e, i]) >> fw, exact; the unshifted sum must fit int64
// (nmc_qk_cuda.cu:560-638). One workgroup per (row, expert): when max|h| * max|w| * width fits int64 the int64
// sum is exact; otherwise one thread runs the exact int128 sum with per-term overflow checks.
__global__ __launch_bounds__(256) void nb_router_kernel(const int64_t* __restrict__ h, int64_t width,
                                                        const int64_t* __restrict__ W, int experts, int fw,
                                                        int64_t* __restrict__ logits, int* __restrict__ status) {
  __shared__ int64_t s_sum[4];
  const int64_t row = blockIdx.y;
  const int e = blockIdx.x;
  const int64_t* hr = h + row * width;
  const int64_t* wr = W + (int64_t)e * width;
  // one pass: the wrapping sum and both maxima together (the sum counts only where the maxima say it is exact)
  __shared__ uint64_t s_h[4], s_w[4];
  uint64_t mh = 0, mw = 0, acc = 0;
#pragma unroll 8
  for (int64_t i = threadIdx.x; i < width; i += 256) {
    const int64_t hv = hr[i], wv = wr[i];
    const uint64_t a = nb_uabs(hv), b = nb_uabs(wv);
    mh = a > mh ? a : mh;
    mw = b > mw ? b : mw;
    acc += (uint64_t)hv * (uint64_t)wv;
  }
  mh = imie_wave_max_u64_full(mh);
  mw = imie_wave_max_u64_full(mw);
  acc = imie_wave_sum_u64_full(acc);
  if ((threadIdx.x & 63) == 0) {
    const int w = threadIdx.x >> 6;
    s_h[w] = mh;
    s_w[w] = mw;
    s_sum[w] = (int64_t)acc;
  }
  __syncthreads();
  if (threadIdx.x) return;
  for (int w = 1; w < 4; ++w) {
    mh = s_h[w] > mh ? s_h[w] : mh;
    mw = s_w[w] > mw ? s_w[w] : mw;
    acc += (uint64_t)s_sum[w];
  }
  if (mh == 0 || mw == 0 || (u128)mh * mw * (u128)(uint64_t)width <= (u128)INT64_MAX) {
    logits[row * experts + e] = (int64_t)acc >> fw;
    return;
  }
  const i128 mx = (i128)(((u128)1 << 127) - 1), mn = -mx - 1;
  i128 sum = 0;
  for (int64_t i = 0; i < width; ++i) {
    const i128 t = (i128)hr[i] * wr[i];
    if ((t > 0 && sum > mx - t) || (t < 0 && sum < mn - t)) {
      atomicOr(status, kGuard);
      logits[row * experts + e] = 0;
      return;
    }
    sum += t;
  }
  if (sum > (i128)INT64_MAX || sum < (i128)INT64_MIN) {
    atomicOr(status, kGuard);
    logits[row * experts + e] = 0;
    return;
  }
  logits[row * experts + e] = (int64_t)sum >> fw;
}

// lowest-index top-k by logit and their sigmoid gates (cohere2.py:162-165, :181-182); one wave per row. The order
// (logit descending, index ascending) is total, so pick k is the first element of that order behind pick k - 1: a
// wave maximum over the lanes' strided elements, then the lowest index that holds it from the lanes' ballots; no list
// of the taken ones. Bound by the latency of its `used` reductions (DPP, no LDS); lane k forms gate k at the end.
// (One thread per row scanning every logit for every pick took 467 us at 128 experts, top-8; this takes 10.)
__global__ __launch_bounds__(64) void nb_topk_kernel(const int64_t* __restrict__ logits, int experts, int used, int fa,
                                                     int* __restrict__ ids, int64_t* __restrict__ gates) {
  const int64_t r = blockIdx.x;
  const int lane = threadIdx.x;
  const int64_t* lr = logits + r * experts;
  constexpr uint64_t kSign = (uint64_t)1 << 63;       // logits as unsigned keys in the same order
  constexpr int kKeep = 4;                            // keys kept in registers: 256 experts without a reload
  uint64_t v[kKeep];
#pragma unroll
  for (int i = 0; i < kKeep; ++i) v[i] = lane + 64 * i < experts ? (uint64_t)lr[lane + 64 * i] ^ kSign : 0;
  const int ni = (experts + 63) / 64;
  uint64_t prev = 0;
  int prev_id = -1;
  for (int k0 = 0; k0 < used; k0 += 64) {
    int64_t mine = 0;
    for (int k = k0; k < used && k < k0 + 64; ++k) {
      auto behind = [&](uint64_t x, int e) {
        return e < experts && (prev_id < 0 || x < prev || (x == prev && e > prev_id));
      };
      uint64_t best = 0;                              // 0: the lowest key, so also the value of "none" in the maximum
#pragma unroll
      for (int i = 0; i < kKeep; ++i) best = behind(v[i], lane + 64 * i) && v[i] > best ? v[i] : best;
      for (int i = kKeep; i < ni; ++i) {
        const int e = lane + 64 * i;
        const uint64_t x = e < experts ? (uint64_t)lr[e] ^ kSign : 0;
        best = behind(x, e) && x > best ? x : best;
      }
      best = imie_wave_max_u64_full(best);
      int id = -1;
#pragma unroll
      for (int i = 0; i < kKeep; ++i) {
        const uint64_t b = __ballot(behind(v[i], lane + 64 * i) && v[i] == best);
        if (id < 0 && b) id = 64 * i + __builtin_ctzll(b);
      }
      for (int i = kKeep; i < ni && id < 0; ++i) {
        const int e = lane + 64 * i;
        const uint64_t x = e < experts ? (uint64_t)lr[e] ^ kSign : 0;
        const uint64_t b = __ballot(behind(x, e) && x == best);
        if (b) id = 64 * i + __builtin_ctzll(b);
      }
      prev = best;
      prev_id = id;
      if (lane == 0) ids[r * used + k] = id;
      if (lane == k - k0) mine = (int64_t)(best ^ kSign);
    }
    if (k0 + lane < used) gates[r * used + k0 + lane] = nb_sigmoid(mine, fa);
  }
}

// Interleaved RoPE of q (in place) and k, the K / V append at `pos` (cache [Hkv][max_len][hd]) and the running
// max|K|, max|V| (kv_max[0..1]); one workgroup per q or kv head. The reference's envelope guard
// (2 max|x| max|cos, sin| <= INT64_MAX over all of q, and over all of k, rope.py:26-39) fires when any head's own
// maximum breaks it, so every workgroup tests its head and none waits for the others; after a guard the outputs
// are discarded, so what is written then does not matter. Latency-bound (one dependent load, two reductions): one
// launch in place of three single-workgroup ones (RoPE 13 us, append and max|q| 5 us each).
__global__ __launch_bounds__(128) void nb_rope_append_kernel(int64_t* __restrict__ q, int heads,
                                                             const int64_t* __restrict__ k,
                                                             const int64_t* __restrict__ v, int hd,
                                                             const int64_t* __restrict__ cs,
                                                             const int64_t* __restrict__ sn, int64_t pos,
                                                             int64_t max_len, int fa, int rope,
                                                             int64_t* __restrict__ ck, int64_t* __restrict__ cv,
                                                             uint64_t* __restrict__ kv_max, int* __restrict__ status) {
  const bool is_q = (int)blockIdx.x < heads;
  const int64_t kvh = is_q ? 0 : (int64_t)blockIdx.x - heads;
  const int64_t* x = is_q ? q + (int64_t)blockIdx.x * hd : k + kvh * hd;
  int64_t* y = is_q ? q + (int64_t)blockIdx.x * hd : ck + (kvh * max_len + pos) * hd;
  const int half = hd / 2;
  uint64_t mx = 0, mc = 0, mk = 0, mv = 0;
  for (int i = threadIdx.x; i < half; i += 128) {
    int64_t a = x[2 * i], b = x[2 * i + 1];
    if (rope) {
      const int64_t c = cs[pos * half + i], s = sn[pos * half + i];
      const uint64_t ua = nb_uabs(a), ub = nb_uabs(b), uc = nb_uabs(c), us = nb_uabs(s);
      mx = ua > mx ? ua : mx;
      mx = ub > mx ? ub : mx;
      mc = uc > mc ? uc : mc;
      mc = us > mc ? us : mc;
      const i128 p0 = (i128)a * c - (i128)b * s, p1 = (i128)a * s + (i128)b * c;
      if (p0 > (i128)INT64_MAX || p0 < (i128)INT64_MIN || p1 > (i128)INT64_MAX || p1 < (i128)INT64_MIN)
        atomicOr(status, kGuard);
      a = (int64_t)p0 >> fa;
      b = (int64_t)p1 >> fa;
    }
    if (rope || !is_q) { y[2 * i] = a; y[2 * i + 1] = b; }
    if (!is_q) {
      const uint64_t ua = nb_uabs(a), ub = nb_uabs(b);
      mk = ua > mk ? ua : mk;
      mk = ub > mk ? ub : mk;
    }
  }
  if (!is_q)
    for (int i = threadIdx.x; i < hd; i += 128) {
      const int64_t a = v[kvh * hd + i];
      cv[(kvh * max_len + pos) * hd + i] = a;
      const uint64_t u = nb_uabs(a);
      mv = u > mv ? u : mv;
    }
  if (rope) {
    mx = imie_wave_max_u64_full(mx);
    mc = imie_wave_max_u64_full(mc);
    __shared__ uint64_t s_m[2][2];
    if ((threadIdx.x & 63) == 0) { s_m[threadIdx.x >> 6][0] = mx; s_m[threadIdx.x >> 6][1] = mc; }
    __syncthreads();
    if (threadIdx.x == 0) {
      const uint64_t m0 = s_m[0][0] > s_m[1][0] ? s_m[0][0] : s_m[1][0];
      const uint64_t m1 = s_m[0][1] > s_m[1][1] ? s_m[0][1] : s_m[1][1];
      if ((u128)2 * m0 * m1 > (u128)INT64_MAX) atomicOr(status, kGuard);
    }
  }
  if (!is_q) {
    mk = imie_wave_max_u64_full(mk);
    mv = imie_wave_max_u64_full(mv);
    if ((threadIdx.x & 63) == 0) {
      atomicMax((unsigned long long*)&kv_max[0], (unsigned long long)mk);
      atomicMax((unsigned long long*)&kv_max[1], (unsigned long long)mv);
    }
  }
}

// GQA fixed-point attention of the new position `pos` over keys [first, pos] (sliding window when window > 0):
// score = (((q . k) >> fa) * inv_sqrt) >> fa, softmax of the 2^-d cubic, out = (p . V) >> fa; every int64
// narrowing is checked (nmc_qk_cuda.cu:343-432).
//
// The keys are split into chunks (a multiple of 64 keys, at most kNbMaxChunks of them); a workgroup takes one chunk of
// one KV head and up to eight of its query heads, so K and V are read once. Four launches: scores and chunk maxima;
// e and chunk Z; p and chunk PV sums; the sum over chunks. Under the envelope (max|q| max|K| hd and 2^fa max|V| within
// int64; otherwise the status is set and the result discarded) the dots and the PV sums fit int64, so 64-bit sums are
// exact in any order; only the narrowing of (q . k >> fa) * inv_sqrt needs 128 bits, once per score.
// Bound by latency (34 MB of K and V at 4096 keys x 4 heads take 5 us at 7 TB/s): at a 4096-key window, 32 / 4 heads
// of 128, 1923 us as one workgroup per query head with 128-bit dots, whose PV walked the keys serially in 128
// threads, against 18 + 5 + 11 + 4 us for the four launches.
constexpr int kNbHeads = 8;                           // query heads of one KV head per workgroup
constexpr int kNbMaxChunks = 128;

struct NbAttn {
  const int64_t *q, *ck, *cv;
  int64_t first, pos, max_len, chunk;                 // keys [first, pos], chunk keys per workgroup
  int heads, nkv, hd, fa;
  int64_t inv_sqrt;
  const uint64_t* kv_max;
  int64_t *prob, *cmax;                               // scores, then e [heads][max_len]; chunk maxima [chunk][heads]
  uint64_t *cz, *part;                                // chunk Z [chunk][heads]; chunk PV sums [chunk][heads][hd]
  int64_t* out;
  int* status;
};

struct NbGroup { int kv, h0, nh; };                   // KV head, first query head, query heads of this workgroup
__device__ inline NbGroup nb_group(const NbAttn& a) {
  const int rep = a.heads / a.nkv, ng = (rep + kNbHeads - 1) / kNbHeads;
  const int kv = (int)blockIdx.x / ng, g = (int)blockIdx.x % ng;
  return NbGroup{kv, kv * rep + g * kNbHeads, min(kNbHeads, rep - g * kNbHeads)};
}

// NIT: 32-dim steps of a key row (hd <= 32 NIT). 16 lanes share a key (2 dims a lane and step), each lane takes four
// keys of the 64-key step at once, so a step's K loads are all in flight together.
template <int NIT>
__global__ __launch_bounds__(256) void nb_scores_kernel(NbAttn a) {
  __shared__ __align__(16) int64_t s_q[kNbHeads][32 * NIT];
  __shared__ int64_t s_b[4][kNbHeads];
  __shared__ uint64_t s_m[4];
  const NbGroup g = nb_group(a);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l16 = tid & 15, grp = tid >> 4;
  uint64_t mq = 0;
  for (int i = tid; i < kNbHeads * 32 * NIT; i += 256) {
    const int hh = i / (32 * NIT), c = i % (32 * NIT);
    const int64_t v = hh < g.nh && c < a.hd ? a.q[(int64_t)(g.h0 + hh) * a.hd + c] : 0;
    s_q[hh][c] = v;
    const uint64_t u = nb_uabs(v);
    mq = u > mq ? u : mq;
  }
  mq = imie_wave_max_u64_full(mq);
  if (lane == 0) s_m[wave] = mq;
  __syncthreads();
  if (blockIdx.y == 0 && tid == 0) {                  // the envelope: any group's max|q| breaks it alone
    for (int w = 1; w < 4; ++w) mq = s_m[w] > mq ? s_m[w] : mq;
    if ((u128)mq * a.kv_max[0] * (u128)(uint64_t)a.hd > (u128)INT64_MAX ||
        ((u128)1 << a.fa) * a.kv_max[1] > (u128)INT64_MAX)
      atomicOr(a.status, kGuard);
  }
  const int64_t jbeg = a.first + (int64_t)blockIdx.y * a.chunk, jend = min(jbeg + a.chunk, a.pos + 1);
  const int64_t* kb = a.ck + (int64_t)g.kv * a.max_len * a.hd;
  int64_t best[2] = {INT64_MIN, INT64_MIN};
  const int key4 = l16 >> 2, hA = 2 * (l16 & 3);
  for (int64_t j0 = jbeg; j0 < jend; j0 += 64) {
    longlong2 kk[NIT][4];
#pragma unroll
    for (int it = 0; it < NIT; ++it) {
      const int c = 2 * l16 + 32 * it;
#pragma unroll
      for (int k4 = 0; k4 < 4; ++k4) {                // keys and dims past the end: an in-range duplicate, not used
        const int64_t j = min(j0 + 16 * k4 + grp, a.pos);
        kk[it][k4] = *(const longlong2*)(kb + j * a.hd + (c < a.hd ? c : 0));
      }
    }
    uint64_t acc[4 * kNbHeads];
#pragma unroll
    for (int i = 0; i < 4 * kNbHeads; ++i) acc[i] = 0;
#pragma unroll
    for (int it = 0; it < NIT; ++it)
#pragma unroll
      for (int hh = 0; hh < kNbHeads; ++hh) {
        const longlong2 qv = *(const longlong2*)&s_q[hh][2 * l16 + 32 * it];   // zero past hd
#pragma unroll
        for (int k4 = 0; k4 < 4; ++k4)
          acc[k4 * kNbHeads + hh] += (uint64_t)qv.x * (uint64_t)kk[it][k4].x + (uint64_t)qv.y * (uint64_t)kk[it][k4].y;
      }
    // the 16 lanes' sums, halving the kept set each step: lane l ends with sums 2 l and 2 l + 1 (key 2 l / 8)
#pragma unroll
    for (int n = 2 * kNbHeads, m = 8; m >= 1; n >>= 1, m >>= 1) {
      const bool up = (l16 & m) != 0;
#pragma unroll
      for (int i = 0; i < n; ++i) {
        const uint64_t send = up ? acc[i] : acc[i + n], keep = up ? acc[i + n] : acc[i];
        acc[i] = keep + (uint64_t)__shfl_xor((long long)send, m, 64);
      }
    }
    const int64_t j = j0 + 16 * key4 + grp;
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      if (j >= jend || hA + r >= g.nh) continue;
      const int64_t sh = (int64_t)acc[r] >> a.fa;
      const i128 sc = ((i128)sh * a.inv_sqrt) >> a.fa;
      int64_t score = 0;
      if (sc > (i128)INT64_MAX || sc < (i128)INT64_MIN) atomicOr(a.status, kGuard);
      else score = (int64_t)sc;
      a.prob[(int64_t)(g.h0 + hA + r) * a.max_len + j] = score;
      best[r] = score > best[r] ? score : best[r];
    }
  }
#pragma unroll
  for (int r = 0; r < 2; ++r) {
#pragma unroll
    for (int o = 32; o >= 4; o >>= 1) {               // lanes of one (l16 & 3) hold the same two heads
      const int64_t u = (int64_t)__shfl_xor((long long)best[r], o, 64);
      best[r] = u > best[r] ? u : best[r];
    }
    if (lane < 4) s_b[wave][hA + r] = best[r];
  }
  __syncthreads();
  if (tid < g.nh) {
    int64_t b = s_b[0][tid];
    for (int w = 1; w < 4; ++w) b = s_b[w][tid] > b ? s_b[w][tid] : b;
    a.cmax[(int64_t)blockIdx.y * a.heads + g.h0 + tid] = b;
  }
}

// e_j = 2^-d_j in place of the scores and the chunk's Z; 32 lanes per query head
__global__ __launch_bounds__(256) void nb_exp_kernel(NbAttn a) {
  const NbGroup g = nb_group(a);
  const int hh = threadIdx.x >> 5, l = threadIdx.x & 31;
  const bool live = hh < g.nh;
  const int64_t h = g.h0 + (live ? hh : 0);
  int64_t best = INT64_MIN;
  for (int c = l; c < (int)gridDim.y; c += 32) {
    const int64_t v = a.cmax[(int64_t)c * a.heads + h];
    best = v > best ? v : best;
  }
#pragma unroll
  for (int o = 16; o >= 1; o >>= 1) {
    const int64_t u = (int64_t)__shfl_xor((long long)best, o, 64);
    best = u > best ? u : best;
  }
  const int64_t l2 = nb_log2e(a.fa);
  int64_t dclip = ((int64_t)(a.fa + 2) << (2 * a.fa)) / l2;
  const int64_t hard = ((int64_t)1 << 62) / l2;
  dclip = hard < dclip ? hard : dclip;
  const int64_t jbeg = a.first + (int64_t)blockIdx.y * a.chunk, jend = min(jbeg + a.chunk, a.pos + 1);
  int64_t* ph = a.prob + h * a.max_len;
  uint64_t z = 0;
  if (live)
    for (int64_t j = jbeg + l; j < jend; j += 32) {
      const uint64_t wide = (uint64_t)best - (uint64_t)ph[j];   // best is the row's maximum: exact below 2^64
      const int64_t d = wide > (uint64_t)dclip ? dclip : (int64_t)wide;
      const int64_t e = nb_exp2_neg((int64_t)((uint64_t)d * (uint64_t)l2) >> a.fa, a.fa);
      ph[j] = e;
      z += (uint64_t)e;
    }
#pragma unroll
  for (int o = 16; o >= 1; o >>= 1) z += (uint64_t)__shfl_xor((long long)z, o, 64);
  if (live && l == 0) a.cz[(int64_t)blockIdx.y * a.heads + h] = z;
}

// p_j = (e_j << fa) / Z, staged per 64 keys, and the chunk's PV sums; thread = dim (DPT dims apart by 128) x key half
template <int DPT>
__global__ __launch_bounds__(256) void nb_pv_kernel(NbAttn a) {
  __shared__ __align__(16) uint32_t s_p[64][kNbHeads];   // p <= 2^fa, fa <= 29
  __shared__ uint64_t s_z[kNbHeads];
  __shared__ uint64_t s_sum[128][kNbHeads + 1];
  const NbGroup g = nb_group(a);
  const int tid = threadIdx.x;
  {
    const int hh = tid >> 5, l = tid & 31;
    const int64_t h = g.h0 + (hh < g.nh ? hh : 0);
    uint64_t z = 0;
    for (int c = l; c < (int)gridDim.y; c += 32) z += a.cz[(int64_t)c * a.heads + h];
#pragma unroll
    for (int o = 16; o >= 1; o >>= 1) z += (uint64_t)__shfl_xor((long long)z, o, 64);
    if (l == 0) s_z[hh] = z;
  }
  const int64_t jbeg = a.first + (int64_t)blockIdx.y * a.chunk, jend = min(jbeg + a.chunk, a.pos + 1);
  const int64_t* vb = a.cv + (int64_t)g.kv * a.max_len * a.hd;
  const int d0 = tid & 127, half = tid >> 7;
  uint64_t acc[DPT][kNbHeads];
#pragma unroll
  for (int x = 0; x < DPT; ++x)
#pragma unroll
    for (int hh = 0; hh < kNbHeads; ++hh) acc[x][hh] = 0;
  for (int64_t j0 = jbeg; j0 < jend; j0 += 64) {
    __syncthreads();                                  // the step before is read; s_z is written
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int hh = (tid >> 6) + 4 * i, k = tid & 63;
      uint32_t p = 0;
      if (hh < g.nh && j0 + k < jend) {
        const uint64_t e = (uint64_t)a.prob[(int64_t)(g.h0 + hh) * a.max_len + j0 + k], z = s_z[hh];
        p = z ? (uint32_t)((e << a.fa) / z) : 0;      // e <= 2^fa: e << fa fits
      }
      s_p[k][hh] = p;
    }
    __syncthreads();
    for (int k0 = 32 * half; k0 < 32 * half + 32 && j0 + k0 < jend; k0 += 16) {
      int64_t v[DPT][16];
#pragma unroll
      for (int k = 0; k < 16; ++k)
#pragma unroll
        for (int x = 0; x < DPT; ++x)                 // keys past the end carry p = 0; dims past hd are not stored
          v[x][k] = vb[min(j0 + k0 + k, a.pos) * a.hd + (d0 + 128 * x < a.hd ? d0 + 128 * x : 0)];
#pragma unroll
      for (int k = 0; k < 16; ++k) {
        const uint4 pa = *(const uint4*)&s_p[k0 + k][0], pb = *(const uint4*)&s_p[k0 + k][4];
        const uint32_t p[kNbHeads] = {pa.x, pa.y, pa.z, pa.w, pb.x, pb.y, pb.z, pb.w};
#pragma unroll
        for (int x = 0; x < DPT; ++x)
#pragma unroll
          for (int hh = 0; hh < kNbHeads; ++hh) acc[x][hh] += (uint64_t)p[hh] * (uint64_t)v[x][k];
      }
    }
  }
#pragma unroll
  for (int x = 0; x < DPT; ++x) {
    __syncthreads();
    if (half == 1)
#pragma unroll
      for (int hh = 0; hh < kNbHeads; ++hh) s_sum[d0][hh] = acc[x][hh];
    __syncthreads();
    const int d = d0 + 128 * x;
    if (half == 0 && d < a.hd)
#pragma unroll
      for (int hh = 0; hh < kNbHeads; ++hh)
        if (hh < g.nh)
          a.part[((int64_t)blockIdx.y * a.heads + g.h0 + hh) * a.hd + d] = acc[x][hh] + s_sum[d0][hh];
  }
}

// out = (sum of the chunks' PV sums) >> fa; 64 outputs x 4 chunk quarters per workgroup
__global__ __launch_bounds__(256) void nb_final_kernel(NbAttn a, int nch) {
  __shared__ uint64_t s_p[4][64];
  const int64_t n = (int64_t)a.heads * a.hd, i = (int64_t)blockIdx.x * 64 + (threadIdx.x & 63);
  const int w = threadIdx.x >> 6;
  uint64_t sum = 0;
  if (i < n) {
#pragma unroll 8
    for (int c = w; c < nch; c += 4) sum += a.part[(int64_t)c * n + i];
  }
  s_p[w][threadIdx.x & 63] = sum;
  __syncthreads();
  if (w == 0 && i < n) {
    const int t = threadIdx.x;
    a.out[i] = (int64_t)(s_p[0][t] + s_p[1][t] + s_p[2][t] + s_p[3][t]) >> a.fa;
  }
}

// The same attention for heads wider than the kernels above take (head_dim > kNbMaxHd): one workgroup per query head,
// 128-bit dots, scores in prob (global).
constexpr int kNbMaxHd = 256;
__global__ __launch_bounds__(256) void nb_attention_wide_kernel(NbAttn a) {
  const int64_t *q = a.q, *ck = a.ck, *cv = a.cv;
  const int64_t first = a.first, pos = a.pos, max_len = a.max_len, inv_sqrt = a.inv_sqrt;
  const int heads = a.heads, nkv = a.nkv, hd = a.hd, fa = a.fa;
  const uint64_t* kv_max = a.kv_max;
  int64_t *prob = a.prob, *out = a.out;
  int* status = a.status;
  __shared__ int64_t s_v[4];
  __shared__ uint64_t s_z[4];
  const int head = blockIdx.x, kv = head / (heads / nkv), t = threadIdx.x;
  const int64_t* qh = q + (int64_t)head * hd;
  // envelope (max|q| max|K| hd and 2^fa max|V| within int64): any head's max|q| breaks it alone
  uint64_t mq = 0;
  for (int i = t; i < hd; i += 256) { const uint64_t u = nb_uabs(qh[i]); mq = u > mq ? u : mq; }
  mq = nb_block_max(mq);
  if (t == 0 && ((u128)mq * kv_max[0] * (u128)(uint64_t)hd > (u128)INT64_MAX ||
                 ((u128)1 << fa) * kv_max[1] > (u128)INT64_MAX))
    atomicOr(status, kGuard);
  int64_t* ph = prob + (int64_t)head * max_len;
  int64_t best = INT64_MIN;
  for (int64_t key = first + t; key <= pos; key += 256) {
    const int64_t* kh = ck + ((int64_t)kv * max_len + key) * hd;
    i128 acc = 0;
    for (int l = 0; l < hd; ++l) acc += (i128)qh[l] * kh[l];
    const i128 sh = acc >> fa, sc = (sh * inv_sqrt) >> fa;
    int64_t score = 0;
    if (sh > (i128)INT64_MAX || sh < (i128)INT64_MIN || sc > (i128)INT64_MAX || sc < (i128)INT64_MIN)
      atomicOr(status, kGuard);
    else
      score = (int64_t)sc;
    ph[key] = score;
    best = score > best ? score : best;
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    const int64_t u = (int64_t)__shfl_xor((long long)best, o, 64);
    best = u > best ? u : best;
  }
  if ((t & 63) == 0) s_v[t >> 6] = best;
  __syncthreads();
  best = s_v[0];
  for (int k = 1; k < 4; ++k) best = s_v[k] > best ? s_v[k] : best;
  const int64_t l2 = nb_log2e(fa);
  int64_t dclip = ((int64_t)(fa + 2) << (2 * fa)) / l2;
  const int64_t hard = ((int64_t)1 << 62) / l2;
  dclip = hard < dclip ? hard : dclip;
  uint64_t z = 0;
  for (int64_t key = first + t; key <= pos; key += 256) {
    const i128 wide = (i128)best - ph[key];
    const int64_t d = wide > dclip ? dclip : (wide < 0 ? 0 : (int64_t)wide);
    const int64_t e = nb_exp2_neg((int64_t)((uint64_t)d * (uint64_t)l2) >> fa, fa);
    ph[key] = e;
    z += (uint64_t)e;
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) z += (uint64_t)__shfl_xor((long long)z, o, 64);
  __syncthreads();
  if ((t & 63) == 0) s_z[t >> 6] = z;
  __syncthreads();
  const uint64_t Z = s_z[0] + s_z[1] + s_z[2] + s_z[3];
  if (Z != 0)
    for (int64_t key = first + t; key <= pos; key += 256)
      ph[key] = (int64_t)(((u128)(uint64_t)ph[key] << fa) / (u128)Z);
  __syncthreads();
  for (int l = t; l < hd; l += 256) {
    i128 acc = 0;
    if (Z != 0)
      for (int64_t key = first; key <= pos; ++key) acc += (i128)ph[key] * cv[((int64_t)kv * max_len + key) * hd + l];
    i128 sh = acc >> fa;
    if (sh > (i128)INT64_MAX || sh < (i128)INT64_MIN) { atomicOr(status, kGuard); sh = 0; }
    out[(int64_t)head * hd + l] = (int64_t)sh;
  }
}

struct Binding { long long g = -1, u = -1, d = -1; bool bound = false; };

struct Layer {
  DevBuf k, v, kvmax;                                 // [Hkv][max_len][hd] int64 each; running max|K|, max|V|
  int64_t length = 0;
  bool poisoned = false;
  int experts = 0, used = 0;
  int64_t d_model = 0, e_ffn = 0;
  std::vector<Binding> bind;
  std::vector<int> pending_cold;
};

struct Bank {
  bool live = false;
  int n_layers = 0, heads = 0, nkv = 0, hd = 0, fa = 0;
  int64_t max_len = 0, d_model = 0;
  DevBuf cos, sin;
  std::vector<Layer> layers;
  DevBuf res[2], norm, logits, gates, attn, qkv, ao, prob, part, status, moe;
  int res_slot = 0;
  bool has_res = false;
  bool status_clear = false;                          // the device status word is known to be 0
  char* host = nullptr;                               // pinned: status, ids and hidden row as read back
  size_t host_cap = 0;
  int retained = -1;
  bool pending = false;
  int pending_layer = -1;
  std::vector<int> route_ids;                         // the pending layer's selected experts
};

std::vector<Bank>& banks() {
  static std::vector<Bank> v;
  return v;
}

Bank* bank_get(long long h) {
  if (h < 0 || h >= (long long)banks().size() || !banks()[(size_t)h].live) return nullptr;
  return &banks()[(size_t)h];
}

bool quant_handle(long long h, int64_t* out_f, int64_t* nb) {
  int qt = -1;
  return imie_qk_info(h, out_f, nb, &qt, nullptr) == IMIE_OK && (qt == 0 || qt == 1);
}

int ensure_layer_kv(Bank& b, Layer& L) {
  const size_t bytes = (size_t)(b.nkv * b.max_len * b.hd) * 8;
  if (!L.k.p) {
    if (L.k.ensure(bytes) || L.v.ensure(bytes) || L.kvmax.ensure(16)) return IMIE_EARG;
    IMIE_HIP(hipMemset(L.kvmax.p, 0, 16));
  }
  return IMIE_OK;
}

size_t bank_bytes(const Bank& b) {
  size_t t = b.cos.cap + b.sin.cap;
  for (const DevBuf* d : {&b.res[0], &b.res[1], &b.norm, &b.logits, &b.gates, &b.attn, &b.qkv, &b.ao, &b.prob,
                          &b.part, &b.status, &b.moe})
    t += d->cap;
  for (const Layer& L : b.layers) t += L.k.cap + L.v.cap + L.kvmax.cap;
  return t;
}

void bank_release(Bank& b) {
  (void)hipStreamSynchronize(imie_stream());
  for (Layer& L : b.layers) { L.k.release(); L.v.release(); L.kvmax.release(); }
  for (DevBuf* d : {&b.cos, &b.sin, &b.res[0], &b.res[1], &b.norm, &b.logits, &b.gates, &b.attn, &b.qkv,
                    &b.ao, &b.prob, &b.part, &b.status, &b.moe})
    d->release();
  if (b.host) (void)hipHostFree(b.host);
  b = Bank();
}

// What the host waits for (n 8-byte words), written straight into its pinned buffer: one small launch and one
// synchronisation where a copy into pageable memory takes a staging copy of its own.
__global__ void nb_publish_kernel(const uint64_t* __restrict__ src, int n, uint64_t* __restrict__ dst) {
  for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) dst[i] = src[i];
}

// The bank's status word (b.status), followed by the routed expert ids. It is zero between calls: a call that
// leaves it otherwise poisons its layer, and the next one clears it first (a new allocation too).
constexpr size_t kIdsAt = 64;
int status_ensure(Bank& b, size_t bytes) {
  if (b.status.cap < bytes) b.status_clear = false;
  return b.status.ensure(bytes);
}
size_t published_bytes(const Bank& b, int n_ids, bool row) {
  return (kIdsAt + (size_t)n_ids * 4 + 7) / 8 * 8 + (row ? (size_t)b.d_model * 8 : 0);
}
// The pinned buffer for n_ids ids and a row, reserved before any work is enqueued; where there is no pinned memory,
// finish() reads back through pageable memory.
void host_reserve(Bank& b, int n_ids) {
  const size_t bytes = published_bytes(b, n_ids, true);
  if (b.host_cap >= bytes) return;
  if (b.host) (void)hipHostFree(b.host);
  b.host = nullptr;
  b.host_cap = 0;
  if (hipHostMalloc((void**)&b.host, bytes) == hipSuccess) {
    b.host_cap = bytes;
  } else {
    b.host = nullptr;
    (void)hipGetLastError();                           // no launch is to report it
  }
}
// validate the attention handles / window and reserve the layer's storage (qk_cuda.py:548-572 envelope)
int attention_preflight(Bank& b, int layer, long long qh, long long kh, long long vh, long long oh, int window) {
  if (layer < 0 || layer >= b.n_layers || window == 0 || window < -1) return IMIE_EARG;
  Layer& L = b.layers[(size_t)layer];
  if (L.poisoned || L.length >= b.max_len) return IMIE_EARG;
  const int64_t qw = (int64_t)b.heads * b.hd, kw = (int64_t)b.nkv * b.hd;
  int64_t of[4], nb[4];
  const long long hs[4] = {qh, kh, vh, oh};
  for (int i = 0; i < 4; ++i) if (!quant_handle(hs[i], &of[i], &nb[i])) return IMIE_EARG;
  if (nb[0] * 256 != b.d_model || nb[1] * 256 != b.d_model || nb[2] * 256 != b.d_model || of[0] != qw ||
      of[1] != kw || of[2] != kw || nb[3] * 256 != qw || of[3] != b.d_model)
    return IMIE_EARG;
  host_reserve(b, L.used);
  if (ensure_layer_kv(b, L) || b.qkv.ensure((size_t)(qw + 2 * kw) * 8) || b.attn.ensure((size_t)qw * 8) ||
      b.ao.ensure((size_t)b.d_model * 8) || b.prob.ensure((size_t)(b.heads * b.max_len) * 8) ||
      b.part.ensure((size_t)(kNbMaxChunks * (qw + 2 * b.heads)) * 8) || status_ensure(b, kIdsAt))
    return IMIE_EARG;
  return IMIE_OK;
}

// normalized x (device) -> Q/K/V -> RoPE -> append -> attention -> O into b.ao; enqueued on st (no sync)
int attention_enqueue(Bank& b, int layer, long long qh, long long kh, long long vh, long long oh, const int64_t* x,
                      int fw, int window, int rope, int64_t inv_sqrt, hipStream_t st) {
  Layer& L = b.layers[(size_t)layer];
  const int64_t qw = (int64_t)b.heads * b.hd, kw = (int64_t)b.nkv * b.hd;
  int64_t* q = (int64_t*)b.qkv.p;
  int64_t *k = q + qw, *v = k + kw;
  int* status = (int*)b.status.p;
  const int64_t hs[3] = {qh, kh, vh};
  int64_t* const ys[3] = {q, k, v};
  const int rc = imie_qk_linears_dev(hs, 3, x, fw, ys, status, st);
  if (rc) return rc;
  hipLaunchKernelGGL(nb_rope_append_kernel, dim3((unsigned)(b.heads + b.nkv)), dim3(128), 0, st, q, b.heads,
                     (const int64_t*)k, (const int64_t*)v, b.hd, (const int64_t*)b.cos.p, (const int64_t*)b.sin.p,
                     L.length, b.max_len, b.fa, rope, (int64_t*)L.k.p, (int64_t*)L.v.p, (uint64_t*)L.kvmax.p, status);
  NbAttn a = {};
  a.q = q; a.ck = (const int64_t*)L.k.p; a.cv = (const int64_t*)L.v.p;
  a.pos = L.length; a.first = (window > 0 && a.pos - window >= 0) ? a.pos - window + 1 : 0;
  a.max_len = b.max_len; a.heads = b.heads; a.nkv = b.nkv; a.hd = b.hd; a.fa = b.fa; a.inv_sqrt = inv_sqrt;
  a.kv_max = (const uint64_t*)L.kvmax.p; a.prob = (int64_t*)b.prob.p; a.out = (int64_t*)b.attn.p; a.status = status;
  if (b.hd > kNbMaxHd) {
    hipLaunchKernelGGL(nb_attention_wide_kernel, dim3((unsigned)b.heads), dim3(256), 0, st, a);
  } else {
    // 64-key chunks (one step a workgroup: the shortest chain) until there would be more than kNbMaxChunks of them
    const int64_t steps = (a.pos - a.first + 64) / 64;
    a.chunk = 64 * ((steps + kNbMaxChunks - 1) / kNbMaxChunks);
    const int nch = (int)((a.pos - a.first + a.chunk) / a.chunk);
    a.part = (uint64_t*)b.part.p;
    a.cz = a.part + (int64_t)kNbMaxChunks * qw;
    a.cmax = (int64_t*)(a.cz + (int64_t)kNbMaxChunks * b.heads);
    const int rep = b.heads / b.nkv;
    const dim3 grid((unsigned)(b.nkv * ((rep + kNbHeads - 1) / kNbHeads)), (unsigned)nch);
    if (b.hd <= 128) hipLaunchKernelGGL(nb_scores_kernel<4>, grid, dim3(256), 0, st, a);
    else hipLaunchKernelGGL(nb_scores_kernel<8>, grid, dim3(256), 0, st, a);
    hipLaunchKernelGGL(nb_exp_kernel, grid, dim3(256), 0, st, a);
    if (b.hd <= 128) hipLaunchKernelGGL(nb_pv_kernel<1>, grid, dim3(256), 0, st, a);
    else hipLaunchKernelGGL(nb_pv_kernel<2>, grid, dim3(256), 0, st, a);
    hipLaunchKernelGGL(nb_final_kernel, dim3((unsigned)((qw + 63) / 64)), dim3(256), 0, st, a, nch);
  }
  IMIE_HIP(hipGetLastError());
  return imie_qk_linear_dev(oh, (const int64_t*)b.attn.p, 1, fw, (int64_t*)b.ao.p, status, st);
}

int status_begin(Bank& b, hipStream_t st) {
  if (!b.status_clear) IMIE_HIP(hipMemsetAsync(b.status.p, 0, 4, st));
  b.status_clear = false;
  return IMIE_OK;
}

// status after the enqueued work: 0 ok, 3 a guard fired (layer poisoned), 1 runtime failure; n_ids routed expert ids
// and a hidden row (d_model words of `row`, to `row_out`) come back with it
int finish(Bank& b, Layer& L, hipStream_t st, int n_ids = 0, int* ids = nullptr, const int64_t* row = nullptr,
           int64_t* row_out = nullptr) {
  const size_t head = published_bytes(b, n_ids, false), bytes = published_bytes(b, n_ids, row != nullptr);
  auto fail = [&]() -> int { L.poisoned = true; return IMIE_EARG; };
  std::vector<char> page;
  const char* src = b.host;
  if (b.host_cap >= bytes) {
    hipLaunchKernelGGL(nb_publish_kernel, dim3(1), dim3(256), 0, st, (const uint64_t*)b.status.p, (int)(head / 8),
                       (uint64_t*)b.host);
    if (row)
      hipLaunchKernelGGL(nb_publish_kernel, dim3((unsigned)((b.d_model + 255) / 256)), dim3(256), 0, st,
                         (const uint64_t*)row, (int)b.d_model, (uint64_t*)(b.host + head));
    if (hipGetLastError() != hipSuccess || hipStreamSynchronize(st) != hipSuccess) return fail();
  } else {
    page.resize(bytes);
    src = page.data();
    if (hipMemcpyAsync(page.data(), b.status.p, head, hipMemcpyDeviceToHost, st) != hipSuccess ||
        (row && hipMemcpyAsync(page.data() + head, row, bytes - head, hipMemcpyDeviceToHost, st) != hipSuccess) ||
        hipStreamSynchronize(st) != hipSuccess) {
      (void)hipStreamSynchronize(st);
      return fail();
    }
  }
  int stat = 0;
  memcpy(&stat, src, 4);
  if (stat) { L.poisoned = true; return 3; }
  b.status_clear = true;
  if (n_ids) memcpy(ids, src + kIdsAt, (size_t)n_ids * 4);
  if (row) memcpy(row_out, src + head, (size_t)b.d_model * 8);
  return IMIE_OK;
}

int64_t imie_rmsnorm_eps(unsigned long long eps) { return eps > (unsigned long long)INT64_MAX ? -1 : (int64_t)eps; }

}  // namespace

extern "C" {

// nmc_qk_cuda.cu:1068 `qk_register_i64` (qk_cuda.py:285-303): dense int64 [rows, cols] (norm gains, router)
long long qk_register_i64(const int64_t* W, long long rows, long long cols) {
  std::lock_guard<std::recursive_mutex> lk(imie_lock());
  return imie_qk_register_i64(W, rows, cols);
}

// nmc_qk_cuda.cu:1116 `qk_rmsnorm_router` (qk_cuda.py:331-372): h = RMSNorm(x) with the resident gain, router
// logits, lowest-index top-`used` ids and their sigmoid gates. rc 3: an exact envelope rejection (the caller
// runs its host path); 1: bad arguments.
int qk_rmsnorm_router(long long gain_h, long long router_h, const int64_t* x, long long rows, int fa, int fw,
                      unsigned long long eps, int used, long long h_capacity, long long route_capacity,
                      int64_t* h_out, int* ids_out, int64_t* gates_out) {
  std::lock_guard<std::recursive_mutex> lk(imie_lock());
  int64_t grows = 0, gcols = 0, rrows = 0, rcols = 0;
  int gq = -1, rq = -1;
  const uint8_t *gp = nullptr, *rp = nullptr;
  if (imie_qk_info(gain_h, &grows, &gcols, &gq, &gp) || imie_qk_info(router_h, &rrows, &rcols, &rq, &rp) || !x ||
      !h_out || !ids_out || !gates_out || rows <= 0 || used <= 0 || fa < 1 || fa > 29 || fw < 0 || fw > 62)
    return IMIE_EARG;
  const int64_t e = imie_rmsnorm_eps(eps);
  if (gq != 2 || rq != 2 || grows != 1 || rcols != gcols || rrows <= 0 || rrows > INT_MAX || used > rrows || e < 0 ||
      rows * gcols > h_capacity || rows * used > route_capacity)
    return IMIE_EARG;
  hipStream_t st = imie_stream();
  static DevBuf dx, dh, dl, di, dg, ds;
  const int64_t width = gcols;
  if (dx.ensure((size_t)(rows * width) * 8) || dh.ensure((size_t)(rows * width) * 8) ||
      dl.ensure((size_t)(rows * rrows) * 8) || di.ensure((size_t)(rows * used) * 4) ||
      dg.ensure((size_t)(rows * used) * 8) || ds.ensure(64))
    return IMIE_EARG;
  IMIE_HIP(hipMemcpyAsync(dx.p, x, (size_t)(rows * width) * 8, hipMemcpyHostToDevice, st));
  IMIE_HIP(hipMemsetAsync(ds.p, 0, 4, st));
  int rc = imie_rmsnorm_launch((const int64_t*)dx.p, rows, width, fa, e, (const int64_t*)gp, (int64_t*)dh.p,
                               (int*)ds.p, st);
  if (rc) return rc;
  hipLaunchKernelGGL(nb_router_kernel, dim3((unsigned)rrows, (unsigned)rows), dim3(256), 0, st, (const int64_t*)dh.p,
                     width, (const int64_t*)rp, (int)rrows, fw, (int64_t*)dl.p, (int*)ds.p);
  hipLaunchKernelGGL(nb_topk_kernel, dim3((unsigned)rows), dim3(64), 0, st, (const int64_t*)dl.p, (int)rrows, used,
                     fa, (int*)di.p, (int64_t*)dg.p);
  IMIE_HIP(hipGetLastError());
  int stat = 0;
  IMIE_HIP(hipMemcpyAsync(&stat, ds.p, 4, hipMemcpyDeviceToHost, st));
  IMIE_HIP(hipStreamSynchronize(st));
  if (stat) return 3;
  IMIE_HIP(hipMemcpy(h_out, dh.p, (size_t)(rows * width) * 8, hipMemcpyDeviceToHost));
  IMIE_HIP(hipMemcpy(ids_out, di.p, (size_t)(rows * used) * 4, hipMemcpyDeviceToHost));
  IMIE_HIP(hipMemcpy(gates_out, dg.p, (size_t)(rows * used) * 8, hipMemcpyDeviceToHost));
  return IMIE_OK;
}

// nmc_qk_cuda.cu:877 `qk_attention_bank_create` (qk_cuda.py:486-519): handle >= 0 or -1
long long qk_attention_bank_create(int n_layers, long long max_length, long long d_model, int heads, int n_kv,
                                   int head_dim, int fa, const int64_t* cos, const int64_t* sin) {
  std::lock_guard<std::recursive_mutex> lk(imie_lock());
  if (!cos || !sin || n_layers <= 0 || max_length <= 0 || d_model <= 0 || d_model % 256 || heads <= 0 || n_kv <= 0 ||
      heads % n_kv || head_dim <= 0 || head_dim % 2 || fa < 1 || fa > 29 || ((int64_t)heads * head_dim) % 256 ||
      imie_device_ready() != 0)
    return -1;
  auto& bs = banks();
  size_t slot = bs.size();
  for (size_t i = 0; i < bs.size(); ++i) if (!bs[i].live) { slot = i; break; }
  if (slot == bs.size()) bs.emplace_back();
  Bank& b = bs[slot];
  b = Bank();
  const size_t tb = (size_t)(max_length * (head_dim / 2)) * 8;
  if (b.cos.ensure(tb) || b.sin.ensure(tb) || hipMemcpy(b.cos.p, cos, tb, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(b.sin.p, sin, tb, hipMemcpyHostToDevice) != hipSuccess) {
    bank_release(b);
    return -1;
  }
  b.n_layers = n_layers; b.max_len = max_length; b.d_model = d_model; b.heads = heads; b.nkv = n_kv;
  b.hd = head_dim; b.fa = fa;
  b.layers.resize((size_t)n_layers);
  b.live = true;
  return (long long)slot;
}

// nmc_qk_cuda.cu:914 `qk_attention_bank_reset`
int qk_attention_bank_reset(long long h) {
  std::lock_guard<std::recursive_mutex> lk(imie_lock());
  Bank* b = bank_get(h);
  if (!b) return IMIE_EARG;
  for (Layer& L : b->layers) {
    L.length = 0;
    L.poisoned = false;
    L.pending_cold.clear();
    if (L.kvmax.p) IMIE_HIP(hipMemset(L.kvmax.p, 0, 16));
  }
  b->res_slot = 0; b->has_res = false; b->retained = -1; b->pending = false; b->pending_layer = -1;
  return IMIE_OK;
}

// nmc_qk_cuda.cu:927 `qk_attention_bank_destroy`
void qk_attention_bank_destroy(long long h) {
  std::lock_guard<std::recursive_mutex> lk(imie_lock());
  Bank* b = bank_get(h);
  if (b) bank_release(*b);
}

// nmc_qk_cuda.cu:1363 `qk_attention_bank_import` (qk_cuda.py:528-546): K/V [n_kv, length, head_dim] of a prefill
int qk_attention_bank_import(long long h, int layer, const int64_t* k, const int64_t* v, long long length) {
  std::lock_guard<std::recursive_mutex> lk(imie_lock());
  Bank* b = bank_get(h);
  if (!b || !k || !v || layer < 0 || layer >= b->n_layers || length < 0 || length > b->max_len) return IMIE_EARG;
  Layer& L = b->layers[(size_t)layer];
  if (L.poisoned || ensure_layer_kv(*b, L)) return IMIE_EARG;
  const size_t per = (size_t)(length * b->hd);
  std::vector<uint64_t> mx(2, 0);
  for (int hh = 0; hh < b->nkv; ++hh) {
    const size_t dst = (size_t)(hh * b->max_len * b->hd);
    if (per && (hipMemcpy((int64_t*)L.k.p + dst, k + hh * per, per * 8, hipMemcpyHostToDevice) != hipSuccess ||
                hipMemcpy((int64_t*)L.v.p + dst, v + hh * per, per * 8, hipMemcpyHostToDevice) != hipSuccess)) {
      L.poisoned = true;
      return IMIE_EARG;
    }
    for (size_t i = 0; i < per; ++i) {
      const int64_t a = k[hh * per + i], c = v[hh * per + i];
      const uint64_t ua = a < 0 ? 0 - (uint64_t)a : (uint64_t)a, uc = c < 0 ? 0 - (uint64_t)c : (uint64_t)c;
      mx[0] = ua > mx[0] ? ua : mx[0];
      mx[1] = uc > mx[1] ? uc : mx[1];
    }
  }
  IMIE_HIP(hipMemcpy(L.kvmax.p, mx.data(), 16, hipMemcpyHostToDevice));
  L.length = length;
  return IMIE_OK;
}

// nmc_qk_cuda.cu:1530 `qk_attention_bank_apply` (qk_cuda.py:548-572): the attention sublayer output (after O) of
// one normalized hidden row; rc 3 = an exact guard fired (the layer is poisoned).
int qk_attention_bank_apply(long long h, int layer, long long qh, long long kh, long long vh, long long oh,
                            const int64_t* x, int fw, int window, int rope, int64_t inv_sqrt,
                            long long output_capacity, int64_t* out) {
  std::lock_guard<std::recursive_mutex> lk(imie_lock());
  Bank* b = bank_get(h);
  if (!b || !x || !out || output_capacity < b->d_model || fw < 0 || fw > 62) return IMIE_EARG;
  if (attention_preflight(*b, layer, qh, kh, vh, oh, window)) return IMIE_EARG;
  if (b->norm.ensure((size_t)b->d_model * 8)) return IMIE_EARG;
  hipStream_t st = imie_stream();
  Layer& L = b->layers[(size_t)layer];
  IMIE_HIP(hipMemcpyAsync(b->norm.p, x, (size_t)b->d_model * 8, hipMemcpyHostToDevice, st));
  int rc = status_begin(*b, st);
  if (rc) return rc;
  rc = attention_enqueue(*b, layer, qh, kh, vh, oh, (const int64_t*)b->norm.p, fw, window, rope, inv_sqrt, st);
  if (rc) { (void)hipStreamSynchronize(st); L.poisoned = true; return IMIE_EARG; }
  if ((rc = finish(*b, L, st, 0, nullptr, (const int64_t*)b->ao.p, out))) return rc;
  ++L.length;
  return IMIE_OK;
}

// nmc_qk_cuda.cu:935 `qk_attention_bank_moe_configure` (qk_cuda.py:574-595): per-layer expert metadata only
int qk_attention_bank_moe_configure(long long h, int layer, int experts, int used, long long d_model,
                                    long long expert_ffn) {
  std::lock_guard<std::recursive_mutex> lk(imie_lock());
  Bank* b = bank_get(h);
  if (!b || layer < 0 || experts <= 0 || used <= 0 || used > experts || d_model <= 0 || expert_ffn <= 0 ||
      d_model % 256 || expert_ffn % 256)
    return IMIE_EARG;
  if (layer >= b->n_layers || d_model != b->d_model || b->pending) return IMIE_EARG;
  Layer& L = b->layers[(size_t)layer];
  if (L.poisoned) return IMIE_EARG;
  if (L.experts)
    return (L.experts == experts && L.used == used && L.d_model == d_model && L.e_ffn == expert_ffn) ? IMIE_OK
                                                                                                     : IMIE_EARG;
  L.experts = experts; L.used = used; L.d_model = d_model; L.e_ffn = expert_ffn;
  L.bind.assign((size_t)experts, Binding());
  L.pending_cold.clear();
  return IMIE_OK;
}

// nmc_qk_cuda.cu:984 `qk_attention_bank_moe_bind` (qk_cuda.py:597-614): one resident expert triplet
int qk_attention_bank_moe_bind(long long h, int layer, int expert, long long gate_h, long long up_h,
                               long long down_h) {
  std::lock_guard<std::recursive_mutex> lk(imie_lock());
  Bank* b = bank_get(h);
  if (!b || layer < 0 || layer >= b->n_layers) return IMIE_EARG;
  Layer& L = b->layers[(size_t)layer];
  if (L.poisoned || expert < 0 || expert >= L.experts) return IMIE_EARG;
  int64_t gof, gnb, uof, unb, dof, dnb;
  if (!quant_handle(gate_h, &gof, &gnb) || !quant_handle(up_h, &uof, &unb) || !quant_handle(down_h, &dof, &dnb))
    return IMIE_EARG;
  if (gof != L.e_ffn || gnb != L.d_model / 256 || uof != L.e_ffn || unb != L.d_model / 256 || dof != L.d_model ||
      dnb != L.e_ffn / 256)
    return IMIE_EARG;
  Binding& bd = L.bind[(size_t)expert];
  if (bd.bound && (bd.g != gate_h || bd.u != up_h || bd.d != down_h)) return IMIE_EARG;
  bd.g = gate_h; bd.u = up_h; bd.d = down_h; bd.bound = true;
  if (b->pending && b->pending_layer == layer)
    for (size_t i = 0; i < L.pending_cold.size(); ++i)
      if (L.pending_cold[i] == expert) { L.pending_cold.erase(L.pending_cold.begin() + (long)i); break; }
  return IMIE_OK;
}

// nmc_qk_cuda.cu:1557 `qk_attention_bank_moe_begin` (qk_cuda.py:616-660): RMSNorm + router + top-k and the
// attention sublayer of one layer, retained on the device; returns the selected experts not yet bound (in
// selected order, without repeats). x is the host hidden row unless use_retained (the previous continuation's).
int qk_attention_bank_moe_begin(long long h, int layer, long long gain_h, long long router_h, long long qh,
                                long long kh, long long vh, long long oh, const int64_t* x, int use_retained, int fw,
                                unsigned long long eps, int window, int rope, int64_t inv_sqrt, int cold_capacity,
                                int* cold_count_out, int* cold_ids_out) {
  std::lock_guard<std::recursive_mutex> lk(imie_lock());
  Bank* b = bank_get(h);
  if (!b || layer < 0 || !cold_count_out || !cold_ids_out || use_retained < 0 || use_retained > 1 || fw < 0 ||
      fw > 62 || window == 0 || window < -1)
    return IMIE_EARG;
  if (layer >= b->n_layers || b->pending) return IMIE_EARG;
  Layer& L = b->layers[(size_t)layer];
  int64_t grows, gcols, rrows, rcols;
  int gq = -1, rq = -1;
  const uint8_t *gp = nullptr, *rp = nullptr;
  if (imie_qk_info(gain_h, &grows, &gcols, &gq, &gp) || imie_qk_info(router_h, &rrows, &rcols, &rq, &rp))
    return IMIE_EARG;
  const int64_t e = imie_rmsnorm_eps(eps);
  if (L.poisoned || L.experts <= 0 || !L.pending_cold.empty() || cold_capacity < L.used || gq != 2 || rq != 2 ||
      grows != 1 || gcols != L.d_model || rrows != L.experts || rcols != L.d_model || e < 0)
    return IMIE_EARG;
  if ((!use_retained && !x) || (use_retained && (!b->has_res || b->retained + 1 != layer))) return IMIE_EARG;
  if (attention_preflight(*b, layer, qh, kh, vh, oh, window)) return IMIE_EARG;
  const size_t dm = (size_t)L.d_model;
  if (b->res[0].ensure(dm * 8) || b->res[1].ensure(dm * 8) || b->norm.ensure(dm * 8) ||
      b->logits.ensure((size_t)L.experts * 8) || status_ensure(*b, kIdsAt + (size_t)(L.used + 1) * 4) ||
      b->gates.ensure((size_t)L.used * 8) || b->moe.ensure(dm * 8))
    return IMIE_EARG;
  hipStream_t st = imie_stream();
  if (!use_retained) {
    IMIE_HIP(hipMemcpyAsync(b->res[0].p, x, dm * 8, hipMemcpyHostToDevice, st));
    b->res_slot = 0;
  }
  const int64_t* resid = (const int64_t*)b->res[b->res_slot].p;
  int* status = (int*)b->status.p;
  int* ids = (int*)((char*)b->status.p + kIdsAt);
  int rc = status_begin(*b, st);
  if (rc) return rc;
  rc = imie_rmsnorm_launch(resid, 1, L.d_model, b->fa, e, (const int64_t*)gp, (int64_t*)b->norm.p, status, st);
  if (rc) return rc;
  hipLaunchKernelGGL(nb_router_kernel, dim3((unsigned)L.experts, 1), dim3(256), 0, st, (const int64_t*)b->norm.p,
                     L.d_model, (const int64_t*)rp, L.experts, fw, (int64_t*)b->logits.p, status);
  hipLaunchKernelGGL(nb_topk_kernel, dim3(1), dim3(64), 0, st, (const int64_t*)b->logits.p, L.experts, L.used,
                     b->fa, ids, (int64_t*)b->gates.p);
  IMIE_HIP(hipGetLastError());
  rc = attention_enqueue(*b, layer, qh, kh, vh, oh, (const int64_t*)b->norm.p, fw, window, rope, inv_sqrt, st);
  if (rc) { (void)hipStreamSynchronize(st); L.poisoned = true; return IMIE_EARG; }
  b->route_ids.assign((size_t)L.used, -1);
  if ((rc = finish(*b, L, st, L.used, b->route_ids.data()))) return rc;
  std::vector<int> cold;
  for (int id : b->route_ids) {
    if (id < 0 || id >= L.experts) { L.poisoned = true; return 3; }
    if (L.bind[(size_t)id].bound) continue;
    bool dup = false;
    for (int c : cold) dup = dup || c == id;
    if (!dup) cold.push_back(id);
  }
  for (size_t i = 0; i < cold.size(); ++i) cold_ids_out[i] = cold[i];
  *cold_count_out = (int)cold.size();
  L.pending_cold = cold;
  ++L.length;
  b->has_res = true; b->pending = true; b->pending_layer = layer;
  return IMIE_OK;
}

// nmc_qk_cuda.cu:1658 `qk_attention_bank_moe_continue` (qk_cuda.py:662-686): the selected experts' MoE and the
// parallel residual x + attention + MoE, retained (publish = 0) or also copied out. rc 4: a selected expert is
// still unbound; rc 3: an envelope guard fired.
int qk_attention_bank_moe_continue(long long h, int layer, int fw, int publish, long long output_capacity,
                                   int64_t* out) {
  std::lock_guard<std::recursive_mutex> lk(imie_lock());
  Bank* b = bank_get(h);
  if (!b || layer < 0 || fw < 0 || fw > 62 || publish < 0 || publish > 1 || (publish && (!out || output_capacity <= 0)))
    return IMIE_EARG;
  if (layer >= b->n_layers || !b->pending || b->pending_layer != layer) return IMIE_EARG;
  Layer& L = b->layers[(size_t)layer];
  if (L.poisoned || L.experts <= 0 || (publish && output_capacity < L.d_model)) return IMIE_EARG;
  if (!L.pending_cold.empty()) return 4;
  std::vector<long long> gh, uh, dh;
  for (int id : b->route_ids) {
    const Binding& bd = L.bind[(size_t)id];
    if (!bd.bound) return 4;
    gh.push_back(bd.g); uh.push_back(bd.u); dh.push_back(bd.d);
  }
  hipStream_t st = imie_stream();
  const int next = b->res_slot ^ 1;
  int rc = status_begin(*b, st);
  if (rc) return rc;
  rc = imie_qk_moe_dev(gh.data(), uh.data(), dh.data(), L.used, (const int64_t*)b->norm.p, (const int64_t*)b->gates.p,
                       L.d_model, L.e_ffn, b->fa, fw, (const int64_t*)b->res[b->res_slot].p, (const int64_t*)b->ao.p,
                       (int64_t*)b->moe.p, (int64_t*)b->res[next].p, (int*)b->status.p, st);
  if (rc) { (void)hipStreamSynchronize(st); L.poisoned = true; return IMIE_EARG; }
  if ((rc = finish(*b, L, st, 0, nullptr, publish ? (const int64_t*)b->res[next].p : nullptr, out))) return rc;
  b->res_slot = next; b->has_res = true; b->retained = layer; b->pending = false; b->pending_layer = -1;
  return IMIE_OK;
}

// nmc_qk_cuda.cu:1748 `qk_attention_bank_moe_export` (qk_cuda.py:688-699): the retained residual row
int qk_attention_bank_moe_export(long long h, long long output_capacity, int64_t* out) {
  std::lock_guard<std::recursive_mutex> lk(imie_lock());
  Bank* b = bank_get(h);
  if (!b || !out || b->pending || !b->has_res || b->retained < 0 || output_capacity < b->d_model) return IMIE_EARG;
  IMIE_HIP(hipMemcpy(out, b->res[b->res_slot].p, (size_t)b->d_model * 8, hipMemcpyDeviceToHost));
  return IMIE_OK;
}

// nmc_qk_cuda.cu:1765 `qk_attention_bank_workspace_bytes`: device bytes owned by the bank (2^64 - 1 if invalid)
unsigned long long qk_attention_bank_workspace_bytes(long long h) {
  std::lock_guard<std::recursive_mutex> lk(imie_lock());
  Bank* b = bank_get(h);
  return b ? (unsigned long long)bank_bytes(*b) : ~0ull;
}

}  // extern "C"
