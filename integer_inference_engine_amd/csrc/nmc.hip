// north-mini-code Q4_K / Q6_K integer linear and the ragged grouped MoE FFN for gfx950.
//
// Semantics (reference: north-mini-code/src/nmc/qk_codec.py:28-206, cohere2.py:102-111, :168-188; producer
// north-mini-code/tools/nmc_qk_cuda.cu:92-237, :2184-2254):
//   y[t, o] = floor( sum_i W[o, i] * x[t, i] / 2^fw )   exactly (big-int in the oracle), W = dequantized block
//   Q4_K (144 B): W = dq*sc_j*q - dmq*m_j, sub-blocks of 32; Q6_K (210 B): W = dq*sc_j*(q6 - 32), sub-blocks of 16
//   dq = round_half_even(fp16 * 2^fw) from the fp16 bits in integer arithmetic (exact; no libm, no FP rounding).
// Evaluation: per sub-block j, sum_i W x = (dq*sc_j) * qdot_j - (dmq*m_j) * xsum_j with qdot_j = sum q*x in
// int64 (|x| < 2^52 keeps it exact; larger staged values take an int128 path), the products and the running sum in
// int128. A result that does not fit int64 (the oracle's astype would raise) sets status bit 2.
//
// Work: a workgroup = (weight group, 64-row tile); the x rows routed to that weight are staged block by block in
// LDS (16 rows per pass) and 4 threads per output row each own a quarter of them, so every weight block is read
// from HBM once per call no matter how many tokens use it.
#include "imie_common.h"
#include "imie_kernels.h"
#include "imie_silu.h"
#include <string.h>
#include <stdlib.h>
#include <algorithm>
#include <map>
#include <tuple>

namespace {

typedef __int128 i128;
constexpr int kRows = 64;        // output rows per workgroup
constexpr int kXRows = 16;       // staged x rows per pass (4 per thread)
// dq * sc * q must fit int64 for every finite fp16 scale (as the oracle's int64 weight arrays require)
constexpr int kMaxFw = 36;

struct QKWeight {
  uint8_t* p = nullptr;
  int64_t out_f = 0, nb = 0;
  int qtype = 0;
  size_t bytes = 0;
};
std::vector<QKWeight> g_qk;
int64_t g_qk_live = 0;

// profile counters (qk_cuda.py:24-34 metric order)
enum { PM_REG_CALLS, PM_REG_NS, PM_H2D_CALLS, PM_H2D_BYTES, PM_H2D_NS, PM_D2H_CALLS, PM_D2H_BYTES, PM_D2H_NS,
       PM_ALLOC_CALLS, PM_ALLOC_BYTES, PM_ALLOC_NS, PM_FREE_CALLS, PM_NATIVE_CALLS, PM_RESIDENT_CALLS,
       PM_GROUPED_CALLS, PM_MOE_CALLS, PM_MOE_BATCHED_CALLS, PM_MOE_BATCHED_DP4A_CALLS, PM_Q_CALLS, PM_Q_NS,
       PM_K_CALLS, PM_K_NS, PM_V_CALLS, PM_V_NS, PM_O_CALLS, PM_O_NS, PM_OTHER_CALLS, PM_OTHER_NS, PM_COUNT };
unsigned long long g_prof[PM_COUNT];
int g_prof_on = 0;
inline void prof(int k, unsigned long long v = 1) { if (g_prof_on) g_prof[k] += v; }

struct MoeWs {
  DevBuf items, pairs, x, y, g, u, d, out, gates, status, tok;
  int64_t grows = 0;
} g_mws;

// round(fp16 h * 2^fw) to the nearest integer, ties to even, without branches (lanes of different rows take different
// exponents): a normal h is (1024 + mant) 2^(e - 25), a subnormal mant 2^-24. A left shift (sh >= 0) is exact; the right
// shift's rounding is done by the float unit: m 2^sh is exact in single precision (m < 2^11) and rint rounds it half to
// even. Exponent 31 is treated as finite.
__device__ inline int64_t fp16_fixed_fast(uint32_t h, int fw) {
  const uint32_t e = (h >> 10) & 31, mant = h & 0x3FF;
  const uint32_t m = e == 0 ? mant : (mant | 0x400);
  const int sh = (e == 0 ? 1 : (int)e) - 25 + fw;
  const int64_t up = (int64_t)((uint64_t)m << (sh > 0 ? sh : 0));
  const int64_t dn = (int64_t)(uint32_t)__builtin_rintf(__builtin_ldexpf((float)m, sh < 0 ? sh : 0));
  const int64_t r = sh >= 0 ? up : dn;
  return ((h >> 15) & 1) ? -r : r;
}

__global__ void fp16_fixed_probe_kernel(const uint16_t* __restrict__ h, int64_t n, int fw, int64_t* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) out[i] = fp16_fixed_fast(h[i], fw);
}

struct Item {               // one weight applied to `count` x rows
  const uint8_t* w;
  int64_t out_f, nb;
  int qtype;
  int first, count;         // into the pair arrays
};

// y[yi[p]][o] = floor(W[o] . x[xi[p]] / 2^fw) for the pairs of one item.
// run_gate (nullable): the launch runs only when *run_gate != 0 (the MFMA path found activations it cannot take)
// One (64-row tile bx, item by) of the exact int128 kernel; every thread of the workgroup calls it with the same
// (bx, by).
__device__ void qk_group_tile(const Item* __restrict__ items, const int* __restrict__ xi, const int* __restrict__ yi,
                              const int64_t* __restrict__ X, int64_t K, int64_t* __restrict__ Y, int64_t ldy, int fw,
                              int* __restrict__ status, int64_t bx, int64_t by) {
  __shared__ int64_t sx[kXRows][257];
  __shared__ int s_wide;
  const Item it = items[by];
  const int64_t o = bx * kRows + (threadIdx.x >> 2);
  if (bx * kRows >= it.out_f) return;
  const int slot = threadIdx.x & 3;
  const bool live = o < it.out_f;
  const int bs = it.qtype == 0 ? 144 : 210;
  const uint8_t* row = it.w + (live ? o : 0) * it.nb * bs;
  for (int c0 = 0; c0 < it.count; c0 += kXRows) {
    const int cn = min(kXRows, it.count - c0);
    i128 acc[4] = {0, 0, 0, 0};
    for (int64_t b = 0; b < it.nb; ++b) {
      __syncthreads();
      if (threadIdx.x == 0) s_wide = 0;
      __syncthreads();
      int wide = 0;
      for (int i = threadIdx.x; i < cn * 256; i += blockDim.x) {
        const int r = i >> 8, c = i & 255;
        const int64_t v = X[(int64_t)xi[it.first + c0 + r] * K + b * 256 + c];
        sx[r][c] = v;
        if (v >= ((int64_t)1 << 52) || v <= -((int64_t)1 << 52)) wide = 1;
      }
      if (wide) s_wide = 1;
      __syncthreads();
      const bool fast = s_wide == 0;
      const uint8_t* blk = row + b * bs;
      if (it.qtype == 0) {
        const int64_t dq = fp16_fixed_fast(blk[0] | (blk[1] << 8), fw), dmq = fp16_fixed_fast(blk[2] | (blk[3] << 8), fw);
        const uint8_t* sc = blk + 4;
        const uint8_t* qs = blk + 16;
#pragma unroll 1
        for (int j = 0; j < 8; ++j) {
          int s, m;
          if (j < 4) { s = sc[j] & 63; m = sc[j + 4] & 63; }
          else { s = (sc[j + 4] & 0xF) | ((sc[j - 4] >> 6) << 4); m = (sc[j + 4] >> 4) | ((sc[j] >> 6) << 4); }
          const int64_t ds = dq * s, dm = dmq * m;
          const int g = j >> 1, hi = j & 1;
          uint8_t q[32];
#pragma unroll
          for (int l = 0; l < 32; ++l) q[l] = hi ? (qs[32 * g + l] >> 4) : (qs[32 * g + l] & 0xF);
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const int r = slot + 4 * k;
            if (r >= cn) break;
            const int64_t* xv = &sx[r][32 * j];
            if (fast) {
              int64_t qd = 0, xs = 0;
#pragma unroll
              for (int l = 0; l < 32; ++l) { qd += (int64_t)q[l] * xv[l]; xs += xv[l]; }
              acc[k] += (i128)ds * qd - (i128)dm * xs;
            } else {
              i128 qd = 0, xs = 0;
              for (int l = 0; l < 32; ++l) { qd += (i128)q[l] * xv[l]; xs += xv[l]; }
              acc[k] += (i128)ds * qd - (i128)dm * xs;
            }
          }
        }
      } else {
        const uint8_t* ql = blk;
        const uint8_t* qh = blk + 128;
        const int8_t* sc = (const int8_t*)(blk + 192);
        const int64_t dq = fp16_fixed_fast(blk[208] | (blk[209] << 8), fw);
#pragma unroll 1
        for (int j = 0; j < 16; ++j) {
          // sub-block j covers positions 16 j .. 16 j + 15: half = j / 8, quarter qq = (j % 8) / 2, is = j % 2
          const int half = j >> 3, qq = (j & 7) >> 1, is = j & 1;
          const int qlo = 64 * half, qho = 32 * half;
          const int64_t ds = dq * sc[8 * half + is + 2 * qq];
          int8_t q[16];
#pragma unroll
          for (int l0 = 0; l0 < 16; ++l0) {
            const int l = 16 * is + l0;
            int v;
            if (qq == 0) v = (ql[qlo + l] & 0xF) | (((qh[qho + l] >> 0) & 3) << 4);
            else if (qq == 1) v = (ql[qlo + l + 32] & 0xF) | (((qh[qho + l] >> 2) & 3) << 4);
            else if (qq == 2) v = (ql[qlo + l] >> 4) | (((qh[qho + l] >> 4) & 3) << 4);
            else v = (ql[qlo + l + 32] >> 4) | (((qh[qho + l] >> 6) & 3) << 4);
            q[l0] = (int8_t)(v - 32);
          }
          const int pos0 = 128 * half + 32 * qq + 16 * is;
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const int r = slot + 4 * k;
            if (r >= cn) break;
            const int64_t* xv = &sx[r][pos0];
            if (fast) {
              int64_t qd = 0;
#pragma unroll
              for (int l = 0; l < 16; ++l) qd += (int64_t)q[l] * xv[l];
              acc[k] += (i128)ds * qd;
            } else {
              i128 qd = 0;
              for (int l = 0; l < 16; ++l) qd += (i128)q[l] * xv[l];
              acc[k] += (i128)ds * qd;
            }
          }
        }
      }
    }
    if (live) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int r = slot + 4 * k;
        if (r >= cn) break;
        const i128 y = acc[k] >> fw;
        if (y > (i128)INT64_MAX || y < (i128)INT64_MIN) atomicOr(status, IMIE_EOVF);
        Y[(int64_t)yi[it.first + c0 + r] * ldy + o] = (int64_t)y;
      }
    }
  }
}

__global__ __launch_bounds__(256) void qk_group_kernel(const Item* __restrict__ items, const int* __restrict__ xi,
                                                       const int* __restrict__ yi, const int64_t* __restrict__ X,
                                                       int64_t K, int64_t* __restrict__ Y, int64_t ldy, int fw,
                                                       int* __restrict__ status, const int* __restrict__ run_gate) {
  if (run_gate && *run_gate == 0) return;
  qk_group_tile(items, xi, yi, X, K, Y, ldy, fw, status, blockIdx.x, blockIdx.y);
}

// The exact kernel as the fallback of a fused MoE stage: a small grid that ends at once unless the prep flagged a
// wide activation row (*run_gate != 0); then its workgroups walk all (tile, item) pairs, ntx tiles per item.
constexpr int kGatedWgs = 128;
__global__ __launch_bounds__(256) void qk_group_gated_kernel(const Item* __restrict__ items, const int* __restrict__ xi,
                                                             const int* __restrict__ yi, const int64_t* __restrict__ X,
                                                             int64_t K, int64_t* __restrict__ Y, int64_t ldy, int fw,
                                                             int* __restrict__ status, const int* __restrict__ run_gate,
                                                             int64_t ntx, int64_t ne) {
  if (*run_gate == 0) return;
  for (int64_t t = blockIdx.x; t < ntx * ne; t += gridDim.x) {
    qk_group_tile(items, xi, yi, X, K, Y, ldy, fw, status, t % ntx, t / ntx);
    __syncthreads();                                  // the tile's shared buffers are free for the next one
  }
}

// nmc SiLU*up: g <- ((g * sigmoid(g)) >> fa) exactly, then gu = (g * u) >> fa exactly (cohere2.py:109-111,
// :183-185); sigmoid without the (1<<62)/log2e cap (north-mini-code/src/nmc/_bonsai/fixedpoint.py:148).
__device__ inline int64_t exp2_neg_fixed(int64_t u, int frac) {
  const int64_t fp = (int64_t)1 << frac;
  const int64_t k = u >> frac, f = u & (fp - 1);
  const int sh = 16 - frac;
  int64_t c0, c1, c2, c3;
  if (sh >= 0) { c0 = 65536 >> sh; c1 = 45426 >> sh; c2 = 15743 >> sh; c3 = 3638 >> sh; }
  else { c0 = (int64_t)65536 << -sh; c1 = (int64_t)45426 << -sh; c2 = (int64_t)15743 << -sh; c3 = (int64_t)3638 << -sh; }
  const int64_t f2 = (int64_t)((uint64_t)f * (uint64_t)f) >> frac;
  const int64_t f3 = (int64_t)((uint64_t)f2 * (uint64_t)f) >> frac;
  int64_t poly = c0 - ((int64_t)((uint64_t)c1 * (uint64_t)f) >> frac) + ((int64_t)((uint64_t)c2 * (uint64_t)f2) >> frac) -
                 ((int64_t)((uint64_t)c3 * (uint64_t)f3) >> frac);
  if (poly < 0) poly = 0;
  if (k < 0) return 0;
  return poly >> (k < 63 ? k : 63);
}

// (silu(x) * u) >> fa in int128 with the int64 range checks (status bit 2)
__device__ inline int64_t qk_silu_elem(int64_t x, int64_t u, int fa, int64_t log2e, int64_t dclip, int* status) {
  const int64_t m = x > 0 ? x : 0;
  int64_t d0 = m, d1 = (int64_t)((uint64_t)m - (uint64_t)x);
  if (d0 > dclip) d0 = dclip;
  if (d1 > dclip) d1 = dclip;
  const int64_t e0 = exp2_neg_fixed((int64_t)((uint64_t)d0 * (uint64_t)log2e) >> fa, fa);
  const int64_t e1 = exp2_neg_fixed((int64_t)((uint64_t)d1 * (uint64_t)log2e) >> fa, fa);
  const int64_t z = e0 + e1;
  const int64_t sig = z == 0 ? 0 : (int64_t)(((uint64_t)e1 << fa) / (uint64_t)z);
  const i128 s = ((i128)x * sig) >> fa;
  if (s > (i128)INT64_MAX || s < (i128)INT64_MIN) atomicOr(status, IMIE_EOVF);
  const i128 gu = ((i128)(int64_t)s * u) >> fa;
  if (gu > (i128)INT64_MAX || gu < (i128)INT64_MIN) atomicOr(status, IMIE_EOVF);
  return (int64_t)gu;
}

__global__ void qk_silu_mul_kernel(const int64_t* __restrict__ g, const int64_t* __restrict__ u, int64_t n, int fa,
                                   int64_t log2e, int64_t dclip, int64_t* __restrict__ out, int* __restrict__ status,
                                   const int* __restrict__ run_gate = nullptr) {
  if (run_gate && *run_gate == 0) return;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    out[i] = qk_silu_elem(g[i], u[i], fa, log2e, dclip, status);
}

// The exact gate and up kernels and SiLU * up as the fallback of the fused gate/up stage, in one launch: a small
// grid that ends at once unless the prep flagged a wide activation row; then each workgroup takes (tile, item)
// pairs, computes the gate tile and the up tile and turns its own tile's elements into silu(gate) * up.
constexpr int kGatedWgs2 = 128;
__global__ __launch_bounds__(256) void qk_gateup_gated_kernel(const Item* __restrict__ ig, const Item* __restrict__ iu,
                                                              const int* __restrict__ xi, const int* __restrict__ yi,
                                                              const int64_t* __restrict__ X, int64_t K,
                                                              int64_t* __restrict__ gb, int64_t* __restrict__ ub,
                                                              int64_t ldy, int fw, int fa, int64_t log2e,
                                                              int64_t dclip, int* __restrict__ status,
                                                              const int* __restrict__ run_gate, int64_t ntx,
                                                              int64_t ne) {
  if (*run_gate == 0) return;
  for (int64_t t = blockIdx.x; t < ntx * ne; t += gridDim.x) {
    const int64_t bx = t % ntx, by = t / ntx;
    qk_group_tile(ig, xi, yi, X, K, gb, ldy, fw, status, bx, by);
    __syncthreads();
    qk_group_tile(iu, xi, yi, X, K, ub, ldy, fw, status, bx, by);
    __threadfence_block();
    __syncthreads();                                  // both tiles written (and the shared buffers free)
    const Item it = ig[by];
    const int64_t o0 = bx * kRows, no = it.out_f - o0 < kRows ? it.out_f - o0 : kRows;
    if (no > 0)
      for (int64_t e = threadIdx.x; e < (int64_t)it.count * no; e += blockDim.x) {
        const int64_t idx = (int64_t)yi[it.first + e / no] * ldy + o0 + e % no;
        gb[idx] = qk_silu_elem(gb[idx], ub[idx], fa, log2e, dclip, status);
      }
    __syncthreads();
  }
}

// out[t][o] = sum_j (dd[t*k + j][o] * gates[t*k + j]) >> fa (exact; cohere2.py:187 then astype int64)
// flags (optional): the fused MoE's two wide-row flags, cleared here, after their last reader, for the next call
__global__ void qk_combine_kernel(const int64_t* __restrict__ dd, int m, int k, int64_t d_model,
                                  const int64_t* __restrict__ gates, int fa, int64_t* __restrict__ out,
                                  int* __restrict__ status, int* __restrict__ flags = nullptr) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (flags && idx < 2) flags[idx] = 0;
  if (idx >= (int64_t)m * d_model) return;
  const int64_t t = idx / d_model, o = idx % d_model;
  i128 acc = 0;
  for (int j = 0; j < k; ++j) acc += ((i128)dd[(t * k + j) * d_model + o] * gates[t * k + j]) >> fa;
  if (acc > (i128)INT64_MAX || acc < (i128)INT64_MIN) atomicOr(status, IMIE_EOVF);
  out[idx] = (int64_t)acc;
}

// out = residual + attention + moe, int64 wrap (the reference's committed numpy int64 addition); the MoE's status
// bits join the layer's
__global__ void qk_add3_kernel(const int64_t* __restrict__ a, const int64_t* __restrict__ b,
                               const int64_t* __restrict__ c, int64_t n, int64_t* __restrict__ out,
                               const int* __restrict__ moe_status, int* __restrict__ status) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = (int64_t)((uint64_t)a[i] + (uint64_t)b[i] + (uint64_t)c[i]);
  if (i == 0 && *moe_status) atomicOr(status, *moe_status);
}

// ---------------------------------------------------------------------------------------------------------
// int8-MFMA path (v_mfma_i32_16x16x32_i8, tokens in M, weight rows in N, one sub-block per K = 32 step):
//   prep  : the activation rows' balanced base-256 digit planes xd[l][row][K] (l < kQkLimbs), the sums of every
//           16 consecutive activations xs16[row][K / 16], and a flag when a row needs more than kQkLimbs limbs
//   Q4_K  : qdot_j = sum_l 256^l D_l with D_l = MFMA(digits_l(x), q) over sub-block j (32 positions, q in 0..15),
//           S1 = sum_j sc_j qdot_j, S2 = sum_j m_j xsum_j (int64: |x| <= 127 (256^5 - 1) / 255 keeps
//           |qdot| < 2^48, |S1| < 2^57, |S2| < 2^53), then acc += dq S1 - dmq S2 (int128) per 256-block
//   Q6_K  : the same with q6 - 32 as int8, sub-blocks of 16 (two MFMAs per 32 positions, each with the other
//           sub-block's K groups zeroed in A), no min term (|S1| < 2^59)
//   y = acc >> fw, refused (status bit 2) outside int64, as the VALU path.
// MFMA operands: A lane l = token l % 16, K group l / 16 (8 bytes); B lane l = weight row l % 16, K group l / 16;
// D lane l holds tokens 4 (l / 16) + r of row l % 16.
// ---------------------------------------------------------------------------------------------------------
constexpr int kQkLimbs = 5;

__global__ __launch_bounds__(256) void qk_prep_kernel(const int64_t* __restrict__ X, int64_t rows, int64_t K,
                                                      int8_t* __restrict__ xd, int64_t* __restrict__ xs16,
                                                      int* __restrict__ Lrow, int* __restrict__ wide) {
  __shared__ uint64_t s_mx[4];
  const int64_t r = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  uint64_t mx = 0;
  // eight consecutive activations per thread: their digits of each limb plane packed into one 64-bit store
  for (int64_t c0 = 8 * (int64_t)tid; c0 < K; c0 += 8 * 256) {
    if (c0 + 8 <= K) {
      int64_t v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = X[r * K + c0 + e];
      // the digits of a value are the bytes of one add and one xor; limbs 0..3 by byte transposes, limb 4 gathered
      uint64_t pk[kQkLimbs];
      uint32_t lo[8], hi[8], ta[4], tb[4];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const uint64_t a = imie_absu64(v[e]), dg = imie_digits64((uint64_t)v[e]);
        mx = a > mx ? a : mx;
        lo[e] = (uint32_t)dg;
        hi[e] = (uint32_t)(dg >> 32);
      }
      imie_bytes4x4(lo[0], lo[1], lo[2], lo[3], ta);
      imie_bytes4x4(lo[4], lo[5], lo[6], lo[7], tb);
#pragma unroll
      for (int l = 0; l < 4; ++l) pk[l] = ((uint64_t)tb[l] << 32) | ta[l];
      imie_bytes4x4(hi[0], hi[1], hi[2], hi[3], ta);
      imie_bytes4x4(hi[4], hi[5], hi[6], hi[7], tb);
      pk[4] = ((uint64_t)tb[0] << 32) | ta[0];
      static_assert(kQkLimbs == 5, "limb 4 is the first of the high halves");
#pragma unroll
      for (int l = 0; l < kQkLimbs; ++l) *(uint64_t*)&xd[((int64_t)l * rows + r) * K + c0] = pk[l];
    } else {
      for (int64_t c = c0; c < K; ++c) {
        int64_t v = X[r * K + c];
        const uint64_t a = imie_absu64(v);
        mx = a > mx ? a : mx;
#pragma unroll
        for (int l = 0; l < kQkLimbs; ++l) {
          const int64_t dg = ((v + 128) & 255) - 128;
          v = (int64_t)((uint64_t)v - (uint64_t)dg) >> 8;
          xd[((int64_t)l * rows + r) * K + c] = (int8_t)dg;
        }
      }
    }
  }
  // sums of 16 consecutive activations (thread per group; callers whose kernels read no sums pass none)
  for (int64_t gq = tid; xs16 && gq < K / 16; gq += 256) {
    int64_t sm = 0;
#pragma unroll
    for (int e = 0; e < 16; ++e) sm = (int64_t)((uint64_t)sm + (uint64_t)X[r * K + 16 * gq + e]);
    xs16[r * (K / 16) + gq] = sm;
  }
  mx = imie_wave_max_u64_full(mx);
  if (lane == 0) s_mx[wave] = mx;
  __syncthreads();
  if (tid == 0) {
    uint64_t m = s_mx[0];
    for (int w = 1; w < 4; ++w) m = s_mx[w] > m ? s_mx[w] : m;
    const bool fits = m <= imie_balanced_cap(kQkLimbs);
    Lrow[r] = fits ? imie_limbs_needed(m) : kQkLimbs;
    if (!fits) atomicOr(wide, 1);
  }
}

__global__ void qk_flag_reset_kernel(int* f) { *f = 0; }

__device__ inline v4i mfma32(int64_t a, int64_t b, v4i c) {
  return __builtin_amdgcn_mfma_i32_16x16x32_i8((long)a, (long)b, c, 0, 0, 0);
}

template <int QT>
__global__ __launch_bounds__(256) void qk_mfma_kernel(const Item* __restrict__ items, const int* __restrict__ xi,
                                                      const int* __restrict__ yi, const int8_t* __restrict__ xd,
                                                      const int64_t* __restrict__ xs16, const int* __restrict__ Lrow,
                                                      int64_t rows, int64_t K, int64_t* __restrict__ Y, int64_t ldy,
                                                      int fw, int* __restrict__ status, const int* __restrict__ wide,
                                                      int dot4_max) {
  if (*wide) return;                                  // the VALU kernel takes this call
  const Item it = items[blockIdx.y];
  if (it.qtype != QT || it.count <= dot4_max) return; // small items: qk_dot4_kernel
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int n = lane & 15, kg = lane >> 4;
  const int64_t o = (int64_t)blockIdx.x * 64 + wave * 16 + n;
  if ((int64_t)blockIdx.x * 64 + wave * 16 >= it.out_f) return;
  const bool orow = o < it.out_f;
  constexpr int BS = QT == 0 ? 144 : 210;
  const uint8_t* wrow = it.w + (orow ? o : 0) * it.nb * BS;
  const int64_t K16 = K / 16;
  for (int c0 = 0; c0 < it.count; c0 += 16) {
    // A rows: token c0 + n of the item (zero past the item's count)
    const bool arow = c0 + n < it.count;
    const int64_t xr = arow ? xi[it.first + c0 + n] : 0;
    int La = arow ? Lrow[xr] : 1;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) { const int t = __shfl_xor(La, off, 64); La = t > La ? t : La; }
    const int L = La;                                 // limbs of this token tile (wave-uniform)
    // D rows: tokens c0 + 4 kg + q
    int64_t drow[4];
    bool dlive[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      dlive[q] = c0 + 4 * kg + q < it.count;
      drow[q] = dlive[q] ? xi[it.first + c0 + 4 * kg + q] : 0;
    }
    i128 acc[4] = {0, 0, 0, 0};
    for (int64_t b = 0; b < it.nb; ++b) {
      const uint8_t* blk = wrow + b * BS;
      int64_t S1[4] = {0, 0, 0, 0}, S2[4] = {0, 0, 0, 0};
      if (QT == 0) {
        const int64_t dq = fp16_fixed_fast(blk[0] | (blk[1] << 8), fw), dmq = fp16_fixed_fast(blk[2] | (blk[3] << 8), fw);
        const uint8_t* scb = blk + 4;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const uint2 qv = *(const uint2*)(blk + 16 + 32 * g + 8 * kg);
#pragma unroll
          for (int hi = 0; hi < 2; ++hi) {
            const int j = 2 * g + hi;
            const uint32_t b0 = hi ? (qv.x >> 4) & 0x0F0F0F0Fu : qv.x & 0x0F0F0F0Fu;
            const uint32_t b1 = hi ? (qv.y >> 4) & 0x0F0F0F0Fu : qv.y & 0x0F0F0F0Fu;
            const int64_t bq = (int64_t)(((uint64_t)b1 << 32) | b0);
            const int64_t pos = b * 256 + 32 * j + 8 * kg;
            int64_t qdot[4] = {0, 0, 0, 0};
#pragma unroll
            for (int l = 0; l < kQkLimbs; ++l) {
              if (l >= L) break;
              const int64_t av = arow ? *(const int64_t*)(xd + ((int64_t)l * rows + xr) * K + pos) : 0;
              const v4i d = mfma32(av, bq, v4i{0, 0, 0, 0});
#pragma unroll
              for (int q = 0; q < 4; ++q) qdot[q] += (int64_t)d[q] << (8 * l);
            }
            int sc, mn;
            if (j < 4) { sc = scb[j] & 63; mn = scb[j + 4] & 63; }
            else { sc = (scb[j + 4] & 0xF) | ((scb[j - 4] >> 6) << 4); mn = (scb[j + 4] >> 4) | ((scb[j] >> 6) << 4); }
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              const int64_t xs = xs16[drow[q] * K16 + (b * 256 + 32 * j) / 16] + xs16[drow[q] * K16 + (b * 256 + 32 * j) / 16 + 1];
              S1[q] += (int64_t)sc * qdot[q];
              S2[q] += (int64_t)mn * xs;
            }
          }
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[q] += (i128)dq * S1[q] - (i128)dmq * S2[q];
      } else {
        const uint8_t* ql = blk;
        const uint8_t* qh = blk + 128;
        const int8_t* scs = (const int8_t*)(blk + 192);
        const int64_t dq = fp16_fixed_fast(blk[208] | (blk[209] << 8), fw);
#pragma unroll
        for (int half = 0; half < 2; ++half)
#pragma unroll
          for (int qq = 0; qq < 4; ++qq) {
            // 32 positions 128 half + 32 qq + (0..31): lane K group kg takes 8 kg .. 8 kg + 7 (sub-block is = kg / 2)
            const uint2 lv = *(const uint2*)(ql + 64 * half + ((qq & 1) ? 32 : 0) + 8 * kg);
            const uint2 hv = *(const uint2*)(qh + 32 * half + 8 * kg);
            const int sl = qq >= 2 ? 4 : 0, sh = 2 * qq;
            uint32_t v0 = ((lv.x >> sl) & 0x0F0F0F0Fu) | (((hv.x >> sh) & 0x03030303u) << 4);
            uint32_t v1 = ((lv.y >> sl) & 0x0F0F0F0Fu) | (((hv.y >> sh) & 0x03030303u) << 4);
            v0 = ((v0 | 0x80808080u) - 0x20202020u) ^ 0x80808080u;   // bytewise q6 - 32 as int8
            v1 = ((v1 | 0x80808080u) - 0x20202020u) ^ 0x80808080u;
            const int64_t bq = (int64_t)(((uint64_t)v1 << 32) | v0);
            const int64_t pos = b * 256 + 128 * half + 32 * qq + 8 * kg;
            int64_t qd0[4] = {0, 0, 0, 0}, qd1[4] = {0, 0, 0, 0};
#pragma unroll
            for (int l = 0; l < kQkLimbs; ++l) {
              if (l >= L) break;
              const int64_t av = arow ? *(const int64_t*)(xd + ((int64_t)l * rows + xr) * K + pos) : 0;
              const v4i d0 = mfma32(kg < 2 ? av : 0, bq, v4i{0, 0, 0, 0});
              const v4i d1 = mfma32(kg < 2 ? 0 : av, bq, v4i{0, 0, 0, 0});
#pragma unroll
              for (int q = 0; q < 4; ++q) {
                qd0[q] += (int64_t)d0[q] << (8 * l);
                qd1[q] += (int64_t)d1[q] << (8 * l);
              }
            }
            const int s0 = scs[8 * half + 2 * qq], s1 = scs[8 * half + 2 * qq + 1];
#pragma unroll
            for (int q = 0; q < 4; ++q) S1[q] += (int64_t)s0 * qd0[q] + (int64_t)s1 * qd1[q];
          }
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[q] += (i128)dq * S1[q];
      }
    }
    if (orow) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        if (!dlive[q]) continue;
        const i128 y = acc[q] >> fw;
        if (y > (i128)INT64_MAX || y < (i128)INT64_MIN) atomicOr(status, IMIE_EOVF);
        Y[(int64_t)yi[it.first + c0 + 4 * kg + q] * ldy + o] = (int64_t)y;
      }
    }
  }
}

// v_dot4_i32_i8 path for items with few tokens (the MoE experts: ~4 tokens each), every token of the item once
// (no 16-row MFMA padding). Workgroup = (item, 64 weight rows); thread = (row, quarter q of each 256-block):
//   Q4_K: q covers qs bytes 32 q .. 32 q + 31, i.e. sub-blocks 2q (low nibbles) and 2q + 1 (high nibbles)
//   Q6_K: q = (half, pair of quarters qq): sub-blocks 8 half + 2 qq + is for qq in {2 (q & 1), 2 (q & 1) + 1}
// The weights are expanded to int8 once per block; per token and limb, 16 dot4s give the sub-block dot products.
// The 256-block's digits of up to 8 tokens are staged in LDS. Partial int128 sums of the 4 quarter-threads of a
// row are added by shuffles at the end (integer addition: order-free).
constexpr int kDotTok = 8;

__device__ inline i128 shfl_xor_i128(i128 v, int m) {
  const uint64_t lo = (uint64_t)v, hi = (uint64_t)((unsigned __int128)v >> 64);
  const uint64_t lo2 = (uint64_t)__shfl_xor((long long)lo, m, 64), hi2 = (uint64_t)__shfl_xor((long long)hi, m, 64);
  return (i128)(((unsigned __int128)hi2 << 64) | lo2);
}

template <int QT>
__global__ __launch_bounds__(256) void qk_dot4_kernel(const Item* __restrict__ items, const int* __restrict__ xi,
                                                      const int* __restrict__ yi, const int8_t* __restrict__ xd,
                                                      const int64_t* __restrict__ xs16, const int* __restrict__ Lrow,
                                                      int64_t rows, int64_t K, int64_t* __restrict__ Y, int64_t ldy,
                                                      int fw, int* __restrict__ status, const int* __restrict__ wide,
                                                      int maxcount) {
  __shared__ __align__(16) int8_t sx[kQkLimbs][kDotTok][256];
  __shared__ int64_t sxs[kDotTok][16];
  __shared__ int s_L;
  if (*wide) return;
  const Item it = items[blockIdx.y];
  if (it.qtype != QT || it.count > maxcount) return;
  const int tid = threadIdx.x, q = tid & 3;
  const int64_t o = (int64_t)blockIdx.x * 64 + (tid >> 2);
  if ((int64_t)blockIdx.x * 64 >= it.out_f) return;
  const bool orow = o < it.out_f;
  constexpr int BS = QT == 0 ? 144 : 210;
  const uint8_t* wrow = it.w + (orow ? o : 0) * it.nb * BS;
  const int64_t K16 = K / 16;
  for (int t0 = 0; t0 < it.count; t0 += kDotTok) {
    const int tn = min(kDotTok, it.count - t0);
    if (tid == 0) {
      int L = 1;
      for (int t = 0; t < tn; ++t) { const int lr = Lrow[xi[it.first + t0 + t]]; L = lr > L ? lr : L; }
      s_L = L;
    }
    __syncthreads();
    const int L = s_L;
    i128 acc[kDotTok];
#pragma unroll
    for (int t = 0; t < kDotTok; ++t) acc[t] = 0;
    for (int64_t b = 0; b < it.nb; ++b) {
      // stage the block's digits (L limbs x tn tokens x 256 bytes, 16 B per thread-step) and 16-sums
      for (int i = tid; i < L * tn * 16; i += 256) {
        const int l = i / (tn * 16), rem = i % (tn * 16), t = rem >> 4, c = rem & 15;
        const int64_t xr = xi[it.first + t0 + t];
        *(uint4*)&sx[l][t][16 * c] = *(const uint4*)(xd + ((int64_t)l * rows + xr) * K + b * 256 + 16 * c);
      }
      if (tid < tn * 16) {
        const int t = tid >> 4, c = tid & 15;
        sxs[t][c] = xs16[(int64_t)xi[it.first + t0 + t] * K16 + b * 16 + c];
      }
      __syncthreads();
      const uint8_t* blk = wrow + b * BS;
      if (QT == 0) {
        const int64_t dq = fp16_fixed_fast(blk[0] | (blk[1] << 8), fw), dmq = fp16_fixed_fast(blk[2] | (blk[3] << 8), fw);
        const uint8_t* scb = blk + 4;
        const uint4 qa = *(const uint4*)(blk + 16 + 32 * q), qb = *(const uint4*)(blk + 32 + 32 * q);
        const uint32_t qd[8] = {qa.x, qa.y, qa.z, qa.w, qb.x, qb.y, qb.z, qb.w};
        int wl[8], wh[8];
#pragma unroll
        for (int d = 0; d < 8; ++d) { wl[d] = (int)(qd[d] & 0x0F0F0F0Fu); wh[d] = (int)((qd[d] >> 4) & 0x0F0F0F0Fu); }
        int sc[2], mn[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int j = 2 * q + h;
          if (j < 4) { sc[h] = scb[j] & 63; mn[h] = scb[j + 4] & 63; }
          else { sc[h] = (scb[j + 4] & 0xF) | ((scb[j - 4] >> 6) << 4); mn[h] = (scb[j + 4] >> 4) | ((scb[j] >> 6) << 4); }
        }
#pragma unroll
        for (int t = 0; t < kDotTok; ++t) {
          if (t >= tn) break;
          int64_t qlo = 0, qhi = 0;
          for (int l = 0; l < L; ++l) {
            const int* xl = (const int*)&sx[l][t][64 * q];
            const int* xh = (const int*)&sx[l][t][64 * q + 32];
            int al = 0, ah = 0;
#pragma unroll
            for (int d = 0; d < 8; ++d) {
              al = __builtin_amdgcn_sdot4(xl[d], wl[d], al, false);
              ah = __builtin_amdgcn_sdot4(xh[d], wh[d], ah, false);
            }
            qlo += (int64_t)al << (8 * l);
            qhi += (int64_t)ah << (8 * l);
          }
          const int64_t S1 = (int64_t)sc[0] * qlo + (int64_t)sc[1] * qhi;
          const int64_t S2 = (int64_t)mn[0] * (sxs[t][4 * q] + sxs[t][4 * q + 1]) +
                             (int64_t)mn[1] * (sxs[t][4 * q + 2] + sxs[t][4 * q + 3]);
          acc[t] += (i128)dq * S1 - (i128)dmq * S2;
        }
      } else {
        const int half = q >> 1, qq0 = 2 * (q & 1);
        const uint8_t* ql = blk + 64 * half;
        const uint8_t* qh = blk + 128 + 32 * half;
        const int8_t* scs = (const int8_t*)(blk + 192);
        const int64_t dq = fp16_fixed_fast(blk[208] | (blk[209] << 8), fw);
        const uint4 l0 = *(const uint4*)ql, l1 = *(const uint4*)(ql + 16), l2 = *(const uint4*)(ql + 32),
                    l3 = *(const uint4*)(ql + 48);
        const uint4 h0 = *(const uint4*)qh, h1 = *(const uint4*)(qh + 16);
        const uint32_t lq[16] = {l0.x, l0.y, l0.z, l0.w, l1.x, l1.y, l1.z, l1.w, l2.x, l2.y, l2.z, l2.w, l3.x, l3.y, l3.z, l3.w};
        const uint32_t hq[8] = {h0.x, h0.y, h0.z, h0.w, h1.x, h1.y, h1.z, h1.w};
        const int sl = (q & 1) ? 4 : 0;
        int w[2][8];                                  // [qq - qq0][dword of the 32 positions]
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const int qq = qq0 + u;
#pragma unroll
          for (int d = 0; d < 8; ++d) {
            uint32_t v = ((lq[((qq & 1) ? 8 : 0) + d] >> sl) & 0x0F0F0F0Fu) | (((hq[d] >> (2 * qq)) & 0x03030303u) << 4);
            v = ((v | 0x80808080u) - 0x20202020u) ^ 0x80808080u;   // bytewise q6 - 32 as int8
            w[u][d] = (int)v;
          }
        }
        int sc[2][2];
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int is = 0; is < 2; ++is) sc[u][is] = scs[8 * half + 2 * (qq0 + u) + is];
#pragma unroll
        for (int t = 0; t < kDotTok; ++t) {
          if (t >= tn) break;
          int64_t qs4[2][2] = {{0, 0}, {0, 0}};
          for (int l = 0; l < L; ++l) {
#pragma unroll
            for (int u = 0; u < 2; ++u) {
              const int* xp = (const int*)&sx[l][t][128 * half + 32 * (qq0 + u)];
              int a0 = 0, a1 = 0;
#pragma unroll
              for (int d = 0; d < 4; ++d) {
                a0 = __builtin_amdgcn_sdot4(xp[d], w[u][d], a0, false);
                a1 = __builtin_amdgcn_sdot4(xp[4 + d], w[u][4 + d], a1, false);
              }
              qs4[u][0] += (int64_t)a0 << (8 * l);
              qs4[u][1] += (int64_t)a1 << (8 * l);
            }
          }
          const int64_t S1 = (int64_t)sc[0][0] * qs4[0][0] + (int64_t)sc[0][1] * qs4[0][1] +
                             (int64_t)sc[1][0] * qs4[1][0] + (int64_t)sc[1][1] * qs4[1][1];
          acc[t] += (i128)dq * S1;
        }
      }
      __syncthreads();
    }
#pragma unroll
    for (int t = 0; t < kDotTok; ++t) {
      if (t >= tn) break;
      i128 v = acc[t];
      v += shfl_xor_i128(v, 1);
      v += shfl_xor_i128(v, 2);
      if (q == 0 && orow) {
        const i128 y = v >> fw;
        if (y > (i128)INT64_MAX || y < (i128)INT64_MIN) atomicOr(status, IMIE_EOVF);
        Y[(int64_t)yi[it.first + t0 + t] * ldy + o] = (int64_t)y;
      }
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------------------------------------
// Fused MoE expert kernels (the batched MoE of cohere2.py:168-188 with Q4_K gate/up and Q6_K down, the
// north-mini-code layout): one item per expert = its gate/up/down weights and the (token, pair) list routed to it.
//   moe_gateup : g = gate . h, u = up . h (the same activation operands feed both), then gu = (silu(g) * u) >> fa
//                in the epilogue (the exact arithmetic of qk_silu_mul_kernel), written per pair
//   moe_down   : d = down . gu per pair
// int8 MFMA v_mfma_i32_16x16x32_i8 with the MFMA M rows = (token t, digit limb l) = 4 t + l: four tokens of up to
// four balanced base-256 limbs per MFMA (a second MFMA takes limbs 4..7), weight rows in N, one sub-block (Q4_K:
// 32 positions; Q6_K: 16, the other half of the K groups zeroed in A) per K = 32 step. D lane (t, n) then holds
// the limb partial sums of token t for weight row n, recombined in place (no cross-lane traffic) into the
// sub-block dot q.x per limb. Per block and limb T = sum_j sc_j D_j and M = sum_j m_j xsum_j stay in int32, and the
// limb's 64-bit sum takes dq T - dmq M by two 32 x 32 + 64 multiply-adds; the four limbs meet in 128 bits once a row.
// That needs |dq|, |dmq| within a bound that keeps the sums below 2^63 (moe_dq_max: 2^31 - 1 up to 129 blocks of Q4_K,
// 17 of Q6_K); a block beyond it adds its products to a 128-bit sum instead. MFMA sums are exact: |D| <= 32 * 128 * 128.
// Up to eight tokens share one walk over the weights: two 16-row groups hold tokens 0..3 and 4..7 (at most four limbs)
// or limbs 0..3 and 4..7 of four tokens, and every block's decode (scales, mins, quants) feeds both groups' MFMAs. A
// group's digits are staged in LDS kMoeChunk blocks at a time; the block loop between has
// no barrier, and the next block's weights are in flight while a block computes.
// Bound by VALU issue, most of it the block decode: about four tokens meet an expert in a batch of 64.
// gate/up: workgroup = (64 weight rows, item), wave = 16 rows. down, whose rows are a few blocks long: workgroup =
// (one or two times 64 weight rows, item), the digits staged once for all of them.
// The kernels run a few rounds of workgroups, so their code is kept short and in one copy (group count at run time): a
// cold workgroup waits on instruction fetches (the same walk with a copy per group count and two blocks ahead: 113 us).
// Measured, 64 tokens, 8 of 128 experts, 2048 -> 768 -> 2048, against 64 x 64 -> 128 products a block, scales decoded
// one by one and 64 rows a workgroup: gate / up 98 -> 89 us, down 93 -> 83 us (the weights alone: 31 and 23 us).
// ---------------------------------------------------------------------------------------------------------
constexpr int kMoeTok = 4;         // tokens per MFMA row group (4 tokens x 4 limbs = 16 rows)
constexpr int kMoeChunk = 8;       // blocks staged at a time
// 16-row tiles of a down wave: two share a workgroup's start and staging where that leaves eight workgroups a CU (64
// tokens: 92.8 us before, 82.5 with two, 84.9 with four), else one (5 tokens, 36 experts: two cost 3 us a call)
constexpr int kMoeDownWgs = 2048;
// LDS row stride of the staged digits: the staged length + 16 bytes (a multiple of 256, + 16). A lane of row r (of the
// 16 (token, limb) rows) and K group kg reads 8 bytes at r stride + 8 kg + 32 j, i.e. 8-byte slot 2 r + kg (mod 32): the
// 32 lanes of a half-wave hit 32 distinct slots (without the 16 bytes all 16 rows of a K group shared one slot: 16-way
// bank conflicts).
// staging for rows of nb blocks: 32 rows x a chunk, and 256 zero bytes
__host__ __device__ inline int moe_chunk(int nb) { return nb < kMoeChunk ? nb : kMoeChunk; }
__host__ __device__ inline size_t moe_lds_bytes(int nb) { return (size_t)32 * (256 * moe_chunk(nb) + 16) + 256; }
// the largest |dq|, |dmq| for which nb blocks' |dq T| + |dmq M| stay below 2^63 (tmax >= |T| + |M|, resp. |T|) and the
// factor fits int32
constexpr int64_t kMoeT4 = (int64_t)8 * 63 * (32 * 128 * 15 + 32 * 128);
constexpr int64_t kMoeT6 = (int64_t)16 * 128 * (16 * 128 * 128);
__host__ __device__ inline int64_t moe_dq_max(int64_t nb, int64_t tmax) {
  const int64_t m = INT64_MAX / (nb * tmax);
  return m < INT32_MAX ? m : INT32_MAX;
}

struct MoeItem {
  const uint8_t* wg;        // gate (Q4_K), up (Q4_K), down (Q6_K) of the expert
  const uint8_t* wu;
  const uint8_t* wd;
  int first, count;         // into the pair arrays: ptok (activation row of h), ppair (gu / d row)
};

struct Acc128 {             // two's-complement 128-bit accumulator
  uint64_t lo;
  int64_t hi;
};

__device__ inline void acc_madd(Acc128& a, int64_t x, int64_t y) {
  const uint64_t pl = (uint64_t)x * (uint64_t)y;
  const int64_t ph = __mul64hi(x, y);
  a.lo += pl;
  a.hi += ph + (a.lo < pl ? 1 : 0);
}

// floor(acc / 2^fw) and whether it fits int64 (0 <= fw < 64)
__device__ inline int64_t acc_shift(Acc128 a, int fw, bool* fits) {
  const i128 v = (i128)(((unsigned __int128)(uint64_t)a.hi << 64) | a.lo);
  const i128 y = v >> fw;
  *fits = y <= (i128)INT64_MAX && y >= (i128)INT64_MIN;
  return (int64_t)y;
}

// exact nmc SiLU * up of one element (qk_silu_mul_kernel): false when an intermediate leaves int64. The sigmoid is the
// one-exponential form (one of the two clipped exponents is 0), the same values as the two-exponential one there.
__device__ inline int64_t nmc_silu_mul(int64_t x, int64_t u, int fa, int64_t log2e, int64_t dclip, bool* ok) {
  const int64_t sig = imie_silu::sigmoid_fixed_fast(x, fa, log2e, dclip);
  const i128 s = ((i128)x * sig) >> fa;
  bool good = s <= (i128)INT64_MAX && s >= (i128)INT64_MIN;
  const i128 gu = ((i128)(int64_t)s * u) >> fa;
  good = good && gu <= (i128)INT64_MAX && gu >= (i128)INT64_MIN;
  *ok = good;
  return (int64_t)gu;
}

// the rows of one walk: up to eight tokens' activation rows, absent ones repeating the last
struct MoeRows {
  int row[2 * kMoeTok];
  int tn, L;                // tokens taken, limbs of the widest
  bool two, hi;             // two 16-row groups; the second holds limbs 4..7 (else tokens 4..7)
};
// the walk that begins at sel[0] with n pairs left: eight tokens of at most four limbs, or four
__device__ inline MoeRows moe_rows(const int* __restrict__ sel, const int* __restrict__ Lrow, int n) {
  MoeRows r;
  int lr[2 * kMoeTok];
#pragma unroll
  for (int i = 0; i < 2 * kMoeTok; ++i) r.row[i] = sel[i < n ? i : n - 1];   // two load rounds, all issued at once
#pragma unroll
  for (int i = 0; i < 2 * kMoeTok; ++i) lr[i] = Lrow[r.row[i]];
  int l4 = 1, l8 = 1;
#pragma unroll
  for (int i = 0; i < 2 * kMoeTok; ++i) {
    l8 = lr[i] > l8 ? lr[i] : l8;
    if (i < kMoeTok) l4 = l8;
  }
  r.tn = min(n, l8 <= 4 ? 2 * kMoeTok : kMoeTok);
  r.L = r.tn > kMoeTok ? l8 : l4;
  r.hi = r.L > 4;
  r.two = r.hi || r.tn > kMoeTok;
  return r;
}

// Stage the digits of blocks b0 .. b0 + cn into LDS rows at stride kp: row 16 g + 4 l + t holds token 4 g + t, limb l (hi:
// token t, limb 4 g + l), in chunks of 16 bytes (thread: chunk tid % 16 of a (block, row)), the loads of four per thread
// issued before their stores. Rows of absent tokens or limbs are written as zeros, so the MFMA A operands need no
// selects. The caller synchronizes before (buffer free) and after (rows visible).
__device__ inline void moe_stage(int8_t* sx, const MoeRows& w, int b0, int cn, int kp, const int8_t* __restrict__ xd,
                                 int64_t rows, int64_t K, int tid, int nt) {
  const int lgr = w.two ? 5 : 4, total = cn << lgr, c = 16 * (tid & 15);
  for (int j0 = tid >> 4; j0 < total; j0 += 4 * (nt >> 4)) {
    uint4 v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int j = j0 + u * (nt >> 4);
      const int r = j & ((1 << lgr) - 1), b = j >> lgr;
      const int l = ((r >> 2) & 3) + (w.hi ? 4 * (r >> 4) : 0), tok = (r & 3) + (w.hi ? 0 : 4 * (r >> 4));
      const bool on = j < total && tok < w.tn && l < w.L;
      int pr = w.row[0];
#pragma unroll
      for (int q = 1; q < 2 * kMoeTok; ++q) pr = tok == q ? w.row[q] : pr;
      v[u] = on ? *(const uint4*)(xd + ((int64_t)l * rows + pr) * K + 256 * (int64_t)(b0 + b) + c) : uint4{0, 0, 0, 0};
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int j = j0 + u * (nt >> 4);
      if (j < total) *(uint4*)(sx + (j & ((1 << lgr) - 1)) * kp + 256 * (j >> lgr) + c) = v[u];
    }
  }
}

// A (token, row)'s sums: per limb in 64 bits; what blocks beyond moe_dq_max add, in 128 bits in memory (rare, and not
// touched before the wave meets such a block: a scratch load would wait for the weights in flight)
struct MoeSum {
  int64_t v[4];
};
struct MoeFactor {          // a block's dq or dmq: exact where ok, else fp16_fixed_fast has it in 64 bits
  int f;
  bool ok;
};
// fp16_fixed_fast in 32 bits (m 2^sh with sh <= 20: single precision holds it exactly either way, so one ldexp and rint
// serve both directions of the shift), without a branch
__device__ inline MoeFactor moe_factor(uint32_t h, int fw, int64_t dqmax) {
  const uint32_t e = (h >> 10) & 31, mant = h & 0x3FF;
  const int sh = (e == 0 ? 1 : (int)e) - 25 + fw;
  const float m = (float)(e == 0 ? mant : (mant | 0x400));
  const int r = (int)__builtin_rintf(__builtin_ldexpf(m, sh < 20 ? sh : 20));
  return {((h >> 15) & 1) ? -r : r, sh <= 20 && r <= (int)dqmax};
}
__device__ inline int64_t limb_sum(v4i d) {           // sum_r d[r] 256^r
  return (int64_t)d[0] + ((int64_t)d[1] << 8) + ((int64_t)d[2] << 16) + ((int64_t)d[3] << 24);
}
__device__ inline void moe_wide_begin(Acc128 (&w)[2], bool& any) {
  if (any) return;                                    // wave-uniform
  w[0] = w[1] = Acc128{0, 0};
  any = true;
}
__device__ __attribute__((noinline)) void moe_wide_add(Acc128* w, uint32_t h, int fw, bool neg, v4i t) {
  const int64_t f = fp16_fixed_fast(h, fw);
  acc_madd(*w, neg ? -f : f, limb_sum(t));
}
__device__ inline i128 moe_total(const MoeSum& s, const Acc128& w, bool any) {
  i128 t = 0;
#pragma unroll
  for (int l = 3; l >= 0; --l) t = (i128)((unsigned __int128)t << 8) + s.v[l];
  if (any) t += (i128)(((unsigned __int128)(uint64_t)w.hi << 64) | w.lo);
  return t;
}
__device__ inline int64_t moe_result(i128 t, int fw, bool* fits) {
  const i128 y = t >> fw;
  *fits = y <= (i128)INT64_MAX && y >= (i128)INT64_MIN;
  return (int64_t)y;
}

// No load in flight (after a staging there is none anyway): the compiler's count of them at a block loop's entry is then
// the loop's own, so it waits for a block's weights and not for whatever the staging may have left.
__device__ inline void moe_settle() { __builtin_amdgcn_s_waitcnt(0x0F70); }   // vmcnt(0)

// The lane's A operand: limb l of token t (row m = 4 t + l of the MFMA), K group kg: byte offset of [l][t][8 kg].
__device__ inline int moe_a_lane(int lane, int kp) {
  const int m = lane & 15, kg = lane >> 4, t = m >> 2, l = m & 3;
  return (l * kMoeTok + t) * kp + 8 * kg;
}
__device__ inline int64_t moe_a(const int8_t* p, int p0) { return *(const int64_t*)(p + p0); }

// Q4_K weights of one block for B lanes (row n, K group kg): the 16-byte header (d, dmin, 12 scale bytes) and the
// qs bytes 32 g + 8 kg .. + 7 for g = 0..3 (sub-blocks 2 g (low nibbles), 2 g + 1 (high nibbles))
struct Q4Lane {
  uint4 h;
  uint2 q[4];
};
// Loads of weight bytes through global-address-space pointers of native vector types. The item pointers come from
// memory, so plain loads through them are flat loads, which count against the LDS counter as well: every LDS wait
// in the block compute would then also wait for the next block's weights in flight.
typedef unsigned gv4u __attribute__((ext_vector_type(4)));
typedef unsigned gv2u __attribute__((ext_vector_type(2)));
template <typename T>
__device__ inline T gload(const uint8_t* p);
template <>
__device__ inline uint4 gload<uint4>(const uint8_t* p) {
  const gv4u v = *(__attribute__((address_space(1))) const gv4u*)p;
  return uint4{v.x, v.y, v.z, v.w};
}
template <>
__device__ inline uint2 gload<uint2>(const uint8_t* p) {
  const gv2u v = *(__attribute__((address_space(1))) const gv2u*)p;
  return uint2{v.x, v.y};
}
template <>
__device__ inline uint8_t gload<uint8_t>(const uint8_t* p) {
  return *(__attribute__((address_space(1))) const uint8_t*)p;
}
template <>
__device__ inline uint16_t gload<uint16_t>(const uint8_t* p) {
  return *(__attribute__((address_space(1))) const uint16_t*)p;
}
__device__ inline Q4Lane q4_lane_load(const uint8_t* blk, int kg) {
  Q4Lane r;
  r.h = gload<uint4>(blk);
#pragma unroll
  for (int g = 0; g < 4; ++g) r.q[g] = gload<uint2>(blk + 16 + 32 * g + 8 * kg);
  return r;
}

// One Q4_K block for the lane's (token, row) of up to two groups (gstride bytes apart in LDS; a: the lane's A pointer at
// the block). T[r] = sum_j sc_j D_j[r] (|D| <= 32 * 128 * 15, 8 sub-blocks x 63: < 2^25); M = sum_j m_j (sum of the
// sub-block's digits) is an MFMA accumulation with B = m_j in every byte (|.| <= 8 * 63 * 32 * 128 < 2^21).
__device__ inline void q4_block_mfma(const Q4Lane& w, const int8_t* a, int gstride, bool two, int fw, int64_t dqmax,
                                     MoeSum (&acc)[2], Acc128 (&accw)[2], bool& any) {
  const MoeFactor dq = moe_factor(w.h.x & 0xFFFF, fw, dqmax), dmq = moe_factor(w.h.x >> 16, fw, dqmax);
  const bool wide = __any(!(dq.ok && dmq.ok));
  if (wide) moe_wide_begin(accw, any);
  // the twelve 6-bit scales and mins, four to a dword: bytes j of sc0 / mn0 (sub-blocks 0..3), of sc1 / mn1 (4..7)
  const uint32_t sc[2] = {w.h.y & 0x3F3F3F3Fu, (w.h.w & 0x0F0F0F0Fu) | ((w.h.y >> 2) & 0x30303030u)};
  const uint32_t mn[2] = {w.h.z & 0x3F3F3F3Fu, ((w.h.w >> 4) & 0x0F0F0F0Fu) | ((w.h.z >> 2) & 0x30303030u)};
  // sub-block j's weights: the low / high nibbles of q bytes 32 (j / 2) + 8 kg ..; the min term's B operand has
  // m_j in every byte
  auto bq = [&](int j) {
    const uint2 qv = w.q[j >> 1];
    const uint32_t b0 = (j & 1) ? (qv.x >> 4) & 0x0F0F0F0Fu : qv.x & 0x0F0F0F0Fu;
    const uint32_t b1 = (j & 1) ? (qv.y >> 4) & 0x0F0F0F0Fu : qv.y & 0x0F0F0F0Fu;
    return (int64_t)(((uint64_t)b1 << 32) | b0);
  };
  auto bm = [&](int j) {
    const uint32_t mb = __builtin_amdgcn_perm(0u, mn[j >> 2], 0x01010101u * (uint32_t)(j & 3));
    return (int64_t)(((uint64_t)mb << 32) | mb);
  };
#pragma unroll
  for (int gi = 0; gi < 2; ++gi) {
    if (gi == 1 && !two) break;                       // wave-uniform
    const int8_t* gb = a + gi * gstride;
    v4i M = {0, 0, 0, 0}, T = {0, 0, 0, 0};
    // two halves of four sub-blocks: four independent MFMAs issued back to back, their results consumed after
#pragma unroll
    for (int hh = 0; hh < 2; ++hh) {
      v4i d[4];
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) {
        const int j = 4 * hh + jj;
        const int64_t av = moe_a(gb, 32 * j);
        d[jj] = mfma32(av, bq(j), v4i{0, 0, 0, 0});
        M = mfma32(av, bm(j), M);
      }
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) {
        const int sj = (int)((sc[hh] >> (8 * jj)) & 0xFF);
#pragma unroll
        for (int r = 0; r < 4; ++r) T[r] += __mul24(sj, d[jj][r]);   // 24-bit: |sc| < 2^6, |D| < 2^17
      }
    }
    if (!wide) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        acc[gi].v[r] += (int64_t)dq.f * T[r];
        acc[gi].v[r] += (int64_t)-dmq.f * M[r];
      }
    } else {
      moe_wide_add(&accw[gi], w.h.x & 0xFFFF, fw, false, T);
      moe_wide_add(&accw[gi], w.h.x >> 16, fw, true, M);
    }
  }
}

// Waves 0..3 walk the gate rows and 4..7 the up rows of the same 64 rows, one block ahead each (two were slower, see
// above); their results meet in LDS for the SiLU pass, a thread per (token, row).
__global__ __launch_bounds__(512, 4) void moe_gateup_kernel(const MoeItem* __restrict__ items, const int* __restrict__ ptok,
                                                         const int* __restrict__ ppair, const int8_t* __restrict__ xd,
                                                         const int* __restrict__ Lrow, int64_t rows, int64_t K,
                                                         int64_t e_ffn, int fw, int fa, int64_t log2e, int64_t dclip,
                                                         int64_t dqmax, int64_t* __restrict__ gu,
                                                         int* __restrict__ status, const int* __restrict__ wide) {
  extern __shared__ __align__(16) int8_t sx[];       // moe_lds_bytes(nb)
  __shared__ int64_t s_y[2][2 * kMoeTok][64];         // [gate, up][token][row]
  if (*wide) return;                                  // the VALU fallback takes this call
  const MoeItem it = items[blockIdx.y];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), proj = wave >> 2;
  const int n = lane & 15, kg = lane >> 4, t = lane >> 4;
  const int nb = (int)(K / 256);
  const int row = 16 * (wave & 3) + n;
  const int64_t ob = (int64_t)blockIdx.x * 64;
  const bool orow = ob + row < e_ffn;
  const uint8_t* wrow = (proj ? it.wu : it.wg) + (orow ? ob + row : 0) * nb * 144;
  for (int t0 = 0; t0 < it.count;) {
    Q4Lane wq = q4_lane_load(wrow, kg);
    const MoeRows w = moe_rows(ptok + it.first + t0, Lrow, it.count - t0);
    const int64_t pair = ppair[it.first + min(t0 + wave, it.count - 1)];   // the SiLU pass's token is the wave
    const int ch = moe_chunk(nb), kp = 256 * ch + 16;
    const int8_t* a0 = sx + moe_a_lane(lane, kp);
    MoeSum acc[2] = {};
    Acc128 accw[2];
    bool any = false;
    for (int c0 = 0; c0 < nb; c0 += ch) {
      const int cn = min(ch, nb - c0);
      __syncthreads();                                // the buffer is free
      moe_stage(sx, w, c0, cn, kp, xd, rows, K, tid, 512);
      __syncthreads();
      moe_settle();
      for (int bb = 0; bb < cn; ++bb) {               // the next block is requested as soon as this one is decoded
        const Q4Lane cur = wq;
        wq = q4_lane_load(wrow + (int64_t)min(c0 + bb + 1, nb - 1) * 144, kg);
        q4_block_mfma(cur, a0 + 256 * bb, 16 * kp, w.two, fw, dqmax, acc, accw, any);
      }
    }
    auto put = [&](i128 v, int tok) {
      bool f;
      s_y[proj][tok][row] = moe_result(v, fw, &f);
      if (!f && orow && tok < w.tn) atomicOr(status, IMIE_EOVF);
    };
    i128 y = moe_total(acc[0], accw[0], any);
    if (w.two) {
      const i128 y1 = moe_total(acc[1], accw[1], any);
      if (w.hi) y += (i128)((unsigned __int128)y1 << 32);
      else put(y1, kMoeTok + t);
    }
    put(y, t);
    __syncthreads();
    if (wave < w.tn && ob + lane < e_ffn) {
      bool f;
      const int64_t v = nmc_silu_mul(s_y[0][wave][lane], s_y[1][wave][lane], fa, log2e, dclip, &f);
      if (!f) atomicOr(status, IMIE_EOVF);
      gu[pair * e_ffn + ob + lane] = v;
    }
    t0 += w.tn;
  }
}

// Q6_K weights of one block for B lanes (row n, K group kg): per K step (half, qq) the ql bytes
// 64 half + 32 (qq & 1) + 8 kg .. + 7 and the qh bytes 32 half + 8 kg .. + 7 (bits 2 qq, 2 qq + 1); the 16
// int8 scales and d
struct Q6Lane {
  uint2 l[2][2];            // [half][qq & 1]
  uint2 h[2];               // [half]
  uint4 sc;
  uint32_t d;
};
__device__ inline Q6Lane q6_lane_load(const uint8_t* blk, int kg) {
  Q6Lane r;
#pragma unroll
  for (int half = 0; half < 2; ++half) {
#pragma unroll
    for (int o = 0; o < 2; ++o) r.l[half][o] = gload<uint2>(blk + 64 * half + 32 * o + 8 * kg);
    r.h[half] = gload<uint2>(blk + 128 + 32 * half + 8 * kg);
  }
  r.sc = gload<uint4>(blk + 192);
  r.d = gload<uint16_t>(blk + 208);                   // blocks are 210 bytes apart: 2-byte aligned
  return r;
}

// One Q6_K block: T[r] = sum_j sc_j D_j[r] with the weights as bytewise 4 (q6 - 32) (the six bits at the top of the byte,
// sign bit flipped: five instructions a dword), so the row's total is a multiple of 4 and shifted back once (|D| <= 16 *
// 128 * 128 = 2^18, 16 sub-blocks x 128: 2^29). A 32-position K step spans two sub-blocks (K groups 0, 1 and 2, 3): two
// MFMAs, whose A pointers (a0, a1; s0, s1: bytes between the groups) lead the other one's lanes to zeros in LDS.
__device__ inline void q6_block_mfma(const Q6Lane& w, const int8_t* a0, const int8_t* a1, int s0, int s1, bool two,
                                     int fw, int64_t dqmax, MoeSum (&acc)[2], Acc128 (&accw)[2], bool& any) {
  const MoeFactor dq = moe_factor(w.d, fw, dqmax);
  const bool wide = __any(!dq.ok);
  if (wide) moe_wide_begin(accw, any);
  const uint32_t scw[4] = {w.sc.x, w.sc.y, w.sc.z, w.sc.w};
  auto scs = [&](int i) { return (int)(int8_t)(uint8_t)(scw[i >> 2] >> (8 * (i & 3))); };
  auto wq = [](uint32_t lv, uint32_t hv, int qq) {
    const uint32_t lo = qq >= 2 ? lv >> 2 : lv << 2, hi = hv << (6 - 2 * qq);
    return (((lo & 0x3C3C3C3Cu) | (hi & ~0x3C3C3C3Cu)) & 0xFCFCFCFCu) ^ 0x80808080u;
  };
  int64_t bq[2][4];
#pragma unroll
  for (int half = 0; half < 2; ++half)
#pragma unroll
    for (int qq = 0; qq < 4; ++qq) {
      const uint2 lv = w.l[half][qq & 1], hv = w.h[half];
      bq[half][qq] = (int64_t)(((uint64_t)wq(lv.y, hv.y, qq) << 32) | wq(lv.x, hv.x, qq));
    }
#pragma unroll
  for (int gi = 0; gi < 2; ++gi) {
    if (gi == 1 && !two) break;                       // wave-uniform
    const int8_t *g0 = a0 + gi * s0, *g1 = a1 + gi * s1;
    v4i T = {0, 0, 0, 0};
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      // the 8 MFMAs of a half are independent: issued back to back, consumed afterwards
      v4i d[4][2];
#pragma unroll
      for (int qq = 0; qq < 4; ++qq) {
        d[qq][0] = mfma32(moe_a(g0, 128 * half + 32 * qq), bq[half][qq], v4i{0, 0, 0, 0});
        d[qq][1] = mfma32(moe_a(g1, 128 * half + 32 * qq), bq[half][qq], v4i{0, 0, 0, 0});
      }
#pragma unroll
      for (int qq = 0; qq < 4; ++qq) {
        const int c0 = scs(8 * half + 2 * qq), c1 = scs(8 * half + 2 * qq + 1);
#pragma unroll
        for (int r = 0; r < 4; ++r) T[r] += __mul24(c0, d[qq][0][r]) + __mul24(c1, d[qq][1][r]);   // |s| < 2^8, |D| <= 2^18
      }
    }
    if (!wide) {
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[gi].v[r] += (int64_t)dq.f * T[r];
    } else {
      moe_wide_add(&accw[gi], w.d, fw, false, T);
    }
  }
}

__global__ __launch_bounds__(256, 4) void moe_down_kernel(const MoeItem* __restrict__ items, const int* __restrict__ ppair,
                                                       const int8_t* __restrict__ xd, const int* __restrict__ Lrow,
                                                       int64_t rows, int64_t K, int64_t d_model, int wtiles, int fw, int64_t dqmax,
                                                       int64_t* __restrict__ dout, int* __restrict__ status,
                                                       const int* __restrict__ wide) {
  extern __shared__ __align__(16) int8_t sx[];       // moe_lds_bytes(nb): 256 zero bytes, the staged digits
  if (*wide) return;
  const MoeItem it = items[blockIdx.y];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int n = lane & 15, kg = lane >> 4, t = lane >> 4;
  const int nb = (int)(K / 256);
  // the wave's tiles: rows o0 + 64 rt
  const int64_t o0 = (int64_t)blockIdx.x * (64 * wtiles) + wave * 16 + n;
  const int tiles = (int)min((int64_t)wtiles, (d_model - (int64_t)blockIdx.x * (64 * wtiles) + 63) / 64);
  auto wrow = [&](int rt) {
    const int64_t o = o0 + 64 * rt;
    return it.wd + (o < d_model ? o : 0) * nb * 210;
  };
  if (tid < 16) ((uint4*)sx)[tid] = uint4{0, 0, 0, 0};   // visible with the first staging
  for (int t0 = 0; t0 < it.count;) {
    Q6Lane wq = q6_lane_load(wrow(0), kg);
    const MoeRows w = moe_rows(ppair + it.first + t0, Lrow, it.count - t0);
    const int ch = moe_chunk(nb), kp = 256 * ch + 16;
    const int al = 256 + moe_a_lane(lane, kp), z = 8 * kg;
    for (int rt = 0; rt < tiles; ++rt) {
      const uint8_t *row = wrow(rt), *next = wrow(min(rt + 1, tiles - 1));
      MoeSum ad[2] = {};
      Acc128 adw[2];
      bool any = false;
      for (int c0 = 0; c0 < nb; c0 += ch) {
        const int cn = min(ch, nb - c0);
        if (rt == 0 || ch < nb) {                     // whole rows that fit are staged once for all tiles
          __syncthreads();                            // the buffer is free
          moe_stage(sx + 256, w, c0, cn, kp, xd, rows, K, tid, 256);
          __syncthreads();
          moe_settle();
        }
        for (int bb = 0; bb < cn; ++bb) {
          const int b = c0 + bb + 1, a = al + 256 * bb;
          const Q6Lane cur = wq;
          wq = q6_lane_load(b < nb ? row + (int64_t)b * 210 : next, kg);
          q6_block_mfma(cur, sx + (kg < 2 ? a : z), sx + (kg < 2 ? z : a), kg < 2 ? 16 * kp : 0, kg < 2 ? 0 : 16 * kp,
                        w.two, fw, dqmax, ad, adw, any);
        }
      }
      const int64_t o = o0 + 64 * rt;
      auto emit = [&](i128 y, int tok) {
        if (o >= d_model || tok >= w.tn) return;
        bool f;
        const int64_t v = moe_result(y >> 2, fw, &f);
        if (!f) atomicOr(status, IMIE_EOVF);
        dout[(int64_t)ppair[it.first + t0 + tok] * d_model + o] = v;
      };
      i128 y = moe_total(ad[0], adw[0], any);
      if (w.two) {
        const i128 y1 = moe_total(ad[1], adw[1], any);
        if (w.hi) y += (i128)((unsigned __int128)y1 << 32);
        else emit(y1, kMoeTok + t);
      }
      emit(y, t);
    }
    t0 += w.tn;
  }
}

// ---------------------------------------------------------------------------------------------------------
// Single-row products (decode): a Q4_K / Q6_K weight against one activation row, and the MoE block of a few tokens.
// One launch each: every workgroup peels the row's balanced base-256 digits into LDS itself (no prep launch, no flag
// to reset, no item list to upload: the weight pointers are kernel arguments), a weight row is spread over a half
// wave, 64 weights (a quarter of a 256-block) per lane, so a row of up to 2048 is one load round and one pass of
// v_dot4_i32_i8 per limb, and the lanes' 128-bit partial sums are added by shuffles. A row beyond kQkLimbs limbs takes
// exact 128-bit products in the same kernel. Bound by latency: the weights of one projection are 1 to 5 MB.
// The digits of 64 consecutive activations are an LDS unit of 80 bytes: 16 lanes reading 16 bytes each at that stride
// touch every bank once (at 64 bytes the same 16 banks four times over).
// Measured: a 4096 x 2048 Q4_K product 3.3 + 1.3 + 28 + 4.4 us (prep, flag, 64 workgroups walking the blocks with two
// barriers each, fallback launch) and three uploads; Q, K and V of one token in one launch, or O: 8.7 us.
// ---------------------------------------------------------------------------------------------------------
constexpr int kG1Unit = 80;
constexpr int kG1MaxNb = 32;       // digits of 32 blocks: 51 KB of LDS
constexpr int kG1Items = 16;
constexpr int kG1Rows = 2;         // weight rows per half wave

struct G1Raw {                     // one lane's 64 weights: Q4_K header, quants; Q6_K low, high bits, scales, d
  uint4 v[6];
  uint32_t s, d;
};

template <int QT>
__device__ inline G1Raw g1_load(const uint8_t* row, int u) {
  const uint8_t* blk = row + (int64_t)(u >> 2) * (QT == 0 ? 144 : 210);
  const int q = u & 3;
  G1Raw r;
  if (QT == 0) {
    r.v[0] = gload<uint4>(blk);
    r.v[1] = gload<uint4>(blk + 16 + 32 * q);
    r.v[2] = gload<uint4>(blk + 32 + 32 * q);
    r.s = r.d = 0;
  } else {
    const int half = q >> 1;
#pragma unroll
    for (int i = 0; i < 4; ++i) r.v[i] = gload<uint4>(blk + 64 * half + 16 * i);
#pragma unroll
    for (int i = 0; i < 2; ++i) r.v[4 + i] = gload<uint4>(blk + 128 + 32 * half + 16 * i);
    const uint8_t* sc = blk + 192 + 8 * half + 4 * (q & 1);
    r.s = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) r.s |= (uint32_t)gload<uint8_t>(sc + i) << (8 * i);
    r.d = (uint32_t)gload<uint8_t>(blk + 208) | ((uint32_t)gload<uint8_t>(blk + 209) << 8);
  }
  return r;
}

// the lane's 64 weights as 16 dwords of int8 (positions 0..31 and 32..63), and their factors: Q4_K sc / mn per 32,
// Q6_K 4 w and sc per 16; dq, dmq
struct G1W {
  int w[16];
  int sc[4], mn[2];
  int64_t dq, dmq;
};
// fp16_fixed_fast, in 32 bits when every lane's result is below 2^31 (m 2^sh with sh <= 20: single precision holds
// it exactly either way, so one ldexp and rint serve both directions of the shift)
__device__ inline int64_t g1_fp16(uint32_t h, int fw) {
  const uint32_t e = (h >> 10) & 31, mant = h & 0x3FF;
  const int sh = (e == 0 ? 1 : (int)e) - 25 + fw;
  if (__any(sh > 20)) return fp16_fixed_fast(h, fw);
  const float m = (float)(e == 0 ? mant : (mant | 0x400));
  const int r = (int)__builtin_rintf(__builtin_ldexpf(m, sh));
  return ((h >> 15) & 1) ? -r : r;
}

template <int QT>
__device__ inline G1W g1_unpack(const G1Raw& r, int q, int fw) {
  G1W o;
  if (QT == 0) {
    o.dq = g1_fp16(r.v[0].x & 0xFFFFu, fw);
    o.dmq = g1_fp16(r.v[0].x >> 16, fw);
    const uint32_t hd[3] = {r.v[0].y, r.v[0].z, r.v[0].w};   // the 12 scale bytes
    const int j0 = 2 * (q & 1);                       // sub-blocks 2 q, 2 q + 1; byte j of a dword each
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int sh = 8 * (j0 + h);
      const uint32_t b0 = (hd[0] >> sh) & 255, b1 = (hd[1] >> sh) & 255, b2 = (hd[2] >> sh) & 255;
      if (q < 2) { o.sc[h] = b0 & 63; o.mn[h] = b1 & 63; }
      else { o.sc[h] = (b2 & 0xF) | ((b0 >> 6) << 4); o.mn[h] = (b2 >> 4) | ((b1 >> 6) << 4); }
    }
    o.sc[2] = o.sc[3] = 0;
    const uint32_t qd[8] = {r.v[1].x, r.v[1].y, r.v[1].z, r.v[1].w, r.v[2].x, r.v[2].y, r.v[2].z, r.v[2].w};
#pragma unroll
    for (int d = 0; d < 8; ++d) {
      o.w[d] = (int)(qd[d] & 0x0F0F0F0Fu);
      o.w[8 + d] = (int)((qd[d] >> 4) & 0x0F0F0F0Fu);
    }
  } else {
    o.dq = g1_fp16(r.d, fw);
    o.dmq = 0;
    o.mn[0] = o.mn[1] = 0;
    const uint32_t lq[16] = {r.v[0].x, r.v[0].y, r.v[0].z, r.v[0].w, r.v[1].x, r.v[1].y, r.v[1].z, r.v[1].w,
                             r.v[2].x, r.v[2].y, r.v[2].z, r.v[2].w, r.v[3].x, r.v[3].y, r.v[3].z, r.v[3].w};
    const uint32_t hq[8] = {r.v[4].x, r.v[4].y, r.v[4].z, r.v[4].w, r.v[5].x, r.v[5].y, r.v[5].z, r.v[5].w};
    // bytewise 4 (q6 - 32) as int8: the 6 bits moved to the top of the byte and its sign bit flipped
    const int sl = (q & 1) ? 4 : 0, sh = (q & 1) ? 4 : 0;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int d = 0; d < 8; ++d) {
        const uint32_t lo = (sl ? lq[8 * u + d] >> 2 : lq[8 * u + d] << 2) & 0x3C3C3C3Cu;
        const uint32_t hi = (sh ? hq[d] << (2 - 2 * u) : hq[d] << (6 - 2 * u)) & 0xC0C0C0C0u;
        o.w[8 * u + d] = (int)((lo | hi) ^ 0x80808080u);
      }
#pragma unroll
    for (int i = 0; i < 4; ++i) o.sc[i] = (int)(int8_t)(uint8_t)(r.s >> (8 * i));
  }
  return o;
}

// acc[r] += the lane's 64 weights of row r x activations, R rows sharing the digits read; xu: the unit's digits of
// limb 0 in LDS, ls: bytes between limbs
template <int QT, int R>
__device__ inline void g1_dot(const G1W (&w)[R], const int8_t* xu, int ls, int L, Acc128 (&acc)[R]) {
  // S1 = sum sc w.x (Q6_K: of the 4 w) and S2 = sum mn xsum: a limb's part stays in int32 (Q4_K: 2 x 63 x 32 x 128 x 15
  // < 2^23, and 2 x 63 x 32 x 128 < 2^19; Q6_K: 4 x 128 x 16 x 128 x 128 = 2^27) and joins with one 32 x 32 + 64
  int64_t S1[R], S2[R];
#pragma unroll
  for (int r = 0; r < R; ++r) S1[r] = S2[r] = 0;
  for (int l = 0; l < L; ++l) {
    const int wt = 1 << (8 * (l & 3));                // limb 4 (2^32): shifted once more below
    int xv[16];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int4 x = *(const int4*)(xu + l * ls + 16 * c);
      xv[4 * c] = x.x;
      xv[4 * c + 1] = x.y;
      xv[4 * c + 2] = x.z;
      xv[4 * c + 3] = x.w;
    }
    int b0 = 0, b1 = 0;
    if (QT == 0) {
#pragma unroll
      for (int d = 0; d < 8; ++d) {
        b0 = __builtin_amdgcn_sdot4(xv[d], 0x01010101, b0, false);
        b1 = __builtin_amdgcn_sdot4(xv[8 + d], 0x01010101, b1, false);
      }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
      int a[4] = {0, 0, 0, 0}, t1, t2 = 0;
#pragma unroll
      for (int d = 0; d < 16; ++d) a[d >> 2] = __builtin_amdgcn_sdot4(xv[d], w[r].w[d], a[d >> 2], false);
      if (QT == 0) {
        t1 = __mul24(w[r].sc[0], a[0] + a[1]) + __mul24(w[r].sc[1], a[2] + a[3]);
        t2 = __mul24(w[r].mn[0], b0) + __mul24(w[r].mn[1], b1);
      } else {
        t1 = __mul24(w[r].sc[0], a[0]) + __mul24(w[r].sc[1], a[1]) + __mul24(w[r].sc[2], a[2]) + __mul24(w[r].sc[3], a[3]);
      }
      if (l < 4) {
        S1[r] += (int64_t)t1 * wt;
        if (QT == 0) S2[r] += (int64_t)t2 * wt;
      } else {
        S1[r] += (int64_t)((uint64_t)(uint32_t)t1 << 32);
        if (QT == 0) S2[r] += (int64_t)((uint64_t)(uint32_t)t2 << 32);
      }
    }
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    acc_madd(acc[r], w[r].dq, QT == 0 ? S1[r] : S1[r] >> 2);   // Q6_K: exact, every weight is a multiple of 4
    if (QT == 0) acc_madd(acc[r], -w[r].dmq, S2[r]);
  }
}

// The lane's 64 weights (unit u of a row) x the 64-bit activations themselves, in 128 bits: a row that needs more than
// kQkLimbs limbs. Rare, so one compact copy that decodes a weight at a time (unrolled into every caller it cost
// registers and instruction fetches on the common path).
__device__ __attribute__((noinline)) void g1_wide(const uint8_t* row, int u, int qtype, int fw, const int64_t* x,
                                                  Acc128* acc) {
  const uint8_t* blk = row + (int64_t)(u >> 2) * (qtype == 0 ? 144 : 210);
  const int q = u & 3;
  i128 a = (i128)(((unsigned __int128)(uint64_t)acc->hi << 64) | acc->lo);
  const int n = qtype == 0 ? 32 : 16;                 // one sub-block at a time
#pragma unroll 1
  for (int e0 = 0; e0 < 64; e0 += n) {
    i128 qd = 0, xs = 0;
#pragma unroll 1
    for (int e = e0; e < e0 + n; ++e) {
      int w;
      if (qtype == 0) {
        const uint8_t b = gload<uint8_t>(blk + 16 + 32 * q + (e & 31));
        w = e < 32 ? b & 15 : b >> 4;
      } else {
        const int half = q >> 1, qq = 2 * (q & 1) + (e >> 5), l = e & 31;
        const uint8_t lo = gload<uint8_t>(blk + 64 * half + 32 * (qq & 1) + l);
        const uint8_t hi = gload<uint8_t>(blk + 128 + 32 * half + l);
        w = (((qq & 2) ? lo >> 4 : lo & 15) | (((hi >> (2 * qq)) & 3) << 4)) - 32;
      }
      qd += (i128)w * x[64 * (int64_t)u + e];
      xs += x[64 * (int64_t)u + e];
    }
    if (qtype == 0) {
      const int j = 2 * q + (e0 >> 5);
      const uint8_t* sc = blk + 4;
      const int s = j < 4 ? gload<uint8_t>(sc + j) & 63
                          : (gload<uint8_t>(sc + j + 4) & 15) | ((gload<uint8_t>(sc + j - 4) >> 6) << 4);
      const int m = j < 4 ? gload<uint8_t>(sc + j + 4) & 63
                          : (gload<uint8_t>(sc + j + 4) >> 4) | ((gload<uint8_t>(sc + j) >> 6) << 4);
      const uint32_t d = gload<uint8_t>(blk) | ((uint32_t)gload<uint8_t>(blk + 1) << 8);
      const uint32_t dm = gload<uint8_t>(blk + 2) | ((uint32_t)gload<uint8_t>(blk + 3) << 8);
      a += (i128)(fp16_fixed_fast(d, fw) * s) * qd - (i128)(fp16_fixed_fast(dm, fw) * m) * xs;
    } else {
      const int s = (int8_t)gload<uint8_t>(blk + 192 + 8 * (q >> 1) + 4 * (q & 1) + (e0 >> 4));
      const uint32_t d = gload<uint8_t>(blk + 208) | ((uint32_t)gload<uint8_t>(blk + 209) << 8);
      a += (i128)(fp16_fixed_fast(d, fw) * s) * qd;
    }
  }
  acc->lo = (uint64_t)a;
  acc->hi = (int64_t)((unsigned __int128)a >> 64);
}

// Digit units of the n activations x (n a multiple of 64) into LDS, kQkLimbs limbs of n / 64 units; returns the limb
// count that all of them need, 0 when one needs more than kQkLimbs. Ends with a barrier.
template <int NT>
__device__ inline int g1_stage(const int64_t* __restrict__ x, int n, int8_t* s_x, uint64_t* s_red) {
  const int ls = (n >> 6) * kG1Unit;
  uint64_t mx = 0;
  for (int c0 = 8 * (int)threadIdx.x; c0 < n; c0 += 8 * NT) {
    int64_t v[8];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const longlong2 p = *(const longlong2*)(x + c0 + 2 * e);
      v[2 * e] = p.x;
      v[2 * e + 1] = p.y;
    }
    uint64_t m8 = 0, d[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const uint64_t a = imie_absu64(v[e]);
      m8 = a > m8 ? a : m8;
    }
    mx = m8 > mx ? m8 : mx;
    if (m8 <= imie_balanced_cap(4)) {
#pragma unroll
      for (int e = 0; e < 8; ++e) d[e] = imie_digits32((uint32_t)v[e]);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) d[e] = imie_digits64((uint64_t)v[e]);
    }
    uint32_t lo[4], hi[4], top[4] = {0, 0, 0, 0};
    imie_bytes4x4((uint32_t)d[0], (uint32_t)d[1], (uint32_t)d[2], (uint32_t)d[3], lo);
    imie_bytes4x4((uint32_t)d[4], (uint32_t)d[5], (uint32_t)d[6], (uint32_t)d[7], hi);
    int8_t* dst = s_x + (c0 >> 6) * kG1Unit + (c0 & 63);
#pragma unroll
    for (int l = 0; l < 4; ++l) *(uint2*)(dst + l * ls) = uint2{lo[l], hi[l]};
    static_assert(kQkLimbs == 5, "one digit above the low four");
    imie_bytes4x4((uint32_t)(d[0] >> 32), (uint32_t)(d[1] >> 32), (uint32_t)(d[2] >> 32), (uint32_t)(d[3] >> 32), top);
    uint2 t5;
    t5.x = top[0];
    imie_bytes4x4((uint32_t)(d[4] >> 32), (uint32_t)(d[5] >> 32), (uint32_t)(d[6] >> 32), (uint32_t)(d[7] >> 32), top);
    t5.y = top[0];
    *(uint2*)(dst + 4 * ls) = t5;
  }
  mx = imie_wave_max_u64_full(mx);
  if ((threadIdx.x & 63) == 0) s_red[threadIdx.x >> 6] = mx;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < NT / 64; ++w) mx = s_red[w] > mx ? s_red[w] : mx;
  return mx <= imie_balanced_cap(kQkLimbs) ? imie_limbs_needed(mx) : 0;
}

// R weight rows (LPR lanes, lane lr of them) against the staged digits of U units at s_x; cur: the lane's first unit
// of each. Every lane gets the rows' sums. next: called once cur is used up (the caller may refill it and row).
template <int QT, int LPR, int R, typename Next>
__device__ inline void g1_rows(const uint8_t* (&row)[R], int lr, int U, G1Raw (&cur)[R], const int8_t* s_x, int ls,
                               int L, int fw, const int64_t* x, Acc128 (&acc)[R], Next next) {
#pragma unroll
  for (int r = 0; r < R; ++r) acc[r] = Acc128{0, 0};
  if (L == 0) {                                       // a wide row
    for (int u = lr; u < U; u += LPR)
#pragma unroll
      for (int r = 0; r < R; ++r) g1_wide(row[r], u, QT, fw, x, &acc[r]);
    next();
  }
  for (int u = lr; L && u - lr < U; u += LPR) {       // every lane walks the same steps; past the end: no product
    G1W w[R];
#pragma unroll
    for (int r = 0; r < R; ++r) w[r] = g1_unpack<QT>(cur[r], u & 3, fw);
    if (u - lr + LPR < U) {
#pragma unroll
      for (int r = 0; r < R; ++r) cur[r] = g1_load<QT>(row[r], u + LPR < U ? u + LPR : 0);
    } else {
      next();                                         // the caller's next rows, requested before this step's products
    }
    if (u < U) g1_dot<QT, R>(w, s_x + u * kG1Unit, ls, L, acc);
  }
  auto add = [&](Acc128& a, uint64_t lo, uint64_t hi) {
    a.lo += lo;
    a.hi += (int64_t)hi + (a.lo < lo ? 1 : 0);
  };
  static_assert(LPR == 16 || LPR == 32, "one or two DPP rows");
#pragma unroll
  for (int r = 0; r < R; ++r) {                       // xor 1, xor 2, half-row mirror, row mirror, xor 16
    add(acc[r], imie_dpp64<0xB1>(acc[r].lo), imie_dpp64<0xB1>((uint64_t)acc[r].hi));
    add(acc[r], imie_dpp64<0x4E>(acc[r].lo), imie_dpp64<0x4E>((uint64_t)acc[r].hi));
    add(acc[r], imie_dpp64<0x141>(acc[r].lo), imie_dpp64<0x141>((uint64_t)acc[r].hi));
    add(acc[r], imie_dpp64<0x140>(acc[r].lo), imie_dpp64<0x140>((uint64_t)acc[r].hi));
    if (LPR == 32)
      add(acc[r], (uint64_t)__shfl_xor((long long)acc[r].lo, 16, 64), (uint64_t)__shfl_xor((long long)acc[r].hi, 16, 64));
  }
}

struct G1Item {
  const uint8_t* w;
  int64_t* y;
  int64_t out_f;
  int qtype, wg0;           // first workgroup of the item
};
struct G1Args {
  G1Item it[kG1Items];
  const int64_t* x;
  int* status;
  int cnt, nb, fw;
};

template <int QT>
__device__ inline void g1_linear(const G1Args& a, const G1Item& it, int8_t* s_x, uint64_t* s_red) {
  const int lane = threadIdx.x & 63, l32 = lane & 31, U = 4 * a.nb;
  const int64_t o0 = ((int64_t)(blockIdx.x - it.wg0) * 8 + (threadIdx.x >> 5)) * kG1Rows;
  const int64_t rb = (int64_t)a.nb * (QT == 0 ? 144 : 210);
  const uint8_t* row[kG1Rows];
  G1Raw first[kG1Rows];
#pragma unroll
  for (int r = 0; r < kG1Rows; ++r) {                 // requested before the digits are formed; past the end: row 0
    row[r] = it.w + (o0 + r < it.out_f ? o0 + r : 0) * rb;
    first[r] = g1_load<QT>(row[r], l32 < U ? l32 : 0);
  }
  const int L = g1_stage<256>(a.x, 64 * U, s_x, s_red);
  Acc128 acc[kG1Rows];
  g1_rows<QT, 32, kG1Rows>(row, l32, U, first, s_x, U * kG1Unit, L, a.fw, a.x, acc, [] {});
#pragma unroll
  for (int r = 0; r < kG1Rows; ++r)
    if (l32 == r && o0 + r < it.out_f) {
      bool fits;
      it.y[o0 + r] = acc_shift(acc[r], a.fw, &fits);
      if (!fits) atomicOr(a.status, IMIE_EOVF);
    }
}

__global__ __launch_bounds__(256) void qk_gemv1_kernel(G1Args a) {
  extern __shared__ __align__(16) int8_t s_x[];
  __shared__ uint64_t s_red[4];
  int i = 0;
  while (i + 1 < a.cnt && (int)blockIdx.x >= a.it[i + 1].wg0) ++i;
  if (a.it[i].qtype == 0) g1_linear<0>(a, a.it[i], s_x, s_red);
  else g1_linear<1>(a, a.it[i], s_x, s_red);
}

// The MoE block of a few tokens (Q4_K gate / up, Q6_K down) in two launches: gate, up and SiLU(g) u per (pair, row) --
// the gate row in one half of the wave, the up row in the other --, then down and the gated sum over a token's
// experts, with the residual of the retained layer chain added when `res` is given. The expert pointers are kernel
// arguments. Each pair reads its expert's weights, so up to kMoe1Pairs pairs, where few experts repeat. Bound by VALU
// (about 500 instructions a weight row pair and half wave at one to two waves per SIMD), 13 + 12 us for one token's
// eight experts of 768 at hidden 2048, where the grouped form's seven launches took 18 + 10 + 20 us.
constexpr int kMoe1Pairs = 32;
constexpr int kMoe1Rows = 2;       // weight rows per lane group
constexpr int kMoe1Wave = 4;       // gate and up rows of a wave (one SiLU pass for all of them)
constexpr int kMoe1Out = 8;        // output rows of a down workgroup
constexpr int kMoe1MaxK = 16;      // experts of a token
struct Moe1Args {
  const uint8_t* w[3][kMoe1Pairs];
  const int64_t *h, *gates;
  int64_t *gu, *out;
  const int64_t *res, *ao;
  int k, d_model, e_ffn, fa, fw;
  int64_t log2e, dclip;
  int* status;
};

__global__ __launch_bounds__(256) void moe1_gateup_kernel(Moe1Args a) {
  extern __shared__ __align__(16) int8_t s_x[];
  __shared__ uint64_t s_red[4];
  const int p = blockIdx.y, lane = threadIdx.x & 63, l32 = lane & 31;
  const int o0 = ((int)blockIdx.x * 4 + (int)(threadIdx.x >> 6)) * kMoe1Wave, U = a.d_model / 64;
  const uint8_t* w = lane < 32 ? a.w[0][p] : a.w[1][p];
  const int64_t rb = (int64_t)(a.d_model / 256) * 144;
  const int64_t* x = a.h + (int64_t)(p / a.k) * a.d_model;
  const uint8_t* row[kMoe1Rows];
  G1Raw cur[kMoe1Rows];
  auto fetch = [&](int o) {
#pragma unroll
    for (int r = 0; r < kMoe1Rows; ++r) {             // rows past the end: the last one again, not stored
      row[r] = w + (o + r < a.e_ffn ? o + r : a.e_ffn - 1) * rb;
      cur[r] = g1_load<0>(row[r], l32 < U ? l32 : 0);
    }
  };
  fetch(o0);
  const int L = g1_stage<256>(x, a.d_model, s_x, s_red);
  int64_t mine = 0;
  bool good = true;
#pragma unroll 1
  for (int i = 0; i < kMoe1Wave; i += kMoe1Rows) {
    Acc128 acc[kMoe1Rows];
    g1_rows<0, 32, kMoe1Rows>(row, l32, U, cur, s_x, U * kG1Unit, L, a.fw, x, acc,
                              [&] { if (i + kMoe1Rows < kMoe1Wave) fetch(o0 + i + kMoe1Rows); });
#pragma unroll
    for (int r = 0; r < kMoe1Rows; ++r)
      if (l32 == i + r) {                             // lanes r / 32 + r keep row r's gate / up
        bool fits;
        mine = acc_shift(acc[r], a.fw, &fits);
        good = fits;
      }
  }
  const int64_t u = (int64_t)__shfl_xor((long long)mine, 32, 64);
  if (lane < kMoe1Wave && o0 + lane < a.e_ffn) {
    bool ok;
    a.gu[(int64_t)p * a.e_ffn + o0 + lane] = nmc_silu_mul(mine, u, a.fa, a.log2e, a.dclip, &ok);
    good = good && ok;
  }
  if (!good) atomicOr(a.status, IMIE_EOVF);
}

__global__ __launch_bounds__(512) void moe1_down_kernel(Moe1Args a) {
  extern __shared__ __align__(16) int8_t s_x[];
  __shared__ uint64_t s_red[8];
  __shared__ int64_t s_d[kMoe1Out][kMoe1MaxK];
  const int t = blockIdx.y, l16 = threadIdx.x & 15, grp = threadIdx.x >> 4;
  const int o0 = (int)blockIdx.x * kMoe1Out, U = a.e_ffn / 64;
  // a job: kMoe1Rows output rows of one expert, 16 lanes; 32 jobs at a time (all of them for eight experts)
  constexpr int kPer = kMoe1Out / kMoe1Rows;
  const int jobs = kPer * a.k;
  const int64_t rb = (int64_t)(a.e_ffn / 256) * 210;
  const int64_t* x = a.gu + (int64_t)t * a.k * a.e_ffn;
  const uint8_t* row[kMoe1Rows];
  G1Raw first[kMoe1Rows];
  auto fetch = [&](int job) {
    const uint8_t* w = a.w[2][t * a.k + job / kPer] + (int64_t)(o0 + (job % kPer) * kMoe1Rows) * rb;
#pragma unroll
    for (int r = 0; r < kMoe1Rows; ++r) {
      row[r] = w + r * rb;
      first[r] = g1_load<1>(row[r], l16 < U ? l16 : 0);
    }
  };
  fetch(grp < jobs ? grp : 0);
  const int L = g1_stage<512>(x, a.k * a.e_ffn, s_x, s_red);
  for (int job = grp; job < jobs; job += 32) {
    const int e = job / kPer;
    Acc128 acc[kMoe1Rows];
    g1_rows<1, 16, kMoe1Rows>(row, l16, U, first, s_x + e * U * kG1Unit, a.k * U * kG1Unit, L, a.fw,
                              x + (int64_t)e * a.e_ffn, acc, [&] { if (job + 32 < jobs) fetch(job + 32); });
#pragma unroll
    for (int r = 0; r < kMoe1Rows; ++r)
      if (l16 == r) {
        bool fits;
        s_d[(job % kPer) * kMoe1Rows + r][e] = acc_shift(acc[r], a.fw, &fits);
        if (!fits) atomicOr(a.status, IMIE_EOVF);
      }
  }
  __syncthreads();
  if (threadIdx.x < kMoe1Out) {
    i128 acc = 0;
    for (int j = 0; j < a.k; ++j) acc += ((i128)s_d[threadIdx.x][j] * a.gates[t * a.k + j]) >> a.fa;
    if (acc > (i128)INT64_MAX || acc < (i128)INT64_MIN) atomicOr(a.status, IMIE_EOVF);
    const int64_t i = (int64_t)t * a.d_model + o0 + threadIdx.x;
    uint64_t y = (uint64_t)acc;
    if (a.res) y += (uint64_t)a.res[i] + (uint64_t)a.ao[i];   // int64 wrap, as the committed numpy addition
    a.out[i] = (int64_t)y;
  }
}

// int8-MFMA path on/off (IMIE_QK_MFMA=0 forces the VALU kernel; tests compare both)
bool qk_mfma_enabled() {
  static const bool v = [] { const char* e = getenv("IMIE_QK_MFMA"); return !(e && atoi(e) == 0); }();
  return v;
}

// a Q4_K / Q6_K handle (int64 matrices registered by qk_register_i64 are qtype 2 and not accepted here)
const QKWeight* qk_get(int64_t h) {
  if (h < 0 || h >= (int64_t)g_qk.size() || !g_qk[(size_t)h].p || g_qk[(size_t)h].qtype > 1) return nullptr;
  return &g_qk[(size_t)h];
}

// One activation row against up to kG1Items weights of the same input width, in one launch (qk_gemv1_kernel).
bool gemv1_ok(int64_t nb) { return nb <= kG1MaxNb && qk_mfma_enabled(); }

int gemv1_launch(const QKWeight* const* ws, int64_t* const* ys, int cnt, const int64_t* x, int fw, int* status,
                 hipStream_t st) {
  G1Args a = {};
  a.x = x; a.status = status; a.cnt = cnt; a.nb = (int)ws[0]->nb; a.fw = fw;
  int64_t wgs = 0;
  for (int i = 0; i < cnt; ++i) {
    a.it[i] = G1Item{ws[i]->p, ys[i], ws[i]->out_f, ws[i]->qtype, (int)wgs};
    wgs += (ws[i]->out_f + 8 * kG1Rows - 1) / (8 * kG1Rows);
  }
  if (wgs > INT32_MAX) return IMIE_EARG;
  imie_prof_mark(IMIE_K_QK, st, true);
  hipLaunchKernelGGL(qk_gemv1_kernel, dim3((unsigned)wgs), dim3(256), (size_t)kQkLimbs * 4 * a.nb * kG1Unit, st, a);
  imie_prof_mark(IMIE_K_QK, st, false);
  IMIE_HIP(hipGetLastError());
  return IMIE_OK;
}

// Enqueue a set of items over device X (rows x K) into device Y (rows x ldy). pairs: host arrays. The int8-MFMA
// kernels run unless an activation row needs more than kQkLimbs limbs (or K is not a multiple of 256); then the
// exact VALU kernel does (both are enqueued, a device flag selects).
struct QkPrepWs {
  DevBuf xd, xs, lr, flag;
} g_qprep;

int run_items(const std::vector<Item>& items, const std::vector<int>& xi, const std::vector<int>& yi,
              const int64_t* X, int64_t K, int64_t* Y, int64_t ldy, int fw, int* status, hipStream_t st,
              DevBuf& ibuf, DevBuf& pbuf) {
  if (items.empty()) return IMIE_OK;
  const size_t np = xi.size();
  if (ibuf.ensure(items.size() * sizeof(Item)) || pbuf.ensure(np * 8)) return IMIE_EARG;
  IMIE_HIP(hipMemcpyAsync(ibuf.p, items.data(), items.size() * sizeof(Item), hipMemcpyHostToDevice, st));
  IMIE_HIP(hipMemcpyAsync(pbuf.p, xi.data(), np * 4, hipMemcpyHostToDevice, st));
  IMIE_HIP(hipMemcpyAsync((int*)pbuf.p + np, yi.data(), np * 4, hipMemcpyHostToDevice, st));
  int64_t maxo = 0;
  for (auto& it : items) maxo = it.out_f > maxo ? it.out_f : maxo;
  int64_t rows = 0;
  for (int r : xi) rows = r + 1 > rows ? r + 1 : rows;
  const bool mfma_ok = K % 256 == 0 && qk_mfma_enabled();
  const int* gate = nullptr;
  imie_prof_mark(IMIE_K_QK, st, true);
  if (mfma_ok) {
    if (g_qprep.xd.ensure((size_t)(kQkLimbs * rows * K)) || g_qprep.xs.ensure((size_t)(rows * (K / 16)) * 8) ||
        g_qprep.lr.ensure((size_t)rows * 4) || g_qprep.flag.ensure(64))
      return IMIE_EARG;
    int* flag = (int*)g_qprep.flag.p;
    hipLaunchKernelGGL(qk_flag_reset_kernel, dim3(1), dim3(1), 0, st, flag);
    hipLaunchKernelGGL(qk_prep_kernel, dim3((unsigned)rows), dim3(256), 0, st, X, rows, K, (int8_t*)g_qprep.xd.p,
                       (int64_t*)g_qprep.xs.p, (int*)g_qprep.lr.p, flag);
    const dim3 grid((unsigned)((maxo + 63) / 64), (unsigned)items.size());
    constexpr int kDot4Max = 32;                      // items with at most this many tokens take the dot4 kernel
    bool q4s = false, q6s = false, q4b = false, q6b = false;
    for (auto& it : items) {
      const bool small = it.count <= kDot4Max;
      q4s = q4s || (it.qtype == 0 && small); q6s = q6s || (it.qtype == 1 && small);
      q4b = q4b || (it.qtype == 0 && !small); q6b = q6b || (it.qtype == 1 && !small);
    }
    const Item* ip = (const Item*)ibuf.p;
    const int *xip = (const int*)pbuf.p, *yip = (const int*)pbuf.p + np;
    const int8_t* xdp = (const int8_t*)g_qprep.xd.p;
    const int64_t* xsp = (const int64_t*)g_qprep.xs.p;
    const int* lrp = (const int*)g_qprep.lr.p;
    if (q4s) hipLaunchKernelGGL(qk_dot4_kernel<0>, grid, dim3(256), 0, st, ip, xip, yip, xdp, xsp, lrp, rows, K, Y, ldy, fw, status, flag, kDot4Max);
    if (q6s) hipLaunchKernelGGL(qk_dot4_kernel<1>, grid, dim3(256), 0, st, ip, xip, yip, xdp, xsp, lrp, rows, K, Y, ldy, fw, status, flag, kDot4Max);
    if (q4b) hipLaunchKernelGGL(qk_mfma_kernel<0>, grid, dim3(256), 0, st, ip, xip, yip, xdp, xsp, lrp, rows, K, Y, ldy, fw, status, flag, kDot4Max);
    if (q6b) hipLaunchKernelGGL(qk_mfma_kernel<1>, grid, dim3(256), 0, st, ip, xip, yip, xdp, xsp, lrp, rows, K, Y, ldy, fw, status, flag, kDot4Max);
    gate = flag;
  }
  hipLaunchKernelGGL(qk_group_kernel, dim3((unsigned)((maxo + kRows - 1) / kRows), (unsigned)items.size()),
                     dim3(256), 0, st, (const Item*)ibuf.p, (const int*)pbuf.p, (const int*)pbuf.p + np, X, K, Y,
                     ldy, fw, status, gate);
  imie_prof_mark(IMIE_K_QK, st, false);
  IMIE_HIP(hipGetLastError());
  return IMIE_OK;
}

void silu_consts_nmc(int fa, int64_t* log2e, int64_t* dclip) {
  const int sh = 16 - fa;
  *log2e = sh >= 0 ? (94548 >> sh) : ((int64_t)94548 << -sh);
  *dclip = (((int64_t)fa + 2) << (2 * fa)) / *log2e;
}

int read_status_and(hipStream_t st, int* stat) {
  IMIE_HIP(hipMemcpyAsync(stat, g_mws.status.p, 4, hipMemcpyDeviceToHost, st));
  IMIE_HIP(hipStreamSynchronize(st));
  return IMIE_OK;
}

// every pair's three weights exist with the shapes of the call; checked on each call, since a handle's number can come to
// name another matrix (qk_free_all and new registrations)
bool moe_shapes_ok(const long long* gate_h, const long long* up_h, const long long* down_h, int64_t P, int64_t d_model,
                   int64_t e_ffn) {
  for (int64_t p = 0; p < P; ++p) {
    const QKWeight *g = qk_get(gate_h[p]), *u = qk_get(up_h[p]), *d = qk_get(down_h[p]);
    if (!g || !u || !d || g->out_f != e_ffn || g->nb * 256 != d_model || u->out_f != e_ffn || u->nb * 256 != d_model ||
        d->out_f != d_model || d->nb * 256 != e_ffn)
      return false;
  }
  return true;
}

// Batched MoE: P = m*k pairs (token-major, pair p belongs to token p / k). Pairs sharing a weight run in one
// item, so each expert's gate/up/down are read once per call. This form runs each projection as its own item list
// (any quantisation types); moe_batched below, which has checked the arguments, takes the fused expert kernels when the
// layout allows.
int moe_batched_items(const long long* gate_h, const long long* up_h, const long long* down_h, int m, int k,
                      const int64_t* h_dev, const int64_t* gates_dev, int64_t d_model, int64_t e_ffn, int fa, int fw,
                      int64_t* out_dev, hipStream_t st) {
  const int64_t P = (int64_t)m * k;
  if (g_mws.g.ensure((size_t)(P * e_ffn) * 8) || g_mws.u.ensure((size_t)(P * e_ffn) * 8) ||
      g_mws.d.ensure((size_t)(P * d_model) * 8) || g_mws.status.ensure(64))
    return IMIE_EARG;
  int64_t *gb = (int64_t*)g_mws.g.p, *ub = (int64_t*)g_mws.u.p, *db = (int64_t*)g_mws.d.p;
  int* status = (int*)g_mws.status.p;
  // group pairs by weight handle
  auto build = [&](const long long* hs, bool x_per_pair, std::vector<Item>& items, std::vector<int>& xi,
                   std::vector<int>& yi) {
    std::map<long long, std::vector<int>> groups;
    for (int64_t p = 0; p < P; ++p) groups[hs[p]].push_back((int)p);
    for (auto& kv : groups) {
      const QKWeight* w = qk_get(kv.first);
      Item it{w->p, w->out_f, w->nb, w->qtype, (int)xi.size(), (int)kv.second.size()};
      for (int p : kv.second) { xi.push_back(x_per_pair ? p : p / k); yi.push_back(p); }
      items.push_back(it);
    }
  };
  std::vector<Item> ig, iu, idn;
  std::vector<int> xg, yg, xu, yu, xd, yd;
  build(gate_h, false, ig, xg, yg);
  build(up_h, false, iu, xu, yu);
  build(down_h, true, idn, xd, yd);
  static DevBuf ib1, pb1, ib2, pb2, ib3, pb3;
  int rc = run_items(ig, xg, yg, h_dev, d_model, gb, e_ffn, fw, status, st, ib1, pb1);
  if (!rc) rc = run_items(iu, xu, yu, h_dev, d_model, ub, e_ffn, fw, status, st, ib2, pb2);
  if (rc) return rc;
  int64_t log2e, dclip;
  silu_consts_nmc(fa, &log2e, &dclip);
  const int64_t n = P * e_ffn;
  hipLaunchKernelGGL(qk_silu_mul_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, gb, ub, n, fa, log2e,
                     dclip, gb, status);
  IMIE_HIP(hipGetLastError());
  rc = run_items(idn, xd, yd, gb, e_ffn, db, d_model, fw, status, st, ib3, pb3);
  if (rc) return rc;
  hipLaunchKernelGGL(qk_combine_kernel, dim3((unsigned)(((int64_t)m * d_model + 255) / 256)), dim3(256), 0, st, db,
                     m, k, d_model, gates_dev, fa, out_dev, status);
  IMIE_HIP(hipGetLastError());
  return IMIE_OK;
}

// whether the fused kernels (Q4_K gate / up, Q6_K down) take the pairs
bool moe_fused_ok(const long long* gate_h, const long long* up_h, const long long* down_h, int64_t P, int fw) {
  bool fused = fw <= kMaxFw && qk_mfma_enabled();
  for (int64_t p = 0; p < P && fused; ++p)
    fused = qk_get(gate_h[p])->qtype == 0 && qk_get(up_h[p])->qtype == 0 && qk_get(down_h[p])->qtype == 1;
  return fused;
}

// A few tokens take moe1_gateup_kernel / moe1_down_kernel (every pair reads its expert's weights, no item lists, two
// launches); more tokens share decoded weights in the grouped kernels below. At 128 experts of 768, top-8, hidden 2048,
// this form against the grouped one for 1, 2, 3, 4 tokens: 23.5 / 41.3, 39 / 44.5, 57.5 / 58.6, 72 / 65 us.
// Two tokens only while their pairs' weights are few, since this form reads and decodes an expert for each of them; beyond
// eight experts a down workgroup needs two rounds of jobs, which count twice. Two tokens, d x e x experts a token (million
// weights), this form against the grouped one: 2048 x 768 x 8 (75) 38.4 / 44.8 us, 8192 x 1024 x 2 (101) 67 / 73, 4096 x
// 512 x 8 (101) 52.6 / 53.2, 4096 x 1536 x 4 (151) 64 / 57, 7168 x 2048 x 2 (176) 86 / 68, 4096 x 1024 x 8 (201) 71 / 64;
// 2048 x 256 x 16 (50) 42 / 45, 2048 x 512 x 16 (101) 52 / 45. One token is faster up to 201 (8192 x 4096 x 2: 77 / 84).
constexpr int kMoe1Tokens = 2;
constexpr int64_t kMoe1Weights = (int64_t)96 << 20;
bool moe1_ok(int64_t m, int64_t k, int64_t d_model, int64_t e_ffn) {
  const int64_t rounds = (kMoe1Out / kMoe1Rows * k + 31) / 32;
  return m <= kMoe1Tokens && k <= kMoe1MaxK && m * k <= kMoe1Pairs && d_model / 256 <= kG1MaxNb &&
         k * (e_ffn / 256) <= kG1MaxNb && d_model % kMoe1Out == 0 &&
         (m == 1 || m * k * 3 * d_model * e_ffn * rounds <= kMoe1Weights);
}

// handles already checked by the caller; res, ao: the residual and attention rows to add (both or none)
int moe1_launch(const long long* gate_h, const long long* up_h, const long long* down_h, int m, int k,
                const int64_t* h_dev, const int64_t* gates_dev, int64_t d_model, int64_t e_ffn, int fa, int fw,
                int64_t* out_dev, const int64_t* res, const int64_t* ao, int* status, hipStream_t st) {
  Moe1Args a = {};
  for (int p = 0; p < m * k; ++p) {
    a.w[0][p] = qk_get(gate_h[p])->p;
    a.w[1][p] = qk_get(up_h[p])->p;
    a.w[2][p] = qk_get(down_h[p])->p;
  }
  a.h = h_dev; a.gates = gates_dev; a.gu = (int64_t*)g_mws.g.p; a.out = out_dev; a.res = res; a.ao = ao;
  a.k = k; a.d_model = (int)d_model; a.e_ffn = (int)e_ffn; a.fa = fa; a.fw = fw; a.status = status;
  silu_consts_nmc(fa, &a.log2e, &a.dclip);
  imie_prof_mark(IMIE_K_QK, st, true);
  hipLaunchKernelGGL(moe1_gateup_kernel, dim3((unsigned)((e_ffn + 4 * kMoe1Wave - 1) / (4 * kMoe1Wave)), (unsigned)(m * k)), dim3(256),
                     (size_t)kQkLimbs * (d_model / 64) * kG1Unit, st, a);
  hipLaunchKernelGGL(moe1_down_kernel, dim3((unsigned)(d_model / kMoe1Out), (unsigned)m), dim3(512),
                     (size_t)kQkLimbs * k * (e_ffn / 64) * kG1Unit, st, a);
  imie_prof_mark(IMIE_K_QK, st, false);
  IMIE_HIP(hipGetLastError());
  return IMIE_OK;
}

// Batched MoE with the fused expert kernels (Q4_K gate/up, Q6_K down): one item per expert, its pairs listed
// once. Sequence: prep(h) -> gate/up + SiLU*up -> prep(gu) -> down -> combine. When an activation row needs more
// than kQkLimbs digit limbs, the prep sets a device flag: the fused kernels return at once and the exact VALU item
// kernels (enqueued behind them, gated by the same flag) compute that stage instead, with no host round trip.
int moe_batched(const long long* gate_h, const long long* up_h, const long long* down_h, int m, int k,
                const int64_t* h_dev, const int64_t* gates_dev, int64_t d_model, int64_t e_ffn, int fa, int fw,
                int64_t* out_dev, hipStream_t st) {
  const int64_t P = (int64_t)m * k;
  if (m <= 0 || k <= 0 || d_model <= 0 || e_ffn <= 0 || d_model % 256 || e_ffn % 256 || fa < 1 || fa > 28 || fw < 0 ||
      fw > 62)
    return IMIE_EARG;
  if (!moe_shapes_ok(gate_h, up_h, down_h, P, d_model, e_ffn)) return IMIE_EARG;
  if (!moe_fused_ok(gate_h, up_h, down_h, P, fw))
    return moe_batched_items(gate_h, up_h, down_h, m, k, h_dev, gates_dev, d_model, e_ffn, fa, fw, out_dev, st);
  if (moe1_ok(m, k, d_model, e_ffn)) {
    if (g_mws.g.ensure((size_t)(P * e_ffn) * 8) || g_mws.status.ensure(64)) return IMIE_EARG;
    return moe1_launch(gate_h, up_h, down_h, m, k, h_dev, gates_dev, d_model, e_ffn, fa, fw, out_dev, nullptr, nullptr,
                       (int*)g_mws.status.p, st);
  }
  if (g_mws.g.ensure((size_t)(P * e_ffn) * 8) || g_mws.u.ensure((size_t)(P * e_ffn) * 8) ||
      g_mws.d.ensure((size_t)(P * d_model) * 8) || g_mws.status.ensure(64))
    return IMIE_EARG;
  int64_t *gb = (int64_t*)g_mws.g.p, *ub = (int64_t*)g_mws.u.p, *db = (int64_t*)g_mws.d.p;
  int* status = (int*)g_mws.status.p;
  // experts = distinct (gate, up, down) handle triples; pairs listed expert by expert
  std::map<std::tuple<long long, long long, long long>, std::vector<int>> groups;
  for (int64_t p = 0; p < P; ++p) groups[std::make_tuple(gate_h[p], up_h[p], down_h[p])].push_back((int)p);
  const size_t ne = groups.size();
  std::vector<MoeItem> mi;
  std::vector<Item> ig, iu, idn;
  std::vector<int> ptok, ppair;
  mi.reserve(ne);
  for (auto& kv : groups) {
    const QKWeight* g = qk_get(std::get<0>(kv.first));
    const QKWeight* u = qk_get(std::get<1>(kv.first));
    const QKWeight* d = qk_get(std::get<2>(kv.first));
    const int first = (int)ptok.size(), count = (int)kv.second.size();
    mi.push_back(MoeItem{g->p, u->p, d->p, first, count});
    ig.push_back(Item{g->p, g->out_f, g->nb, g->qtype, first, count});
    iu.push_back(Item{u->p, u->out_f, u->nb, u->qtype, first, count});
    idn.push_back(Item{d->p, d->out_f, d->nb, d->qtype, first, count});
    for (int p : kv.second) { ptok.push_back(p / k); ppair.push_back(p); }
  }
  // one upload: [MoeItem x ne][Item gate x ne][Item up x ne][Item down x ne][ptok P][ppair P]
  static DevBuf meta;
  const size_t o_items = 0, o_ig = o_items + ne * sizeof(MoeItem), o_iu = o_ig + ne * sizeof(Item),
               o_id = o_iu + ne * sizeof(Item), o_pt = o_id + ne * sizeof(Item), o_pp = o_pt + (size_t)P * 4,
               total = o_pp + (size_t)P * 4;
  static std::vector<uint8_t> hb;                     // pageable staging: the async copy reads it before returning
  hb.resize(total);
  memcpy(hb.data() + o_items, mi.data(), ne * sizeof(MoeItem));
  memcpy(hb.data() + o_ig, ig.data(), ne * sizeof(Item));
  memcpy(hb.data() + o_iu, iu.data(), ne * sizeof(Item));
  memcpy(hb.data() + o_id, idn.data(), ne * sizeof(Item));
  memcpy(hb.data() + o_pt, ptok.data(), (size_t)P * 4);
  memcpy(hb.data() + o_pp, ppair.data(), (size_t)P * 4);
  if (meta.ensure(total)) return IMIE_EARG;
  IMIE_HIP(hipMemcpyAsync(meta.p, hb.data(), total, hipMemcpyHostToDevice, st));
  const uint8_t* mb = (const uint8_t*)meta.p;
  const MoeItem* d_items = (const MoeItem*)(mb + o_items);
  const Item *d_ig = (const Item*)(mb + o_ig), *d_iu = (const Item*)(mb + o_iu), *d_id = (const Item*)(mb + o_id);
  const int *d_pt = (const int*)(mb + o_pt), *d_pp = (const int*)(mb + o_pp);
  const int64_t prow = P > m ? P : m, pk = d_model > e_ffn ? d_model : e_ffn;
  if (g_qprep.xd.ensure((size_t)(kQkLimbs * prow * pk)) || g_qprep.lr.ensure((size_t)prow * 4) ||
      g_qprep.flag.ensure(64))
    return IMIE_EARG;
  int* flagA = (int*)g_qprep.flag.p;
  int* flagB = flagA + 1;
  int8_t* xdp = (int8_t*)g_qprep.xd.p;
  int* lrp = (int*)g_qprep.lr.p;
  int64_t log2e, dclip;
  silu_consts_nmc(fa, &log2e, &dclip);
  imie_prof_mark(IMIE_K_QK, st, true);
  // the wide-row flags start clear: the previous call's combine kernel cleared them (a fresh or foreign value
  // only costs a run of the exact fallbacks, whose results equal the fused kernels')
  // the fused expert kernels read no 16-element sums (their min terms are MFMA accumulations)
  hipLaunchKernelGGL(qk_prep_kernel, dim3((unsigned)m), dim3(256), 0, st, h_dev, (int64_t)m, d_model, xdp, nullptr, lrp,
                     flagA);
  hipLaunchKernelGGL(moe_gateup_kernel, dim3((unsigned)((e_ffn + 63) / 64),
                     (unsigned)ne), dim3(512), moe_lds_bytes((int)(d_model / 256)), st, d_items,
                     d_pt, d_pp, xdp, lrp, (int64_t)m, d_model, e_ffn, fw, fa, log2e, dclip,
                     moe_dq_max(d_model / 256, kMoeT4), gb, status, flagA);
  // exact VALU fallback of the gate/up stage (runs only when the prep flagged a wide activation row)
  const int64_t ntg = (e_ffn + kRows - 1) / kRows;
  hipLaunchKernelGGL(qk_gateup_gated_kernel, dim3(kGatedWgs2), dim3(256), 0, st, d_ig, d_iu, d_pt, d_pp, h_dev,
                     d_model, gb, ub, e_ffn, fw, fa, log2e, dclip, status, flagA, ntg, (int64_t)ne);
  // down over the P rows of gu
  hipLaunchKernelGGL(qk_prep_kernel, dim3((unsigned)P), dim3(256), 0, st, gb, P, e_ffn, xdp, nullptr, lrp, flagB);
  const int wtiles = (int64_t)ne * ((d_model + 63) / 64) >= kMoeDownWgs ? 2 : 1;
  hipLaunchKernelGGL(moe_down_kernel, dim3((unsigned)((d_model + 64 * wtiles - 1) / (64 * wtiles)), (unsigned)ne),
                     dim3(256), moe_lds_bytes((int)(e_ffn / 256)), st, d_items, d_pp, xdp, lrp, P, e_ffn, d_model,
                     wtiles, fw, moe_dq_max(e_ffn / 256, kMoeT6), db, status, flagB);
  hipLaunchKernelGGL(qk_group_gated_kernel, dim3(kGatedWgs), dim3(256), 0, st, d_id, d_pp, d_pp, gb, e_ffn, db,
                     d_model, fw, status, flagB, (int64_t)((d_model + kRows - 1) / kRows), (int64_t)ne);
  hipLaunchKernelGGL(qk_combine_kernel, dim3((unsigned)(((int64_t)m * d_model + 255) / 256)), dim3(256), 0, st, db,
                     m, k, d_model, gates_dev, fa, out_dev, status, flagA);
  imie_prof_mark(IMIE_K_QK, st, false);
  IMIE_HIP(hipGetLastError());
  return IMIE_OK;
}

int host_linear(const std::vector<int64_t>& handles, const int64_t* x, int64_t T, int fw, int64_t* out_flat) {
  // all handles share the input width; outputs concatenated handle-major (each T x out_f)
  hipStream_t st = imie_stream();
  const QKWeight* w0 = qk_get(handles[0]);
  const int64_t K = w0->nb * 256;
  int64_t total = 0;
  for (auto h : handles) total += T * qk_get(h)->out_f;
  if (g_mws.x.ensure((size_t)(T * K) * 8) || g_mws.y.ensure((size_t)total * 8) || g_mws.status.ensure(64))
    return IMIE_EARG;
  IMIE_HIP(hipMemcpyAsync(g_mws.x.p, x, (size_t)(T * K) * 8, hipMemcpyHostToDevice, st));
  IMIE_HIP(hipMemsetAsync(g_mws.status.p, 0, 4, st));
  prof(PM_H2D_CALLS); prof(PM_H2D_BYTES, (unsigned long long)(T * K * 8));
  int64_t off = 0;
  const bool one = T == 1 && gemv1_ok(w0->nb);
  for (size_t i0 = 0; one && i0 < handles.size(); i0 += kG1Items) {   // one row: all weights in one launch
    const QKWeight* ws[kG1Items];
    int64_t* ys[kG1Items];
    int cnt = 0;
    for (; cnt < kG1Items && i0 + cnt < handles.size(); ++cnt) {
      ws[cnt] = qk_get(handles[i0 + cnt]);
      ys[cnt] = (int64_t*)g_mws.y.p + off;
      off += ws[cnt]->out_f;
    }
    const int rc = gemv1_launch(ws, ys, cnt, (const int64_t*)g_mws.x.p, fw, (int*)g_mws.status.p, st);
    if (rc) return rc;
  }
  static DevBuf ib, pb;
  for (auto h : handles) {
    if (one) break;
    const QKWeight* w = qk_get(h);
    std::vector<Item> items{Item{w->p, w->out_f, w->nb, w->qtype, 0, (int)T}};
    std::vector<int> xi((size_t)T), yi((size_t)T);
    for (int64_t t = 0; t < T; ++t) { xi[(size_t)t] = (int)t; yi[(size_t)t] = (int)t; }
    int rc = run_items(items, xi, yi, (const int64_t*)g_mws.x.p, K, (int64_t*)g_mws.y.p + off, w->out_f, fw,
                       (int*)g_mws.status.p, st, ib, pb);
    if (rc) return rc;
    IMIE_HIP(hipStreamSynchronize(st));   // ib/pb are reused by the next handle
    off += T * w->out_f;
  }
  int stat = 0;
  if (read_status_and(st, &stat)) return IMIE_EARG;
  IMIE_HIP(hipMemcpy(out_flat, g_mws.y.p, (size_t)total * 8, hipMemcpyDeviceToHost));
  prof(PM_D2H_CALLS); prof(PM_D2H_BYTES, (unsigned long long)(total * 8));
  return stat ? IMIE_EOVF : IMIE_OK;
}

int64_t qk_register(const uint8_t* W, int64_t out_f, int64_t nb, int qtype) {
  if (!W || out_f <= 0 || nb <= 0 || (qtype != 0 && qtype != 1) || imie_device_ready() != 0) return -1;
  QKWeight w;
  w.out_f = out_f; w.nb = nb; w.qtype = qtype;
  w.bytes = (size_t)(out_f * nb) * (qtype == 0 ? 144 : 210);
  if (hipMalloc((void**)&w.p, w.bytes) != hipSuccess) return -1;
  if (hipMemcpy(w.p, W, w.bytes, hipMemcpyHostToDevice) != hipSuccess) { imie_free(w.p); return -1; }
  g_qk.push_back(w);
  ++g_qk_live;
  prof(PM_REG_CALLS); prof(PM_ALLOC_CALLS); prof(PM_ALLOC_BYTES, w.bytes);
  return (int64_t)g_qk.size() - 1;
}

}  // namespace

// ---- internal API for the resident attention bank (csrc/nmcbank.hip) --------------------------------------------
int imie_qk_info(int64_t h, int64_t* out_f, int64_t* nb, int* qtype, const uint8_t** p) {
  if (h < 0 || h >= (int64_t)g_qk.size() || !g_qk[(size_t)h].p) return IMIE_EARG;
  const QKWeight& w = g_qk[(size_t)h];
  if (out_f) *out_f = w.out_f;
  if (nb) *nb = w.nb;
  if (qtype) *qtype = w.qtype;
  if (p) *p = w.p;
  return IMIE_OK;
}

// int64 matrix [rows, cols] registered as qtype 2 (nb holds cols)
int64_t imie_qk_register_i64(const int64_t* W, int64_t rows, int64_t cols) {
  if (!W || rows <= 0 || cols <= 0 || imie_device_ready() != 0) return -1;
  QKWeight w;
  w.out_f = rows; w.nb = cols; w.qtype = 2;
  w.bytes = (size_t)(rows * cols) * 8;
  if (hipMalloc((void**)&w.p, w.bytes) != hipSuccess) return -1;
  if (hipMemcpy(w.p, W, w.bytes, hipMemcpyHostToDevice) != hipSuccess) { imie_free(w.p); return -1; }
  g_qk.push_back(w);
  ++g_qk_live;
  prof(PM_REG_CALLS); prof(PM_ALLOC_CALLS); prof(PM_ALLOC_BYTES, w.bytes);
  return (int64_t)g_qk.size() - 1;
}

// y[t, :] = (W . x[t, :]) >> fw for T device rows into device out (T x out_f); status gets IMIE_EOVF where the
// oracle's int64 conversion would raise
int imie_qk_linear_dev(int64_t h, const int64_t* x, int64_t T, int fw, int64_t* out, int* status, hipStream_t st) {
  const QKWeight* w = qk_get(h);
  if (!w || !x || !out || !status || T <= 0) return IMIE_EARG;
  if (T == 1 && gemv1_ok(w->nb)) return gemv1_launch(&w, &out, 1, x, fw, status, st);
  std::vector<Item> items{Item{w->p, w->out_f, w->nb, w->qtype, 0, (int)T}};
  std::vector<int> xi((size_t)T), yi((size_t)T);
  for (int64_t t = 0; t < T; ++t) { xi[(size_t)t] = (int)t; yi[(size_t)t] = (int)t; }
  static DevBuf ib[4], pb[4];
  static int slot = 0;
  slot = (slot + 1) & 3;                              // distinct item buffers for back-to-back launches
  return run_items(items, xi, yi, x, w->nb * 256, out, w->out_f, fw, status, st, ib[slot], pb[slot]);
}

// one row against cnt weights of the same input width (the Q / K / V projections of one token)
int imie_qk_linears_dev(const int64_t* hs, int cnt, const int64_t* x, int fw, int64_t* const* outs, int* status,
                        hipStream_t st) {
  const QKWeight* ws[kG1Items];
  bool one = cnt <= kG1Items;
  for (int i = 0; i < cnt && one; ++i) {
    if (!(ws[i] = qk_get(hs[i]))) return IMIE_EARG;
    one = ws[i]->nb == ws[0]->nb && gemv1_ok(ws[i]->nb);
  }
  if (one) return gemv1_launch(ws, outs, cnt, x, fw, status, st);
  for (int i = 0; i < cnt; ++i) {
    const int rc = imie_qk_linear_dev(hs[i], x, 1, fw, outs[i], status, st);
    if (rc) return rc;
  }
  return IMIE_OK;
}

// One token's MoE over k selected experts (host handle arrays), gates on the device, and the layer's residual:
// out = res + ao + moe (int64 wrap). Enqueued on st (no synchronisation); *status_dev gets IMIE_EOVF where the
// oracle's int64 conversions would raise.
int imie_qk_moe_dev(const long long* gate_h, const long long* up_h, const long long* down_h, int k,
                    const int64_t* h_dev, const int64_t* gates_dev, int64_t d_model, int64_t e_ffn, int fa, int fw,
                    const int64_t* res, const int64_t* ao, int64_t* moe, int64_t* out_dev, int* status_dev,
                    hipStream_t st) {
  if (!moe_shapes_ok(gate_h, up_h, down_h, k, d_model, e_ffn)) return IMIE_EARG;
  if (moe_fused_ok(gate_h, up_h, down_h, k, fw) && moe1_ok(1, k, d_model, e_ffn) && fa >= 1 && fa <= 28 && fw >= 0) {
    if (g_mws.g.ensure((size_t)(k * e_ffn) * 8)) return IMIE_EARG;
    return moe1_launch(gate_h, up_h, down_h, 1, k, h_dev, gates_dev, d_model, e_ffn, fa, fw, out_dev, res, ao,
                       status_dev, st);
  }
  if (g_mws.status.ensure(64)) return IMIE_EARG;
  hipLaunchKernelGGL(qk_flag_reset_kernel, dim3(1), dim3(1), 0, st, (int*)g_mws.status.p);
  const int rc = moe_batched(gate_h, up_h, down_h, 1, k, h_dev, gates_dev, d_model, e_ffn, fa, fw, moe, st);
  if (rc) return rc;
  hipLaunchKernelGGL(qk_add3_kernel, dim3((unsigned)((d_model + 255) / 256)), dim3(256), 0, st, res, ao, moe, d_model,
                     out_dev, (const int*)g_mws.status.p, status_dev);
  IMIE_HIP(hipGetLastError());
  return IMIE_OK;
}

extern "C" {

// fp16 -> fixed point as the Q4_K / Q6_K kernels compute it (fp16_fixed_fast), over n host values; synchronous.
// Test hook (no reference counterpart): the exhaustive check against the oracle's integer rule.
int imie_fp16_fixed_probe(const uint16_t* h, int64_t n, int fw, int64_t* out) {
  std::lock_guard<std::recursive_mutex> lk(imie_lock());
  if (!h || !out || n <= 0 || fw < 0 || fw > 62 || imie_device_ready() != 0) return IMIE_EARG;
  hipStream_t st = imie_stream();
  static DevBuf a, b;                                 // grow-only staging, like the other host-pointer entry points
  if (a.ensure((size_t)n * 2) || b.ensure((size_t)n * 8)) return IMIE_EARG;
  IMIE_HIP(hipMemcpyAsync(a.p, h, (size_t)n * 2, hipMemcpyHostToDevice, st));
  hipLaunchKernelGGL(fp16_fixed_probe_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, (const uint16_t*)a.p,
                     n, fw, (int64_t*)b.p);
  IMIE_HIP(hipGetLastError());
  IMIE_HIP(hipMemcpyAsync(out, b.p, (size_t)n * 8, hipMemcpyDeviceToHost, st));
  IMIE_HIP(hipStreamSynchronize(st));
  return IMIE_OK;
}

// nmc_qk_cuda.cu:755 `qk_cuda_abi_version`; the reference bridge requires 5 (qk_cuda.py:22, 83-92).
int qk_cuda_abi_version(void) { return 5; }

// nmc_qk_cuda.cu `qk_cuda_available`: 0 iff usable.
int qk_cuda_available(void) {
  std::lock_guard<std::recursive_mutex> lk(imie_lock());
  return imie_device_ready();
}

// nmc_qk_cuda.cu:720 `qk_linear_cuda` (qk_cuda.py:230-244): per-call weight upload, y [T, out_f].
int qk_linear_cuda(const uint8_t* W, const int64_t* x, long long T, long long out_f, long long n_blocks, int fw,
                   int qtype, int64_t* out) {
  std::lock_guard<std::recursive_mutex> lk(imie_lock());
  prof(PM_NATIVE_CALLS);
  if (!W || !x || !out || T < 0 || out_f <= 0 || n_blocks <= 0 || fw < 0 || fw > kMaxFw) return IMIE_EARG;
  if (T == 0) return IMIE_OK;
  const int64_t h = qk_register(W, out_f, n_blocks, qtype);
  if (h < 0) return IMIE_EARG;
  const int rc = host_linear({h}, x, T, fw, out);
  imie_free(g_qk[(size_t)h].p);
  g_qk[(size_t)h].p = nullptr;
  --g_qk_live;
  if (h == (int64_t)g_qk.size() - 1) g_qk.pop_back();
  return rc;
}

// nmc_qk_cuda.cu:1046 `qk_register_weight` (qk_cuda.py:252-270): raw Q4_K (0) / Q6_K (1) bytes -> handle.
long long qk_register_weight(const uint8_t* W, long long out_f, long long n_blocks, int qtype) {
  std::lock_guard<std::recursive_mutex> lk(imie_lock());
  return qk_register(W, out_f, n_blocks, qtype);
}

// nmc_qk_cuda.cu:1040 `qk_resident_reserve`: registry metadata only.
int qk_resident_reserve(long long count) {
  std::lock_guard<std::recursive_mutex> lk(imie_lock());
  if (count < 0) return IMIE_EARG;
  g_qk.reserve((size_t)count);
  return IMIE_OK;
}

// nmc_qk_cuda.cu:1252 `qk_apply_resident` (qk_cuda.py:387-397).
int qk_apply_resident(long long h, const int64_t* x, long long T, int fw, int64_t* out) {
  std::lock_guard<std::recursive_mutex> lk(imie_lock());
  prof(PM_RESIDENT_CALLS);
  if (!qk_get(h) || !x || !out || T < 0 || fw < 0 || fw > kMaxFw) return IMIE_EARG;
  if (T == 0) return IMIE_OK;
  return host_linear({(int64_t)h}, x, T, fw, out);
}

// nmc_qk_cuda.cu:1284 `qk_apply_resident_grouped` (qk_cuda.py:405-442): same-input projections, one H2D and
// one D2H; outputs concatenated handle-major. phase_ids only feed the Q/K/V/O counters.
int qk_apply_resident_grouped(const long long* handles, const int* phase_ids, int count, const int64_t* x,
                              long long rows, int fw, long long total, int64_t* out) {
  std::lock_guard<std::recursive_mutex> lk(imie_lock());
  prof(PM_GROUPED_CALLS);
  if (!handles || !x || !out || count <= 0 || count > 16 || rows <= 0 || fw < 0 || fw > kMaxFw) return IMIE_EARG;
  std::vector<int64_t> hs;
  int64_t K = -1, want = 0;
  for (int i = 0; i < count; ++i) {
    const QKWeight* w = qk_get(handles[i]);
    if (!w || (K >= 0 && w->nb * 256 != K)) return IMIE_EARG;
    K = w->nb * 256;
    want += rows * w->out_f;
    hs.push_back(handles[i]);
    if (phase_ids) {
      const int ph = phase_ids[i];
      prof(ph == 1 ? PM_Q_CALLS : ph == 2 ? PM_K_CALLS : ph == 3 ? PM_V_CALLS : ph == 4 ? PM_O_CALLS : PM_OTHER_CALLS);
    }
  }
  if (want != total) return IMIE_EARG;
  return host_linear(hs, x, rows, fw, out);
}

// DP4A entries (nmc_qk_cuda.cu:1932, :2003): on gfx950 the same exact kernel serves every limb count, so these
// return the apply_resident result after the reference's argument checks (Ln in [1, 8], matching qtype).
int qk_apply_resident_q6k_dp4a(long long h, const int64_t* x, long long T, int fw, int Ln, int64_t* out) {
  std::lock_guard<std::recursive_mutex> lk(imie_lock());
  const QKWeight* w = qk_get(h);
  if (!w || w->qtype != 1 || Ln < 1 || Ln > 8) return IMIE_EARG;
  return qk_apply_resident(h, x, T, fw, out);
}
int qk_apply_resident_q4k_dp4a(long long h, const int64_t* x, long long T, int fw, int Ln, int64_t* out) {
  std::lock_guard<std::recursive_mutex> lk(imie_lock());
  const QKWeight* w = qk_get(h);
  if (!w || w->qtype != 0 || Ln < 1 || Ln > 8) return IMIE_EARG;
  return qk_apply_resident(h, x, T, fw, out);
}

// nmc_qk_cuda.cu:2203-2254 `qk_moe_ffn_batched` (qk_cuda.py:1073-1101): host h [m, d_model], gates [m*k],
// handles flattened token-major; out [m, d_model]. rc 2 where the oracle's int64 conversions would raise.
int qk_moe_ffn_batched(const long long* gate_h, const long long* up_h, const long long* down_h, int m, int k,
                       const int64_t* h, const int64_t* gates, long long d_model, long long e_ffn, int fa, int fw,
                       int64_t* out) {
  std::lock_guard<std::recursive_mutex> lk(imie_lock());
  prof(PM_MOE_BATCHED_CALLS);
  if (!gate_h || !up_h || !down_h || !h || !gates || !out || m <= 0 || k <= 0) return IMIE_EARG;
  hipStream_t st = imie_stream();
  const int64_t P = (int64_t)m * k;
  if (g_mws.x.ensure((size_t)(m * d_model) * 8) || g_mws.gates.ensure((size_t)P * 8) ||
      g_mws.out.ensure((size_t)(m * d_model) * 8) || g_mws.status.ensure(64))
    return IMIE_EARG;
  IMIE_HIP(hipMemcpyAsync(g_mws.x.p, h, (size_t)(m * d_model) * 8, hipMemcpyHostToDevice, st));
  IMIE_HIP(hipMemcpyAsync(g_mws.gates.p, gates, (size_t)P * 8, hipMemcpyHostToDevice, st));
  IMIE_HIP(hipMemsetAsync(g_mws.status.p, 0, 4, st));
  int rc = moe_batched(gate_h, up_h, down_h, m, k, (const int64_t*)g_mws.x.p, (const int64_t*)g_mws.gates.p,
                       d_model, e_ffn, fa, fw, (int64_t*)g_mws.out.p, st);
  if (rc) return rc;
  int stat = 0;
  if (read_status_and(st, &stat)) return IMIE_EARG;
  if (stat) return IMIE_EOVF;
  IMIE_HIP(hipMemcpy(out, g_mws.out.p, (size_t)(m * d_model) * 8, hipMemcpyDeviceToHost));
  return IMIE_OK;
}

// Guarded-limb batched entry (nmc_qk_cuda.cu:2261): exact for every activation here, never rc 2 for the limb
// envelope; overflow of the int64 results still returns 2 (the caller then runs the int128 entry, which agrees).
int qk_moe_ffn_batched_dp4a(const long long* gate_h, const long long* up_h, const long long* down_h, int m, int k,
                            const int64_t* h, const int64_t* gates, long long d_model, long long e_ffn, int fa, int fw,
                            int64_t* out) {
  prof(PM_MOE_BATCHED_DP4A_CALLS);
  return qk_moe_ffn_batched(gate_h, up_h, down_h, m, k, h, gates, d_model, e_ffn, fa, fw, out);
}

// nmc_qk_cuda.cu:1816 `qk_moe_ffn` (qk_cuda.py:1104-1124): one token, n_e selected experts, out [d_model].
int qk_moe_ffn(const long long* gate_h, const long long* up_h, const long long* down_h, int n_e, const int64_t* h,
               const int64_t* gates, long long d_model, long long e_ffn, int fa, int fw, int64_t* out) {
  prof(PM_MOE_CALLS);
  return qk_moe_ffn_batched(gate_h, up_h, down_h, 1, n_e, h, gates, d_model, e_ffn, fa, fw, out);
}
int qk_moe_ffn_dp4a(const long long* gate_h, const long long* up_h, const long long* down_h, int n_e, const int64_t* h,
                    const int64_t* gates, long long d_model, long long e_ffn, int fa, int fw, int64_t* out) {
  return qk_moe_ffn(gate_h, up_h, down_h, n_e, h, gates, d_model, e_ffn, fa, fw, out);
}

// Device-pointer batched MoE (no reference counterpart): h_dev [m, d_model], gates_dev [m*k], out_dev [m, d_model];
// status_dev receives bit 2 on an int64 envelope miss. Asynchronous on `stream`.
int imie_moe_ffn_batched_dev(const long long* gate_h, const long long* up_h, const long long* down_h, int m, int k,
                             const int64_t* h_dev, const int64_t* gates_dev, long long d_model, long long e_ffn,
                             int fa, int fw, int64_t* out_dev, void* stream) {
  std::lock_guard<std::recursive_mutex> lk(imie_lock());
  if (!gate_h || !up_h || !down_h || !h_dev || !gates_dev || !out_dev) return IMIE_EARG;
  if (g_mws.status.ensure(64)) return IMIE_EARG;
  return moe_batched(gate_h, up_h, down_h, m, k, h_dev, gates_dev, d_model, e_ffn, fa, fw, out_dev,
                     (hipStream_t)stream);
}

int imie_moe_status(int clear, void* stream) {
  std::lock_guard<std::recursive_mutex> lk(imie_lock());
  if (g_mws.status.ensure(64)) return -1;
  hipStream_t st = (hipStream_t)stream;
  if (clear) return hipMemsetAsync(g_mws.status.p, 0, 4, st) == hipSuccess ? 0 : -1;
  int stat = 0;
  if (hipMemcpyAsync(&stat, g_mws.status.p, 4, hipMemcpyDeviceToHost, st) != hipSuccess ||
      hipStreamSynchronize(st) != hipSuccess)
    return -1;
  return stat;
}

void qk_free_all(void) {
  std::lock_guard<std::recursive_mutex> lk(imie_lock());
  (void)hipDeviceSynchronize();
  for (auto& w : g_qk) if (w.p) { imie_free(w.p); prof(PM_FREE_CALLS); }
  g_qk.clear();
  g_qk_live = 0;
}

long long qk_resident_count(void) { return (long long)g_qk_live; }
long long qk_resident_capacity(void) { return (long long)g_qk.capacity(); }
long long qk_moe_workspace_allocations(void) { return 0; }
unsigned long long qk_moe_workspace_bytes(void) {
  return (unsigned long long)(g_mws.g.cap + g_mws.u.cap + g_mws.d.cap + g_mws.x.cap + g_mws.out.cap);
}
void qk_moe_workspace_release(void) {
  std::lock_guard<std::recursive_mutex> lk(imie_lock());
  (void)hipDeviceSynchronize();
  g_mws.g.release(); g_mws.u.release(); g_mws.d.release(); g_mws.x.release(); g_mws.out.release();
}

void qk_profile_reset(void) { memset(g_prof, 0, sizeof(g_prof)); }
void qk_profile_set_enabled(int enabled) { g_prof_on = enabled ? 1 : 0; }
// Copies min(capacity, PM_COUNT) counters; returns the number of counters the library keeps.
int qk_profile_snapshot(unsigned long long* out, int capacity) {
  if (out) for (int i = 0; i < capacity && i < PM_COUNT; ++i) out[i] = g_prof[i];
  return PM_COUNT;
}

}  // extern "C"
