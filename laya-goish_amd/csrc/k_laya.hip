// Kernels of the Laya encoder (src/models/laya/model.rs:301-416, src/tensor.rs:103-192) that the
// decoder path does not have: LayerNorm (with optional weight and bias, into f16 planes or f32,
// optionally gathering rows and adding a per-sequence type row), bidirectional RoPE attention
// with a local window, and the small pieces of the decision tail.  Projections and MLPs run on
// the shared MFMA GEMM (GEGLU and ReLU epilogues).
#include <hip/hip_runtime.h>

#include <cfloat>

#include "common.h"
#include "kernels.h"
#include "f16split.h"
#include "wave.h"

namespace lg {
namespace {

constexpr int kT = 256;

__device__ float block_sum_ln(float v, float *red) {
  v = wave_sum_dpp(v);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  return (red[0] + red[1]) + (red[2] + red[3]);
}

__device__ __forceinline__ float gelu_tanh_f(float x) {
  return 0.5f * x * (1.0f + tanhf(0.7978845608028654f * x * (1.0f + 0.044715f * x * x)));
}

// One workgroup per output row: y = (x - mean) * (1/sqrt(var + eps)) * w + b (+ add row), the
// row read once into registers (d <= 4096, d % 4 == 0).  Row r of the output reads input row
// rows[r] (rows == nullptr: r).  Output: f16 hi/lo planes (y16, y16lo) or f32 (y32).  The add
// row (f32 [3][d]) is add + sel[seq[r]] * d.
template <int NI>
__global__ __launch_bounds__(kT) void layer_norm_kernel(const float *__restrict__ x, const int32_t *__restrict__ rows,
                                                        int d, const float *__restrict__ w, const float *__restrict__ b,
                                                        float eps, const float *__restrict__ add,
                                                        const int32_t *__restrict__ seq, const int32_t *__restrict__ sel,
                                                        _Float16 *__restrict__ y16, _Float16 *__restrict__ y16lo,
                                                        float *__restrict__ y32) {
  __shared__ float red[8];
  const int r = blockIdx.x;
  const float4 *row = reinterpret_cast<const float4 *>(x + int64_t(rows ? rows[r] : r) * d);
  const int n4 = d >> 2;
  const float *addrow = add ? add + int64_t(sel[seq[r]]) * d : nullptr;
  // the row, its weights, biases and added row in one round trip (clamped indices: no load waits for a sum), 16 bytes each
  // (weights after the two sums: 31,488 rows of 768 37.9 us against 34.4, 45 rows 3.5 against 3.2)
  float4 v[NI], wr[NI], br[NI], ar[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int k = min(int(threadIdx.x) + i * kT, n4 - 1);
    v[i] = row[k];
    wr[i] = w ? reinterpret_cast<const float4 *>(w)[k] : make_float4(1.0f, 1.0f, 1.0f, 1.0f);
    br[i] = b ? reinterpret_cast<const float4 *>(b)[k] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    ar[i] = addrow ? reinterpret_cast<const float4 *>(addrow)[k] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  }
  float s = 0.0f;
#pragma unroll
  for (int i = 0; i < NI; ++i)
    if (int(threadIdx.x) + i * kT < n4) s += (v[i].x + v[i].y) + (v[i].z + v[i].w);
  const float mean = block_sum_ln(s, red) / float(d);
  float q = 0.0f;
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int k = threadIdx.x + i * kT;
    if (k < n4) {
      const float a = v[i].x - mean, bb = v[i].y - mean, c = v[i].z - mean, e = v[i].w - mean;
      q += (a * a + bb * bb) + (c * c + e * e);
    }
  }
  const float scale = 1.0f / sqrtf(block_sum_ln(q, red + 4) / float(d) + eps);
  // a thread's four consecutive values: one 16-byte f32 or 8-byte store per f16 plane
  typedef _Float16 half4_ __attribute__((ext_vector_type(4)));
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int k = threadIdx.x + i * kT;
    if (k >= n4) continue;
    const float in[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
    const float wv[4] = {wr[i].x, wr[i].y, wr[i].z, wr[i].w}, bv[4] = {br[i].x, br[i].y, br[i].z, br[i].w},
                av[4] = {ar[i].x, ar[i].y, ar[i].z, ar[i].w};
    float4v o;
    half4_ h4, l4;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      o[e] = (in[e] - mean) * scale * wv[e] + bv[e];
      if (addrow) o[e] = o[e] + av[e];
      _Float16 h, hl;
      split_f16(o[e], h, hl);
      h4[e] = h;
      l4[e] = hl;
    }
    const int64_t at = int64_t(r) * d + 4 * k;
    if (y32) {
      *reinterpret_cast<float4v *>(y32 + at) = o;
    } else {
      *reinterpret_cast<half4_ *>(y16 + at) = h4;
      if (y16lo) *reinterpret_cast<half4_ *>(y16lo + at) = l4;
    }
  }
}

constexpr int kHD = 64;

// RoPE in place on the q and k parts of q|k|v rows [T][3d] (model.rs:336-350 rotates q and k
// before attention): pairs (j, j + 32) of every 64-wide head, angle tables [pos][64].
__global__ __launch_bounds__(kT) void laya_rope_kernel(float *__restrict__ qkv, int d, const float *__restrict__ cosT,
                                                       const float *__restrict__ sinT,
                                                       const int32_t *__restrict__ tok_pos) {
  const int t = blockIdx.x;
  const int p = tok_pos[t];
  float *row = qkv + int64_t(t) * 3 * d;
  const float *cs = cosT + int64_t(p) * kHD, *sn = sinT + int64_t(p) * kHD;
  for (int e = threadIdx.x; e < d; e += kT) {  // 2 parts x (d / 64) heads x 32 pairs
    const int part = e / (d / 2), rem = e % (d / 2), hh = rem / 32, j = rem % 32;
    float *x = row + part * d + hh * kHD;
    float a, c;
    rope_pair(x[j], x[j + 32], cs[j], sn[j], cs[j + 32], sn[j + 32], a, c);  // as the wide GEMM's epilogue
    x[j] = a;
    x[j + 32] = c;
  }
}

// Bidirectional attention over q|k|v rows [T][3d] (f32, q and k already rotated), head dim 64, on
// v_mfma_f32_16x16x32_f16 with every f32 operand split into f16 hi + lo parts and three products per pair (lo.hi,
// hi.lo, hi.hi; lo.lo is below f32 rounding), f32 accumulation.  Keys j with |i - j| <= window (window < 0: the whole
// sequence); scores q.k / sqrt(64) in base 2; online softmax in f32.  Output f16 planes [T][d].
//
// One workgroup per (group of at most four consecutive 32-row tiles of one sequence, head): its four waves walk the same
// 64-key blocks (aligned to the sequence's start, so a query's arithmetic depends on its position only), and each
// block's K and V rows are read, split and staged in LDS once for up to 128 queries, V transposed, the next block's rows
// on their way in registers.  (The former form gave every 16 queries a workgroup that read and split all keys
// again, on the 16x16x16 instruction: 657 us a full and 301 a windowed layer of 64 inputs of 492 tokens, 12 heads, against
// 207 and 125.)  QB 16-query blocks a wave: 2, a wave takes a tile; 1, half a tile, two workgroups (z) a group, when whole
// groups would leave CUs idle.
// S^T = K Q^T in 16 x 16 blocks: lane l feeds row lr = l % 16 of key block (ck, hh), which is key ck * 32 + 8 (lr / 4) + 4 hh +
// lr % 4, so that it receives, for query lr, keys ck * 32 + 8 qg + 4 hh + 0..3, qg = l / 16: blocks (ck, 0) and (ck, 1)
// together are the eight keys its P^T operand of O^T = V^T P^T takes (the decoder's prefill attention has the same form).
// Rounding: a block's output is summed from zero, its small products first, and added to the running O once, so O is rounded
// once per 64 keys and not with each of six products (an MFMA's own sum truncates).  The exponent is one fused operation on the
// raw score.  Error against 64 bits over 492-token inputs, this form / one chain with a rounded product / the former four
// chains of a quarter of the keys: flat scores 4.0 / 4.6 / 4.1 e-7, scores of deviation 4 3.8 / 4.6 / 5.1 e-7; the same time.
// LDS: 16-byte chunk x of a K row at slot x ^ kswz(row); V rows (one dim, 64 keys) with one pad slot: operand reads
// without bank conflicts.
// scores to base-2 units; applied to them and not to q, whose f16 range stays the operand's own
constexpr float kScoreLog2 = 0.125f * 1.44269504088896341f;
constexpr int kKB = 64;                     // keys per block
constexpr int kKSlots = kKB * 8, kVSlots = kHD * 9;  // 16-byte slots of a plane

__device__ __forceinline__ int laya_kswz(int row) { return (row & 3) | (((row >> 3) & 1) << 2); }

template <int QB>
__global__ __launch_bounds__(256, 2) void laya_attn_kernel(const float *__restrict__ qkv, int d, int window, int ngroups,
                                                           int per_head, const int32_t *__restrict__ grp_first,
                                                           const int32_t *__restrict__ grp_count,
                                                           const int32_t *__restrict__ tile_row0,
                                                           const int32_t *__restrict__ tile_pos0,
                                                           const int32_t *__restrict__ tile_n,
                                                           const int32_t *__restrict__ tile_seq,
                                                           const int32_t *__restrict__ seq_n, _Float16 *__restrict__ y,
                                                           _Float16 *__restrict__ ylo) {
  __shared__ __align__(16) f16x8 lds[2 * kKSlots + 2 * kVSlots];
  f16x8 *const Kh = lds, *const Kl = Kh + kKSlots, *const Vh = Kl + kKSlots, *const Vl = Vh + kVSlots;
  // workgroups go to the 8 XCDs round-robin; each XCD takes a contiguous range of (head, group) pairs, groups fastest, so
  // the workgroups of one sequence and head read its rows through one L2
  const int total = gridDim.x, xcd = blockIdx.x % 8, per = total / 8, rem = total % 8;
  const int logical = xcd * per + min(xcd, rem) + blockIdx.x / 8;
  const int h = logical / per_head, part = logical % per_head, grp = part % ngroups, z = part / ngroups;
  const int t0 = grp_first[grp], cnt = grp_count[grp];
  const int first = QB == 2 ? 0 : 2 * z, last = min(cnt, QB == 2 ? 4 : first + 2) - 1;
  if (first >= cnt) return;  // whole workgroup, before any barrier
  const int tid = threadIdx.x, w = tid >> 6, l = tid & 63, lr = l & 15, qg = l >> 4;
  const int ti = QB == 2 ? w : first + w / 2, sub = QB == 2 ? 0 : 16 * (w & 1);
  const int tile = t0 + min(ti, last);
  const int nq = tile_n[tile] - sub;  // queries of this wave: rows sub .. sub + min(nq, 16 QB) of the tile
  const bool active = ti <= last && nq > 0;
  const int row0 = tile_row0[tile] + sub, pos0 = tile_pos0[tile] + sub;
  const int n = seq_n[tile_seq[t0]];
  const int ld = 3 * d;
  const float *kbase = qkv + int64_t(tile_row0[t0] - tile_pos0[t0]) * ld + d + h * kHD;  // key rows of the sequence
  const int plast = tile_pos0[t0 + last] + tile_n[t0 + last];
  const int wlo = window < 0 ? 0 : max(0, tile_pos0[t0 + first] - window), whi = window < 0 ? n : min(n, plast + window);
  const int kb1 = (whi + kKB - 1) / kKB;

  f16x8 qh[QB][2], ql[QB][2];
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    // rows past the tile repeat its last row and are never written
    const float *qr = qkv + int64_t(row0 - sub + min(sub + qb * 16 + lr, sub + nq - 1)) * ld + h * kHD + 8 * qg;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      float v[8];
#pragma unroll
      for (int e = 0; e < 2; ++e) *reinterpret_cast<float4v *>(v + 4 * e) = *reinterpret_cast<const float4v *>(qr + 32 * c + 4 * e);
      split8_pk(v, qh[qb][c], ql[qb][c]);
    }
  }
  float4v acc[QB][4];
  float m[QB], lsum[QB];
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
#pragma unroll
    for (int b = 0; b < 4; ++b) acc[qb][b] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
    m[qb] = -1e30f;  // finite: 2^(-inf - m) = 0 while no key of a window has been seen
    lsum[qb] = 0.0f;
  }
  // this thread's part of a block: K chunks of rows tid / 8 and 32 + tid / 8, V of dim l, keys 16 w .. 16 w + 15 (key rows
  // past the sequence repeat its last row and are masked)
  float4v kf[2][2];
  float vf[16];
  auto load = [&](int kb) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const float *kr = kbase + int64_t(min(kb * kKB + 32 * i + (tid >> 3), n - 1)) * ld + (tid & 7) * 8;
      kf[i][0] = *reinterpret_cast<const float4v *>(kr);
      kf[i][1] = *reinterpret_cast<const float4v *>(kr + 4);
    }
#pragma unroll
    for (int e = 0; e < 16; ++e) vf[e] = kbase[int64_t(min(kb * kKB + 16 * w + e, n - 1)) * ld + d + l];
  };
  auto stage = [&] {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      float v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = kf[i][e / 4][e % 4];
      const int row = 32 * i + (tid >> 3), slot = row * 8 + ((tid & 7) ^ laya_kswz(row));
      split8_pk(v, Kh[slot], Kl[slot]);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) split8_pk(vf + 8 * i, Vh[l * 9 + 2 * w + i], Vl[l * 9 + 2 * w + i]);
  };
  const int kr0 = 8 * (lr >> 2) + (lr & 3), ksw = laya_kswz(kr0);
  load(wlo / kKB);
  for (int kb = wlo / kKB; kb < kb1; ++kb) {
    if (kb > wlo / kKB) __syncthreads();  // every wave is done with the previous block
    stage();
    __syncthreads();
    if (kb + 1 < kb1) load(kb + 1);
    const int k0 = kb * kKB;
    // a block outside every window of the wave adds nothing
    if (!active || (window >= 0 && (k0 + kKB - 1 < pos0 - window || k0 > pos0 + min(nq, 16 * QB) - 1 + window))) continue;
    float4v s[QB][2][2];
#pragma unroll
    for (int qb = 0; qb < QB; ++qb)
#pragma unroll
      for (int i = 0; i < 4; ++i) s[qb][i / 2][i % 2] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
    // the small products of both halves of the head dim first, then the two hi.hi: two roundings at a score's magnitude
#pragma unroll
    for (int ck = 0; ck < 2; ++ck) {
      f16x8 kh[2][2], kl[2][2];  // [hh][c]
#pragma unroll
      for (int hh = 0; hh < 2; ++hh)
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          const int slot = (ck * 32 + kr0 + 4 * hh) * 8 + ((4 * c + qg) ^ ksw);
          kh[hh][c] = Kh[slot];
          kl[hh][c] = Kl[slot];
        }
#pragma unroll
      for (int n = 0; n < 6; ++n) {
        const int c = n % 2;
#pragma unroll
        for (int hh = 0; hh < 2; ++hh)
#pragma unroll
          for (int qb = 0; qb < QB; ++qb)
            s[qb][ck][hh] = __builtin_amdgcn_mfma_f32_16x16x32_f16(n < 2 ? kl[hh][c] : kh[hh][c],
                                                                   n / 2 == 1 ? ql[qb][c] : qh[qb][c], s[qb][ck][hh], 0, 0, 0);
      }
    }
    if (k0 + kKB > n || (window >= 0 && (k0 + kKB - 1 - pos0 > window || pos0 + 16 * QB - 1 - k0 > window))) {
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) {
        const int qpos = pos0 + qb * 16 + lr;
        const int hi = min(n - 1, window < 0 ? n - 1 : qpos + window) - k0 - 8 * qg;
        const int lo = (window < 0 ? 0 : qpos - window) - k0 - 8 * qg;
#pragma unroll
        for (int ck = 0; ck < 2; ++ck)
#pragma unroll
          for (int hh = 0; hh < 2; ++hh)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int j = ck * 32 + 4 * hh + e;
              if (j > hi || j < lo) s[qb][ck][hh][e] = -INFINITY;
            }
      }
    }
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
      float mt = -INFINITY;
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) mt = fmaxf(mt, s[qb][i / 2][i % 2][e]);
      mt = fmaxf(mt, __shfl_xor(mt, 16));
      mt = fmaxf(mt, __shfl_xor(mt, 32));
      mt *= kScoreLog2;
      // The exponent base m moves when a score exceeds it by more than 2 (an exponent's rounding grows with its size); lanes
      // that keep theirs multiply by exactly 1.  Probabilities are held 2^12 times larger (an exact factor that cancels in
      // O / l), which keeps the lo part of a small one clear of the f16 subnormals' 2^-24 floor; their sum is taken pairwise.
      const bool grow = mt > m[qb] + 2.0f;
      if (__any(grow)) {
        const float mn = grow ? mt : m[qb];
        const float alpha = __builtin_amdgcn_exp2f(m[qb] - mn);
        lsum[qb] *= alpha;
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[qb][b][r] *= alpha;
        m[qb] = mn;
      }
      float part[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float4v &p = s[qb][i / 2][i % 2];
#pragma unroll
        for (int e = 0; e < 4; ++e) p[e] = __builtin_amdgcn_exp2f(fmaf(p[e], kScoreLog2, -m[qb])) * 4096.0f;
        part[i] = (p[0] + p[1]) + (p[2] + p[3]);
      }
      float rs = (part[0] + part[1]) + (part[2] + part[3]);
      rs += __shfl_xor(rs, 16);
      rs += __shfl_xor(rs, 32);
      lsum[qb] += rs;
    }
    f16x8 ph[QB][2], pl[QB][2];
#pragma unroll
    for (int qb = 0; qb < QB; ++qb)
#pragma unroll
      for (int ck = 0; ck < 2; ++ck) {
        float pv[8];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          pv[e] = s[qb][ck][0][e];
          pv[4 + e] = s[qb][ck][1][e];
        }
        split8_pk(pv, ph[qb][ck], pl[qb][ck]);
      }
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      f16x8 vh[2], vl[2];
#pragma unroll
      for (int ck = 0; ck < 2; ++ck) {
        const int slot = (b * 16 + lr) * 9 + 4 * ck + qg;
        vh[ck] = Vh[slot];
        vl[ck] = Vl[slot];
      }
      float4v t[QB];
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) t[qb] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int n = 0; n < 6; ++n)
#pragma unroll
        for (int qb = 0; qb < QB; ++qb)
          t[qb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(n < 2 ? vl[n % 2] : vh[n % 2], n / 2 == 1 ? pl[qb][n % 2] : ph[qb][n % 2], t[qb], 0, 0, 0);
#pragma unroll
      for (int qb = 0; qb < QB; ++qb)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[qb][b][r] += t[qb][r];
    }
  }
  if (!active) return;
  // acc[qb][b][r]: dim 16 b + 4 qg + r of query qb * 16 + lr
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    if (qb * 16 + lr >= nq) continue;
    const float inv = 1.0f / lsum[qb];
    const int64_t base = int64_t(row0 + qb * 16 + lr) * d + h * kHD + 4 * qg;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      typedef _Float16 half4v __attribute__((ext_vector_type(4)));
      half4v oh, ol;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        _Float16 hi, lo;
        split_f16(acc[qb][b][j] * inv, hi, lo);
        oh[j] = hi;
        ol[j] = lo;
      }
      *reinterpret_cast<half4v *>(y + base + 16 * b) = oh;
      if (ylo) *reinterpret_cast<half4v *>(ylo + base + 16 * b) = ol;
    }
  }
}

__global__ void gelu_inplace_kernel(float *__restrict__ x, int64_t n) {
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) x[i] = gelu_tanh_f(x[i]);
}

// model.rs:392-403, one workgroup per sequence: pooled = [h[first row], top1, top1 - top2,
// entropy / ln max(k, 2), max(k, 2) / 255] from the softmax of the sequence's option logits.
__global__ __launch_bounds__(kT) void laya_act_features_kernel(const float *__restrict__ h, int d,
                                                               const int32_t *__restrict__ seq_row0,
                                                               const int32_t *__restrict__ lg_first,
                                                               const int32_t *__restrict__ lg_count,
                                                               const float *__restrict__ logits,
                                                               float *__restrict__ pooled) {
  const int sq = blockIdx.x;
  const float *row = h + int64_t(seq_row0[sq]) * d;
  float *out = pooled + int64_t(sq) * (d + 4);
  for (int j = threadIdx.x; j < d; j += kT) out[j] = row[j];
  if (threadIdx.x == 0) {
    const int k = lg_count[sq];
    const float *z = logits + lg_first[sq];
    float mx = -INFINITY;
    for (int i = 0; i < k; ++i) mx = fmaxf(mx, z[i]);
    float p[16], sum = 0.0f;
    for (int i = 0; i < k; ++i) {
      p[i] = expf(z[i] - mx);
      sum += p[i];
    }
    float top1 = 0.0f;
    for (int i = 0; i < k; ++i) {
      p[i] = p[i] / sum;
      top1 = fmaxf(top1, p[i]);
    }
    float top2 = 0.0f, es = 0.0f;
    for (int i = 0; i < k; ++i) {
      top2 = fmaxf(top2, p[i] * (top1 - p[i]) / ((top1 - p[i]) + 1e-6f));
      es += p[i] * logf(fmaxf(p[i], 1e-9f));
    }
    const float kk = float(k > 2 ? k : 2);
    out[d] = top1;
    out[d + 1] = top1 - top2;
    out[d + 2] = -es / logf(kk);
    out[d + 3] = kk / 255.0f;
  }
}

}  // namespace

void launch_layer_norm(const float *x, const int32_t *rows, int nrows, int d, const float *w, const float *b, float eps,
                       const float *add, const int32_t *seq, const int32_t *sel, _Float16 *y16, _Float16 *y16lo,
                       float *y32, hipStream_t st) {
  LG_REQUIRE(nrows > 0 && d > 0 && d % 4 == 0 && d <= 4 * 4 * kT, "layer norm: d=%d outside 4..4096 (multiple of 4)", d);
  LG_REQUIRE((y32 != nullptr) != (y16 != nullptr), "layer norm: exactly one output form");
  LG_REQUIRE(!add || (seq && sel), "layer norm: an add row needs its selectors");
  const auto fn = d <= 4 * kT ? layer_norm_kernel<1> : d <= 8 * kT ? layer_norm_kernel<2> : layer_norm_kernel<4>;
  hipLaunchKernelGGL(fn, dim3(nrows), dim3(kT), 0, st, x, rows, d, w, b, eps, add, seq, sel, y16, y16lo, y32);
  HIP_CHECK(hipGetLastError());
}

void launch_laya_rope(float *qkv, int T, int d, int hd, const float *cosT, const float *sinT, const int32_t *tok_pos,
                      hipStream_t st) {
  LG_REQUIRE(hd == kHD && T > 0 && d % kHD == 0 && cosT && sinT && tok_pos, "laya rope: bad shape");
  hipLaunchKernelGGL(laya_rope_kernel, dim3(T), dim3(kT), 0, st, qkv, d, cosT, sinT, tok_pos);
  HIP_CHECK(hipGetLastError());
}

void launch_laya_attn(const float *qkv, int d, int hd, int window, const int32_t *tile_row0, const int32_t *tile_pos0,
                      const int32_t *tile_n, const int32_t *tile_seq, const int32_t *seq_n, const int32_t *grp_first,
                      const int32_t *grp_count, int ngroups, _Float16 *y, _Float16 *ylo, hipStream_t st) {
  LG_REQUIRE(hd == kHD, "laya attention: head_dim %d (kernel is built for 64)", hd);
  LG_REQUIRE(ngroups > 0 && d % kHD == 0 && d >= kHD, "laya attention: bad shape");
  const int heads = d / kHD;
  const bool small = int64_t(ngroups) * heads < device_cus();
  const int per_head = small ? 2 * ngroups : ngroups;
  LG_REQUIRE(int64_t(per_head) * heads < (1ll << 31), "laya attention: too many tiles");
  const auto fn = small ? laya_attn_kernel<1> : laya_attn_kernel<2>;
  hipLaunchKernelGGL(fn, dim3(per_head * heads), dim3(256), 0, st, qkv, d, window, ngroups, per_head, grp_first, grp_count,
                     tile_row0, tile_pos0, tile_n, tile_seq, seq_n, y, ylo);
  HIP_CHECK(hipGetLastError());
}

void launch_gelu_inplace(float *x, int64_t n, hipStream_t st) {
  if (n <= 0) return;
  hipLaunchKernelGGL(gelu_inplace_kernel, dim3(unsigned((n + 255) / 256)), dim3(256), 0, st, x, n);
  HIP_CHECK(hipGetLastError());
}

void launch_laya_act_features(const float *h, int d, const int32_t *seq_row0, const int32_t *lg_first,
                              const int32_t *lg_count, const float *logits, int nseq, float *pooled, hipStream_t st) {
  LG_REQUIRE(nseq > 0 && d > 0, "act features: bad shape");
  hipLaunchKernelGGL(laya_act_features_kernel, dim3(nseq), dim3(kT), 0, st, h, d, seq_row0, lg_first, lg_count, logits,
                     pooled);
  HIP_CHECK(hipGetLastError());
}

}  // namespace lg
