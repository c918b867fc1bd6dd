// Small memory-bound kernels of the forward pass: RMSNorm, embedding gather, RoPE fused
// with the paged KV-cache write, the option head and option scores, full-vocab argmax.
#include <hip/hip_runtime.h>

#include <algorithm>

#include <cfloat>
#include <cmath>
#include <type_traits>

#include "common.h"
#include "kernels.h"
#include "quant.h"
#include "f16split.h"
#include "wave.h"

namespace lg {
namespace {

constexpr int kT = 256;

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
  return v;
}

__device__ float block_sum(float v, float *red) {
  v = wave_sum(v);
  const int t = threadIdx.x;
  if ((t & 63) == 0) red[t >> 6] = v;
  __syncthreads();
  float s = 0.0f;
  for (int i = 0; i < int(blockDim.x) / 64; ++i) s += red[i];
  __syncthreads();
  return s;
}

// RMSNorm, src/models/openthai/model.rs:84-94: y = (x * (1/sqrt(dot(x,x)/d + eps))) * w.
template <typename Out>
__global__ __launch_bounds__(kT) void rmsnorm_kernel(const float *__restrict__ x, int d,
                                                     const float *__restrict__ w, float eps,
                                                     Out *__restrict__ y, Out *__restrict__ ylo) {
  __shared__ float red[kT / 64];
  const float *row = x + int64_t(blockIdx.x) * d;
  float ss = 0.0f;
  for (int k = threadIdx.x; k < d; k += kT) ss += row[k] * row[k];
  const float inv = 1.0f / sqrtf(block_sum(ss, red) / float(d) + eps);
  Out *out = y + int64_t(blockIdx.x) * d;
  Out *lo = ylo ? ylo + int64_t(blockIdx.x) * d : nullptr;
  for (int k = threadIdx.x; k < d; k += kT) {
    const float v = f32_pin(row[k] * inv * w[k]);
    const Out h = Out(v);
    out[k] = h;
    if (lo) lo[k] = Out(v - float(h));
  }
}

// The same into f16 (+ lo plane) for d % 4 == 0, d <= 1024 NI: the row and the weights are loaded together, as float4 at
// clamped indices (no load waits for the sum of squares or for another), and kept in registers; one barrier.  Latency-bound for
// a request's rows (weights after the sum, a shuffle reduction and two barriers: 3.3 us against 2.8 for 144 rows of 512),
// HBM-bound for a batch's (34,560 rows of 2048: 91.3 -> 89.2 us).
template <int NI>
__global__ __launch_bounds__(kT) void rmsnorm_f16_vec_kernel(const float *__restrict__ x, int d,
                                                             const float *__restrict__ w, float eps,
                                                             _Float16 *__restrict__ y, _Float16 *__restrict__ ylo) {
  typedef _Float16 half4 __attribute__((ext_vector_type(4)));
  __shared__ float red[kT / 64];
  const float4 *row = reinterpret_cast<const float4 *>(x + int64_t(blockIdx.x) * d);
  const float4 *w4 = reinterpret_cast<const float4 *>(w);
  const int n4 = d >> 2;
  float4 v[NI], ww[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) v[i] = row[min(int(threadIdx.x) + i * kT, n4 - 1)];
#pragma unroll
  for (int i = 0; i < NI; ++i) ww[i] = w4[min(int(threadIdx.x) + i * kT, n4 - 1)];
  float ss = 0.0f;
#pragma unroll
  for (int i = 0; i < NI; ++i)
    if (int(threadIdx.x) + i * kT < n4) {
      ss += v[i].x * v[i].x;
      ss += v[i].y * v[i].y;
      ss += v[i].z * v[i].z;
      ss += v[i].w * v[i].w;
    }
  // block_sum's order: an f16 KV cache turns a last-bit change of the norm into whole f16 steps
  ss = wave_sum_butterfly(ss);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
  __syncthreads();
  const float inv = 1.0f / sqrtf((((red[0] + red[1]) + red[2]) + red[3]) / float(d) + eps);
  half4 *out = reinterpret_cast<half4 *>(y + int64_t(blockIdx.x) * d);
  half4 *lo = ylo ? reinterpret_cast<half4 *>(ylo + int64_t(blockIdx.x) * d) : nullptr;
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int k = threadIdx.x + i * kT;
    if (k >= n4) continue;
    const float r[4] = {v[i].x * inv * ww[i].x, v[i].y * inv * ww[i].y, v[i].z * inv * ww[i].z, v[i].w * inv * ww[i].w};
    half4 h, l;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      _Float16 a, b;
      split_f16(r[e], a, b);
      h[e] = a;
      l[e] = b;
    }
    out[k] = h;
    if (lo) lo[k] = l;
  }
}

// Eight values a thread where rows and addresses allow 16-byte accesses (34,560 rows of 2048: 225 us one value a thread,
// 84 here).
__global__ __launch_bounds__(kT) void embed_vec_kernel(const void *__restrict__ table, uint32_t kind,
                                                       const int32_t *__restrict__ ids, int T, int d, int vocab,
                                                       float *__restrict__ x) {
  const int64_t e = int64_t(blockIdx.x) * kT + threadIdx.x;
  const int n8 = d >> 3;
  if (e >= int64_t(T) * n8) return;
  const int t = int(e / n8), k = int(e % n8) * 8;
  const int64_t src = int64_t(min(max(ids[t], 0), vocab - 1)) * d + k;  // ids are validated on the host
  float4 o[2];
  if (kind == LG_F16) {
    const uint4 q = *reinterpret_cast<const uint4 *>(static_cast<const uint16_t *>(table) + src);
    o[0] = make_float4(half_bits(q.x & 0xffffu), half_bits(q.x >> 16), half_bits(q.y & 0xffffu), half_bits(q.y >> 16));
    o[1] = make_float4(half_bits(q.z & 0xffffu), half_bits(q.z >> 16), half_bits(q.w & 0xffffu), half_bits(q.w >> 16));
  } else {
    o[0] = reinterpret_cast<const float4 *>(static_cast<const float *>(table) + src)[0];
    o[1] = reinterpret_cast<const float4 *>(static_cast<const float *>(table) + src)[1];
  }
  float4 *dst = reinterpret_cast<float4 *>(x + int64_t(t) * d + k);
  dst[0] = o[0];
  dst[1] = o[1];
}

__global__ void embed_kernel(const void *__restrict__ table, uint32_t kind, const int32_t *__restrict__ ids,
                             int T, int d, int vocab, float *__restrict__ x) {
  const int64_t e = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (e >= int64_t(T) * d) return;
  const int t = int(e / d), k = int(e % d);
  const int id = min(max(ids[t], 0), vocab - 1);  // ids are validated on the host
  const int64_t src = int64_t(id) * d + k;
  x[e] = kind == LG_F16 ? half_bits(static_cast<const uint16_t *>(table)[src])
                        : static_cast<const float *>(table)[src];
}

// One KV value into a pool: offset r inside the (page, kv head) block that starts at value
// `block` (page * page_stride + head * plane).  Split pools hold the block as an f16 hi plane
// and then an f16 lo plane of `plane` values each; f16 pools as one plane.
// RoPE everywhere is the rotate-half form with the model's tables (src/tensor.rs:158-172).
template <bool SPLIT>
__device__ __forceinline__ void kv_put(void *pool, int64_t block, int r, int plane, float v) {
  _Float16 *p = static_cast<_Float16 *>(pool);
  if constexpr (SPLIT) {
    _Float16 hi, lo;
    split_f16(v, hi, lo);
    p[2 * block + r] = hi;
    p[2 * block + plane + r] = lo;
  } else {
    p[block + r] = _Float16(v);
  }
}

// Decode form: one token whose position and KV page the host already knows (kernel arguments,
// so the only memory round trip is the q|k|v row and the table rows).  q goes out in f32.
// Prefill form: one workgroup per (attention tile of <= 32 consecutive tokens of one sequence,
// part: first or second half of the q heads, the k heads, the v heads).  q and k rotations are
// flat (token, quad of pairs) items dealt to the threads in rounds whose loads are all issued
// before any is used; v is staged through LDS a few kv heads at a time so that its transposed
// page layout is written as runs of consecutive slots instead of one 4-byte store per cache line.
template <bool SPLIT, int HD>
__global__ __launch_bounds__(kT) void rope_kv_tile_kernel(
    const float *__restrict__ qkv, int hq, KvGeom g, const float *__restrict__ cosT,
    const float *__restrict__ sinT, const int32_t *__restrict__ pages, int max_pages,
    const int32_t *__restrict__ tile_seq, const int32_t *__restrict__ tile_row0,
    const int32_t *__restrict__ tile_pos0, const int32_t *__restrict__ tile_n,
    _Float16 *__restrict__ q16, _Float16 *__restrict__ q16lo, void *__restrict__ kpool,
    void *__restrict__ vpool, float qscale) {
  constexpr int TT = 32, HALF = HD / 2;        // tokens per tile, pair offset
  constexpr int HB = HD == 64 ? 4 : 2;         // V heads per LDS round (32 values per thread)
  constexpr int RI = 4;                        // rotation items whose loads one round issues together
  constexpr int TPR = kT / HD, VT = TT / TPR;  // V: token lanes per dim, tokens per thread
  static_assert(kT % HALF == 0 && kT % HD == 0, "thread blocks must tile the head");
  __shared__ float vs[HB][TT][HD + 1];
  const int tile = blockIdx.x, tid = threadIdx.x;
  const int row0 = tile_row0[tile], pos0 = tile_pos0[tile], n = tile_n[tile];
  const int32_t *ptab = pages + int64_t(tile_seq[tile]) * max_pages;
  // a tile of <= 32 tokens spans at most two pages (page_tokens >= 32): look both up once
  const int pg0 = pos0 / g.page_tokens;
  const int64_t page_lo = ptab[pg0], page_hi = ptab[(pos0 + n - 1) / g.page_tokens];
  auto page_base = [&](int pos) { return (pos / g.page_tokens == pg0 ? page_lo : page_hi) * g.page_stride; };
  const int plane = g.page_tokens * HD;  // values per plane of one (page, kv head) block
  const int qw = hq * HD, kvw = g.hkv * HD, rw = qw + 2 * kvw;
  // rotations: flat items (token, quad of four consecutive pairs j..j+3 of a q|k head), quads
  // fastest so that neighbouring threads read neighbouring 16 bytes of a row and of the tables;
  // RI items per thread per round with every load issued before any value is used (one memory
  // round trip per round: a 32-token tile of the d512 model's q heads is one round); float4
  // loads, 8-byte stores of four f16
  constexpr int QPH = HALF / 4;  // quads per head
  // the tile's work is split over four workgroups (blockIdx.y): the first and second half of the q
  // heads, the k heads, the v heads
  const int part = blockIdx.y;
  const int h_lo = part == 0 ? 0 : part == 1 ? hq / 2 : hq, h_hi = part == 0 ? hq / 2 : part == 1 ? hq : hq + g.hkv;
  const int nquads = part < 3 ? (h_hi - h_lo) * QPH : 0;
  const int items = n * nquads;
  typedef _Float16 half4 __attribute__((ext_vector_type(4)));
  for (int i0 = 0; i0 < items; i0 += RI * kT) {
    float4 u[RI], v[RI], c0[RI], c1[RI], s0[RI], s1[RI];
#pragma unroll
    for (int b = 0; b < RI; ++b) {
      const int it = min(i0 + b * kT + tid, items - 1);  // past the end: a valid item, not stored
      const int tk = it / nquads, p = it % nquads;
      const int hh = h_lo + p / QPH, j = (p % QPH) * 4;
      const float *row = qkv + int64_t(row0 + tk) * rw + hh * HD;
      const int64_t cb = int64_t(pos0 + tk) * HD;
      u[b] = *reinterpret_cast<const float4 *>(row + j);
      v[b] = *reinterpret_cast<const float4 *>(row + j + HALF);
      c0[b] = *reinterpret_cast<const float4 *>(cosT + cb + j);
      c1[b] = *reinterpret_cast<const float4 *>(cosT + cb + j + HALF);
      s0[b] = *reinterpret_cast<const float4 *>(sinT + cb + j);
      s1[b] = *reinterpret_cast<const float4 *>(sinT + cb + j + HALF);
    }
#pragma unroll
    for (int b = 0; b < RI; ++b) {
      const int it = i0 + b * kT + tid;
      if (it >= items) continue;
      const int tk = it / nquads, p = it % nquads;
      const int hh = h_lo + p / QPH, j = (p % QPH) * 4;
      const float uu[4] = {u[b].x, u[b].y, u[b].z, u[b].w}, vv[4] = {v[b].x, v[b].y, v[b].z, v[b].w};
      const float cc0[4] = {c0[b].x, c0[b].y, c0[b].z, c0[b].w}, cc1[4] = {c1[b].x, c1[b].y, c1[b].z, c1[b].w};
      const float ss0[4] = {s0[b].x, s0[b].y, s0[b].z, s0[b].w}, ss1[4] = {s1[b].x, s1[b].y, s1[b].z, s1[b].w};
      float a[4], c[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) rope_pair(uu[e], vv[e], cc0[e], ss0[e], cc1[e], ss1[e], a[e], c[e]);
      if (hh < hq) {
        const int64_t at = int64_t(row0 + tk) * qw + hh * HD + j;
        half4 ah, al, ch, cl;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          _Float16 x, y;
          split_f16(a[e] * qscale, x, y);
          ah[e] = x;
          al[e] = y;
          split_f16(c[e] * qscale, x, y);
          ch[e] = x;
          cl[e] = y;
        }
        *reinterpret_cast<half4 *>(q16 + at) = ah;
        *reinterpret_cast<half4 *>(q16 + at + HALF) = ch;
        if (q16lo) {
          *reinterpret_cast<half4 *>(q16lo + at) = al;
          *reinterpret_cast<half4 *>(q16lo + at + HALF) = cl;
        }
      } else {
        const int pos = pos0 + tk;
        const int64_t blk = page_base(pos) + int64_t(hh - hq) * plane;
        const int r = (pos % g.page_tokens) * HD + j;
        _Float16 *kp = static_cast<_Float16 *>(kpool);
        half4 ah, al, ch, cl;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if constexpr (SPLIT) {
            _Float16 x, y;
            split_f16(a[e], x, y);
            ah[e] = x;
            al[e] = y;
            split_f16(c[e], x, y);
            ch[e] = x;
            cl[e] = y;
          } else {
            ah[e] = _Float16(a[e]);
            ch[e] = _Float16(c[e]);
          }
        }
        if constexpr (SPLIT) {
          *reinterpret_cast<half4 *>(kp + 2 * blk + r) = ah;
          *reinterpret_cast<half4 *>(kp + 2 * blk + r + HALF) = ch;
          *reinterpret_cast<half4 *>(kp + 2 * blk + plane + r) = al;
          *reinterpret_cast<half4 *>(kp + 2 * blk + plane + r + HALF) = cl;
        } else {
          *reinterpret_cast<half4 *>(kp + blk + r) = ah;
          *reinterpret_cast<half4 *>(kp + blk + r + HALF) = ch;
        }
      }
    }
  }
  if (part != 3) return;
  // v: HB kv heads per round staged through LDS (thread -> dim tid % HD, tokens tid / HD + TPR i),
  // then written as runs of consecutive slots; the next round's loads are issued before this
  // round's stores, so one memory round trip overlaps the stores of the round before
  const int dd = tid % HD, tq = tid / HD;
  float val[HB][VT];
  auto load_v = [&](int h0) {
#pragma unroll
    for (int hh = 0; hh < HB; ++hh)
#pragma unroll
      for (int i = 0; i < VT; ++i) {
        const int tk = min(tq + TPR * i, n - 1), h = min(h0 + hh, g.hkv - 1);
        val[hh][i] = qkv[int64_t(row0 + tk) * rw + qw + kvw + h * HD + dd];
      }
  };
  load_v(0);
  for (int h0 = 0; h0 < g.hkv; h0 += HB) {
    const int nh = min(HB, g.hkv - h0);
#pragma unroll
    for (int hh = 0; hh < HB; ++hh)
#pragma unroll
      for (int i = 0; i < VT; ++i) vs[hh][tq + TPR * i][dd] = val[hh][i];
    __syncthreads();
    if (h0 + HB < g.hkv) load_v(h0 + HB);
    // thread -> (head, dim, four tokens) with the tokens fastest: runs of consecutive slots per dim row,
    // four slots (one 8-byte store per plane) when the quad is whole and 4-aligned in its page
    for (int i = tid; i < nh * (TT / 4) * HD; i += kT) {
      const int hh = i / ((TT / 4) * HD), r = i % ((TT / 4) * HD), tk0 = (r % (TT / 4)) * 4, d2 = r / (TT / 4);
      if (tk0 >= n) continue;
      if ((pos0 & 3) == 0 && tk0 + 3 < n) {
        const int pos = pos0 + tk0;
        const int64_t blk = page_base(pos) + int64_t(h0 + hh) * plane;
        const int idx = d2 * g.page_tokens + pos % g.page_tokens;
        _Float16 *vp = static_cast<_Float16 *>(vpool);
        half4 vh, vl;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if constexpr (SPLIT) {
            _Float16 x, y;
            split_f16(vs[hh][tk0 + e][d2], x, y);
            vh[e] = x;
            vl[e] = y;
          } else {
            vh[e] = _Float16(vs[hh][tk0 + e][d2]);
          }
        }
        if constexpr (SPLIT) {
          *reinterpret_cast<half4 *>(vp + 2 * blk + idx) = vh;
          *reinterpret_cast<half4 *>(vp + 2 * blk + plane + idx) = vl;
        } else {
          *reinterpret_cast<half4 *>(vp + blk + idx) = vh;
        }
      } else {
        for (int tk = tk0; tk < min(tk0 + 4, n); ++tk) {
          const int pos = pos0 + tk;
          kv_put<SPLIT>(vpool, page_base(pos) + int64_t(h0 + hh) * plane, d2 * g.page_tokens + pos % g.page_tokens,
                        plane, vs[hh][tk][d2]);
        }
      }
    }
    __syncthreads();
  }
}

// Eight consecutive weights (k a multiple of 8) of row n of the option head, loaded raw.
template <uint32_t KIND>
struct HeadChunk {
  uint4 q, q2;
  float a, b;
  int shift;
  __device__ __forceinline__ void load(const DevMatrix &W, int64_t n, int k) {
    const int64_t cols = W.cols;
    if constexpr (KIND == LG_F32) {
      const uint4 *p = reinterpret_cast<const uint4 *>(static_cast<const float *>(W.q) + n * cols + k);
      q = p[0];
      q2 = p[1];
    } else if constexpr (KIND == LG_F16) {
      q = *reinterpret_cast<const uint4 *>(static_cast<const uint16_t *>(W.q) + n * cols + k);
    } else {
      const uint8_t *p = static_cast<const uint8_t *>(W.q);
      p += KIND == LG_Q4_K ? n * (cols / 2) + (k / 64) * 32 + (k % 32) : n * cols + k;
      const uint2 v = *reinterpret_cast<const uint2 *>(p);
      q.x = v.x;
      q.y = v.y;
      if constexpr (KIND == LG_Q8_0) {
        a = float(static_cast<const _Float16 *>(W.s)[n * (cols / 32) + k / 32]);
      } else if constexpr (KIND == LG_Q4_K) {
        const float2 ab = static_cast<const float2 *>(W.s)[n * (cols / 32) + k / 32];
        a = ab.x;
        b = ab.y;
        shift = (k % 64) >= 32 ? 4 : 0;
      } else {
        a = static_cast<const float *>(W.s)[n * (cols / 16) + k / 16];
      }
    }
  }
  __device__ __forceinline__ float value(int j) const {
    const uint32_t w[8] = {q.x, q.y, q.z, q.w, q2.x, q2.y, q2.z, q2.w};
    if constexpr (KIND == LG_F32) return __uint_as_float(w[j]);
    if constexpr (KIND == LG_F16) return float(__builtin_bit_cast(_Float16, uint16_t(w[j / 2] >> (16 * (j % 2)))));
    const uint32_t byte = w[j / 4] >> (8 * (j % 4));
    if constexpr (KIND == LG_Q4_K) return kq4_weight(a, (byte >> shift) & 15u, b);
    return kq6_weight(a, int8_t(byte));
  }
};

// Final RMSNorm and option head: a wave takes RB gathered rows against NO option rows, its lanes eight consecutive
// columns at a time, and needs one pass and no LDS: logit = (sum_k (x_k norm_k) w_k) / sqrt(mean x^2 + eps), both sums
// taken over the same loads.  The order of both is the same for every RB and NO, so a row's logits do not depend on the
// batch around it.  Latency-bound for a few rows (the former form, one element a load after a workgroup-wide norm, took
// 20 us for one row of F16 d 512, 68 for three of Q8_0 d 2048, 93 for three of Q6_K d 3584; this one 3.6, 6.0 and 9.8), L2-bound for many; RB = NO = 4 reads a batch's weights and rows once per four.
template <uint32_t KIND, int RB, int NO>
__global__ __launch_bounds__(kT) void head_rows_kernel(const float *__restrict__ x, const int32_t *__restrict__ rows,
                                                       int R, int d, const float *__restrict__ norm_w, float eps,
                                                       DevMatrix W, const float *__restrict__ bias,
                                                       const int32_t *__restrict__ ids, int nv,
                                                       float *__restrict__ logits) {
  const int lane = threadIdx.x & 63, r0 = blockIdx.x * RB;
  const int j0 = (blockIdx.y * (kT / 64) + (threadIdx.x >> 6)) * NO;
  if (j0 >= nv) return;
  constexpr int U = RB == 1 ? 8 : 1;  // chunks loaded together
  int64_t n[NO];
  const float *row[RB];
#pragma unroll
  for (int o = 0; o < NO; ++o) n[o] = ids[min(j0 + o, nv - 1)];
#pragma unroll
  for (int r = 0; r < RB; ++r) row[r] = x + int64_t(rows[min(r0 + r, R - 1)]) * d;
  float ss[RB], s[RB][NO];
#pragma unroll
  for (int r = 0; r < RB; ++r) {
    ss[r] = 0.0f;
#pragma unroll
    for (int o = 0; o < NO; ++o) s[r][o] = 0.0f;
  }
  for (int k0 = lane * 8; k0 < d; k0 += 512 * U) {
    HeadChunk<KIND> w[U][NO];
    float4 nw[U][2], xv[U][RB][2];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = min(k0 + 512 * u, d - 8);
#pragma unroll
      for (int o = 0; o < NO; ++o) w[u][o].load(W, n[o], k);
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        nw[u][e] = *reinterpret_cast<const float4 *>(norm_w + k + 4 * e);
#pragma unroll
        for (int r = 0; r < RB; ++r) xv[u][r][e] = *reinterpret_cast<const float4 *>(row[r] + k + 4 * e);
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (k0 + 512 * u >= d) break;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float nj = reinterpret_cast<const float *>(&nw[u][j / 4])[j % 4];
#pragma unroll
        for (int r = 0; r < RB; ++r) {
          const float xj = reinterpret_cast<const float *>(&xv[u][r][j / 4])[j % 4];
          ss[r] = fmaf(xj, xj, ss[r]);
#pragma unroll
          for (int o = 0; o < NO; ++o) s[r][o] = fmaf(xj * nj, w[u][o].value(j), s[r][o]);
        }
      }
    }
  }
#pragma unroll
  for (int r = 0; r < RB; ++r) {
    const float inv = 1.0f / sqrtf(wave_sum_dpp(ss[r]) / float(d) + eps);
#pragma unroll
    for (int o = 0; o < NO; ++o) {
      float v = wave_sum_dpp(s[r][o]) * inv;
      if (bias) v = f32_pin(v) + bias[n[o]];
      if (lane == 0 && r0 + r < R && j0 + o < nv) logits[int64_t(r0 + r) * nv + j0 + o] = v;
    }
  }
}

template <int RB, int NO>
void launch_head_kind(const float *x, const int32_t *rows, int R, int d, const float *norm_w, float eps,
                      const DevMatrix &W, const float *bias, const int32_t *vocab_ids, int nv, float *logits, hipStream_t st) {
  const dim3 grid((R + RB - 1) / RB, (nv + NO * kT / 64 - 1) / (NO * kT / 64));
#define HEAD(K)                                                                                                       \
  case K:                                                                                                             \
    hipLaunchKernelGGL((head_rows_kernel<K, RB, NO>), grid, dim3(kT), 0, st, x, rows, R, d, norm_w, eps, W, bias,     \
                       vocab_ids, nv, logits);                                                                        \
    break;
  switch (W.kind) {
    HEAD(LG_F32) HEAD(LG_F16) HEAD(LG_Q8_0) HEAD(LG_Q4_K) HEAD(LG_Q6_K)
    default: fail(LG_ERR_UNSUPPORTED, "head: GGML type %u", W.kind);
  }
#undef HEAD
}

// Option scores for one answer position per thread (src/models/openthai/decision.rs:268-279,
// 297-303): z = l / T; p = softmax(z); p /= max(sum p, 1e-12); final renormalisation; and the
// option log-softmax z - max - log(sum exp(z - max)).
__global__ void option_scores_kernel(const float *__restrict__ logits, int R, int k, float temp,
                                     float *__restrict__ probs, float *__restrict__ logprobs) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= R) return;
  const float *l = logits + int64_t(r) * k;
  float z[32], p[32];
  float m = -INFINITY;
  for (int i = 0; i < k; ++i) {
    z[i] = l[i] / temp;
    m = fmaxf(m, z[i]);
  }
  float s = 0.0f;
  for (int i = 0; i < k; ++i) {
    p[i] = expf(z[i] - m);
    s += p[i];
  }
  const float lse = logf(s);
  float sum = 0.0f;
  for (int i = 0; i < k; ++i) {
    p[i] = p[i] / s;
    sum += p[i];
  }
  sum = fmaxf(sum, 1e-12f);
  float s2 = 0.0f;
  for (int i = 0; i < k; ++i) {
    p[i] = p[i] / sum;
    s2 += p[i];
  }
  s2 = fmaxf(s2, 1e-12f);
  for (int i = 0; i < k; ++i) {
    if (probs) probs[int64_t(r) * k + i] = p[i] / s2;
    if (logprobs) logprobs[int64_t(r) * k + i] = z[i] - m - lse;
  }
}

// Argmax: ties and NaN follow the strict ">" scan (first maximum wins).
// Each thread scans increasing indices with a strict ">", so it keeps its first maximum;
// NaN never compares greater.  Merges prefer the larger value, then the smaller index.
__device__ __forceinline__ void better(float &bv, int &bi, float v, int i) {
  if (v > bv) {
    bv = v;
    bi = i;
  }
}

// Two launches for long vectors (a single workgroup reads the 608 KB of a 152,064-entry vocabulary in 15.2 us, limited by what
// one CU can load; the two together take 9.4): kArgParts workgroups each take a range, the last one merges.  At 32,000
// entries the single launch below is ahead (5.7 us against 8.4).
constexpr int kArgParts = 64;
__global__ __launch_bounds__(kT) void argmax_part_kernel(const float *__restrict__ v, int n, float *__restrict__ part_v,
                                                         int32_t *__restrict__ part_i) {
  __shared__ float sv[kT / 64];
  __shared__ int si[kT / 64];
  const int per = ((n + kArgParts - 1) / kArgParts + 3) & ~3, lo = min(int(blockIdx.x) * per, n), hi = min(lo + per, n);
  const int t = threadIdx.x, lane = t & 63;
  float bv = -INFINITY;
  int bi = -1;
  constexpr int U = 4;
  for (int k0 = lo + 4 * t; k0 < hi; k0 += 4 * kT * U) {
    float w[U][4];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e) w[u][e] = v[min(k0 + 4 * kT * u + e, n - 1)];  // all loads before any compare
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (k0 + 4 * kT * u + e < hi) better(bv, bi, w[u][e], k0 + 4 * kT * u + e);
  }
  auto merge = [&](float ov, int oi) {
    if (oi >= 0 && (bi < 0 || ov > bv || (ov == bv && oi < bi))) {
      bv = ov;
      bi = oi;
    }
  };
#pragma unroll
  for (int m = 1; m < 64; m <<= 1) merge(__shfl_xor(bv, m), __shfl_xor(bi, m));
  if (lane == 0) {
    sv[t >> 6] = bv;
    si[t >> 6] = bi;
  }
  __syncthreads();
  if (t == 0) {
#pragma unroll
    for (int w = 1; w < kT / 64; ++w) merge(sv[w], si[w]);
    part_v[blockIdx.x] = bv;
    part_i[blockIdx.x] = bi;
  }
}

// The token's embedding row (ids clamped as embed_kernel clamps them) to x, four loads of a thread in flight.
template <int THREADS>
__device__ __forceinline__ void token_row(int tok, int n, const void *__restrict__ table, uint32_t kind, int d,
                                          float *__restrict__ x) {
  const int64_t row = int64_t(min(max(tok, 0), n - 1)) * d;
  for (int k0 = threadIdx.x; k0 < d; k0 += 4 * THREADS) {
    float w[4];
    if (kind == LG_F16) {
      uint16_t b[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) b[u] = static_cast<const uint16_t *>(table)[row + min(k0 + u * THREADS, d - 1)];
#pragma unroll
      for (int u = 0; u < 4; ++u) w[u] = half_bits(b[u]);
    } else {
#pragma unroll
      for (int u = 0; u < 4; ++u) w[u] = static_cast<const float *>(table)[row + min(k0 + u * THREADS, d - 1)];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (k0 + u * THREADS < d) x[k0 + u * THREADS] = w[u];
  }
}

// Merges the parts; with x, also writes the token's embedding row, as argmax_one<true>.
__global__ __launch_bounds__(1024) void argmax_merge_kernel(const float *__restrict__ part_v, const int32_t *__restrict__ part_i,
                                                          int n, int32_t *__restrict__ out, const void *__restrict__ table,
                                                          uint32_t kind, int d, float *__restrict__ x) {
  static_assert(kArgParts == 64, "one part a lane");
  const int t = threadIdx.x, lane = t & 63;
  float bv = part_v[lane];
  int bi = part_i[lane];
#pragma unroll
  for (int m = 1; m < 64; m <<= 1) {  // every wave merges for itself
    const float ov = __shfl_xor(bv, m);
    const int oi = __shfl_xor(bi, m);
    if (oi >= 0 && (bi < 0 || ov > bv || (ov == bv && oi < bi))) {
      bv = ov;
      bi = oi;
    }
  }
  const int tok = bi >= 0 && bv > -INFINITY && bv < INFINITY ? bi : -1;  // -1: no finite maximum
  if (t == 0) out[0] = tok;
  if (x) token_row<1024>(tok, n, table, kind, d, x);
}

// from this length two launches
constexpr int kArgLong = 65536;

// One workgroup of 1024 threads over the whole vector (one launch: a decode step's argmax sits between
// two dependent launches).  Thread t takes float4 words t, t + 1024, ... (their elements in index
// order, so the strict `better` keeps the first of equal values), then the merge rule of the two-stage
// form over the wave (butterfly) and over the 16 waves.  The rule is a total order (larger value,
// then smaller index; no index loses), so the merge order does not change the result.
// EMB: the workgroup then writes the token's embedding row (ids clamped as embed_kernel clamps
// them) to x, the next decode step's input, which saves that step its embedding launch.
template <bool EMB>
__global__ __launch_bounds__(1024) void argmax_one(const float *__restrict__ v, int n, int32_t *__restrict__ out,
                                                   const void *__restrict__ table, uint32_t kind, int d,
                                                   float *__restrict__ x) {
  __shared__ float sv[16];
  __shared__ int si[16];
  __shared__ int stok;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  float bv = -INFINITY;
  int bi = -1;
  const int n4 = (reinterpret_cast<uintptr_t>(v) & 15) == 0 ? n >> 2 : 0;
  const float4 *v4 = reinterpret_cast<const float4 *>(v);
  for (int k0 = t; k0 < n4; k0 += 8 * 1024) {
    float4 w[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) w[u] = v4[min(k0 + u * 1024, n4 - 1)];  // all loads before any compare
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int k = k0 + u * 1024;
      if (k < n4) {
        better(bv, bi, w[u].x, 4 * k);
        better(bv, bi, w[u].y, 4 * k + 1);
        better(bv, bi, w[u].z, 4 * k + 2);
        better(bv, bi, w[u].w, 4 * k + 3);
      }
    }
  }
  for (int i = 4 * n4 + t; i < n; i += 1024) better(bv, bi, v[i], i);  // the tail (or all, unaligned)
  auto merge = [&](float ov, int oi) {
    if (oi >= 0 && (bi < 0 || ov > bv || (ov == bv && oi < bi))) {
      bv = ov;
      bi = oi;
    }
  };
#pragma unroll
  for (int m = 1; m < 64; m <<= 1) merge(__shfl_xor(bv, m), __shfl_xor(bi, m));
  if (lane == 0) {
    sv[wave] = bv;
    si[wave] = bi;
  }
  __syncthreads();
  if (wave == 0) {
    bv = lane < 16 ? sv[lane] : -INFINITY;
    bi = lane < 16 ? si[lane] : -1;
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) merge(__shfl_xor(bv, m), __shfl_xor(bi, m));
    if (lane == 0) {
      const int tok = bi >= 0 && bv > -INFINITY && bv < INFINITY ? bi : -1;  // -1: no finite maximum
      out[0] = tok;
      stok = tok;
    }
  }
  if constexpr (EMB) {
    __syncthreads();
    token_row<1024>(stok, n, table, kind, d, x);
  }
}

__global__ void cvt_f16_kernel(const float *__restrict__ x, int64_t n, _Float16 *__restrict__ y,
                               _Float16 *__restrict__ ylo) {
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  _Float16 h, l;
  split_f16(x[i], h, l);
  y[i] = h;
  if (ylo) ylo[i] = l;
}

__global__ void fill_i32_kernel(int32_t *p, int n, int32_t v) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

}  // namespace

void launch_rmsnorm_f16(const float *x, int rows, int d, const float *w, float eps, _Float16 *y,
                        _Float16 *y_lo, hipStream_t st) {
  LG_REQUIRE(rows > 0 && d > 0, "rmsnorm: empty");
  const auto vec = [&](auto ni) {
    hipLaunchKernelGGL(rmsnorm_f16_vec_kernel<decltype(ni)::value>, dim3(rows), dim3(kT), 0, st, x, d, w, eps, y, y_lo);
  };
  if (d % 4 == 0 && d <= 4 * kT) vec(std::integral_constant<int, 1>{});
  else if (d % 4 == 0 && d <= 8 * kT) vec(std::integral_constant<int, 2>{});
  else if (d % 4 == 0 && d <= 16 * kT) vec(std::integral_constant<int, 4>{});
  else
    hipLaunchKernelGGL(rmsnorm_kernel<_Float16>, dim3(rows), dim3(kT), 0, st, x, d, w, eps, y, y_lo);
  HIP_CHECK(hipGetLastError());
}

void launch_rmsnorm_f32(const float *x, int rows, int d, const float *w, float eps, float *y,
                        hipStream_t st) {
  LG_REQUIRE(rows > 0 && d > 0, "rmsnorm: empty");
  hipLaunchKernelGGL(rmsnorm_kernel<float>, dim3(rows), dim3(kT), 0, st, x, d, w, eps, y,
                     static_cast<float *>(nullptr));
  HIP_CHECK(hipGetLastError());
}

void launch_embed(const void *table, uint32_t kind, const int32_t *ids, int T, int d, int vocab,
                  float *x, hipStream_t st) {
  LG_REQUIRE(kind == LG_F16 || kind == LG_F32, "embed: table must be F16/F32");
  const int64_t n = int64_t(T) * d;
  LG_REQUIRE(n > 0 && n / kT < (1ll << 31), "embed: bad size");
  if (d % 8 == 0 && (reinterpret_cast<uintptr_t>(table) & 15) == 0 && (reinterpret_cast<uintptr_t>(x) & 15) == 0)
    hipLaunchKernelGGL(embed_vec_kernel, dim3(unsigned((n / 8 + kT - 1) / kT)), dim3(kT), 0, st, table, kind, ids, T, d,
                       vocab, x);
  else
    hipLaunchKernelGGL(embed_kernel, dim3(unsigned((n + kT - 1) / kT)), dim3(kT), 0, st, table, kind, ids,
                       T, d, vocab, x);
  HIP_CHECK(hipGetLastError());
}

void launch_rope_kv_tiles(const float *qkv, int hq, const KvGeom &g, const float *cosT,
                          const float *sinT, const int32_t *pages, int max_pages,
                          const int32_t *tile_seq, const int32_t *tile_row0, const int32_t *tile_pos0,
                          const int32_t *tile_n, int ntiles, _Float16 *q16, _Float16 *q16_lo,
                          void *kpool, void *vpool, hipStream_t st) {
  LG_REQUIRE(ntiles > 0 && q16, "rope_kv: bad arguments");
  LG_REQUIRE(g.page_tokens >= 32, "rope_kv: a 32-token tile must span at most two pages");
  // the attention consumes base-2 logits: fold log2(e) / sqrt(hd) into q once here
  const float qscale = attn_q_scale(g.hd);
#define LAUNCH(K32, HDV)                                                                                  \
  hipLaunchKernelGGL((rope_kv_tile_kernel<K32, HDV>), dim3(ntiles, 4), dim3(kT), 0, st, qkv, hq, g, cosT, sinT, \
                     pages, max_pages, tile_seq, tile_row0, tile_pos0, tile_n, q16, q16_lo, kpool, vpool, qscale)
  if (g.hd == 128) {
    if (g.split) LAUNCH(true, 128); else LAUNCH(false, 128);
  } else if (g.hd == 64) {
    if (g.split) LAUNCH(true, 64); else LAUNCH(false, 64);
  } else {
    fail(LG_ERR_UNSUPPORTED, "rope_kv: head_dim %d not supported (64, 128)", g.hd);
  }
#undef LAUNCH
  HIP_CHECK(hipGetLastError());
}

void launch_head_rows(const float *x, const int32_t *rows, int R, int d, const float *norm_w,
                      float eps, const DevMatrix &W, const float *bias, const int32_t *vocab_ids, int nv,
                      float *logits, hipStream_t st) {
  LG_REQUIRE(R > 0 && nv > 0 && W.cols == d, "head: bad shape");
  LG_REQUIRE(d % 8 == 0, "head: d=%d is not a multiple of 8", d);
  LG_REQUIRE(d <= 16384, "head: d=%d is past the widths that forwards take", d);
  // a few rows: one row and one option a wave, every load of the row in flight; from 16 rows blocks of four by four
  if (R < 16) launch_head_kind<1, 1>(x, rows, R, d, norm_w, eps, W, bias, vocab_ids, nv, logits, st);
  else launch_head_kind<4, 4>(x, rows, R, d, norm_w, eps, W, bias, vocab_ids, nv, logits, st);
  HIP_CHECK(hipGetLastError());
}

void launch_option_scores(const float *logits, int R, int k, float temperature, float *probs,
                          float *logprobs, hipStream_t st) {
  LG_REQUIRE(R > 0 && k > 0 && k <= 32, "option scores: need 1..32 options");
  hipLaunchKernelGGL(option_scores_kernel, dim3((R + 63) / 64), dim3(64), 0, st, logits, R, k,
                     temperature, probs, logprobs);
  HIP_CHECK(hipGetLastError());
}

static void launch_argmax_long(const float *logits, int V, int32_t *out, float *part_v, int32_t *part_i, const void *table,
                               uint32_t kind, int d, float *x, hipStream_t st) {
  LG_REQUIRE(part_v && part_i, "argmax: missing partials");
  hipLaunchKernelGGL(argmax_part_kernel, dim3(kArgParts), dim3(kT), 0, st, logits, V, part_v, part_i);
  hipLaunchKernelGGL(argmax_merge_kernel, dim3(1), dim3(1024), 0, st, part_v, part_i, V, out, table, kind, d, x);
  HIP_CHECK(hipGetLastError());
}

void launch_argmax(const float *logits, int V, int32_t *out, float *part_v, int32_t *part_i,
                   hipStream_t st) {
  LG_REQUIRE(V > 0, "argmax: empty");
  if (V >= kArgLong) return launch_argmax_long(logits, V, out, part_v, part_i, nullptr, 0, 0, nullptr, st);
  hipLaunchKernelGGL(argmax_one<false>, dim3(1), dim3(1024), 0, st, logits, V, out, static_cast<const void *>(nullptr),
                     0u, 0, static_cast<float *>(nullptr));
  HIP_CHECK(hipGetLastError());
}

void launch_argmax_embed(const float *logits, int V, int32_t *out, const void *table, uint32_t kind, int d, float *x,
                         float *part_v, int32_t *part_i, hipStream_t st) {
  LG_REQUIRE(V > 0 && d > 0 && table && x, "argmax: bad arguments");
  LG_REQUIRE(kind == LG_F16 || kind == LG_F32, "embed: table must be F16/F32");
  if (V >= kArgLong) return launch_argmax_long(logits, V, out, part_v, part_i, table, kind, d, x, st);
  hipLaunchKernelGGL(argmax_one<true>, dim3(1), dim3(1024), 0, st, logits, V, out, table, kind, d, x);
  HIP_CHECK(hipGetLastError());
}

void launch_cvt_f16(const float *x, int64_t n, _Float16 *y, _Float16 *y_lo, hipStream_t st) {
  LG_REQUIRE(n > 0 && n / 256 < (1ll << 31), "cvt_f16: bad size");
  hipLaunchKernelGGL(cvt_f16_kernel, dim3(unsigned((n + 255) / 256)), dim3(256), 0, st, x, n, y, y_lo);
  HIP_CHECK(hipGetLastError());
}

void launch_fill_i32(int32_t *p, int n, int32_t v, hipStream_t st) {
  if (n <= 0) return;
  hipLaunchKernelGGL(fill_i32_kernel, dim3((n + 255) / 256), dim3(256), 0, st, p, n, v);
  HIP_CHECK(hipGetLastError());
}

namespace {
// Plain read of n16 16-byte words for the launch-floor probe: each thread issues its four loads
// before using any, one workgroup covers 16 KiB; the single store is conditional on a value the
// zero-filled buffer never holds, so the kernel writes nothing.
__global__ __launch_bounds__(256) void probe_read_kernel(const uint4 *__restrict__ p, int64_t n16,
                                                         uint32_t *__restrict__ sink) {
  constexpr int PER = 4;
  const int64_t base = int64_t(blockIdx.x) * 256 * PER + threadIdx.x;
  uint4 v[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) v[i] = p[min(base + int64_t(i) * 256, n16 - 1)];
  uint32_t acc = 0;
#pragma unroll
  for (int i = 0; i < PER; ++i) acc ^= v[i].x ^ v[i].y ^ v[i].z ^ v[i].w;
  if (acc == 0x9e3779b9u) sink[blockIdx.x & 255] = acc;
}
}  // namespace

double probe_read_chain(size_t bytes, int launches) {
  LG_REQUIRE(bytes >= 16 && launches > 0 && launches <= 100000, "probe: need >= 16 bytes and 1..100000 launches");
  const int64_t n16 = int64_t(bytes / 16);
  const int64_t blocks = (n16 + 1023) / 1024;
  LG_REQUIRE(blocks < (int64_t(1) << 31), "probe: buffer too large");
  // consecutive launches read distinct slices, about 2 GiB in all (8x the memory-side cache), so the
  // bytes come from HBM as a decode step's distinct weight matrices do
  const size_t stride = (size_t(n16) * 16 + 255) / 256 * 256;
  const int64_t nslice = std::max<int64_t>(1, std::min<int64_t>(launches, int64_t((size_t(2) << 30) / stride) + 1));
  void *buf = nullptr, *sink = nullptr;
  hipStream_t st = nullptr;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  struct Cleanup {
    void *&b, *&s;
    hipStream_t &st;
    hipEvent_t &a, &z;
    ~Cleanup() {
      if (st) (void)hipStreamSynchronize(st);
      if (b) (void)hipFree(b);
      if (s) (void)hipFree(s);
      if (a) (void)hipEventDestroy(a);
      if (z) (void)hipEventDestroy(z);
      if (st) (void)hipStreamDestroy(st);
    }
  } cleanup{buf, sink, st, e0, e1};
  HIP_CHECK(hipMalloc(&buf, stride * size_t(nslice)));
  HIP_CHECK(hipMalloc(&sink, 256 * 4));
  HIP_CHECK(hipStreamCreate(&st));
  HIP_CHECK(hipMemsetAsync(buf, 0, stride * size_t(nslice), st));
  HIP_CHECK(hipEventCreate(&e0));
  HIP_CHECK(hipEventCreate(&e1));
  auto run = [&](int k) {
    for (int i = 0; i < k; ++i) {
      const uint4 *slice = reinterpret_cast<const uint4 *>(static_cast<const uint8_t *>(buf) + stride * size_t(i % nslice));
      hipLaunchKernelGGL(probe_read_kernel, dim3(unsigned(blocks)), dim3(256), 0, st, slice, n16,
                         static_cast<uint32_t *>(sink));
    }
  };
  run(std::min(launches, 20));  // warm-up
  HIP_CHECK(hipEventRecord(e0, st));
  run(launches);
  HIP_CHECK(hipEventRecord(e1, st));
  HIP_CHECK(hipEventSynchronize(e1));
  HIP_CHECK(hipGetLastError());
  float ms = 0.0f;
  HIP_CHECK(hipEventElapsedTime(&ms, e0, e1));
  return double(ms) * 1e3 / launches;
}

}  // namespace lg
