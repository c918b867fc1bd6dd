// Exact GEMM for launches too small for the 256 x 256 tiles of gemm_wide.h (single requests, option passes, narrow
// outputs of batches): C = A . W^T, A as f16 hi/lo planes, W from its prefill copy (DevMatrix::pc, pcl, pcs), the
// modes and the per-element operation order of gemm_wide.h, so every tiling gives the same bits.
//
// What bounds these launches is the time from a load's issue to its use: a workgroup walks K alone, and tiles that
// stage through registers keep one K step in flight (the tiles of gemm_tiles.h: ~2 us a 128-deep step of 64 x 128 at 80
// workgroups).  Here every operand byte moves by LDS-DMA (buffer_load ... lds) with no registers, no conversion, and
// S stages of 64-deep steps: up to S - 1 steps are in flight while one is consumed.  Measured (chained launches): Q8_0 down
// (2048 x 5632) at 301 rows 87 -> 45 us, Q6_K down (3584 x 18944) at 700 rows 768 -> 385 us, F16 512 x 512 at 144 rows 8.0 ->
// 3.8 us.  A step's time then follows the bytes that pass through the LDS (24 KB in, 48 KB out for 64 x 64), not the depth
// of the pipeline: five stages of 64 x 64 take as long as three.
//
// Geometry: 256 threads = 4 waves in a 2 x 2 arrangement, each a (16 HM) x (16 HN) part of a (32 HM) x (32 HN)
// tile, so the epilogues are those of gemm_tiles.h.  A plane's LDS row is 64 halves = 128 bytes = eight 16-byte
// slots, chunk c of row r at slot c ^ (r % 8): eight consecutive lanes of an operand read take the eight 16-byte
// groups of 128 bytes, without bank conflicts.
#pragma once
#include <type_traits>

#include "gemm_tiles.h"
#include "gemm_wide.h"

namespace lg {
namespace mid {

constexpr int BK = 64, ROWB = BK * 2;

template <int NPB, bool SCALED, int HM, int HN>
struct Stage {
  static constexpr int kAP = 32 * HM * ROWB, kBP = 32 * HN * ROWB;
  static constexpr int kALo = kAP, kBHi = 2 * kAP, kBLo = 2 * kAP + kBP, kScl = 2 * kAP + NPB * kBP;
  static constexpr int kBytes = kScl + (SCALED ? 1024 : 0);
  static constexpr int kDma = 2 * HM + NPB * HN + (SCALED ? 1 : 0);  // DMA instructions of a wave per step
};

template <int MODE>
constexpr bool kScaledMode = MODE == wide::WQ8 || MODE == wide::WQ4;

template <int MODE, int HM, int HN, int S>
constexpr int lds_bytes() {
  constexpr int main = S * Stage<MODE == wide::W2 ? 2 : 1, kScaledMode<MODE>, HM, HN>::kBytes;
  constexpr int corr = 2 * Stage<2, false, HM, HN>::kBytes;  // a two-pass Q4_K launch's correction: two stages
  return MODE == wide::WQ4 && corr > main ? corr : main;
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t resource(const void *p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, bytes, kBufferFlags);
}

template <int N>
__device__ __forceinline__ void wait_vm() {
  static_assert(N >= 0 && N < 64, "vmcnt is a 6-bit count");
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// a bare barrier: DMA in flight stays in flight across it, and no instruction is scheduled across it
__device__ __forceinline__ void bare_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

struct Operands {
  __amdgpu_buffer_rsrc_t ah, al, bh, bl, sc;
};

// acc += the K loop over nk steps of 64.  aoff / boff: this lane's byte offsets of DMA instruction q of an A / W
// plane (rows 32 q + 8 wave + lane / 8), soff: of the scale block, sstep its bytes per step.
// Step k: the reads of its second 32-deep chunk issue before the MFMAs of the first; then (barrier) step k + 1 has
// landed and every wave has read all of step k, so the reads of step k + 1's first chunk issue, and the DMA of step k + S
// into step k's stage goes with the MFMAs of the second chunk (ahead of the reads it held them back: Q6_K 3584 x 18944 at
// 700 rows 473 -> 385 us, F16 1024 x 3584 at 1024 rows 24.3 -> 21.9).  No step past the last is fetched; once none is left
// to issue, the wait is for all that is in flight.
template <int NPB, bool SCALED, int HM, int HN, int S>
__device__ __forceinline__ void k_loop(uint8_t *lds, f32x4 (&acc)[HM][HN], const Operands &o, const uint32_t (&aoff)[HM],
                                       const uint32_t (&boff)[HN], uint32_t soff, uint32_t sstep, int nk, int wave,
                                       int lane) {
  using G = Stage<NPB, SCALED, HM, HN>;
#if defined(__HIP_DEVICE_COMPILE__)
  typedef __attribute__((address_space(3))) void *lds_ptr;
#endif
  // DMA instruction i of step k into stage st
  auto dma = [&](int k, int st, int i) {
#if defined(__HIP_DEVICE_COMPILE__)
    // device pass only: with a run-time voffset this builtin keeps the host pass from emitting the launch stub
    uint8_t *base = lds + st * G::kBytes + wave * 1024;
    const uint32_t kb = uint32_t(k) * ROWB;
    if (i < 2 * HM) {
      const int q = i / 2;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(i % 2 ? o.al : o.ah, (lds_ptr)(base + (i % 2 ? G::kALo : 0) + q * 4096), 16,
                                               aoff[q], kb, 0, 0);
    } else if (i < 2 * HM + NPB * HN) {
      const int q = (i - 2 * HM) / NPB, lo = (i - 2 * HM) % NPB;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(lo ? o.bl : o.bh, (lds_ptr)(base + (lo ? G::kBLo : G::kBHi) + q * 4096), 16,
                                               boff[q], kb, 0, 0);
    } else {  // every wave moves the scale block (the same bytes to the same place): one count of DMA for all waves
      __builtin_amdgcn_raw_ptr_buffer_load_lds(o.sc, (lds_ptr)(lds + st * G::kBytes + G::kScl), 16, soff,
                                               uint32_t(k) * sstep, 0, 0);
    }
#endif
  };
  auto issue = [&](int k, int st) {
#pragma unroll
    for (int i = 0; i < G::kDma; ++i) dma(k, st, i);
  };
  const int lr = lane & 15, g = lane >> 4, wm = wave >> 1, wn = wave & 1;
  const int arow = (wm * 16 * HM + lr) * ROWB, brow = (wn * 16 * HN + lr) * ROWB;
  const int slot0 = ((g ^ (lr & 7)) * 16), slot1 = (((4 + g) ^ (lr & 7)) * 16);
  struct Frag {
    half8 ah[HM], al[HM], b[HN], c[NPB == 2 ? HN : 1];
    float d[SCALED ? HN : 1];
  };
  auto read = [&](int st, int ck, Frag &f) {
    const uint8_t *p = lds + st * G::kBytes;
    const int sl = ck ? slot1 : slot0;
#pragma unroll
    for (int i = 0; i < HM; ++i) {
      f.ah[i] = *reinterpret_cast<const half8 *>(p + arow + i * 16 * ROWB + sl);
      f.al[i] = *reinterpret_cast<const half8 *>(p + G::kALo + arow + i * 16 * ROWB + sl);
    }
#pragma unroll
    for (int j = 0; j < HN; ++j) {
      f.b[j] = *reinterpret_cast<const half8 *>(p + G::kBHi + brow + j * 16 * ROWB + sl);
      if constexpr (NPB == 2) f.c[j] = *reinterpret_cast<const half8 *>(p + G::kBLo + brow + j * 16 * ROWB + sl);
      if constexpr (SCALED)
        f.d[j] = *reinterpret_cast<const float *>(p + G::kScl + (ck * 32 * HN + wn * 16 * HN + j * 16 + lr) * 4);
    }
  };
  // The MFMAs of one 32-deep chunk; with DMA, the instructions of step dk into stage dst spread between them (a wave's
  // next MFMA waits behind a DMA instruction that the texture unit has not taken yet).
  constexpr int kMfma = HM * HN * (NPB == 2 ? 3 : 2);
  auto compute = [&](const Frag &f, auto with_dma, int dk, int dst) {
    if constexpr (SCALED) {
      // column j's MFMAs (hi then lo chains of its row blocks) issue between the scale FMAs of column j - 1
      const f32x4 zero = {};
      f32x4 p[2][HM];
#pragma unroll
      for (int j = 0; j <= HN; ++j) {
        if (j < HN) {
#pragma unroll
          for (int i = 0; i < HM; ++i) p[j & 1][i] = MFMA(f.ah[i], f.b[j], zero);
#pragma unroll
          for (int i = 0; i < HM; ++i) p[j & 1][i] = MFMA(f.al[i], f.b[j], p[j & 1][i]);
        }
        if (j > 0) {
#pragma unroll
          for (int i = 0; i < HM; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[i][j - 1][r] += f.d[j - 1] * p[(j - 1) & 1][i][r];
        }
#pragma unroll
        for (int q = 0; q < 2 * HM; ++q) {
          if (j < HN) __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one MFMA of column j
          if (j > 0) __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);   // two FMAs of column j - 1
        }
      }
    } else {
#pragma unroll
      for (int n = 0; n < kMfma; ++n) {
        const int pass = n / (HM * HN), j = n / HM % HN, i = n % HM;
        acc[i][j] = MFMA(pass == 1 ? f.al[i] : f.ah[i], pass == 2 ? f.c[NPB == 2 ? j : 0] : f.b[j], acc[i][j]);
#pragma unroll
        for (int q = 0; q < G::kDma; ++q)
          if (decltype(with_dma)::value && q * kMfma / G::kDma == n) {
            __builtin_amdgcn_sched_barrier(0);
            dma(dk, dst, q);
            __builtin_amdgcn_sched_barrier(0);
          }
      }
    }
  };

#pragma unroll
  for (int s = 0; s < S; ++s)
    if (s < nk) issue(s, s);
  if (nk >= S) wait_vm<(S - 1) * G::kDma>();
  else wait_vm<0>();
  bare_barrier();
  Frag f0, f1;
  read(0, 0, f0);
  int st = 0;
  for (int k = 0; k < nk; ++k) {
    read(st, 1, f1);
    __builtin_amdgcn_sched_barrier(0);  // the reads issue ahead of the MFMAs that cover them
    compute(f0, std::false_type{}, 0, 0);
    const int nst = st + 1 == S ? 0 : st + 1;
    if (k + 1 < nk) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // this wave has read all of step k
      if (k + S - 1 < nk) wait_vm<(S - 2) * G::kDma>();
      else wait_vm<0>();
      bare_barrier();
      read(nst, 0, f0);
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (SCALED) {  // spread among the scale FMAs the DMA cost 8-15%
      if (k + S < nk) issue(k + S, st);
      compute(f1, std::false_type{}, 0, 0);
    } else if (k + S < nk) {
      compute(f1, std::true_type{}, k + S, st);
    } else {
      compute(f1, std::false_type{}, 0, 0);
    }
    st = nst;
  }
}

template <int EPI, int MODE, int HM, int HN, int S>
__global__ __launch_bounds__(256, (2 * lds_bytes<MODE, HM, HN, S>() <= 160 * 1024 ? 2 : 1)) void gemm_mid_kernel(
    const _Float16 *__restrict__ A, const _Float16 *__restrict__ Alo, int M, int K, const _Float16 *__restrict__ Wh,
    const _Float16 *__restrict__ Wl, const float *__restrict__ Ws, int N, float *__restrict__ C,
    _Float16 *__restrict__ C16, _Float16 *__restrict__ C16lo, int ldc, const float *__restrict__ bias, int MT, int NT,
    int ffn, RopeKvOut ro, int ro_row0, wide::KqCorr kq) {
  constexpr bool kScaled = kScaledMode<MODE>;
  constexpr bool kRope = EPI == kTileEpiRope || EPI == kTileEpiLayaRope;
  static_assert(!kRope || HN == 2, "the rotating epilogues take 64-column tiles");
  static_assert(HN % 2 == 0 || (EPI != int(Epi::SWIGLU) && EPI != int(Epi::GEGLU)), "gate and up blocks share a wave");
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  // Tile order: workgroups go to the 8 XCDs round-robin; each XCD takes a contiguous range of tiles, walked in groups
  // of up to GM M-tiles, M fastest, so an XCD's tiles share weight rows (each read from HBM by few XCDs) and A rows
  // through its L2.
  int mt, nt;
  {
    constexpr int GM = 16;
    const int per = gridDim.x >> 3, rem = gridDim.x & 7, xcd = blockIdx.x & 7;
    const int id = xcd * per + min(xcd, rem) + (blockIdx.x >> 3);
    const int group = id / (GM * NT), first = group * GM;
    const int gm = min(MT - first, GM), in = id - group * GM * NT;
    mt = first + in % gm;
    nt = in / gm;
  }
  const int m0 = mt * (32 * HM);
  // rows of this lane's part of DMA instruction q: 32 q + 8 wave + lane / 8, its chunk (lane % 8) ^ (row % 8).  Rows
  // past M read row M - 1 (their results are not stored), so every access is inside its buffer.
  const int r0 = wave * 8 + (lane >> 3), c16 = ((lane & 7) ^ (lane >> 3)) * 16;
  f32x4 acc[HM][HN];
#pragma unroll
  for (int i = 0; i < HM; ++i)
#pragma unroll
    for (int j = 0; j < HN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[i][j][r] = 0.0f;
  uint32_t aoff[HM], boff[HN];
  auto offsets = [&](int depth) {
#pragma unroll
    for (int q = 0; q < HM; ++q) aoff[q] = uint32_t(min(m0 + 32 * q + r0, M - 1)) * uint32_t(depth) * 2u + c16;
#pragma unroll
    for (int q = 0; q < HN; ++q) boff[q] = uint32_t(tile_wrow<EPI, HN>(32 * q + r0, nt, ffn, ro)) * uint32_t(depth) * 2u + c16;
  };
  Operands o;
  if constexpr (MODE == wide::WQ4) {
    // the correction of the two-pass form first: acc = (sum_c ks[m][c] (-B[n][c] 2^e_n)) 2^-e_n, depth kq.kp
    const int kp = kq.kp;
    offsets(kp);
    o.ah = resource(kq.ks, uint32_t(M) * kp * 2u);
    o.al = resource(kq.kslo, uint32_t(M) * kp * 2u);
    o.bh = resource(kq.bh, uint32_t(N) * kp * 2u);
    o.bl = resource(kq.bl, uint32_t(N) * kp * 2u);
    o.sc = o.bh;
    k_loop<2, false, HM, HN, 2>(lds, acc, o, aoff, boff, 0, 0, kp / BK, wave, lane);
#pragma unroll
    for (int j = 0; j < HN; ++j) {
      const float rs = kq.rs[tile_wrow<EPI, HN>((wave & 1) * (16 * HN) + j * 16 + (lane & 15), nt, ffn, ro)];
#pragma unroll
      for (int i = 0; i < HM; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[i][j][r] *= rs;
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");  // the main loop's waits count its own DMA only
    bare_barrier();                                             // and its stages reuse the LDS
  }
  offsets(K);
  o.ah = resource(A, uint32_t(M) * uint32_t(K) * 2u);
  o.al = resource(Alo, uint32_t(M) * uint32_t(K) * 2u);
  o.bh = resource(Wh, uint32_t(N) * uint32_t(K) * 2u);
  o.bl = MODE == wide::W2 ? resource(Wl, uint32_t(N) * uint32_t(K) * 2u) : o.bh;
  o.sc = o.bh;
  uint32_t soff = 0;
  if constexpr (kScaled) {
    // scales f32 [K/32][N]: a step's two chunks, four consecutive columns a lane (lanes past them repeat chunk 1 into
    // the pad of the scale block)
    o.sc = resource(Ws, uint32_t(N) * uint32_t(K / 32) * 4u);
    constexpr int kLanes = 8 * HN;  // lanes per chunk
    soff = (uint32_t(min(lane / kLanes, 1)) * uint32_t(N) + uint32_t(tile_wrow<EPI, HN>(4 * (lane % kLanes), nt, ffn, ro))) * 4u;
  }
  k_loop<MODE == wide::W2 ? 2 : 1, kScaled, HM, HN, S>(lds, acc, o, aoff, boff, soff, uint32_t(N) * 8u, K / BK, wave, lane);
  tile_epilogue<EPI, HM, HN>(acc, M, m0, nt, wave >> 1, wave & 1, lane, C, C16, C16lo, ldc, bias, ro, ro_row0);
}

}  // namespace mid
}  // namespace lg
