// Launches of the exact GEMM tiles of gemm_mid.h, and the choice between them and the 256 x 256 tiles.  Built with
// MFMA results in VGPRs (-mllvm -amdgpu-mfma-vgpr-form), as k_gemm_q8.hip.
#include <algorithm>
#include <cmath>

#include "gemm_mid.h"

namespace lg {
namespace {

using wide::W1;
using wide::W2;
using wide::WQ4;
using wide::WQ8;

// Tile configurations: (HM, HN, stages).
enum Tile { T11, T12, T22, T24, T24D, T44, kTiles, kNoTile = -1 };

// What a launch takes beyond ~3 us: microseconds per 64-deep K step of a workgroup alone on a CU (one) and of two sharing
// it (two; 0: the LDS holds one), and a round's fill and drain.  Fitted to launches of M 24-1437 over the q|k|v, o, gate|up
// and down shapes of the workload models (weights rotating through 1 GB).  one = 0: not a configuration of the mode.
struct StepCost {
  float one, two, fill;
};
constexpr StepCost kCost[4][kTiles] = {
    /* WQ8 */ {{0.23f, 0.40f, 1}, {0.30f, 0.54f, 1}, {0.46f, 0.78f, 1}, {0.84f, 1.03f, 1}, {0.68f, 0, 1}, {1.14f, 0, 1}},
    /* W1  */ {{0.19f, 0.36f, 0.5f}, {0.23f, 0.46f, 1}, {0.27f, 0.68f, 2}, {0.78f, 0.90f, 2}, {0.41f, 0, 2}, {0.66f, 0, 6.5f}},
    /* W2  */ {{0.26f, 0.50f, 1}, {0.43f, 0.74f, 1}, {0.44f, 0, 2}, {0, 0, 0}, {0.73f, 0, 2}, {1.29f, 0, 6}},
    /* WQ4 */ {{0.24f, 0.40f, 1}, {0.31f, 0.54f, 1}, {0.46f, 0.78f, 2}, {0, 0, 0}, {0.70f, 0, 2}, {1.14f, 0, 3}},
};
// What whole layers of 24-32,768 rows measure as a multiple of the table's cost: a launch of several rounds runs at a lower
// clock and shares L2, most of all where one workgroup fills a CU (F16 3584 x 18944 at 3,000 rows: 892 us for 605).  The table
// chooses among these tiles; against the 256 x 256 tiles and the RoPE pass this cost counts.
constexpr float kLong[4][kTiles] = {
    /* WQ8 */ {1.1f, 1.1f, 1.1f, 1.1f, 1.1f, 1.1f},
    /* W1  */ {1.06f, 1.06f, 1.06f, 1.1f, 1.4f, 1.3f},
    /* W2  */ {1.1f, 1.1f, 1.1f, 1.1f, 1.2f, 1.2f},
    /* WQ4 */ {1.1f, 1.1f, 1.1f, 1.1f, 1.2f, 1.25f},
};
constexpr int kHM[kTiles] = {1, 1, 2, 2, 2, 4}, kHN[kTiles] = {1, 2, 2, 4, 4, 4};
// a 256 x 256 tile's microseconds per 64-deep step, one workgroup per CU (mode order as above; F16 at 168 and 198 tiles
// of K 1024, the others from full rounds)
constexpr float kWideStep[4] = {3.5f, 2.75f, 4.7f, 3.5f};

// What the rotating epilogue adds to a round (table reads, eight stores a value pair): measured against the table's
// costs over F16, Q8_0 and Q4_K q|k|v at 1,100-32,768 rows.
constexpr float kRopeFill = 2.2f;

// Microseconds of `nk` steps on n CUs over rounds of two workgroups per CU (the last round alone when half of it or less is
// left), or of one; `extra` a round.
float cost(const StepCost &c, int64_t n, int64_t tiles, int nk, float extra) {
  const float fill = c.fill + extra;
  if (c.two == 0) return float((tiles + n - 1) / n) * (c.one * nk + fill);
  const int64_t rounds = tiles / (2 * n), rest = tiles - rounds * 2 * n;
  return float(rounds) * (c.two * nk + fill) + (rest == 0 ? 0.0f : (rest <= n ? c.one : c.two) * nk + fill);
}

// The cheapest configuration for M rows of a matrix of `rows` weight rows (only those of 64 columns when rope), and
// its cost; kNoTile when none divides the output.
int best_tile(int mode, int M, const DevMatrix &W, bool glu, bool rope, float *best) {
  const int rows = W.rows;
  const int64_t n = device_cus();
  int t = kNoTile;
  for (int i = 0; i < kTiles; ++i) {
    const int bm = 32 * kHM[i], bn = 32 * kHN[i];
    if (kCost[mode][i].one == 0 || rows % bn || (glu && kHN[i] % 2) || (rope && kHN[i] != 2)) continue;
    const float c = cost(kCost[mode][i], n, int64_t((M + bm - 1) / bm) * (rows / bn), W.cols / mid::BK, rope ? kRopeFill : 0.0f);
    if (t == kNoTile || c < *best) {
      t = i;
      *best = c;
    }
  }
  return t;
}

// the mode of an M-row launch of W, or -1 when these tiles do not take it
int mid_mode(int M, const DevMatrix &W) {
  const int mode = wide::prefill_mode(W);
  if (M <= 0 || mode < 0 || W.cols % mid::BK != 0) return -1;
  if (int64_t(W.rows) * W.cols * 2 >= (int64_t(1) << 32)) return -1;  // 32-bit buffer offsets of the weights
  return mode;
}

struct Launch {
  const _Float16 *A, *Alo;
  int M;
  const DevMatrix &W;
  float *C;
  _Float16 *C16, *C16lo;
  int ldc;
  const float *bias;
  const RopeKvOut &ro;
  hipStream_t st;
  const _Float16 *ks;
};

template <int EPI, int MODE, int HM, int HN, int S>
void launch_rows(const Launch &l) {
  const DevMatrix &W = l.W;
  const int N = W.rows, K = W.cols, NT = N / (32 * HN);
  constexpr int BM = 32 * HM, lds = mid::lds_bytes<MODE, HM, HN, S>();
  // activation rows per launch: the planes' buffer offsets are 32-bit
  const int64_t rows_cap = ((int64_t(1) << 31) - 1) / (int64_t(K) * 2) / BM * BM;
  LG_REQUIRE(rows_cap > 0, "gemm: K=%d too large", K);
  const auto fn = mid::gemm_mid_kernel<EPI, MODE, HM, HN, S>;
  grant_lds(reinterpret_cast<const void *>(fn), lds);
  KernelTimer *timer = kernel_timer();
  const KernelTimer whole = timer ? *timer : KernelTimer{};
  for (int m0 = 0; m0 < l.M;) {
    const int Mc = int(std::min<int64_t>(l.M - m0, rows_cap));
    if (timer) {
      timer->start = m0 == 0 ? whole.start : nullptr;
      timer->stop = m0 + Mc >= l.M ? whole.stop : nullptr;
    }
    const int MT = (Mc + BM - 1) / BM;
    LG_REQUIRE(int64_t(MT) * NT < (int64_t(1) << 31), "gemm: grid too large");
    wide::KqCorr kq;
    if (MODE == WQ4) {
      kq.kp = W.pkp;
      kq.ks = l.ks + int64_t(m0) * W.pkp;
      kq.kslo = l.ks + (int64_t(l.M) + m0) * W.pkp;
      kq.bh = W.pcl;
      kq.bl = W.pcl + int64_t(N) * W.pkp;
      kq.rs = W.pcr;
    }
    const int64_t co = int64_t(m0) * l.ldc;
    launch_timed(fn, dim3(MT * NT), dim3(256), lds, l.st, l.A + int64_t(m0) * K, l.Alo + int64_t(m0) * K, Mc, K,
                 static_cast<const _Float16 *>(W.pc), static_cast<const _Float16 *>(W.pcl),
                 static_cast<const float *>(W.pcs), N, l.C ? l.C + co : nullptr, l.C16 ? l.C16 + co : nullptr,
                 l.C16lo ? l.C16lo + co : nullptr, l.ldc, l.bias, MT, NT, N / 2, l.ro, m0, kq);
    m0 += Mc;
  }
  if (timer) *timer = whole;
  HIP_CHECK(hipGetLastError());
}

template <int EPI, int MODE>
void launch_tile(int tile, const Launch &l) {
  constexpr bool kRope = EPI == kTileEpiRope || EPI == kTileEpiLayaRope;
  constexpr bool kGlu = EPI == int(Epi::SWIGLU) || EPI == int(Epi::GEGLU);
  constexpr bool w2 = MODE == W2, wq4 = MODE == WQ4;
  switch (tile) {
    case T11:
      if constexpr (!kRope && !kGlu) launch_rows<EPI, MODE, 1, 1, w2 ? 5 : 6>(l);
      break;
    case T12: launch_rows<EPI, MODE, 1, 2, w2 ? 3 : 4>(l); break;
    case T22: launch_rows<EPI, MODE, 2, 2, w2 ? 4 : 3>(l); break;
    case T24:  // two workgroups per CU
      if constexpr (!kRope && !w2 && !wq4) launch_rows<EPI, MODE, 2, 4, 2>(l);
      break;
    case T24D:  // one, with more steps in flight
      if constexpr (!kRope) launch_rows<EPI, MODE, 2, 4, w2 ? 3 : 4>(l);
      break;
    case T44:
      if constexpr (!kRope) launch_rows<EPI, MODE, 4, 4, w2 ? 2 : 3>(l);
      break;
  }
}

template <int EPI>
void launch_mode(int mode, int tile, const Launch &l) {
  // GeGLU, ReLU and the encoder's rotation come with F16 weights only
  constexpr bool kF16Only = EPI == int(Epi::GEGLU) || EPI == int(Epi::RELU16) || EPI == kTileEpiLayaRope;
  if constexpr (kF16Only) {
    launch_tile<EPI, W1>(tile, l);
  } else {
    if (mode == WQ8) launch_tile<EPI, WQ8>(tile, l);
    else if (mode == W1) launch_tile<EPI, W1>(tile, l);
    else if (mode == W2) launch_tile<EPI, W2>(tile, l);
    else launch_tile<EPI, WQ4>(tile, l);
  }
}

}  // namespace

namespace {

// Whether launch_gemm_mid has the epilogue for weights of `mode`.
bool mid_epi(int mode, Epi epi) {
  return epi != Epi::F16 && ((epi != Epi::GEGLU && epi != Epi::RELU16) || mode == W1);
}

// Microseconds of the tile that a launch takes among many rounds; infinity when there is none.
float long_cost(int M, const DevMatrix &W, bool glu, bool rope) {
  const int mode = mid_mode(M, W);
  float c = 0.0f;
  const int t = best_tile(mode, M, W, glu, rope, &c);
  return t == kNoTile ? INFINITY : c * kLong[mode][t];
}

// The 256 x 256 tiles (where they take the launch) or those of gemm_mid.h (where they do); *us, if asked for: the
// modelled microseconds.  Fewer 256 x 256 tiles than 5/8 of the CUs leaves too many idle.  Between that and one tile
// per CU they still win (F16 at 1437 rows x 7168 gated, 168 tiles: 47.8 us against 53.4 of the best smaller tiles), and
// below it they lose.  A last round that is nearly empty loses too (301 rows x 37888 gated F16, 296 tiles, against 170
// us), so up to two rounds the modelled costs decide, with 8% for the larger tiles: over 60 shapes and row counts the
// choice is the faster one or within 4% of it (F16 3584 x 18944 at 3,000 rows 757 us against 892, at 4,800 rows 1623
// against 1529; Q4_K 3584 x 3584 at 4,800 rows 371 against 432).  Over more the card holds its power and the larger
// tiles, with fewer instructions an MFMA, win whatever their last round (the 16-request Q4_K/Q6_K batch, 3.5 rounds of
// Q6_K down: 31.4 against 34.0 ms).
GemmForm choose(int M, const DevMatrix &W, bool wide_takes, bool mid_takes, bool glu, bool rope, float *us) {
  const int64_t n = device_cus(), tiles = int64_t((M + wide::BM - 1) / wide::BM) * (W.rows / wide::BN);
  const auto mid_us = [&] { return mid_takes ? long_cost(M, W, glu, rope) : INFINITY; };
  if (wide_takes && tiles * 8 >= n * 5) {
    const int64_t rounds = (tiles + n - 1) / n;
    const float wide_us = float(rounds) * (kWideStep[wide::prefill_mode(W)] * (W.cols / mid::BK) + 1.0f);
    if (rounds > 2 || !(mid_us() * 1.08f < wide_us)) {
      if (us) *us = wide_us;
      return GemmForm::Wide;
    }
  }
  if (us) *us = mid_us();
  return mid_takes ? GemmForm::Mid : GemmForm::None;
}

}  // namespace

GemmForm gemm_form(int M, const DevMatrix &W, Epi epi, float *us) {
  const int mode = mid_mode(M, W);
  return choose(M, W, gemm_wide_takes(M, W, epi), mode >= 0 && mid_epi(mode, epi), epi == Epi::SWIGLU || epi == Epi::GEGLU,
                false, us);
}

GemmForm gemm_rope_form(int M, const DevMatrix &W, int hd, float *us) {
  return choose(M, W, gemm_wide_rope_takes(M, W, hd), gemm_mid_rope_takes(M, W, hd), false, true, us);
}

GemmForm gemm_laya_rope_form(int M, const DevMatrix &W, int heads) {
  return choose(M, W, heads % 2 == 0 && gemm_wide_takes(M, W, Epi::F32), gemm_mid_laya_rope_takes(M, W), false, true, nullptr);
}

bool launch_gemm_mid(const _Float16 *A, const _Float16 *Alo, int M, const DevMatrix &W, Epi epi, float *C,
                     _Float16 *C16, _Float16 *C16lo, int ldc, const float *bias, hipStream_t st, const _Float16 *ks) {
  const int mode = mid_mode(M, W);
  if (mode < 0 || !A || !Alo) return false;
  const bool glu = epi == Epi::SWIGLU || epi == Epi::GEGLU;
  if (!mid_epi(mode, epi)) return false;
  LG_REQUIRE(mode != WQ4 || ks, "gemm: an exact Q4_K launch needs its activation's chunk sums");
  float c = 0.0f;
  const int tile = best_tile(mode, M, W, glu, false, &c);
  if (tile == kNoTile) return false;
  const RopeKvOut none;
  const Launch l{A, Alo, M, W, C, C16, C16lo, ldc, bias, none, st, ks};
  switch (epi) {
    case Epi::F32: launch_mode<int(Epi::F32)>(mode, tile, l); break;
    case Epi::ADD: launch_mode<int(Epi::ADD)>(mode, tile, l); break;
    case Epi::SWIGLU: launch_mode<int(Epi::SWIGLU)>(mode, tile, l); break;
    case Epi::GEGLU: launch_mode<int(Epi::GEGLU)>(mode, tile, l); break;
    case Epi::RELU16: launch_mode<int(Epi::RELU16)>(mode, tile, l); break;
    default: return false;
  }
  return true;
}

bool gemm_mid_rope_takes(int M, const DevMatrix &W, int hd) {
  return (hd == 64 || hd == 128) && W.rows % hd == 0 && mid_mode(M, W) >= 0;
}

void launch_gemm_mid_rope(const _Float16 *A, const _Float16 *Alo, int M, const DevMatrix &W, const float *bias,
                          const RopeKvOut &ro, hipStream_t st, const _Float16 *ks) {
  LG_REQUIRE(A && Alo && gemm_mid_rope_takes(M, W, ro.hd) && ro.col0 % ro.hd == 0 &&
                 ro.col0 / ro.hd + W.rows / ro.hd <= ro.hq + 2 * ro.hkv,
             "gemm rope: %d rows of this projection are not a launch of the 64-column tiles", M);
  LG_REQUIRE(ro.cosT && ro.sinT && ro.tok_pos && ro.tok_page && ro.q16 && ro.q16lo && ro.kpool && ro.vpool,
             "gemm rope: missing output");
  LG_REQUIRE(ro.page_tokens >= 4 && ro.page_tokens % 4 == 0 && ro.page_stride > 0, "gemm rope: bad page geometry");
  LG_REQUIRE(ro.kv_planes == 1 || ro.kv_planes == 2, "gemm rope: KV pools hold 1 or 2 planes, not %d", ro.kv_planes);
  const int mode = mid_mode(M, W);
  LG_REQUIRE(mode != WQ4 || ks, "gemm: an exact Q4_K launch needs its activation's chunk sums");
  float c = 0.0f;
  const int tile = best_tile(mode, M, W, false, true, &c);
  launch_mode<kTileEpiRope>(mode, tile, Launch{A, Alo, M, W, nullptr, nullptr, nullptr, 0, bias, ro, st, ks});
}

bool gemm_mid_laya_rope_takes(int M, const DevMatrix &W) { return W.rows % 64 == 0 && mid_mode(M, W) == W1; }

void launch_gemm_mid_laya_rope(const _Float16 *A, const _Float16 *Alo, int M, const DevMatrix &W, const float *bias,
                               const float *cosT, const float *sinT, const int32_t *tok_pos, int heads, float *C,
                               int ldc, hipStream_t st) {
  LG_REQUIRE(A && Alo && C && cosT && sinT && tok_pos, "gemm laya rope: missing operand");
  LG_REQUIRE(gemm_mid_laya_rope_takes(M, W) && heads > 0 && W.rows == 3 * heads * 64 && ldc >= W.rows,
             "gemm laya rope: %d rows are not q|k|v of %d 64-dim heads", W.rows, heads);
  RopeKvOut ro;
  ro.cosT = cosT;
  ro.sinT = sinT;
  ro.tok_pos = tok_pos;
  ro.hq = heads;
  ro.hd = 64;
  float c = 0.0f;
  const int tile = best_tile(W1, M, W, false, true, &c);
  launch_mode<kTileEpiLayaRope>(W1, tile, Launch{A, Alo, M, W, C, nullptr, nullptr, ldc, bias, ro, st, nullptr});
}

}  // namespace lg
