// Linear y[M,N] = x[M,K] . w[N,K]^T above 8 tokens for gfx950 (bf16/fp16,
// 16-byte rows): the verify forwards (up to 64 rows or so), where it streams
// the weight, and prompts, where the matrix cores bound it.
//
// A workgroup computes a tile of BN weight rows x BM tokens over its share of
// K, 64 k elements (128 bytes of every row) a stage.  Both operands go from
// memory straight into LDS (buffer_load ... lds), ST - 1 stages ahead of the
// one being multiplied, so a stage costs its wave no registers and one
// barrier, and each operand byte is fetched once per workgroup: the row-block
// kernels of thin_gemm.hip fetch the activations once per wave and hold at
// most two batches of registers in flight.
//
// The waves split the tile WM x WN; a wave's TN x TM blocks of 16 x 16 reuse
// each LDS operand TM (TN) times.  The tiles (kTiles):
//   32 x 64, 64 x 64   up to 32 / 64 tokens: many small workgroups with three
//                      stages in flight, the weight loads non-temporal
//   64 x 128           the same where the rows alone fill the chip
//   128 x 64           above that, where rows are few
//   128 x 128, 256 x 128, 128 x 256   prompts, with 8 waves: a stage of the
//                      last two is 1.0k cycles of MFMA a SIMD and 1.4k of LDS,
//                      and of two waves on a SIMD one multiplies while the
//                      other reads (four waves of twice the blocks: 1.1k of
//                      LDS, but one after the other).  Reading a k step's
//                      operands during the products of the one before, within
//                      a wave, cost 3 to 8% on top of that and was left out.
// Whole calls, the sum of their partials included, in a graph over 2.5 to 7 GB
// of weights (us, against the row-block kernels): 36 tokens: gate/up
// 4096->2x12288 42.1 (45.3), down 12288->4096 21.8 (25.6), qkv 4096->6144 14.6
// (17.9), o 4096->4096 11.1 (12.5); 1024 tokens: gate/up 192 us, 1076 TFLOP/s
// (1.3 ms, 160), with 4 waves 222; down in 2 partials 98 (4 waves 112), qkv 58
// (75), both without their sum.
#include "simsd_kernels.h"
#include "thin_common.hpp"
#include "thin_tile.hpp"
#include "tile_core.hpp"

namespace simsd {

template <int DT, int WM, int WN, int TM, int TN, int ST, int AUXW, bool PARTIAL, bool GLU>
__global__ __launch_bounds__(64 * WM * WN, tile_waves_per_simd(WM * WN, TM * TN, ST * TileShape<WM, WN, TM, TN, ST, GLU>::kStage)) void thin_tile_kernel(ThinArgs a, int tiles_n, int tiles_m) {
  constexpr int ES = DTypeInfo<DT>::kSize;
  using S = TileShape<WM, WN, TM, TN, ST, GLU>;
  constexpr int BM = S::BM, OUT = S::OUT, LN = S::LN, LM = S::LM;
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int wn = wv % WN, wm = wv / WN;
  const int g = lane >> 4, r = lane & 15;

  // workgroup -> tile: workgroups go to the XCDs in turn, so XCD x takes a
  // run of consecutive tiles, token tiles first: its L2 then serves a weight
  // panel to all of its token tiles
  const int total = gridDim.x, q8 = total >> 3, r8 = total & 7;
  const int xcd = blockIdx.x & 7;
  int tile = xcd * q8 + min(xcd, r8) + (int)(blockIdx.x >> 3);
  const int tm = tile % tiles_m;
  tile /= tiles_m;
  const int tn = tile % tiles_n;
  const int split_id = tile / tiles_n;
  const int64_t n_tile = (int64_t)tn * OUT, m_tile = (int64_t)tm * BM;

  const uint32_t Kb = (uint32_t)(a.K * ES);
  const uint32_t swn_b = (uint32_t)(a.swn * ES), sxm_b = (uint32_t)(a.sxm * ES), sw2n_b = (uint32_t)(a.sw2n * ES);
  const int k0 = split_id * a.steps_per_split, k1 = min(a.steps, k0 + a.steps_per_split);
  const int rows_valid = (int)min((int64_t)OUT, a.N - n_tile);
  const int cols_valid = (int)min((int64_t)BM, a.M - m_tile);
  const rsrc_t rW = make_rsrc(a.w + n_tile * swn_b, (uint32_t)(rows_valid - 1) * swn_b + Kb);
  const rsrc_t rW2 = GLU ? make_rsrc(a.w2 + n_tile * sw2n_b, (uint32_t)(rows_valid - 1) * sw2n_b + Kb) : rW;
  const rsrc_t rX = make_rsrc(a.x + m_tile * sxm_b, (uint32_t)(cols_valid - 1) * sxm_b + Kb);

  uint32_t won[LN], xon[LM];
  const int lr = lane >> 3;
#pragma unroll
  for (int i = 0; i < LN; ++i) {
    const int R = (wv * LN + i) * 8 + lr;
    won[i] = (uint32_t)S::weight_row(R) * (S::up(wv, i) ? sw2n_b : swn_b) + S::piece(lane, R);
  }
#pragma unroll
  for (int i = 0; i < LM; ++i) {
    const int R = (wv * LM + i) * 8 + lr;
    xon[i] = (uint32_t)R * sxm_b + S::piece(lane, R);
  }

  f32x4_t acc[TN][TM];
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  tile_main_loop<DT, WM, WN, TM, TN, ST, AUXW, GLU>(rW, rW2, rX, won, xon, Kb, k0, k1, lane, wv, acc);

  // epilogue: lane (g, r) of block (i, c): columns 4g .. 4g + 3 of token r,
  // stored through descriptors (offsets of columns past N or rows past M: out
  // of range, dropped)
  constexpr int OB = GLU ? TN / 2 : TN;   // output blocks of a wave
  constexpr int OS = PARTIAL ? 4 : ES;
  const int64_t out_ld = PARTIAL ? (GLU ? 2 * a.N : a.N) : a.sym;
  char* obase = PARTIAL ? reinterpret_cast<char*>(a.part) + ((int64_t)split_id * a.M + m_tile) * out_ld * 4
                        : a.y + m_tile * out_ld * ES;
  const int n_left = (int)(a.N - n_tile);
  const uint32_t out_b = (uint32_t)(out_ld * OS), res_b = (uint32_t)(a.srm * ES);
  const rsrc_t rO = make_rsrc(obase, (uint32_t)(cols_valid - 1) * out_b + (uint32_t)((PARTIAL && GLU ? 2 : 1) * a.N * OS));
  const rsrc_t rR = make_rsrc(a.res + m_tile * a.srm * ES, a.res != nullptr ? (uint32_t)(cols_valid - 1) * res_b + (uint32_t)(a.N * ES) : 0u);
  const rsrc_t rBias = make_rsrc(a.bias, a.bias != nullptr ? (uint32_t)(a.N * ES) : 0u);
  const bool vec = ((out_b | (uint32_t)reinterpret_cast<uintptr_t>(obase)) & (4 * OS - 1)) == 0 && a.N % 4 == 0 &&
                   (PARTIAL || a.res == nullptr || ((res_b | (uint32_t)reinterpret_cast<uintptr_t>(a.res)) & 7) == 0);
  auto finish = [&](float v, float u, float bias, float res) {
    if (GLU) return silu_mul<DT>(v, u);
    if (a.bias != nullptr) v = round_to<DT>(v) + bias;
    if (a.res != nullptr) v = round_to<DT>(v) + res;
    return v;
  };
#pragma unroll
  for (int i = 0; i < OB; ++i) {
    const int nl = (wn * OB + i) * 16 + 4 * g;   // first of the lane's columns within the tile
    const uint32_t n = (uint32_t)(n_tile + nl);
    float bias[4] = {0.f, 0.f, 0.f, 0.f};
    if (!PARTIAL && !GLU && a.bias != nullptr) {
#pragma unroll
      for (int j = 0; j < 4; ++j) bias[j] = h16_to_f32<DT>(buf_load2(rBias, nl + j < n_left ? (n + j) * ES : kOob));
    }
#pragma unroll
    for (int c = 0; c < TM; ++c) {
      const int ml = (wm * TM + c) * 16 + r;
      const f32x4_t v = acc[i][c], u = acc[GLU ? i + OB : i][c];
      const uint32_t ro = (uint32_t)ml * out_b + n * OS;
      const bool ok = ml < cols_valid && nl < n_left;
      if (vec) {
        if (PARTIAL) {
          buf_store16(rO, ok ? ro : kOob, __builtin_bit_cast(u32x4_t, v));
          if (GLU) buf_store16(rO, ok ? ro + (uint32_t)(a.N * 4) : kOob, __builtin_bit_cast(u32x4_t, u));
        } else {
          u32x2_t rs = u32x2_t{0u, 0u};
          if (!GLU && a.res != nullptr) rs = buf_load8(rR, ok ? (uint32_t)ml * res_b + n * ES : kOob);
          uint32_t o[4];
#pragma unroll
          for (int j = 0; j < 4; ++j)
            o[j] = f32_to_h16<DT>(finish(v[j], u[j], bias[j], h16_to_f32<DT>(rs[j >> 1] >> (16 * (j & 1)))));
          buf_store8(rO, ok ? ro : kOob, u32x2_t{o[0] | (o[1] << 16), o[2] | (o[3] << 16)});
        }
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const bool okj = ml < cols_valid && nl + j < n_left;
          const uint32_t o = okj ? ro + j * OS : kOob;
          if (PARTIAL) {
            buf_store4(rO, o, __float_as_uint(v[j]));
            if (GLU) buf_store4(rO, okj ? o + (uint32_t)(a.N * 4) : kOob, __float_as_uint(u[j]));
          } else {
            float rs = 0.f;
            if (!GLU && a.res != nullptr) rs = h16_to_f32<DT>(buf_load2(rR, okj ? (uint32_t)ml * res_b + (n + j) * ES : kOob));
            buf_store2(rO, o, f32_to_h16<DT>(finish(v[j], u[j], bias[j], rs)));
          }
        }
      }
    }
  }
}

// ------------------------------------------------------------------ host side
namespace {

inline int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

// The tiles and what one costs, for the choice below: a workgroup's fixed
// time, its time per stage alone on its CU and as one of two on it (us), and
// the rate at which a whole launch streams weights (bytes / us).  The first
// four are fitted to 11500 timings of whole calls (plain, gated, and partials
// with their consumer) over 27 weight shapes x 16 token counts (9 .. 80) x
// splits 1 .. 8, the weights from a 1.6 GB pool: the choice by them is within
// 1% (geometric mean; at most 14%) of the best tile and split timed.  The others
// to 900 timings of prompts (up to 2048 tokens): within 1.3%, at most 20%.
struct Tile {
  int wm, wn, tm, tn, st;
  int per_cu;        // workgroups a CU holds (LDS)
  float launch, wg, alone, pair, rate;
};
constexpr Tile kTiles[] = {
    {2, 2, 1, 2, 4, 3, 1.94f, 0.37f, 0.277f, 0.558f, 5.81e6f},
    {2, 2, 2, 2, 4, 2, 1.12f, 1.11f, 0.325f, 0.623f, 5.5e6f},
    {1, 4, 4, 2, 4, 1, 0.229f, 2.49f, 0.493f, 0.493f, 5.5e6f},
    {2, 2, 4, 2, 4, 1, 0.904f, 1.69f, 0.427f, 0.427f, 4.39e6f},
    {2, 4, 4, 2, 4, 1, 0.0f, 6.0f, 0.52f, 0.52f, 3.7e6f},
    {4, 2, 4, 4, 3, 1, 0.0f, 8.4f, 0.78f, 0.78f, 3.4e6f},
    {2, 4, 4, 4, 3, 1, 0.0f, 8.8f, 0.83f, 0.83f, 3.1e6f},
};
constexpr int kNumTiles = sizeof(kTiles) / sizeof(kTiles[0]);
constexpr int kCus = 256;
constexpr double kTileFloorUs = 1.48;      // a launch, beside streaming its weights
// summing the partials of a split: a launch of its own, or (partials calls)
// what more of them cost the launch that consumes them; us and bytes / us
constexpr float kSumUs = 2.21f, kSumRate = 1.84e6f, kConsumeUs = 0.147f, kConsumeRate = 0.822e6f;

float tile_cost(const Tile& t, int64_t wgs, int64_t stages, double weight_bytes) {
  const double s = (double)(cdiv(stages, t.st) * t.st);
  const int64_t per_cu = cdiv(wgs, kCus), rounds = per_cu / t.per_cu, rest = per_cu % t.per_cu;
  const double full = t.per_cu == 1 ? t.alone : t.pair * t.per_cu / 2;
  double us = t.launch + rounds * (s * full + t.wg);
  if (rest) us += s * (rest == 1 ? t.alone : t.pair) + t.wg;
  const double stream = kTileFloorUs + weight_bytes / t.rate;
  return (float)(us > stream ? us : stream);
}

template <int DT, int I, bool PARTIAL, bool GLU>
void launch_tile(const TilePlan& p, const ThinArgs& a, hipStream_t stream) {
  constexpr Tile t = kTiles[I];
  // up to 64 tokens the weight is read once: non-temporal loads
  constexpr int kAuxW = 16 * t.tm * t.wm <= 64 ? kAuxStream : kAuxKeep;
  hipLaunchKernelGGL((thin_tile_kernel<DT, t.wm, t.wn, t.tm, t.tn, t.st, kAuxW, PARTIAL, GLU>),
                     dim3((unsigned)(p.tiles_n * p.tiles_m * p.split)), dim3(64 * t.wm * t.wn), 0, stream, a,
                     (int)p.tiles_n, (int)p.tiles_m);
}

template <int DT, int I>
void launch_form(const TilePlan& p, const ThinArgs& a, bool glu, bool part, hipStream_t stream) {
  if (glu && part) launch_tile<DT, I, true, true>(p, a, stream);
  else if (glu) launch_tile<DT, I, false, true>(p, a, stream);
  else if (part) launch_tile<DT, I, true, false>(p, a, stream);
  else launch_tile<DT, I, false, false>(p, a, stream);
}

template <int DT>
void launch_cfg(const TilePlan& p, const ThinArgs& a, bool glu, bool part, hipStream_t stream) {
  switch (p.cfg) {
    case 0: launch_form<DT, 0>(p, a, glu, part, stream); break;
    case 1: launch_form<DT, 1>(p, a, glu, part, stream); break;
    case 2: launch_form<DT, 2>(p, a, glu, part, stream); break;
    case 3: launch_form<DT, 3>(p, a, glu, part, stream); break;
    case 4: launch_form<DT, 4>(p, a, glu, part, stream); break;
    case 5: launch_form<DT, 5>(p, a, glu, part, stream); break;
    default: launch_form<DT, 6>(p, a, glu, part, stream); break;
  }
}

}  // namespace

TilePlan thin_tile_plan(int64_t M, int64_t rows, int64_t K, bool partials, int split_k) {
  TilePlan best{};
  float best_us = 0.f;
  const int64_t stages = cdiv(K * 2, kTileK);
  for (int i = 0; i < kNumTiles; ++i) {
    const Tile& t = kTiles[i];
    const int bm = 16 * t.tm * t.wm, bn = 16 * t.tn * t.wn;
    if (bm < 64 ? M > 32 : bm > 64 && M <= 64) continue;   // half the tile or more would be padding, or x read twice
    const int64_t tn = cdiv(rows, bn), tm = cdiv(M, bm);
    for (int s : {1, 2, 4, 8}) {
      if (split_k > 0 ? s > 1 : s > 1 && stages < 4 * s) continue;
      const int sp = split_k > 0 ? split_k : s;
      float us = tile_cost(t, tn * tm * sp, cdiv(stages, sp), (double)rows * K * 2);
      if (sp > 1) us += (partials ? kConsumeUs : kSumUs) + (float)sp * M * rows * 4 / (partials ? kConsumeRate : kSumRate);
      if (best_us == 0.f || us < best_us) {
        best_us = us;
        best.cfg = i;
        best.bm = bm;
        best.bn = bn;
        best.waves = t.wm * t.wn;
        best.split = sp;
        best.tiles_n = tn;
        best.tiles_m = tm;
      }
    }
  }
  best.steps = (int)stages;
  best.steps_per_split = (int)cdiv(stages, best.split);
  return best;
}

bool thin_tile_fits(int64_t M, int64_t N, int64_t K, int64_t sxm, int64_t swn, int64_t sw2n, int64_t sym, int64_t srm) {
  // every row's bytes from a tile's first row, within 31 bits (kTileOob is past them)
  const auto ok = [](int64_t rows, int64_t stride, int64_t len, int64_t es) {
    return stride >= 0 && (rows - 1) * stride * es + len * es < (int64_t)kTileOob;
  };
  const int64_t m = M < 256 ? M : 256;
  return ok(256, M > 1 ? sxm : 0, K, 2) && ok(256, N > 1 ? swn : 0, K, 2) && ok(256, N > 1 ? sw2n : 0, K, 2) && ok(m, sym, N, 2) &&
         ok(m, srm, N, 2) && ok(m, 2 * N, 2 * N, 4);
}

void launch_thin_tile(const TilePlan& p, ThinArgs a, int dtype, bool glu, bool part, hipStream_t stream) {
  a.steps = p.steps;
  a.steps_per_split = p.steps_per_split;
  if (dtype == kBF16) launch_cfg<kBF16>(p, a, glu, part, stream);
  else launch_cfg<kF16>(p, a, glu, part, stream);
}

}  // namespace simsd
