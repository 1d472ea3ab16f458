// Grouped expert projections for steps whose experts hold more slots than one
// 16-slot tile (gfx950, bf16/fp16).
//
// The align tables group an expert's slots in tiles of 16, and the single-tile
// kernels stream the expert's weights once per tile: 2.4 times at 1001 tokens
// of 8 picks over 256 experts.  Here a workgroup takes a run of up to 4
// consecutive tiles of one expert as one 64-row activation tile of the linear
// layers' tile kernel, whose activation loads gather the slots' rows (every
// load into LDS has its own address), and the weights are read once for it.
// 1001 tokens, H 2048, I 512 (traced): gate_up 258 us (4.2 TB/s of weights),
// down 155; the case's step, with the align kernel's parallel scatter and the
// wide combine, 893 -> 447.  What bounds it now is streaming 32 (gate_up) and 8 (down)
// stages per short-lived workgroup, and the workgroups of the tiles that are
// not the first of a run, which exit after a load.
#include "moe_common.hpp"
#include "simsd_kernels.h"
#include "tile_core.hpp"

namespace simsd {
namespace {

constexpr int kGroup = 4;   // tiles of one expert a workgroup takes

struct MoeTileArgs {
  const char* x;             // activation rows: x (gate_up) or h (down)
  uint32_t x_b, x_rows;      // their stride in bytes and count (routed)
  const char *w, *w2;        // routed weights: gate and up, or down
  int64_t we, w2e;           // expert strides in bytes
  uint32_t w_b, w2_b;        // row strides in bytes
  const char *sx, *sw, *sw2; // the shared expert's
  uint32_t sx_b, sw_b, sw2_b;
  char *out, *sout;          // routed (slot rows) and shared (token rows) outputs
  uint32_t N, sN, Kb, sKb;   // output columns and row bytes
  const int32_t *slots, *tile_expert;
  int num_tiles, E, k, T;
  uint32_t k_magic;          // floor(2^32 / k) + 1: slots below 2^16 divide exactly
};

// grid (tiles, column tiles).  A workgroup whose tile is the first of a run of
// kGroup within its expert's tiles computes the run; the others exit.
// GLU: h = silu(gate) * up of the slots' tokens; else the rows of h times down.
template <int DT, int WM, int WN, int TM, int TN, int ST, int AUXW, bool GLU>
__global__ __launch_bounds__(64 * WM * WN, tile_waves_per_simd(WM * WN, TM * TN, ST * TileShape<WM, WN, TM, TN, ST, GLU>::kStage))
void moe_tile_kernel(MoeTileArgs a) {
  using S = TileShape<WM, WN, TM, TN, ST, GLU>;
  constexpr int ES = 2;
  constexpr int LN = S::LN, LM = S::LM;
  static_assert(S::BM == kGroup * kTile, "a run of tiles");
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int wn = wv % WN, wm = wv / WN;
  const int g = lane >> 4, r = lane & 15, lr = lane >> 3;
  const int t = blockIdx.x;
  const bool shared = t >= a.num_tiles;
  int e = -1, rows = 0;   // rows: of the run
  if (shared) {
    const int first = (t - a.num_tiles) * kTile;
    if ((t - a.num_tiles) % kGroup != 0) return;
    rows = min(kGroup * kTile, a.T - first);
  } else {
    e = a.tile_expert[t];
    if (e < 0 || e >= a.E) return;
    // this tile's place among its expert's: lane l looks l + 1 tiles back,
    // and l + 1 ahead for the run's length
    int back = 0;
    for (int b0 = t - 1;; b0 -= 64) {
      const int b = b0 - lane;
      const uint64_t other = __ballot(b < 0 || a.tile_expert[max(b, 0)] != e);
      if (other != 0) {
        back += __builtin_ctzll(other);
        break;
      }
      back += 64;
    }
    if (back % kGroup != 0) return;
    const int f = t + 1 + lane;
    const uint64_t other = __ballot(f >= a.num_tiles || a.tile_expert[min(f, a.num_tiles - 1)] != e);
    rows = min(other != 0 ? __builtin_ctzll(other) + 1 : 64, kGroup) * kTile;
  }
  const uint32_t N = shared ? a.sN : a.N, Kb = shared ? a.sKb : a.Kb;
  const uint32_t n_tile = blockIdx.y * S::OUT;
  if (n_tile >= N) return;
  const int n_left = (int)(N - n_tile), cols = min(n_left, S::OUT);
  const uint32_t w_b = shared ? a.sw_b : a.w_b, w2_b = shared ? a.sw2_b : a.w2_b, x_b = shared ? a.sx_b : a.x_b;
  const char* w = shared ? a.sw : a.w + (int64_t)e * a.we;
  const char* w2 = shared ? a.sw2 : a.w2 + (int64_t)e * a.w2e;
  const rsrc_t rW = make_rsrc(w + (int64_t)n_tile * w_b, (uint32_t)(cols - 1) * w_b + Kb);
  const rsrc_t rW2 = GLU ? make_rsrc(w2 + (int64_t)n_tile * w2_b, (uint32_t)(cols - 1) * w2_b + Kb) : rW;
  const rsrc_t rX = make_rsrc(shared ? a.sx : a.x, ((shared ? (uint32_t)a.T : a.x_rows) - 1) * x_b + Kb);
  // row R of the run: its slot (shared: token), -1 past the group's last
  auto slot_of = [&](int R) {
    if (R >= rows) return -1;
    return shared ? (t - a.num_tiles) * kTile + R : a.slots[t * kTile + R];
  };
  uint32_t won[LN], xon[LM];
#pragma unroll
  for (int i = 0; i < LM; ++i) {
    const int R = (wv * LM + i) * 8 + lr;
    const int s = slot_of(R);
    // gate_up reads the slot's token, down the slot's h row
    const uint32_t row = GLU && !shared && a.k > 1 ? __umulhi((uint32_t)s, a.k_magic) : (uint32_t)s;
    xon[i] = s >= 0 ? row * x_b + S::piece(lane, R) : kTileOob;
  }
#pragma unroll
  for (int i = 0; i < LN; ++i) {
    const int R = (wv * LN + i) * 8 + lr;
    won[i] = (uint32_t)S::weight_row(R) * (S::up(wv, i) ? w2_b : w_b) + S::piece(lane, R);
  }
  f32x4_t acc[TN][TM];
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  tile_main_loop<DT, WM, WN, TM, TN, ST, AUXW, GLU>(rW, rW2, rX, won, xon, Kb, 0, (int)((Kb + kTileK - 1) / kTileK),
                                                        lane, wv, acc);
  // lane (g, r) of block (i, c): columns 4g .. 4g + 3 of row c * 16 + r, at its slot's row
  constexpr int OB = GLU ? TN / 2 : TN;
  const uint32_t o_b = N * ES;
  const rsrc_t rO = make_rsrc(shared ? a.sout : a.out, (shared ? (uint32_t)a.T : (uint32_t)(a.T * a.k)) * o_b);
  const bool vec = N % 4 == 0;
#pragma unroll
  for (int c = 0; c < TM; ++c) {
    const int s = slot_of((wm * TM + c) * 16 + r);
#pragma unroll
    for (int i = 0; i < OB; ++i) {
      const int nl = (wn * OB + i) * 16 + 4 * g;
      uint32_t o[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float v = acc[i][c][j];
        if (GLU) {
          const float gv = round_to<DT>(v), uv = round_to<DT>(acc[GLU ? i + OB : i][c][j]);
          v = round_to<DT>(silu_f32(gv)) * uv;
        }
        o[j] = f32_to_h16<DT>(v);
      }
      const uint32_t ro = (uint32_t)s * o_b + (n_tile + nl) * ES;
      if (vec) {
        buf_store8(rO, s >= 0 && nl < n_left ? ro : kOob, u32x2_t{o[0] | (o[1] << 16), o[2] | (o[3] << 16)});
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) buf_store2(rO, s >= 0 && nl + j < n_left ? ro + j * ES : kOob, o[j]);
      }
    }
  }
}

MoeTileArgs common(const MoeArgs& a) {
  MoeTileArgs t{};
  t.slots = a.slots;
  t.tile_expert = a.tile_expert;
  t.num_tiles = a.num_tiles;
  t.E = a.E;
  t.k = a.k;
  t.T = (int)a.T;
  t.k_magic = (uint32_t)((1ull << 32) / (uint64_t)a.k) + 1u;
  return t;
}

// Few experts hold more slots than a run: their weights are read once, and
// non-temporal (1001 tokens, 31 slots an expert: 464 -> 447 us a layer; at 94
// slots it would cost 399 -> 451).
bool weights_once(const MoeArgs& a) { return a.T * a.k <= 40ll * a.E; }

template <int DT>
void gate_up(const MoeArgs& a, hipStream_t stream) {
  MoeTileArgs t = common(a);
  t.x = a.x; t.x_b = (uint32_t)(a.sxt * 2); t.x_rows = (uint32_t)a.T;
  t.w = a.wg; t.we = a.sge * 2; t.w_b = (uint32_t)(a.sgi * 2);
  t.w2 = a.wu; t.w2e = a.sue * 2; t.w2_b = (uint32_t)(a.sui * 2);
  t.sx = a.x; t.sx_b = t.x_b;
  t.sw = a.shg; t.sw_b = (uint32_t)(a.shg_i * 2);
  t.sw2 = a.shu; t.sw2_b = (uint32_t)(a.shu_i * 2);
  t.out = a.h; t.sout = a.hs;
  t.N = (uint32_t)a.I; t.sN = (uint32_t)a.Is;
  t.Kb = t.sKb = (uint32_t)(a.H * 2);
  const int64_t imax = a.I > a.Is ? a.I : a.Is;
  constexpr unsigned OUT = TileShape<2, 2, 2, 2, 4, true>::OUT;
  const dim3 grid((unsigned)(a.num_tiles + a.shared_tiles), (unsigned)((imax + OUT - 1) / OUT));
  if (weights_once(a)) hipLaunchKernelGGL((moe_tile_kernel<DT, 2, 2, 2, 2, 4, kAuxStream, true>), grid, dim3(256), 0, stream, t);
  else hipLaunchKernelGGL((moe_tile_kernel<DT, 2, 2, 2, 2, 4, kAuxKeep, true>), grid, dim3(256), 0, stream, t);
}

template <int DT>
void down(const MoeArgs& a, hipStream_t stream) {
  MoeTileArgs t = common(a);
  t.x = a.h; t.x_b = (uint32_t)(a.I * 2); t.x_rows = (uint32_t)(a.T * a.k);
  t.w = a.wd; t.we = a.sde * 2; t.w_b = (uint32_t)(a.sdh * 2);
  t.sx = a.hs; t.sx_b = (uint32_t)(a.Is * 2);
  t.sw = a.shd; t.sw_b = (uint32_t)(a.shd_h * 2);
  t.out = a.y; t.sout = a.ys;
  t.N = t.sN = (uint32_t)a.H;
  t.Kb = (uint32_t)(a.I * 2);
  t.sKb = (uint32_t)(a.Is * 2);
  constexpr unsigned OUT = TileShape<1, 4, 4, 2, 3, false>::OUT;
  const dim3 grid((unsigned)(a.num_tiles + a.shared_tiles), (unsigned)((a.H + OUT - 1) / OUT));
  if (weights_once(a)) hipLaunchKernelGGL((moe_tile_kernel<DT, 1, 4, 4, 2, 3, kAuxStream, false>), grid, dim3(256), 0, stream, t);
  else hipLaunchKernelGGL((moe_tile_kernel<DT, 1, 4, 4, 2, 3, kAuxKeep, false>), grid, dim3(256), 0, stream, t);
}

}  // namespace

bool moe_tile_fits(const MoeArgs& a, int dtype) {
  const auto ok = [](int64_t bytes) { return bytes >= 0 && bytes < (int64_t)kTileOob; };
  const int64_t M = a.T * a.k, imax = a.I > a.Is ? a.I : a.Is;
  return dtype != kF32 && M < 65536 && ok(a.T * a.sxt * 2 + a.H * 2) && ok(M * imax * 2) && ok(M * a.H * 2) &&
         ok(128 * a.sgi * 2 + a.H * 2) && ok(128 * a.sui * 2 + a.H * 2) && ok(128 * a.sdh * 2 + a.I * 2) &&
         ok(128 * a.shg_i * 2 + a.H * 2) && ok(128 * a.shu_i * 2 + a.H * 2) && ok(128 * a.shd_h * 2 + a.Is * 2) &&
         (a.H + 127) / 128 <= 65535 && (imax + 31) / 32 <= 65535;
}

void launch_moe_tile_gate_up(const MoeArgs& a, int dtype, hipStream_t stream) {
  if (dtype == kBF16) gate_up<kBF16>(a, stream);
  else gate_up<kF16>(a, stream);
}

void launch_moe_tile_down(const MoeArgs& a, int dtype, hipStream_t stream) {
  if (dtype == kBF16) down<kBF16>(a, stream);
  else down<kF16>(a, stream);
}

}  // namespace simsd
