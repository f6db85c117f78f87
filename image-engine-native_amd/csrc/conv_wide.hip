// conv_wide.hip -- 3 x 3 stride-1 convolutions of NHWC f16 maps whose
// channels come in 64s, on gfx950: the general kernel's implicit GEMM
// (conv.hip) with the loads of the reduction kept in flight throughout.
//
// What bounds the general kernel on these shapes is what it fetches and how
// it waits: 128 pixels x 64 channels a workgroup read 10 bytes of L2 a
// KFLOP, 32-channel chunks take half of each 128-byte line of a pixel, and
// every chunk ends in a barrier behind its own loads (MFMA busy 26 % of the
// cycles on 71 x 472, 512 -> 128).  Here a workgroup of 8 waves owns a CU
// and a tile of TR x 32 pixels x BN channels:
//  - the input halo of 64 channels (a whole line a pixel) is staged twice
//    over, the next chunk's pieces requested a tap at a time behind the
//    current one's products;
//  - the weights run through a ring of taps (64 channels x BN, S slots): tap
//    n + S - 1 is requested when tap n starts, so a load has some 1.5 to 3
//    thousand cycles to land;
//  - 4 x 32 x 64 tiles halve a tap's steps between two sets of four waves,
//    whose sums meet in the epilogue's LDS (a wave of 32 pixels x 32 channels
//    would read 2 KiB of LDS a product, past what a CU's LDS gives);
//  - one barrier a tap, which makes the next tap's weights visible, so that
//    every 16-deep step's fragments are read a step ahead, across taps.
// The loads are buffer loads straight into LDS, from inline assembly the
// compiler does not see; each iteration issues the same number of them
// (past the last tap or chunk they are out of range: zeros into a slot that
// nothing reads), so a constant vmcnt covers what a tap needs.  The buffer
// range check gives the zero padding.
//
// Split-K over blockIdx.y in whole 64-channel chunks, counted in per tile as
// in the general kernel (count_in).

#include "conv_common.h"

namespace ien {
namespace {

constexpr int HC = 34;              // halo columns
constexpr int PIXEL = 128;          // bytes of 64 channels
constexpr int OOB = 0x7ffffff0;     // past every buffer (launch checks)

template <int T>
struct Const {
  static constexpr int value = T;
};

// The barrier alone: nothing is written to LDS but by the counted loads.
__device__ __forceinline__ void tap_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

template <int TR, int NW, int KG, int S>
struct WideCfg {
  static constexpr int BN = 64 * NW, MW = 8 / NW / KG, MB = TR / MW;
  static constexpr int HALO = (TR + 2) * HC;
  static constexpr int A_KIB = (HALO * PIXEL + 1023) / 1024;
  static constexpr int PIECES = (A_KIB + 7) / 8;   // halo loads a wave and chunk
  static constexpr int SLOT = 8192 * NW;           // a tap's weights
  static constexpr int B0 = 2 * A_KIB * 1024;
  static constexpr int SP = 72;                    // staged f32 pitch
  static constexpr int STAGE = MB * 32 * SP * 4;   // per wave
  static constexpr int LDS = B0 + S * SLOT > 8 * STAGE ? B0 + S * SLOT : 8 * STAGE;
  static_assert(PIECES <= 8 && S >= 10 - PIECES && S <= 9 && LDS <= 160 * 1024, "budget");
  // Loads issued in an iteration of tap t, and those after tap t + 1's
  // weights when tap t starts (they went out S - 2 iterations ago).
  static constexpr int loads(int t) { return NW + (t < PIECES); }
  static constexpr int pending(int t) {
    int n = ((t + 11 - S) % 9) < PIECES;  // the halo piece behind them
    for (int m = 3 - S; m < 0; m++) n += loads((t + 9 + m) % 9);
    if (t == 8) {  // the next chunk's halo too: its last piece went out at tap PIECES - 1
      const int after = NW * (8 - PIECES);
      n = n < after ? n : after;
    }
    return n;
  }
};

// A doubling transposed convolution (UP): its four output phases' products
// over offset taps in one launch.  Phase p = 2 py + px reads the pixel and,
// where py or px is set, the next one down or across: nine (phase, tap)
// pairs in all, which take the nine taps' places above; the phases' sums stay
// in registers side by side and the halo serves them all.
struct UpWeights {
  const uint16_t *wp[4];
  const float *bias[4];
  int kb[4];  // 16-deep blocks of each matrix
};
constexpr int UP_PHASE[9] = {0, 1, 1, 2, 2, 3, 3, 3, 3}, UP_TAP[9] = {0, 0, 1, 0, 1, 0, 1, 2, 3};
constexpr int UP_DY[9] = {0, 0, 0, 0, 1, 0, 0, 1, 1}, UP_DX[9] = {0, 0, 1, 0, 0, 0, 1, 0, 1};

template <int TR, int NW, int KG, int S, bool UP>
__global__ __launch_bounds__(512, 2) void conv_wide(ConvArgs a, UpWeights up) {
  using Cfg = WideCfg<TR, NW, KG, S>;
  constexpr int MB = Cfg::MB, MW = Cfg::MW, PH = UP ? 4 : 1, P = UP ? 0 : 1;  // phases, halo border
  __shared__ __attribute__((aligned(1024))) unsigned char lds[Cfg::LDS];
  const int bid = xcd_remap(blockIdx.x, gridDim.x);
  const int tpix = a.tiles_x * a.tiles_y;
  const int tn = a.n_major ? bid / tpix : bid % a.tiles_n;
  const int tile = a.n_major ? bid % tpix : bid / a.tiles_n;
  const int ty = tile / a.tiles_x;
  const int oy0 = (ty + a.ty_begin) * TR, ox0 = (tile - ty * a.tiles_x) * 32;
  const int tid = threadIdx.x, lane = tid & 63, hi = lane >> 5, l32 = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int mg = wave % MW, ng = wave / MW % NW, kg = wave / (MW * NW);
  constexpr int KS = 4 / KG;  // 16-deep steps of a tap for each wave
  const int nblk = tn * 2 * NW;  // first 32-channel block of the tile
  const int4v xr = uniform_rsrc(a.x, (long)a.H * a.W * a.xs * 2);
  int4v wr[PH];
#pragma unroll
  for (int q = 0; q < PH; q++)
    wr[q] = UP ? uniform_rsrc(up.wp[q], (long)a.NB * up.kb[q] * 1024)
               : uniform_rsrc(a.wp, (long)a.NB * a.KB * 1024);
  const unsigned l0 = lds_addr(lds);
  const int c_begin = (int)blockIdx.y * a.kchunks;
  const int chunks = min(a.C / 64 - c_begin, a.kchunks);

  // Byte offsets of this lane's 16 bytes of the halo pieces at channel 0:
  // 16-byte slot s of halo pixel p holds channels 8 (s ^ (p / 2 % 8)) ...
  // (A wave's last piece may lie past the halo: it repeats the last KiB.)
  int piece[Cfg::PIECES];
#pragma unroll
  for (int i = 0; i < Cfg::PIECES; i++) {
    const int item = min(wave + 8 * i, Cfg::A_KIB - 1) * 64 + lane, p = item >> 3;
    const int hy = p / HC;
    int iy = oy0 + hy - P, ix = ox0 + p - hy * HC - P;
    bool ok = p < Cfg::HALO;
    if (iy < 0 || iy >= a.H || ix < 0 || ix >= a.W) {
      ok = ok && a.pad_reflect;
      // (Clamped as well: pixels that feed no stored output may lie further
      // out than one reflection reaches.)
      iy = min(max(reflect_idx(iy, a.H), 0), a.H - 1);
      ix = min(max(reflect_idx(ix, a.W), 0), a.W - 1);
    }
    piece[i] = ok ? (iy * a.W + ix) * a.xs * 2 + 16 * ((item & 7) ^ ((p >> 1) & 7)) : OOB;
  }
  // Piece i of chunk c (of this split) into its buffer.
  auto issue_halo = [&](int c, int i) {
    const unsigned base = l0 + (c & 1) * (Cfg::A_KIB * 1024) + min(wave + 8 * i, Cfg::A_KIB - 1) * 1024;
    int off = piece[i];
    if (off != OOB) off += (c_begin + c) * PIXEL;
    dma_lds(xr, __builtin_amdgcn_readfirstlane(base), c < chunks ? off : OOB);
  };
  // Weights of tap t of chunk c: fragments [32-channel block][16-deep step].
  auto issue_weights = [&](int c, int t, int slot) {
    const int q = UP ? UP_PHASE[t] : 0, tap = UP ? UP_TAP[t] : t, kbs = UP ? up.kb[q] : a.KB;
#pragma unroll
    for (int i = 0; i < NW; i++) {
      const int f = wave + 8 * i;
      const int kb = tap * (a.C / 16) + (c_begin + c) * 4 + (f & 3);
      const int off = ((nblk + (f >> 2)) * kbs + kb) * 1024 + lane * 16;
      const unsigned base = l0 + Cfg::B0 + (unsigned)slot * Cfg::SLOT + f * 1024;
      dma_lds(wr[q], __builtin_amdgcn_readfirstlane(base), c < chunks ? off : OOB);
    }
  };

  floatx16 acc[PH][MB][2] = {};
  // The fragments of step s (of this wave's) of tap (c, t): its rows and 64 channels.
  auto frag = [&](int c, int t, int slot, int s, half8 *av, half8 *bv) {
    const int ks = kg * KS + s;
    const unsigned char *ab = lds + (c & 1) * (Cfg::A_KIB * 1024);
    const int dy = UP ? UP_DY[t] : t / 3, dx = UP ? UP_DX[t] : t % 3;
#pragma unroll
    for (int i = 0; i < MB; i++) {
      const int p = (mg * MB + i + dy) * HC + l32 + dx;
      av[i] = *(const half8 *)(ab + p * PIXEL + 16 * ((2 * ks + hi) ^ ((p >> 1) & 7)));
    }
    const unsigned char *bb = lds + Cfg::B0 + slot * Cfg::SLOT + ng * 8192 + lane * 16;
#pragma unroll
    for (int j = 0; j < 2; j++) bv[j] = *(const half8 *)(bb + (4 * j + ks) * 1024);
  };

  // The loads before the first tap, in the order the iterations would have
  // issued them.
#pragma unroll
  for (int m = -9; m < 0; m++) {
    if (m + S - 1 >= 0) issue_weights(0, m + S - 1, m + S - 1);
    if (m + 9 < Cfg::PIECES) issue_halo(0, m + 9);
  }
  wait_vm<Cfg::pending(8)>();
  tap_barrier();
  half8 av[2][MB], bv[2][2];
  frag(0, 0, 0, 0, av[0], bv[0]);
  int slot = 0;
  auto tap = [&](int c, auto tc) {
    constexpr int t = decltype(tc)::value, q = UP ? UP_PHASE[t] : 0;
    wait_vm<Cfg::pending(t)>();
    tap_barrier();  // the next tap (and at tap 8 the next halo) is in; every wave is done with the last one
    issue_weights(c + (t + S - 1) / 9, (t + S - 1) % 9, slot == 0 ? S - 1 : slot - 1);
    if constexpr (t < Cfg::PIECES) issue_halo(c + 1, t);
    const int next = slot + 1 == S ? 0 : slot + 1;
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
      const int now = ks & 1;
      if (ks < KS - 1)
        frag(c, t, slot, ks + 1, av[now ^ 1], bv[now ^ 1]);
      else
        frag(t < 8 ? c : c + 1, (t + 1) % 9, next, 0, av[now ^ 1], bv[now ^ 1]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < MB; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
          acc[q][i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av[now][i], bv[now][j], acc[q][i][j], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    slot = next;
  };
  for (int c = 0; c < chunks; c++) {
    tap(c, Const<0>{});
    tap(c, Const<1>{});
    tap(c, Const<2>{});
    tap(c, Const<3>{});
    tap(c, Const<4>{});
    tap(c, Const<5>{});
    tap(c, Const<6>{});
    tap(c, Const<7>{});
    tap(c, Const<8>{});
  }
  wait_vm<0>();  // (the loads past the end too: the stages reuse their LDS)
  __syncthreads();

  if constexpr (KG == 1 && !UP)
    if (a.ksplit > 1 && !count_in<MB, 2, 512>(a, acc[0], (int *)lds, tid)) return;
  __syncthreads();

  // Epilogue: acc + bias as f32 per wave in LDS, then 16-byte items of 8
  // channels of a pixel: old output, activation, f16, added map.
  float *stage = (float *)(lds + wave % (MW * NW) * Cfg::STAGE);
  constexpr int SP = Cfg::SP, ITEMS = MB * 4 / KG;
  auto put = [&](auto phase, bool add) {
    constexpr int ph = decltype(phase)::value;
    const float *bias = UP ? up.bias[ph] : a.bias;
#pragma unroll
    for (int j = 0; j < 2; j++) {
      const float b = kg == 0 ? bias[(nblk + 2 * ng + j) * 32 + l32] : 0.0f;
#pragma unroll
      for (int i = 0; i < MB; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
          float *s = stage + (i * 32 + 8 * (r >> 2) + 4 * hi + (r & 3)) * SP + j * 32 + l32;
          *s = (add ? acc[ph][i][j][r] + *s : acc[ph][i][j][r]) + b;
        }
    }
  };
  const int n0 = (nblk + 2 * ng) * 32 + 8 * (lane & 7);
  uint16_t *y = (uint16_t *)a.y;
  auto finish = [&](auto phase) {
    constexpr int ph = decltype(phase)::value;
    if constexpr (KG == 1) {
      put(phase, false);
      __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): this wave's LDS writes done
      __builtin_amdgcn_wave_barrier();
    } else {  // the second half of the steps, then the first half and the bias
      if (kg == 1) put(phase, false);
      __syncthreads();
      if (kg == 0) put(phase, true);
      __syncthreads();
    }
    int at[ITEMS];
#pragma unroll
    for (int t = 0; t < ITEMS; t++) {
      const int q = (lane >> 3) + 8 * (KG * t + kg);
      const int oy = oy0 + mg * MB + q / 32, ox = ox0 + (q & 31), p = oy * a.OW + ox;
      const bool ok = oy < a.OH && ox < a.OW && p >= a.p_begin && p < a.p_end && n0 < a.N;
      const int pixel = UP ? (2 * oy + (ph >> 1)) * 2 * a.OW + 2 * ox + (ph & 1) : p - a.p_begin;
      at[t] = ok ? pixel * a.ys + n0 : -1;
    }
    u32x4 old[ITEMS], add[ITEMS];
    if (a.accumulate) {
#pragma unroll
      for (int t = 0; t < ITEMS; t++) old[t] = *(const u32x4 *)(y + max(at[t], 0));
    }
    if (a.add2) {
#pragma unroll
      for (int t = 0; t < ITEMS; t++) add[t] = *(const u32x4 *)(a.add2 + max(at[t], 0));
    }
    auto store = [&](auto actf) {
#pragma unroll
      for (int t = 0; t < ITEMS; t++) {
        if (at[t] < 0) continue;
        const float *s = stage + ((lane >> 3) + 8 * (KG * t + kg)) * SP + 8 * (lane & 7);
        const float4v s0 = *(const float4v *)s, s1 = *(const float4v *)(s + 4);
        float v[8] = {s0[0], s0[1], s0[2], s0[3], s1[0], s1[1], s1[2], s1[3]};
        uint16_t o[8], h[8];
        if (a.accumulate) {
          __builtin_memcpy(h, &old[t], 16);
#pragma unroll
          for (int e = 0; e < 8; e++) v[e] += h2f(h[e]);
        }
#pragma unroll
        for (int e = 0; e < 8; e++) o[e] = f2h(actf(v[e], n0 + e));
        if (a.add2) {
          __builtin_memcpy(h, &add[t], 16);
#pragma unroll
          for (int e = 0; e < 8; e++) o[e] = f2h(h2f(o[e]) + h2f(h[e]));
        }
        __builtin_memcpy(y + at[t], o, 16);
      }
    };
    switch (a.act) {
      case IEN_ACT_RELU: store([](float v, int) { return act_c<IEN_ACT_RELU>(v, 0.0f); }); break;
      case IEN_ACT_GELU: store([](float v, int) { return act_c<IEN_ACT_GELU>(v, 0.0f); }); break;
      case IEN_ACT_SIGMOID: store([](float v, int) { return act_c<IEN_ACT_SIGMOID>(v, 0.0f); }); break;
      case IEN_ACT_PRELU: {
        const float *sl = a.slope;
        store([sl](float v, int n) { return v < 0.0f ? v * sl[n] : v; });
        break;
      }
      default: store([](float v, int) { return v; }); break;
    }
  };
  finish(Const<0>{});
  if constexpr (UP) {  // (a wave's stage is its own: its reads are done when its next writes are)
    finish(Const<1>{});
    finish(Const<2>{});
    finish(Const<3>{});
  }
}

template <int TR, int NW, int KG, int S, bool UP = false>
ien_status launch(ien_ctx *ctx, ConvArgs a, int ksplit, const UpWeights &up = {}) {
  using Cfg = WideCfg<TR, NW, KG, S>;
  a.ty_begin = a.p_begin / a.OW / TR;
  a.tiles_y = (a.p_end - 1) / a.OW / TR + 1 - a.ty_begin;
  a.tiles_x = (a.OW + 31) / 32;
  a.tiles_n = (a.N + Cfg::BN - 1) / Cfg::BN;
  const long tpix = (long)a.tiles_y * a.tiles_x, blocks = tpix * a.tiles_n;
  IEN_CHECK(blocks > 0 && blocks < (1L << 31) && a.tiles_n * 2 * NW <= a.NB, IEN_ERR_INPUT,
            "grid of %ld tiles", blocks);
  // The order of the tiles that fetches fewer bytes a band (as conv.hip).
  const double wb = (double)a.tiles_n * 2 * NW * a.KB * 1024.0, xb = (double)tpix * Cfg::HALO * a.C * 2.0;
  const double by_n = xb * std::max(1.0, 8.0 / tpix) + wb * std::min(8L, tpix);
  const double by_pix = wb * std::max(1.0, 8.0 / a.tiles_n) + xb * std::min(8, a.tiles_n);
  a.n_major = a.tiles_n > 1 && (blocks & 7) == 0 && by_pix < by_n;
  const int chunks = a.C / 64;
  a.kchunks = (chunks + ksplit - 1) / ksplit;
  a.ksplit = (chunks + a.kchunks - 1) / a.kchunks;
  IEN_CHECK(a.ksplit == 1 || (KG == 1 && blocks <= ien_ctx::SPLITK_TILES &&
                              blocks * a.ksplit * Cfg::MB * 16384 <= (long)ctx->splitk_floats),
            IEN_ERR_INPUT, "%ld tiles in %d splits past the workspace", blocks, a.ksplit);
  a.part = ctx->splitk;
  a.tile_count = (int *)(ctx->splitk + ctx->splitk_floats);
  hipLaunchKernelGGL((conv_wide<TR, NW, KG, S, UP>), dim3((unsigned)blocks, (unsigned)a.ksplit), dim3(512), 0,
                     ctx->stream, a, up);
  IEN_HIP(hipGetLastError());
  return IEN_OK;
}

// The tiles, with the microseconds of a round of workgroups: `round` and
// `chunk` a 64-channel chunk.  A CU takes one workgroup at a time, so a
// launch's time goes in whole rounds; a split costs its f32 sums' way
// through memory (at device scope), some 6 us whatever the size.
struct Tile {
  int rows, cols;  // pixels and channels: rows x 32 x cols
  double round, chunk;
  long sums;       // floats of a workgroup's sums (0: not split over workgroups)
};
constexpr Tile TILES[] = {
    {8, 64, 5.5, 2.8, 16384},
    {4, 128, 5.9, 2.65, 16384},
    {8, 128, 8.0, 5.0, 32768},
    {4, 64, 5.7, 1.77, 0},
};
constexpr double SPLIT_US = 6.0;

}  // namespace

// Whole 16-byte groups of f16 NHWC outputs, ranges in 31 bits.  Measured
// against the general kernel on one idle MI355X (us, general -> here; the same
// shape moves by some 3 % from box to box): 85 x 125, 512 -> 128 23.0 -> 19.2
// (4 x 64 tiles; 22.9 as 4 x 128 in 2 splits) and 128 -> 384 19.1 -> 18.3
// (8 x 128); 64 x 96, 256 -> 256 15.0 -> 12.8 and 64 x 64, 128 -> 384 10.1 ->
// 9.3 (4 x 64); 71 x 472, 512 -> 128 60 -> 49 (8 x 128); 200 x 200, 256 -> 256
// 66 -> 63; 95 x 95, 512 -> 256 32 -> 29; and, left to the general kernel's
// deep splits, 64 x 64, 512 -> 128 14.4 against 17.9.  Over 215 sizes of 1 ..
// 400 rows and 4 .. 400 columns, 64 .. 1024 -> 64 .. 512 channels, the choice
// took 0.95 of the general kernel's time in the mean, at worst 1.02 of it.  Not
// compact launches: a workgroup leaves another branch's kernels no LDS.
bool wide_supported(const ien_ctx *ctx, const ConvArgs &a) {
  return a.C % 64 == 0 && a.N % 8 == 0 && a.ys % 8 == 0 && (((uintptr_t)a.y | (uintptr_t)a.add2) & 15) == 0 &&
         !a.out_nchw && !a.out_f32 && !ctx->compact && (long)a.H * a.W * a.xs * 2 <= 0x7fff0000L &&
         (long)a.NB * a.KB * 1024 <= 0x7fff0000L;
}

WidePlan wide_plan(int cus, long workspace, int ow, int c, int n, long p_begin, long p_end) {
  WidePlan best{-1.0, 0, 1};
  const int chunks = c / 64;
  for (int i = 0; i < (int)(sizeof TILES / sizeof TILES[0]); i++) {
    const Tile &t = TILES[i];
    const long blocks = range_tiles(ow, p_begin, p_end, n, t.rows, t.cols);
    for (int s = 1; s <= 4 && s <= chunks; s++) {
      if (s > 1 && (!t.sums || blocks > ien_ctx::SPLITK_TILES || blocks * s * t.sums > workspace)) break;
      const double rounds = (double)((blocks * s + cus - 1) / cus);
      const double us = rounds * (t.round + t.chunk * ((chunks + s - 1) / s)) + (s > 1 ? SPLIT_US : 0.0);
      if (best.us < 0 || us < best.us) best = WidePlan{us, i, s};
    }
  }
  return best;
}

ien_status launch_wide(ien_ctx *ctx, const ConvArgs &a, int tile, int ksplit) {
  switch (tile) {
    case 0: return launch<8, 1, 1, 8>(ctx, a, ksplit);
    case 1: return launch<4, 2, 1, 6>(ctx, a, ksplit);
    case 2: return launch<8, 2, 1, 4>(ctx, a, ksplit);
    default: return launch<4, 1, 2, 8>(ctx, a, 1);
  }
}

// Input bytes up to the padding loads' out-of-range offset, outputs in 31 bits
// of elements: every map that LaMa's first convolution can write at full scale
// (2^31 values of 64 channels) comes up again.
bool conv_up_fits(long h, long w, long c, long n, long ys) {
  return h > 0 && w > 0 && c > 0 && c % 64 == 0 && n > 0 && n % 8 == 0 && ys % 8 == 0 && ys >= n &&
         h * w * c * 2 <= OOB && 4 * h * w * ys < (1L << 31);
}

// LaMa's doublings (1000 x 680 images, us): 85 x 125, 512 -> 256 as four
// launches of the general kernel 108, here 37; 170 x 250, 256 -> 128 109 and
// 48; 340 x 500, 128 -> 64 107 and 62.
ien_status conv_up(ien_ctx *ctx, const uint16_t *x, int h, int w, int c, ien_matrix *const *phases, uint16_t *y,
                   int ys, ien_act act) {
  const int n = (int)phases[0]->n;
  IEN_CHECK(act != IEN_ACT_PRELU, IEN_ERR_INPUT, "a doubling takes no slopes");
  UpWeights up{};
  for (int p = 0; p < 4; p++) {
    const int taps = (1 + p / 2) * (1 + p % 2);
    IEN_CHECK(phases[p]->d_packed && phases[p]->k == (size_t)taps * c && (int)phases[p]->n == n &&
                  (long)phases[p]->nb * phases[p]->kb * 1024 <= 0x7fff0000L,
              IEN_ERR_INPUT, "phase %d of %zu x %zu for %d channels", p, phases[p]->k, phases[p]->n, c);
    up.wp[p] = phases[p]->d_packed;
    up.bias[p] = phases[p]->d_bias;
    up.kb[p] = phases[p]->kb;
  }
  IEN_CHECK(conv_up_fits(h, w, c, n, ys) && (((uintptr_t)x | (uintptr_t)y) & 15) == 0, IEN_ERR_INPUT, "doubling of a %d x %d map, %d -> %d channels", w, h, c, n);
  ConvArgs a{};
  a.x = x;
  a.H = a.OH = h;
  a.W = a.OW = w;
  a.C = a.xs = c;
  a.p_end = h * w;
  a.NB = phases[0]->nb;
  a.KB = phases[3]->kb;
  a.N = n;
  a.y = y;
  a.ys = ys;
  a.act = act;
  return launch<8, 1, 1, 8, true>(ctx, a, 1, up);
}

}  // namespace ien
