// conv_pair.hip -- consecutive 3x3 64 -> 64 convolutions, each with bias
// and PReLU, two per pass over the map: pairs of Real-ESRGAN's body layers
// (crates/realesrgan-native/src/network.rs:96-109; gemm.rs multiply order).
//
// Two kernels.  conv_pair runs one pair on a map of any size in strips
// (below, at the kernel).  conv_chain runs up to 16 pairs in one launch on
// maps whose tiles fit the device at once: a launch per pair spends as long
// on fixed costs (the gap after the previous kernel, the weights landing,
// the last stores draining) as on a small map's products, and a chain pays
// them once.  Every accumulator of either is seeded with the bias and sums
// the 36 steps (9 taps x 16 channels, taps first) in the order of the
// one-layer resident kernel, and the first layer's results are rounded to
// f16 as the map between two launches would hold them, so both give the
// same bits as single-layer launches.
//
// A chain's workgroup of 8 waves (two per SIMD) computes a TR x TC tile of
// each pair's second layer:
//  - The input halo, TR + 4 by TC + 4 pixels of 64 channels, is in LDS
//    (zeros outside the image), each pixel followed by a 16-byte pad chunk
//    and each row by padding, so that the B fragments of packed pixel
//    blocks read LDS without bank conflicts.
//  - Phase 1: the first layer on the TR + 2 by TC + 2 pixels the second one
//    reads, packed row after row into blocks of 32 (each lane addresses its
//    own pixel, so a block may span rows and only the halo itself is
//    computed twice).  Pixels outside the image are stored as zeros: the
//    second layer's zero padding.
//  - Phase 2: the second layer on the TR x TC output pixels.
// Wave w takes the 32 output channels of half w / 4 and the blocks w % 4,
// w % 4 + 4, ...; it holds that half of one layer's packed weights in
// registers (36 fragments, the A operand of v_mfma_f32_32x32x16_f16, so the
// product is C^T = W^T X^T), each layer's loaded once per pair into LDS and
// from there into registers.
//
// All of a chain's workgroups, one per tile, are resident at once (at most
// one per CU).  A tile keeps its pair output in
// LDS as the centre of the next pair's halo and exchanges only the 2-pixel
// ring with its 8 neighbours: after pair k it stores the outer 2 rows and
// columns of its output to border map k % 2 and, once those stores are
// complete, publishes epoch k + 1; pair k + 1 waits until each neighbour's
// epoch reaches k + 1 and loads its ring from that map.  The neighbours may
// run on other XCDs, whose L2 caches are not kept coherent with this one:
// the border stores, the ring loads and the epoch words all use device
// scope (the sc1 cache policy: written through to, and read from, the
// device's point of coherence), so no cache-wide write-back or invalidate
// is needed.  A neighbour only publishes after it has
// read its own ring from the other map, so a border map is never rewritten
// while a reader still needs it.  Every wait is bounded by a wall-clock
// limit; a tile that runs out sets an abort word that every other waiting
// tile sees, so all workgroups end (the run reports the failure).  The last
// pair stores the whole tile.  Each workgroup counts itself out as its last
// act; the last one out returns the epochs, the abort word and the count to
// zero, so the next chain on the stream starts from clear flags without a
// launch of its own for them.

#include "conv_common.h"

namespace ien {
namespace {

constexpr int C = 64;                      // channels in, between and out
constexpr int PB = 2 * C + 16;             // bytes of a staged pixel
constexpr int WBYTES = 2 * (9 * C / 16) * 1024;  // both halves of a layer
constexpr int STEPS = 9 * C / 16;
constexpr int WAVES = 8, THREADS = 64 * WAVES;
constexpr int WLOADS = WBYTES / (1024 * WAVES);  // 1 KiB weight loads per wave
constexpr int MAXPAIRS = 16;
#ifndef IEN_PAIR_PREFETCH
#define IEN_PAIR_PREFETCH 1
#endif
constexpr int PREFETCH = IEN_PAIR_PREFETCH;  // steps a B fragment is loaded ahead of its products
static_assert(WLOADS * 1024 * WAVES == WBYTES, "weight loads");

// A TR x TC output tile.  LDS: the halo, the first layer's results, with
// OWN a buffer for one layer's weights (without: the first layer's weights
// lie where its results go, the second's where the halo was), then the
// biases and slopes of both layers.
template <int TR, int TC, bool OWN_>
struct Geo {
  static constexpr bool OWN = OWN_;
  static constexpr int OTR = TR, OTC = TC;
  static constexpr int MR = OTR + 2, MC = OTC + 2;  // first layer's pixels
  static constexpr int IR = OTR + 4, IC = OTC + 4;  // input halo
  static constexpr int MPIX = MR * MC, OPIX = OTR * OTC;
  static constexpr int MBLK = (MPIX + 31) / 32, OBLK = OPIX / 32;
  static constexpr int INNER = (MR - 4) * (MC - 4);  // first-layer pixels that read no halo ring
  // Blocks of the first layer that read only the halo's centre and come
  // before the ring (whole blocks, whole rounds of the 4 block groups
  // except where there are fewer), and the blocks a wave takes before and
  // after it; the output blocks a wave takes in one sequence of products.
  static constexpr int IBLK = INNER / 32 < 4 ? INNER / 32 : INNER / 32 / 4 * 4;
  static constexpr int PASS0 = (IBLK + 3) / 4, PASS1 = (MBLK - IBLK + 3) / 4;
  static constexpr int OUTN = OBLK / 4 < 2 ? (OBLK + 3) / 4 : 2;
  // Staged rows end with padding, which with 144-byte pixels (16
  // consecutive pixels on disjoint banks) makes a block's step from the
  // last pixel of one of its rows to the first of the next land on the
  // banks of a one-pixel step, so no B-fragment read conflicts even where a
  // block spans rows: the first layer's results are read in rows of OTC (of
  // MC), the halo, interior first, in rows of MC - 4 (of IC).
  static constexpr int MROW = MC * PB + 224;  // bytes a staged row of the first layer's results
  static constexpr int HROW = IC * PB + 160;  // bytes a staged halo row
  static constexpr int HALO = OWN ? (IR * HROW + 1024 * WAVES - 1) / (1024 * WAVES) * (1024 * WAVES)
                                  : IR * HROW;
  static constexpr int MID = HALO;
  static constexpr int MBYTES = OWN ? MR * MROW : std::max(MR * MROW, WBYTES);
  static constexpr int W1AT = OWN ? MID + MBYTES : MID, W2AT = OWN ? W1AT : 0;
  static constexpr int PARAM = OWN ? W1AT + WBYTES : MID + MBYTES;
  // A chain's tail: the final layer's results (f32, over the first layer's)
  // and the tile's image, behind them or in room of its own.
  static constexpr int RES = OPIX * 48 * 4, IMG = OWN ? MID + RES : PARAM + 4 * C * 4;
  static constexpr int LDS = PARAM + 4 * C * 4 + (OWN ? 0 : OPIX * 3 * 4);
  static constexpr int HLOADS = (HALO + 1024 * WAVES - 1) / (1024 * WAVES);  // 1 KiB loads a wave
  static constexpr int RING = (9 * IC + 63) / 64;  // 1 KiB loads of a whole ring row
  static_assert(LDS <= 160 * 1024 && HALO % 16 == 0 && W1AT % 16 == 0, "LDS budget");
  static_assert((MROW - (OTC - 1) * PB) % 256 == PB, "first layer's rows");
  static_assert((HROW - (MC - 5) * PB) % 256 == PB, "halo rows");
  static_assert(HLOADS + WLOADS < 64, "load split");
  static_assert((WAVES - 1 + WAVES * (HLOADS - 2)) * 1024 + 1024 <= HALO, "halo loads before the last");
  static_assert(RES + (OWN ? OPIX * 3 * 4 : 0) <= MBYTES, "the final layer's results");
  static_assert(OWN || WBYTES <= HALO, "second layer's weights in the halo");
  static_assert(MBLK <= 16 && OPIX % 32 == 0 && OBLK <= 12 && PASS0 <= 2 && PASS1 <= 2, "block split");
};

// The first layer's pixel i (of MPIX) in pass order: the INNER pixels that
// read only the halo's centre first (rows 2 .. MR - 3, columns 2 .. MC - 3,
// row-major), then rows 0, 1, then the outer columns 0, 1, MC - 2, MC - 1
// of rows 2 .. MR - 3, then the last two rows.
template <class G>
__device__ __forceinline__ int first_pixel(int i) {
  constexpr int MR = G::MR, MC = G::MC;
  if (i < G::INNER) return (2 + i / (MC - 4)) * MC + 2 + i % (MC - 4);
  i -= G::INNER;
  if (i < 2 * MC) return i;
  i -= 2 * MC;
  if (i < 4 * (MR - 4)) {
    const int c = i & 3;
    return (2 + (i >> 2)) * MC + (c < 2 ? c : c + MC - 4);
  }
  return (MR - 2) * MC + i - 4 * (MR - 4);
}

struct PairArgs {
  const uint16_t *x;  // H x W x 64 f16 input (pixels 64 halves apart)
  uint16_t *y;        // the same shape: the last pair's output
  int H, W, tiles_x, tiles_y;
  int KB;     // fragments along k of each layer (36)
  int pairs;  // 1, or the chain's length
  // Layer 2 k and 2 k + 1 of pair k: packed weights (fragment (kb, nb) at
  // (nb KB + kb) 512 halves), biases and PReLU slopes (64 each).
  const uint16_t *w[2 * MAXPAIRS];
  const float *b[2 * MAXPAIRS], *s[2 * MAXPAIRS];
  // Chain only: the border maps (pair k stores to border[k % 2]); the
  // flags: the abort word, the failure word (raised to this launch's
  // sequence number `seq` when a wait gives up, never lowered, so the host
  // tells which launches failed without clearing it), the count of
  // workgroups done, then the tile epochs (tiles_x tiles_y words); all but
  // the failure word are zero at launch and again at the end; and the
  // wall-clock ticks (100 MHz) a wait for neighbours may take (negative: no
  // wait succeeds, every tile with a neighbour gives up at its first wait --
  // the failure path on demand).
  uint16_t *border[2];
  int *flags;
  int seq;
  long spin_limit;
  // Chain only, optional (wl null: none): a final 3x3 64 -> 48 layer
  // (weights packed with n padded, bias; no activation) whose 48 channels
  // are pixel-shuffled x4 and added to the f32 RGB image (H x W x 3) into
  // out ((4 H) x (4 W) x 3 f32) instead of the last pair storing its map.
  const uint16_t *wl;
  const float *bl;
  const float *image;
  float *out;
  // Chain only, optional (w0 null: none): the first layer, 3x3 over the
  // image's RGB and a zero fourth channel (weights packed with k = 36 in
  // 3 fragments, bias, PReLU slopes), computed by the first pair on its
  // halo from the f32 image instead of reading x.
  const uint16_t *w0;
  const float *b0, *s0;
};

constexpr int OOB = 0x7ffffff0;
constexpr int SC1 = 16;  // cache policy bits of a device-scope buffer access

// dma_lds at device scope (sc1): the load bypasses copies in this XCD's
// caches that another XCD's device-scope stores may have made stale.
__device__ __forceinline__ void dma_lds_device(int4v rsrc, unsigned wave_base, int off) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen sc1 lds"
               :: "s"(wave_base), "v"(off), "s"(rsrc) : "memory", "m0");
}

// What a chain does with a tile, on geometry G: one wave's view.
template <class G>
struct Tile {
  unsigned char *lds;
  unsigned lds0;
  float *par;  // both layers' biases and slopes, in LDS
  int tid, lane, wave, hf, grp;  // channel half, block group
  // Lane l's 16 bytes of fragment (step s, channel half hf): rows 16 s +
  // 8 (l / 32) .. + 7 of output channel 32 hf + l % 32.
  half8 w[STEPS];

  __device__ __forceinline__ Tile(unsigned char *l)
      : lds(l), lds0(lds_addr(l)), par((float *)(l + G::PARAM)), tid(threadIdx.x), lane(tid & 63),
        wave(__builtin_amdgcn_readfirstlane(tid >> 6)), hf(wave >> 2), grp(wave & 3) {}

  // A layer's fragments of both halves, (hf 36 + s) KiB from `at`, once per
  // workgroup.
  __device__ __forceinline__ void stage_weights(const uint16_t *wp, int at) const {
    const int4v wr = buffer_rsrc(wp, WBYTES);
#pragma unroll
    for (int i = 0; i < WLOADS; i++) {
      const int f = wave + WAVES * i;
      dma_lds(wr, __builtin_amdgcn_readfirstlane(lds0 + at + f * 1024), f * 1024 + lane * 16);
    }
  }
  __device__ __forceinline__ void params(const PairArgs &a, int k) const {
    if (tid < C) {
      par[tid] = a.b[2 * k][tid];
      par[C + tid] = a.s[2 * k][tid];
      par[2 * C + tid] = a.b[2 * k + 1][tid];
      par[3 * C + tid] = a.s[2 * k + 1][tid];
    }
  }

  // The accumulators of a block, seeded with the bias: register 4 g + e is
  // channel 32 hf + 8 g + 4 (lane / 32) + e of pixel lane % 32.
  __device__ __forceinline__ floatx16 seed(const float *bias) const {
    floatx16 acc;
#pragma unroll
    for (int g = 0; g < 4; g++) {
      const float4v b4 = *(const float4v *)(bias + 32 * hf + 8 * g + 4 * (lane >> 5));
#pragma unroll
      for (int e = 0; e < 4; e++) acc[4 * g + e] = b4[e];
    }
    return acc;
  }
  // acc[j] += W^T X^T over the 36 steps for NB blocks whose lane bases are
  // base[j] in a staged map of rows ROW bytes apart.  With STREAM the
  // weights come into w from their staging at `wat` in step with the B
  // fragments (the first products after a layer's weights are staged), so
  // that their loads overlap the products instead of preceding them.
  template <int NB, int ROW, bool STREAM>
  __device__ __forceinline__ void products(const int *base, floatx16 *acc, int wat) {
    constexpr int DEPTH = PREFETCH;  // steps the B fragments are loaded ahead
    auto frag = [&](int j, int s) {
      const int tap = s / 4, kc = s % 4;
      return *(const half8 *)(lds + base[j] + (tap / 3) * ROW + (tap % 3) * PB + 32 * kc);
    };
    half8 xv[NB][DEPTH + 1];
#pragma unroll
    for (int s = 0; s < DEPTH; s++) {
      if (STREAM) w[s] = *(const half8 *)(lds + wat + (hf * STEPS + s) * 1024 + lane * 16);
#pragma unroll
      for (int j = 0; j < NB; j++) xv[j][s] = frag(j, s);
    }
#pragma unroll
    for (int s = 0; s < STEPS; s++) {
      if (s + DEPTH < STEPS) {
        if (STREAM)
          w[s + DEPTH] = *(const half8 *)(lds + wat + (hf * STEPS + s + DEPTH) * 1024 + lane * 16);
#pragma unroll
        for (int j = 0; j < NB; j++) xv[j][(s + DEPTH) % (DEPTH + 1)] = frag(j, s + DEPTH);
      }
#pragma unroll
      for (int j = 0; j < NB; j++)
        acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(w[s], xv[j][s % (DEPTH + 1)], acc[j], 0, 0, 0);
      // Keeps each step's loads ahead of the products they feed: left to
      // itself the scheduler sinks them to just before their use, and every
      // product then waits out an LDS round trip.
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  // The PReLU slopes of the lane's 16 channels, the same for every block.
  __device__ __forceinline__ void slopes(const float *slope, float4v *s4) const {
#pragma unroll
    for (int g = 0; g < 4; g++) s4[g] = *(const float4v *)(slope + 32 * hf + 8 * g + 4 * (lane >> 5));
  }
  // Activation and f16 of a block's accumulators, all bits cleared where
  // keep is 0: out[g] holds channels 32 hf + 8 g + 4 (lane / 32) .. + 3 of
  // pixel lane % 32.
  __device__ __forceinline__ void finish(const floatx16 &acc, const float4v *s4, unsigned keep,
                                         uint2 *out) const {
#pragma unroll
    for (int g = 0; g < 4; g++) {
      uint16_t h[4];
#pragma unroll
      for (int e = 0; e < 4; e++) h[e] = f2h(act_c<IEN_ACT_PRELU>(acc[4 * g + e], s4[g][e]));
      __builtin_memcpy(&out[g], h, 8);
      out[g].x &= keep;
      out[g].y &= keep;
    }
  }
  // One pass of phase 1: the first layer on blocks FIRST + grp + 4 j (j <
  // NB) below LIMIT of its pixels in first_pixel order; blocks past that
  // are computed on its final pixel and dropped.  Results to LDS as f16
  // (zeros outside the H x W image whose pixel (y0, x0) is the tile's: the
  // second layer's padding).  With STREAM the layer's weights come from
  // their staging.  after() runs once the products are issued, before the
  // results are stored.
  template <int FIRST, int NB, int LIMIT, bool STREAM, class After>
  __device__ __forceinline__ void first_pass(int y0, int x0, int H, int W, After after) {
    int base[NB], pix[NB];
#pragma unroll
    for (int j = 0; j < NB; j++) {
      const int blk = FIRST + grp + 4 * j, i = 32 * blk + (lane & 31);
      const bool ok = (FIRST + 4 * j + 3 < LIMIT || blk < LIMIT) && i < G::MPIX;
      const int pc = first_pixel<G>(ok ? i : G::MPIX - 1);
      pix[j] = ok ? pc : -1;
      base[j] = (pc / G::MC) * G::HROW + (pc % G::MC) * PB + 16 * (lane >> 5);
    }
    floatx16 acc[NB];
#pragma unroll
    for (int j = 0; j < NB; j++) acc[j] = seed(par);
    products<NB, G::HROW, STREAM>(base, acc, G::W1AT);
    __builtin_amdgcn_sched_barrier(0);
    after();
    float4v s4[4];
    slopes(par + C, s4);
#pragma unroll
    for (int j = 0; j < NB; j++) {
      const int p = pix[j];
      if (p < 0) continue;
      const int gy = y0 - 1 + p / G::MC, gx = x0 - 1 + p % G::MC;
      const bool inside = (unsigned)gy < (unsigned)H && (unsigned)gx < (unsigned)W;
      uint2 o[4];
      finish(acc[j], s4, inside ? ~0u : 0u, o);
#pragma unroll
      for (int g = 0; g < 4; g++) {
        const int ch = 32 * hf + 8 * g + 4 * (lane >> 5);
        *(uint2 *)(lds + G::MID + (p / G::MC) * G::MROW + (p % G::MC) * PB + ch * 2) = o[g];
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  // The products of a wave's output blocks (grp, grp + 4, ...: 32 output
  // pixels q each), seeded with `bias`, on a staged map whose output pixel
  // q's tap (0, 0) is at base_of(q) (rows ROW bytes apart): up to two
  // blocks, then a third, each passed to emit(j, acc) as soon as its
  // products are issued, so that no more than two blocks' accumulators and
  // fragments are live beside the weights; emit is not called for blocks
  // past the last.  The first ones stream the layer's weights from their
  // staging at `wat`; held() then runs, before the first emit.
  template <int ROW, class BaseOf, class Held, class Emit>
  __device__ __forceinline__ void out_blocks(const float *bias, int wat, BaseOf base_of, Held held,
                                             Emit emit) {
    constexpr int N = G::OUTN;
    auto lane_base = [&](int blk) {
      return base_of(32 * (blk < G::OBLK ? blk : G::OBLK - 1) + (lane & 31));
    };
    {
      int base[N];
      floatx16 acc[N];
#pragma unroll
      for (int j = 0; j < N; j++) base[j] = lane_base(grp + 4 * j), acc[j] = seed(bias);
      products<N, ROW, true>(base, acc, wat);
      __builtin_amdgcn_sched_barrier(0);
      held();
#pragma unroll
      for (int j = 0; j < N; j++)
        if (4 * j + 3 < G::OBLK || grp + 4 * j < G::OBLK) emit(j, acc[j]);
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (G::OBLK > 8) {
      static_assert(G::OBLK <= 8 || G::OBLK == 12, "a third block for every group");
      int base[1] = {lane_base(grp + 8)};
      floatx16 acc[1] = {seed(bias)};
      products<1, ROW, false>(base, acc, 0);
      __builtin_amdgcn_sched_barrier(0);
      emit(2, acc[0]);
    }
  }
  // The lane's base of output pixel q in the first layer's results.
  __device__ __forceinline__ int mid_base(int q) const {
    return G::MID + (q / G::OTC) * G::MROW + (q % G::OTC) * PB + 16 * (lane >> 5);
  }
};

// One pair on the whole map, as strips: a workgroup takes MW - 2 columns of
// the output and marches down a segment of rows, R at a time.  Waves 0-3
// are the first layer and waves 4-7 the second (wave w and w + 4 share a
// SIMD), each with a channel half of its layer's weights in registers from
// start to end, so nothing but pixels moves after the start:
//  - input rows come straight into a ring of 4 batches of R rows, requested
//    three batches ahead;
//  - step i: the first layer computes batch i of its rows (y0 - 1 + R i ..)
//    into a ring of 3 batches, the second the R output rows that need no
//    later row than batch i - 1's last (y0 + R (i - 1) - 2 ..);
//  - one barrier a step.  The second layer's waves store a step's results
//    at the start of the next, the first layer's at the end of their own,
//    so that on each SIMD one wave's epilogue runs beside the other's
//    products.
// A wave takes 32 columns of two neighbouring rows: a B fragment of an
// input row serves both (as tap row dy of the upper and dy - 1 of the
// lower), 48 LDS reads for 72 products, each accumulator still summed in
// tap order.  No row is computed twice within a segment.
//
// Bound by the matrix cores: 836 x 836 pixels (103 GFLOP a pair) take 96 us
// a pair, MFMA busy 59 % of the device's SIMD cycles over the launch, its
// start and drain included.  16 x 24 tiles, which stage 144 KiB of weights and
// wait for them and for the halo once a tile, took 130 us there (the whole
// network 2.28 -> 1.64 ms); 12 x 16 tiles with every load overlapped 142.
// B fragments 1, 2, 3, 4 products ahead: 1725, 1655, 1647, 1647 us.
template <int R>
struct Strip {
  static constexpr int MW = 128 / R, OW = MW - 2, IW = MW + 2;  // columns of the two layers, the input
  static constexpr int IROW = IW * PB, MROW = MW * PB;
  static constexpr int IBATCH = R * IROW, IRING = 4, MRING = 3;
  static constexpr int KIBS = (IBATCH + 1023) / 1024;
  static constexpr int LOADS = (KIBS + WAVES - 1) / WAVES;  // a batch's 1 KiB loads a wave
  static constexpr int AHEAD = 3;  // products a B fragment is loaded ahead of
  static constexpr int MID = (IRING * IBATCH + 1023) / 1024 * 1024;
  static constexpr int STAGE = MID + MRING * R * MROW;  // a wave's 64 pixels x 32 channels (second layer)
  static constexpr int PARAM = STAGE + 4 * 4096;
  static constexpr int LDS = PARAM + 4 * C * 4;
  static_assert(R % 2 == 0 && MW % 32 == 0 && LDS <= 160 * 1024, "strip");
  static_assert(LOADS < 64, "vmcnt range");
};

template <int R>
__global__ __launch_bounds__(THREADS) void conv_pair(PairArgs a) {
  using S = Strip<R>;
  __shared__ __attribute__((aligned(1024))) unsigned char lds[S::LDS];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int layer = wave >> 2, hf = (wave >> 1) & 1, part = wave & 1;
  // The wave's 32 columns and two rows of a batch.
  const int col = 32 * (R == 2 ? part : 0) + (lane & 31), row = R == 2 ? 0 : 2 * part;
  const int tile = xcd_remap(blockIdx.x, gridDim.x);
  const int x0 = tile % a.tiles_x * S::OW, seg = tile / a.tiles_x;
  const int y0 = (int)((long)a.H * seg / a.tiles_y), y1 = (int)((long)a.H * (seg + 1) / a.tiles_y);
  const int steps = (y1 - y0 + 2 + R - 1) / R;  // batches of the first layer
  const unsigned lds0 = lds_addr(lds);
  const long map_bytes = (long)a.H * a.W * C * 2;
  const int4v xr = buffer_rsrc(a.x, map_bytes);
  const __amdgpu_buffer_rsrc_t yr =
      __builtin_amdgcn_make_buffer_rsrc(a.y, 0, (int)map_bytes, 0x00020000);

  // Batch b's loads: KiB k of the batch, lane l's 16 bytes: chunk ch of
  // column hx of the batch's row hy (the pad chunk and what lies outside the
  // image read zeros).  Waves without a KiB of their own repeat the last, so
  // that each has the same number of loads in flight.
  auto load_batch = [&](int b) {
    const int gy0 = y0 - 2 + R * b;
#pragma unroll
    for (int i = 0; i < S::LOADS; i++) {
      const int k = std::min(wave + WAVES * i, S::KIBS - 1);
      const int byte = k * 1024 + lane * 16;
      const int hy = byte / S::IROW, within = byte - hy * S::IROW;
      const int hx = within / PB, ch = (within - hx * PB) >> 4;
      const int gy = gy0 + hy, gx = x0 - 2 + hx;
      const bool ok = b <= steps && hy < R && ch < 8 && (unsigned)gy < (unsigned)a.H &&
                      (unsigned)gx < (unsigned)a.W;
      if (byte < S::IBATCH)
        dma_lds(xr, __builtin_amdgcn_readfirstlane(lds0 + (b % S::IRING) * S::IBATCH + k * 1024),
                ok ? ((gy * a.W + gx) * C + 8 * ch) * 2 : OOB);
    }
  };
  load_batch(0);
  load_batch(1);
  load_batch(2);

  // Lane l's 16 bytes of fragment (step s, channel half hf): rows 16 s +
  // 8 (l / 32) .. + 7 of output channel 32 hf + l % 32.
  half8 w[STEPS];
  {
    const half8 *wp = (const half8 *)(a.w[layer] + (size_t)hf * STEPS * 512) + lane;
#pragma unroll
    for (int s = 0; s < STEPS; s++) w[s] = wp[s * 64];
  }
  float *par = (float *)(lds + S::PARAM);
  if (tid < C) {
    par[tid] = a.b[0][tid];
    par[C + tid] = a.s[0][tid];
    par[2 * C + tid] = a.b[1][tid];
    par[3 * C + tid] = a.s[1][tid];
  }
#pragma unroll
  for (int s = 0; s < STEPS; s++) asm volatile("" : "+v"(w[s]));  // loaded here, once
  const float *bias = par + 2 * C * layer + 32 * hf + 4 * (lane >> 5), *slope = bias + C;

  floatx16 acc[2];
  // acc[j] (row `row` + j of the wave's batch) = bias + W^T X^T, the staged
  // rows it reads being rows base[0 .. 3] (LDS addresses of the lane's
  // pixel at tap column 0).
  auto products = [&](const int *base) {
#pragma unroll
    for (int g = 0; g < 4; g++) {
      const float4v b4 = *(const float4v *)(bias + 8 * g);
#pragma unroll
      for (int e = 0; e < 4; e++) acc[0][4 * g + e] = acc[1][4 * g + e] = b4[e];
    }
    constexpr int N = 4 * 12;  // fragments: 4 rows x 3 tap columns x 4 channel steps
    auto frag = [&](int n) {
      return *(const half8 *)(lds + base[n / 12] + n % 12 / 4 * PB + n % 4 * 32);
    };
    half8 xv[S::AHEAD + 1];
#pragma unroll
    for (int n = 0; n < S::AHEAD; n++) xv[n] = frag(n);
#pragma unroll
    for (int n = 0; n < N; n++) {
      if (n + S::AHEAD < N) xv[(n + S::AHEAD) % (S::AHEAD + 1)] = frag(n + S::AHEAD);
      const half8 x = xv[n % (S::AHEAD + 1)];
      if (n < 36) acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(w[n], x, acc[0], 0, 0, 0);
      if (n >= 12) acc[1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(w[n - 12], x, acc[1], 0, 0, 0);
      // Keeps each step's loads ahead of the products they feed: left to
      // itself the scheduler sinks them to just before their use.
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // PReLU and f16 of acc[j], all bits cleared where keep is 0: out[g] holds
  // channels 32 hf + 8 g + 4 (lane / 32) .. + 3 of the lane's pixel.
  auto finish = [&](int j, unsigned keep, uint2 *out) {
#pragma unroll
    for (int g = 0; g < 4; g++) {
      const float4v s4 = *(const float4v *)(slope + 8 * g);
      uint16_t h[4];
#pragma unroll
      for (int e = 0; e < 4; e++) h[e] = f2h(act_c<IEN_ACT_PRELU>(acc[j][4 * g + e], s4[e]));
      __builtin_memcpy(&out[g], h, 8);
      out[g].x &= keep;
      out[g].y &= keep;
    }
  };

  const int lane_at = col * PB + 16 * (lane >> 5);
  wait_vm<S::LOADS>();  // batches 0 and 1 (and the weights)
  if (layer == 0) {
    const int gx = x0 - 1 + col;
    const unsigned in_col = (unsigned)gx < (unsigned)a.W ? ~0u : 0u;
    for (int i = 0; i <= steps; i++) {
      lds_barrier();
      load_batch(i + 3);
      if (i < steps) {
        int base[4];
#pragma unroll
        for (int n = 0; n < 4; n++)
          base[n] = (R * i + row + n) % (S::IRING * R) * S::IROW + lane_at;
        products(base);
#pragma unroll
        for (int j = 0; j < 2; j++) {
          const int gy = y0 - 1 + R * i + row + j;
          uint2 o[4];
          finish(j, (unsigned)gy < (unsigned)a.H ? in_col : 0u, o);
          unsigned char *d = lds + S::MID + (R * i + row + j) % (S::MRING * R) * S::MROW + col * PB +
                             (32 * hf + 4 * (lane >> 5)) * 2;
#pragma unroll
          for (int g = 0; g < 4; g++) *(uint2 *)(d + 16 * g) = o[g];
        }
      }
      wait_vm<S::LOADS>();  // all but this step's loads
    }
  } else {
    // Staged pixel wp = 32 j + l % 32 holds its 4 chunks of 8 channels at
    // chunk c ^ (wp / 4 % 4), which keeps both the writes (16 pixels, one
    // chunk) and the reads (4 pixels, 4 chunks) free of bank conflicts; a
    // lane then stores 16 bytes and 4 lanes a pixel's 64 contiguous bytes.
    unsigned char *stage = lds + S::STAGE + (wave - 4) * 4096;
    // The results of the products of step i - 1: output rows from r0 + row.
    auto emit = [&](int r0) {
#pragma unroll
      for (int j = 0; j < 2; j++) {
        uint2 o[4];
        finish(j, ~0u, o);
        const int wp = 32 * j + (lane & 31);
#pragma unroll
        for (int pr = 0; pr < 2; pr++) {
          // Lanes < 32 hold channels 16 pr + 0..3 (o[2 pr]) and 16 pr +
          // 8..11 (o[2 pr + 1]), lanes >= 32 the runs 4 above; swapping the
          // upper half's o[2 pr] with the lower half's o[2 pr + 1] gives
          // lane l < 32 channels 16 pr + 0..7 and lane l + 32 channels
          // 16 pr + 8..15.
          const auto sx = __builtin_amdgcn_permlane32_swap(o[2 * pr].x, o[2 * pr + 1].x, false, false);
          const auto sy = __builtin_amdgcn_permlane32_swap(o[2 * pr].y, o[2 * pr + 1].y, false, false);
          const uint4 v = {sx[0], sy[0], sx[1], sy[1]};
          const int c = 2 * pr + (lane >> 5);
          *(uint4 *)(stage + wp * 64 + 16 * (c ^ ((wp >> 2) & 3))) = v;
        }
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
      for (int n = 0; n < 4; n++) {
        const int v = lane + 64 * n, wp = v >> 2, c = v & 3;
        const u32x4 d = *(const u32x4 *)(stage + wp * 64 + 16 * (c ^ ((wp >> 2) & 3)));
        const int gy = r0 + row + (wp >> 5), oc = col - (lane & 31) + (wp & 31), gx = x0 + oc;
        const bool ok = gy >= y0 && gy < y1 && oc < S::OW && gx < a.W;
        __builtin_amdgcn_raw_buffer_store_b128(d, yr, ok ? (gy * a.W + gx) * C * 2 + 64 * hf + 16 * c : OOB,
                                               0, 0);
      }
    };
    for (int i = 0; i <= steps; i++) {
      lds_barrier();
      if (i >= 2) emit(y0 + R * (i - 2) - 2);
      load_batch(i + 3);
      if (i >= 1) {
        // Output row y0 + R (i - 1) - 2 + row + j reads the first layer's
        // rows numbered R (i - 1) - 2 + row + j .. + 2 from its first one.
        int base[4];
#pragma unroll
        for (int n = 0; n < 4; n++)
          base[n] = S::MID + (R * (i - 1) - 2 + S::MRING * R + row + n) % (S::MRING * R) * S::MROW + lane_at;
        products(base);
      }
      wait_vm<S::LOADS>();  // all but this step's loads
    }
    emit(y0 + R * (steps - 1) - 2);
  }
}

template <class G>
__global__ __launch_bounds__(THREADS) void conv_chain(PairArgs a) {
  constexpr int OTR = G::OTR, OTC = G::OTC, IR = G::IR, IC = G::IC, HROW = G::HROW;
  __shared__ __attribute__((aligned(1024))) unsigned char lds[G::LDS];
  __shared__ int go;  // 1 when every neighbour is ready
  Tile<G> t(lds);
  float *par = t.par;
  const int tid = t.tid, lane = t.lane, wave = t.wave, hf = t.hf, grp = t.grp;
  const int tile = xcd_remap(blockIdx.x, gridDim.x);
  const int ty = tile / a.tiles_x, tx = tile % a.tiles_x;
  const int y0 = ty * OTR, x0 = tx * OTC;
  const unsigned lds0 = t.lds0;
  const long map_bytes = (long)a.H * a.W * C * 2;

  // Global offset of chunk ch (8 channels) of halo pixel (hy, hx), or OOB
  // for the pad chunk and pixels outside the image.
  auto halo_src = [&](int hy, int hx, int ch) {
    const int gy = y0 - 2 + hy, gx = x0 - 2 + hx;
    const bool ok = hy < IR && hx < IC && ch < 8 && (unsigned)gy < (unsigned)a.H &&
                    (unsigned)gx < (unsigned)a.W;
    return ok ? ((gy * a.W + gx) * C + 8 * ch) * 2 : OOB;
  };

  // First pair with a first layer: the first layer's outputs on the whole
  // halo, from the image patch around it (two more rows and columns of f16
  // RGB and a zero fourth channel) and the layer's 6 fragments, both
  // staged in MID; as the separate 4-channel kernel computes them (one
  // v_mfma_f32_32x32x16_f16 step covers 4 taps of 4 channels, lane half h
  // reading taps 4 s + 2 h and 4 s + 2 h + 1; taps 9 .. 11 read tap 0
  // against zero weights), PReLU, zeros outside the image.
  constexpr int PR = IR + 2, PC = IC + 2;  // the patch
  auto first_layer = [&]() {
    for (int i = tid; i < PR * PC; i += THREADS) {
      const int gy = y0 - 3 + i / PC, gx = x0 - 3 + i % PC;
      uint16_t h[4] = {0, 0, 0, 0};
      if ((unsigned)gy < (unsigned)a.H && (unsigned)gx < (unsigned)a.W) {
        const float *im = a.image + ((long)gy * a.W + gx) * 3;
        h[0] = f2h(im[0]);
        h[1] = f2h(im[1]);
        h[2] = f2h(im[2]);
      }
      uint2 v;
      __builtin_memcpy(&v, h, 8);
      *(uint2 *)(lds + G::MID + i * 8) = v;
    }
    constexpr int W0AT = (G::MID + PR * PC * 8 + 15) / 16 * 16;  // the fragments after the patch
    static_assert(W0AT + 6 * 1024 <= G::MID + G::MBYTES, "patch");
    if (wave < 6) {
      const int4v w0r = buffer_rsrc(a.w0, 6 * 1024);
      dma_lds(w0r, __builtin_amdgcn_readfirstlane(lds0 + W0AT + wave * 1024), wave * 1024 + lane * 16);
    }
    if (tid < C) {
      par[tid] = a.b0[tid];
      par[C + tid] = a.s0[tid];
    }
    wait_vm<0>();
    __syncthreads();
    half8 w0[3];
#pragma unroll
    for (int s = 0; s < 3; s++) w0[s] = *(const half8 *)(lds + W0AT + (hf * 3 + s) * 1024 + lane * 16);
    float4v s4[4];
    t.slopes(par + C, s4);
    auto tap = [](int t) { return t < 9 ? ((t / 3) * PC + t % 3) * 8 : 0; };
    for (int blk = grp; blk * 32 < IR * IC; blk += 4) {
      const int p = 32 * blk + (lane & 31), pc = p < IR * IC ? p : IR * IC - 1;
      const int hy = pc / IC, hx = pc % IC;
      const unsigned char *pb = lds + G::MID + (hy * PC + hx) * 8;
      floatx16 acc = t.seed(par);
#pragma unroll
      for (int s = 0; s < 3; s++) {
        const int t0 = 4 * s + 2 * (lane >> 5);
        typedef unsigned u32x2v __attribute__((ext_vector_type(2)));
        const u32x2v q0 = *(const u32x2v *)(pb + tap(t0)), q1 = *(const u32x2v *)(pb + tap(t0 + 1));
        const u32x4 raw = {q0[0], q0[1], q1[0], q1[1]};
        half8 xb;
        __builtin_memcpy(&xb, &raw, 16);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(w0[s], xb, acc, 0, 0, 0);
      }
      if (p >= IR * IC) continue;
      const int gy = y0 - 2 + hy, gx = x0 - 2 + hx;
      const bool inside = (unsigned)gy < (unsigned)a.H && (unsigned)gx < (unsigned)a.W;
      uint2 o[4];
      t.finish(acc, s4, inside ? ~0u : 0u, o);
#pragma unroll
      for (int g = 0; g < 4; g++) {
        const int ch = 32 * hf + 8 * g + 4 * (lane >> 5);
        *(uint2 *)(lds + hy * HROW + hx * PB + ch * 2) = o[g];
      }
    }
    __syncthreads();  // the halo is complete; MID and the parameters are free
  };

  int *abort_word = a.flags;
  int *epochs = a.flags + 3;
  // The workgroup's last act on every way out.  Only wave 0 writes
  // the flags (the epoch stores, the abort and failure words); every wave
  // reads the epochs and the abort word, always before the barrier that
  // ends a ring wait, so once wave 0 counts the workgroup out no access of
  // it to the flags remains.  The count's release orders wave 0's flag
  // stores before it, and the workgroup that brings it to the grid size
  // (every other one has left) clears the flags.
  auto leave = [&]() {
    if (wave != 0) return;
    int done = 0;
    if (lane == 0)
      done = __hip_atomic_fetch_add(a.flags + 2, 1, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
    done = __builtin_amdgcn_readfirstlane(done);
    if (done != (int)gridDim.x - 1) return;
    for (int i = lane; i < (int)gridDim.x; i += 64)
      __hip_atomic_store(epochs + i, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (lane == 0) {
      __hip_atomic_store(abort_word, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(a.flags + 2, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  };
  const int pairs = a.pairs;
  // Lane n < 9 (n != 4) of a wave watches neighbour (ty + n / 3 - 1,
  // tx + n % 3 - 1): its epoch word, or null where there is none.
  auto neighbour = [&]() -> const int * {
    if (lane < 9 && lane != 4) {
      const int ny = ty + lane / 3 - 1, nx = tx + lane % 3 - 1;
      if (ny >= 0 && ny < a.tiles_y && nx >= 0 && nx < a.tiles_x) return epochs + ny * a.tiles_x + nx;
    }
    return nullptr;
  };
  // This wave's share of the loads of the halo's 2-pixel ring from
  // the neighbours' border map (k - 1) % 2, at device scope.  A load fills
  // one contiguous KiB of LDS, 16 bytes a lane: staged chunk q of a run of
  // pixels is chunk q % 9 of pixel q / 9 (chunk 8, the pad, and pixels
  // outside the image read zeros).
  auto ring_loads = [&](int k) {
    // The lane index through an opaque move: the offsets below are then
    // computed where they are used rather than kept live (or spilled) from
    // the kernel's start, so that no spill reload, whose wait would also
    // wait for every load in flight, lands between these loads.
    int lane;
    asm volatile("v_mov_b32 %0, %1" : "=v"(lane) : "v"(tid & 63));
    const int4v rr = buffer_rsrc(a.border[(k - 1) & 1], map_bytes);
    auto src = [&](int gy, int gx, int c) {
      const bool ok = c < 8 && (unsigned)gx < (unsigned)a.W && (unsigned)gy < (unsigned)a.H;
      return ok ? ((gy * a.W + gx) * C + 8 * c) * 2 : OOB;
    };
    // The first and last two halo rows whole: 9 chunks a pixel, RING loads
    // a row (lanes past a row's pixels write zeros into its padding, or
    // nothing where they would pass it).
    for (int i = wave; i < 4 * G::RING; i += WAVES) {
      const int r = i / G::RING, part = i - r * G::RING, hy = r < 2 ? r : r + IR - 4;
      const int q = 64 * part + lane, p = (int)((unsigned)q / 9u);
      if (G::RING * 1024 <= HROW || q < 9 * IC)
        dma_lds_device(rr, __builtin_amdgcn_readfirstlane(lds0 + hy * HROW + part * 1024),
                       q < 9 * IC ? src(y0 - 2 + hy, x0 - 2 + p, q - 9 * p) : OOB);
    }
    // The outer two pixels of the rows between: 18 chunks (lanes 0 .. 17) a load.
    for (int i = wave; i < 2 * (IR - 4); i += WAVES) {
      const int hy = 2 + (i >> 1), hx0 = (i & 1) ? IC - 2 : 0;
      const int p = lane >= 9 ? 1 : 0;
      if (lane < 18)
        dma_lds_device(rr, __builtin_amdgcn_readfirstlane(lds0 + hy * HROW + hx0 * PB),
                       src(y0 - 2 + hy, x0 - 2 + hx0 + p, lane - 9 * p));
    }
  };
  // The ring of pair k.  Each wave waits for its neighbours' epoch k
  // (lane n for neighbour n) and issues its share of the loads, then waits
  // for them; the barrier follows.  False when a wait gave up: wave 0 then
  // raises the abort word (which every waiting tile watches) and the
  // failure word.
  auto ring = [&](int k) {
    bool fail = false;
    if (const int *f = neighbour()) {
      const unsigned long long t0 = wall_clock64();
      while (a.spin_limit < 0 ||
             __hip_atomic_load(f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < k) {
        if (__hip_atomic_load(abort_word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0 ||
            (long)(wall_clock64() - t0) > a.spin_limit) {
          fail = true;
          break;
        }
        __builtin_amdgcn_s_sleep(1);
      }
    }
    if (__builtin_amdgcn_ballot_w64(fail) != 0) {
      if (lane == 0) go = 0;
    } else {
      ring_loads(k);
    }
    wait_vm<0>();
    __syncthreads();
    if (go != 0) return true;
    if (tid == 0) {
      __hip_atomic_store(abort_word, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_fetch_max(abort_word + 1, a.seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    return false;
  };
  if (tid == 0) go = 1;  // (seen after the first pair's opening barrier)
  // The tile's image rows (OTC pixels x RGB each), which the final layer
  // adds; rows past the image read zeros.
  auto load_image = [&]() {
    const int4v ir = buffer_rsrc(a.image, (long)a.H * a.W * 12);
    const unsigned i0 = lds0 + G::IMG;
    constexpr int PARTS = (OTC * 3 + 63) / 64;
    for (int i = wave; i < PARTS * OTR; i += WAVES) {
      const int r = i / PARTS, part = i % PARTS, e = 64 * part + lane;
      if (e < OTC * 3)
        dma_lds4(ir, __builtin_amdgcn_readfirstlane(i0 + (r * OTC * 3 + 64 * part) * 4),
                 y0 + r < a.H ? (((y0 + r) * a.W + x0) * 3 + e) * 4 : OOB);
    }
  };
  if (!G::OWN && a.wl) load_image();  // (the first pair's waits cover it)
  if (G::OWN) t.stage_weights(a.w[0], G::W1AT);  // (their buffer is no one else's)
  for (int k = 0; k < pairs; k++) {
    // ---- the first layer's weights and, for the first pair, the whole
    // halo from the input; later pairs find the weights staged and the
    // halo's centre left in LDS by the pair before ----
    if (k == 0 && a.w0) {
      first_layer();
      if (!G::OWN) t.stage_weights(a.w[0], G::W1AT);
    } else if (k == 0) {
      if (!G::OWN) t.stage_weights(a.w[0], G::W1AT);
      // KiB g of the halo: lane l's 16 bytes belong to halo row hy, pixel
      // hx, chunk ch (chunk 8 and the row padding read zeros, as do
      // offsets past the input); lanes past the halo's end load nothing.
      const int4v xr = buffer_rsrc(a.x, map_bytes);
#pragma unroll
      for (int i = 0; i < G::HLOADS; i++) {
        const int g = wave + WAVES * i, byte = g * 1024 + lane * 16;
        const int hy = byte / HROW, within = byte - hy * HROW;
        const int hx = within / PB, ch = (within - hx * PB) >> 4;
        if (i < G::HLOADS - 1 || byte < G::HALO)  // only the last KiB runs past the halo
          dma_lds(xr, __builtin_amdgcn_readfirstlane(lds0 + g * 1024), halo_src(hy, hx, ch));
      }
    }
    t.params(a, k);
    wait_vm<0>();  // (later pairs: also the previous border stores)
    __syncthreads();
    if (k > 0 && tid == 0)  // publish epoch k: this tile's pair k - 1 border is out
      __hip_atomic_store(epochs + tile, k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);

    // ---- phase 1: the first layer on its pixels in two passes; the first
    // reads only the halo's centre, and the ring comes in between them.
    // Pass 0 streams the layer's weights, so that behind it every wave
    // holds them ----
    t.template first_pass<0, G::PASS0, G::IBLK, true>(y0, x0, a.H, a.W, [&] {
      __syncthreads();  // every wave holds its weights: their staging is free
      if (G::OWN) t.stage_weights(a.w[2 * k + 1], G::W2AT);
    });
    if (k > 0 && !ring(k)) {  // (it waited for every load of this workgroup)
      leave();
      return;
    }
    // ---- and, without a buffer of their own, the second layer's weights
    // staged where the halo was ----
    t.template first_pass<G::IBLK, G::PASS1, G::MBLK, false>(y0, x0, a.H, a.W, [&] {
      if (G::OWN) return;
      __syncthreads();  // every wave is done with the halo
      t.stage_weights(a.w[2 * k + 1], G::W2AT);
    });
    wait_vm<0>();
    __syncthreads();  // the first layer's results complete, the weights staged

    // ---- phase 2: the second layer on the tile's outputs, which become
    // the centre of the next pair's halo (zeros outside the image: its
    // padding) ----
    float4v s4[4];
    t.slopes(par + 3 * C, s4);
    {
      const bool last = k == pairs - 1 && !a.wl;  // (a final layer follows the last pair)
      const __amdgpu_buffer_rsrc_t br =
          __builtin_amdgcn_make_buffer_rsrc(a.border[k & 1], 0, (int)map_bytes, 0x00020000);
      t.template out_blocks<G::MROW>(
          par + 2 * C, G::W2AT, [&](int q) { return t.mid_base(q); },
          [&] {
            if (!G::OWN) __syncthreads();  // every wave holds its weights: the halo may be written
          },
          [&](int j, const floatx16 &acc) {
            const int q = 32 * (grp + 4 * j) + (lane & 31), r = q / OTC, col = q % OTC;
            const bool inside = y0 + r < a.H && x0 + col < a.W;
            uint2 o[4];
            t.finish(acc, s4, inside ? ~0u : 0u, o);
#pragma unroll
            for (int g = 0; g < 4; g++) {
              const int ch = 32 * hf + 8 * g + 4 * (lane >> 5);
              *(uint2 *)(lds + (2 + r) * HROW + (2 + col) * PB + ch * 2) = o[g];
            }
          });
      __syncthreads();  // the centre is complete; the first layer's results are read
      if (last) {
        // The whole tile out, 16 bytes a lane (8 lanes a pixel).
        const __amdgpu_buffer_rsrc_t yr =
            __builtin_amdgcn_make_buffer_rsrc(a.y, 0, (int)map_bytes, 0x00020000);
        for (int v = tid; v < G::OPIX * 8; v += THREADS) {
          const int c = v & 7, b = v >> 3, r = b / OTC, col = b % OTC;
          const uint4 d = *(const uint4 *)(lds + (2 + r) * HROW + (2 + col) * PB + 16 * c);
          const int gy = y0 + r, gx = x0 + col;
          typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
          const u32x4 dv = {d.x, d.y, d.z, d.w};
          __builtin_amdgcn_raw_buffer_store_b128(
              dv, yr, gy < a.H && gx < a.W ? (gy * a.W + gx) * C * 2 + 16 * c : OOB, 0, 0);
        }
      } else {
        // The pixels of the outer 2 rows and columns, which the
        // neighbours read, to border map k % 2 at device scope, with the
        // next pair's first weights staged behind them
        // (their completion, and so the epoch, is awaited at the next
        // pair's start).  (Stored straight from the registers during phase
        // 2 instead, they cost more than this pass.)
        // All of a thread's chunks are read from LDS before any is stored.
        constexpr int CHUNKS = (4 * OTC + 4 * (OTR - 4)) * 8;
        constexpr int PER = (CHUNKS + THREADS - 1) / THREADS;
        typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
        u32x4 dv[PER];
        int at[PER];
#pragma unroll
        for (int i = 0; i < PER; i++) {
          const int v = tid + THREADS * i, vc = v < CHUNKS ? v : CHUNKS - 1;
          const int c = vc & 7, b = vc >> 3;
          int r, col;
          if (b < 4 * OTC) {
            r = b / OTC;
            r = r < 2 ? r : r + OTR - 4;
            col = b % OTC;
          } else {
            r = 2 + ((b - 4 * OTC) >> 2);
            col = (b - 4 * OTC) & 3;
            col = col < 2 ? col : col + OTC - 4;
          }
          const uint4 d = *(const uint4 *)(lds + (2 + r) * HROW + (2 + col) * PB + 16 * c);
          dv[i] = u32x4{d.x, d.y, d.z, d.w};
          const int gy = y0 + r, gx = x0 + col;
          at[i] = v < CHUNKS && gy < a.H && gx < a.W ? (gy * a.W + gx) * C * 2 + 16 * c : OOB;
        }
#pragma unroll
        for (int i = 0; i < PER; i++) __builtin_amdgcn_raw_buffer_store_b128(dv[i], br, at[i], 0, SC1);
        t.stage_weights(k + 1 < pairs ? a.w[2 * k + 2] : a.wl, G::W1AT);
      }
    }
  }

  {
    if (!a.wl) {
      leave();
      return;
    }
    // ---- the final layer on the tile, read from the halo (its
    // 1-pixel ring inside the 2-pixel one), no activation; then the pixel
    // shuffle x4 plus the image, as f32 RGB ----
    const int k = pairs;
    if (G::OWN) load_image();
    if (tid < C) par[tid] = a.bl[tid];  // zero past channel 48
    wait_vm<0>();  // the last border stores
    __syncthreads();
    if (tid == 0) __hip_atomic_store(epochs + tile, k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (!ring(k)) {
      leave();
      return;
    }
    // Results [pixel][48] in MID, rounded through f16 as the last layer's
    // map between separate launches holds them, so that the chain's output
    // is bit for bit that of the separate launches.
    float *res = (float *)(lds + G::MID);
    const float *img = (const float *)(lds + G::IMG);
    auto r16 = [](float v) { return h2f(f2h(v)); };
    t.template out_blocks<HROW>(
        par, G::W1AT,
        [&](int q) { return (1 + q / OTC) * HROW + (1 + q % OTC) * PB + 16 * (lane >> 5); },
        [&] {
          if (!G::OWN) __syncthreads();  // every wave holds its weights: MID may take the results
        },
        [&](int j, const floatx16 &acc) {
          const int q = 32 * (grp + 4 * j) + (lane & 31);
#pragma unroll
          for (int g = 0; g < 4; g++) {
            const int ch = 32 * hf + 8 * g + 4 * (lane >> 5);
            if (ch < 48)
              *(float4v *)(res + q * 48 + ch) = float4v{r16(acc[4 * g]), r16(acc[4 * g + 1]),
                                                        r16(acc[4 * g + 2]), r16(acc[4 * g + 3])};
          }
        });
    __syncthreads();
    // Output row 4 r + i (r < OTR) of the tile holds 4 OTC pixels x RGB:
    // chunks of 4 floats, three per input pixel; float f of chunk q is
    // output pixel 4 x + j (x = f / 12, j = f / 3 % 4), colour c = f % 3:
    // channel 16 c + 4 i + j of input pixel (r, x) plus the image's colour c.
    const long ow = 4L * a.W;
    for (int v = tid; v < 4 * OTR * 3 * OTC; v += THREADS) {
      const int row = v / (3 * OTC), q = v - row * (3 * OTC);
      const int r = row >> 2, i = row & 3, x = q / 3;
      const int gy = y0 + r, gx = x0 + x;
      if (gy >= a.H || gx >= a.W) continue;
      const float *px = res + (r * OTC + x) * 48;
      const float *im = img + (r * OTC + x) * 3;
      float o[4];
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int f = 4 * q + e - 12 * x, j = f / 3, c = f - 3 * j;
        o[e] = px[16 * c + 4 * i + j] + im[c];
      }
      *(float4v *)(a.out + ((4L * gy + i) * ow + 4L * x0) * 3 + 4 * q) = float4v{o[0], o[1], o[2], o[3]};
    }
    leave();
  }
}

bool layer_ok(const ien_matrix *m, const float *slope) {
  return m && m->k == 9 * C && m->n == C && m->kb == STEPS && m->nb >= 2 && m->d_packed &&
         m->d_bias && slope;
}

bool maps_ok(const uint16_t *x, const uint16_t *y, int H, int W) {
  const long bytes = (long)H * W * C * 2;
  const uintptr_t xa = (uintptr_t)x, ya = (uintptr_t)y;
  return H > 0 && W > 0 && bytes <= 0x7fff0000L && ((xa | ya) & 15) == 0 &&
         (xa + bytes <= ya || ya + bytes <= xa);
}

void fill_layers(PairArgs &a, const ien_matrix *const *w, const float *const *s, int layers) {
  for (int i = 0; i < layers; i++) {
    a.w[i] = w[i]->d_packed;
    a.b[i] = w[i]->d_bias;
    a.s[i] = s[i];
  }
  a.KB = w[0]->kb;
}

// How a pair's map is cut: strips of Strip<R>::OW columns by segments of
// rows.  A step of any strip takes the same time, a workgroup needs one for
// each R rows of its segment and the two above and below, one more for the
// second layer and about two to start; of all cuts the one with the least
// time in rounds of a workgroup a CU.
struct PairCut {
  int rows = 0, strips = 0, segments = 0;
  long cost = 0;
};
PairCut pair_cut(int H, int W, int cus) {
  PairCut best;
  for (int R : {2, 4}) {
    const int ow = 128 / R - 2, strips = (W + ow - 1) / ow;
    for (int fill = 1; fill <= 4; fill++) {  // as many segments as `fill` rounds hold
      const int segments = std::min(H, std::max(1, fill * cus / strips));
      const long rounds = ((long)strips * segments + cus - 1) / cus;
      const int h = (H + segments - 1) / segments;
      const long cost = rounds * ((h + 2 + R - 1) / R + 3);
      if (best.segments == 0 || cost < best.cost) best = {R, strips, segments, cost};
    }
  }
  return best;
}

// A chain's tiles, smallest first.  A pair on a 16 x 24 tile takes about
// 14 us whatever the map's size, most of it products; on smaller tiles each CU
// has fewer of them, and LDS has room for a weight buffer of its own, so that
// the second layer's weights land behind the ring and the first layer.  The
// whole network on 64 x 48 pixels: 229 us on 16 x 24 tiles, 127 us on 8 x 16.
//
// The smaller ones only up to a quarter of the CUs: a process runs kernels of
// up to 4 streams at once, and as many chains of small maps, each waiting for
// tiles of its own, have to fit side by side, as they did on 16 x 24 tiles.
// (With up to a tile a CU two contexts on 128 x 256 pixels, 88 tiles of 16 x 24
// or 256 of 8 x 16, now and then started together, kept CUs from each other and
// gave up waiting: once in 3000 runs.)  Maps over some 12000 pixels stay on
// 16 x 24 tiles: 128 x 128 pixels 221 us, where 128 tiles of 8 x 16 took 141.
using SmallTile = Geo<8, 16, true>;
using MiddleTile = Geo<12, 16, true>;
using LargeTile = Geo<16, 24, false>;
struct ChainTile {
  int rows, cols;
  void (*kernel)(PairArgs);
};
const ChainTile CHAIN_TILES[ien_ctx::CHAIN_TILINGS] = {
    {SmallTile::OTR, SmallTile::OTC, conv_chain<SmallTile>},
    {MiddleTile::OTR, MiddleTile::OTC, conv_chain<MiddleTile>},
    {LargeTile::OTR, LargeTile::OTC, conv_chain<LargeTile>},
};

long tile_count(const ChainTile &t, int H, int W) {
  return (long)((W + t.cols - 1) / t.cols) * ((H + t.rows - 1) / t.rows);
}

}  // namespace

int chain_choice(int cus, int H, int W) {
  constexpr int LAST = ien_ctx::CHAIN_TILINGS - 1;
  for (int i = 0; i < LAST; i++)
    if (4 * tile_count(CHAIN_TILES[i], H, W) <= cus) return i;
  return tile_count(CHAIN_TILES[LAST], H, W) <= cus ? LAST : -1;
}

namespace {

// The smallest tiling of a map whose workgroups are all resident at once
// (one per CU at most), or null.
const ChainTile *chain_tile(ien_ctx *ctx, int H, int W) {
  for (int i = chain_choice(ctx->cus, H, W); i >= 0 && i < ien_ctx::CHAIN_TILINGS; i++) {
    if (tile_count(CHAIN_TILES[i], H, W) > ctx->chain_tiles) continue;
    int &per_cu = ctx->chain_per_cu[i];
    if (per_cu < 0) {
      int n = 0;
      if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, CHAIN_TILES[i].kernel, THREADS, 0) != hipSuccess)
        n = 0;
      per_cu = n;
    }
    if (per_cu >= 1) return &CHAIN_TILES[i];
  }
  return nullptr;
}

}  // namespace

bool pair_supported(const PairCall &p) {
  return layer_ok(p.w1, p.s1) && layer_ok(p.w2, p.s2) && maps_ok(p.x, p.y, p.H, p.W);
}

ien_status launch_pair(ien_ctx *ctx, const PairCall &p) {
  IEN_CHECK(pair_supported(p), IEN_ERR_INPUT, "not a pair of 3x3 64-channel PReLU layers");
  PairArgs a = {};
  a.x = p.x;
  a.y = p.y;
  a.H = p.H;
  a.W = p.W;
  const PairCut cut = pair_cut(p.H, p.W, ctx->cus);
  a.tiles_x = cut.strips;
  a.tiles_y = cut.segments;
  a.pairs = 1;
  const ien_matrix *w[2] = {p.w1, p.w2};
  const float *s[2] = {p.s1, p.s2};
  fill_layers(a, w, s, 2);
  const dim3 grid((unsigned)(cut.strips * cut.segments));
  if (cut.rows == 2)
    hipLaunchKernelGGL(conv_pair<2>, grid, dim3(THREADS), 0, ctx->stream, a);
  else
    hipLaunchKernelGGL(conv_pair<4>, grid, dim3(THREADS), 0, ctx->stream, a);
  IEN_HIP(hipGetLastError());
  return IEN_OK;
}

bool chain_supported(ien_ctx *ctx, const ChainCall &c) {
  if (!ctx->chain_flags || c.pairs < 1 || c.pairs > MAXPAIRS || !maps_ok(c.a, c.b, c.H, c.W))
    return false;
  for (int i = 0; i < 2 * c.pairs; i++)
    if (!layer_ok(c.w[i], c.s[i])) return false;
  if (c.first) {
    const ien_matrix *m = c.first;
    if (m->k != 36 || m->n != C || m->kb != 3 || m->nb < 2 || !m->d_packed || !m->d_bias ||
        !c.first_slope || !c.image)
      return false;
  }
  if (c.last) {
    const ien_matrix *m = c.last;
    if (m->k != 9 * C || m->n != 48 || m->kb != STEPS || m->nb < 2 || !m->d_packed || !m->d_bias ||
        !c.image || !c.out || ((uintptr_t)c.out & 15) != 0 ||
        (long)c.H * c.W * 48 > 0x7fff0000L)
      return false;
  }
  return chain_tile(ctx, c.H, c.W) != nullptr;
}

ien_status launch_chain(ien_ctx *ctx, const ChainCall &c, uint16_t **out) {
  IEN_CHECK(chain_supported(ctx, c), IEN_ERR_INPUT, "not a chain this device runs at once");
  PairArgs a = {};
  a.x = c.a;
  a.border[0] = c.b;
  a.border[1] = c.a;
  a.y = a.border[(c.pairs - 1) & 1];
  a.H = c.H;
  a.W = c.W;
  const ChainTile *tile = chain_tile(ctx, c.H, c.W);
  a.tiles_x = (c.W + tile->cols - 1) / tile->cols;
  a.tiles_y = (c.H + tile->rows - 1) / tile->rows;
  a.pairs = c.pairs;
  fill_layers(a, c.w, c.s, 2 * c.pairs);
  a.flags = ctx->chain_flags;
  a.seq = ++ctx->chain_seq;
  a.spin_limit = ctx->chain_spin;
  if (c.first) {
    a.w0 = c.first->d_packed;
    a.b0 = c.first->d_bias;
    a.s0 = c.first_slope;
    a.image = c.image;
  }
  if (c.last) {
    a.wl = c.last->d_packed;
    a.bl = c.last->d_bias;
    a.image = c.image;
    a.out = c.out;
  }
  const int tiles = a.tiles_x * a.tiles_y;
  hipLaunchKernelGGL(tile->kernel, dim3((unsigned)tiles), dim3(THREADS), 0, ctx->stream, a);
  IEN_HIP(hipGetLastError());
  *out = c.last ? nullptr : a.y;
  return IEN_OK;
}

ien_status chain_status(ien_ctx *ctx, int first) {
  int word = 0;
  IEN_HIP(hipMemcpyAsync(&word, ctx->chain_flags + 1, 4, hipMemcpyDeviceToHost, ctx->stream));
  IEN_HIP(hipStreamSynchronize(ctx->stream));
  if (word < first || word <= ctx->chain_reported) return IEN_OK;
  ctx->chain_reported = word;
  return fail(IEN_ERR_GPU, "body chain: a tile's wait for its neighbours timed out");
}

}  // namespace ien

using namespace ien;

extern "C" ien_status ien_conv3_pair(ien_ctx *ctx, const uint16_t *d_x, uint16_t *d_y,
                                     size_t height, size_t width, const ien_matrix *w1,
                                     const float *d_slope1, const ien_matrix *w2,
                                     const float *d_slope2) {
  IEN_CHECK(ctx && d_x && d_y && w1 && w2 && d_slope1 && d_slope2, IEN_ERR_INPUT,
            "null argument");
  IEN_CHECK(height > 0 && width > 0 && height < (1u << 20) && width < (1u << 20), IEN_ERR_INPUT,
            "map of %zu x %zu", height, width);
  for (const ien_matrix *m : {w1, w2})
    IEN_CHECK(m->k == 9 * C && m->n == C, IEN_ERR_INPUT,
              "pair layers are 3x3 64->64 (k 576, n 64), not k %zu, n %zu", m->k, m->n);
  const size_t bytes = height * width * C * 2;
  IEN_CHECK(bytes <= 0x7fff0000UL, IEN_ERR_INPUT, "map of %zu bytes over 2 GiB", bytes);
  IEN_CHECK((((uintptr_t)d_x | (uintptr_t)d_y) & 15) == 0, IEN_ERR_INPUT,
            "maps must be 16-byte aligned");
  const uintptr_t x = (uintptr_t)d_x, y = (uintptr_t)d_y;
  IEN_CHECK(x + bytes <= y || y + bytes <= x, IEN_ERR_INPUT, "input and output maps overlap");
  PairCall p;
  p.x = d_x;
  p.y = d_y;
  p.H = (int)height;
  p.W = (int)width;
  p.w1 = w1;
  p.s1 = d_slope1;
  p.w2 = w2;
  p.s2 = d_slope2;
  return launch_pair(ctx, p);
}

extern "C" ien_status ien_conv3_chain(ien_ctx *ctx, uint16_t *d_a, uint16_t *d_b, size_t height,
                                      size_t width, size_t pairs, const ien_matrix *const *w,
                                      const float *const *d_slopes, uint16_t **d_out) {
  IEN_CHECK(ctx && d_a && d_b && w && d_slopes && d_out, IEN_ERR_INPUT, "null argument");
  IEN_CHECK(pairs >= 1 && pairs <= MAXPAIRS, IEN_ERR_INPUT, "%zu pairs (1 to %d)", pairs, MAXPAIRS);
  IEN_CHECK(height > 0 && width > 0 && height < (1u << 20) && width < (1u << 20), IEN_ERR_INPUT,
            "map of %zu x %zu", height, width);
  ChainCall c;
  c.a = d_a;
  c.b = d_b;
  c.H = (int)height;
  c.W = (int)width;
  c.pairs = (int)pairs;
  for (size_t i = 0; i < 2 * pairs; i++) {
    IEN_CHECK(w[i] && d_slopes[i], IEN_ERR_INPUT, "layer %zu: null argument", i);
    IEN_CHECK(w[i]->k == 9 * C && w[i]->n == C, IEN_ERR_INPUT,
              "layer %zu: chain layers are 3x3 64->64 (k 576, n 64), not k %zu, n %zu", i, w[i]->k,
              w[i]->n);
    c.w[i] = w[i];
    c.s[i] = d_slopes[i];
  }
  const size_t bytes = height * width * C * 2;
  IEN_CHECK(bytes <= 0x7fff0000UL, IEN_ERR_INPUT, "map of %zu bytes over 2 GiB", bytes);
  IEN_CHECK((((uintptr_t)d_a | (uintptr_t)d_b) & 15) == 0, IEN_ERR_INPUT,
            "maps must be 16-byte aligned");
  const uintptr_t a = (uintptr_t)d_a, b = (uintptr_t)d_b;
  IEN_CHECK(a + bytes <= b || b + bytes <= a, IEN_ERR_INPUT, "the two maps overlap");
  IEN_CHECK(chain_supported(ctx, c), IEN_ERR_INPUT,
            "a %zu x %zu map has more 16 x 24 tiles than this device holds at once", height, width);
  return launch_chain(ctx, c, d_out);
}

extern "C" ien_status ien_conv3_chain_status(ien_ctx *ctx) {
  IEN_CHECK(ctx, IEN_ERR_INPUT, "null argument");
  IEN_HIP(hipSetDevice(ctx->device));
  return chain_status(ctx, 1);
}

