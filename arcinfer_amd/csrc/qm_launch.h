// Host-side launchers of the qmatmul kernels (one per kernel family, defined next to the kernels).
// All return hipSuccess or the launch error; shapes are validated by the C-ABI layer (qm_api.hip) beforehand.
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "qm_device.h"
#include "qm_workspace.h"

namespace qm {

// GGUF rows -> prepared planes (qm_prep.hip)
// K: the prepared row length (a multiple of 256); kraw: 32-blocks per raw row (K / 32, or fewer for a padded
// Q8_0 / Q4_0 / IQ4_NL row)
hipError_t launch_repack(int type, const uint8_t* raw, int rows, int K, int kraw, uint8_t* qs, uint8_t* hdr,
                         hipStream_t s);
// f32 rows -> int8 + per-32 scales + per-16 sums (qm_prep.hip)
hipError_t launch_quantize(const float* x, int ldx, int M, int M_stride, int K, bool act32, int8_t* aq, float* asc,
                           int16_t* absum, hipStream_t s);

struct GemvArgs {
  WView w;
  const int8_t* aq;
  const float* asc;
  const int16_t* absum;
  int M_stride, T;
  float* C;
  int ldc, c_off, accumulate;
  int32_t* dbg_isum;  // non-null: write the block sums instead of C
  int32_t* dbg_msum;
  int split = 0;      // batch-1 sweep: work-groups of the first dispatch round (0: every group takes the same rows)
};
hipError_t launch_gemv(int type, const GemvArgs& a, hipStream_t s);

// Products of 1 to 32 tokens against one read of the weight on the int8 matrix pipe (qm_skinny_*.hip). Any weight type,
// rows and K; dbg_isum: block-sum mode.
struct SkinnyArgs {
  WView w;
  const int8_t* aq;
  const float* asc;
  const int16_t* absum;
  int M, M_stride;
  int ash;  // asc row of 32-block b: b >> ash
  float* C;
  int ldc, c_off, accumulate;
  int32_t* dbg_isum;
  int32_t* dbg_msum;
};
constexpr int kSkinnyMax = 32;
// whether a decode GEMV (prompt = false) or prompt GEMM of M tokens goes there
bool skinny_supported(int type, bool prompt, int M, int rows, int K);
hipError_t launch_skinny(int type, const SkinnyArgs& a, hipStream_t s);

// Row source of a GEMM's activation tile: dense (row m = token m), gathered (row r = token rowmap[r]) or slots.
struct GemmArgs {
  WView w;       // weight (MoE: gate or down, stacked experts)
  WView w2;      // MoE gate/up: the up projection
  const int8_t* aq;
  const float* asc;
  const int16_t* absum;
  int M, M_stride;
  float* C;
  int ldc, c_off, accumulate;
  int32_t* dbg_isum;
  // Dense products: tiles from split_from on are cut into `splits` pieces of K each, whose partial tiles go to part (see
  // gemm_split); part null: no tile is cut
  float* part = nullptr;
  int split_from = 0, splits = 1;
  int ash = 0;  // activation scales per 32 << ash values: asc row of 32-block b is b >> ash (0, or 3 = per 256)
  // MoE tile mode
  const int* tiles;    // [0] = count, then (expert, first slot, rows) per tile
  const int* rowmap;   // slot -> token (gate/up), or null (down: slot rows)
  const float* rowscale;  // slot -> routing weight (down), or null
  int8_t* hq;          // gate/up: quantized h rows [slots][ldc] (ldc = F, the down projection's K)
  float* hsc;          // gate/up: h scales [F/32][slots]
  int slots;           // row stride of hsc
  int max_tiles;
  int expert_rows;     // rows per expert in w (Fv <= F for gate/up, E for down)
};
// MoE tile modes: GATEUP (gate and up of one type in one launch: h quantized), G (gate alone: f32 g into C),
// UH (up alone after G: h from u and g, quantized), DOWN (routing-weighted y)
// How a dense product's tiles are dealt. The chip holds kGemmSlots work-groups of the prompt kernels at once (two per CU), so
// tiles run in rounds and the last one is often nearly empty (520 tiles take the time of 1024). The tiles past the last
// whole round -- all of them for a small product -- are cut along K into `splits` pieces, each with its share of the
// superblocks, whose partial tiles are added by a second kernel (in piece order: the result does not depend on timing).
constexpr int kGemmSlots = 512;
constexpr size_t kSplitBytes = (size_t)32 << 20;  // most partial tiles of one call
struct GemmSplit {
  int from, splits;  // tiles [0, from) whole, [from, tiles) in `splits` pieces each (splits = 1: none)
  size_t bytes;      // partial tiles
  bool halves;       // uncut, two K halves added into a zeroed C
  float us;          // the call's modelled time
};
// A kernel's times in microseconds, fitted to some 2000 measured products of 14 types (rms 3 %): `us` a superblock of a full round;
// `alone`, `last` the part of it that a superblock of a round takes which fills half the slots or less (a work-group that has its
// CU to itself runs faster than two that share it), as the only round or after another; what a call costs besides when it runs
// whole (and per 512 work-groups), in halves (and per 512 of them, as far as they hold results, and as far as not) and cut (and per 512 pieces; `stream` at least);
// `host` what a call with its own workspace takes the host (0: it has one anyway). A call is cut for a gain of `part` of its time
// and of `least` us; `even`: how much of pieces that differ by a superblock runs as their mean (the rest as the longest).
struct GemmRates {
  float us, alone, last, whole, whole_wg, half, half_wg, half_pad, cut, cut_wg, host, part, least, even, stream;
};
// Rounds that n equal work-groups take. (With more than two whole rounds the last one starts while others still run.)
inline float gemm_rounds(int n, const GemmRates& g) {
  const int f = n / kGemmSlots, rem = n % kGemmSlots;
  if (rem == 0) return (float)f;
  if (f >= 2) return (float)f + (2 * rem <= kGemmSlots ? 0.38f : 0.82f);
  return (float)f + (2 * rem > kGemmSlots ? 1.0f : f ? g.last : g.alone);
}
// tiles of bm x 128 results, filled to `fill`; K of nsb superblocks; halves: a small product may add two K halves into a zeroed C.
// A work-group costs its superblocks and about one more (its prologue and store). With more than one whole round cutting the last
// measured level (Q4_K 2048 x 5120 -> 17408, 2176 tiles: 572 us either way), so only products of fewer than 1024 tiles are
// cut, of K 2048 and more.
inline GemmSplit gemm_split(int tiles, int nsb, int bm, float fill, bool halves, const GemmRates& g) {
  GemmSplit r{tiles, 1, 0, false, g.whole + g.whole_wg * (float)tiles / kGemmSlots + g.us * gemm_rounds(tiles, g) * (float)(nsb + 1)};
  const int full = tiles / kGemmSlots * kGemmSlots, rem = tiles - full;
  if (halves && nsb >= 8 && tiles < kGemmSlots) {
    const float p = 2.0f * (float)tiles / kGemmSlots;
    const float t = g.half + p * (g.half_wg * fill + g.half_pad * (1.0f - fill)) + g.us * gemm_rounds(2 * tiles, g) * (0.5f * (float)nsb + 1.0f);
    // (up to one tile per CU always: IQ4_XS 333 x 17408 -> 5120, 240 tiles, 131 us in halves against 156, 200 x 5120 -> 5120, 160
    //  tiles, 45 against 51; above, unless whole tiles are faster: 416 tiles of Q5_K 777 x 4096 -> 4096
    //  93 us in halves against 75, but 360 of IQ4_XS 142 x 3072 -> 15312, the last token tile nearly empty, 46.6 against 48.5)
    if (2 * tiles <= kGemmSlots || 0.97f * t < r.us) {
      r.us = t;
      r.halves = true;
    }
  }
  if (rem == 0 || full > kGemmSlots || nsb < 8) return r;
  const float uncut = r.us, whole = (float)(full / kGemmSlots) * (float)(nsb + 1);
  GemmRates pieces = g;
  if (full) pieces.alone = g.last;
  // (pieces of two superblocks only where there are few: IQ2_XXS 75 x 2560 -> 8800, 138 tiles in five, 28.6 us against 25.2 in halves)
  for (int s = 2; s <= 8 && nsb / s >= (halves && rem > 128 ? 3 : 2); ++s) {
    const size_t bytes = (size_t)rem * s * bm * 128 * sizeof(float);
    const float deep = g.even * (float)nsb / (float)s + (1.0f - g.even) * (float)((nsb + s - 1) / s) + 1.0f;  // a piece's superblocks
    const float t = g.cut + g.cut_wg * (float)(rem * s) / kGemmSlots + g.us * (whole + gemm_rounds(rem * s, pieces) * deep);
    const float least = fmaxf(t, fmaxf(g.host, g.stream * (float)rem / (float)tiles));
    if (least < (1.0f - g.part) * uncut && least <= uncut - g.least && t < 0.999f * r.us && bytes <= kSplitBytes) r = GemmSplit{full, s, bytes, r.halves, t};
  }
  return r;
}
// The same for one call, on the f16 path or by launch_gemm (splits = 1 where that takes the few-token kernels)
GemmSplit gemm_split_for(int type, int M, int rows, int K, bool f16);
// C (op)= the sums of the cut tiles' pieces (bm x 128 each); tile t: rows bm * (t % gy).., columns 128 * (t / gy).. when
// m_fast, else bm * (t / gx).., 128 * (t % gx)..
hipError_t launch_split_sum(const GemmArgs& a, int bm, int tiles, int gx, int gy, bool m_fast, hipStream_t s);
enum GemmMode : int { GEMM_DENSE = 0, GEMM_MOE_GATEUP = 1, GEMM_MOE_DOWN = 2, GEMM_MOE_G = 3, GEMM_MOE_UH = 4 };
hipError_t launch_gemm(int type, int mode, const GemmArgs& a, hipStream_t s);
// Prompt GEMM on the f16 matrix pipe (qm_gemm_f16.hip): the types and shapes it takes, its per-call workspace, and
// the launcher (ws = null: the workspace comes from a per-device stream-ordered pool). dbg_isum: block-sum mode.
bool f16_gemm_supported(int type, int M, int rows, int K);
size_t f16_workspace_bytes(int type, int M, int K);
hipError_t launch_gemm_f16(int type, const GemmArgs& a, void* ws, hipStream_t s);
// The current device's copies of the static scratch arrays for the allocation-free entry: ptr (bytes) the f16 path's
// workspace, part (kSplitBytes) the partial tiles
hipError_t f16_scratch(void** ptr, size_t* bytes, void** part);
// slots per MoE tile (one expert each); a 64-row tile (fewer, larger tiles) measured slower under the Zipf skew
constexpr int kMoeTileRows = 32;

// Activation producers (qm_producers.hip)
hipError_t launch_rmsnorm_quant(const float* x, int ldx, const float* w, int K, int M, int M_stride, float eps,
                                int8_t* aq, float* asc, int16_t* absum, float* h, int ldh, bool act32, hipStream_t s);
hipError_t launch_swiglu_quant(const float* gu, int ldg, int F, int M, int M_stride, int fused, int gelu, int8_t* aq,
                               float* asc, int16_t* absum, bool act32, hipStream_t s);
hipError_t launch_add_norm_quant(float* x, const float* t, const float* w, int K, float eps, float scale,
                                 const float* w2, int M, int M_stride, int8_t* aq, float* asc, int16_t* absum,
                                 bool act32, hipStream_t s);

// The shared expert of an MoE layer: sh [T][ldsh] (null: none), added times g_t = sigmoid(gl[t * ldl]) (gl null:
// g_t = 1). zero/kernels/moe.cl:332-340, 37-41.
struct MoeShared {
  const float* sh;
  int ldsh;
  const float* gl;
  int ldl;
};

// MoE routing (qm_moe.hip); escale [NE] (or null): each chosen expert's weight times its scale
// Tokens per wave of the routing kernel, and its work-groups (four waves each) for T tokens.
// (about 2048 waves, two per SIMD: the selection is latency-bound, T = 4096 measured 20 us for the route + scan +
// scatter chain at 2 tokens per wave, 23 at 4, 22 at 1)
inline int moe_route_tpw(int T) { return T >= 4096 ? (T / 2048 < 16 ? T / 2048 : 16) : 1; }
inline int moe_route_groups(int T) { return (T + 4 * moe_route_tpw(T) - 1) / (4 * moe_route_tpw(T)); }
// counts (or null): per-expert counts by global atomics (counts zeroed first); part (or null): each work-group's
// expert histogram as row blockIdx.x of part [moe_route_groups(T)][NE], plain stores
hipError_t launch_moe_route(const float* logits, int ldl, int T, int NE, int NU, int* ids, float* wts, int* counts,
                            const float* escale, int* part, hipStream_t s);
// From the routing histograms: counts; part's columns become running sums over the routing work-groups
hipError_t launch_moe_scan(int* part, int groups, int* counts, int NE, hipStream_t s);
// The slot permutation (stok, swt, inv) and the scan's outputs: first slots (cursor), tile starts, the tile list
hipError_t launch_moe_scatter(const int* ids, const float* wts, int T, int NU, int NE, const int* part,
                              const int* counts, int* cursor, int* tstart, int* tiles, int tile_rows, int* stok,
                              float* swt, int* inv, hipStream_t s);
// Expert products over the slot tiles for small expert sets (qm_moe_few.hip): gate and up of one type (hq / hsc), or down; and
// whether a layer of `slots` slots, NE experts, hidden E and expert width Fv (F padded) takes them
bool moe_few(int type, int slots, int NE, int E, int Fv);
bool moe_few_down(int type, int slots, int NE, int E, int F);
hipError_t launch_moe_few(int type, bool down, const GemmArgs& a, hipStream_t s);
hipError_t launch_moe_combine(float* x, const float* y, const int* inv, int T, int NU, int E, int accumulate,
                              const MoeShared& sh, hipStream_t s);
hipError_t launch_fill_i32(int* p, int value, size_t n, hipStream_t s);
// MoE at decode sizes (qm_moe_dec.hip): routing + gate/up -> ids, wts, h (f32 [T*NU][F]), then down + combine into x
// (gate, up, down of types tg, tu, td; escale: routing expert scales or null; sh: the shared expert or sh.sh null)
hipError_t launch_moe_decode(int tg, int tu, int td, const WView& gate, const WView& up, const WView& down, int T,
                             int NU, int E, int F, int Fv, const float* logits, int ldl, int NE, const float* escale,
                             int* ids, float* wts, const int8_t* aq, const float* asc, int M_stride, float* h, float* x,
                             int accumulate, const MoeShared& sh, hipStream_t s);

}  // namespace qm
