// Products of a few tokens (multi-token decode, short prompts) on the int8 matrix pipe: C[t][n] (op)= sum_k W[n][k] a_t[k]
// for up to 32 tokens against one read of the weight.
//
// Bound by the weight decode's VALU work (about 130 instructions per 64 blocks of 32, paid once whatever the token
// count), with the weight stream from HBM close behind; the products themselves are 16 x 16 x 32 int8 MFMAs.
//
// A wave works on quads: four consecutive 32-blocks (128 elements) of 16 weight rows. Lane (c, g) = (lane % 16,
// lane / 16) loads and decodes block g of the quad of weight row c as the decode GEMVs do (lanes g read consecutive
// records) and holds block g of token c. The MFMA of block j wants word g of block j in lane group g for both operands:
// a 4 x 4 transpose over the lane groups, four v_permlane32_swap / v_permlane16_swap per four words (no LDS). Per quad
// one four-block f32 outer product gives asc * d * sc for the four blocks (each lane group contributes its own block's
// scales, so every scale is decoded once); the int32 block sums are scaled and added in f32, as the prompt GEMM does
// (zero/kernels/gemm.cl:367-412). Types with a scale per 16 elements take two MFMAs per block, each with the other half
// of the token operand zero; mins are one f32 16 x 16 x 4 MFMA per quad (and half) into the accumulator.
// 16x16 result layout: lane (c, g) holds column c (weight row) and rows 4 g + r (tokens), r = 0..3.
#pragma once
#include <type_traits>

#include "qm_decode.h"

namespace qm {

typedef int sk_v4i __attribute__((ext_vector_type(4)));
typedef float sk_v4f __attribute__((ext_vector_type(4)));
typedef float sk_v16f __attribute__((ext_vector_type(16)));

// per-16 scales: the block sums of the two halves are needed separately
template <int TYPE> constexpr bool kHalves = Traits<TYPE>::SC16 || Traits<TYPE>::SPLIT;

// lane group g holds x[0..3] of block g -> lane group g holds word g of block j in x[j]
__device__ __forceinline__ void group_transpose(uint32_t x[4]) {
  const auto a = __builtin_amdgcn_permlane32_swap(x[0], x[2], false, false);
  const auto b = __builtin_amdgcn_permlane32_swap(x[1], x[3], false, false);
  const auto c = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false);
  const auto d = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
  x[0] = c[0];
  x[1] = c[1];
  x[2] = d[0];
  x[3] = d[1];
}

__device__ __forceinline__ long pair64(uint32_t lo, uint32_t hi) { return (long)(((uint64_t)hi << 32) | lo); }

// A lane's token operands of one quad: words (both halves) of block j, the scale of block g, and (types with mins) the
// scale times the block's sum, Q2_K per half
template <int TYPE> struct TokQuad {
  uint32_t x[2][4];
  float asc;
  float u[kMin16<TYPE> ? 2 : 1];
};

// raw: the token's 32 bytes of block g
template <int TYPE, bool DUMP>
__device__ __forceinline__ void tok_quad(const u32x4_t raw[2], float asc, int bs0, int bs1, TokQuad<TYPE>& q) {
#pragma unroll
  for (int h = 0; h < 2; ++h) {
#pragma unroll
    for (int k = 0; k < 4; ++k) q.x[h][k] = raw[h][k];
    group_transpose(q.x[h]);
  }
  if constexpr (DUMP) return;
  q.asc = asc;
  if constexpr (kMin16<TYPE>) {
    q.u[0] = asc * (float)bs0;
    q.u[1] = asc * (float)bs1;
  } else if constexpr (Traits<TYPE>::MINS) {
    q.u[0] = asc * (float)(bs0 + bs1);
  }
}

// One quad of one row tile times NT token tiles, added to acc. q: the quad, live: whether it lies in the row (a quad past
// the row's end repeats the last one and is scaled by 0), n: the lane's weight row (block-sum mode).
template <int TYPE, int NT, bool DUMP>
__device__ __forceinline__ void quad_product(const SkinnyArgs& a, const RawBlk& w, int q, bool live, int n,
                                             const typename LdsFor<TYPE>::type* tab, const KvTab& kv,
                                             const TokQuad<TYPE>* tk, sk_v4f* acc) {
  constexpr bool HALVES = kHalves<TYPE>;
  const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
  const sk_v4i zero4 = {0, 0, 0, 0};
  uint32_t wd[8];
  int sc, sc1, mn;
  float d, dmin;
  decode_block32<TYPE>(w, tab, 4 * (q & 1) + g, kv, wd, sc, sc1, mn, d, dmin);
  group_transpose(wd);
  group_transpose(wd + 4);
  const float dsc[2] = {live ? (kBlockScales<TYPE> ? d : d * (float)sc) : 0.0f, HALVES && live ? d * (float)sc1 : 0.0f};
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    // (Q6_K's decoded values are q + 32: a constant operand of -32 takes it off in the integer sums)
    const long m32 = pair64(0xE0E0E0E0u, 0xE0E0E0E0u);
    auto sums = [&](int h, int j) {  // block j's int32 sums: of half h, or of the whole block
      if constexpr (HALVES) {
        const long aop = h ? pair64(0u, tk[nt].x[1][j]) : pair64(tk[nt].x[0][j], 0u);
        sk_v4i c0 = zero4;
        if constexpr (TYPE == T_Q6_K) c0 = __builtin_amdgcn_mfma_i32_16x16x32_i8(aop, m32, zero4, 0, 0, 0);
        return __builtin_amdgcn_mfma_i32_16x16x32_i8(aop, pair64(wd[j], wd[4 + j]), c0, 0, 0, 0);
      } else {
        return __builtin_amdgcn_mfma_i32_16x16x32_i8(pair64(tk[nt].x[0][j], tk[nt].x[1][j]), pair64(wd[j], wd[4 + j]), zero4,
                                                     0, 0, 0);
      }
    };
    if constexpr (DUMP) {
      const int rows = a.w.rows, nb = a.w.K / 32;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int src = c + 16 * j, blk = 4 * q + j;
        const int scj = __shfl(sc, src), sc1j = __shfl(sc1, src), mnj = __shfl(mn, src);
        const sk_v4i lo = sums(0, j), hi = HALVES ? sums(1, j) : zero4;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int t = 16 * nt + 4 * g + r;
          if (!live || t >= a.M || n >= rows) continue;
          const size_t o = ((size_t)t * rows + n) * nb + blk;
          a.dbg_isum[o] = HALVES ? scj * lo[r] + sc1j * hi[r] : kBlockScales<TYPE> ? lo[r] : scj * lo[r];
          if constexpr (Traits<TYPE>::MINS) {
            if (a.dbg_msum) {
              const int b0 = (int)a.absum[(size_t)(2 * blk) * a.M_stride + t],
                        b1 = (int)a.absum[(size_t)(2 * blk + 1) * a.M_stride + t];
              a.dbg_msum[o] = kMin16<TYPE> ? (mnj & 0xFFFF) * b0 + (mnj >> 16) * b1 : mnj * (b0 + b1);
            }
          }
        }
      }
    } else {
      sk_v16f zero16;
#pragma unroll
      for (int r = 0; r < 16; ++r) zero16[r] = 0.0f;
      // the quad's own sum, from its min term, then onto the accumulator: min terms cancel against products of the same four
      // blocks, and the long chain of f32 additions is a quarter as long (4 additions per quad and token tile)
      sk_v4f sum = {0.0f, 0.0f, 0.0f, 0.0f};
      if constexpr (Traits<TYPE>::MINS) {
        sum = __builtin_amdgcn_mfma_f32_16x16x4f32(tk[nt].u[0], live ? -dmin * (float)(kMin16<TYPE> ? mn & 0xFFFF : mn) : 0.0f,
                                                   sum, 0, 0, 0);
        if constexpr (kMin16<TYPE>)
          sum = __builtin_amdgcn_mfma_f32_16x16x4f32(tk[nt].u[1], live ? -dmin * (float)(mn >> 16) : 0.0f, sum, 0, 0, 0);
      }
#pragma unroll
      for (int h = 0; h < (HALVES ? 2 : 1); ++h) {
        const sk_v16f scl = __builtin_amdgcn_mfma_f32_16x16x1f32(tk[nt].asc, dsc[h], zero16, 0, 0, 0);
        sk_v4i s[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) s[j] = sums(h, j);
        // (one token tile: the second half's sum by itself, as one chain of eight rounds more than two of four)
        constexpr bool APART = NT == 1;
        sk_v4f hs = sum;
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float v = (float)s[j][r];
            const bool first = j == 0 && (h == 0 ? !Traits<TYPE>::MINS : APART);
            hs[r] = first ? scl[r] * v : fmaf(scl[4 * j + r], v, hs[r]);
          }
#pragma unroll
        for (int r = 0; r < 4; ++r) sum[r] = h > 0 && APART ? sum[r] + hs[r] : hs[r];
        // (one half and token tile at a time: free to move, the compiler starts them all and runs out of registers)
        if constexpr (HALVES) __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[nt][r] += sum[r];
    }
  }
}

// Adds the W waves' partial tiles (part[wave][element][lane], element = 4 * tile + r) in 64 bits and stores NTOT result
// tiles; tile e / 4 is token tile (e / 4) % NT of row tile (e / 4) / NT from row n0.
template <int NT, int NTOT, int W>
__device__ __forceinline__ void store_tiles(const SkinnyArgs& a, const float (*part)[NTOT * 4][64], int n0, int wave) {
  const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
  for (int e = wave; e < NTOT * 4; e += W) {
    double sum = part[0][e][lane];
#pragma unroll
    for (int k = 1; k < W; ++k) sum += (double)part[k][e][lane];
    float v = (float)sum;
    const int t = 16 * ((e >> 2) % NT) + 4 * g + (e & 3), n = n0 + 16 * ((e >> 2) / NT) + c;
    if (t < a.M && n < a.w.rows) {
      float* cp = a.C + (size_t)t * a.ldc + a.c_off + n;
      if (a.accumulate == 1) {
        v += *cp;
      } else if (a.accumulate == 2) {
        const float gt = *cp;
        v *= gt / (1.0f + expf(-gt));
      }
      *cp = v;
    }
  }
}

// A work-group owns RT row tiles; its W waves split K (wave w: quads w, w + W, ...), each with PF quads' loads in flight.
// Tokens are read from L2 with every quad (two row tiles halve that), so any K goes. Every fourth quad a wave's one tile
// (decode) goes to 64 bits: added up in f32, 34 quads a wave, 5 tokens of 17408 were 1.27e-7 off the exact product against the GEMV's 8.8e-8; now 7.2e-8, for 1
// to 4 % of the time (every eighth quad: as long, and up to 1.07 of the GEMV's error).
template <int TYPE, int RT, int NT, int W, int PF, bool DUMP>
__global__ __launch_bounds__(64 * W, 4) void skinny_kernel(SkinnyArgs a) {
  using Tr = Traits<TYPE>;
  __shared__ typename LdsFor<TYPE>::type tab;
  __shared__ float part[DUMP ? 1 : W][RT * NT * 4][64];
  // (the wave's index as a scalar: its quads, trip count and base addresses are then scalar too)
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
  const int K = a.w.K, nb = K / 32, nq = K / 128, rows = a.w.rows;
  const int n0 = blockIdx.x * (16 * RT);
  // each address is a scalar base (the tile's first row, advanced by quads) plus a lane's 32-bit offset
  const uint8_t* qbase = a.w.qs + (size_t)n0 * nb * Tr::QB;
  const uint8_t* hbase = a.w.hdr + (size_t)n0 * (nb / 8) * Tr::HB;
  uint32_t qoff[RT], hoff[RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    const int n = min(16 * rt + c, rows - 1 - n0);
    qoff[rt] = (uint32_t)(n * nb + g) * Tr::QB;
    hoff[rt] = (uint32_t)(n * (nb / 8)) * Tr::HB;
  }
  int tok[NT];
  const int8_t* arow[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    tok[nt] = min(16 * nt + c, a.M - 1);  // (rows past the last token repeat it and are not stored)
    arow[nt] = a.aq + (size_t)tok[nt] * K + 32 * g;
  }
  const int steps = wave < nq ? (nq - 1 - wave) / W + 1 : 0;
  struct Stage {
    RawBlk w[RT];
    u32x4_t a[NT][2];
    float asc[NT];
    int16_t bs[NT][2];
  } st[PF];
  auto fetch = [&](int i, Stage& s) {
    const int q = min(wave + W * i, nq - 1);  // (past the end: the last quad again, unused)
    const uint8_t *qp = qbase + (uint32_t)(4 * q * Tr::QB), *hp = hbase + (uint32_t)((q >> 1) * Tr::HB);
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) s.w[rt] = load_block_ptr<TYPE, false>(qp + qoff[rt], hp + hoff[rt], 4 * (q & 1) + g);
    const int b = 4 * q + g;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      s.a[nt][0] = *(const u32x4_t*)(arow[nt] + 128 * q);
      s.a[nt][1] = *(const u32x4_t*)(arow[nt] + 128 * q + 16);
      if constexpr (!DUMP) s.asc[nt] = a.asc[(size_t)(b >> a.ash) * a.M_stride + tok[nt]];
      // (kept as loaded: packing the two sums here would wait for the loads)
      if constexpr (Tr::MINS && !DUMP) {
        s.bs[nt][0] = a.absum[(size_t)(2 * b) * a.M_stride + tok[nt]];
        s.bs[nt][1] = a.absum[(size_t)(2 * b + 1) * a.M_stride + tok[nt]];
      }
    }
  };
#pragma unroll
  for (int p = 0; p < PF; ++p) fetch(p, st[p]);
  lds_fill<TYPE>(&tab);
  if constexpr (!std::is_same_v<typename LdsFor<TYPE>::type, typename LdsFor<T_Q8_0>::type>) __syncthreads();
  const KvTab kv = kv_tab();
  sk_v4f acc[RT][NT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[rt][nt] = sk_v4f{0.0f, 0.0f, 0.0f, 0.0f};
  constexpr bool WIDE = !DUMP && RT * NT == 1;  // (decode's one tile; more have no registers for it)
  double tot[WIDE ? 4 : 1] = {};
  auto fold = [&] {
    if constexpr (WIDE)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        tot[r] += (double)acc[0][0][r];
        acc[0][0][r] = 0.0f;
      }
  };
  auto step = [&](int i, const Stage& s) {
    TokQuad<TYPE> tk[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
      tok_quad<TYPE, DUMP>(s.a[nt], DUMP ? 0.0f : s.asc[nt], Tr::MINS && !DUMP ? s.bs[nt][0] : 0,
                           Tr::MINS && !DUMP ? s.bs[nt][1] : 0, tk[nt]);
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
      quad_product<TYPE, NT, DUMP>(a, s.w[rt], wave + W * i, true, n0 + 16 * rt + c, &tab, kv, tk, acc[rt]);
  };
  int i = 0;
  for (; i + PF <= steps; i += PF) {
#pragma unroll
    for (int p = 0; p < PF; ++p) {
      step(i + p, st[p]);
      // (the next loads stay between the steps: free to move, the compiler gathers every stage's loads behind the last)
      __builtin_amdgcn_sched_barrier(0);
      fetch(i + p + PF, st[p]);
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (WIDE)
      if (i & PF) fold();
  }
#pragma unroll
  for (int p = 0; p < PF - 1; ++p)
    if (i + p < steps) step(i + p, st[p]);
  if constexpr (!DUMP) {
    fold();
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int r = 0; r < 4; ++r) part[wave][(rt * NT + nt) * 4 + r][lane] = WIDE ? (float)tot[WIDE ? r : 0] : acc[rt][nt][r];
    __syncthreads();
    store_tiles<NT, RT * NT, W>(a, part, n0, wave);
  }
}

// The same product as a persistent sweep, for rows short enough that a wave can keep its share of the tokens in
// registers: one work-group per CU, its W waves split K by quads (wave w: quads w, w + W, ..., CH of them) and hold
// those quads' token operands, scales and sums for the whole launch; the work-groups walk the row tiles b, b + G, ...,
// so the grid moves through the matrix together (consecutive rows stream from HBM at the same time) and the tokens are
// read from L2 once per CU. The next tile's loads are issued before the current tile is decoded; the waves' partial
// tiles are added through LDS, one barrier per tile.
// Measured and not kept (16 tokens, IQ4_XS 5120 -> 17408, 19.5 us): scaling a quad's sums behind the next quad's products
// (19.3), 16 waves of three quads (20.7), two tiles of loads ahead (21.5), one combine per four tiles (19.6-21).
template <int TYPE, int NT, int W, int CH, bool DUMP>
__global__ __launch_bounds__(64 * W, W / 4) void skinny_sweep_kernel(SkinnyArgs a) {
  using Tr = Traits<TYPE>;
  __shared__ typename LdsFor<TYPE>::type tab;
  __shared__ float part[DUMP ? 1 : 2][W][NT * 4][64];
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
  const int K = a.w.K, nb = K / 32, nq = K / 128, rows = a.w.rows;
  const int ntile = (rows + 15) / 16, G = gridDim.x;
  const int steps = (ntile - 1 - (int)blockIdx.x) / G + 1;
  RawBlk cur[CH], nxt[CH];
  auto fetch = [&](int i, RawBlk* dst) {
    const int n0 = 16 * min((int)blockIdx.x + G * i, ntile - 1), n = min(c, rows - 1 - n0);
    const uint8_t* qb = a.w.qs + (size_t)n0 * nb * Tr::QB;
    const uint8_t* hb = a.w.hdr + (size_t)n0 * (nb / 8) * Tr::HB;
    const uint32_t qo = (uint32_t)(n * nb + g) * Tr::QB, ho = (uint32_t)(n * (nb / 8)) * Tr::HB;
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      const int q = min(wave + W * u, nq - 1);  // (a quad past the row's end: the last one again, scaled by 0)
      dst[u] = load_block_ptr<TYPE, false>(qb + (uint32_t)(4 * q * Tr::QB) + qo, hb + (uint32_t)((q >> 1) * Tr::HB) + ho,
                                           4 * (q & 1) + g);
    }
  };
  fetch(0, cur);
  lds_fill<TYPE>(&tab);
  TokQuad<TYPE> tk[CH][NT];
#pragma unroll
  for (int u = 0; u < CH; ++u) {
    const int b = 4 * min(wave + W * u, nq - 1) + g;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const int t = min(16 * nt + c, a.M - 1);  // (rows past the last token repeat it and are not stored)
      const int8_t* ap = a.aq + (size_t)t * K + 32 * b;
      const u32x4_t raw[2] = {*(const u32x4_t*)ap, *(const u32x4_t*)(ap + 16)};
      float sa = 0.0f;
      int b0 = 0, b1 = 0;
      if constexpr (!DUMP) {
        sa = a.asc[(size_t)(b >> a.ash) * a.M_stride + t];
        if constexpr (Tr::MINS) {
          b0 = (int)a.absum[(size_t)(2 * b) * a.M_stride + t];
          b1 = (int)a.absum[(size_t)(2 * b + 1) * a.M_stride + t];
        }
      }
      tok_quad<TYPE, DUMP>(raw, sa, b0, b1, tk[u][nt]);
    }
  }
  __syncthreads();
  const KvTab kv = kv_tab();
  auto tile_step = [&](int i, const RawBlk* w) {
    const int n0 = 16 * ((int)blockIdx.x + G * i);
    sk_v4f acc[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[nt] = sk_v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      const int q = wave + W * u;
      quad_product<TYPE, NT, DUMP>(a, w[u], q, q < nq, n0 + c, &tab, kv, tk[u], acc);
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (!DUMP) {
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int r = 0; r < 4; ++r) part[i & 1][wave][nt * 4 + r][lane] = acc[nt][r];
      __syncthreads();
      store_tiles<NT, NT, W>(a, part[i & 1], n0, wave);
    }
  };
  int i = 0;
  for (; i + 1 < steps; i += 2) {
    fetch(i + 1, nxt);
    __builtin_amdgcn_sched_barrier(0);
    tile_step(i, cur);
    fetch(i + 2, cur);
    __builtin_amdgcn_sched_barrier(0);
    tile_step(i + 1, nxt);
  }
  if (i < steps) tile_step(i, cur);
}

template <int TYPE, int RT, int NT, bool DUMP>
static hipError_t skinny_go(const SkinnyArgs& a, hipStream_t s) {
  constexpr int W = 4, PF = 2;
  skinny_kernel<TYPE, RT, NT, W, PF, DUMP><<<dim3((unsigned)((a.w.rows + 16 * RT - 1) / (16 * RT))), dim3(64 * W), 0, s>>>(a);
  return hipGetLastError();
}

template <int TYPE, int NT, int CH, bool DUMP>
static hipError_t skinny_sweep_go(const SkinnyArgs& a, hipStream_t s) {
  constexpr int W = 8;
  static const int cus = [] {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        n < 1)
      n = 256;
    return n;
  }();
  const int ntile = (a.w.rows + 15) / 16;
  skinny_sweep_kernel<TYPE, NT, W, CH, DUMP><<<dim3((unsigned)(ntile < cus ? ntile : cus)), dim3(64 * W), 0, s>>>(a);
  return hipGetLastError();
}

// Most quads per wave of the sweep kernel whose registers fit without spilling (per-16-scale types need more)
template <int TYPE>
constexpr int skinny_max_ch(int nt) { return kHalves<TYPE> && nt == 2 ? 3 : TYPE == T_Q6_K ? 4 : 5; }

template <int TYPE, int NT, bool DUMP>
static hipError_t skinny_sweep_ch(int ch, const SkinnyArgs& a, hipStream_t s) {
  if (ch == 1) return skinny_sweep_go<TYPE, NT, 1, DUMP>(a, s);
  if (ch == 2) return skinny_sweep_go<TYPE, NT, 2, DUMP>(a, s);
  if (ch == 3) return skinny_sweep_go<TYPE, NT, 3, DUMP>(a, s);
  if constexpr (skinny_max_ch<TYPE>(NT) >= 4)
    if (ch == 4) return skinny_sweep_go<TYPE, NT, 4, DUMP>(a, s);
  if constexpr (skinny_max_ch<TYPE>(NT) >= 5)
    if (ch == 5) return skinny_sweep_go<TYPE, NT, 5, DUMP>(a, s);
  return hipErrorInvalidValue;  // (the route never asks)
}

// The sweep takes matrices of more than two row tiles per CU (below that its prologue costs more than it saves: 4096 x 5120,
// 16 tokens, 7.2 against 6.5 us; at 17408 rows 19.5 against 26.7) whose row fits its waves' registers.
template <int TYPE>
constexpr bool skinny_sweeps(int M, int rows, int K) {
  return rows > 8192 && (K / 128 + 7) / 8 <= skinny_max_ch<TYPE>(M <= 16 ? 1 : 2);
}

// Two row tiles per work-group halve the token traffic from 9 tokens on (IQ4_XS 17408 -> 5120, 16 tokens: 31.7 -> 26.8 us; at
// 8 tokens 25.6 against 24.7); the per-16-scale types' two tiles spill (Q6_K 89 us against 65 at 32 tokens).
template <int TYPE, bool DUMP>
static hipError_t skinny_route(const SkinnyArgs& a, hipStream_t s) {
  if (skinny_sweeps<TYPE>(a.M, a.w.rows, a.w.K)) {
    const int ch = (a.w.K / 128 + 7) / 8;
    return a.M <= 16 ? skinny_sweep_ch<TYPE, 1, DUMP>(ch, a, s) : skinny_sweep_ch<TYPE, 2, DUMP>(ch, a, s);
  }
  if (a.M > 16) return skinny_go<TYPE, 1, 2, DUMP>(a, s);
  if constexpr (!kHalves<TYPE>)
    if (a.M > 8 && a.w.rows > 4096) return skinny_go<TYPE, 2, 1, DUMP>(a, s);
  return skinny_go<TYPE, 1, 1, DUMP>(a, s);
}

// Which calls the few-token kernels take. Decode (T <= 8): from 5 tokens on always (1.2-3.3 x the GEMV's time before). 3 and
// 4 tokens: rows past 16384, where the GEMV splits its tokens over launches (5120 x 17408: IQ4_XS 41.9 -> 22.4 us, Q4_K 34.8 ->
// 25.8, Q8_0 37.7 -> 34.0; Q2_K, with mins per 16, only at four: 33.9 -> 30.9, at three 28.4 against 30.9; past 32768 the GEMV takes two tokens at most), and the types of 16-byte records up to 8192 rows of at most 5120 (4096 x 4096: 7.3 -> 5.5 us; the
// others' heavier decode leaves them level or behind: Q8_0 512 x 5120 6.6 against 7.1, Q6_K 1024 x 1024 3.6 against 3.75).
// Prompts: up to 16 tokens always (1.2-5.7 x); 17 to 32 unless the matrix is too large for one-tile work-groups to fit the
// chip in a round or two and its rows too long for the sweep (17408 x 8192: IQ4_XS 54.5 against 63.0 us; Q6_K 89.6 against 84.7,
// kept: its prompt kernel is slower).
// Q8_0 prompts, whose int8 kernel decodes nothing: not from 24 tokens on at 4096 rows and more of over 2560 (31 x 4096 -> 4560 17.6 us
// against 15.3), nor past 8192 rows of over 3072 where that kernel's K halves fill the chip once (20 x 3584 -> 15504 18.9 against 16.7,
// 13 x 9216 -> 8304 34.8 against 27.6, 5 x 11264 -> 12640 43.1 against 32.8; but 9 x 7424 -> 22672, 178 column tiles, 35.8 against 41.9,
// 9 x 4864 -> 10400, 82, 14.0 against 17.8).
inline bool skinny_takes_q8(int M, int rows, int K) {
  const int tiles = (rows + 127) / 128;
  if (rows <= 8192) return M < 24 || rows <= 4096 || K <= 2560;
  return K <= 3072 || (M <= 16 && (tiles > 128 || (K <= 5120 && tiles < 96)));
}

template <int TYPE>
bool skinny_takes(bool prompt, int M, int rows, int K) {
  if (M > kSkinnyMax || M < 3) return prompt && M < 3;
  if (prompt && TYPE == T_Q8_0) return skinny_takes_q8(M, rows, K);
  if (prompt) return M <= 16 || kHalves<TYPE> || rows <= 8192 || skinny_sweeps<TYPE>(M, rows, K);
  return M >= 5 || (K > 16384 && (M == 4 || K > 32768 || !kMin16<TYPE>)) || (Traits<TYPE>::QB == 16 && rows <= 8192 && K <= 5120);
}

template <int TYPE>
hipError_t skinny_dispatch(const SkinnyArgs& a, hipStream_t s) {
  return a.dbg_isum ? skinny_route<TYPE, true>(a, s) : skinny_route<TYPE, false>(a, s);
}

}  // namespace qm
