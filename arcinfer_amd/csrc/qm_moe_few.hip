// Expert products of an MoE layer with few experts, or few tokens, on the chip: the quad scheme of qm_skinny_impl.h over the
// slot tiles. The prompt kernels' work-groups of 128 columns x 64 slots are too few there to fill the CUs, and each walks
// the whole K alone; these cut the columns four times finer and split K.
//
// Gate and up: a work-group owns 32 columns of h (one 32-block) of one slot tile: two row tiles of gate and two of up against
// the tile's up to 32 gathered tokens, K split over its four waves; the partial sums meet in LDS, where each half-wave forms
// one slot's h = silu(g) * u over the 32 columns and quantizes it (zero/kernels/moe.cl:251-282).
// Down: a wave owns 32 output columns over the whole (short) K, a work-group 128; the routing weight is applied on the store.
// A tile of 16 slots or fewer runs with one token tile.
#include "qm_skinny_impl.h"

namespace qm {

template <int TYPE, int NT>
__device__ __forceinline__ void few_gateup(const GemmArgs& a, const typename LdsFor<TYPE>::type* tab,
                                           float (*part)[4 * 2 * 4][64], int e, int m0, int nvalid) {
  using Tr = Traits<TYPE>;
  constexpr int W = 4, PF = TYPE == T_Q6_K ? 1 : 2;  // (Q6_K spills 56 bytes with one stage, more with two)
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
  const int K = a.w.K, nb = K / 32, nq = K / 128;
  const int n0 = blockIdx.x * 32;
  const size_t row0 = (size_t)e * a.expert_rows + n0;
  const uint8_t *qg = a.w.qs + row0 * nb * Tr::QB, *hg = a.w.hdr + row0 * (nb / 8) * Tr::HB;
  const uint8_t *qu = a.w2.qs + row0 * nb * Tr::QB, *hu = a.w2.hdr + row0 * (nb / 8) * Tr::HB;
  uint32_t qoff[2], hoff[2];
#pragma unroll
  for (int rt = 0; rt < 2; ++rt) {
    const int n = 16 * rt + c;  // (expert rows are a multiple of 32)
    qoff[rt] = (uint32_t)(n * nb + g) * Tr::QB;
    hoff[rt] = (uint32_t)(n * (nb / 8)) * Tr::HB;
  }
  int tok[NT];
  const int8_t* arow[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    tok[nt] = a.rowmap[m0 + min(16 * nt + c, nvalid - 1)];
    arow[nt] = a.aq + (size_t)tok[nt] * K + 32 * g;
  }
  const int steps = wave < nq ? (nq - 1 - wave) / W + 1 : 0;
  struct Stage {
    RawBlk w[4];
    u32x4_t a[NT][2];
    float asc[NT];
  } st[PF];
  auto fetch = [&](int i, Stage& s) {
    const int q = min(wave + W * i, nq - 1);  // (past the end: the last quad again, unused)
    const uint32_t qo = (uint32_t)(4 * q * Tr::QB), ho = (uint32_t)((q >> 1) * Tr::HB);
    const int ib = 4 * (q & 1) + g;
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
      s.w[rt] = load_block_ptr<TYPE, false>(qg + qo + qoff[rt], hg + ho + hoff[rt], ib);
      s.w[2 + rt] = load_block_ptr<TYPE, false>(qu + qo + qoff[rt], hu + ho + hoff[rt], ib);
    }
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      s.a[nt][0] = *(const u32x4_t*)(arow[nt] + 128 * q);
      s.a[nt][1] = *(const u32x4_t*)(arow[nt] + 128 * q + 16);
      s.asc[nt] = a.asc[(size_t)(4 * q + g) * a.M_stride + tok[nt]];
    }
  };
#pragma unroll
  for (int p = 0; p < PF; ++p) fetch(p, st[p]);
  const KvTab kv = kv_tab();
  const SkinnyArgs unused{};
  sk_v4f acc[4][NT];
#pragma unroll
  for (int rt = 0; rt < 4; ++rt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[rt][nt] = sk_v4f{0.0f, 0.0f, 0.0f, 0.0f};
  auto step = [&](int i, const Stage& s) {
    TokQuad<TYPE> tk[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) tok_quad<TYPE, false>(s.a[nt], s.asc[nt], 0, 0, tk[nt]);
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) {
      quad_product<TYPE, NT, false>(unused, s.w[rt], wave + W * i, true, 0, tab, kv, tk, acc[rt]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  int i = 0;
  for (; i + PF <= steps; i += PF) {
#pragma unroll
    for (int p = 0; p < PF; ++p) {
      step(i + p, st[p]);
      __builtin_amdgcn_sched_barrier(0);
      fetch(i + p + PF, st[p]);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int p = 0; p < PF - 1; ++p)
    if (i + p < steps) step(i + p, st[p]);
#pragma unroll
  for (int rt = 0; rt < 4; ++rt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int r = 0; r < 4; ++r) part[wave][(rt * NT + nt) * 4 + r][lane] = acc[rt][nt][r];
  __syncthreads();
  // half-wave hw: slots hw, hw + 8, ...; its lane j: column n0 + j
  const int j = threadIdx.x & 31, hw = threadIdx.x >> 5, n = n0 + j;
#pragma unroll
  for (int s0 = 0; s0 < 16 * NT; s0 += 8) {
    const int s = s0 + hw, el = ((j >> 4) * NT + (s >> 4)) * 4 + (s & 3), ln = 16 * ((s >> 2) & 3) + (j & 15);
    float gv = part[0][el][ln], uv = part[0][2 * NT * 4 + el][ln];
#pragma unroll
    for (int k = 1; k < W; ++k) {
      gv += part[k][el][ln];
      uv += part[k][2 * NT * 4 + el][ln];
    }
    const float h = uv * (gv / (1.0f + expf(-gv)));
    const float amax = max32(fabsf(h));
    const float inv = amax > 0.0f ? 127.0f / amax : 0.0f;
    const int q = (int)__builtin_rintf(h * inv);
    if (s < nvalid) {
      a.hq[(size_t)(m0 + s) * a.ldc + n] = (int8_t)q;
      if (j == 0) a.hsc[(size_t)(n / 32) * a.slots + m0 + s] = amax / 127.0f;
    }
  }
}

template <int TYPE>
__global__ __launch_bounds__(256, 2) void moe_few_gateup_kernel(GemmArgs a) {
  __shared__ typename LdsFor<TYPE>::type tab;
  __shared__ float part[4][4 * 2 * 4][64];
  const int t = blockIdx.y;
  if (t >= a.tiles[0]) return;
  const int e = a.tiles[1 + 3 * t], m0 = a.tiles[2 + 3 * t], nvalid = a.tiles[3 + 3 * t];
  if (nvalid <= 0) return;
  lds_fill<TYPE>(&tab);
  __syncthreads();
  if (nvalid <= 16) few_gateup<TYPE, 1>(a, &tab, part, e, m0, nvalid);
  else few_gateup<TYPE, 2>(a, &tab, part, e, m0, nvalid);
}

template <int TYPE, int NT>
__device__ __forceinline__ void few_down(const GemmArgs& a, const typename LdsFor<TYPE>::type* tab, int e, int m0, int nvalid) {
  using Tr = Traits<TYPE>;
  constexpr int PF = 2;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
  const int K = a.w.K, nb = K / 32, nq = K / 128;
  const int n0 = blockIdx.x * 128 + wave * 32;
  if (n0 >= a.expert_rows) return;
  const size_t row0 = (size_t)e * a.expert_rows + n0;
  const uint8_t *qb = a.w.qs + row0 * nb * Tr::QB, *hb = a.w.hdr + row0 * (nb / 8) * Tr::HB;
  uint32_t qoff[2], hoff[2];
#pragma unroll
  for (int rt = 0; rt < 2; ++rt) {
    const int n = min(16 * rt + c, a.expert_rows - 1 - n0);
    qoff[rt] = (uint32_t)(n * nb + g) * Tr::QB;
    hoff[rt] = (uint32_t)(n * (nb / 8)) * Tr::HB;
  }
  int slot[NT];
  const int8_t* arow[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    slot[nt] = m0 + min(16 * nt + c, nvalid - 1);
    arow[nt] = a.aq + (size_t)slot[nt] * K + 32 * g;
  }
  struct Stage {
    RawBlk w[2];
    u32x4_t a[NT][2];
    float asc[NT];
  } st[PF];
  auto fetch = [&](int i, Stage& s) {
    const int q = min(i, nq - 1);
#pragma unroll
    for (int rt = 0; rt < 2; ++rt)
      s.w[rt] = load_block_ptr<TYPE, false>(qb + (uint32_t)(4 * q * Tr::QB) + qoff[rt], hb + (uint32_t)((q >> 1) * Tr::HB) + hoff[rt],
                                            4 * (q & 1) + g);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      s.a[nt][0] = *(const u32x4_t*)(arow[nt] + 128 * q);
      s.a[nt][1] = *(const u32x4_t*)(arow[nt] + 128 * q + 16);
      s.asc[nt] = a.asc[(size_t)(4 * q + g) * a.M_stride + slot[nt]];
    }
  };
#pragma unroll
  for (int p = 0; p < PF; ++p) fetch(p, st[p]);
  const KvTab kv = kv_tab();
  const SkinnyArgs unused{};
  sk_v4f acc[2][NT];
#pragma unroll
  for (int rt = 0; rt < 2; ++rt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[rt][nt] = sk_v4f{0.0f, 0.0f, 0.0f, 0.0f};
  // (K is a multiple of 256: an even number of quads)
  for (int i = 0; i < nq; i += PF) {
#pragma unroll
    for (int p = 0; p < PF; ++p) {
      TokQuad<TYPE> tk[NT];
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) tok_quad<TYPE, false>(st[p].a[nt], st[p].asc[nt], 0, 0, tk[nt]);
#pragma unroll
      for (int rt = 0; rt < 2; ++rt) {
        quad_product<TYPE, NT, false>(unused, st[p].w[rt], i + p, true, 0, tab, kv, tk, acc[rt]);
        __builtin_amdgcn_sched_barrier(0);
      }
      fetch(i + p + PF, st[p]);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int s = 16 * nt + 4 * g + r;
      if (s >= nvalid) continue;
      const float ws = a.rowscale[m0 + s];
#pragma unroll
      for (int rt = 0; rt < 2; ++rt) {
        const int n = n0 + 16 * rt + c;
        if (n < a.expert_rows) a.C[(size_t)(m0 + s) * a.ldc + n] = ws * acc[rt][nt][r];
      }
    }
}

template <int TYPE>
__global__ __launch_bounds__(256, 2) void moe_few_down_kernel(GemmArgs a) {
  __shared__ typename LdsFor<TYPE>::type tab;
  const int t = blockIdx.y;
  if (t >= a.tiles[0]) return;
  const int e = a.tiles[1 + 3 * t], m0 = a.tiles[2 + 3 * t], nvalid = a.tiles[3 + 3 * t];
  if (nvalid <= 0) return;
  lds_fill<TYPE>(&tab);
  __syncthreads();
  if (nvalid <= 16) few_down<TYPE, 1>(a, &tab, e, m0, nvalid);
  else few_down<TYPE, 2>(a, &tab, e, m0, nvalid);
}

template <int TYPE>
static hipError_t few_go(bool down, const GemmArgs& a, hipStream_t s) {
  const dim3 grid((unsigned)(down ? (a.expert_rows + 127) / 128 : a.expert_rows / 32), (unsigned)a.max_tiles);
  if (down) moe_few_down_kernel<TYPE><<<grid, dim3(256), 0, s>>>(a);
  else moe_few_gateup_kernel<TYPE><<<grid, dim3(256), 0, s>>>(a);
  return hipGetLastError();
}

// Which products come here: by the work-groups of 128 columns that the prompt kernels launch, wgs, and their decode (one pass, or two
// for the types with scales per 16 elements, s16). The two are chosen apart, from 460 layers of 8 to 256 experts, E 768 to 4096, F 256
// to 1024 and 66 to 6600 slots, each product on both (whole layers, us, old -> new); of those no layer is slower by over 3 %.
// Gate and up: up to 256 (one a CU there; IQ4_XS 8 experts of 512, E 2048, 330 slots 91 -> 57, Q6_K 8 of 256, E 1792, 118 slots 107 ->
// 48), 192 where an expert has many slots (IQ2_XXS 8 of 512, E 2048, 1812 slots, 256: 78 -> 87); to 320 where tiles are few, narrow or
// nearly empty, or the prompt kernels run twice (but Q6_K 64 of 512, E 4096, 222 slots, 280: 155 -> 183). Q8_0, whose stream is
// twice as long, to 128 (32 of 512, E 2048, 96 slots, 140: 67 -> 73), to 160 with over four slots an expert.
static bool s16(int t) { return t == T_Q6_K || t == T_Q3_K || t == T_IQ2_XS || t == T_IQ2_S; }
static int few_tiles(int slots, int NE) { return (slots < NE ? slots : NE) + slots / kMoeTileRows; }

bool moe_few(int type, int slots, int NE, int E, int Fv) {
  const int tiles = few_tiles(slots, NE), wgs = (Fv + 127) / 128 * tiles;
  if (wgs > 192 && slots > 16 * NE) return false;
  if (type == T_Q8_0) return wgs < 128 || (wgs <= 160 && slots > 4 * NE);
  if (wgs <= 256 || wgs > 320) return wgs <= 256;
  if (s16(type)) return type != T_Q6_K || E < 2048 || tiles <= 52 || slots <= 2 * NE;
  return tiles <= 52 || Fv <= 256 || slots <= 4 * NE;
}

// Down, IQ4_XS 32 of 512, E 1024, 160 slots, 296: 66 -> 52; the prompt kernels catch up with more work-groups (E 4096, 1302 slots,
// 2304: 137 -> 144) and longer rows (32 of 1024, E 2048, 220 slots, 608: Q8_0 90 -> 111; but 8 of 1024, E 1280, 164 slots, 130: IQ3_S
// 72 -> 65).
bool moe_few_down(int type, int slots, int NE, int E, int F) {
  const int wgs = (E + 127) / 128 * few_tiles(slots, NE);
  if (s16(type)) return wgs <= (slots > 16 * NE ? 256 : 200);
  if (type == T_Q8_0) return wgs <= (F <= 512 ? 550 : F <= 768 ? 750 : 0);
  return wgs <= 200 || (F <= 768 && (wgs <= 850 || (wgs <= (F > 512 ? 1600 : 1100) && slots <= 16 * NE)));
}

hipError_t launch_moe_few(int type, bool down, const GemmArgs& a, hipStream_t s) {
  switch (type) {
    case T_Q8_0: return few_go<T_Q8_0>(down, a, s);
    case T_Q4_0: return few_go<T_Q4_0>(down, a, s);
    case T_IQ4_NL: return few_go<T_IQ4_NL>(down, a, s);
    case T_Q2_0: return few_go<T_Q2_0>(down, a, s);
    case T_IQ4_XS: return few_go<T_IQ4_XS>(down, a, s);
    case T_IQ3_S: return few_go<T_IQ3_S>(down, a, s);
    case T_IQ3_XXS: return few_go<T_IQ3_XXS>(down, a, s);
    case T_IQ2_XXS: return few_go<T_IQ2_XXS>(down, a, s);
    case T_IQ2_XS: return few_go<T_IQ2_XS>(down, a, s);
    case T_IQ2_S: return few_go<T_IQ2_S>(down, a, s);
    case T_Q6_K: return few_go<T_Q6_K>(down, a, s);
    case T_Q3_K: return few_go<T_Q3_K>(down, a, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace qm
