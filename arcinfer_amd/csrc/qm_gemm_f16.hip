// Prompt GEMM on the f16 matrix pipe for the types whose per-block weight scale is an integer and whose block values
// times that scale fit an f16 exactly (Q4_K: sc * q <= 63 * 15 = 945 < 2048).
//
// The reference's product (zero/kernels/gemm.cl:367-398) is, per token m, weight row n, 32-block b and superblock s,
//   I[m,n,b] = sc[n,b] * sum_k a[m,k] q[n,k]                  (the int32 block sum times the integer block scale)
//   tq  = sum_b fma(asc[m,b], I, .)        tmn = sum_b fma(asc[m,b], mn[n,b] * bsum[m,b], .)     (Q4_K mins)
//   res = fma(d[n,s], tq, fma(-dmin[n,s], tmn, res))
// Here I comes from two v_mfma_f32_32x32x16_f16 per block and 32 x 32 tile: the weights are decoded to sc * q in f16
// and the activations are their int8 values in f16, so every product is exact and the f32 sum of 32 of them
// (|I| <= 32 * 127 * 945 < 2^24) is the exact integer. The per-block activation scale is then applied with one f32 fma
// per element, as the reference does; with tokens on the MFMA's columns, asc is one value per lane. tmn is one bf16
// MFMA per superblock (asc * bsum split into two bf16 parts, 16 bits; mn exact), and d, dmin are applied once per
// superblock in the reference's order. Q5_K: kF16Centred.
//
// Work-group: 4 waves, a tile of 128 weight rows x 128 tokens; wave w owns weight rows 32w..32w+31 (one MFMA row
// tile, decoded once per block in registers) for all 128 tokens (four 32-token column tiles). Two work-groups per CU,
// so one wave's scaling and decoding overlaps the other wave's MFMAs. The activations (f16, written by a prepass in
// MFMA operand order) are staged in LDS a block pair at a time, one pair ahead.
// MFMA orientation: A = weights (rows: weight rows n), B = activations (columns: tokens m).
// 32x32 result layout: lane l holds column l % 32 and rows 8 * (r / 4) + 4 * (l / 32) + r % 4, r = 0..15.
#include <stdlib.h>

#include <mutex>

#include "qm_decode.h"
#include "qm_launch.h"

namespace qm {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kF16BM = 128;                        // tokens per work-group tile
constexpr int kF16BN = 128;                        // weight rows per work-group tile
constexpr int kF16Piece = 1024;                    // one MFMA operand piece of a 32-token tile: 64 lanes x 16 bytes
constexpr int kF16PairTile = 4 * kF16Piece;        // per 32-token tile and block pair: (block, chunk) pieces
constexpr int kF16PairBytes = 4 * kF16PairTile;    // per 128-token tile and block pair (16 KB)

// Element order inside a lane's 8-value f16 operand: the weight decode turns a word of nibble bytes t0..t3 into the
// f16 pairs (t0, t2), (t1, t3), so operand position i holds element 8h + f16_perm8(i) of its 16-element chunk.
__host__ __device__ constexpr int f16_perm8(int i) { return (i & 4) | ((i & 1) << 1) | ((i >> 1) & 1); }

static size_t round_up(size_t v, size_t a) { return (v + a - 1) / a * a; }

// Workspace of one call (device bytes), for M tokens and K columns: the f16 activations, then the mins operand (Q5_K: twice,
// kF16Centred).
size_t f16_workspace_bytes(int type, int M, int K) {
  const size_t Mp = round_up((size_t)M, kF16BM);
  return round_up(Mp * (size_t)K * 2, 256) + Mp * (size_t)(K / 32) * (type == T_Q5_K ? 8 : 4);
}

// The types of this kernel: Q4_K (Q5_K's and IQ3_S's values times their integer block scales fit an f16 exactly too: 31 * 63 =
// 1953, 15 * 31 = 465). kF16Half: see f16_act_kernel.
template <int TYPE> constexpr bool kF16Half = TYPE == T_Q5_K || TYPE == T_IQ3_S;

// Q5_K: values less 16, and the 16 in the min term: d sc q - dmin mn = d sc (q - 16) + kappa, kappa = 16 d sc - dmin mn. Weights
// without a mean times activations with one make d sc q and dmin mn cancel almost wholly, and what is rounded before they meet
// shows; q - 16 and kappa are small by themselves. kappa and u = asc * bsum enter the matrix pipe as three bf16 parts each, 24
// bits, what the int8 kernel of Q5_K's shorter products holds them in (per-256 scales: u = bsum, exact in two parts). Error of
// 500 x 5376 -> 4624 on such rows 3.3e-7 (the int8 kernel 6.3e-7; q, mn and two parts of u 2.3e-5, with three 1.4e-6), on random
// ones a third of the int8 kernel's. 2048 x 5120 -> 17408: 697 us against 683 of two parts and 806 of int8; 333 x 17408 -> 5120
// 143.5, 146.5, 157 (the parts lie by superblock, 1 KB a load, where rows of them took a cache line each).
template <int TYPE> constexpr bool kF16Centred = TYPE == T_Q5_K;

// ---- prepass: the int8 activations as f16 in MFMA operand order, and (MINS) the mins operand u = asc * bsum split
// into two bf16 parts (one 32-bit word per token and block: bf16 hi | lo << 16; per superblock the 8 words are the
// bf16 MFMA's B operand, slot 8h + i = block 4h + i / 2, part i % 2). CENTRED: both parts of all tokens by superblock; PARTS = 3: u2
// has the first and the third part the same way. asc null: u = bsum.
// One thread per (token, 32-block, k-half h); consecutive threads take consecutive lanes of one operand piece
// (token % 32, then h), so each wave writes whole 1 KB pieces. A thread writes lane (token % 32, h)'s 16 bytes of the
// block's two pieces: chunk c = 0 holds elements 8h + perm8(i), chunk 1 elements 16 + 8h + perm8(i).
// HALF: lane half h holds the 16 elements of half h (chunk c: 16h + 8c + perm8(i)) instead, for the types whose records keep
// a half together (kF16Half).
template <int PARTS, bool HALF, bool CENTRED>
__global__ __launch_bounds__(256) void f16_act_kernel(const int8_t* aq, const float* asc, const int16_t* absum, int M,
                                                      int M_stride, int ash, int Mp, int K, uint8_t* af, uint32_t* u,
                                                      uint32_t* u2) {
  const int nb = K / 32;
  const size_t gid = (size_t)blockIdx.x * 256 + threadIdx.x;
  const int lanei = (int)(gid & 63), h = lanei >> 5;
  const int b = (int)((gid >> 6) % nb), mtile = (int)((gid >> 6) / nb);
  const int m = mtile * 32 + (lanei & 31);
  if (m >= Mp) return;
  uint32_t hw[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  if (m < M) {
    const int8_t* src = aq + (size_t)m * K + 32 * b;
    const uint2 q0 = *(const uint2*)(src + (HALF ? 16 : 8) * h), q1 = *(const uint2*)(src + (HALF ? 8 + 16 * h : 16 + 8 * h));
    const uint32_t qw[4] = {q0.x, q0.y, q1.x, q1.y};
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int i = 0; i < 8; i += 2) {
        uint32_t pr = 0;
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const int e = f16_perm8(i + t);  // element 16c + 8h + e (HALF: 16h + 8c + e)
          const int8_t qv = (int8_t)(qw[2 * c + (e >> 2)] >> (8 * (e & 3)));
          pr |= (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)qv) << (16 * t);
        }
        hw[4 * c + i / 2] = pr;
      }
  }
  // destination: [m / 128][pair b / 2][token tile (m % 128) / 32][piece 2 * (b % 2) + c][lane][16 B]
  uint8_t* base = af + ((size_t)(m / kF16BM) * (K / 64) + b / 2) * kF16PairBytes + ((m % kF16BM) / 32) * kF16PairTile +
                  (2 * (b & 1)) * kF16Piece + lanei * 16;
  *(uint4*)(base) = make_uint4(hw[0], hw[1], hw[2], hw[3]);
  *(uint4*)(base + kF16Piece) = make_uint4(hw[4], hw[5], hw[6], hw[7]);
  if constexpr (PARTS > 0) {
    if (h == 0) {
      float uv = 0.0f;
      if (m < M) {
        const int bs = (int)absum[(size_t)(2 * b) * M_stride + m] + (int)absum[(size_t)(2 * b + 1) * M_stride + m];
        uv = asc ? asc[(size_t)(b >> ash) * M_stride + m] * (float)bs : (float)bs;
      }
      const __bf16 uh = (__bf16)uv;
      const __bf16 ul = (__bf16)(uv - (float)uh);
      const size_t at = CENTRED ? ((size_t)(b >> 3) * Mp + m) * 8 + (b & 7) : (size_t)m * nb + b;
      u[at] =
          (uint32_t)__builtin_bit_cast(uint16_t, uh) | ((uint32_t)__builtin_bit_cast(uint16_t, ul) << 16);
      if constexpr (PARTS == 3)
        u2[at] = (uint32_t)__builtin_bit_cast(uint16_t, uh) |
                 ((uint32_t)__builtin_bit_cast(uint16_t, (__bf16)(uv - (float)uh - (float)ul)) << 16);
    }
  }
}

// ---- the GEMM

struct F16Args {
  WView w;
  const uint8_t* af;   // prepass output
  const uint32_t* u;   // mins operand
  const uint32_t* u2;  // (three parts: the first and third)
  const float* asc;
  int M, M_stride, Mp;  // (Mp: M rounded up to whole tiles)
  int ash;             // asc row of 32-block b: b >> ash (per-32 scales: 0; per-256: 3)
  float* C;
  int ldc, c_off, accumulate;
  float* part;         // partial tiles of the cut tiles (tiles from split_from on, in `splits` pieces of K), or null
  int split_from, splits;
  int32_t* dbg_isum;   // non-null: write the exact block sums sc * isum [M][rows][K/32] instead of C
};

// one VALU op: (x & mask) | c
__device__ __forceinline__ uint32_t and_or(uint32_t x, uint32_t mask, uint32_t c) {
  uint32_t r;
  asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(x), "s"(mask), "v"(c));
  return r;
}

// Q4_K: the lane's 16 values of one 32-block (payload bytes 8h..8h+7: x, y) times the integer block scale, as two
// f16 operands: chunk 0 the low nibbles (elements 8h + perm8(i)), chunk 1 the high nibbles (16 + 8h + perm8(i)).
// (1024 + q) as f16 is the bit pattern 0x6400 | q; one packed fma makes (1024 + q) sc - 1024 sc = sc q exactly. The
// high nibbles are not shifted down: left in mantissa bits 4-7 under the exponent of 16384 (0x7400 | q << 4) they
// read as 16384 + 256 q, and (16384 + 256 q) (sc / 256) - 64 sc = sc q exactly too (sc / 256 and 64 sc are exact in
// f16, and the fused multiply-add rounds only its exact integer result).
__device__ __forceinline__ void q4k_f16_decode(uint32_t x, uint32_t y, int sc, uint32_t c64, f16x8& b0, f16x8& b1) {
  const _Float16 s = (_Float16)sc;
  const f16x2 sc2 = {s, s}, off2 = {(_Float16)(-1024.0f) * s, (_Float16)(-1024.0f) * s};
  const _Float16 sh = s * (_Float16)0.00390625f;  // sc / 256
  const f16x2 sch2 = {sh, sh}, offh2 = {(_Float16)(-64.0f) * s, (_Float16)(-64.0f) * s};
  const uint32_t m = 0x000F000Fu, mh = 0x00F000F0u, c74 = 0x74007400u;
  const uint32_t x8 = x >> 8, y8 = y >> 8;
  const uint32_t w[8] = {and_or(x, m, c64), and_or(x8, m, c64), and_or(y, m, c64), and_or(y8, m, c64),
                         and_or(x, mh, c74), and_or(x8, mh, c74), and_or(y, mh, c74), and_or(y8, mh, c74)};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const f16x2 v0 = __builtin_bit_cast(f16x2, w[i]) * sc2 + off2;
    const f16x2 v1 = __builtin_bit_cast(f16x2, w[4 + i]) * sch2 + offh2;
    b0[2 * i] = v0[0];
    b0[2 * i + 1] = v0[1];
    b1[2 * i] = v1[0];
    b1[2 * i + 1] = v1[1];
  }
}

// A lane's share of a 32-block: Q4_K its 8 nibble bytes (x y); Q5_K the 8 nibble bytes of its half and the word of fifth bits
// (z); IQ3_S the four index bytes of its half (x) and the block's sign bytes (y)
struct F16Pay {
  uint32_t x, y, z;
};
template <int TYPE>
__device__ __forceinline__ F16Pay f16_load(const uint8_t* qrow, int blk, int h) {
  const uint8_t* r = qrow + (size_t)blk * Traits<TYPE>::QB;
  if constexpr (TYPE == T_IQ3_S) {
    return F16Pay{*(const uint32_t*)(r + 4 * h), *(const uint32_t*)(r + 8), 0u};
  } else {
    const uint2 v = *(const uint2*)(r + 8 * h);
    return F16Pay{v.x, v.y, TYPE == T_Q5_K ? *(const uint32_t*)(r + 16) : 0u};
  }
}

// Block b (0..7) of a superblock with header hdr: the lane's 16 values times the integer block scale, as the two f16 operands
// (CENTRED: values less 16)
template <int TYPE, bool CENTRED>
__device__ __forceinline__ void f16_decode(const F16Pay& p, uint4 hdr, int b, int h, const typename LdsFor<TYPE>::type* tab,
                                           f16x8& b0, f16x8& b1) {
  if constexpr (TYPE == T_Q4_K) {
    int sc, mn;
    q4k_scale_min(hdr.y, hdr.z, hdr.w, b, sc, mn);
    (void)mn;
    q4k_f16_decode(p.x, p.y, sc, 0x64006400u, b0, b1);
  } else {
    // words w[k] of bytes u (elements 16h + 4k ..): IQ3_S (1024 + u) as f16 is 0x6400 | u, and (1024 + u) sc - (1024 + bias) sc is
    // exact as in q4k_f16_decode (bias 128 takes the signed bytes, flipped to unsigned, back). Q5_K u = 4 q under the exponent of
    // 256, 0x5C00 | 4 q, where the offset less 16 fits too: (256 + q) sc - 272 sc, and 272 * 63 = 17136 is an f16 (1040 * 63 is not)
    uint32_t w[4];
    int sc;
    if constexpr (TYPE == T_Q5_K) {
      int mn;
      q4k_scale_min(hdr.y, hdr.z, hdr.w, b, sc, mn);
      (void)mn;
      const uint32_t hb = p.z >> (4 * h);
      w[0] = ((p.x << 2) & 0x3C3C3C3Cu) | ((hb & 0x01010101u) << 6);
      w[1] = ((p.y << 2) & 0x3C3C3C3Cu) | ((hb & 0x02020202u) << 5);
      w[2] = ((p.x >> 2) & 0x3C3C3C3Cu) | ((hb & 0x04040404u) << 4);
      w[3] = ((p.y >> 2) & 0x3C3C3C3Cu) | ((hb & 0x08080808u) << 3);
    } else {
      const uint32_t qh = ((b < 4 ? hdr.x : hdr.y) >> (8 * (b & 3) + 4 * h)) & 0xFu, sg = p.y >> (16 * h);
      sc = 1 + 2 * (int)((hdr.z >> (4 * b)) & 0xFu);
      const uint4 m0 = tab->sgn[sg & 0xFFu], m1 = tab->sgn[(sg >> 8) & 0xFFu];
      w[0] = (tab->grid[(p.x & 0xFFu) | ((qh << 8) & 256u)] ^ m0.x) + m0.z;
      w[1] = (tab->grid[((p.x >> 8) & 0xFFu) | ((qh << 7) & 256u)] ^ m0.y) + m0.w;
      w[2] = (tab->grid[((p.x >> 16) & 0xFFu) | ((qh << 6) & 256u)] ^ m1.x) + m1.z;
      w[3] = (tab->grid[(p.x >> 24) | ((qh << 5) & 256u)] ^ m1.y) + m1.w;
#pragma unroll
      for (int k = 0; k < 4; ++k) w[k] ^= 0x80808080u;
    }
    constexpr uint32_t hi = TYPE == T_IQ3_S ? 0x64646464u : 0x5C5C5C5Cu;
    const _Float16 s = (_Float16)sc, o = (_Float16)(TYPE == T_IQ3_S ? -1152.0f : CENTRED ? -272.0f : -256.0f) * s;
    const f16x2 sc2 = {s, s}, off2 = {o, o};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const f16x2 v0 = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(hi, w[k], 0x04020400u)) * sc2 + off2;
      const f16x2 v1 = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(hi, w[k], 0x04030401u)) * sc2 + off2;
      f16x8& d = k < 2 ? b0 : b1;
      const int i = 4 * (k & 1);
      d[i] = v0[0];
      d[i + 1] = v0[1];
      d[i + 2] = v1[0];
      d[i + 3] = v1[1];
    }
  }
}

__device__ __forceinline__ uint32_t bf16_pair(float lo, float hi) {
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, bf16x2{(__bf16)lo, (__bf16)hi});
}

// Work-group -> (128-row weight tile, 128-token tile, K piece); consecutive work-groups of one XCD (work-groups are dealt to
// the 8 XCDs round-robin) take neighbouring weight tiles of one token tile, so the token tile stays in that XCD's L2.
// Returns the index of the piece among the cut tiles' pieces, or -1 for a whole tile.
template <bool CUT>
__device__ __forceinline__ int f16_tile(const F16Args& a, int& nt, int& mt) {
  const int gx = (a.w.rows + kF16BN - 1) / kF16BN;
  int lin = blockIdx.x, piece = -1;
  const int whole = CUT ? a.split_from : (int)gridDim.x;
  if (CUT && lin >= whole) {
    piece = lin - whole;
    lin = whole + piece / a.splits;
  } else if (whole % 8 == 0) {
    lin = (lin % 8) * (whole / 8) + lin / 8;
  }
  mt = lin / gx;
  nt = lin % gx;
  return piece;
}

// S256: per-256 activation scales (the reference's act32 = false, gemm.cl:413-447): one scale per token and superblock,
// so the f16 MFMAs accumulate the whole superblock's products (sum_b sc * isum, in f32: exact while the partial sums
// stay below 2^24, i.e. for all but extreme rows, and within f32 rounding otherwise) and the scale is applied once per
// superblock, res = fma(d * asc, I, fma(-dmin, tmn, res)) -- no per-block VALU work.
template <int TYPE, bool DUMP, bool S256 = false, bool CUT = false>
__global__ __launch_bounds__(256, 2) void gemm_f16_kernel(F16Args a) {
  // two activation stages of 16 KB, reused at the end to transpose the result tiles (4 waves x 32 x 33 floats)
  __shared__ __attribute__((aligned(16))) uint8_t lds[2 * kF16PairBytes];
  __shared__ float dtab[4][2][32];  // per wave: d and dmin of its 32 rows (current superblock)
  __shared__ float sasc[2][2][kF16BM];  // per stage: the activation scales of the pair's two blocks, [block][token]
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, h = lane >> 5, lc = lane & 31;
  const int K = a.w.K, nb = K / 32, nsb = K / 256, npair = K / 64;
  int nt, mt;
  const int piece = f16_tile<CUT>(a, nt, mt);
  const int z = CUT && piece >= 0 ? piece % a.splits : 0, nz = CUT && piece >= 0 ? a.splits : 1;
  const int sb0 = z * nsb / nz, sb1 = (z + 1) * nsb / nz;  // (its piece of a cut tile, or all superblocks)
  const int m0 = mt * kF16BM;
  const int n_rows = a.w.rows;
  const int nbase = nt * kF16BN + wave * 32;
  const int nrow = min(nbase + lc, n_rows - 1);  // this lane's A-operand row
  constexpr bool CENTRED = kF16Centred<TYPE> && !DUMP, MINS = Traits<TYPE>::MINS && !CENTRED;
  static_assert(Traits<TYPE>::HB == 16, "16-byte headers");
  __shared__ typename LdsFor<TYPE>::type tab;
  lds_fill<TYPE>(&tab);
  const uint8_t* qrow = a.w.qs + (size_t)nrow * nb * Traits<TYPE>::QB;
  const uint8_t* hrow = a.w.hdr + (size_t)nrow * nsb * 16;
  const uint8_t* abase = a.af + (size_t)mt * npair * kF16PairBytes;

  // activation staging: 16 KB per block pair, 4 x 16 bytes per thread
  u32x4_t st[4];
  auto fetch = [&](int g) {
#pragma unroll
    for (int c = 0; c < 4; ++c) st[c] = *(const u32x4_t*)(abase + (size_t)g * kF16PairBytes + (tid + 256 * c) * 16);
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int c = 0; c < 4; ++c) *(u32x4_t*)(lds + buf * kF16PairBytes + (tid + 256 * c) * 16) = st[c];
  };
  // activation scales of a block pair, staged with its activations: thread tid takes block tid / 128, token tid % 128
  float st_sc;
  const int sc_row = min(m0 + (tid & (kF16BM - 1)), a.M - 1);
  // (the block-sum mode has no activation scales: a.asc is null there and is never read)
  auto fetch_sa = [&](int g) {
    if constexpr (!DUMP) st_sc = a.asc[(size_t)((2 * g + (tid >> 7)) >> a.ash) * a.M_stride + sc_row];
  };
  auto store_sa = [&](int buf) {
    if constexpr (!DUMP) sasc[buf][tid >> 7][tid & (kF16BM - 1)] = st_sc;
  };

  f32x16 tq[4], res[4];
  float sv256[4];  // S256: the superblock's activation scale of each token tile
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) res[t][r] = 0.0f;
  const f32x16 zero16 = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};

  uint4 hdr = *(const uint4*)(hrow + (size_t)sb0 * 16), hdr_n;
  F16Pay pay[2], pay_n[2];
#pragma unroll
  for (int bb = 0; bb < 2; ++bb) pay[bb] = f16_load<TYPE>(qrow, 8 * sb0 + bb, h);
  fetch_sa(4 * sb0);
  fetch(4 * sb0);
  store(0);
  store_sa(0);
  __syncthreads();

  for (int s = sb0; s < sb1; ++s) {
    const int sn = s + 1 < sb1 ? s + 1 : s;
    hdr_n = *(const uint4*)(hrow + (size_t)sn * 16);
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const int g = 4 * s + p, cur = g & 1;
      const int gn = g + 1 < 4 * sb1 ? g + 1 : g;
      fetch(gn);
#pragma unroll
      for (int bb = 0; bb < 2; ++bb) pay_n[bb] = f16_load<TYPE>(qrow, 2 * gn + bb, h);
      fetch_sa(gn);
      // (keeps the loads here: issued a whole pair of MFMA work before their data is needed)
      __builtin_amdgcn_sched_barrier(0);
      f16x8 aw[2][2];
#pragma unroll
      for (int bb = 0; bb < 2; ++bb) f16_decode<TYPE, CENTRED>(pay[bb], hdr, 2 * p + bb, h, &tab, aw[bb][0], aw[bb][1]);
      const uint8_t* L = lds + cur * kF16PairBytes + lane * 16;
      if constexpr (S256) {
        // items block-major (k = 4 bb + t): consecutive MFMAs feed different token tiles' accumulators
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const int t = k & 3, bb = k >> 2;
          const uint8_t* Lt = L + t * kF16PairTile;
          const f16x8 b0 = *(const f16x8*)(Lt + (2 * bb) * kF16Piece);
          const f16x8 b1 = *(const f16x8*)(Lt + (2 * bb + 1) * kF16Piece);
          const f32x16 c = (p == 0 && bb == 0) ? zero16 : tq[t];
          tq[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(aw[bb][0], b0, c, 0, 0, 0);
          tq[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(aw[bb][1], b1, tq[t], 0, 0, 0);
        }
      } else {
        // items k = (token tile t, block bb), t = k / 2, bb = k % 2. Stage k: item k's first MFMA, item k + 1's
        // operands read from LDS, half of item k - 1's scaling fmas, item k's second MFMA (it accumulates onto the
        // first, so it waits for it: the eight fmas fill that wait), the other half of the fmas. One MFMA result is in
        // flight while the previous one is consumed, and the next item's LDS round trip runs under both (605 -> 579 ->
        // 561 us on the 2048 x 5120 x 17408 shape for the operand prefetch and then the split fmas, A/B in one process).
        f32x16 Iprev;
        f16x8 nb0 = *(const f16x8*)(L), nb1 = *(const f16x8*)(L + kF16Piece);  // (item 0)
        float nsv = DUMP ? 0.0f : sasc[cur][0][lc], svprev = 0.0f;
#pragma unroll
        for (int k = 0; k <= 8; ++k) {
          f32x16 Icur;
          float svcur = 0.0f;
          const int bb = k & 1;
          const f16x8 b1 = nb1;
          if (k < 8) {
            const f16x8 b0 = nb0;
            svcur = nsv;
            Icur = __builtin_amdgcn_mfma_f32_32x32x16_f16(aw[bb][0], b0, zero16, 0, 0, 0);
            if (k + 1 < 8) {
              const int t1 = (k + 1) >> 1, bb1 = (k + 1) & 1;
              const uint8_t* Lt = L + t1 * kF16PairTile;
              nb0 = *(const f16x8*)(Lt + (2 * bb1) * kF16Piece);
              nb1 = *(const f16x8*)(Lt + (2 * bb1 + 1) * kF16Piece);
              if constexpr (!DUMP) nsv = sasc[cur][bb1][32 * t1 + lc];
            }
          }
          __builtin_amdgcn_sched_barrier(0);
          const int tp = (k - 1) >> 1, bbp = (k - 1) & 1;
          if constexpr (!DUMP) {
            if (k > 0) {
#pragma unroll
              for (int r = 0; r < 8; ++r)
                tq[tp][r] = (p == 0 && bbp == 0) ? svprev * Iprev[r] : fmaf(svprev, Iprev[r], tq[tp][r]);
            }
          }
          __builtin_amdgcn_sched_barrier(0);
          if (k < 8) Icur = __builtin_amdgcn_mfma_f32_32x32x16_f16(aw[bb][1], b1, Icur, 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
          if (k > 0) {
            if constexpr (DUMP) {
              const int m = m0 + 32 * tp + lc, blk = 8 * s + 2 * p + bbp;
#pragma unroll
              for (int r = 0; r < 16; ++r) {
                const int n = nbase + 8 * (r >> 2) + 4 * h + (r & 3);
                if (m < a.M && n < n_rows) a.dbg_isum[((size_t)m * n_rows + n) * nb + blk] = (int)Iprev[r];
              }
            } else {
#pragma unroll
              for (int r = 8; r < 16; ++r)
                tq[tp][r] = (p == 0 && bbp == 0) ? svprev * Iprev[r] : fmaf(svprev, Iprev[r], tq[tp][r]);
              // (pins the scaled sums here: otherwise the compiler defers every fma to the superblock end and keeps
              // each block's MFMA result alive meanwhile, in scratch memory)
#pragma unroll
              for (int r = 0; r < 16; ++r) asm volatile("" : "+v"(tq[tp][r]));
            }
          }
          if (k < 8) {
            Iprev = Icur;
            svprev = svcur;
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (S256 && !DUMP) {
        // the superblock's scale (its last pair's stage) is read before this pair's barrier: the next superblock's
        // first pair overwrites that stage after the barrier, possibly while a slower wave is still in this epilogue
        if (p == 3)
#pragma unroll
          for (int t = 0; t < 4; ++t) sv256[t] = sasc[cur][0][32 * t + lc];
      }
      store(cur ^ 1);
      store_sa(cur ^ 1);
#pragma unroll
      for (int bb = 0; bb < 2; ++bb) pay[bb] = pay_n[bb];
      __syncthreads();
    }
    if constexpr (!DUMP) {
      // superblock epilogue: res = fma(d, tq, fma(-dmin, tmn, res)) (gemm.cl:395-398). d and dmin are per weight row,
      // i.e. per result register: each lane publishes its row's pair in LDS and reads those of its 16 rows.
      if (h == 0) {
        dtab[wave][0][lc] = h2f(TYPE == T_IQ3_S ? hdr.w : hdr.x);
        if constexpr (MINS) dtab[wave][1][lc] = h2f(hdr.x >> 16);
      }
      // kappa's parts for the blocks 4h + j: slots 2j, 2j + 1 hold parts (0, 0), (1, 1), (2, 0) (S256, with two parts of u: (2, 2))
      u32x4_t kop[CENTRED ? 3 : 1];
      if constexpr (CENTRED) {
        const float d16 = 16.0f * h2f(hdr.x), dm = h2f(hdr.x >> 16);
        const uint32_t m0 = 0x0F0F0F0Fu, m1 = 0x30303030u, m2 = 0x3F3F3F3Fu;
        const uint32_t scw = h ? (hdr.w & m0) | ((hdr.y >> 2) & m1) : hdr.y & m2;
        const uint32_t mnw = h ? ((hdr.w >> 4) & m0) | ((hdr.z >> 2) & m1) : hdr.z & m2;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float k = fmaf(d16, (float)((scw >> (8 * j)) & 0xFFu), -dm * (float)((mnw >> (8 * j)) & 0xFFu));
          kop[0][j] = bf16_pair(k, k);
          const float r1 = k - __builtin_bit_cast(float, kop[0][j] & 0xFFFF0000u);
          kop[1][j] = bf16_pair(r1, r1);
          const float r2 = r1 - __builtin_bit_cast(float, kop[1][j] & 0xFFFF0000u);
          kop[2][j] = bf16_pair(r2, S256 ? r2 : k);
        }
      }
      int mn[8];
#pragma unroll
      for (int b = 0; b < 8; ++b) {
        int scv;
        if constexpr (MINS) q4k_scale_min(hdr.y, hdr.z, hdr.w, b, scv, mn[b]);
        else mn[b] = 0;
      }
      // mins operand (A: weight rows): slot 8h + i = mn of block 4h + i / 2 (a bit select on the two candidates: a
      // lane-dependent array index would put mn in scratch memory)
      bf16x8 mnop;
      const int hm = -h;
#pragma unroll
      for (int i = 0; i < 8; ++i) mnop[i] = (__bf16)(float)((mn[i / 2] & ~hm) | (mn[4 + i / 2] & hm));
      float dr[16], dmr[16];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const float4 dv = *(const float4*)&dtab[wave][0][8 * q + 4 * h];
        dr[4 * q] = dv.x; dr[4 * q + 1] = dv.y; dr[4 * q + 2] = dv.z; dr[4 * q + 3] = dv.w;
        if constexpr (MINS) {
          const float4 mv = *(const float4*)&dtab[wave][1][8 * q + 4 * h];
          dmr[4 * q] = -mv.x; dmr[4 * q + 1] = -mv.y; dmr[4 * q + 2] = -mv.z; dmr[4 * q + 3] = -mv.w;
        }
      }
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        if constexpr (CENTRED) {
          const size_t uo = ((size_t)s * a.Mp + m0 + 32 * t + lc) * 8 + 4 * h;
          const bf16x8 u01 = __builtin_bit_cast(bf16x8, *(const uint4*)(a.u + uo));
          f32x16 tk = zero16;
          if constexpr (!S256) {
            const bf16x8 u02 = __builtin_bit_cast(bf16x8, *(const uint4*)(a.u2 + uo));
            tk = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, kop[2]), u02, tk, 0, 0, 0);
          } else {
            tk = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, kop[2]), u01, tk, 0, 0, 0);
          }
          tk = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, kop[1]), u01, tk, 0, 0, 0);
          tk = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, kop[0]), u01, tk, 0, 0, 0);
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const float v = fmaf(dr[r], tq[t][r], tk[r]);
            res[t][r] = S256 ? fmaf(sv256[t], v, res[t][r]) : v + res[t][r];
          }
          continue;
        }
        if constexpr (!MINS) {
          const float sv = S256 ? sv256[t] : 1.0f;
#pragma unroll
          for (int r = 0; r < 16; ++r) res[t][r] = fmaf(S256 ? dr[r] * sv : dr[r], tq[t][r], res[t][r]);
          continue;
        }
        const uint4 uv = *(const uint4*)(a.u + (size_t)(m0 + 32 * t + lc) * nb + 8 * s + 4 * h);
        const f32x16 tmn = __builtin_amdgcn_mfma_f32_32x32x16_bf16(mnop, __builtin_bit_cast(bf16x8, uv), zero16, 0, 0, 0);
        if constexpr (S256) {
          const float sv = sv256[t];
#pragma unroll
          for (int r = 0; r < 16; ++r) res[t][r] = fmaf(dr[r] * sv, tq[t][r], fmaf(dmr[r], tmn[r], res[t][r]));
        } else {
#pragma unroll
          for (int r = 0; r < 16; ++r) res[t][r] = fmaf(dr[r], tq[t][r], fmaf(dmr[r], tmn[r], res[t][r]));
        }
      }
    }
    hdr = hdr_n;
  }
  if constexpr (DUMP) return;

  // ---- store through LDS: each wave writes a 32 x 32 result tile as [row n][token m], then lanes 0-31 / 32-63 store
  // tokens 2k / 2k + 1 with 32 consecutive weight rows each (128-byte rows of C)
  float* T = (float*)lds + wave * 32 * 33;
#pragma unroll
  for (int t = 0; t < 4; ++t) {
#pragma unroll
    for (int r = 0; r < 16; ++r) T[(8 * (r >> 2) + 4 * h + (r & 3)) * 33 + lc] = res[t][r];
    __builtin_amdgcn_wave_barrier();
    const int n = nbase + lc;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      const int ml = 2 * k + h, m = m0 + 32 * t + ml;
      const float v0 = T[lc * 33 + ml];
      if (CUT && piece >= 0) {  // (piece-local [128 tokens][128 rows])
        a.part[(size_t)piece * (kF16BM * kF16BN) + (32 * t + ml) * kF16BN + wave * 32 + lc] = v0;
        continue;
      }
      if (m < a.M && n < n_rows) {
        float* cp = a.C + (size_t)m * a.ldc + a.c_off + n;
        float v = v0;
        if (a.accumulate == 1) {
          v += *cp;
        } else if (a.accumulate == 2) {
          const float gv = *cp;
          v *= gv / (1.0f + expf(-gv));
        }
        *cp = v;
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
}

// ---- host side

// Q4_K: every prompt of 128 tokens and more. Q5_K and IQ3_S, whose int8 kernels run without a workspace: where the product
// is long enough for the call to wait for the GPU (the workspace costs the host about 20 us), 128-token tiles waste at most a
// fifth of their rows, and the modelled time here, with the prepass's 7 us and 0.16 per million values, is under the int8 kernel's
// (2048 x 5120 -> 17408 Q5_K 773 -> 697 us, IQ3_S 695 -> 650; 512 x 5120 -> 5120 86.6 -> 72.7 and 79.3 -> 70.3; but 1024 x 4096 ->
// 4096, 256 tiles here and 512 there, 86.7 against 79.7 and 84.7 against 71.9, and Q5_K 1167 x 1792 -> 13120, 1030 tiles here, a
// third round of six, 146 against 142).
bool f16_gemm_supported(int type, int M, int rows, int K) {
  if (M < 128 || K % 256) return false;
  if (type == T_Q4_K) return true;
  if (type != T_Q5_K && type != T_IQ3_S) return false;
  if ((double)M * rows * K < 1.2e10 || round_up((size_t)M, kF16BM) * 4 > (size_t)M * 5) return false;
  const float here = 7.0f + 1.03f * gemm_split_for(type, M, rows, K, true).us + 0.16e-6f * (float)M * (float)K;
  return here < gemm_split_for(type, M, rows, K, false).us;
}

// Allocation-free workspace for qmatmul_gemm_noalloc: a file-scope device array (each GPU holds its own copy until
// the process ends). Host code never passes the array's name to a kernel or a copy -- in host code it is only a
// stand-in for the symbol -- but the device address that hipGetSymbolAddress returns for the current device, looked
// up once per device (under a lock) and kept.
constexpr size_t kF16ScratchBytes = (size_t)32 << 20;
static __device__ __align__(256) uint8_t scratch[kF16ScratchBytes];
static __device__ __align__(256) uint8_t split_scratch[kSplitBytes];  // (partial tiles of the cut tiles)

hipError_t f16_scratch(void** out, size_t* bytes, void** part) {
  static std::mutex mu;
  static void *ptrs[64] = {}, *parts[64] = {};
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= 64) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lock(mu);
  if (!ptrs[dev]) {
    void *p = nullptr, *q = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e == hipSuccess) e = hipGetSymbolAddress(&q, HIP_SYMBOL(split_scratch));
    if (e != hipSuccess) return e;
    ptrs[dev] = p;
    parts[dev] = q;
  }
  *out = ptrs[dev];
  *bytes = kF16ScratchBytes;
  *part = parts[dev];
  return hipSuccess;
}

template <int TYPE>
static hipError_t go_f16(const GemmArgs& g, void* ws, hipStream_t s) {
  constexpr int PARTS = !Traits<TYPE>::MINS ? 0 : kF16Centred<TYPE> ? 3 : 2;
  constexpr bool HALF = kF16Half<TYPE>, CENTRED = kF16Centred<TYPE>;
  const int M = g.M, K = g.w.K;
  const int Mp = (int)round_up((size_t)M, kF16BM);
  void* buf = ws;
  hipError_t e = hipSuccess;
  if (!buf) {
    e = pool_alloc(&buf, f16_workspace_bytes(TYPE, M, K), s);
    if (e != hipSuccess) return e;
  }
  uint8_t* af = (uint8_t*)buf;
  uint32_t* u = (uint32_t*)(af + round_up((size_t)Mp * K * 2, 256));
  uint32_t* u2 = u + (size_t)Mp * (K / 32);
  const dim3 agrid((unsigned)(((size_t)Mp * (K / 32) * 2 + 255) / 256));
  // (the block-sum mode reads no activation scales: no mins operand)
  if (g.dbg_isum)
    f16_act_kernel<0, HALF, CENTRED><<<agrid, dim3(256), 0, s>>>(g.aq, nullptr, nullptr, M, g.M_stride, 0, Mp, K, af, u, u2);
  else if (CENTRED && g.ash == 3)
    f16_act_kernel<2, HALF, CENTRED><<<agrid, dim3(256), 0, s>>>(g.aq, nullptr, g.absum, M, g.M_stride, 0, Mp, K, af, u, u2);
  else
    f16_act_kernel<PARTS, HALF, CENTRED><<<agrid, dim3(256), 0, s>>>(g.aq, g.asc, g.absum, M, g.M_stride, g.ash, Mp, K, af, u, u2);
  e = hipGetLastError();
  if (e == hipSuccess) {
    F16Args a{};
    a.w = g.w;
    a.af = af;
    a.Mp = Mp;
    a.u = u;
    a.u2 = u2;
    a.asc = g.asc;
    a.M = M;
    a.M_stride = g.M_stride;
    a.ash = g.ash;
    a.C = g.C;
    a.ldc = g.ldc;
    a.c_off = g.c_off;
    a.accumulate = g.accumulate;
    a.dbg_isum = g.dbg_isum;
    a.part = g.part;
    a.split_from = g.split_from;
    a.splits = g.splits;
    const int gx = (g.w.rows + kF16BN - 1) / kF16BN, gy = Mp / kF16BM, tiles = gx * gy;
    const dim3 grid((unsigned)(g.part ? g.split_from + (tiles - g.split_from) * g.splits : tiles));
    if (g.dbg_isum) gemm_f16_kernel<TYPE, true><<<grid, dim3(256), 0, s>>>(a);
    else if (g.ash == 3 && g.part) gemm_f16_kernel<TYPE, false, true, true><<<grid, dim3(256), 0, s>>>(a);
    else if (g.ash == 3) gemm_f16_kernel<TYPE, false, true><<<grid, dim3(256), 0, s>>>(a);
    else if (g.part) gemm_f16_kernel<TYPE, false, false, true><<<grid, dim3(256), 0, s>>>(a);
    else gemm_f16_kernel<TYPE, false><<<grid, dim3(256), 0, s>>>(a);
    e = hipGetLastError();
    if (e == hipSuccess && g.part) e = launch_split_sum(g, kF16BM, tiles, gx, gy, false, s);
  }
  if (!ws) {
    const hipError_t e2 = hipFreeAsync(buf, s);
    if (e == hipSuccess) e = e2;
  }
  return e;
}

hipError_t launch_gemm_f16(int type, const GemmArgs& g, void* ws, hipStream_t s) {
  switch (type) {
    case T_Q4_K: return go_f16<T_Q4_K>(g, ws, s);
    case T_Q5_K: return go_f16<T_Q5_K>(g, ws, s);
    case T_IQ3_S: return go_f16<T_IQ3_S>(g, ws, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace qm
