// ── fused skinny GEMM, up to 16 pseudo-tokens: half a tile per wave, 16 rows x 16 tokens per matrix-core product ──────
// Decode + dequant + Y[m][N] = X[m][K] W^T for 2..16 pseudo-tokens of fp16 activations (fp32 activations enter as fp16
// hi + lo pseudo-tokens), every K-quant format, any mix of formats in one launch.
//
// What bounds it (gfx950, Q4_K gate + up 2 x 14336 x 4096 at 5 tokens, counters): the LDS pipe, busy 2507 cycles per
// tile (408 reads, 2 table gathers and 1 window read per pair of symbols and chain, 1675 of the cycles bank conflicts),
// and VALU issue, 2463 instructions per tile = as many cycles on a CU's 4 SIMDs: 14 tiles per CU take at least 16 us of
// the launch's 26; the rest is its start (4 us until the first units are in LDS) and the last blocks' ends. The matrix
// cores do 128 products of 16 cycles per tile.
//
// Units. A wave takes half a tile (rows 32 f .. 32 f + 31, contiguous word rows) and copies them to its LDS buffer. Lane
// 16 g + j decodes 4 chains c = 2 p + i: run 4 p + g (32 symbols, a load-time chain start) of row 16 i + j, interleaved
// instruction by instruction. The 16 lanes of one g so hold 16 rows at the same columns: that is the B operand of
// v_mfma_f32_16x16x16_f16 (lane 16 g + j: column j, k = 4 g .. 4 g + 3) with no data moved between lanes, and the A
// operand (lane 16 g + i: row i, the same k) is a piece of token i's activations that launch_wide_x has laid out so that
// a wave's load is one run (read row by row its 64 lanes lie in 64 cache lines: a layer's step of 16 tokens took 145 us
// so, 106 us reordered, the launch that reorders them included). A product costs 16 cycles for 16 tokens x 16 rows x 16 weights; the 4-row blocks of
// v_mfma_f32_4x4x4f16 (k_fused_tiles_mma) take 8 cycles per 4 tokens, and their 16 tokens' x and accumulators would not
// fit the registers. Products of 32 weights (two pairs of symbols at once) were 3 % slower: 116 registers against 98.
//
// Weights. A product's weights lie in 4 sub-blocks (the runs g), so they are scaled by their sub-blocks' integer scales
// before it, exactly in fp16:
//   Q4_K: sc q 2^-24 from the table's grid byte as a denormal, Q5_K: sc (q - c) (at most 63 x 31);
//   Q6_K, IQ4_XS: s f(q) has up to 13 bits, so s = s1 + s0 with s1 even and s0 = 1 or 2 of its sign (split_scale): s1 f(q)
//   and s0 f(q) are exact and go into one product of k = 32 (v_mfma_f32_16x16x32_f16, as long as one of 16), each with the
//   activations. Neither part is 0 unless s is, nor do their signs differ, so an infinite activation stays infinite;
//   IQ4_XS's kv / 16 = fp16(64 + b / 16) - 72 of the grid byte b = kv + 128, one fma per weight pair.
// d is applied in fp32 when the super-block is complete. Mins (Q4_K / Q5_K): one product per row group and super-block of
// the mins with the sub-blocks' fp32 x sums, formed by launch_wide_x and held as three bf16 parts that add up to all 24
// bits (as fp16 hi and lo a sum past 65504, 32 activations of 2047, would be infinite): parts in lane groups 0, 1 and 2 of
// v_mfma_f32_16x16x32_bf16, the mins (at most 63) exact in bf16. Q5_K takes its mean code c
// (DevMat::centre, in its table) off every code and with the sums instead: c d (sc . Sx), as exact, leaves products of sc (q - c), whose
// rounding counts for less.
// Distance from 64 bits 1.3e-7 (2-norm), against 3e-6 of the ring kernel's fp16 dot products and 2e-7 .. 8e-7 of
// k_fused_tiles_mma.
//
// Block = up to W waves of one matrix: whole rows of units where a row has no more units than that, else 4 consecutive
// units of a row. Results [token][32 rows] replace the words in a wave's buffer and the block sums the units of each row
// in tile-column order, four by four. A row in one block is stored; else the sums go to the row's partial slots (one per
// block) and the block that counts the row's last part takes them by the exchanges of sum_partials, its waves sharing
// the tokens (2 us more at the end of a launch).
//
// Measured before (the ring kernel, block per tile column, and a reduction launch) and now, us: a Q4_K layer's step of 16
// tokens in the forward order (4 calls: q + k + v, o, gate + up, down) 339.7 / 83.0; the 4 matrices of a 3072-wide Q4_K
// layer with 4 tokens of fp32 x (4 calls) 159.1 / 66.2; IQ4_XS gate + up and Q6_K down with 5 tokens (2 calls, before:
// k_fused_tiles_mma) 78.0 / 63.3.
#include <algorithm>
#include <cstddef>

#include "lw_device.h"

namespace lw {

namespace {

typedef __attribute__((address_space(3))) const uint32_t LdsU32;
typedef __attribute__((address_space(4))) const char KChar;
typedef __attribute__((address_space(4))) const WideEntry KWide;
typedef __attribute__((address_space(4))) const uint16_t KU16;
typedef __attribute__((address_space(4))) const uint32_t KU32;

constexpr int WIDE_TOKENS = 16;
constexpr int WIDE_MIN_ROWS = WIDE_TOKENS * 32 * 4 / 128;  // a buffer also holds its unit's results

__device__ __forceinline__ h2v dup(float v) { return h2v{(_Float16)v, (_Float16)v}; }

// s0 of a scale v in -128 .. 127: 1 or 2 with v's sign so that v - s0 is even, half of v up to 2
__device__ __forceinline__ float split_scale(int v) {
  const float f = (float)v, part = __builtin_copysignf((float)(2 - (v & 1)), f);
  return __builtin_fabsf(f) <= 2.f ? 0.5f * f : part;
}

// Half a tile (rows 32 f .. 32 f + 31) by one wave: chain c = 2 p + i is run 4 p + g of row 32 f + 16 i + j. PK: of a
// packed matrix, each chain's 32 symbol bytes in registers and 256 table entries; the products, and so the results, are
// those of the coded matrix with the same codes.
template <int KQ, bool PK>
struct WideUnit {
  static constexpr int SYMB = kq_symbits(KQ);
  static constexpr int TW = SYMB == 4 ? 2 * TK : TK;
  static constexpr int SB = kq_sbytes(KQ), NSB = TW / 256;
  static constexpr bool MINS = KQ == KQ_Q4_K || KQ == KQ_Q5_K, SPLIT = !MINS;
  // the accumulators' scale: Q4_K codes enter as fp16 denormals q 2^-24, IQ4_XS grid values as kv / 16
  static constexpr float WSCALE = KQ == KQ_Q4_K ? 16777216.f : KQ == KQ_IQ4_XS ? 16.f : 1.f;
  static constexpr int RUN = TW / 8;     // weights of a run (32 symbols)
  static constexpr int NST = RUN / 8;    // products per run
  static constexpr int PPS = 16 / NST;   // pairs of symbols per product
  static constexpr int XD = 2;           // products (of both passes) whose activations are in flight
  static constexpr int NA = 2 * NSB;     // side records: a super-block of a row each (index 2 sb + i)
  // chain starts; side records as loaded (Q6_K: d and the scales of the run's sub-blocks of both passes)
  uint32_t start[4], raw[NA][5];
  u32x4 sym[4][2];  // PK
  u32x4 x[XD][2], sx[NSB];
  __amdgpu_buffer_rsrc_t xr;
  uint32_t xv;  // the lane's 16 bytes of a piece (a lane past the tokens: past the buffer, reads zeros)
  int x0, xs;   // the tile column's first piece, the piece stride

  __device__ __forceinline__ void load_x(int st) {
#pragma unroll
    for (int p = 0; p < 2; ++p)
      x[st % XD][p] = __builtin_amdgcn_raw_buffer_load_b128(xr, xv, x0 + (p * NST + st) * xs, 0);
  }

  __device__ __forceinline__ void load(KWide* e, int t, int f, int mt, int lane) {
    const auto& M = e->M;
    const int g = lane >> 4, j = lane & 15;
    const int KT = M.KT, K = M.K, tc = t % KT, tr = t / KT;
    const uint8_t* srec = M.side + (side_record(tr * TN, tc * NSB, KT, NSB) + (uint32_t)(32 * f + j)) * SB;
#pragma unroll
    for (int a = 0; a < NA; ++a) {
      const uint8_t* r = srec + ((a >> 1) * TN + 16 * (a & 1)) * SB;
      if constexpr (KQ == KQ_Q6_K) {  // int8 scales of sub-blocks 2 g, 2 g + 1 and 8 + 2 g, 9 + 2 g
        const uint16_t* h = reinterpret_cast<const uint16_t*>(r);
        raw[a][0] = h[8];
        raw[a][1] = (uint32_t)h[g];
        raw[a][2] = (uint32_t)h[4 + g];
      } else {
        side_load<KQ>(r, raw[a]);
      }
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      if constexpr (PK) {  // 16-byte pieces 2 r and 2 r + 1 of run r, [16 pieces][64 rows]
        const u32x4* w = reinterpret_cast<const u32x4*>(M.words) + (size_t)t * 1024 + 512 * (c >> 1) + 32 * f + 16 * (c & 1);
#pragma unroll
        for (int u = 0; u < 2; ++u) sym[c][u] = w[128 * g + 64 * u + j];
      } else {
        start[c] = M.hsplit[(((size_t)t * 2 + (uint32_t)f) * 64 + 32 * (c >> 1) + 16 * (c & 1)) * 4 + (uint32_t)(4 * j + g)];
      }
    }
    const int xbytes = 2 * mt * K;
    xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(e->X), (short)0, xbytes + xbytes / 32 * 3, kBufferRsrcWord3);
    xv = j < mt ? (uint32_t)(16 * (g * mt + j)) : 0x7FFFFFF0u;
    x0 = tc * 2 * NST * 64 * mt;
    xs = 64 * mt;
    // lanes g < 3 part g of a super-block's 8 x sums
    if constexpr (MINS) {
#pragma unroll
      for (int sb = 0; sb < NSB; ++sb)
        sx[sb] = __builtin_amdgcn_raw_buffer_load_b128(xr, g < 3 ? xv : 0x7FFFFFF0u, xbytes + (NSB * tc + sb) * 48 * mt, 0);
    }
#pragma unroll
    for (int st = 0; st < XD; ++st) load_x(st);
  }

  // results [16 tokens][32 rows] of the unit in tot[i][r] (token 4 g + r, row 16 i + j); buf: its word rows in LDS, row
  // 0 of the buffer the tile's row r0
  __device__ __forceinline__ void decode(const uint32_t* buf, int r0, int lane, int centre, f4v (&tot)[2]) {
    const int g = lane >> 4;
    // the sub-block scales of the runs of chains 2 p and 2 p + 1 (two bytes each; Q5_K one of them) and d of rows
    // 0 and 1 of a super-block, two to a word
    uint32_t sc[2] = {0, 0}, d2[NA / 2];
    auto put = [&](int c, uint32_t v) { sc[c >> 1] |= (v & 0xFFFFu) << (16 * (c & 1)); };
    tot[0] = tot[1] = f4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int a = 0; a < NA; ++a) {
      const uint32_t* w = raw[a];
      if (a & 1) d2[a / 2] |= w[0] << 16;
      else d2[a / 2] = w[0] & 0xFFFFu;
      if constexpr (KQ == KQ_Q6_K) {
        put(a, w[1]);
        put(2 + a, w[2]);
      } else if constexpr (KQ == KQ_IQ4_XS) {  // sub-blocks 2 g, 2 g + 1
        const uint32_t lo = w[1] >> (8 * g), hi = w[0] >> (16 + 4 * g);
        put(a, ((lo & 15u) | (hi & 3u) << 4) | ((lo >> 4 & 15u) | (hi >> 2 & 3u) << 4) << 8);
      } else {
        const uint32_t s0 = w[1] & 0x3F3F3F3Fu, s1 = (w[3] & 0x0F0F0F0Fu) | ((w[1] >> 2) & 0x30303030u);
        if constexpr (KQ == KQ_Q4_K) {  // sub-blocks 2 g, 2 g + 1
          put(a, ((g & 2) ? s1 : s0) >> (16 * (g & 1)));
        } else {  // sub-blocks g, 4 + g
          put(a, s0 >> (8 * g) & 255u);
          put(2 + a, s1 >> (8 * g) & 255u);
        }
        float mf[8];
        side_mins(w, mf);
        u32x4 m;  // as bf16, the upper halves
#pragma unroll
        for (int k = 0; k < 4; ++k)
          m[k] = __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, mf[2 * k + 1]), __builtin_bit_cast(uint32_t, mf[2 * k]),
                                       0x07060302u);
        f4v mb = {0.f, 0.f, 0.f, 0.f};
        if constexpr (KQ == KQ_Q5_K) {  // the scales with the sums
          u32x4 sb;
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const uint32_t v = (k < 2 ? s0 : s1) >> (16 * (k & 1));
            sb[k] = __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, (float)(v >> 8 & 255u)),
                                          __builtin_bit_cast(uint32_t, (float)(v & 255u)), 0x07060302u);
          }
          mb = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(b8v, sx[a >> 1]), __builtin_bit_cast(b8v, sb), mb, 0,
                                                       0, 0);
        }
        const float off = -h2f(w[0] >> 16), dc = (float)centre * h2f(w[0]);
        const f4v ma = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(b8v, sx[a >> 1]), __builtin_bit_cast(b8v, m),
                                                               f4v{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 4; ++r) tot[a & 1][r] = fmaf(off, ma[r], KQ == KQ_Q5_K ? dc * mb[r] : tot[a & 1][r]);
      }
    }
    const uint32_t rlb =
        (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const uint32_t*)(buf + (lane & 15));
    // sums of a chain (Q5_K, for the registers: of a row's two), Q6_K's folded into tot every 16 symbols (one run of
    // additions over 256 weights was 1.3 .. 1.6 times as far from 64 bits)
    constexpr int NACC = KQ == KQ_Q5_K ? 2 : 4;
    f4v acc[NACC];
#pragma unroll
    for (int c = 0; c < NACC; ++c) acc[c] = f4v{0.f, 0.f, 0.f, 0.f};
    auto fold = [&]() {
#pragma unroll
      for (int c = 0; c < NACC; ++c) {
        const float d = h2f(d2[NSB == 2 ? c >> 1 : 0] >> (16 * (c & 1))) * WSCALE;
#pragma unroll
        for (int r = 0; r < 4; ++r) tot[c & 1][r] = fmaf(d, acc[c][r], tot[c & 1][r]);
        acc[c] = f4v{0.f, 0.f, 0.f, 0.f};
      }
    };
    // P form: bit position in the buffer - GUARD_BITS + 64; slot = P >> 5 is the window row after the two in A and B
    uint32_t P[4], slot[4], A[4], B[4], C[4];
#pragma unroll
    for (int c = 0; c < 4 && !PK; ++c) {
      P[c] = start[c] - (uint32_t)(32 * r0) - GUARD_BITS + 64u;
      slot[c] = __builtin_amdgcn_ubfe(P[c], 5, 8);
      const uint32_t a = rlb + (slot[c] << 7) + 64u * (c & 1);
      A[c] = *(LdsU32*)(a - 256u);
      B[c] = *(LdsU32*)(a - 128u);
      C[c] = *(LdsU32*)a;
    }
    h2v s1[4], n1[4], s0[4], n0[4];  // the chains' current scales (SPLIT: s1 + s0) and IQ4_XS's -72 s
    uint32_t w4[4][2];
    static_for<16>([&](auto pc) {
      constexpr int q = decltype(pc)::value, st = q / PPS;
      // scales of the sub-block that starts here: 8 pairs of symbols each (Q5_K: the whole run)
      if constexpr (q == 0 || (KQ != KQ_Q5_K && q == 8)) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const uint32_t b = sc[c >> 1] >> (16 * (c & 1) + q) & 255u;
          if constexpr (!SPLIT) {
            s1[c] = dup((float)b);
          } else {
            const int v = KQ == KQ_Q6_K ? (int)(int8_t)(uint8_t)b : (int)b - 32;
            const float b0 = split_scale(v), b1 = (float)v - b0;
            s1[c] = dup(b1);
            s0[c] = dup(b0);
            n1[c] = dup(-72.f * b1);
            n0[c] = dup(-72.f * b0);
          }
        }
      }
      uint32_t w1[4], e1[4], e2[4];
      if constexpr (PK) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          w1[c] = sym[c][q >> 3][q >> 1 & 3] >> (16 * (q & 1));
          e1[c] = *(LdsU32*)(4u * (w1[c] & 255u));  // (the table lies at LDS address 0)
          e2[c] = *(LdsU32*)(4u * (w1[c] >> 8 & 255u));
        }
      } else {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          w1[c] = __builtin_amdgcn_alignbit(B[c], A[c], P[c]);
          e1[c] = *(LdsU32*)(w1[c] & 0x1FFCu);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int c = 0; c < 4; ++c) e2[c] = *(LdsU32*)(w1[c] >> (e1[c] & 31u) & 0x1FFCu);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          P[c] = P[c] + e1[c] + e2[c];
          const uint32_t nslot = __builtin_amdgcn_ubfe(P[c], 5, 8);
          const bool slide = nslot != slot[c];
          A[c] = slide ? B[c] : A[c];
          B[c] = slide ? C[c] : B[c];
          slot[c] = nslot;
          C[c] = *(LdsU32*)(rlb + (nslot << 7) + 64u * (c & 1));
        }
      }
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        if constexpr (KQ == KQ_IQ4_XS) {  // fp16(64 + b / 16) of each grid byte b = kv + 128
          w4[c][0] = __builtin_amdgcn_perm(0x54545454u, e1[c], 0x04030402u);
          w4[c][1] = __builtin_amdgcn_perm(0x54545454u, e2[c], 0x04030402u);
        } else if constexpr (SYMB == 4) {
          w4[c][0] = __builtin_amdgcn_perm(e1[c], e1[c], 0x0C030C02u);
          w4[c][1] = __builtin_amdgcn_perm(e2[c], e2[c], 0x0C030C02u);
        } else {
          w4[c][q & 1] = __builtin_amdgcn_perm(e2[c], e1[c], 0x07060302u);
        }
      }
      if constexpr (SYMB == 4 || (q & 1)) {  // 4 weights per lane
        constexpr int h = SYMB == 4 ? q & 1 : (q >> 1) & 1;
        auto scaled = [&](uint32_t w, h2v sv, h2v nv) {
          const h2v v = __builtin_bit_cast(h2v, w);
          return __builtin_bit_cast(uint32_t, KQ == KQ_IQ4_XS ? __builtin_elementwise_fma(v, sv, nv) : v * sv);
        };
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const u32x4 xp = x[st % XD][c >> 1];
          const uint32_t x0 = xp[2 * h], x1 = xp[2 * h + 1];
          const uint32_t v0 = scaled(w4[c][0], s1[c], n1[c]), v1 = scaled(w4[c][1], s1[c], n1[c]);
          f4v& a = acc[c % NACC];
          if constexpr (SPLIT) {  // both parts in one product, the activations twice
            const uint32_t u0 = scaled(w4[c][0], s0[c], n0[c]), u1 = scaled(w4[c][1], s0[c], n0[c]);
            a = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8v, make_uint4(x0, x1, x0, x1)),
                                                       __builtin_bit_cast(h8v, make_uint4(v0, v1, u0, u1)), a, 0, 0, 0);
          } else {
            a = __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(h4v, make_uint2(x0, x1)),
                                                      __builtin_bit_cast(h4v, make_uint2(v0, v1)), a, 0, 0, 0);
          }
        }
        if constexpr (q % PPS == PPS - 1 && st + XD < NST) load_x(st + XD);
        if constexpr (KQ == KQ_Q6_K && q == 7) fold();
      }
    });
    fold();
  }
};

template <int V>
struct WideTag {
  static constexpr int value = V;
};

}  // namespace

// KQ: the entries' K-quant type, 0 for a plan over several; PK: packed matrices
template <int KQ, bool PK>
__global__ void __launch_bounds__(64 * WIDE_MAX_WAVES) __attribute__((amdgpu_waves_per_eu(KQ == KQ_Q5_K || KQ == KQ_Q6_K ? 5 : 4)))
k_fused_wide(WidePlan plan, int buf_rows) {
  __shared__ uint32_t lut4[LUTN + 4];  // the table first: table_addr takes it to lie at LDS address 0
  extern __shared__ __align__(16) uint32_t tbuf[];
  KChar* kbase = (KChar*)__builtin_amdgcn_kernarg_segment_ptr();
  const int b = (int)blockIdx.x, W = plan.W, mt = plan.mt, per = plan.per;
  int me = 0;
#pragma unroll
  for (int i = 1; i < MAX_GROUP; ++i)
    if (i < plan.n && b >= plan.e[i].block0) me = i;
  KWide* e = (KWide*)(kbase + offsetof(WidePlan, e) + (size_t)me * sizeof(WideEntry));
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  // half-tile rows hr = 2 tr + f (32 matrix rows each) of KT units. A block has whole rows (hr0 .. hr0 + nseg - 1), or
  // the units c0 .. c0 + nu - 1 of one row, its part `part` of np
  const int KT = e->M.KT, N = e->M.N, bl = b - e->block0, upb = e->w;
  int hr0, nseg = 1, c0 = 0, nu, part = 0, np = 1;
  if (KT <= upb) {
    const int rpb = upb / KT;
    hr0 = bl * rpb;
    nseg = min(rpb, 2 * e->M.NT - hr0);
    nu = nseg * KT;
  } else {
    np = (KT + upb - 1) / upb;
    hr0 = bl / np;
    part = bl - hr0 * np;
    c0 = part * upb;
    nu = min(upb, KT - c0);
  }
  const bool have = wave < nu;
  uint32_t* buf = tbuf + (size_t)wave * buf_rows * 32;
  uint32_t* last = lut4 + LUTN;            // this block sums its row's parts
  const int mo = per == 2 ? mt >> 1 : mt;  // output tokens
  if (threadIdx.x == 0) *last = 0u;
  f4v tot[2];
  auto run = [&](auto kq) __attribute__((always_inline)) {
    WideUnit<decltype(kq)::value, PK> unit;
    const int sg = np > 1 ? 0 : wave / KT, hr = hr0 + sg, f = hr & 1, t = (hr >> 1) * KT + c0 + wave - sg * KT;
    int r0 = 0, nc = 0;
    if (have) {
      unit.load(e, t, f, mt, lane);
    }
    if (!PK && have) {
      // the unit's word rows (8 per instruction, the last masked)
      const uint32_t h = ((KU32*)e->M.hrow)[t];
      const uint32_t rw = ((KU32*)e->M.rows)[t >> 1] >> (16 * (t & 1)) & 0xFFFFu;
      r0 = f ? (int)(h >> 16) : 0;
      const int nrow = f ? (int)rw - r0 : (int)(h & 0xFFFFu);
      const uint4* src = reinterpret_cast<const uint4*>(e->M.words + ((KU32*)e->M.tbase)[t] + 32u * (uint32_t)r0) + lane;
      nc = (nrow + 7) / 8;
      for (int i = 0; i < nc; ++i)
        if (lane < 8 * (nrow - 8 * i))
          __builtin_amdgcn_global_load_lds(src + 64 * i, (__attribute__((address_space(3))) void*)(buf + 256 * i), 16, 0, 0);
    }
    {  // the decode table: 1 KB direct-to-LDS loads, chunk c by wave c mod W
      const uint4* ta = reinterpret_cast<const uint4*>(e->M.lutw);
      for (int c = wave; c < (PK ? 1 : 8); c += W)
        __builtin_amdgcn_global_load_lds(ta + 64 * c + lane, (__attribute__((address_space(3))) void*)(lut4 + 256 * c), 16,
                                         0, 0);
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (have) unit.decode(buf, r0, lane, e->M.centre, tot);
  };
  const int kqt = KQ ? KQ : e->M.kqt;
  if (kqt == KQ_Q4_K) run(WideTag<KQ_Q4_K>{});
  else if (kqt == KQ_Q5_K) run(WideTag<KQ_Q5_K>{});
  else if (kqt == KQ_Q6_K) run(WideTag<KQ_Q6_K>{});
  else run(WideTag<KQ_IQ4_XS>{});
  if (have) {  // the wave's own buffer, its decode done, takes the results [token][32 rows]
    asm volatile("" ::: "memory");
    float* res = reinterpret_cast<float*>(buf) + (lane & 15);
    const int g = lane >> 4;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      if (per == 2) {  // hi + lo of tokens 2 g, 2 g + 1
        res[(2 * g) * 32 + 16 * i] = tot[i][0] + tot[i][1];
        res[(2 * g + 1) * 32 + 16 * i] = tot[i][2] + tot[i][3];
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) res[(4 * g + r) * 32 + 16 * i] = tot[i][r];
      }
    }
  }
  __syncthreads();
  // per row and token the block's units in tile-column order, summed four by four (the parts of a row are multiples of
  // four units, so a row's sum does not depend on how the units lie in blocks): 32 lanes a token
  const int l32 = lane & 31, nc = np > 1 ? nu : KT;
  for (int it = 2 * wave + (lane >> 5); it < nseg * mo; it += 2 * W) {
    const int sg = it / mo, tok = it - sg * mo;
    const float* res = reinterpret_cast<const float*>(tbuf) + (size_t)(sg * nc) * buf_rows * 32 + tok * 32 + l32;
    float a = 0.f;
    for (int w = 0; w < nc; w += 4) {
      float v[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) v[k] = w + k < nc ? res[(size_t)(w + k) * buf_rows * 32] : 0.f;
      a += (v[0] + v[1]) + (v[2] + v[3]);
    }
    const size_t o = (size_t)(hr0 + sg) * 32 + (uint32_t)l32;
    if (np == 1)
      e->Y[(size_t)tok * e->ldy + o] = a;
    else
      __hip_atomic_store(e->P + ((size_t)part * mo + tok) * N + o, a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  if (np == 1) return;
  // the block that counts the row's last part sums the parts in order; it counts its own once every wave's partials are
  // stored (a workgroup barrier alone does not wait for global stores)
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0) {
    const uint32_t old = __hip_atomic_fetch_add(e->cnt + hr0, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (old == (uint32_t)(np - 1)) {
      __hip_atomic_store(e->cnt + hr0, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      *last = 1u;
    }
  }
  __syncthreads();
  if (!*last) return;
  const size_t o = (size_t)hr0 * 32 + (uint32_t)l32;
  for (int tok = 2 * wave + (lane >> 5); tok < mo; tok += 2 * W)
    e->Y[(size_t)tok * e->ldy + o] =
        sum_partials(reinterpret_cast<uint32_t*>(e->P + (size_t)tok * N + o), (size_t)mo * N, np);
}

// blocks of an entry with at most w units per block
int wide_blocks(const DevMat& M, int w) {
  return M.KT <= w ? (2 * M.NT + w / M.KT - 1) / (w / M.KT) : 2 * M.NT * ((M.KT + w - 1) / w);
}

// Activations in the products' order: fp16 X [mt][K] (per = 1), or fp32 X [mt / 2][K] split into fp16 hi and lo tokens
// (per = 2), to pieces of 64 mt bytes per (tile column, pass, product): 16 bytes (8 weights' activations) of token j at
// (g mt + j) 16, g the quarter of the pass. Read row by row, the 64 lanes of a product's load lie in 64 cache lines;
// in pieces they are one run.
__global__ void __launch_bounds__(256) k_wide_x(WideXJobs q) {
  int jb = 0;
#pragma unroll
  for (int i = 1; i < MAX_GROUP; ++i)
    if (i < q.n && (int)blockIdx.x >= q.b0[i]) jb = i;
  const int K = q.K[jb], mt = q.mt, n8 = K / 8;        // 8 consecutive weights of one token per thread
  const int i = ((int)blockIdx.x - q.b0[jb]) * 256 + threadIdx.x;
  const int tok = i / n8, c = i - tok * n8;
  if (tok >= (q.per == 2 ? mt / 2 : mt)) return;
  const int run8 = q.symbits[jb] == 4 ? 8 : 4;          // products per run
  const int st = c % run8, g = c / run8 % 4, piece = c / (4 * run8) * run8 + st;
  uint4* out = static_cast<uint4*>(q.XT[jb]) + (size_t)piece * 4 * mt + g * mt;
  // the sum of the thread's 8, then of the sub-block's 32 (4 threads), as three bf16 parts, each what is left cut to 8
  // bits: its place in the super-block's 8 first parts of each token, then 8 second and 8 third ones, after the pieces
  uint16_t* sxo = reinterpret_cast<uint16_t*>(static_cast<uint4*>(q.XT[jb]) + (size_t)n8 * mt) +
                  (size_t)(c / 32) * 24 * mt + (c >> 2 & 7);
  auto put_sum = [&](float a, int tk) {
    a += __shfl_xor(a, 1);
    a += __shfl_xor(a, 2);
    if (c & 3) return;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const uint32_t u = __builtin_bit_cast(uint32_t, a) & 0xFFFF0000u;
      sxo[8 * (k * mt + tk)] = (uint16_t)(u >> 16);
      a -= __builtin_bit_cast(float, u);
    }
  };
  auto sum8 = [&](const uint32_t* v) {
    float a = 0.f;
#pragma unroll
    for (int k = 0; k < 4; ++k) a += h2f(v[k]) + h2f(v[k] >> 16);
    return a;
  };
  if (q.per == 1) {
    const uint16_t* x = static_cast<const uint16_t*>(q.X[jb]) + (size_t)tok * K + 8 * c;
    uint4 v;
    if (((uintptr_t)x & 15) == 0) {
      v = *reinterpret_cast<const uint4*>(x);
    } else {
      v = make_uint4(x[0] | (uint32_t)x[1] << 16, x[2] | (uint32_t)x[3] << 16, x[4] | (uint32_t)x[5] << 16,
                     x[6] | (uint32_t)x[7] << 16);
    }
    out[tok] = v;
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
    put_sum(sum8(w), tok);
  } else {
    const float* x = static_cast<const float*>(q.X[jb]) + (size_t)tok * K + 8 * c;
    uint32_t hi[4], lo[4];
#pragma unroll
    for (int k = 0; k < 8; k += 2) {
      const _Float16 h0 = (_Float16)x[k], h1 = (_Float16)x[k + 1];
      hi[k / 2] = (uint32_t)__builtin_bit_cast(uint16_t, h0) | (uint32_t)__builtin_bit_cast(uint16_t, h1) << 16;
      lo[k / 2] = f2h(x[k] - (float)h0) | f2h(x[k + 1] - (float)h1) << 16;
    }
    out[2 * tok] = make_uint4(hi[0], hi[1], hi[2], hi[3]);
    out[2 * tok + 1] = make_uint4(lo[0], lo[1], lo[2], lo[3]);
    put_sum(sum8(hi), 2 * tok);
    put_sum(sum8(lo), 2 * tok + 1);
  }
}

size_t wide_x_bytes(int mt, int K) { return (size_t)mt * K * 2 + (size_t)mt * (K / 256) * 48; }

hipError_t launch_wide_x(WideXJobs q, hipStream_t s) {
  if (q.n < 1 || q.n > MAX_GROUP || q.mt < 1 || q.mt > WIDE_TOKENS || (q.per != 1 && q.per != 2) || q.mt % q.per)
    return hipErrorInvalidValue;
  int blocks = 0;
  for (int i = 0; i < q.n; ++i) {
    if (!q.X[i] || !q.XT[i] || q.K[i] < 256 || q.K[i] % (q.symbits[i] == 4 ? 512 : 256)) return hipErrorInvalidValue;
    q.b0[i] = blocks;
    blocks += (q.mt / q.per * (q.K[i] / 8) + 255) / 256;
  }
  hipLaunchKernelGGL(k_wide_x, dim3(blocks), dim3(256), 0, s, q);
  return hipGetLastError();
}

bool wide_ok(const DevMat& M) {
  return M.kqt >= KQ_Q4_K && M.kqt <= KQ_IQ4_XS && M.words && M.lutw && M.side &&
         (M.packed || (M.hsplit && M.rows && M.tbase && M.hrow && M.max_rows + 2 <= 256));
}

int wide_buf_rows(const WidePlan& p) {
  int r = WIDE_MIN_ROWS;
  for (int i = 0; i < p.n; ++i) r = std::max(r, p.e[i].M.max_hrows + 2);
  return r;
}

size_t wide_lds_bytes(int waves, int buf_rows) { return (size_t)4 * (LUTN + 4) + (size_t)waves * buf_rows * 128; }

hipError_t launch_fused_wide(const WidePlan& p, hipStream_t s) {
  if (p.n < 1 || p.n > MAX_GROUP || p.W < 1 || p.W > WIDE_MAX_WAVES || p.mt < 1 || p.mt > WIDE_TOKENS ||
      (p.per != 1 && p.per != 2) || p.mt % p.per)
    return hipErrorInvalidValue;
  int blocks = 0, kqt = p.e[0].M.kqt;
  for (int i = 0; i < p.n; ++i) {
    const WideEntry& e = p.e[i];
    if (!wide_ok(e.M) || e.M.packed != p.e[0].M.packed || !e.X || ((uintptr_t)e.X & 15) || !e.Y || !e.P || !e.cnt || e.block0 != blocks || e.M.KT < 1 ||
        e.M.NT < 1 || e.w < 1 || (e.M.KT <= e.w ? e.w / e.M.KT * e.M.KT : e.w) > p.W || (e.M.KT > e.w && e.w % 4))
      return hipErrorInvalidValue;
    blocks += wide_blocks(e.M, e.w);
    if (e.M.kqt != kqt) kqt = 0;
  }
  const int rows = wide_buf_rows(p);
  if (wide_lds_bytes(p.W, rows) > 160 * 1024) return hipErrorInvalidValue;
  const size_t smem = (size_t)p.W * rows * 128;
  auto* const kernel = p.e[0].M.packed ? k_fused_wide<0, true>
                     : kqt == KQ_Q4_K ? k_fused_wide<KQ_Q4_K, false> : kqt == KQ_Q5_K ? k_fused_wide<KQ_Q5_K, false>
                     : kqt == KQ_Q6_K ? k_fused_wide<KQ_Q6_K, false> : kqt == KQ_IQ4_XS ? k_fused_wide<KQ_IQ4_XS, false>
                                                                     : k_fused_wide<0, false>;
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kernel, dim3(blocks), dim3(64 * p.W), smem, s, p, rows);
  return hipGetLastError();
}

}  // namespace lw
