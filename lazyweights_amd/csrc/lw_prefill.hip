// Prefill (m > 8): codes decoded to a tiled layout, activations split and tiled, GEMM on the matrix cores.
#include <algorithm>

#include "lw_device.h"

namespace lw {

// x of the prefill GEMM: fp32 X [m][K] -> XT (fp16 hi = fp16(x), lo = fp16(x - hi)) and SXT (per sub-block of 32
// weights s = ((a0 + a1) + (a2 + a3)), a_q the in-order fp32 sum of its q-th 8 values, as fp16 hi / lo), tokens
// padded with zeros to a multiple of 64. Thread = (chunk, q, token c of the tile): the 32 threads of one q write one
// lane-linear 512-byte run of a piece; the chunk's four a_q meet in LDS (part: PREFILL_X_LDS floats).
constexpr int PREFILL_X_LDS = 2 * 4 * 32;
__device__ __forceinline__ void prefill_x_block(const PrefillX& px, int block, float* part) {
  const float* __restrict__ const X = px.X;
  uint16_t* __restrict__ const XT = px.XT;
  uint16_t* __restrict__ const SXT = px.SXT;
  const int m = px.m, K = px.K;
  const int KC = K / 32, NB = K / 256;
  const int i = block * 256 + (int)threadIdx.x;          // the blocks cover the padded tokens exactly
  const int c = i & 31, q = (i >> 5) & 3, ci = i >> 7;
  const int tt = ci / KC, kc = ci - tt * KC, t = tt * 32 + c, hh = q >> 1, st = q & 1;
  float v[8];
  if (t < m) {
    const float* x = X + (size_t)t * K + 32 * kc + 8 * q;
    const float4 a = *reinterpret_cast<const float4*>(x), b = *reinterpret_cast<const float4*>(x + 4);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = 0.f;
  }
  uint32_t hw[4], lw[4];
  float sum = 0.f;
#pragma unroll
  for (int e = 0; e < 8; e += 2) {
    const _Float16 h0 = (_Float16)v[e], h1 = (_Float16)v[e + 1];
    const _Float16 l0 = (_Float16)(v[e] - (float)h0), l1 = (_Float16)(v[e + 1] - (float)h1);
    hw[e / 2] = (uint32_t)__builtin_bit_cast(uint16_t, h0) | (uint32_t)__builtin_bit_cast(uint16_t, h1) << 16;
    lw[e / 2] = (uint32_t)__builtin_bit_cast(uint16_t, l0) | (uint32_t)__builtin_bit_cast(uint16_t, l1) << 16;
    sum += v[e];
    sum += v[e + 1];
  }
  uint4* o = reinterpret_cast<uint4*>(XT) + ((((size_t)tt * KC + kc) * 2) * 2 + st) * 64 + 32 * hh + c;
  o[0] = make_uint4(hw[0], hw[1], hw[2], hw[3]);
  o[2 * 64] = make_uint4(lw[0], lw[1], lw[2], lw[3]);
  if (!SXT) return;  // formats without mins
  float* const p = part + ((threadIdx.x >> 7) & 1) * 128 + c;  // of the block's two chunks
  p[32 * q] = sum;
  __syncthreads();
  if (q == 0) {
    const float s = (p[0] + p[32]) + (p[64] + p[96]);
    const _Float16 hi = (_Float16)s;
    uint16_t* sx = SXT + ((((size_t)tt * NB + (kc >> 3)) * 2) * 32 + c) * 8 + (kc & 7);
    sx[0] = __builtin_bit_cast(uint16_t, hi);
    sx[32 * 8] = __builtin_bit_cast(uint16_t, (_Float16)(s - (float)hi));
  }
}

// Codes in the prefill GEMM's tiled layout (launch_prefill_prep): one block of 4 waves per tile as k_decode_split,
// but each lane runs the two 32-symbol chains of its 64-symbol segment (split starts 2k and 2k + 1) interleaved, and
// stores its codes straight from registers: 16 codes make one lane's piece of the tiled layout, and the 32 lanes of a
// row half write 32 consecutive pieces (512 B) per store. No code rows in LDS: the block holds the table and the tile.
// The first px.blocks blocks prepare the activations (prefill_x_block): the two need nothing from each other, and in one
// launch the second costs neither a launch nor the first's last wave: a Q4_K layer's prompt of 128 tokens (7 calls) 321 ->
// 290 us, with the 4-bit formats' codes taken from the decode table's grid bytes (no nibbles to part).
template <int SYMB>
__global__ void __launch_bounds__(256) k_prefill_prep(DevMat M, uint8_t* __restrict__ out, int tr0, int tr1,
                                                      int stage_rows, PrefillX px) {
  typedef __attribute__((address_space(3))) const uint32_t LdsU32;
  // the only static LDS object, so at LDS address 0 (table_addr ORs its base in); an activation block's sums lie in it too
  __shared__ __align__(16) uint32_t lut4[LUTN];
  extern __shared__ __align__(16) uint32_t tw[];
  const int KT = M.KT, KC = M.K / 32;
  if ((int)blockIdx.x < px.blocks) {
    prefill_x_block(px, (int)blockIdx.x, reinterpret_cast<float*>(lut4));
    return;
  }
  const int t = tr0 * KT + (int)blockIdx.x - px.blocks;
  const int tc = t % KT, tr = t / KT;
  const int R = min((int)M.rows[t] + 2, stage_rows);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, l = lane & 31, f = lane >> 5;
  // the tile's rows, 8 per direct-to-LDS load, the waves in turn, and the table: every load in flight at once (through
  // registers in a loop each turn waited for its own: 4096 x 4096 with m = 128 9.8 us, so 8.1; 14336 x 4096 18.7 and 15.5)
  const uint4* src = reinterpret_cast<const uint4*>(M.words + M.tbase[t]) + lane;
  for (int i = wave; 8 * i < R; i += 4)
    if (lane < 8 * (R - 8 * i))
      __builtin_amdgcn_global_load_lds(src + 64 * i, (__attribute__((address_space(3))) void*)(tw + 256 * i), 16, 0, 0);
  if (SYMB == 4) {  // entries len | grid byte of the pair's first code << 16 | second << 24 (decode_table4)
    const uint4* ta = reinterpret_cast<const uint4*>(M.lut4) + lane;
#pragma unroll
    for (int i = 0; i < 2; ++i)
      __builtin_amdgcn_global_load_lds(ta + 64 * (wave + 4 * i),
                                       (__attribute__((address_space(3))) void*)(lut4 + 256 * (wave + 4 * i)), 16, 0, 0);
  } else {  // sym | len << 8 -> len | sym << 16, 8 entries a thread
    static_assert(LUTN == 8 * 256, "8 entries per thread");
    const uint4 v = reinterpret_cast<const uint4*>(M.lut)[threadIdx.x];
    auto entry = [](uint32_t e) { return (e >> 8 & 255u) | (e & 255u) << 16; };
    uint4* o = reinterpret_cast<uint4*>(lut4) + 2 * threadIdx.x;
    o[0] = make_uint4(entry(v.x), entry(v.x >> 16), entry(v.y), entry(v.y >> 16));
    o[1] = make_uint4(entry(v.z), entry(v.z >> 16), entry(v.w), entry(v.w >> 16));
  }
  const int k = 4 * f + wave;  // segment of bit-lane l: row f * 32 + l, symbols 64 wave .. 64 wave + 63
  const uint32_t tsel = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const uint32_t*)lut4;
  uint32_t tmask = 0x1FFCu;
  asm volatile("" : "+v"(tmask));
  const uint32_t rlb = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint32_t*)(tw + l);
  uint32_t P[2], slot[2], A[2], B[2], C[2];
#pragma unroll
  for (int ch = 0; ch < 2; ++ch)
    P[ch] = (uint32_t)M.split[((size_t)t * SPLITS + 2 * k + ch) * 32 + (uint32_t)l] - GUARD_BITS + 64u;
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
  for (int ch = 0; ch < 2; ++ch) {
    slot[ch] = __builtin_amdgcn_ubfe(P[ch], 5, 8);
    A[ch] = *(LdsU32*)(rlb + ((slot[ch] - 2u) << 7));
    B[ch] = *(LdsU32*)(rlb + ((slot[ch] - 1u) << 7));
    C[ch] = *(LdsU32*)(rlb + (slot[ch] << 7));
  }
  // chain ch holds codes [2 (64 wave + 32 ch), + 64) (SYMB 4) or [64 wave + 32 ch, + 32) (SYMB 8) of the row
  const size_t rt = (size_t)(tr - tr0) * 2 + f;
  uint8_t* const obase = out + (rt * KC * 64 + l) * 16;
  const int kc0 = SYMB == 4 ? tc * (2 * TK / 32) + 4 * wave : tc * (TK / 32) + 2 * wave;
  uint32_t acc[2][4];
#pragma unroll
  for (int p = 0; p < 16; ++p) {
#pragma unroll
    for (int ch = 0; ch < 2; ++ch) {
      const uint32_t w1 = __builtin_amdgcn_alignbit(B[ch], A[ch], P[ch]);
      const uint32_t e1 = *(LdsU32*)table_addr(w1, tsel, tmask);
      const uint32_t w2 = w1 >> (e1 & 31u);
      const uint32_t e2 = *(LdsU32*)table_addr(w2, tsel, tmask);
      P[ch] = P[ch] + e1 + e2;
      const uint32_t nslot = __builtin_amdgcn_ubfe(P[ch], 5, 8);
      const bool slide = nslot != slot[ch];
      A[ch] = slide ? B[ch] : A[ch];
      B[ch] = slide ? C[ch] : B[ch];
      slot[ch] = nslot;
      C[ch] = *(LdsU32*)(rlb + (nslot << 7));
      const uint32_t s1 = e1 >> 16, s2 = e2 >> 16;
      if (SYMB == 4) {  // 4 grid bytes per pair; a piece every 4 pairs
        acc[ch][p & 3] = s1 | s2 << 16;
        if ((p & 3) == 3) {
          const int q = p >> 2;  // piece q of the chain's 64 codes: chunk kc0 + 2 ch + q / 2, half q % 2
          *reinterpret_cast<uint4*>(obase + ((size_t)(kc0 + 2 * ch + (q >> 1)) * 64 + 32 * (q & 1)) * 16) =
              make_uint4(acc[ch][0], acc[ch][1], acc[ch][2], acc[ch][3]);
        }
      } else {  // 2 codes per pair; a piece every 8 pairs
        const uint32_t v = s1 | s2 << 8;
        if (p & 1) acc[ch][(p >> 1) & 3] |= v << 16;
        else acc[ch][(p >> 1) & 3] = v;
        if ((p & 7) == 7)
          *reinterpret_cast<uint4*>(obase + ((size_t)(kc0 + ch) * 64 + 32 * (p >> 3)) * 16) =
              make_uint4(acc[ch][0], acc[ch][1], acc[ch][2], acc[ch][3]);
      }
    }
  }
}

bool decode_tiled_ok(const DevMat& M) {
  return M.K % 32 == 0 && (M.symbits != 4 || M.lut4) &&
         (M.packed || (M.split && M.rows && M.lut && M.max_rows + 2 <= 256));
}

size_t prefill_x_bytes(int m, int K) { return (size_t)((m + 63) / 64 * 64) * K * 4; }
size_t prefill_sx_bytes(int m, int K) { return (size_t)((m + 63) / 64 * 64) * (K / 32) * 4; }

__global__ void __launch_bounds__(256) k_prefill_x(PrefillX px) {
  __shared__ float part[PREFILL_X_LDS];
  prefill_x_block(px, (int)blockIdx.x, part);
}

hipError_t launch_prefill_prep(const DevMat& M, uint8_t* out, int tr0, int tr1, const PrefillX* x, hipStream_t s) {
  if (!decode_tiled_ok(M) || tr0 < 0 || tr0 >= tr1 || tr1 > M.NT) return hipErrorInvalidValue;
  PrefillX px{};
  if (x) {
    if (x->m < 1 || x->K % 256) return hipErrorInvalidValue;
    px = *x;
    px.blocks = (int)((size_t)((x->m + 63) / 64 * 64) * (x->K / 8) / 256);  // (a multiple of 256 threads)
  }
  if (M.packed) {
    if (px.blocks) hipLaunchKernelGGL(k_prefill_x, dim3(px.blocks), dim3(256), 0, s, px);
    return launch_unpack_tiled(M, out, tr0, tr1, s);
  }
  const int rows = M.max_rows + 2;
  const size_t sm = (size_t)rows * 128;
  auto* const kernel = M.symbits == 4 ? k_prefill_prep<4> : k_prefill_prep<8>;
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)sm);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kernel, dim3((unsigned)((tr1 - tr0) * M.KT + px.blocks)), dim3(256), sm, s, M, out, tr0, tr1, rows, px);
  return hipGetLastError();
}

// ── prefill GEMM on the matrix cores, Q4_K / Q5_K (path 2 and m > 8, the default for these formats) ─────────
// Y[t][n] = sum over super-blocks of d_n (x_t . w'_n) - dmin_n (Sx_t . m_n), where w'_k = sc_j q_k is the code scaled
// by its sub-block's 6-bit scale (at most 63 x 31 = 1953) and Sx_t,j the sum of x_t over sub-block j, m_n,j the
// sub-block's 6-bit min. Both dot products run on v_mfma_f32_32x32x16_f16 with x split into fp16 hi + lo (two
// products per weight, fp32 accumulation), the mins term as one K = 16 product per super-block (8 sub-blocks,
// zero-padded) with Sx split likewise; d and dmin applied once per super-block.
// Weights enter the products as w'/16, exact in fp16: a byte permute against 0x54 bytes makes fp16(64 + q/16) of each
// code, and one fma with sc and -64 sc leaves sc q / 16 (every intermediate exact); the 16 goes into d.
// Operand layout (32x32x16): lane l holds A[i = l % 32][k = 8 (l / 32) + 0..7] (token i) and B[k = 8 (l / 32) + 0..7]
// [j = l % 32] (weight row j), and receives D[i = 8 (r / 4) + 4 (l / 32) + r % 4][j = l % 32] in register r: a lane owns
// one weight row (one set of scales) per row tile and 16 tokens of the token tile.
// Block = WV waves over 64 weight rows (two row tiles) x 32 TT tokens; the waves split K by super-block (wave w takes
// super-blocks w, w + WV, ...) and their partial tiles are summed through LDS in wave order, so the result does not
// depend on timing.
// What bounds it: a wave of TT = 1 reads 6 KB of operands per 8 products (256 cycles of a SIMD's matrix core), 96 bytes a
// cycle of a CU where its vector cache gives 64; with TT = 2 the same codes serve 16 products (80 bytes a cycle, and half
// the scaling of codes per product). 64 x 64 tiles take all 256 registers of 2 waves per SIMD (128 in accumulators): the
// operand rings are 2 chunks deep instead of 4, side records and x sums are read through buffers (no per-lane addresses)
// two chunks ahead, and a tile's registers take its mins product before its own. Q4_K 14336 x 4096, m = 2048: 737 -> 520 us
// with the preparation, the totals put aside (below) included: 462 useful TFLOP/s a call, two products per weight, where a
// library fp16 GEMM of 8192 x 8192 x 8192 reaches 1176 on this card. Mins folded after the products instead: 527 us, 5
// registers spilled, and 1.2 % further from 64 bits.
// codes q0..q3 (bytes of qw) -> sc q / 16 as 4 fp16 in two words (nsc = -64 sc)
__device__ __forceinline__ uint2 scaled_codes16(uint32_t qw, h2v sc, h2v nsc) {
  const h2v a = __builtin_bit_cast(h2v, __builtin_amdgcn_perm(0x54545454u, qw, 0x04010400u));
  const h2v b = __builtin_bit_cast(h2v, __builtin_amdgcn_perm(0x54545454u, qw, 0x04030402u));
  return make_uint2(__builtin_bit_cast(uint32_t, __builtin_elementwise_fma(a, sc, nsc)),
                    __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(b, sc, nsc)));
}

// a row's Q4_K / Q5_K super-block record, compacted: the 8 scales and the 8 mins as bytes, d x 16 and dmin
struct KSide {
  uint32_t sc_lo, sc_hi, m_lo, m_hi;
  float d16, dmin;
};
__device__ __forceinline__ KSide kside(const uint32_t* w) {
  KSide k;
  k.sc_lo = w[1] & 0x3F3F3F3Fu;
  k.sc_hi = (w[3] & 0x0F0F0F0Fu) | ((w[1] >> 2) & 0x30303030u);
  k.m_lo = w[2] & 0x3F3F3F3Fu;
  k.m_hi = ((w[3] >> 4) & 0x0F0F0F0Fu) | ((w[2] >> 2) & 0x30303030u);
  k.d16 = 16.f * h2f(w[0]);
  k.dmin = h2f(w[0] >> 16);
  return k;
}
// sub-block j's scale as an fp16 pair
__device__ __forceinline__ h2v kside_sc(const KSide& k, int j) {
  const _Float16 v = (_Float16)(float)((((j < 4) ? k.sc_lo : k.sc_hi) >> (8 * (j & 3))) & 255u);
  return h2v{v, v};
}
// the 8 mins as the B operand of the mins product
__device__ __forceinline__ h8v kside_mins(const KSide& k) {
  h8v v;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    v[i] = (_Float16)(float)((k.m_lo >> (8 * i)) & 255u);
    v[4 + i] = (_Float16)(float)((k.m_hi >> (8 * i)) & 255u);
  }
  return v;
}

// Layouts (all lane-linear: one wave's load of a piece is one contiguous 1 KB read):
//   codes CT: per 32-row tile rt and 32-code chunk kc (the weights of one sub-block) a 1 KB piece at
//     (rt KC + kc) 1024, lane (h, c) = 32 h + c holding row c's codes 16 h .. 16 h + 15 of the chunk;
//   x XT: per 32-token tile tt, chunk kc, half (hi / lo) and step s a 1 KB piece at (((tt KC + kc) 2 + half) 2 + s)
//     1024, lane (h, c) holding x[token c][32 kc + 16 h + 8 s + 0..7] as fp16;
//   SXT: per token tile tt, super-block sb and half a 512-byte piece, lane c (< 32) holding Sx[token c][8 sb + 0..7].
// Step s of chunk kc gives lane (h, c) the weights 32 kc + 16 h + 8 s + 0..7 in both operands: the products of the
// 32 weights of the chunk are all taken once, in a different order than k, which a dot product does not see.
// The side records of one row of a wave's 64 through a buffer (no per-lane addresses): as the words side_load gives, but
// Q6_K's 18 bytes as the 5 aligned dwords that hold them (side_words; a side tensor ends with 16 bytes of padding).
template <int KQ>
__device__ __forceinline__ uint32_t side_voffset(int c) { return (uint32_t)(c * kq_sbytes(KQ)) & (KQ == KQ_Q6_K ? ~3u : ~0u); }
template <int KQ>
__device__ __forceinline__ void side_fetch(__amdgpu_buffer_rsrc_t r, uint32_t vo, int so, uint32_t* w) {
  if constexpr (KQ == KQ_IQ4_XS) {
    const auto v = __builtin_amdgcn_raw_buffer_load_b64(r, vo, so, 0);
    w[0] = v[0];
    w[1] = v[1];
  } else {
    const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, vo, so, 0);
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] = v[i];
    if constexpr (KQ == KQ_Q6_K) w[4] = __builtin_amdgcn_raw_buffer_load_b32(r, vo + 16, so, 0);
  }
}
template <int KQ>
__device__ __forceinline__ void side_words(const uint32_t* raw, int c, uint32_t* w) {
  const uint32_t sh = KQ == KQ_Q6_K ? 16u * (c & 1) : 0u;
#pragma unroll
  for (int i = 0; i < 4; ++i) w[i] = KQ == KQ_Q6_K ? __builtin_amdgcn_alignbit(raw[i + 1], raw[i], sh) : raw[i];
  w[4] = KQ == KQ_Q6_K ? raw[4] >> sh : 0u;
}

// The block's pair of row tiles and first token tile. With TT = 2 (many blocks) in an order by XCD: hardware deals
// consecutive blocks to the 8 XCDs, so block id takes place (id % 8) n / 8 + id / 8 of a list that runs over groups of 4
// token tile pairs and inside a group over row pairs: an XCD's L2 keeps a group's activations while each row pair's codes
// come by once (Q4_K 14336 x 4096, m = 2048: 528 -> 516 us, m = 512: 147 -> 143; groups of 1, 2 and 8: 529, 515, 529).
template <int TT>
__device__ __forceinline__ void block_tile(int& rp, int& tt) {
  rp = blockIdx.x;
  tt = blockIdx.y;
  if constexpr (TT > 1) {
    constexpr int G = 4;
    const int gx = gridDim.x, gy = gridDim.y, per = gx * gy / 8;
    int id = tt * gx + rp;
    if (id < 8 * per) id = (id & 7) * per + (id >> 3);
    const int g = id / (gx * G), rem = id - g * gx * G, gw = min(G, gy - g * G);
    rp = rem / gw;
    tt = g * G + rem - rp * gw;
  }
  tt *= TT;
}

// TT: token tiles of 32 per wave; WV: waves per block (the K split). The block's partial tiles -> LDS as
// part[wave][tile][r][lane] (lane-contiguous, no bank conflicts), then each thread sums its outputs over the waves in
// order; consecutive threads take consecutive lanes = consecutive weight rows. Tile = row tile + 2 token tile.
template <int TT, int WV>
__device__ __forceinline__ void store_tiles(const f16x16 (&tot)[2][TT], float* part, int wave, int lane, int row0, int tt0,
                                            int m, float* __restrict__ Y, int ldy) {
  constexpr int TILES = 2 * TT;
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < TT; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) part[((wave * TILES + a + 2 * b) * 16 + r) * 64 + lane] = tot[a][b][r];
  __syncthreads();
  for (int e = threadIdx.x; e < TILES * 16 * 64; e += 64 * WV) {
    const int tile = e >> 10, r = (e >> 6) & 15, l = e & 63;
    float acc = 0.f;
#pragma unroll
    for (int w = 0; w < WV; ++w) acc += part[w * TILES * 1024 + e];
    const int t = tt0 * 32 + 32 * (tile >> 1) + 8 * (r / 4) + 4 * (l >> 5) + (r % 4);
    if (t < m) Y[(size_t)t * ldy + row0 + 32 * (tile & 1) + (l & 31)] = acc;
  }
}

// A wave's totals to its part of the LDS (own: [tile][r / 4][lane]) and zero again, and added back.
template <int TT>
__device__ __forceinline__ void put_aside(f16x16 (&tot)[2][TT], f4v* own) {
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < TT; ++b) {
#pragma unroll
      for (int r = 0; r < 16; r += 4)
        own[(a + 2 * b) * 256 + r * 16] = f4v{tot[a][b][r], tot[a][b][r + 1], tot[a][b][r + 2], tot[a][b][r + 3]};
      tot[a][b] = f16x16{};
    }
}

template <int TT>
__device__ __forceinline__ void take_back(f16x16 (&tot)[2][TT], const f4v* own) {
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < TT; ++b)
#pragma unroll
      for (int r = 0; r < 16; r += 4) {
        const f4v v = own[(a + 2 * b) * 256 + r * 16];
#pragma unroll
        for (int k = 0; k < 4; ++k) tot[a][b][r + k] += v[k];
      }
}

template <int KQ, int TT, int WV>
__global__ void __launch_bounds__(64 * WV, 2 * 4 / WV) k_gemm_prefill(DevMat M, const uint8_t* __restrict__ CT, int row0,
                                                                     const uint16_t* __restrict__ XT,
                                                                     const uint16_t* __restrict__ SXT, int m,
                                                                     float* __restrict__ Y, int ldy) {
  static_assert(KQ == KQ_Q4_K || KQ == KQ_Q5_K, "scaled weights are exact in fp16 for Q4_K / Q5_K only");
  constexpr int SB = kq_sbytes(KQ), NSB = kq_symbits(KQ) == 4 ? 2 : 1;
  constexpr int RD = TT == 1 ? 4 : 2;  // chunks on the operand rings (RD - 1 ahead)
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, c = lane & 31;
  int rp, tt;  // pair of 32-row tiles of the chunk, first 32-token tile
  block_tile<TT>(rp, tt);
  const int K = M.K, KC = K / 32, NB = K / 256;
  // buffer resources over the block's codes (its two row tiles) and x (its token tiles): the lane's byte offset is
  // the only per-lane address, the chunk offset a scalar
  const __amdgpu_buffer_rsrc_t rc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint8_t*>(CT + (size_t)rp * 2 * KC * 1024), (short)0, 2 * KC * 1024, kBufferRsrcWord3);
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(XT + (size_t)tt * KC * 2048), (short)0, TT * KC * 4096, kBufferRsrcWord3);
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint8_t*>(M.side + side_record(row0 + rp * 64, 0, M.KT, NSB) * SB), (short)0, NB * 64 * SB + 16, kBufferRsrcWord3);
  const uint32_t vs = side_voffset<KQ>(c);  // row c's record, row c + 32's 32 SB on (a super-block's 64 records in a run)
  const __amdgpu_buffer_rsrc_t rsx = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(SXT + (size_t)tt * NB * 512), (short)0, TT * NB * 1024, kBufferRsrcWord3);
  const uint32_t vo = (uint32_t)lane * 16;
  // operands in flight: codes and x RD - 1 chunks ahead (one depth for both: the load counter completes in issue order);
  // 8 chunks per super-block keep the rings aligned
  auto load_q = [&](int kc, u32x4& qa, u32x4& qb) {
    qa = __builtin_amdgcn_raw_buffer_load_b128(rc, vo, kc * 1024, 0);
    qb = __builtin_amdgcn_raw_buffer_load_b128(rc, vo, (KC + kc) * 1024, 0);
  };
  auto load_x = [&](int kc, u32x4* x) {
#pragma unroll
    for (int b = 0; b < TT; ++b)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        x[4 * b + i] = __builtin_amdgcn_raw_buffer_load_b128(rx, vo + i * 1024, (b * KC + kc) * 4096, 0);
  };
  f16x16 tot[2][TT] = {};
  extern __shared__ float part[];
  // with 4 waves sharing K the totals are put aside half way, as in k_gemm_prefill_sub: 14336 x 4096, m = 2048 1.8e-7
  // from 64 bits without, 1.7e-7 with 8 waves and with this, for 1 to 2 % of the time
  int left = WV < 8 ? ((NB - wave + WV - 1) / WV + 1) / 2 : 0;
  bool aside = false;
  f4v* const own = reinterpret_cast<f4v*>(part) + wave * 2 * TT * 256 + lane;
  uint32_t swa[5] = {}, swb[5] = {};
  u32x4 qa[RD] = {}, qb[RD] = {}, xr[RD][4 * TT] = {};
  u32x4 sx[TT] = {};  // Sx of the super-block: lanes h = 0 the hi, h = 1 the lo halves
  auto load_sx = [&](int sb) {
#pragma unroll
    for (int b = 0; b < TT; ++b) sx[b] = __builtin_amdgcn_raw_buffer_load_b128(rsx, vo, (b * NB + sb) * 1024, 0);
  };
  if (wave < NB) {
    side_fetch<KQ>(rs, vs, wave * (64 * SB), swa);
    side_fetch<KQ>(rs, vs + 32 * SB, wave * (64 * SB), swb);
    load_sx(wave);
#pragma unroll
    for (int i = 0; i < RD - 1; ++i) {
      load_q(wave * 8 + i, qa[i], qb[i]);
      load_x(wave * 8 + i, xr[i]);
    }
  }
  for (int sb = wave; sb < NB; sb += WV) {
    const KSide ka = kside(swa), kb = kside(swb);
    const int nsb = sb + WV;
    f16x16 d[2][TT];
    // mins, into the totals before the super-block's products (which are the larger term): A2 = the tokens' Sx over the 8
    // sub-blocks, hi in k 0..7 and lo in k 8..15, B2 = the row's 8 mins in both; in the tiles' registers
    const h8v mn[2] = {kside_mins(ka), kside_mins(kb)};
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < TT; ++b)
        d[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(h8v, sx[b]), mn[a], f16x16{}, 0, 0, 0);
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      const float dmin = a ? kb.dmin : ka.dmin;
#pragma unroll
      for (int b = 0; b < TT; ++b) {
#pragma unroll
        for (int r = 0; r < 16; ++r) tot[a][b][r] = fmaf(-dmin, d[a][b][r], tot[a][b][r]);
        asm volatile("" : "+v"(tot[a][b]));
        d[a][b] = f16x16{};
      }
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {  // the super-block's 8 chunks (sub-blocks)
      if (j < 9 - RD || nsb < NB) {
        const int kn = j < 9 - RD ? sb * 8 + j + RD - 1 : nsb * 8 + j - (9 - RD);
        load_q(kn, qa[(j + RD - 1) % RD], qb[(j + RD - 1) % RD]);
        load_x(kn, xr[(j + RD - 1) % RD]);
      }
      if (j == 6 && nsb < NB) {  // the next super-block's records and sums (from chunk 5 on they would spill 8 registers)
        side_fetch<KQ>(rs, vs, nsb * (64 * SB), swa);
        side_fetch<KQ>(rs, vs + 32 * SB, nsb * (64 * SB), swb);
        load_sx(nsb);
      }
      __builtin_amdgcn_sched_barrier(0);  // keep the loads issued here, ahead of this chunk's products
      const u32x4 ca = qa[j % RD], cb = qb[j % RD];
      const u32x4* xc = xr[j % RD];
      const h2v sca = kside_sc(ka, j), scb = kside_sc(kb, j);
      const h2v n64 = {(_Float16)-64.f, (_Float16)-64.f};
      const h2v nsa = sca * n64, nsb2 = scb * n64;
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        const uint2 a0 = scaled_codes16(ca[2 * st], sca, nsa), a1 = scaled_codes16(ca[2 * st + 1], sca, nsa);
        const uint2 b0 = scaled_codes16(cb[2 * st], scb, nsb2), b1 = scaled_codes16(cb[2 * st + 1], scb, nsb2);
        const h8v w[2] = {__builtin_bit_cast(h8v, make_uint4(a0.x, a0.y, a1.x, a1.y)),
                          __builtin_bit_cast(h8v, make_uint4(b0.x, b0.y, b1.x, b1.y))};
#pragma unroll
        for (int half = 0; half < 2; ++half)  // x hi, then lo
#pragma unroll
          for (int b = 0; b < TT; ++b)
#pragma unroll
            for (int a = 0; a < 2; ++a)
              d[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(h8v, xc[4 * b + 2 * half + st]), w[a], d[a][b], 0, 0, 0);
      }
    }
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      const float d16 = a ? kb.d16 : ka.d16;
#pragma unroll
      for (int b = 0; b < TT; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) tot[a][b][r] = fmaf(d16, d[a][b][r], tot[a][b][r]);
    }
    if (WV < 8 && --left == 0 && nsb < NB) {
      aside = true;
      put_aside<TT>(tot, own);
    }
  }
  if (aside) take_back<TT>(tot, own);
  store_tiles<TT, WV>(tot, part, wave, lane, row0 + rp * 64, tt, m, Y, ldy);
}

// ── prefill GEMM on the matrix cores, Q6_K / IQ4_XS: unscaled grid weights, folded per sub-block ─────────────
// Y[t][n] = sum over sub-blocks j of d_n s_n,j (x_t . f(q_n)) with f(q) = q - 32 (Q6_K) or kv[q] (IQ4_XS): integers of
// at most 8 bits, exact in fp16, where the scaled s f(q) (up to 128 x 32 or 32 x 127) is not. Each sub-block's
// products go to a fresh accumulator tile (x split into fp16 hi + lo, as k_gemm_prefill), folded into the fp32 total
// with d s_j (exact in fp32) once the sub-block is in. No offsets: neither format has mins.
// The block, the waves' split of K, the rings and the wave-order LDS sum are those of k_gemm_prefill; the fold (an FMA per
// output and sub-block) is as much VALU as there is matrix-core time for Q6_K: 4096 x 14336, m = 512 takes 170 us (64 x 32
// tiles 200). A step's K = 16
// must lie in one sub-block:
//   IQ4_XS (32-weight sub-blocks) takes k_gemm_prefill's steps (a chunk = a sub-block) over the grid bytes kv[q] + 128
//   of the tiled codes; weights fp16(1024 + g) from a byte permute against 0x64, minus 1152.
//   Q6_K (16-weight sub-blocks) takes weights 16 s + 8 h + 0..7 of the chunk in step s for lane (h, c), so that step s
//   is sub-block 2 kc + s: 8 bytes of the codes piece at lane slot 32 s + c, byte 8 h, and the x piece of step h at
//   lane slot 32 s + c (the products of a chunk are still each taken once); weights fp16(1024 + q) minus 1056.
template <int KQ, int TT, int WV>
__global__ void __launch_bounds__(64 * WV, 2 * 4 / WV) k_gemm_prefill_sub(DevMat M, const uint8_t* __restrict__ CT, int row0,
                                                                   const uint16_t* __restrict__ XT, int m,
                                                                   float* __restrict__ Y, int ldy) {
  static_assert(KQ == KQ_Q6_K || KQ == KQ_IQ4_XS, "per-sub-block folding: Q6_K and IQ4_XS");
  constexpr bool Q6 = KQ == KQ_Q6_K;
  constexpr int SB = kq_sbytes(KQ), NSB = kq_symbits(KQ) == 4 ? 2 : 1;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, c = lane & 31, h = lane >> 5;
  constexpr int RD = TT == 1 ? 4 : 2;  // chunks on the operand rings (RD - 1 ahead)
  int rp, tt;
  block_tile<TT>(rp, tt);
  const int K = M.K, KC = K / 32, NB = K / 256;
  const __amdgpu_buffer_rsrc_t rc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint8_t*>(CT + (size_t)rp * 2 * KC * 1024), (short)0, 2 * KC * 1024, kBufferRsrcWord3);
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(XT + (size_t)tt * KC * 2048), (short)0, TT * KC * 4096, kBufferRsrcWord3);
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint8_t*>(M.side + side_record(row0 + rp * 64, 0, M.KT, NSB) * SB), (short)0, NB * 64 * SB + 16, kBufferRsrcWord3);
  const uint32_t vs = side_voffset<KQ>(c);  // row c's record, row c + 32's 32 SB on (a super-block's 64 records in a run)
  // the lane's byte offsets of step s's operands in a chunk's codes piece and in its x pieces (hi, then lo 2 KB on)
  uint32_t vq[2], vx[2];
#pragma unroll
  for (int st = 0; st < 2; ++st) {
    vq[st] = Q6 ? (uint32_t)(32 * st + c) * 16 + 8 * h : (uint32_t)lane * 16;
    vx[st] = Q6 ? (uint32_t)h * 1024 + (uint32_t)(32 * st + c) * 16 : (uint32_t)st * 1024 + (uint32_t)lane * 16;
  }
  // a chunk's codes as 4 words per row tile, words 2 s and 2 s + 1 = the 8 weights of step s
  auto load_q = [&](int kc, u32x4& qa, u32x4& qb) {
    if (Q6) {
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        const auto a = __builtin_amdgcn_raw_buffer_load_b64(rc, vq[st], kc * 1024, 0);
        const auto b = __builtin_amdgcn_raw_buffer_load_b64(rc, vq[st], (KC + kc) * 1024, 0);
        qa[2 * st] = a[0];
        qa[2 * st + 1] = a[1];
        qb[2 * st] = b[0];
        qb[2 * st + 1] = b[1];
      }
    } else {
      qa = __builtin_amdgcn_raw_buffer_load_b128(rc, vq[0], kc * 1024, 0);
      qb = __builtin_amdgcn_raw_buffer_load_b128(rc, vq[0], (KC + kc) * 1024, 0);
    }
  };
  auto load_x = [&](int kc, u32x4* x) {  // x[2 half + s]
#pragma unroll
    for (int b = 0; b < TT; ++b)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        x[4 * b + i] = __builtin_amdgcn_raw_buffer_load_b128(rx, vx[i & 1] + (i >> 1) * 2048, (b * KC + kc) * 4096, 0);
  };
  // 4 weights (bytes of qw) -> fp16 f(q) in two words
  const h2v bias = Q6 ? h2v{(_Float16)-1056.f, (_Float16)-1056.f} : h2v{(_Float16)-1152.f, (_Float16)-1152.f};
  auto grid16 = [&](uint32_t qw) -> uint2 {
    const h2v a = __builtin_bit_cast(h2v, __builtin_amdgcn_perm(0x64646464u, qw, 0x04010400u));
    const h2v b = __builtin_bit_cast(h2v, __builtin_amdgcn_perm(0x64646464u, qw, 0x04030402u));
    return make_uint2(__builtin_bit_cast(uint32_t, a + bias), __builtin_bit_cast(uint32_t, b + bias));
  };
  // d s_j of sub-block j of a super-block record (words as side_load)
  auto sub_scale = [&](const uint32_t* w, int j) -> float {
    if (Q6) return h2f(w[4]) * (float)(int)(int8_t)(uint8_t)(w[j >> 2] >> (8 * (j & 3)));
    const uint32_t ls = ((w[1] >> (4 * j)) & 15u) | ((w[0] >> (16 + 2 * j)) & 3u) << 4;
    return h2f(w[0]) * (float)((int)ls - 32);
  };
  f16x16 tot[2][TT] = {};
  extern __shared__ float part[];
  // a total takes 8 or 16 rounded additions per super-block: half way (with 4 waves sharing K)
  // it is put aside in the wave's part of the LDS, which keeps the sums' distance from 64 bits (Q6_K, K = 14336 and 4096:
  // 2.1e-7 and 1.3e-7 with 8 waves and with this, 2.8e-7 and 1.6e-7 with 4 waves without it)
  int left = WV < 8 ? ((NB - wave + WV - 1) / WV + 1) / 2 : 0;
  bool aside = false;
  f4v* const own = reinterpret_cast<f4v*>(part) + wave * 2 * TT * 256 + lane;  // [tile][r / 4][lane]
  uint32_t swa[5] = {}, swb[5] = {};
  u32x4 qa[RD] = {}, qb[RD] = {}, xr[RD][4 * TT] = {};
  if (wave < NB) {
    side_fetch<KQ>(rs, vs, wave * (64 * SB), swa);
    side_fetch<KQ>(rs, vs + 32 * SB, wave * (64 * SB), swb);
#pragma unroll
    for (int i = 0; i < RD - 1; ++i) {
      load_q(wave * 8 + i, qa[i], qb[i]);
      load_x(wave * 8 + i, xr[i]);
    }
  }
  for (int sb = wave; sb < NB; sb += WV) {
    uint32_t wr[2][5];
    side_words<KQ>(swa, c, wr[0]);
    side_words<KQ>(swb, c, wr[1]);
    const int nsb = sb + WV;
#pragma unroll
    for (int j = 0; j < 8; ++j) {  // the super-block's 8 chunks
      if (j < 9 - RD || nsb < NB) {
        const int kn = j < 9 - RD ? sb * 8 + j + RD - 1 : nsb * 8 + j - (9 - RD);
        load_q(kn, qa[(j + RD - 1) % RD], qb[(j + RD - 1) % RD]);
        load_x(kn, xr[(j + RD - 1) % RD]);
      }
      if (j == 5 && nsb < NB) {  // the next super-block's records (from the start they would cost 10 registers more)
        side_fetch<KQ>(rs, vs, nsb * (64 * SB), swa);
        side_fetch<KQ>(rs, vs + 32 * SB, nsb * (64 * SB), swb);
      }
      __builtin_amdgcn_sched_barrier(0);  // keep the loads issued here, ahead of this chunk's products
      const u32x4 ca = qa[j % RD], cb = qb[j % RD];
      const u32x4* xc = xr[j % RD];
      f16x16 d[2][TT] = {};
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        const uint2 a0 = grid16(ca[2 * st]), a1 = grid16(ca[2 * st + 1]);
        const uint2 b0 = grid16(cb[2 * st]), b1 = grid16(cb[2 * st + 1]);
        const h8v w[2] = {__builtin_bit_cast(h8v, make_uint4(a0.x, a0.y, a1.x, a1.y)),
                          __builtin_bit_cast(h8v, make_uint4(b0.x, b0.y, b1.x, b1.y))};
#pragma unroll
        for (int b = 0; b < TT; ++b)
#pragma unroll
          for (int a = 0; a < 2; ++a) {
            if (Q6 && st == 1) d[a][b] = f16x16{};
#pragma unroll
            for (int half = 0; half < 2; ++half)
              d[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(h8v, xc[4 * b + 2 * half + st]), w[a], d[a][b], 0, 0, 0);
          }
        if (Q6 || st == 1) {  // the sub-block is in: fold it
          const int js = Q6 ? 2 * j + st : j;
#pragma unroll
          for (int a = 0; a < 2; ++a) {
            const float sc = sub_scale(wr[a], js);
#pragma unroll
            for (int b = 0; b < TT; ++b) {
#pragma unroll
              for (int r = 0; r < 16; ++r) tot[a][b][r] = fmaf(sc, d[a][b][r], tot[a][b][r]);
              // keep the fold here: sunk below the chunk loop's branches it would hold every chunk's tiles live (spills)
              asm volatile("" : "+v"(tot[a][b]));
            }
          }
          if (Q6 && TT > 1) __builtin_amdgcn_sched_barrier(0);  // (else the next step's operands spill)
        }
      }
    }
    if (WV < 8 && --left == 0 && nsb < NB) {
      aside = true;
      put_aside<TT>(tot, own);
    }
  }
  if (aside) take_back<TT>(tot, own);
  store_tiles<TT, WV>(tot, part, wave, lane, row0 + rp * 64, tt, m, Y, ldy);
}

template <int KQ, int TT, int WV>
static hipError_t gemm_prefill(const DevMat& M, const uint8_t* CT, int row0, int nrows, const uint16_t* x, const uint16_t* sx,
                               int m, float* Y, int ldy, hipStream_t s) {
  const dim3 grid(nrows / 64, (m + 32 * TT - 1) / (32 * TT)), block(64 * WV);
  const size_t smem = (size_t)WV * 2 * TT * 16 * 64 * 4;
  if constexpr (KQ == KQ_Q4_K || KQ == KQ_Q5_K) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_gemm_prefill<KQ, TT, WV>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((k_gemm_prefill<KQ, TT, WV>), grid, block, smem, s, M, CT, row0, x, sx, m, Y, ldy);
  } else {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_gemm_prefill_sub<KQ, TT, WV>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((k_gemm_prefill_sub<KQ, TT, WV>), grid, block, smem, s, M, CT, row0, x, m, Y, ldy);
  }
  return hipGetLastError();
}

// 64 x 64 or 64 x 32 tiles (rows x tokens) per wave, for a matrix of `rows` row pairs whose GEMM runs over at most `chunk` of
// them at a time (both of the matrix alone, not of what the scratch has grown to: the same bits from call to call). A larger
// tile takes 3/4 of the time per product, but its blocks fill the 256 CUs in coarser steps and may hold 32 tokens of
// padding. Time goes with the fullest CU's blocks and, a quarter as much, with all of them: c(b) = 3 ceil(b / 256) + b / 256
// per launch. Fitted to 230 shapes of all formats (m = 9 .. 2048, N = 2048 .. 28672, K = 512 .. 14336): within 1 % of the best
// of the four on the mean. us per call, preparation included, of 64 x 64 by 4 waves / by 8 / 64 x 32 by 4 / by 8: Q4_K
// 14336 x 4096, m = 9 36.6 / 34.0 / 32.9 / 30.1, m = 33 36.5 / 34.0 / 39.2 / 42.4, m = 2048 546 / 580 / 674 / 736; Q6_K
// 16384 x 1024, m = 65 29.0 / 30.5 / 24.4 / 27.4; IQ4_XS 6400 x 14336 (two launches), m = 200 192 / 190 / 157 / 157, m = 300
// 204 / 204 / 226 / 231; Q4_K 2048 x 14336, m = 300 75 / 68 / 78 / 82.
// K split over 4 waves where the blocks are more than the CUs, else over 8.
int prefill_tiles(int rows, int chunk, int m) {
  long long c64 = 0, c32 = 0;
  const long long t64 = (m + 63) / 64, t32 = (m + 31) / 32, first = std::min(rows, chunk);
  for (long long r = rows; r > 0; r -= chunk) {
    const long long n = std::min<long long>(r, chunk), b64 = n * t64, b32 = n * t32;
    c64 += (b64 + 255) / 256 * 768 + b64;
    c32 += (b32 + 255) / 256 * 768 + b32;
  }
  if (2 * c32 > 3 * c64) return first * t64 > 256 ? PREFILL_64X64_4 : PREFILL_64X64_8;
  return first * t32 > 256 ? PREFILL_64X32_4 : PREFILL_64X32_8;
}

template <int KQ>
static hipError_t gemm_prefill_any(const DevMat& M, const uint8_t* CT, int row0, int nrows, const uint16_t* x,
                                   const uint16_t* sx, int m, int tiles, float* Y, int ldy, hipStream_t s) {
  switch (tiles) {
    case PREFILL_64X64_4: return gemm_prefill<KQ, 2, 4>(M, CT, row0, nrows, x, sx, m, Y, ldy, s);
    case PREFILL_64X64_8: return gemm_prefill<KQ, 2, 8>(M, CT, row0, nrows, x, sx, m, Y, ldy, s);
    case PREFILL_64X32_4: return gemm_prefill<KQ, 1, 4>(M, CT, row0, nrows, x, sx, m, Y, ldy, s);
    case PREFILL_64X32_8: return gemm_prefill<KQ, 1, 8>(M, CT, row0, nrows, x, sx, m, Y, ldy, s);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_gemm_prefill(const DevMat& M, const uint8_t* CT, int row0, int nrows, const void* XT,
                               const void* SXT, int m, int tiles, float* Y, int ldy, hipStream_t s) {
  if (nrows < 1 || m < 1 || nrows % 64 || M.K % 256) return hipErrorInvalidValue;
  const uint16_t* x = static_cast<const uint16_t*>(XT);
  const uint16_t* sx = static_cast<const uint16_t*>(SXT);
  switch (M.kqt) {
    case KQ_Q4_K: return gemm_prefill_any<KQ_Q4_K>(M, CT, row0, nrows, x, sx, m, tiles, Y, ldy, s);
    case KQ_Q5_K: return gemm_prefill_any<KQ_Q5_K>(M, CT, row0, nrows, x, sx, m, tiles, Y, ldy, s);
    case KQ_Q6_K: return gemm_prefill_any<KQ_Q6_K>(M, CT, row0, nrows, x, sx, m, tiles, Y, ldy, s);
    case KQ_IQ4_XS: return gemm_prefill_any<KQ_IQ4_XS>(M, CT, row0, nrows, x, sx, m, tiles, Y, ldy, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace lw
