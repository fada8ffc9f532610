// Prefill (m > 8): codes decoded to a tiled layout, activations split and tiled, GEMM on the matrix cores.
#include "lw_device.h"

namespace lw {

// x of the prefill GEMM: fp32 X [m][K] -> XT (fp16 hi = fp16(x), lo = fp16(x - hi)) and SXT (per sub-block of 32
// weights s = ((a0 + a1) + (a2 + a3)), a_q the in-order fp32 sum of its q-th 8 values, as fp16 hi / lo), tokens
// padded with zeros to a multiple of 64. Thread = (chunk, q, token c of the tile): the 32 threads of one q write one
// lane-linear 512-byte run of a piece; the chunk's four a_q meet in LDS.
__device__ __forceinline__ void prefill_x_block(const PrefillX& px, int block) {
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
  __shared__ float part[2][4][32];                       // the block's two chunks
  const int cb = (threadIdx.x >> 7) & 1;
  part[cb][q][c] = sum;
  __syncthreads();
  if (q == 0) {
    const float s = (part[cb][0][c] + part[cb][1][c]) + (part[cb][2][c] + part[cb][3][c]);
    const _Float16 hi = (_Float16)s;
    uint16_t* sx = SXT + ((((size_t)tt * NB + (kc >> 3)) * 2) * 32 + c) * 8 + (kc & 7);
    sx[0] = __builtin_bit_cast(uint16_t, hi);
    sx[32 * 8] = __builtin_bit_cast(uint16_t, (_Float16)(s - (float)hi));
  }
}


// Codes in the prefill GEMM's tiled layout (launch_decode_tiled): one block of 4 waves per tile as k_decode_split,
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
  __shared__ __align__(16) uint32_t lut4[LUTN];  // the only static LDS object: at LDS address 0 (table_addr ORs it in)
  extern __shared__ __align__(16) uint32_t tw[];
  const int KT = M.KT, KC = M.K / 32;
  if ((int)blockIdx.x < px.blocks) {
    prefill_x_block(px, (int)blockIdx.x);
    return;
  }
  const int t = tr0 * KT + (int)blockIdx.x - px.blocks;
  const int tc = t % KT, tr = t / KT;
  const int R = min((int)M.rows[t] + 2, stage_rows);
  if (SYMB == 4) {  // entries len | grid byte of the pair's first code << 16 | second << 24 (decode_table4)
    for (int i = threadIdx.x; i < LUTN / 4; i += 256)
      reinterpret_cast<uint4*>(lut4)[i] = reinterpret_cast<const uint4*>(M.lut4)[i];
  } else {  // sym | len << 8 -> len | sym << 16, 8 entries a thread
    static_assert(LUTN == 8 * 256, "8 entries per thread");
    const uint4 v = reinterpret_cast<const uint4*>(M.lut)[threadIdx.x];
    auto entry = [](uint32_t e) { return (e >> 8 & 255u) | (e & 255u) << 16; };
    uint4* o = reinterpret_cast<uint4*>(lut4) + 2 * threadIdx.x;
    o[0] = make_uint4(entry(v.x), entry(v.x >> 16), entry(v.y), entry(v.y >> 16));
    o[1] = make_uint4(entry(v.z), entry(v.z >> 16), entry(v.w), entry(v.w >> 16));
  }
  const uint4* src = reinterpret_cast<const uint4*>(M.words + M.tbase[t]);
  for (int i = threadIdx.x; i < 8 * R; i += 256) reinterpret_cast<uint4*>(tw)[i] = src[i];
  __syncthreads();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, l = lane & 31, f = lane >> 5;
  const int k = 4 * f + wave;  // segment of bit-lane l: row f * 32 + l, symbols 64 wave .. 64 wave + 63
  const uint32_t tsel = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const uint32_t*)lut4;
  uint32_t tmask = 0x1FFCu;
  asm volatile("" : "+v"(tmask));
  const uint32_t rlb = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint32_t*)(tw + l);
  uint32_t P[2], slot[2], A[2], B[2], C[2];
#pragma unroll
  for (int ch = 0; ch < 2; ++ch) {
    P[ch] = (uint32_t)M.split[((size_t)t * SPLITS + 2 * k + ch) * 32 + (uint32_t)l] - GUARD_BITS + 64u;
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

__global__ void __launch_bounds__(256) k_prefill_x(PrefillX px) { prefill_x_block(px, (int)blockIdx.x); }

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
// Block = GEMM_WAVES waves over 64 weight rows (two row tiles) x 32 tokens; the waves split K by super-block (wave w
// takes super-blocks w, w + GEMM_WAVES, ...) and their partial tiles are summed through LDS in wave order, so the
// result does not depend on timing. A skinny prefill (m = 128, N = 4096) gives 256 blocks.
constexpr int GEMM_WAVES = 8;
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
// the 8 mins as the B operand of the mins product (k 0..7; lanes h = 1 pass zeros)
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
template <int KQ>
__global__ void __launch_bounds__(64 * GEMM_WAVES) k_gemm_prefill(DevMat M, const uint8_t* __restrict__ CT, int row0,
                                                               const uint16_t* __restrict__ XT,
                                                               const uint16_t* __restrict__ SXT, int m,
                                                               float* __restrict__ Y, int ldy) {
  static_assert(KQ == KQ_Q4_K || KQ == KQ_Q5_K, "scaled weights are exact in fp16 for Q4_K / Q5_K only");
  constexpr int SB = kq_sbytes(KQ), NSB = kq_symbits(KQ) == 4 ? 2 : 1;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, c = lane & 31, h = lane >> 5;
  const int rp = blockIdx.x, tt = blockIdx.y;            // pair of 32-row tiles of the chunk, 32-token tile
  const int K = M.K, KC = K / 32, NB = K / 256;
  const int nA = rp * 64 + c, nB = nA + 32;              // the lane's weight rows within the chunk
  // buffer resources over the block's codes (its two row tiles) and x (its token tile): the lane's byte offset is
  // the only per-lane address, the chunk offset a scalar
  const __amdgpu_buffer_rsrc_t rc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint8_t*>(CT + (size_t)rp * 2 * KC * 1024), (short)0, 2 * KC * 1024, kBufferRsrcWord3);
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(XT + (size_t)tt * KC * 2048), (short)0, KC * 4096, kBufferRsrcWord3);
  const uint16_t* sxw = SXT + (size_t)tt * NB * 512 + c * 8;
  const uint32_t vo = (uint32_t)lane * 16;
  // operands in flight: codes and x three chunks ahead on 4-slot rings (one depth for both: the load counter
  // completes in issue order); 8 chunks per super-block keep the rings aligned
  auto load_q = [&](int kc, u32x4& qa, u32x4& qb) {
    qa = __builtin_amdgcn_raw_buffer_load_b128(rc, vo, kc * 1024, 0);
    qb = __builtin_amdgcn_raw_buffer_load_b128(rc, vo, (KC + kc) * 1024, 0);
  };
  auto load_x = [&](int kc, u32x4* x) {
#pragma unroll
    for (int i = 0; i < 4; ++i) x[i] = __builtin_amdgcn_raw_buffer_load_b128(rx, vo + i * 1024, kc * 4096, 0);
  };
  f16x16 totA = {}, totB = {};
  uint32_t swa[5] = {}, swb[5] = {};
  u32x4 qa[4] = {}, qb[4] = {}, xr[4][4] = {};
  if (wave < NB) {
    side_load<KQ>(M.side + side_record(row0 + nA, wave, M.KT, NSB) * SB, swa);
    side_load<KQ>(M.side + side_record(row0 + nB, wave, M.KT, NSB) * SB, swb);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      load_q(wave * 8 + i, qa[i], qb[i]);
      load_x(wave * 8 + i, xr[i]);
    }
  }
  for (int sb = wave; sb < NB; sb += GEMM_WAVES) {
    const KSide ka = kside(swa), kb = kside(swb);
    const int nsb = sb + GEMM_WAVES;
    if (nsb < NB) {
      side_load<KQ>(M.side + side_record(row0 + nA, nsb, M.KT, NSB) * SB, swa);
      side_load<KQ>(M.side + side_record(row0 + nB, nsb, M.KT, NSB) * SB, swb);
    }
    uint4 sxh = {}, sxl = {};  // Sx of this super-block, loaded at chunk 5
    f16x16 dA = {}, dB = {};
#pragma unroll
    for (int j = 0; j < 8; ++j) {  // the super-block's 8 chunks (sub-blocks)
      if (j < 5 || nsb < NB) {
        const int kn = j < 5 ? sb * 8 + j + 3 : nsb * 8 + j - 5;
        load_q(kn, qa[(j + 3) & 3], qb[(j + 3) & 3]);
        load_x(kn, xr[(j + 3) & 3]);
      }
      if (j == 5 && h == 0) {  // lanes h = 0 hold the mins product's k 0..7; k 8..15 stay zero
        sxh = *reinterpret_cast<const uint4*>(sxw + (size_t)sb * 512);
        sxl = *reinterpret_cast<const uint4*>(sxw + (size_t)sb * 512 + 256);
      }
      __builtin_amdgcn_sched_barrier(0);  // keep the loads issued here, ahead of this chunk's products
      const u32x4 ca = qa[j & 3], cb = qb[j & 3];
      const u32x4* xc = xr[j & 3];
      const h2v sca = kside_sc(ka, j), scb = kside_sc(kb, j);
      const h2v n64 = {(_Float16)-64.f, (_Float16)-64.f};
      const h2v nsa = sca * n64, nsb2 = scb * n64;
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        const uint2 a0 = scaled_codes16(ca[2 * st], sca, nsa), a1 = scaled_codes16(ca[2 * st + 1], sca, nsa);
        const uint2 b0 = scaled_codes16(cb[2 * st], scb, nsb2), b1 = scaled_codes16(cb[2 * st + 1], scb, nsb2);
        const h8v wa = __builtin_bit_cast(h8v, make_uint4(a0.x, a0.y, a1.x, a1.y));
        const h8v wb = __builtin_bit_cast(h8v, make_uint4(b0.x, b0.y, b1.x, b1.y));
        const h8v xh = __builtin_bit_cast(h8v, xc[st]), xl = __builtin_bit_cast(h8v, xc[2 + st]);
        dA = __builtin_amdgcn_mfma_f32_32x32x16_f16(xh, wa, dA, 0, 0, 0);
        dB = __builtin_amdgcn_mfma_f32_32x32x16_f16(xh, wb, dB, 0, 0, 0);
        dA = __builtin_amdgcn_mfma_f32_32x32x16_f16(xl, wa, dA, 0, 0, 0);
        dB = __builtin_amdgcn_mfma_f32_32x32x16_f16(xl, wb, dB, 0, 0, 0);
      }
    }
    // mins: A2 = the tokens' Sx over the super-block's 8 sub-blocks, B2 = the row's 8 mins
    h8v ma = {}, mb = {};
    if (h == 0) {
      ma = kside_mins(ka);
      mb = kside_mins(kb);
    }
    f16x16 mA = {}, mB = {};
    mA = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(h8v, sxh), ma, mA, 0, 0, 0);
    mB = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(h8v, sxh), mb, mB, 0, 0, 0);
    mA = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(h8v, sxl), ma, mA, 0, 0, 0);
    mB = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(h8v, sxl), mb, mB, 0, 0, 0);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      totA[r] = fmaf(ka.d16, dA[r], fmaf(-ka.dmin, mA[r], totA[r]));
      totB[r] = fmaf(kb.d16, dB[r], fmaf(-kb.dmin, mB[r], totB[r]));
    }
  }
  // partial tiles -> LDS as part[wave][row tile][r][lane] (lane-contiguous, no bank conflicts), then each thread
  // sums its outputs over the waves in order; consecutive threads take consecutive lanes = consecutive weight rows
  __shared__ float part[GEMM_WAVES][2][16][64];
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    part[wave][0][r][lane] = totA[r];
    part[wave][1][r][lane] = totB[r];
  }
  __syncthreads();
  for (int e = threadIdx.x; e < 2 * 16 * 64; e += 64 * GEMM_WAVES) {
    const int half = e >> 10, r = (e >> 6) & 15, l = e & 63;
    float acc = 0.f;
#pragma unroll
    for (int w = 0; w < GEMM_WAVES; ++w) acc += part[w][half][r][l];
    const int t = tt * 32 + 8 * (r / 4) + 4 * (l >> 5) + (r % 4);
    if (t < m) Y[(size_t)t * ldy + row0 + rp * 64 + 32 * half + (l & 31)] = acc;
  }
}

// ── prefill GEMM on the matrix cores, Q6_K / IQ4_XS: unscaled grid weights, folded per sub-block ─────────────
// Y[t][n] = sum over sub-blocks j of d_n s_n,j (x_t . f(q_n)) with f(q) = q - 32 (Q6_K) or kv[q] (IQ4_XS): integers of
// at most 8 bits, exact in fp16, where the scaled s f(q) (up to 128 x 32 or 32 x 127) is not. Each sub-block's
// products go to a fresh accumulator tile (x split into fp16 hi + lo, as k_gemm_prefill), folded into the fp32 total
// with d s_j (exact in fp32) once the sub-block is in. No offsets: neither format has mins.
// The block, the waves' split of K, the rings and the wave-order LDS sum are those of k_gemm_prefill. A step's K = 16
// must lie in one sub-block:
//   IQ4_XS (32-weight sub-blocks) takes k_gemm_prefill's steps (a chunk = a sub-block) over the grid bytes kv[q] + 128
//   of the tiled codes; weights fp16(1024 + g) from a byte permute against 0x64, minus 1152.
//   Q6_K (16-weight sub-blocks) takes weights 16 s + 8 h + 0..7 of the chunk in step s for lane (h, c), so that step s
//   is sub-block 2 kc + s: 8 bytes of the codes piece at lane slot 32 s + c, byte 8 h, and the x piece of step h at
//   lane slot 32 s + c (the products of a chunk are still each taken once); weights fp16(1024 + q) minus 1056.
template <int KQ>
__global__ void __launch_bounds__(64 * GEMM_WAVES) k_gemm_prefill_sub(DevMat M, const uint8_t* __restrict__ CT, int row0,
                                                                   const uint16_t* __restrict__ XT, int m,
                                                                   float* __restrict__ Y, int ldy) {
  static_assert(KQ == KQ_Q6_K || KQ == KQ_IQ4_XS, "per-sub-block folding: Q6_K and IQ4_XS");
  constexpr bool Q6 = KQ == KQ_Q6_K;
  constexpr int SB = kq_sbytes(KQ), NSB = kq_symbits(KQ) == 4 ? 2 : 1;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, c = lane & 31, h = lane >> 5;
  const int rp = blockIdx.x, tt = blockIdx.y;
  const int K = M.K, KC = K / 32, NB = K / 256;
  const int nA = rp * 64 + c, nB = nA + 32;
  const __amdgpu_buffer_rsrc_t rc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint8_t*>(CT + (size_t)rp * 2 * KC * 1024), (short)0, 2 * KC * 1024, kBufferRsrcWord3);
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(XT + (size_t)tt * KC * 2048), (short)0, KC * 4096, kBufferRsrcWord3);
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
    for (int i = 0; i < 4; ++i) x[i] = __builtin_amdgcn_raw_buffer_load_b128(rx, vx[i & 1] + (i >> 1) * 2048, kc * 4096, 0);
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
  f16x16 totA = {}, totB = {};
  uint32_t swa[5] = {}, swb[5] = {};
  u32x4 qa[4] = {}, qb[4] = {}, xr[4][4] = {};
  if (wave < NB) {
    side_load<KQ>(M.side + side_record(row0 + nA, wave, M.KT, NSB) * SB, swa);
    side_load<KQ>(M.side + side_record(row0 + nB, wave, M.KT, NSB) * SB, swb);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      load_q(wave * 8 + i, qa[i], qb[i]);
      load_x(wave * 8 + i, xr[i]);
    }
  }
  for (int sb = wave; sb < NB; sb += GEMM_WAVES) {
    uint32_t wa[5], wb[5];
#pragma unroll
    for (int i = 0; i < 5; ++i) {
      wa[i] = swa[i];
      wb[i] = swb[i];
    }
    const int nsb = sb + GEMM_WAVES;
    if (nsb < NB) {
      side_load<KQ>(M.side + side_record(row0 + nA, nsb, M.KT, NSB) * SB, swa);
      side_load<KQ>(M.side + side_record(row0 + nB, nsb, M.KT, NSB) * SB, swb);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {  // the super-block's 8 chunks
      if (j < 5 || nsb < NB) {
        const int kn = j < 5 ? sb * 8 + j + 3 : nsb * 8 + j - 5;
        load_q(kn, qa[(j + 3) & 3], qb[(j + 3) & 3]);
        load_x(kn, xr[(j + 3) & 3]);
      }
      __builtin_amdgcn_sched_barrier(0);  // keep the loads issued here, ahead of this chunk's products
      const u32x4 ca = qa[j & 3], cb = qb[j & 3];
      const u32x4* xc = xr[j & 3];
      f16x16 dA = {}, dB = {};
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        if (Q6 && st == 1) {
          dA = f16x16{};
          dB = f16x16{};
        }
        const uint2 a0 = grid16(ca[2 * st]), a1 = grid16(ca[2 * st + 1]);
        const uint2 b0 = grid16(cb[2 * st]), b1 = grid16(cb[2 * st + 1]);
        const h8v wva = __builtin_bit_cast(h8v, make_uint4(a0.x, a0.y, a1.x, a1.y));
        const h8v wvb = __builtin_bit_cast(h8v, make_uint4(b0.x, b0.y, b1.x, b1.y));
        const h8v xh = __builtin_bit_cast(h8v, xc[st]), xl = __builtin_bit_cast(h8v, xc[2 + st]);
        dA = __builtin_amdgcn_mfma_f32_32x32x16_f16(xh, wva, dA, 0, 0, 0);
        dB = __builtin_amdgcn_mfma_f32_32x32x16_f16(xh, wvb, dB, 0, 0, 0);
        dA = __builtin_amdgcn_mfma_f32_32x32x16_f16(xl, wva, dA, 0, 0, 0);
        dB = __builtin_amdgcn_mfma_f32_32x32x16_f16(xl, wvb, dB, 0, 0, 0);
        if (Q6 || st == 1) {  // the sub-block is in: fold it
          const int js = Q6 ? 2 * j + st : j;
          const float sa = sub_scale(wa, js), sbb = sub_scale(wb, js);
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            totA[r] = fmaf(sa, dA[r], totA[r]);
            totB[r] = fmaf(sbb, dB[r], totB[r]);
          }
          // keep the fold here: sunk below the chunk loop's branches it would hold every chunk's tiles live (spills)
          asm volatile("" : "+v"(totA), "+v"(totB));
        }
      }
    }
  }
  __shared__ float part[GEMM_WAVES][2][16][64];
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    part[wave][0][r][lane] = totA[r];
    part[wave][1][r][lane] = totB[r];
  }
  __syncthreads();
  for (int e = threadIdx.x; e < 2 * 16 * 64; e += 64 * GEMM_WAVES) {
    const int half = e >> 10, r = (e >> 6) & 15, l = e & 63;
    float acc = 0.f;
#pragma unroll
    for (int w = 0; w < GEMM_WAVES; ++w) acc += part[w][half][r][l];
    const int t = tt * 32 + 8 * (r / 4) + 4 * (l >> 5) + (r % 4);
    if (t < m) Y[(size_t)t * ldy + row0 + rp * 64 + 32 * half + (l & 31)] = acc;
  }
}

hipError_t launch_gemm_prefill(const DevMat& M, const uint8_t* CT, int row0, int nrows, const void* XT,
                               const void* SXT, int m, float* Y, int ldy, hipStream_t s) {
  if (nrows < 1 || m < 1 || nrows % 64 || M.K % 256) return hipErrorInvalidValue;
  const dim3 grid(nrows / 64, (m + 31) / 32), block(64 * GEMM_WAVES);
  const uint16_t* x = static_cast<const uint16_t*>(XT);
  const uint16_t* sx = static_cast<const uint16_t*>(SXT);
  switch (M.kqt) {
    case KQ_Q4_K: hipLaunchKernelGGL(k_gemm_prefill<KQ_Q4_K>, grid, block, 0, s, M, CT, row0, x, sx, m, Y, ldy); break;
    case KQ_Q5_K: hipLaunchKernelGGL(k_gemm_prefill<KQ_Q5_K>, grid, block, 0, s, M, CT, row0, x, sx, m, Y, ldy); break;
    case KQ_Q6_K: hipLaunchKernelGGL(k_gemm_prefill_sub<KQ_Q6_K>, grid, block, 0, s, M, CT, row0, x, m, Y, ldy); break;
    case KQ_IQ4_XS: hipLaunchKernelGGL(k_gemm_prefill_sub<KQ_IQ4_XS>, grid, block, 0, s, M, CT, row0, x, m, Y, ldy); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace lw
