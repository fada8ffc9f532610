// Device helpers shared by the kernel sources.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "lw_format.h"
#include "lw_kernels.h"

namespace lw {

typedef _Float16 h2v __attribute__((ext_vector_type(2)));

// leading zero bits of every device lane stream (lw_layout.h GUARD)
constexpr int GUARD_BITS = 2;
constexpr int kBufferRsrcWord3 = 0x00020000;  // buffer descriptor word 3 for raw dword loads on CDNA (32-bit data format)

typedef _Float16 h4v __attribute__((ext_vector_type(4)));
typedef float f4v __attribute__((ext_vector_type(4)));
typedef int v4i32 __attribute__((ext_vector_type(4)));
typedef float f16x16 __attribute__((ext_vector_type(16)));

typedef _Float16 h8v __attribute__((ext_vector_type(8)));
typedef __bf16 b8v __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float h2f(uint32_t bits16) {
  return (float)__builtin_bit_cast(_Float16, (uint16_t)(bits16 & 0xFFFFu));
}
__device__ __forceinline__ uint32_t f2h(float v) { return (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)v); }

// side bytes of one super-block as words (byte i at bits 8 (i & 3) of w[i / 4]); Q6_K records are 2-byte aligned
template <int KQ>
__device__ __forceinline__ void side_load(const uint8_t* p, uint32_t* w) {
  if (KQ == KQ_Q6_K) {
    const uint16_t* h = reinterpret_cast<const uint16_t*>(p);
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] = (uint32_t)h[2 * i] | (uint32_t)h[2 * i + 1] << 16;
    w[4] = h[8];
  } else if (KQ == KQ_IQ4_XS) {
    const uint2 v = *reinterpret_cast<const uint2*>(p);
    w[0] = v.x;
    w[1] = v.y;
  } else {
    const uint4 v = *reinterpret_cast<const uint4*>(p);
    w[0] = v.x;
    w[1] = v.y;
    w[2] = v.z;
    w[3] = v.w;
  }
}
__device__ __forceinline__ uint32_t side_byte(const uint32_t* w, int i) { return (w[i >> 2] >> (8 * (i & 3))) & 255u; }

// Sub-block scales of one super-block packed as bytes, consumed low byte first (reference llmrt.cu:125-149; Q4_K /
// Q5_K fields per llama.cpp get_scale_min_k4, four at a time): s_j = dA * byte_j (Q6_K: signed bytes, 16 of them in
// scq then scq2; IQ4_XS: ls_j - 32, also signed), o_j = dB * m_j (side_mins).
template <int KQ>
__device__ __forceinline__ void side_packed(const uint32_t* w, uint64_t& scq, uint64_t& scq2, float& dA, float& dB) {
  if (KQ == KQ_Q4_K || KQ == KQ_Q5_K) {
    const uint32_t sc_lo = w[1] & 0x3F3F3F3Fu;
    const uint32_t sc_hi = (w[3] & 0x0F0F0F0Fu) | ((w[1] >> 2) & 0x30303030u);
    scq = (uint64_t)sc_lo | (uint64_t)sc_hi << 32;
    scq2 = 0;
    dA = h2f(w[0]);
    dB = h2f(w[0] >> 16);
  } else if (KQ == KQ_Q6_K) {
    scq = (uint64_t)w[0] | (uint64_t)w[1] << 32;
    scq2 = (uint64_t)w[2] | (uint64_t)w[3] << 32;
    dA = h2f(w[4]);
    dB = 0.f;
  } else {
    const uint32_t hi = w[0] >> 16, lo = w[1];
    uint64_t q = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint32_t ls = ((lo >> (4 * i)) & 15u) | (((hi >> (2 * i)) & 3u) << 4);
      q |= (uint64_t)((ls - 32u) & 255u) << (8 * i);
    }
    scq = q;
    scq2 = 0;
    dA = h2f(w[0]);
    dB = 0.f;
  }
}
// Q4_K / Q5_K sub-block mins as floats
__device__ __forceinline__ void side_mins(const uint32_t* w, float* mf) {
  const uint32_t m_lo = w[2] & 0x3F3F3F3Fu;
  const uint32_t m_hi = ((w[3] >> 4) & 0x0F0F0F0Fu) | ((w[2] >> 2) & 0x30303030u);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    mf[i] = (float)((m_lo >> (8 * i)) & 255u);
    mf[4 + i] = (float)((m_hi >> (8 * i)) & 255u);
  }
}

// LDS address of the table entry indexed by window bits 2..12 of w: (w & 0x1FFC) | table base, one instruction (the
// base is a multiple of 8 KB and wave-uniform)
__device__ __forceinline__ uint32_t table_addr(uint32_t w, uint32_t base, uint32_t mask) {
  uint32_t a;  // VOP3 takes no literal here: the mask 0x1FFC lives in a register
  asm("v_and_or_b32 %0, %1, %3, %2" : "=v"(a) : "v"(w), "s"(base), "v"(mask));
  return a;
}

// compile-time loop: f(std::integral_constant<int, i>) for i = 0 .. N - 1 (indices that must be constants: MFMA
// broadcast fields, register-array indices; bodies past the loop unroller's size limit)
template <int I, int N, class F>
__device__ __forceinline__ void static_for_from(F& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for_from<I + 1, N>(f);
  }
}
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_from<0, N>(f);
}

// s_waitcnt vmcnt(n) for a wave-uniform n in [0, 63] (the count is an immediate: one wait per value; larger n wait
// for 63). The compiler does not see which value ran, so it still waits for every vector load whose result a later
// instruction reads; this is for loads whose results only LDS reads see (direct-to-LDS copies).
template <int N = 63>
__device__ __forceinline__ void wait_vmcnt_upto(int n) {
  if constexpr (N == 0) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  } else {
    if (n >= N) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
    else wait_vmcnt_upto<N - 1>(n);
  }
}

// The sum over columns c < KT, in order, of the partial slots q + c cs. Each slot is taken by an exchange with
// kNoPartial, 32 in flight. A slot still holding kNoPartial (its partial counted but not yet visible here) makes the
// running sum NaN, so one test per batch finds it; the batch is then summed again once every such slot has its
// partial (at most kPartialSpins re-reads each, a few hundred cycles apiece; past that the sum is NaN rather than a
// hang). A NaN of the data itself only costs the re-summation: no arithmetic result has kNoPartial's bits.
__device__ __forceinline__ float sum_partials(uint32_t* q, size_t cs, int KT) {
  constexpr int B = 32;
  auto take = [&](int c) {
    return __hip_atomic_exchange(q + (size_t)c * cs, kNoPartial, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  float a = 0.f;
  for (int c0 = 0; c0 < KT; c0 += B) {
    uint32_t v[B];
#pragma unroll
    for (int u = 0; u < B; ++u) v[u] = c0 + u < KT ? take(c0 + u) : 0u;
    const float a0 = a;
#pragma unroll
    for (int u = 0; u < B; ++u)
      if (c0 + u < KT) a += __builtin_bit_cast(float, v[u]);
    if (__builtin_expect(a != a, 0)) {
      a = a0;
      for (int u = 0; u < B && c0 + u < KT; ++u) {
        uint32_t w = v[u];
        for (int i = 0; w == kNoPartial && i < kPartialSpins; ++i) {
          __builtin_amdgcn_s_sleep(2);
          w = take(c0 + u);
        }
        a += w == kNoPartial ? __builtin_nanf("") : __builtin_bit_cast(float, w);
      }
    }
  }
  return a;
}

}  // namespace lw
