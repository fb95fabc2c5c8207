// Device helpers shared by the MFMA product kernels (gemm.hip, gemm_few.hip).
#pragma once

#include "gemm.h"

#pragma clang fp contract(off)

namespace frhip {

typedef float f16v __attribute__((ext_vector_type(16)));
typedef float f4v __attribute__((ext_vector_type(4)));

// sigmoid_h of the W accumulators a lane holds of one MFMA block (16 of 32 x 32, 4 of 16 x 16), the same bits at a
// fraction of the cost.  Called element by element, sigmoid_h makes a wave take its double branch whenever
// any of its 64 lanes needs it (every other element), and its fp32 estimate alone (expf and a
// correctly rounded division, ~35 VALU instructions) is 128 x 35 instructions per lane and tile:
// the sigmoid epilogue of a 128 x 224 tile took 26 us where a plain store takes 2.5 us.
// Here the estimate is v_exp_f32 and v_rcp_f32.  Its error: t = -x log2(e) is one rounded product,
// |dt| <= 9e-8 |t|, so exp2(t) is off by at most 6.2e-8 |t| relative, which reaches the result
// scaled by e/(1+e); over the range that is not handed to the exact path anyway (x > -9.3) that
// is below 1e-6, plus one ulp each for v_exp_f32, the sum and v_rcp_f32: under 20 fp32 ulps.  An
// estimate further than 64 ulps from the midpoint of two binary16 values therefore rounds as the
// exact value does; the others (about 1 in 60) are queued per lane and evaluated in double
// afterwards, one per lane and pass.  `live`: the elements that are stored.  Rows past the matrix hold copies of its
// last row, so one pending element would be sixteen: 777 x 2048 x (2048 sigmoid + 8192), whose last strip of 256 rows has
// nine, took 89 us with all of them queued and takes 57.5 (1024 rows: 59).
template <int W, class V>
__device__ __forceinline__ void sigmoid_batch(const V& c, h1 (&y)[W], uint32_t live) {
  h1 x[W];
  uint32_t pend = 0;
#pragma unroll
  for (int v = 0; v < W; v++) {
    x[v] = (h1)c[v];
    const float e = __builtin_amdgcn_exp2f((float)x[v] * -1.44269504088896340736f);
    const float s32 = __builtin_amdgcn_rcpf(1.0f + e);
    const uint32_t frac = __float_as_uint(s32) & 0x1FFFu;  // the 13 fp32 mantissa bits binary16 drops
    const bool safe = s32 > 1e-4f && (frac - (0x1000u - 64u)) > 128u;
    y[v] = (h1)s32;
    pend |= safe ? 0u : (1u << v);
  }
  pend &= live;
  while (pend) {
    const int v = __builtin_ctz(pend);
    pend &= pend - 1;
    h1 xv = x[0];
#pragma unroll
    for (int u = 1; u < W; u++) xv = (v == u) ? x[u] : xv;
    const h1 r = sigmoid_h_exact(xv);
#pragma unroll
    for (int u = 0; u < W; u++) y[u] = (v == u) ? r : y[u];
  }
}

// silu_h of a block's accumulators, the same bits, built like sigmoid_batch.  silu_h rounds
// e^-x to binary16, adds 1 in binary16 and divides x by the sum in fp32.  The estimates (v_exp_f32
// for the exponential, v_rcp_f32 for the quotient: under 20 and 3 fp32 ulps off) are taken when
// they are further than 64 ulps from a binary16 rounding boundary and in the normal binary16
// range; the other elements are queued and go through silu_h itself.
template <int W, class V>
__device__ __forceinline__ void silu_batch(const V& c, h1 (&y)[W], uint32_t live) {
  h1 x[W];
  uint32_t pend = 0;
  auto far_from_boundary = [](float v) {
    const uint32_t frac = __float_as_uint(v) & 0x1FFFu;
    const float m = __builtin_fabsf(v);
    return m > 1e-4f && m < 60000.f && (frac - (0x1000u - 64u)) > 128u;
  };
#pragma unroll
  for (int v = 0; v < W; v++) {
    x[v] = (h1)c[v];
    const float xf = (float)x[v];
    const float ef = __builtin_amdgcn_exp2f(xf * -1.44269504088896340736f);
    const h1 d = (h1)1.0f + (h1)ef;
    const float qf = xf * __builtin_amdgcn_rcpf((float)d);
    const bool safe = far_from_boundary(ef) && far_from_boundary(qf);
    y[v] = (h1)qf;
    pend |= safe ? 0u : (1u << v);
  }
  pend &= live;
  while (pend) {
    const int v = __builtin_ctz(pend);
    pend &= pend - 1;
    h1 xv = x[0];
#pragma unroll
    for (int u = 1; u < W; u++) xv = (v == u) ? x[u] : xv;
    const h1 r = silu_h(xv);
#pragma unroll
    for (int u = 0; u < W; u++) y[u] = (v == u) ? r : y[u];
  }
}

// global_load_lds_dwordx4 with the address as a scalar base plus a 32-bit lane offset.  The builtin
// takes a 64-bit address per lane, which costs the loader one vector add per load; on the SIMD it
// shares with an MFMA wave each of those waits for a gap between that wave's MFMAs, and the whole
// workgroup waits for the loader at the step's barrier (per K-step of a 128 x 256 tile: loader 2150
// cycles from barrier to barrier, MFMA waves 1550-1700 plus 540-700 waiting).  In this form a load
// needs scalar instructions only.  `lds` is the destination's LDS byte address (lane l writes 16 bytes
// at lds + 16 l); the wait counts are the caller's business, as with the builtin.
// M0 is written here without the compiler knowing (it refuses m0 in a clobber list: a reserved register).  That is safe
// as used: a workgroup issues either these loads or the builtin's (a tile lies wholly inside the matrices or it does not),
// never both, so no value the compiler keeps in M0 for the builtin is ever live across this statement.
__device__ __forceinline__ void load_lds_saddr(unsigned voff, const void* sbase, unsigned lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(sbase), "s"(lds) : "memory");
}

// The same address for every lane, in scalar registers (the compiler cannot always prove it).
__device__ __forceinline__ const unsigned char* uniform_ptr(const void* p) {
  const unsigned long long v = reinterpret_cast<unsigned long long>(p);
  const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)v), hi = __builtin_amdgcn_readfirstlane((unsigned)(v >> 32));
  return reinterpret_cast<const unsigned char*>(((unsigned long long)hi << 32) | lo);
}

// The barrier between K-steps whose waits the kernel places itself.  The builtin is no memory fence for the compiler:
// without the empty statements it could move a fragment read across (nothing else stands between the barrier and the
// reads in a step that issues no loads).  No instruction of its own.
__device__ __forceinline__ void step_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

}  // namespace frhip
