// Device helpers shared by the MFMA product kernels (gemm.hip, gemm_few.hip, gemm_ring.hip, gemm_q8.hip).
#pragma once

#include "gemm.h"

#pragma clang fp contract(off)

namespace frhip {

typedef float f16v __attribute__((ext_vector_type(16)));
typedef float f4v __attribute__((ext_vector_type(4)));
// 16 bytes at any address of an element: the same one instruction (device memory is accessed in unaligned mode)
typedef h1 h8_any __attribute__((ext_vector_type(8), aligned(2)));
typedef float f4v_any __attribute__((ext_vector_type(4), aligned(4)));

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
// as used: no kernel issues the builtin's loads besides, so the compiler keeps no value in M0 across this statement.
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
// Behind it the loading waves write over what the MFMA waves read ahead of it, so those reads have to be complete here.  The compiler waits for
// them ahead of the MFMAs that take them, in the same loop body, so ahead of the barrier; that this is what it built
// is checked in the library's code (test_kernel_isa.py).  lgkmcnt(0) ahead of the barrier besides made uint8 products up to 2.4 %
// slower (93 of more than 25 us: 0.3 %).
__device__ __forceinline__ void step_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Between lanes of one wave that pass values through LDS: LDS serves a wave's accesses in their order, this keeps the compiler to it.
__device__ __forceinline__ void lanes_in_order() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_wave_barrier();
  asm volatile("" ::: "memory");
}

// 4 bytes per lane, each lane from its own address (see load_lds_saddr for M0 and the wait counts)
__device__ __forceinline__ void load_lds_dword(const void* p, unsigned lds) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off" ::"v"(p), "s"(lds) : "memory");
}

// c * ry and mx + my, each rounded once to fp32, with the binary16 operand taken from its half of a register
template <int HI>
__device__ __forceinline__ float mul_h(float c, h2 v) {
  float r;
  if constexpr (HI) asm("v_fma_mix_f32 %0, %1, %2, -%3 op_sel:[0,1,0] op_sel_hi:[0,1,0]" : "=v"(r) : "v"(c), "v"(v), "s"(0.0f));
  else asm("v_fma_mix_f32 %0, %1, %2, -%3 op_sel_hi:[0,1,0]" : "=v"(r) : "v"(c), "v"(v), "s"(0.0f));
  return r;
}
template <int HI>
__device__ __forceinline__ float add_h(float m, h2 v) {
  float r;
  if constexpr (HI) asm("v_fma_mix_f32 %0, 1.0, %2, %1 op_sel:[0,1,0] op_sel_hi:[0,1,0]" : "=v"(r) : "v"(m), "v"(v));
  else asm("v_fma_mix_f32 %0, 1.0, %2, %1 op_sel_hi:[0,1,0]" : "=v"(r) : "v"(m), "v"(v));
  return r;
}

// dequant_pair's two values, the same bits, in 9 instead of up to 13 instructions: no conversion of ry and my
template <int HI>
__device__ __forceinline__ h2 few_dequant(uint32_t word, float c, float mx, h2 ry, h2 my) {
  float w0 = __builtin_fmaf((float)((word >> (HI ? 16 : 0)) & 0xffu), mul_h<0>(c, ry), add_h<0>(mx, my));
  float w1 = __builtin_fmaf((float)((word >> (HI ? 24 : 8)) & 0xffu), mul_h<1>(c, ry), add_h<1>(mx, my));
  asm("" : "+v"(w0), "+v"(w1));  // rounded to fp32 before the conversion (not v_fma_mixlo_f16, which rounds once)
  return (h2){(h1)w0, (h1)w1};
}

template <int N>
__device__ __forceinline__ void wait_loads() {  // at most N of this wave's loads outstanding
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// An operand's K-step of 64 in LDS: 8 rows x 128 bytes are 1 KB, k-segment q of row r in slot q ^ (r % 8) ^ (r / 8 % 2)
// (gemm.hip, "LDS layout").
constexpr int kLdwBK = 64;
__device__ __forceinline__ int ldw_at(int row, int q) {
  return (row >> 3) * 1024 + (row & 7) * 128 + ((q ^ (row & 7) ^ ((row >> 3) & 1)) * 16);
}

// Workgroups are dealt to the eight XCDs in turn (linear index mod 8), each with an L2 of its own.  XCD x takes the
// x-th eighth of the tiles, counted in blocks of four strips of rows by all N tiles, so that the 32 it runs at a time
// share about four strips and eight N tiles.  Blocks of four N tiles by all strips, the other way round, gave the
// tiles of a segment with a costly epilogue to one or two XCDs: the 4099-token prompt of a 1.5B model took 19.2 ms
// so, 18.3 this way (same box, in turn; up to four strips the two are the same map).  (A matter of traffic and balance
// only: the map is one to one, and any assignment of tiles to workgroups gives the same results.)
__device__ __forceinline__ void xcd_tile(int& bx, int& by) {
  const int gx = gridDim.x, gy = gridDim.y, lin = blockIdx.y * gx + blockIdx.x, n = gx * gy;
  const int x = lin & 7, id = x * (n >> 3) + min(x, n & 7) + (lin >> 3);
  const int blk = id / (4 * gx), rem = id - blk * 4 * gx, bw = min(4, gy - 4 * blk);
  bx = rem / bw;
  by = 4 * blk + rem % bw;
}

// Fused epilogues, shared by the product kernels: acc[i][j] is the 32x32 block (i, j) of the wave's
// (32 MI) x (32 NJ) tile whose first element is (row0, col0); acc[i][j][v] is
// C[row = 8*(v/4) + 4*(lane/32) + v%4][col = lane%32] of the block.
// FULL: the workgroup's tile lies inside the matrix, nothing is predicated.  (With a predicate per
// element every store becomes a branch to an out-of-line block; on the 1024 x 6144 product that
// was 11 of 59 us.)  The epilogue kind is uniform over the launch segment: one switch, and for the
// kinds that read operands all 16 of a block are requested before the first is used.
template <int MI, int NJ, bool FULL>
__device__ __forceinline__ void gemm_epilogue_t(const GemmArgs& a, const GemmSeg& sg, const f16v (&acc)[MI][NJ],
                                                int row0, int col0, int M, int N, int lane) {
  auto for_tile = [&](int i, int j, auto&& f) {
    const int col = col0 + j * 32 + (lane & 31);
#pragma unroll
    for (int v = 0; v < 16; v++) {
      const int row = row0 + i * 32 + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
      if constexpr (FULL)
        f(v, true, (size_t)row * N + col);
      else
        f(v, row < M && col < N, (size_t)(row < M ? row : M - 1) * N + (col < N ? col : N - 1));
    }
  };
  auto for_blocks = [&](auto&& g) {
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
      for (int j = 0; j < NJ; j++) g(i, j, acc[i][j]);
  };
  // blocks without a stored element; only for the costly epilogues: with the test in all of them the short launches of
  // 64-row tiles took 0.4-0.8 us longer (33 x 1024 x 5120: 6.5 -> 6.9)
  auto outside = [&](int i, int j) { return !FULL && (row0 + i * 32 >= M || col0 + j * 32 >= N); };
  auto live_of = [&](int i, int j) {  // bit v: element v of the block lies inside the matrix
    uint32_t m = 0;
    for_tile(i, j, [&](int v, bool ok, size_t) { m |= ok ? 1u << v : 0u; });
    return m;
  };
  switch (sg.epi) {
    case G_STORE_F16:
      for_blocks([&](int i, int j, const f16v& c) {
        for_tile(i, j, [&](int v, bool ok, size_t o) { if (ok) static_cast<h1*>(sg.out)[o] = (h1)c[v]; });
      });
      break;
    case G_STORE_F32:
      for_blocks([&](int i, int j, const f16v& c) {
        for_tile(i, j, [&](int v, bool ok, size_t o) { if (ok) static_cast<float*>(sg.out)[o] = c[v]; });
      });
      break;
    case G_SIGMOID:
      for_blocks([&](int i, int j, const f16v& c) {
        if (outside(i, j)) return;
        h1 y[16];
        sigmoid_batch(c, y, live_of(i, j));
        for_tile(i, j, [&](int v, bool ok, size_t o) { if (ok) static_cast<h1*>(sg.out)[o] = y[v]; });
      });
      break;
    case G_RELU2:
      for_blocks([&](int i, int j, const f16v& c) {
        for_tile(i, j, [&](int v, bool ok, size_t o) {
          const h1 t = (h1)c[v];
          if (ok) static_cast<h1*>(sg.out)[o] = (t > (h1)0.0f) ? (t * t) : (h1)0.0f;
        });
      });
      break;
    case G_SILU:
      for_blocks([&](int i, int j, const f16v& c) {
        if (outside(i, j)) return;
        h1 y[16];
        silu_batch(c, y, live_of(i, j));
        for_tile(i, j, [&](int v, bool ok, size_t o) { if (ok) static_cast<h1*>(sg.out)[o] = y[v]; });
      });
      break;
    case G_RESIDUAL:
      for_blocks([&](int i, int j, const f16v& c) {
        h1 rx[16];
        for_tile(i, j, [&](int v, bool, size_t o) { rx[v] = a.res_x[o]; });
        for_tile(i, j, [&](int v, bool ok, size_t o) { if (ok) static_cast<h1*>(sg.out)[o] = rx[v] + (h1)c[v]; });
      });
      break;
    case G_FFN_OUT:
      for_blocks([&](int i, int j, const f16v& c) {
        h1 rx[16], rr[16];
        for_tile(i, j, [&](int v, bool, size_t o) {
          rx[v] = a.res_x[o];
          rr[v] = a.res_r[o];
        });
        for_tile(i, j, [&](int v, bool ok, size_t o) {
          h1 r = __builtin_fmaf16((h1)c[v], rr[v], rx[v]);
          if (a.div2) r = r / (h1)2.0f;
          if (ok) static_cast<h1*>(sg.out)[o] = r;
        });
      });
      break;
    default: break;
  }
}

// The epilogue of G groups of eight consecutive outputs of a row, whose sums are in `acc`; o: the groups' places in [M][N].  VEC:
// operands and outputs go 16 bytes at a time, at any address; otherwise one at a time, the first n of every group.
template <int G, bool VEC = true>
__device__ __forceinline__ void store_groups(const GemmArgs& a, const GemmSeg& sg, const float (&acc)[8 * G], const size_t (&o)[G], int n = 8) {
  constexpr int W = 8 * G;
  if (sg.epi == G_STORE_F32) {
#pragma unroll
    for (int g = 0; g < G; g++) {
      float* out = static_cast<float*>(sg.out) + o[g];
      if constexpr (VEC) {
#pragma unroll
        for (int q = 8 * g; q < 8 * g + 8; q += 4) *reinterpret_cast<f4v_any*>(out + q - 8 * g) = (f4v){acc[q], acc[q + 1], acc[q + 2], acc[q + 3]};
      } else {
#pragma unroll
        for (int i = 0; i < 8; i++)
          if (i < n) out[i] = acc[8 * g + i];
      }
    }
    return;
  }
  auto operand = [&](const h1* p, h1 (&v)[W]) {
#pragma unroll
    for (int g = 0; g < G; g++) {
      if constexpr (VEC) {
        const h8_any t = *reinterpret_cast<const h8_any*>(p + o[g]);
#pragma unroll
        for (int i = 0; i < 8; i++) v[8 * g + i] = t[i];
      } else {
#pragma unroll
        for (int i = 0; i < 8; i++) v[8 * g + i] = i < n ? p[o[g] + i] : (h1)0.0f;
      }
    }
  };
  static_assert(VEC || G == 1, "one bound for one group");
  const uint32_t live = VEC ? (1u << W) - 1 : (1u << n) - 1;
  h1 y[W], x[W], r[W];
  switch (sg.epi) {
    case G_STORE_F16:
#pragma unroll
      for (int i = 0; i < W; i++) y[i] = (h1)acc[i];
      break;
    case G_SIGMOID: sigmoid_batch(acc, y, live); break;
    case G_SILU: silu_batch(acc, y, live); break;
    case G_RELU2:
#pragma unroll
      for (int i = 0; i < W; i++) {
        const h1 t = (h1)acc[i];
        y[i] = (t > (h1)0.0f) ? (t * t) : (h1)0.0f;
      }
      break;
    case G_RESIDUAL:
      operand(a.res_x, x);
#pragma unroll
      for (int i = 0; i < W; i++) y[i] = x[i] + (h1)acc[i];
      break;
    default:  // G_FFN_OUT
      operand(a.res_x, x);
      operand(a.res_r, r);
#pragma unroll
      for (int i = 0; i < W; i++) {
        y[i] = __builtin_fmaf16((h1)acc[i], r[i], x[i]);
        if (a.div2) y[i] = y[i] / (h1)2.0f;
      }
      break;
  }
#pragma unroll
  for (int g = 0; g < G; g++) {
    h1* out = static_cast<h1*>(sg.out) + o[g];
    if constexpr (VEC) {
      h8_any v;
#pragma unroll
      for (int i = 0; i < 8; i++) v[i] = y[8 * g + i];
      *reinterpret_cast<h8_any*>(out) = v;
    } else {
#pragma unroll
      for (int i = 0; i < 8; i++)
        if (i < n) out[i] = y[8 * g + i];
    }
  }
}

// The end of a tile through LDS (where the operands were): an output row goes out 16 bytes a lane instead of one element a lane and
// instruction, and a lane holds eight or sixteen sums at a time instead of its whole part of the tile.
// Rows of sums are `pitch` floats apart: 32 columns a block and 4 more.
__host__ __device__ constexpr int sums_pitch(int blocks) { return 32 * blocks + 4; }

// One row of 32 x 32 blocks of a wave's sums: acc[j][v] is C[row = 8 * (v / 4) + 4 * (lane / 32) + v % 4][col = lane % 32] of block j.
template <int NJ>
__device__ __forceinline__ void sums_to_lds(const f16v (&acc)[NJ], float* sums, int pitch, int lane) {
  float* const p = sums + 4 * (lane >> 5) * pitch + (lane & 31);
#pragma unroll
  for (int j = 0; j < NJ; j++)
#pragma unroll
    for (int v = 0; v < 16; v++) p[(8 * (v >> 2) + (v & 3)) * pitch + j * 32] = acc[j][v];
}

__device__ __forceinline__ void read_sums(float (&s)[8], const float* sums) {
#pragma unroll
  for (int h = 0; h < 2; h++) {
    const f4v v = *reinterpret_cast<const f4v*>(sums + 4 * h);
#pragma unroll
    for (int t = 0; t < 4; t++) s[4 * h + t] = v[t];
  }
}

// Eight sums of row `row` from column `col`; nothing if they are not all inside the matrix (finish_ends)
__device__ __forceinline__ void finish_group(const GemmArgs& a, const GemmSeg& sg, const float* sums, int row, int col, int M, int N) {
  if (row >= M || col + 8 > N) return;
  float s[8];
  read_sums(s, sums);
  const size_t o[1] = {(size_t)row * N + col};
  store_groups<1>(a, sg, s, o);
}

// The last outputs of rows that are no whole groups of eight, a row a thread, after those: as a branch of finish_group every pass over the
// rows went through it.  Whole groups go out 16 bytes a lane at whatever address such rows begin; with one output a lane and instruction,
// 16 bytes apart from lane to lane, 384 x 768 x 50277 took 74.5 us, so 52.3, 200 rows 44.3 and 31.1, 1024 x 2048 x 16377 81.2 and 71.7.
__device__ __forceinline__ void finish_ends(const GemmArgs& a, const GemmSeg& sg, const float* sums, int pitch, int rows, int cols,
                                            int row0, int col0, int M, int N, int t) {
  const int col = (N - col0) & ~7;
  if (col0 >= N || col0 + cols <= N || col0 + col == N || t >= rows || row0 + t >= M) return;
  float s[8];
  read_sums(s, sums + t * pitch + col);
  const size_t o[1] = {(size_t)(row0 + t) * N + col0 + col};
  store_groups<1, false>(a, sg, s, o, N - col0 - col);
}

// A wave's part of a tile, from row row0 and column col0, through a place in LDS of its own, 32 rows at a time: no barriers, and
// only the rows that follow stay in registers.  For tiles over the edge of the matrix, where a predicate per element makes every
// store of gemm_epilogue_t a branch: 300 x 2560 x (2560 + 8960) 49.3 -> 43.7 us, 1000 x 2048 x (3 x 2048) 46.7 -> 42.5, 1000 x 768 x
// (3 x 768) 20.1 -> 16.8.  Whole tiles store straight from the accumulators: 4099 x 2048 x (3 x 2048) 129 us, 136 through LDS.
constexpr int wave_sums_bytes(int blocks) { return 32 * sums_pitch(blocks) * 4; }
template <int MI, int NJ>
__device__ __forceinline__ void finish_wave(const GemmArgs& a, const GemmSeg& sg, const f16v (&acc)[MI][NJ], float* sums, int row0,
                                            int col0, int M, int N, int lane) {
  const bool full = row0 + MI * 32 <= M && col0 + NJ * 32 <= N;
#pragma unroll
  for (int i = 0; i < MI; i++) {
    if (i > 0) lanes_in_order();  // the rows before have been read
    sums_to_lds(acc[i], sums, sums_pitch(NJ), lane);
    lanes_in_order();
    if (full) {
#pragma unroll 1
      for (int t = lane; t < 32 * NJ * 4; t += 128) {
        float s[16];
        size_t o[2];
#pragma unroll
        for (int g = 0; g < 2; g++) {
          const int row = (t + 64 * g) / (NJ * 4), col = (t + 64 * g - row * (NJ * 4)) * 8;
          read_sums(*reinterpret_cast<float(*)[8]>(s + 8 * g), sums + row * sums_pitch(NJ) + col);
          o[g] = (size_t)(row0 + i * 32 + row) * N + col0 + col;
        }
        store_groups<2>(a, sg, s, o);
      }
      continue;
    }
#pragma unroll 1
    for (int t = lane; t < 32 * NJ * 4; t += 64) {
      const int row = t / (NJ * 4), col = (t - row * (NJ * 4)) * 8;
      finish_group(a, sg, sums + row * sums_pitch(NJ) + col, row0 + i * 32 + row, col0 + col, M, N);
    }
    finish_ends(a, sg, sums, sums_pitch(NJ), 32, NJ * 32, row0 + i * 32, col0, M, N, lane);
  }
}

// A tile of ROWS rows and `blocks` blocks of 32 columns, shared by all waves of the workgroup
template <int ROWS, int THREADS>
__device__ __forceinline__ void finish_tile(const GemmArgs& a, const GemmSeg& sg, const float* sums, int pitch, int blocks, int m0,
                                            int n0, int M, int N) {
  const int groups = blocks * 4;  // of 8 outputs
  for (int i = threadIdx.x; i < ROWS * groups; i += THREADS) {
    const int row = i / groups, col = (i - row * groups) * 8;
    finish_group(a, sg, sums + row * pitch + col, m0 + row, n0 + col, M, N);
  }
  static_assert(ROWS <= THREADS, "finish_ends");
  finish_ends(a, sg, sums, pitch, ROWS, blocks * 32, m0, n0, M, N, threadIdx.x);
}

}  // namespace frhip
