// Seq-mode (prefill) matrix products on the MFMA units of gfx950.
//
//   Y[T, N] = X[T, K] . W        with W held output-major, Wt[N][K]
//
// Both operands are K-contiguous, which is the layout v_mfma_f32_32x32x16_f16 wants:
// a lane's A (or B) fragment is 8 consecutive k of one row, i.e. one 16-byte load.
// The kernels:
//   gemm_ring_kernel   (gemm_ring.hip) binary16 weights: four waves multiply a tile of 64 or 128 rows, four load;
//   gemm_vw_kernel, gemm_vw256_kernel  binary16 weights, many rows of wide products: tiles of 256 rows, eight MFMA waves,
//                      with a loader wave, or loading themselves;
//   gemm_q8_kernel     (gemm_q8.hip) uint8 weights, dequantised on their way into LDS by waves of their own;
//   gemm_few_kernel    (gemm_few.hip) a few rows: K split over the waves of a workgroup;
//   gemm_kernel        tiles go global -> registers -> LDS (rows padded by 16 bytes against bank conflicts), the loads of step
//                      k+1 issued before the MFMAs of step k, uint8 ones dequantised on the way: what none of the others takes
//                      (uint8 products of fewer than four rows or of columns that are no multiple of 16, without scratch to
//                      expand them; rows of more than 8 million elements).
// Products are exact in fp32, accumulation is fp32 in ascending k, and the result is rounded once
// to the output type (kernels/cuda/matmul.cpp:38-42,64-68); all kernels but gemm_few_kernel give the same bits, except
// that a launch split over K (launch_gemm) adds its slices' fp32 sums at the end.
// Independent products over the same T and K share one launch ("segments"), each with
// its own X, W and fused epilogue.
#include <climits>
#include <cstring>

#include "gemm_device.h"

#pragma clang fp contract(off)

namespace frhip {

constexpr int BN = 128;
constexpr int kGemmThreads = 256;
template <int BM>
__device__ __forceinline__ void gemm_epilogue(const GemmArgs& a, const GemmSeg& sg, const f16v (&acc)[BM / 64][2], int m0,
                                              int n0, int M, int N, int lane, int wm, int wn) {
  if (m0 + BM <= M && n0 + BN <= N)
    gemm_epilogue_t<BM / 64, 2, true>(a, sg, acc, m0 + wm * (BM / 2), n0 + wn * 64, M, N, lane);
  else
    gemm_epilogue_t<BM / 64, 2, false>(a, sg, acc, m0 + wm * (BM / 2), n0 + wn * 64, M, N, lane);
}

// BM = 128 (waves 2 x 2 of 64 x 64) or 64 (waves of 32 x 64), for launches that would otherwise
// leave compute units idle.  BK = 64, or 128 for launches with about one workgroup per CU: with a
// single wave per SIMD nothing hides the round trip of the next tile's loads, so a K step lasts
// about one memory latency whatever its depth, and a deeper step halves their number.
template <int BM, int BK, bool U8>
__global__ __launch_bounds__(kGemmThreads) void gemm_kernel(GemmArgs a) {
  constexpr int LDSK = BK + 8;
  constexpr int MI = BM / 64;                      // 32-row MFMA blocks per wave
  constexpr int CPR = BK / 8;                      // 16-byte chunks of 8 halves per tile row
  constexpr int AC = BM * CPR / kGemmThreads;      // chunks of the A tile per thread
  constexpr int BC = BN * CPR / kGemmThreads;      // chunks of a binary16 B tile per thread
  constexpr int QPR = BK / 16;                     // 16-code chunks per tile row (uint8)
  constexpr int QC = BN * QPR / kGemmThreads;      // chunks of a uint8 B tile per thread
  extern __shared__ __attribute__((aligned(16))) unsigned char gemm_smem[];  // gemm_lds_bytes(BM, BK)
  h1* const As = reinterpret_cast<h1*>(gemm_smem);  // [BM][LDSK]
  h1* const Bs = As + BM * LDSK;                    // [BN][LDSK]

  // which segment does this N-tile belong to
  int sidx = 0;
#pragma unroll
  for (int i = 1; i < kGemmMaxSeg; i++) sidx += (i < a.nseg && (int)blockIdx.x >= a.tile_start[i]) ? 1 : 0;
  const GemmSeg& sg = a.seg[sidx];
  const int n0 = ((int)blockIdx.x - a.tile_start[sidx]) * BN;
  const int m0 = blockIdx.y * BM;
  const int M = a.M, K = a.K, N = sg.N;

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;

  // global -> register staging: a tile is 128 rows x 64 k.
  //   A (binary16): 1024 chunks of 8 halves, 4 per thread: chunk c -> row c/8, k (c%8)*8
  //   B binary16: same.  B uint8: 512 chunks of 16 codes, 2 per thread: row c/4, k (c%4)*16
  struct Stage {
    h8 ra[AC];
    h8 rb[U8 ? 1 : BC];
    u32x4 rq[U8 ? QC : 1];
  };
  auto load_tiles = [&](Stage& st, int k0) {
#pragma unroll
    for (int i = 0; i < AC; i++) {
      const int c = tid + i * kGemmThreads;
      int row = m0 + c / CPR;
      row = row < M ? row : M - 1;  // rows past M are computed on a copy of the last row and never stored
      st.ra[i] = *reinterpret_cast<const h8*>(sg.A + (size_t)row * K + k0 + (c % CPR) * 8);
    }
    if constexpr (!U8) {
#pragma unroll
      for (int i = 0; i < BC; i++) {
        const int c = tid + i * kGemmThreads;
        int row = n0 + c / CPR;
        row = row < N ? row : N - 1;
        st.rb[i] = __builtin_nontemporal_load(reinterpret_cast<const h8*>(sg.B + ((size_t)row * K + k0 + (c % CPR) * 8) * 2));
      }
    } else {
#pragma unroll
      for (int i = 0; i < QC; i++) {
        const int c = tid + i * kGemmThreads;
        int row = n0 + c / QPR;
        row = row < N ? row : N - 1;
        st.rq[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(sg.B + (size_t)row * K + k0 + (c % QPR) * 16));
      }
    }
  };
  auto store_tiles = [&](const Stage& st, int k0) {
#pragma unroll
    for (int i = 0; i < AC; i++) {
      const int c = tid + i * kGemmThreads;
      *reinterpret_cast<h8*>(&As[(c / CPR) * LDSK + (c % CPR) * 8]) = st.ra[i];
    }
    if constexpr (!U8) {
#pragma unroll
      for (int i = 0; i < BC; i++) {
        const int c = tid + i * kGemmThreads;
        *reinterpret_cast<h8*>(&Bs[(c / CPR) * LDSK + (c % CPR) * 8]) = st.rb[i];
      }
    } else {
#pragma unroll
      for (int i = 0; i < QC; i++) {
        const int c = tid + i * kGemmThreads;
        int row = n0 + c / QPR;
        row = row < N ? row : N - 1;
        const int kk = k0 + (c % QPR) * 16;
        const float c2 = dequant_c(sg.rx[row]);
        const float m2 = (float)sg.mx[row];
#pragma unroll
        for (int hh = 0; hh < 2; hh++) {
          const h8 ry = *reinterpret_cast<const h8*>(sg.ry + kk + hh * 8);
          const h8 my = *reinterpret_cast<const h8*>(sg.my + kk + hh * 8);
          const uint32_t w0 = st.rq[i][2 * hh], w1 = st.rq[i][2 * hh + 1];
          h2 p0 = dequant_pair<0>(w0, c2, m2, ry.s01, my.s01);
          h2 p1 = dequant_pair<1>(w0, c2, m2, ry.s23, my.s23);
          h2 p2 = dequant_pair<0>(w1, c2, m2, ry.s45, my.s45);
          h2 p3 = dequant_pair<1>(w1, c2, m2, ry.s67, my.s67);
          h8 o = {p0.x, p0.y, p1.x, p1.y, p2.x, p2.y, p3.x, p3.y};
          *reinterpret_cast<h8*>(&Bs[(c / QPR) * LDSK + (c % QPR) * 16 + hh * 8]) = o;
        }
      }
    }
  };

  f16v acc[MI][2];
#pragma unroll
  for (int i = 0; i < MI; i++)
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int v = 0; v < 16; v++) acc[i][j][v] = 0.f;

  // the fragments of FG * 16 k are requested from LDS together; the MFMAs then start as the first
  // ones arrive instead of paying the LDS latency once per 16-deep sub-step
  auto compute_tile = [&]() {
    constexpr int FG = 4;
#pragma unroll
    for (int kh = 0; kh < BK; kh += FG * 16) {
      h8 fa[FG][MI], fb[FG][2];
#pragma unroll
      for (int kq = 0; kq < FG; kq++) {
        const int kofs = kh + kq * 16 + (lane >> 5) * 8;
#pragma unroll
        for (int i = 0; i < MI; i++)
          fa[kq][i] = *reinterpret_cast<const h8*>(&As[(wm * (BM / 2) + i * 32 + (lane & 31)) * LDSK + kofs]);
#pragma unroll
        for (int j = 0; j < 2; j++)
          fb[kq][j] = *reinterpret_cast<const h8*>(&Bs[(wn * 64 + j * 32 + (lane & 31)) * LDSK + kofs]);
      }
#pragma unroll
      for (int kq = 0; kq < FG; kq++)
#pragma unroll
        for (int i = 0; i < MI; i++)
#pragma unroll
          for (int j = 0; j < 2; j++)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[kq][i], fb[kq][j], acc[i][j], 0, 0, 0);
    }
  };

  Stage s0;
  load_tiles(s0, 0);
  for (int k0 = 0; k0 < K; k0 += BK) {
    __syncthreads();  // everyone is done reading the previous tile
    store_tiles(s0, k0);
    __syncthreads();
    if (k0 + BK < K) load_tiles(s0, k0 + BK);
    compute_tile();
  }

  gemm_epilogue<BM>(a, sg, acc, m0, n0, M, N, lane, wm, wn);
}

// ---------------------------------------------------------------------------
// binary16 weights: waves that multiply and waves that only move data.
//
// A compute unit keeps about 64 KB of loads in flight, and a wave that asks for more stands at its
// load instruction with everything behind it, MFMAs included.  In gemm_kernel the waves that
// compute also load, so requests are outstanding only between "issue" and "store to LDS".  In gemm_ring_kernel (gemm_ring.hip)
// and gemm_vw_kernel waves of their own stream tiles global -> LDS directly (global_load_lds_dwordx4, no registers)
// into a ring of K-steps of 64, two or three of which are in flight all the time, and the MFMA waves meet them at one barrier
// per step.  Same products in the same order as gemm_kernel: the results are bit-identical.
//
// LDS layout.  One load instruction brings 8 rows x 64 k = 8 x 128 contiguous bytes (fully
// coalesced) and lands as 1 KB in lane order: lane l = row l/8, 16-byte slot l%8.  The lane asks
// for k-segment (l%8) ^ (row%8) ^ (row/8 % 2), so k-segment q of row r sits in slot
// q ^ (r%8) ^ (r/8 % 2).  A fragment read (32 consecutive rows, one k-segment) is served 16 lanes
// per cycle over 64 banks; rows r and r+8 lie 1 KB apart, i.e. on the same banks, and the last
// term moves them one slot apart: SQ_LDS_BANK_CONFLICT is 0 and a read takes 4 cycles (without
// that term every read was a two-way conflict: 8 cycles).
// ---------------------------------------------------------------------------
// Adds the K slices of a split launch in slice order and applies each product's epilogue; a thread
// takes W consecutive outputs of a row: 16, the unit the batched sigmoid / silu work on, when one of
// the epilogues is one of those, else 8 (N % 16 == 0 either way).
// og: the thread's place within a slice, over all segments; o: within its segment's [M][N]
template <int W>
__device__ __forceinline__ void splitk_reduce_body(const GemmArgs& a, const GemmSeg& sg, size_t og, size_t o) {
  constexpr int Q = W / 4;
  float acc[W];
#pragma unroll
  for (int q = 0; q < Q; q++) {
    const f4v p = *reinterpret_cast<const f4v*>(a.partial + og + 4 * q);
#pragma unroll
    for (int i = 0; i < 4; i++) acc[4 * q + i] = p[i];
  }
  // many slices (a short prompt's launch): four are requested together and then added in slice order
  if (a.ksplit <= 4) {
    for (int z = 1; z < a.ksplit; z++) {
      const float* pz = a.partial + (size_t)z * a.partial_stride + og;
#pragma unroll
      for (int q = 0; q < Q; q++) {
        const f4v p = *reinterpret_cast<const f4v*>(pz + 4 * q);
#pragma unroll
        for (int i = 0; i < 4; i++) acc[4 * q + i] += p[i];
      }
    }
  } else
  for (int z0 = 1; z0 < a.ksplit; z0 += 4) {
    f4v p[4][Q];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      if (z0 + j < a.ksplit) {
        const float* pz = a.partial + (size_t)(z0 + j) * a.partial_stride + og;
#pragma unroll
        for (int q = 0; q < Q; q++) p[j][q] = *reinterpret_cast<const f4v*>(pz + 4 * q);
      }
    }
#pragma unroll
    for (int j = 0; j < 4; j++)
      if (z0 + j < a.ksplit)
#pragma unroll
        for (int q = 0; q < Q; q++)
#pragma unroll
          for (int i = 0; i < 4; i++) acc[4 * q + i] += p[j][q][i];
  }
  size_t at[W / 8];
#pragma unroll
  for (int g = 0; g < W / 8; g++) at[g] = o + 8 * g;
  store_groups<W / 8>(a, sg, acc, at);
}

template <int W>
__global__ __launch_bounds__(256) void gemm_splitk_reduce_kernel(GemmArgs a) {
  const size_t og = ((size_t)blockIdx.x * blockDim.x + threadIdx.x) * W;
  if (a.nseg == 1) {  // the segment's description stays in scalar registers
    if (og < a.part_off[1]) splitk_reduce_body<W>(a, a.seg[0], og, og);
    return;
  }
  if (og >= a.part_off[a.nseg]) return;
  int sidx = 0;
#pragma unroll
  for (int i = 1; i < kGemmMaxSeg; i++) sidx += (i < a.nseg && og >= a.part_off[i]) ? 1 : 0;
  splitk_reduce_body<W>(a, a.seg[sidx], og, og - a.part_off[sidx]);
}

// Small reductions go out in workgroups of one wave, so that they spread over the compute units.
static void launch_splitk_reduce(hipStream_t st, const GemmArgs& a) {
  bool wide = false;
  for (int i = 0; i < a.nseg; i++) wide = wide || a.seg[i].epi == G_SIGMOID || a.seg[i].epi == G_SILU;
  const size_t threads = (a.part_off[a.nseg] + (wide ? 15 : 7)) / (wide ? 16 : 8);
  const unsigned block = threads >= 65536 ? 256 : 64;
  const dim3 grid((unsigned)((threads + block - 1) / block));
  if (wide)
    hipLaunchKernelGGL(gemm_splitk_reduce_kernel<16>, grid, dim3(block), 0, st, a);
  else
    hipLaunchKernelGGL(gemm_splitk_reduce_kernel<8>, grid, dim3(block), 0, st, a);
}

// ---------------------------------------------------------------------------
// binary16 weights, tiles of 256 rows and a width chosen per launch.
//
// A launch of fixed tiles rarely comes out as a whole number of rounds over the compute units, and a
// wider tile moves fewer bytes per product.  Here, and for gemm_ring_kernel's tiles of 64 and 128 rows, the host cuts every segment
// of a launch into tiles of 32 w columns, w = base or base + 1 per segment, so that the launch fills
// a whole number of rounds over the compute units, and no tile straddles two segments.  The two wave columns of a workgroup take
// ceil(w/2) and floor(w/2) 32-column blocks; the loops are instantiated per block count, so the products are the same
// MFMAs in the same k order as in the other kernels and the results are bit-identical.  gemm_vw_kernel has eight MFMA waves
// (4 x 2 of 64 rows each) and a loader wave with a ring of three K-steps, and takes whole tiles of at most 160 columns;
// gemm_vw256_kernel below takes the others.
// ---------------------------------------------------------------------------
constexpr int kVwMaxW = 8, kVwABytes = 256 * kLdwBK * 2;
constexpr int kVwStages = 3, kVw256LoaderMaxW = 5;  // three stages of (256 + 160) x 64 halves are 156 KB of the 160 KB

template <int W>
__device__ __forceinline__ void vw_loader(const GemmSeg& sg, unsigned char* smem, int stage_bytes, int m0, int n0, int K, int lane) {
  constexpr int kAInstr = kVwABytes / 1024, kBInstr = 4 * W, kPer = kAInstr + kBInstr;
  static_assert(kPer <= 63, "the wait counter's range");
  const int lr = lane >> 3, ls = (lane & 7) ^ lr;
  const int nk = K / kLdwBK;
  // the tile lies wholly inside the matrices: rows are 8 K halves apart for every lane, so the address of
  // load b is a uniform base (row group b, this step's k) plus one of two lane offsets
  const unsigned voff[2] = {(unsigned)(lr * K * 2 + ls * 16), (unsigned)(lr * K * 2 + (ls ^ 1) * 16)};
  const unsigned char* abase = uniform_ptr(reinterpret_cast<const unsigned char*>(sg.A) + (size_t)m0 * K * 2);
  const unsigned char* bbase = uniform_ptr(reinterpret_cast<const unsigned char*>(sg.B) + (size_t)n0 * K * 2);
  const unsigned lds0 = (unsigned)(size_t)((__attribute__((address_space(3))) unsigned char*)smem);
  const size_t group = (size_t)__builtin_amdgcn_readfirstlane(K) * 16;  // bytes between row groups of 8
  auto issue = [&](int step, int slot) {
    const unsigned st = lds0 + slot * stage_bytes;
    const unsigned char* ak = abase + (size_t)step * (kLdwBK * 2);
    const unsigned char* bk = bbase + (size_t)step * (kLdwBK * 2);
#pragma unroll
    for (int b = 0; b < kAInstr; b++) load_lds_saddr(voff[b & 1], ak + b * group, st + b * 1024);
#pragma unroll
    for (int b = 0; b < kBInstr; b++) load_lds_saddr(voff[b & 1], bk + b * group, st + kVwABytes + b * 1024);
  };
  issue(0, 0);
  if (nk > 1) issue(1, 1);
  int slot = 2;
  for (int k = 0; k < nk; k++) {
    if (k + 1 < nk)
      __builtin_amdgcn_s_waitcnt(((kPer >> 4) << 14) | 0x0F70 | (kPer & 15));  // vmcnt(kPer): step k has landed
    else
      __builtin_amdgcn_s_waitcnt(0x0F70);
    step_barrier();  // step k may be read; step k-1 has been read by all
    if (k + 2 < nk) {
      issue(k + 2, slot);  // not the slot of step k or k+1
      slot = slot + 1 == kVwStages ? 0 : slot + 1;
    }
  }
}

template <int NJ>
__device__ __forceinline__ void vw_mma(const GemmArgs& a, const GemmSeg& sg, const unsigned char* smem, int stage_bytes, int brow0,
                                       int m0, int n0, int M, int N, int lane, int wave) {
  const int wm = wave >> 1;
  f16v acc[2][NJ];
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < NJ; j++)
#pragma unroll
      for (int v = 0; v < 16; v++) acc[i][j][v] = 0.f;
  const int nk = a.K / kLdwBK;
  int slot = 0;
  for (int k = 0; k < nk; k++) {
    step_barrier();
    const unsigned char* st = smem + slot * stage_bytes;
    slot = slot + 1 == kVwStages ? 0 : slot + 1;
    // fragments of KG x 16 k are requested together; with eight MFMA waves and the loader a lane has 168
    // registers and holds two of the four k-blocks of a step at a time
    constexpr int KG = 2;
#pragma unroll
    for (int kh = 0; kh < 4; kh += KG) {
      h8 fa[KG][2], fb[KG][NJ];
#pragma unroll
      for (int kb = 0; kb < KG; kb++) {
        const int q = (kh + kb) * 2 + (lane >> 5);
#pragma unroll
        for (int i = 0; i < 2; i++) fa[kb][i] = *reinterpret_cast<const h8*>(st + ldw_at(wm * 64 + i * 32 + (lane & 31), q));
#pragma unroll
        for (int j = 0; j < NJ; j++)
          fb[kb][j] = *reinterpret_cast<const h8*>(st + kVwABytes + ldw_at(brow0 + j * 32 + (lane & 31), q));
      }
#pragma unroll
      for (int kb = 0; kb < KG; kb++)
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
          for (int j = 0; j < NJ; j++)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[kb][i], fb[kb][j], acc[i][j], 0, 0, 0);
    }
  }
  gemm_epilogue_t<2, NJ, true>(a, sg, acc, m0 + wm * 64, n0 + brow0, M, N, lane);
}

// Eight MFMA waves of 64 rows x half the width, then the loader: launches of whole tiles of at most kVw256LoaderMaxW blocks,
// of rows of at most 8 million elements (plan_vw).
__global__ __launch_bounds__(576) void gemm_vw_kernel(GemmArgs a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char gemm_smem[];
  int bx, by;
  xcd_tile(bx, by);
  int sidx = 0;
#pragma unroll
  for (int i = 1; i < kGemmMaxSeg; i++) sidx += (i < a.nseg && bx >= a.tile_start[i]) ? 1 : 0;
  const GemmSeg& sg = a.seg[sidx];
  const int ti = bx - a.tile_start[sidx];
  const int base = a.vw_base[sidx], wide = a.vw_wide[sidx];
  const int width = base + (ti < wide ? 1 : 0);                  // 32-column blocks of this tile
  const int n0 = (ti * base + (ti < wide ? ti : wide)) * 32;
  const int m0 = by * 256;
  const int M = a.M, K = a.K, N = sg.N;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int stage_bytes = kVwABytes + a.vw_maxw * 4096;
  if (wave == 8) {
    switch (width) {
      case 2: vw_loader<2>(sg, gemm_smem, stage_bytes, m0, n0, K, lane); break;
      case 3: vw_loader<3>(sg, gemm_smem, stage_bytes, m0, n0, K, lane); break;
      case 4: vw_loader<4>(sg, gemm_smem, stage_bytes, m0, n0, K, lane); break;
      default: vw_loader<kVw256LoaderMaxW>(sg, gemm_smem, stage_bytes, m0, n0, K, lane); break;
    }
    return;
  }
  const int wn = wave & 1;
  const int nj0 = (width + 1) >> 1;
  const int nj = wn ? width - nj0 : nj0;
  const int brow0 = wn ? nj0 * 32 : 0;
  switch (nj) {
    case 1: vw_mma<1>(a, sg, gemm_smem, stage_bytes, brow0, m0, n0, M, N, lane, wave); break;
    case 2: vw_mma<2>(a, sg, gemm_smem, stage_bytes, brow0, m0, n0, M, N, lane, wave); break;
    default: vw_mma<3>(a, sg, gemm_smem, stage_bytes, brow0, m0, n0, M, N, lane, wave); break;
  }
}

// ---------------------------------------------------------------------------
// The same tiles, 256 rows high: eight waves, 4 x 2, each 64 rows x half the width.
//
// With one MFMA wave per SIMD (gemm_ring_kernel) nothing runs while the first fragments of a step come
// out of LDS after the barrier.  Here every SIMD has two, and a step is twice the
// products for 1.33 times the bytes (256 x 256 against 128 x 256).  There is no loader wave: a ninth
// wave would leave each wave 168 registers (three on one SIMD), too few for 128 accumulators; the waves
// issue their share of a step's loads (at most 8 instructions of 1 KB) right behind a barrier, one step
// ahead into the second stage.  (A third stage, which tiles of up to 160 columns leave room for, and loads
// two steps ahead were measured: no faster, 4099 x 8192 x 2048 166 us against 161.)
// Rows past the matrix are clamped in the lane offsets, so edge tiles load like the others.
// What bounds it: a step of 256 x 256 reads 192 KB of fragments from LDS and writes 64 KB to it, 2048 cycles at
// 128 bytes per cycle, as many as its MFMAs take on each SIMD.  3000 x 5120 x 20480: 811 -> 580 us (1.08 PFLOP/s),
// 4099 x 2048 x 10240: 229 -> 172 us, against the fixed 128 x 128 tiles both launches had before (in turn on one part).
// ---------------------------------------------------------------------------
constexpr int kVw256Threads = 512;
static_assert(kVwStages * (kVwABytes + kVw256LoaderMaxW * 4096) <= 160 * 1024 && 2 * (kVwABytes + kVwMaxW * 4096) <= 160 * 1024 &&
                  8 * wave_sums_bytes((kVwMaxW + 1) / 2) <= 160 * 1024, "LDS of a compute unit");

template <int NJ>
__device__ __forceinline__ void vw256_body(const GemmArgs& a, const GemmSeg& sg, unsigned char* smem, int width, int brow0,
                                           int m0, int n0, int lane, int wave) {
  const int M = a.M, K = a.K, N = sg.N, nk = K / kLdwBK, wm = wave >> 1;
  const unsigned stage_bytes = kVwABytes + a.vw_maxw * 4096;
  // this wave's loads: row groups 4 wave .. + 3 of A, row groups wave, wave + 8, ... of B (there are 4 width)
  unsigned va[4], vb[4];
  const int lr = lane >> 3, ls = (lane & 7) ^ lr;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int ga = wave * 4 + i, gb = wave + 8 * i;
    const int ra = m0 + ga * 8 + lr, rb = n0 + gb * 8 + lr;
    va[i] = (unsigned)((ra < M ? ra : M - 1) - m0) * (unsigned)(K * 2) + (ls ^ (ga & 1)) * 16;
    vb[i] = (unsigned)((rb < N ? rb : N - 1) - n0) * (unsigned)(K * 2) + (ls ^ (gb & 1)) * 16;
  }
  const unsigned char* abase = uniform_ptr(reinterpret_cast<const unsigned char*>(sg.A) + (size_t)m0 * K * 2);
  const unsigned char* bbase = uniform_ptr(sg.B + (size_t)n0 * K * 2);
  const unsigned lds0 = (unsigned)(size_t)((__attribute__((address_space(3))) unsigned char*)smem);
  const int nb = 4 * width;
  auto issue = [&](int step) {
    const unsigned st = lds0 + (step & 1) * stage_bytes;
    const unsigned char* ak = abase + (size_t)step * (kLdwBK * 2);
    const unsigned char* bk = bbase + (size_t)step * (kLdwBK * 2);
#pragma unroll
    for (int i = 0; i < 4; i++) load_lds_saddr(va[i], ak, st + (wave * 4 + i) * 1024);
#pragma unroll
    for (int i = 0; i < 4; i++)
      if (wave + 8 * i < nb) load_lds_saddr(vb[i], bk, st + kVwABytes + (wave + 8 * i) * 1024);
  };
  f16v acc[2][NJ];
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < NJ; j++)
#pragma unroll
      for (int v = 0; v < 16; v++) acc[i][j][v] = 0.f;
  issue(0);
  for (int k = 0; k < nk; k++) {
    // this wave's loads of step k have landed and its fragments of step k-1 are in registers; behind the
    // barrier that holds for all eight, so step k may be read and the slot of step k-1 refilled
    __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) lgkmcnt(0)
    step_barrier();
    if (k + 1 < nk) issue(k + 1);
    const unsigned char* st = smem + (k & 1) * stage_bytes;
#pragma unroll
    for (int kb = 0; kb < 4; kb++) {
      h8 fa[2], fb[NJ];
      const int q = kb * 2 + (lane >> 5);
#pragma unroll
      for (int i = 0; i < 2; i++) fa[i] = *reinterpret_cast<const h8*>(st + ldw_at(wm * 64 + i * 32 + (lane & 31), q));
#pragma unroll
      for (int j = 0; j < NJ; j++)
        fb[j] = *reinterpret_cast<const h8*>(st + kVwABytes + ldw_at(brow0 + j * 32 + (lane & 31), q));
#pragma unroll
      for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < NJ; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[i], fb[j], acc[i][j], 0, 0, 0);
    }
  }
  if (m0 + 256 <= M && n0 + width * 32 <= N) {
    gemm_epilogue_t<2, NJ, true>(a, sg, acc, m0 + wm * 64, n0 + brow0, M, N, lane);
  } else {
    step_barrier();  // all fragments have been read
    finish_wave(a, sg, acc, reinterpret_cast<float*>(smem + wave * wave_sums_bytes((a.vw_maxw + 1) / 2)), m0 + wm * 64, n0 + brow0, M, N, lane);
  }
}

__global__ __launch_bounds__(kVw256Threads) void gemm_vw256_kernel(GemmArgs a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char gemm_smem[];
  int bx, by;
  xcd_tile(bx, by);
  int sidx = 0;
#pragma unroll
  for (int i = 1; i < kGemmMaxSeg; i++) sidx += (i < a.nseg && bx >= a.tile_start[i]) ? 1 : 0;
  const GemmSeg& sg = a.seg[sidx];
  const int ti = bx - a.tile_start[sidx];
  const int base = a.vw_base[sidx], wide = a.vw_wide[sidx];
  const int width = base + (ti < wide ? 1 : 0);  // 32-column blocks of this tile
  const int n0 = (ti * base + (ti < wide ? ti : wide)) * 32;
  const int m0 = by * 256;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nj0 = (width + 1) >> 1;
  const int nj = (wave & 1) ? width - nj0 : nj0;
  const int brow0 = (wave & 1) ? nj0 * 32 : 0;
  switch (nj) {  // every wave passes the same barriers, whatever its width
    case 1: vw256_body<1>(a, sg, gemm_smem, width, brow0, m0, n0, lane, wave); break;
    case 2: vw256_body<2>(a, sg, gemm_smem, width, brow0, m0, n0, lane, wave); break;
    case 3: vw256_body<3>(a, sg, gemm_smem, width, brow0, m0, n0, lane, wave); break;
    default: vw256_body<4>(a, sg, gemm_smem, width, brow0, m0, n0, lane, wave); break;
  }
}

// How one launch of binary16 weights, not split over K, is cut into tiles.
struct GemmRoute {
  int rows = 0;        // of a tile: 64 or 128 (with a loader wave; gemm_ring_kernel has taken their place), 256; 0: none of these
  bool loader = true;  // 256 rows: gemm_vw_kernel, not gemm_vw256_kernel
  int blocks = 0;      // widest tile, in blocks of 32 columns
  int rounds = 0;      // over the compute units
  double us = 0;       // what the launch is expected to take
  dim3 grid;
  size_t lds = 0;
  GemmArgs a;          // with the tile tables of this cut
};

static long tiles64(const GemmArgs& a) {
  long n = 0;
  for (int s = 0; s < a.nseg; s++) n += (long)((a.seg[s].N + BN - 1) / BN) * ((a.M + 63) / 64);
  return n;
}

// Expected times, us, with k = K / 2048: 2 + rounds x (a part that does not depend on K + k x (fixed + slope x widest
// tile)).  Fitted to 825 products of 65 to 4099 rows, K 768 to 20480, N 768 to 65536, weights from memory: the kernels
// chosen by them take 0.3 % longer than the best of each product's, none but a few at equal prices more than 4 %.
// Rounds at K = 2048 as measured: 64 rows 14-18; 128 rows, widths 3 / 5 / 8: 22 / 26 / 38; 256 rows, widths 3 / 5 / 7 /
// 8: 36 / 44 / 54 / 65 (the widest tiles of full strips run at the lowest clock).  300 x 2048 x 6144: 19.2 us as one
// round of 64-row tiles, 22.7 as 128 x 96; 3000 x 2048 x 8192: 105.5 as 256 rows, 119 as 128; 640 x 2048 x 65536, three
// strips of 256 rows, half of the last one empty: 200 as 128 rows, 217 as 256.
static double us_64(int rounds, double k) { return 2 + rounds * (2.4 + 14.2 * k); }
static double us_128(int rounds, double k, int w) { return 2 + rounds * (5 + k * (5 + 3.55 * w)); }
static double us_256(int rounds, double k, int w) { return 2 + rounds * (6.6 + k * (11.8 + 5.45 * w + (w == 8 ? 3 : 0))); }
static double us_256_loader(int rounds, double k, int w) { return 2 + rounds * (5.7 + k * (5.8 + 6.8 * w)); }
constexpr double kLaunchUs = 3;  // one more launch

bool deal_tiles(GemmArgs& a, int P) {
  if (P < a.nseg) return false;
  int cb[kGemmMaxSeg], t[kGemmMaxSeg], total = 0, used = 0;
  for (int s = 0; s < a.nseg; s++) {
    cb[s] = (a.seg[s].N + 31) / 32;
    total += cb[s];
  }
  for (int s = 0; s < a.nseg; s++) {
    t[s] = (int)((long)P * cb[s] / total);
    if (t[s] < 1) t[s] = 1;
    used += t[s];
  }
  if (used > P) return false;
  // the spare tiles go where the tiles are widest; among equals, to the segment whose epilogue
  // costs most (a transcendental per element), so that its tiles are the narrow ones
  auto heavy = [&](int s) { return a.seg[s].epi == G_SIGMOID || a.seg[s].epi == G_SILU ? 1 : 0; };
  while (used < P) {
    int best = 0;
    for (int s = 1; s < a.nseg; s++) {
      const long l = (long)cb[s] * t[best], q = (long)cb[best] * t[s];
      if (l > q || (l == q && heavy(s) > heavy(best))) best = s;
    }
    t[best]++;
    used++;
  }
  int tiles = 0;
  a.vw_maxw = 0;
  for (int s = 0; s < a.nseg; s++) {
    const int w = (cb[s] + t[s] - 1) / t[s];
    a.vw_maxw = w > a.vw_maxw ? w : a.vw_maxw;
    a.tile_start[s] = tiles;
    a.vw_base[s] = cb[s] / t[s];
    a.vw_wide[s] = cb[s] % t[s];
    tiles += t[s];
  }
  for (int s = a.nseg; s <= kGemmMaxSeg; s++) a.tile_start[s] = INT_MAX;
  a.tile_start[a.nseg] = tiles;
  return true;
}

// Cuts the launch into tiles of bm rows (256, or 128 for the price alone): the fewest rounds over `cus` compute units whose widest tile
// fits.  r.rows stays 0 if it is too small for tiles of at least bm x 96, or too ragged.
static GemmRoute plan_vw(const GemmArgs& args, int bm, int cus) {
  GemmRoute r;
  r.a = args;
  GemmArgs& a = r.a;
  // gemm_vw256_kernel addresses the 256 rows of a tile with 32-bit byte offsets
  if (bm == 256 && (size_t)a.K * 2 * 256 > 0xffffffffull) return r;
  const int mt = (a.M + bm - 1) / bm;
  int total = 0;
  for (int s = 0; s < a.nseg; s++) total += (a.seg[s].N + 31) / 32;
  // From the fewest rounds that tiles of the largest width allow; it ends at tiles of one block at the latest.  (With a
  // limit of 32 rounds 8193 x 2048 x 65536 took 3.14 ms on fixed 128 x 128 tiles, 2.06 so, one row less 1.97.)
  for (long rounds = ((long)total * mt + (long)kVwMaxW * cus - 1) / ((long)kVwMaxW * cus);; rounds++) {
    const int P = (int)(rounds * cus / mt);  // tiles per strip of rows
    if (!deal_tiles(a, P)) continue;
    const int maxw = a.vw_maxw, tiles = a.tile_start[a.nseg];
    int minw = INT_MAX;
    for (int s = 0; s < a.nseg; s++) minw = a.vw_base[s] < minw ? a.vw_base[s] : minw;
    if (maxw > kVwMaxW) continue;
    if (minw < 2 || maxw < 3) return r;
    if (bm == 256) {
      // Whole tiles of up to 160 columns: the loader wave's form, whose loads are two steps ahead.  All 256 compute
      // units multiply real data then and the clock is the lowest, which costs it less: 512 x 5120 x 20480 101 us
      // against 115, 2048 x 20480 x 5120 375 against 423, 1024 x 2048 x 10240 44 against 46.  With a part of a tile
      // empty the other form is the faster one (1793 x 5120 x 5120: 101 against 119): its edge tiles load like whole ones.
      r.loader = a.M % 256 == 0 && maxw <= kVw256LoaderMaxW;
      for (int s = 0; s < a.nseg; s++) r.loader = r.loader && a.seg[s].N % 32 == 0;
      r.lds = (r.loader ? kVwStages : 2) * (size_t)(kVwABytes + maxw * 4096);
      const size_t sums = 8 * (size_t)wave_sums_bytes((maxw + 1) / 2);  // the epilogue's place (finish_wave)
      if (r.lds < sums) r.lds = sums;
      r.grid = dim3(tiles, mt);
    }
    r.blocks = maxw;
    r.rounds = (int)rounds;
    r.us = bm == 128 ? us_128(r.rounds, a.K / 2048.0, maxw)
           : r.loader ? us_256_loader(r.rounds, a.K / 2048.0, maxw)
                      : us_256(r.rounds, a.K / 2048.0, maxw);
    r.rows = bm;
    return r;
  }
  return r;
}

// The cheapest cut.  rows stays 0 where the planned tiles do not fit and fixed 64-row tiles take more than a round.
static GemmRoute gemm_route(const GemmArgs& a, int cus) {
  GemmRoute r = plan_vw(a, 128, cus);
  const GemmRoute r2 = plan_vw(a, 256, cus);
  if (r2.rows && (!r.rows || r2.us < r.us)) r = r2;
  const int rounds = (int)((tiles64(a) + cus - 1) / cus);
  const double us = us_64(rounds, a.K / 2048.0);
  if (r.rows ? us < r.us : rounds == 1) {
    r.rows = 64;
    r.blocks = BN / 32;
    r.rounds = rounds;
    r.us = us;
    r.a = a;
    int tiles = 0;
    for (int s = 0; s < a.nseg; s++) {
      r.a.tile_start[s] = tiles;
      tiles += (a.seg[s].N + BN - 1) / BN;
    }
    for (int s = a.nseg; s <= kGemmMaxSeg; s++) r.a.tile_start[s] = INT_MAX;
    r.a.tile_start[a.nseg] = tiles;
    r.grid = dim3(tiles, (a.M + 63) / 64);
  }
  return r;
}

// A grouped launch whose products are cheaper one by one (2048 columns in one round of 64 x 128 tiles, 8192 in two of
// 128 x 192, together three) goes out as separate launches.  FRHIP_GEMM_SEPARATE=0: never.
// -> what that is expected to take, us; 0: it stays one launch
static double one_by_one(const GemmArgs& a, const GemmRoute& whole, int cus) {
  static const bool separate = !(getenv("FRHIP_GEMM_SEPARATE") && atoi(getenv("FRHIP_GEMM_SEPARATE")) == 0);
  if (!separate || a.nseg < 2) return 0;
  double us = kLaunchUs * (a.nseg - 1);
  for (int s = 0; s < a.nseg; s++) {
    GemmArgs one = a;
    one.nseg = 1;
    one.seg[0] = a.seg[s];
    const GemmRoute r = gemm_route(one, cus);
    if (!r.rows) return 0;
    us += r.us;
  }
  return !whole.rows || us < whole.us ? us : 0;
}

static void gemm_vw_launch(const GemmRoute& r, hipStream_t st) {
  static const bool raised = [] {
    for (const void* f : {reinterpret_cast<const void*>(&gemm_vw_kernel), reinterpret_cast<const void*>(&gemm_vw256_kernel)})
      (void)hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    return true;
  }();
  (void)raised;
  if (r.loader)
    hipLaunchKernelGGL(gemm_vw_kernel, r.grid, dim3(576), r.lds, st, r.a);
  else
    hipLaunchKernelGGL(gemm_vw256_kernel, r.grid, dim3(kVw256Threads), r.lds, st, r.a);
}

// How a launch of binary16 weights that is not split over K goes out: gemm_ring_kernel's tiles in place of every cut of 64 or 128
// rows (1.20 and 1.11 times as fast over 75 products of 200 to 2048 rows, none slower: 512 x 2048 x 2048 15.8 -> 11.5 us, 300 x 4096 x
// (4 x 4096) 71.1 -> 60.5), and of 256 rows or product by product where they are expected to be quicker by a twentieth (29
// products: five, all of them the quicker ones; 1536 x 2048 x (3 x 2048) 58.2 -> 51.7; 1024 x 2560 x (2560 + 8960) stays, 70 against 79).
struct WholePlan {
  bool separate = false;
  TilePlan ring;  // rows = 0: the route
  GemmRoute route;
  double us = 0;
};
static WholePlan plan_whole(const GemmArgs& a, int cus) {
  WholePlan w;
  w.route = gemm_route(a, cus);
  w.ring = plan_ring(a, cus);
  const double apart = one_by_one(a, w.route, cus), other = apart ? apart : w.route.rows == 256 ? w.route.us : 0;
  w.us = w.ring.us;
  if (other && (!w.ring.rows || other <= w.ring.us * 1.05)) {
    w.separate = apart != 0;
    w.ring.rows = 0;
    w.us = other;
  }
  return w;
}

static constexpr size_t gemm_lds_bytes(int bm, int bk) { return (size_t)(bm + BN) * (bk + 8) * 2; }

// Tiles above 64 KB of LDS need the limit raised once per kernel.
template <int BM, int BK, bool U8>
static void gemm_launch_one(dim3 grid, hipStream_t st, const GemmArgs& a) {
  constexpr size_t lds = gemm_lds_bytes(BM, BK);
  static bool raised = false;
  if (lds > 64 * 1024 && !raised) {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_kernel<BM, BK, U8>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    raised = true;
  }
  hipLaunchKernelGGL((gemm_kernel<BM, BK, U8>), grid, dim3(kGemmThreads), lds, st, a);
}
#define FR_GEMM_LAUNCH(BM_, BK_)                         \
  do {                                                   \
    if (u8)                                              \
      gemm_launch_one<BM_, BK_, true>(grid, st, a);      \
    else                                                 \
      gemm_launch_one<BM_, BK_, false>(grid, st, a);     \
  } while (0)

// FRHIP_GEMM_BK=64|128 forces the K-step depth (measurement aid); default: 128 where K allows
// (256 was measured no faster than 128).
static int env_bk() {
  const char* e = getenv("FRHIP_GEMM_BK");
  return e ? atoi(e) : 0;
}

static bool env_on(const char* name) {
  const char* e = getenv(name);
  return !(e && atoi(e) == 0);
}

// Few rows (a short prompt): 64 x 128 tiles leave most compute units without a workgroup, and a workgroup pulls its
// weights through a ring of a few K-steps, so a launch takes about K / 64 round trips to memory however few
// rows there are (64 x 2048 x 2048, two steps in flight: 16 workgroups, 17-25 us for 8 MB).  With scratch for the partial sums such a
// launch is split over K into as many slices as there are idle compute units (at least four K-steps each), and the
// reduction pass adds the slices in order and applies each product's epilogue.  A group that is too wide for that as a
// whole goes out product by product, so that its narrow members still can.  FRHIP_GEMM_FEW_ROWS=0: off.
// *taken stays false, and nothing is launched, if the launch is not of this form.

// Slices of K for a launch of few rows on 64 x 128 tiles, 0 if it is not split as a whole.
static int few_rows_slices(const GemmArgs& a, size_t few_rows_floats, int cus) {
  long tiles = 0;
  size_t cols = 0;
  for (int s = 0; s < a.nseg; s++) {
    if (a.seg[s].N % 16 != 0) return 0;
    tiles += (a.seg[s].N + BN - 1) / BN;
    cols += (size_t)a.seg[s].N;
  }
  const int m64 = (a.M + 63) / 64, ksteps = a.K / kLdwBK;
  if (tiles * m64 * 2 > cus) return 0;
  const size_t stride = ((size_t)a.M * cols + 63) / 64 * 64;
  long S = cus / (tiles * m64);
  if (S > ksteps / 4) S = ksteps / 4;  // at least four K-steps per slice: twice the ring's depth in flight
  if ((size_t)S * stride > few_rows_floats) S = (long)(few_rows_floats / stride);
  return S < 2 ? 0 : (int)S;
}

// ... or, a group that does not fill the part, product by product, so that its narrow members are.  A group that fits as a
// whole and still gets no two slices has a K of four to seven steps: nor would its members get any, it stays one launch.
static bool few_rows_one_by_one(const GemmArgs& a, int cus) {
  const int m64 = (a.M + 63) / 64;
  long tiles = 0;
  bool any = false, all = true;
  for (int s = 0; s < a.nseg; s++) {
    const long t = (a.seg[s].N + BN - 1) / BN;
    tiles += t;
    any = any || (t * m64 * 2 <= cus && a.seg[s].N % 16 == 0);
    all = all && a.seg[s].N % 16 == 0;
  }
  return a.nseg > 1 && tiles * m64 < cus && any && !(all && tiles * m64 * 2 <= cus);
}

// S slices of K with their sums in `partial`: the segments side by side in every slice
static void split_over(GemmArgs& a, int S, float* partial) {
  size_t cols = 0;
  for (int s = 0; s < a.nseg; s++) {
    a.part_off[s] = (size_t)a.M * cols;
    cols += (size_t)a.seg[s].N;
  }
  a.part_off[a.nseg] = (size_t)a.M * cols;
  a.ksplit = S;
  a.partial = partial;
  a.partial_stride = (a.part_off[a.nseg] + 63) / 64 * 64;
}

// A launch in slices of K, and the launch that adds them
static int launch_split(const GemmArgs& a, int cus, hipStream_t st, const char* what) {
  const TilePlan p = plan_ring(a, cus);
  if (!p.rows) return set_error(FRHIP_ESHAPE, "gemm: rows too long");
  if (int rc = launch_gemm_ring(p, st, what)) return rc;
  launch_splitk_reduce(st, a);
  return check_launch(what);
}

static int launch_few_rows(GemmArgs& a, hipStream_t st, const char* what, float* few_rows, size_t few_rows_floats, bool* taken) {
  const int cus = compute_units();
  if (a.K / kLdwBK < 4) return 0;
  if (const int S = few_rows_slices(a, few_rows_floats, cus)) {
    split_over(a, S, few_rows);
    *taken = true;
    return launch_split(a, cus, st, what);
  }
  if (!few_rows_one_by_one(a, cus)) return 0;
  *taken = true;
  for (int s = 0; s < a.nseg; s++) {
    GemmArgs one = a;
    one.nseg = 1;
    one.seg[0] = a.seg[s];
    if (int rc = launch_gemm(one, false, st, what, nullptr, nullptr, 0, 0, few_rows, few_rows_floats)) return rc;
  }
  return 0;
}

// Slices of K of a single product with few outputs and a long K on 128 x 128 tiles (below), 0 if it is not split.
static int long_k_slices(const GemmArgs& a, size_t partial_stride, int max_split, int cus) {
  const int epi = a.seg[0].epi;
  if (max_split < 2 || a.nseg != 1 || a.K < 4096 || a.seg[0].N % 16 != 0 || (size_t)a.M * a.seg[0].N > partial_stride ||
      (epi != G_STORE_F16 && epi != G_STORE_F32 && epi != G_RESIDUAL && epi != G_FFN_OUT))
    return 0;
  const long t128 = (long)((a.seg[0].N + BN - 1) / BN) * ((a.M + 127) / 128);
  int S = (int)(cus / t128);
  if (S > max_split) S = max_split;
  while (S >= 2 && a.K / (kLdwBK * S) < 16) S--;
  return S >= 2 && t128 * S * 5 >= (long)cus * 3 ? S : 0;  // the slices fill at least 60 % of the CUs
}

// What launch_gemm's other binary16 forms are expected to take, us, in its order: split over K on 64-row tiles, product by
// product, split over K on 128-row tiles, planned tiles; all with a single loader wave, which gemm_ring_kernel has replaced
// since.  It is up to 1.4 times as quick, and still only 14 of 299 launches of 8 to 512 rows that go to gemm_few_kernel by this
// estimate would be the quicker on its tiles (widths 768 to 5120; 77 x 5120 x 5120 20.8 us against 26.6, the others by a seventh
// at most), of uint8 codes two: the line stays, and with it every launch's order of sums.  The split forms are fitted to 600 measured products (5 to 7 % rms),
// their reduction launch included.  Over 476 others of 4 to 512 rows all forms together came out 5 % quicker than expected (11 %
// rms), and what is chosen by it and few_us 0.9 % slower than the quicker form (gemm_few_kernel 295 times, 10 of them wrongly, by 14 %
// at most).  An expansion of uint8 codes is left out, so that codes and their image take the same form: uint8 products are 10 %
// over the quicker one, all of them among those that stay on tiles.
static double tiled_us(const GemmArgs& a, size_t partial_stride, int max_split, size_t few_rows_floats, int cus) {
  const double outs = [&] { double n = 0; for (int s = 0; s < a.nseg; s++) n += (double)a.M * a.seg[s].N; return n; }();
  auto each = [&](size_t floats) {
    double us = 0;
    for (int s = 0; s < a.nseg; s++) {
      GemmArgs one = a;
      one.nseg = 1;
      one.seg[0] = a.seg[s];
      us += tiled_us(one, 0, 0, floats, cus);
    }
    return us;
  };
  const int ksteps = a.K / kLdwBK;
  if (few_rows_floats && ksteps >= 4) {
    if (const int S = few_rows_slices(a, few_rows_floats, cus))
      return 6.8 + 0.37 * ((ksteps + S - 1) / S) + outs / a.M * a.K * 2 / 11.3e6 + 0.067 * S + outs * S * 8 / 4.27e6;
    if (few_rows_one_by_one(a, cus)) return each(few_rows_floats);
  }
  if (const int S = long_k_slices(a, partial_stride, max_split, cus)) return 10 + 0.66 * ((ksteps + S - 1) / S) + outs * S * 8 / 7.1e6;
  const GemmRoute r = gemm_route(a, cus);
  if (one_by_one(a, r, cus)) return each(0);
  return r.rows ? r.us : us_64((int)((tiles64(a) + cus - 1) / cus), a.K / 2048.0);
}

// plan_few's tile where it is worth it, with the scratch that the other forms would have
static FewPlan few_plan(const GemmArgs& a, size_t partial_stride, int max_split, size_t few_rows_floats, int cus) {
  const FewPlan p = plan_few(a, cus);
  return p.mt && p.us * 1.1 <= tiled_us(a, partial_stride, max_split, few_rows_floats, cus) ? p : FewPlan();
}

// uint8 weights through gemm_q8_kernel, in the slices of K that the binary16 launch would take, so with the same bits.  A group
// whose members are split one by one stays one launch where they take the same slices and their sums fit the scratch.
// With scratch for it (dq) the codes can be expanded instead, a launch of 5.5 us and 3 bytes of traffic a weight at 6.3 TB/s, and
// multiplied as binary16; many strips of rows dequantise every code once each, so from about 512 rows of a wide product on that is
// quicker.  Both ways measured over 488 launches of 65 to 4099 rows, widths 768 to 5120, us (expanded / on the codes): 777 x 14336
// x 4096 142 / 162, 1024 x 5120 x (5120 + 20480) 331 / 365; 384 x 768 x (768 + 3072) 18.1 / 13.3, 1024 x 768 x 768 10.0 / 9.2.  What is
// chosen with these figures, the 1.12 among them, is 0.7 % slower than the quicker way on average; with 2 us, 5 TB/s and 1 it was 2.5 %.
// (Prompts of 1024 tokens of the 1.5B shape 6479 -> 6112 us, of 700 of the 7B RWKV-5.2 width 1593 -> 1508, two layers of it.)
struct CodesPlan {
  int way = FRHIP_CODES_EXPANDED;  // or FRHIP_CODES_TILES: q, FRHIP_CODES_ONE_BY_ONE: a launch per product, each with a plan of its own
  TilePlan q;
};
// dq: with scratch for the expanded codes.  max_split, few_rows_floats: 0 without scratch for slices of that kind.
static CodesPlan plan_codes(const GemmArgs& a, bool dq, float* partial, size_t partial_stride, int max_split, float* few_rows,
                            size_t few_rows_floats, int cus) {
  CodesPlan c;
  const int ksteps = a.K / kLdwBK;
  GemmArgs b = a;
  if (few_rows_floats && ksteps >= 4) {
    if (const int S = few_rows_slices(a, few_rows_floats, cus)) {
      split_over(b, S, few_rows);
    } else if (few_rows_one_by_one(a, cus)) {
      int S = 0;
      for (int s = 0; s < a.nseg; s++) {
        GemmArgs one = a;
        one.nseg = 1;
        one.seg[0] = a.seg[s];
        const int Si = few_rows_slices(one, few_rows_floats, cus);
        S = s == 0 || Si == S ? Si : -1;
        if (S < 2) break;
      }
      // (not where a member could be one of gemm_few_kernel: its binary16 image would be)
      if (S >= 2 && a.tiled_sums) split_over(b, S, few_rows);
      if (b.ksplit < 2 || b.ksplit * b.partial_stride > few_rows_floats) {
        c.way = FRHIP_CODES_ONE_BY_ONE;
        return c;
      }
    }
  }
  if (b.ksplit < 2 && max_split)
    if (const int S = long_k_slices(a, partial_stride, max_split, cus)) {
      split_over(b, S, partial);
      b.partial_stride = partial_stride;
    }
  WholePlan w;
  if (b.ksplit < 2) w = plan_whole(a, cus);
  if (w.separate && !a.tiled_sums)
    for (int s = 0; s < a.nseg; s++) {  // the binary16 image's members could be gemm_few_kernel's
      GemmArgs one = a;
      one.nseg = 1;
      one.seg[0] = a.seg[s];
      if (few_plan(one, 0, 0, 0, cus).mt) return c;
    }
  c.q = plan_q8(b, cus);
  if (!c.q.rows) return c;
  if (dq) {
    double weights = 0;
    for (int s = 0; s < a.nseg; s++) weights += (double)a.seg[s].N * a.K;
    if (c.q.us * 1.12 > 5.5 + weights * 3 / 6.3e6 + (b.ksplit < 2 ? w.us : plan_ring(b, cus).us)) return c;
  }
  c.way = FRHIP_CODES_TILES;
  return c;
}

// *taken stays false, and nothing is launched, where the codes are to be expanded.
static int launch_codes(GemmArgs& a, hipStream_t st, const char* what, void* dq, float* partial, size_t partial_stride, int max_split,
                        float* few_rows, size_t few_rows_floats, bool* taken) {
  if (!q8_takes(a)) return 0;
  const CodesPlan c = plan_codes(a, dq != nullptr, partial, partial_stride, partial ? max_split : 0, few_rows, few_rows_floats, compute_units());
  if (c.way == FRHIP_CODES_EXPANDED) return 0;
  *taken = true;
  if (c.way == FRHIP_CODES_ONE_BY_ONE) {
    for (int s = 0; s < a.nseg; s++) {
      GemmArgs one = a;
      one.nseg = 1;
      one.seg[0] = a.seg[s];
      if (int rc = launch_gemm(one, true, st, what, dq, nullptr, 0, 0, few_rows, few_rows_floats)) return rc;
    }
    return 0;
  }
  if (int rc = launch_gemm_q8(c.q, st, what)) return rc;
  if (c.q.a.ksplit < 2) return 0;
  launch_splitk_reduce(st, c.q.a);
  return check_launch(what);
}

int launch_gemm(GemmArgs& a, bool u8, hipStream_t st, const char* what, void* dq, float* partial, size_t partial_stride,
                int max_split, float* few_rows, size_t few_rows_floats) {
  if (a.M <= 0) return 0;
  if (a.K <= 0 || a.K % 64 != 0) return set_error(FRHIP_ESHAPE, "gemm: K must be a positive multiple of 64");
  static const bool splitk = env_on("FRHIP_GEMM_SPLITK");
  // FRHIP_GEMM_LDW=0 selects gemm_kernel (measurement aid), which also takes rows too long for 32-bit byte offsets within a tile
  static const bool ldw_on = env_on("FRHIP_GEMM_LDW"), few = env_on("FRHIP_GEMM_FEW_ROWS");
  const bool ldw = ldw_on && (size_t)a.K * 2 * 256 <= 0xffffffffull;
  const bool few_ok = ldw && splitk && few && few_rows;
  // Few rows: one launch with K split over the waves of a workgroup where that is expected to be the quicker form by a
  // tenth (both estimates are good to that).  Every workgroup of it reads all rows of X: a long K over few columns is quicker
  // split over K in memory (64 x 20480 x 5120: 45 us against 64; 77 x 8192 x 2048: 17.3 both), many rows of wide products on
  // planned tiles (256 x 5120 x (5120 + 20480): 91 against 143).  Decided by the sizes alone: uint8 codes and their binary16
  // image, expanded here or kept by the caller, give the same bits.
  const FewPlan fp = ldw && splitk && few && !a.tiled_sums
                         ? few_plan(a, partial ? partial_stride : 0, partial ? max_split : 0, few_ok ? few_rows_floats : 0, compute_units())
                         : FewPlan();
  if (fp.mt && few_takes(a, u8)) return launch_gemm_few(a, fp, u8, st, what);
  if (u8 && !fp.mt && a.M >= kDequantRows && ldw && splitk) {
    bool taken = false;
    const int rc = launch_codes(a, st, what, dq, partial, partial_stride, max_split, few_ok ? few_rows : nullptr, few_ok ? few_rows_floats : 0, &taken);
    if (taken) return rc;
  }
  if (u8 && dq && a.M >= kDequantRows) {
    // Expanding N x K codes costs 3 bytes of traffic per weight, once for all strips of rows (launch_codes).
    h1* dst = static_cast<h1*>(dq);
    const unsigned char* qs[kGemmMaxSeg];
    const h1 *mxs[kGemmMaxSeg], *rxs[kGemmMaxSeg], *mys[kGemmMaxSeg], *rys[kGemmMaxSeg];
    h1* dsts[kGemmMaxSeg];
    int ns[kGemmMaxSeg];
    for (int s = 0; s < a.nseg; s++) {
      GemmSeg& g = a.seg[s];
      qs[s] = g.B; mxs[s] = g.mx; rxs[s] = g.rx; mys[s] = g.my; rys[s] = g.ry; ns[s] = g.N;
      dsts[s] = dst;
      g.B = reinterpret_cast<const unsigned char*>(dst);
      dst += (size_t)g.N * a.K;
    }
    if (int rc = dequant_u8_group_async(a.nseg, qs, mxs, rxs, mys, rys, dsts, a.K, ns, st)) return rc;
    u8 = false;
    if (fp.mt && few_takes(a, false)) return launch_gemm_few(a, fp, false, st, what);
  }
  if (!u8 && few_ok) {
    bool taken = false;
    const int rc = launch_few_rows(a, st, what, few_rows, few_rows_floats, &taken);
    if (taken) return rc;
  }
  const int cus = compute_units();
  // Split K: a single product with few outputs and a long K (ffn value: 1024 x 8192 x 2048) fills the compute units only
  // with 64 x 128 tiles, which ask L2 for 1.5 times the bytes of 128 x 128 tiles per product and are bound by just that
  // (786 MB in 57 us).  With scratch for the partial sums the launch runs ksplit slices of K, and a
  // second kernel adds the slices in order and applies the epilogue.  The sums are grouped by slice, so the result can
  // differ from the unsplit launch in the last fp32 bit before the rounding to binary16.  FRHIP_GEMM_SPLITK=0: off.
  if (!u8 && ldw && splitk && partial) {
    if (const int S = long_k_slices(a, partial_stride, max_split, cus)) {
      split_over(a, S, partial);
      a.partial_stride = partial_stride;
      return launch_split(a, cus, st, what);
    }
  }
  if (!u8 && ldw) {
    const WholePlan w = plan_whole(a, cus);
    if (w.separate) {
      for (int sgi = 0; sgi < a.nseg; sgi++) {
        GemmArgs one = a;
        one.nseg = 1;
        one.seg[0] = a.seg[sgi];
        if (int rc = launch_gemm(one, false, st, what, nullptr, nullptr, 0, 0, nullptr, 0)) return rc;
      }
      return 0;
    }
    if (w.ring.rows) return launch_gemm_ring(w.ring, st, what);
    gemm_vw_launch(w.route, st);
    return check_launch(what);
  }
  int tiles = 0;
  for (int s = 0; s < a.nseg; s++) {
    a.tile_start[s] = tiles;
    tiles += (a.seg[s].N + BN - 1) / BN;
  }
  for (int s = a.nseg; s <= kGemmMaxSeg; s++) a.tile_start[s] = INT_MAX;
  a.tile_start[a.nseg] = tiles;
  // 128-row tiles unless that leaves fewer than ~1.5 workgroups per CU; then 64-row tiles
  const int m128 = (a.M + 127) / 128;
  static const int force_bk = env_bk();
  const bool deep_ok = (force_bk ? force_bk == 128 : true) && a.K % 128 == 0;
  if ((long)tiles * m128 < (long)cus * 3 / 2) {
    dim3 grid(tiles, (a.M + 63) / 64);
    if (deep_ok) FR_GEMM_LAUNCH(64, 128); else FR_GEMM_LAUNCH(64, 64);
  } else {
    dim3 grid(tiles, m128);
    if (deep_ok) FR_GEMM_LAUNCH(128, 128); else FR_GEMM_LAUNCH(128, 64);
  }
  return check_launch(what);
}

void gemm_add_seg(GemmArgs& a, const void* A, const frhip_weight* w, void* out, int epi) {
  GemmSeg& s = a.seg[a.nseg++];
  s.A = static_cast<const h1*>(A);
  s.B = static_cast<const unsigned char*>(w->data);
  s.mx = static_cast<const h1*>(w->mx);
  s.rx = static_cast<const h1*>(w->rx);
  s.my = static_cast<const h1*>(w->my);
  s.ry = static_cast<const h1*>(w->ry);
  s.out = out;
  s.N = w->N;
  s.epi = epi;
}

}  // namespace frhip

using namespace frhip;

// matmul, matrix x matrix (kernels/cuda/matmul.cpp:110-121): x [T][K] binary16, y [T][N].
extern "C" int frhip_gemm(const void* x, const frhip_weight* w, void* y, int T, int out_dtype, frhip_stream s) {
  if (!x || !w || !w->data || !y) return set_error(FRHIP_EINVAL, "gemm: null pointer");
  if (T < 0) return set_error(FRHIP_ESHAPE, "gemm: negative T");
  if (out_dtype != FRHIP_F16 && out_dtype != FRHIP_F32) return set_error(FRHIP_EINVAL, "gemm: out_dtype must be F16 or F32");
  if (w->dtype != FRHIP_F16 && w->dtype != FRHIP_U8) return set_error(FRHIP_EINVAL, "gemm: weight dtype must be F16 or U8");
  if (w->dtype == FRHIP_U8 && (!w->mx || !w->rx || !w->my || !w->ry)) return set_error(FRHIP_EINVAL, "gemm: uint8 weight without mx/rx/my/ry");
  if (reinterpret_cast<uintptr_t>(x) % 16 != 0 || reinterpret_cast<uintptr_t>(w->data) % 16 != 0)
    return set_error(FRHIP_EINVAL, "gemm: operands must be 16-byte aligned");
  GemmArgs a;
  memset(&a, 0, sizeof(a));
  a.M = T;
  a.K = w->K;
  gemm_add_seg(a, x, w, y, out_dtype == FRHIP_F32 ? G_STORE_F32 : G_STORE_F16);
  return launch_gemm(a, w->dtype == FRHIP_U8, static_cast<hipStream_t>(s), "gemm");
}

extern "C" int frhip_gemm_route(int T, int K, int nproducts, const int* N, int compute_units, int* out) {
  if (!N || !out) return set_error(FRHIP_EINVAL, "gemm_route: null pointer");
  if (T <= 0 || K <= 0 || K % 64 != 0 || nproducts < 1 || nproducts > kGemmMaxSeg || compute_units < 1)
    return set_error(FRHIP_ESHAPE, "gemm_route: no such launch");
  GemmArgs a;
  memset(&a, 0, sizeof(a));
  a.M = T;
  a.K = K;
  for (int s = 0; s < nproducts; s++) {
    if (N[s] <= 0) return set_error(FRHIP_ESHAPE, "gemm_route: no such launch");
    a.seg[s].N = N[s];
  }
  a.nseg = nproducts;
  if ((size_t)K * 2 * 256 > 0xffffffffull) {  // launch_gemm: gemm_kernel
    memset(out, 0, sizeof(int) * 4 * nproducts);
    return 1;
  }
  const WholePlan whole = plan_whole(a, compute_units);
  for (int s = 0; s < nproducts; s++) {
    WholePlan w = whole;
    if (whole.separate) {
      GemmArgs one = a;
      one.nseg = 1;
      one.seg[0] = a.seg[s];
      w = plan_whole(one, compute_units);
    }
    const bool ring = w.ring.rows != 0;
    out[4 * s] = ring ? w.ring.rows : w.route.rows;
    out[4 * s + 1] = ring ? w.ring.a.vw_maxw : w.route.blocks;
    out[4 * s + 2] = ring ? w.ring.rounds : w.route.rounds;
    out[4 * s + 3] = ring || w.route.loader;
  }
  return whole.separate ? nproducts : 1;
}

static int tile_args(GemmArgs& a, int T, int K, int nproducts, const int* N, int slices, int compute_units, const int* out, const char* what) {
  if (!N || !out) return set_error(FRHIP_EINVAL, what);
  if (T <= 0 || K <= 0 || K % 64 != 0 || nproducts < 1 || nproducts > kGemmMaxSeg || compute_units < 1 || slices < 1 || slices > K / 64)
    return set_error(FRHIP_ESHAPE, what);
  memset(&a, 0, sizeof(a));
  a.M = T;
  a.K = K;
  a.nseg = nproducts;
  a.ksplit = slices;
  for (int s = 0; s < nproducts; s++) {
    if (N[s] <= 0) return set_error(FRHIP_ESHAPE, what);
    a.seg[s].N = N[s];
  }
  return 0;
}

static void tell(const TilePlan& p, int* out) {
  out[0] = p.rows;
  out[1] = p.rows ? p.a.vw_maxw : 0;
  out[2] = p.rounds;
}

extern "C" int frhip_gemm_ring_tile(int T, int K, int nproducts, const int* N, int slices, int compute_units, int* out) {
  GemmArgs a;
  if (int rc = tile_args(a, T, K, nproducts, N, slices, compute_units, out, "gemm_ring_tile: no such launch")) return rc;
  tell(plan_ring(a, compute_units), out);
  out[3] = plan_whole(a, compute_units).ring.rows != 0;
  return 0;
}

extern "C" int frhip_gemm_q8_tile(int T, int K, int nproducts, const int* N, int slices, int compute_units, int* out) {
  GemmArgs a;
  if (int rc = tile_args(a, T, K, nproducts, N, slices, compute_units, out, "gemm_q8_tile: no such launch")) return rc;
  tell(plan_q8(a, compute_units), out);
  return 0;
}

extern "C" int frhip_gemm_few_tile(int T, int K, int nproducts, const int* N, int compute_units, int* out) {
  if (!N || !out) return set_error(FRHIP_EINVAL, "gemm_few_tile: null pointer");
  if (T <= 0 || K <= 0 || K % 64 != 0 || nproducts < 1 || nproducts > kGemmMaxSeg || compute_units < 1)
    return set_error(FRHIP_ESHAPE, "gemm_few_tile: no such launch");
  GemmArgs a;
  memset(&a, 0, sizeof(a));
  a.M = T;
  a.K = K;
  a.nseg = nproducts;
  for (int s = 0; s < nproducts; s++) {
    if (N[s] <= 0) return set_error(FRHIP_ESHAPE, "gemm_few_tile: no such launch");
    a.seg[s].N = N[s];
  }
  const FewPlan p = few_plan(a, 0, 0, 0, compute_units);
  out[0] = p.mt;
  out[1] = p.nt;
  return 0;
}

// A launch of the seq operators as frhip_seq_gemm_form and frhip_seq_codes_way are asked about, with the scratch it has
struct AskedLaunch {
  GemmArgs a;
  size_t stride = 0, floats = 0;
  int max_split = 0;
  bool v4 = false;
};
static int asked_launch(AskedLaunch& q, int T, int K, int nproducts, const int* N, int which, int compute_units, const int* out, const char* what) {
  if (int rc = tile_args(q.a, T, K, nproducts, N, 1, compute_units, out, what)) return rc;
  q.v4 = (which & FRHIP_SEQ_V4) != 0;
  q.floats = T <= kFewRowsMax ? kFewRowsFloats : 0;
  if (which & FRHIP_SEQ_FFN_VALUE) {
    q.a.seg[0].epi = G_FFN_OUT;
    q.stride = (size_t)T * N[0];
    q.max_split = kSeqMaxSplit;
  }
  return 0;
}

extern "C" int frhip_seq_gemm_form(int T, int K, int nproducts, const int* N, int which, int compute_units, int* out) {
  AskedLaunch q;
  if (int rc = asked_launch(q, T, K, nproducts, N, which, compute_units, out, "seq_gemm_form: no such launch")) return rc;
  out[0] = out[1] = 0;
  if (q.v4) {
    const FewPlan p = few_plan(q.a, q.stride, q.max_split, q.floats, compute_units);
    out[0] = p.mt;
    out[1] = p.nt;
    if (p.mt) return FRHIP_FORM_FEW;
  }
  if (q.floats && K / kLdwBK >= 4) {
    out[0] = few_rows_slices(q.a, q.floats, compute_units);
    if (out[0]) return FRHIP_FORM_SPLIT;
    if (few_rows_one_by_one(q.a, compute_units)) return FRHIP_FORM_ONE_BY_ONE;
  }
  out[0] = long_k_slices(q.a, q.stride, q.max_split, compute_units);
  return out[0] ? FRHIP_FORM_SPLIT : FRHIP_FORM_TILES;
}

extern "C" int frhip_seq_codes_way(int T, int K, int nproducts, const int* N, int which, int compute_units, int* out) {
  AskedLaunch q;
  if (int rc = asked_launch(q, T, K, nproducts, N, which, compute_units, out, "seq_codes_way: no such launch")) return rc;
  out[0] = out[1] = out[2] = 0;
  q.a.tiled_sums = !q.v4;
  if (q.v4 && few_plan(q.a, q.stride, q.max_split, q.floats, compute_units).mt) return FRHIP_CODES_FEW;
  if (T < kDequantRows || (size_t)K * 2 * 256 > 0xffffffffull) return FRHIP_CODES_EXPANDED;
  const CodesPlan c = plan_codes(q.a, true, nullptr, q.stride, q.max_split, nullptr, q.floats, compute_units);
  if (c.way == FRHIP_CODES_TILES) {
    tell(c.q, out);
    out[2] = c.q.a.ksplit > 1 ? c.q.a.ksplit : 1;
  }
  return c.way;
}

static_assert(FRHIP_ACT_SIGMOID == G_SIGMOID && FRHIP_ACT_RELU2 == G_RELU2 && FRHIP_ACT_SILU == G_SILU, "activation codes");

// matmul + in-place activation (kernels/cuda/ffn_seq.cu:78-81, att_seq.cu:394-395) in one launch.
extern "C" int frhip_gemm_act(const void* x, const frhip_weight* w, void* y, int T, int act, frhip_stream s) {
  if (!x || !w || !w->data || !y) return set_error(FRHIP_EINVAL, "gemm_act: null pointer");
  if (T < 0) return set_error(FRHIP_ESHAPE, "gemm_act: negative T");
  if (act != FRHIP_ACT_SIGMOID && act != FRHIP_ACT_RELU2 && act != FRHIP_ACT_SILU)
    return set_error(FRHIP_EINVAL, "gemm_act: act must be SIGMOID, RELU2 or SILU");
  if (w->dtype != FRHIP_F16 && w->dtype != FRHIP_U8) return set_error(FRHIP_EINVAL, "gemm_act: weight dtype must be F16 or U8");
  if (w->dtype == FRHIP_U8 && (!w->mx || !w->rx || !w->my || !w->ry)) return set_error(FRHIP_EINVAL, "gemm_act: uint8 weight without mx/rx/my/ry");
  if (reinterpret_cast<uintptr_t>(x) % 16 != 0 || reinterpret_cast<uintptr_t>(w->data) % 16 != 0)
    return set_error(FRHIP_EINVAL, "gemm_act: operands must be 16-byte aligned");
  GemmArgs a;
  memset(&a, 0, sizeof(a));
  a.M = T;
  a.K = w->K;
  gemm_add_seg(a, x, w, y, act);
  return launch_gemm(a, w->dtype == FRHIP_U8, static_cast<hipStream_t>(s), "gemm_act");
}
