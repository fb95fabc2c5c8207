// Products of binary16 weights on the MFMA units: four MFMA waves and four that load, tiles of 64 or 128 rows.
//
// Tiles, MFMAs and their order in k are those of gemm_vw_kernel (gemm.hip), so the bits are, too.  The loaders, one per SIMD, share
// a K-step's loads (global -> LDS, a scalar base and one of a few lane offsets each) and keep two or three steps in flight behind the
// one that is multiplied; they meet the MFMA waves at one barrier a step, behind which the slot of the step before is refilled.
// The sums go through LDS to the epilogue, which all eight waves share; fp32 outputs (k and v of the attention, slices of K)
// go straight from the accumulators, 128 bytes a row.
//
// What bounds it: a loader wave brings 1 KB in about 37 cycles and a compute unit keeps about 64 KB in flight, so that a step of 128 x
// 192 lasts as long as its loads (384 x 4096 x 16384: 66.8 us with a single loader two steps ahead, 55 without the products, 56 without
// the loads).  One loader and five waves -> four and eight, three steps ahead, us: 512 x 2048 x 2048 15.8 -> 11.5, 300 x 4096 x 4096
// 33.4 -> 24.3, 300 x 4096 x (4 x 4096) 71.1 -> 60.5, 1000 x 768 x (3 x 768) 16.4 -> 11.5, 1024 x 2048 x 2048 17.0 -> 14.8; in slices
// of K 300 x 8960 x 2560 40.0 -> 30.4, 1024 x 8192 x 2048 50.0 -> 44.9, 65 x 8960 x 2560 22.3 -> 18.3.
//
#include <climits>
#include <cmath>
#include <cstring>

#include "gemm_device.h"

#pragma clang fp contract(off)

namespace frhip {

constexpr int kRingLoaders = 4, kRingThreads = 64 * (4 + kRingLoaders), kRingMostBlocks = 8;
// K-steps in LDS: as many as 160 KB hold, up to four; tiles of 64 rows and up to 96 columns run two workgroups on a compute unit
constexpr int ring_stages(int bm, int w) { return bm == 128 && w > 6 ? 3 : 4; }
static_assert(4 * (128 * 128 + 6 * 4096) <= 160 * 1024 && 3 * (128 * 128 + 8 * 4096) <= 160 * 1024 && 4 * (64 * 128 + 8 * 4096) <= 160 * 1024, "LDS");

template <int BM, int S, int W>
__device__ __forceinline__ void ring_loader(const GemmSeg& sg, unsigned char* smem, int stage, int p, int m0, int n0, int M, int K, int kbase,
                                            int nk, int lane) {
  constexpr int NA = BM / 8 / kRingLoaders, NL = NA + W;
  static_assert(S == 3 || S == 4, "the waits of the last steps");
  static_assert((S - 1) * NL <= 63, "the wait counter's range");
  const int N = sg.N, lr = lane >> 3;
  unsigned va[NA], vb[W];
#pragma unroll
  for (int i = 0; i < NA; i++) {  // groups of 8 rows; rows past the matrix repeat its last one and are never stored
    const int g = p + kRingLoaders * i;
    va[i] = (unsigned)(min(m0 + g * 8 + lr, M - 1) - m0) * (unsigned)(K * 2) + (((lane & 7) ^ lr ^ (g & 1)) * 16);
  }
#pragma unroll
  for (int i = 0; i < W; i++) {
    const int g = p + kRingLoaders * i;
    vb[i] = (unsigned)(min(n0 + g * 8 + lr, N - 1) - n0) * (unsigned)(K * 2) + (((lane & 7) ^ lr ^ (g & 1)) * 16);
  }
  const unsigned char* ak = uniform_ptr(reinterpret_cast<const unsigned char*>(sg.A) + ((size_t)m0 * K + kbase) * 2);
  const unsigned char* bk = uniform_ptr(sg.B + ((size_t)n0 * K + kbase) * 2);
  const unsigned lds0 = (unsigned)(size_t)((__attribute__((address_space(3))) unsigned char*)smem) + p * 1024;
  unsigned at = lds0;
  const unsigned end = lds0 + S * stage;
  auto issue = [&] {
#pragma unroll
    for (int i = 0; i < W; i++) load_lds_saddr(vb[i], bk, at + BM * 128 + i * (kRingLoaders * 1024));
#pragma unroll
    for (int i = 0; i < NA; i++) load_lds_saddr(va[i], ak, at + i * (kRingLoaders * 1024));
    ak += 128;
    bk += 128;
    at += stage;
    at = at == end ? lds0 : at;
  };
#pragma unroll
  for (int i = 0; i < S - 1; i++)
    if (i < nk) issue();
  int k = 0;
  for (; k + S - 1 < nk; k++) {
    wait_loads<(S - 2) * NL>();  // step k has landed
    step_barrier();              // and step k - 1 has been read
    issue();                     // step k + S - 1, into the slot of step k - 1
  }
  for (; k < nk; k++) {
    const int behind = nk - 1 - k;
    if (S > 3 && behind >= 2) wait_loads<2 * NL>();
    else if (behind >= 1) wait_loads<NL>();
    else wait_loads<0>();
    step_barrier();
  }
}

template <int BM, int S, int NJ>
__device__ __forceinline__ void ring_mma(const GemmArgs& a, const GemmSeg& sg, unsigned char* smem, int stage, int maxw, bool direct, int m0,
                                         int n0, int brow0, int nk, int lane, int wm) {
  constexpr int MI = BM / 64, KG = MI * NJ >= 6 ? 2 : 4;
  if constexpr (NJ == 0) {  // a tile of one block: the first wave column has it
    for (int k = 0; k < nk; k++) step_barrier();
    if (!direct) step_barrier();
    return;
  } else {
  f16v acc[MI][NJ];
#pragma unroll
  for (int i = 0; i < MI; i++)
#pragma unroll
    for (int j = 0; j < NJ; j++)
#pragma unroll
      for (int v = 0; v < 16; v++) acc[i][j][v] = 0.f;
  const unsigned char* as = smem;
  for (int k = 0; k < nk; k++) {
    step_barrier();
    const unsigned char* bs = as + BM * 128;
#pragma unroll
    for (int kh = 0; kh < 4; kh += KG) {
      h8 fa[KG][MI], fb[KG][NJ];
#pragma unroll
      for (int kb = 0; kb < KG; kb++) {
        const int q = (kh + kb) * 2 + (lane >> 5);
#pragma unroll
        for (int i = 0; i < MI; i++) fa[kb][i] = *reinterpret_cast<const h8*>(as + ldw_at(wm * (BM / 2) + i * 32 + (lane & 31), q));
#pragma unroll
        for (int j = 0; j < NJ; j++) fb[kb][j] = *reinterpret_cast<const h8*>(bs + ldw_at(brow0 + j * 32 + (lane & 31), q));
      }
#pragma unroll
      for (int kb = 0; kb < KG; kb++)
#pragma unroll
        for (int i = 0; i < MI; i++)
#pragma unroll
          for (int j = 0; j < NJ; j++)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[kb][i], fb[kb][j], acc[i][j], 0, 0, 0);
    }
    as += stage;
    as = as == smem + S * stage ? smem : as;
  }
  if (direct) {
    const int row0 = m0 + wm * (BM / 2) + 4 * (lane >> 5), rows = a.M - row0;
    float* const out = static_cast<float*>(sg.out) + (size_t)row0 * sg.N + n0 + brow0 + (lane & 31);
    if (m0 + BM <= a.M) {
#pragma unroll
      for (int i = 0; i < MI; i++)
#pragma unroll
        for (int j = 0; j < NJ; j++)
#pragma unroll
          for (int v = 0; v < 16; v++) out[(size_t)(i * 32 + 8 * (v >> 2) + (v & 3)) * sg.N + j * 32] = acc[i][j][v];
    } else {
#pragma unroll
      for (int i = 0; i < MI; i++)
#pragma unroll
        for (int v = 0; v < 16; v++)
          if (i * 32 + 8 * (v >> 2) + (v & 3) < rows) {
#pragma unroll
            for (int j = 0; j < NJ; j++) out[(size_t)(i * 32 + 8 * (v >> 2) + (v & 3)) * sg.N + j * 32] = acc[i][j][v];
          }
    }
    return;
  }
  step_barrier();  // all fragments have been read
  const int pitch = sums_pitch(maxw);
#pragma unroll
  for (int i = 0; i < MI; i++) sums_to_lds(acc[i], reinterpret_cast<float*>(smem) + (wm * (BM / 2) + i * 32) * pitch + brow0, pitch, lane);
  }
}

template <int BM, int S>
__global__ __launch_bounds__(kRingThreads) void gemm_ring_kernel(GemmArgs a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char ring_smem[];
  constexpr int kMost = BM == 128 && S == 4 ? 6 : kRingMostBlocks;
  int bx, by;
  xcd_tile(bx, by);
  int sidx = 0;
#pragma unroll
  for (int i = 1; i < kGemmMaxSeg; i++) sidx += (i < a.nseg && bx >= a.tile_start[i]) ? 1 : 0;
  GemmSeg sg = a.seg[sidx];
  const int ti = bx - a.tile_start[sidx], base = a.vw_base[sidx], wide = a.vw_wide[sidx];
  const int width = base + (ti < wide ? 1 : 0);
  const int n0 = (ti * base + (ti < wide ? ti : wide)) * 32, m0 = by * BM;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ksplit = a.ksplit > 1 ? a.ksplit : 1, kz = blockIdx.z, ksteps = a.K / kLdwBK, kper = ksteps / ksplit, krem = ksteps % ksplit;
  const int nk = kper + (kz < krem ? 1 : 0), kbase = (kz * kper + (kz < krem ? kz : krem)) * kLdwBK;
  const int stage = BM * 128 + a.vw_maxw * 4096;
  if (a.ksplit > 1) {
    sg.out = a.partial + (size_t)kz * a.partial_stride + a.part_off[sidx];
    sg.epi = G_STORE_F32;
  }
  const bool direct = sg.epi == G_STORE_F32 && n0 + width * 32 <= sg.N;
  if (wave >= 4) {
    const int p = wave - 4;
    switch (width) {
      case 1: ring_loader<BM, S, 1>(sg, ring_smem, stage, p, m0, n0, a.M, a.K, kbase, nk, lane); break;
      case 2: ring_loader<BM, S, 2>(sg, ring_smem, stage, p, m0, n0, a.M, a.K, kbase, nk, lane); break;
      case 3: ring_loader<BM, S, 3>(sg, ring_smem, stage, p, m0, n0, a.M, a.K, kbase, nk, lane); break;
      case 4: ring_loader<BM, S, 4>(sg, ring_smem, stage, p, m0, n0, a.M, a.K, kbase, nk, lane); break;
      case 5: ring_loader<BM, S, 5>(sg, ring_smem, stage, p, m0, n0, a.M, a.K, kbase, nk, lane); break;
      case 6: ring_loader<BM, S, 6>(sg, ring_smem, stage, p, m0, n0, a.M, a.K, kbase, nk, lane); break;
      case 7: ring_loader<BM, S, kMost < 7 ? kMost : 7>(sg, ring_smem, stage, p, m0, n0, a.M, a.K, kbase, nk, lane); break;
      default: ring_loader<BM, S, kMost>(sg, ring_smem, stage, p, m0, n0, a.M, a.K, kbase, nk, lane); break;
    }
    if (!direct) step_barrier();
  } else {
    const int wm = wave >> 1, nj0 = (width + 1) >> 1, nj = (wave & 1) ? width - nj0 : nj0, brow0 = (wave & 1) ? nj0 * 32 : 0;
    switch (nj) {  // every wave passes the same barriers, whatever its width
      case 0: ring_mma<BM, S, 0>(a, sg, ring_smem, stage, a.vw_maxw, direct, m0, n0, brow0, nk, lane, wm); break;
      case 1: ring_mma<BM, S, 1>(a, sg, ring_smem, stage, a.vw_maxw, direct, m0, n0, brow0, nk, lane, wm); break;
      case 2: ring_mma<BM, S, 2>(a, sg, ring_smem, stage, a.vw_maxw, direct, m0, n0, brow0, nk, lane, wm); break;
      case 3: ring_mma<BM, S, 3>(a, sg, ring_smem, stage, a.vw_maxw, direct, m0, n0, brow0, nk, lane, wm); break;
      default: ring_mma<BM, S, kMost / 2>(a, sg, ring_smem, stage, a.vw_maxw, direct, m0, n0, brow0, nk, lane, wm); break;
    }
  }
  if (direct) return;
  __syncthreads();
  finish_tile<BM, kRingThreads>(a, sg, reinterpret_cast<const float*>(ring_smem), sums_pitch(a.vw_maxw), width, m0, n0, a.M, sg.N);
}

// What a launch of such tiles is expected to take, us (slices of K: with their reduction launch): fitted to 1985 measured ones (13 to
// 2048 rows, widths 768 to 4096, the products of a layer, weights from memory; 11 % rms, the tile chosen by it 1 % slower than the best).
static double ring_us(const GemmArgs& a, int bm, long rounds, int w) {
  const int S = a.ksplit > 1 ? a.ksplit : 1, steps = (a.K / kLdwBK + S - 1) / S;
  double cols = 0;
  for (int s = 0; s < a.nseg; s++) cols += a.seg[s].N;
  const double r = bm == 64 && w <= 3 ? 1 + (rounds - 1) * 0.81 : rounds;  // two workgroups on a compute unit
  const double x = r * (bm == 128 ? 3.0 + 0.101 * w + steps * (0.124 + 0.108 * w - (w >= 7 ? 0.028 : 0)) : 1.31 + 0.32 * w + steps * (0.088 + 0.072 * w));
  const double y = cols * a.K * 2 / 4.71e6;
  return 2.6 + sqrt(sqrt(x * x * x * x + y * y * y * y)) + (S > 1 ? 2.5 + S * a.M * cols * 8 / 6.5e6 : 0);
}

TilePlan plan_ring(const GemmArgs& args, int cus) {
  TilePlan best;
  const int S = args.ksplit > 1 ? args.ksplit : 1;
  if ((size_t)args.K * 2 * 256 > 0xffffffffull) return best;  // 32-bit byte offsets within a tile
  for (int bm : {128, 64}) {
    const long slots = (args.M + bm - 1) / bm * (long)S;  // workgroups per column of tiles
    for (int w = kRingMostBlocks; w >= 1; w--) {
      // as few tiles as this width allows, then as many as their rounds hold
      long need = 0;
      for (int s = 0; s < args.nseg; s++) need += ((args.seg[s].N + 31) / 32 + w - 1) / w;
      const long rounds = (need * slots + cus - 1) / cus;
      TilePlan p;
      p.a = args;
      auto dealt = [&](long tiles) {
        if (tiles > INT_MAX || !deal_tiles(p.a, (int)tiles) || p.a.vw_maxw > w) return false;
        for (int s = 0; s < args.nseg; s++)
          if (p.a.vw_base[s] < 1) return false;
        return true;
      };
      if (!dealt(rounds * cus / slots) && !dealt(need)) continue;
      p.us = ring_us(args, bm, rounds, p.a.vw_maxw);
      p.rows = bm;
      p.rounds = (int)rounds;
      p.grid = dim3(p.a.tile_start[p.a.nseg], (args.M + bm - 1) / bm, S);
      if (!best.rows || p.us < best.us) best = p;
    }
  }
  return best;
}

template <int BM, int S>
static void ring_launch(const TilePlan& p, hipStream_t st) {
  static const bool raised = [] {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_ring_kernel<BM, S>), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    return true;
  }();
  (void)raised;
  const int ring = S * (BM * 128 + p.a.vw_maxw * 4096), sums = BM * sums_pitch(p.a.vw_maxw) * 4;
  hipLaunchKernelGGL((gemm_ring_kernel<BM, S>), p.grid, dim3(kRingThreads), ring > sums ? ring : sums, st, p.a);
}

int launch_gemm_ring(const TilePlan& p, hipStream_t st, const char* what) {
  if (p.rows == 64) ring_launch<64, 4>(p, st);
  else if (ring_stages(128, p.a.vw_maxw) == 4) ring_launch<128, 4>(p, st);
  else ring_launch<128, 3>(p, st);
  return check_launch(what);
}

}  // namespace frhip
