// Products of uint8 weights on the MFMA units, the codes dequantised on their way into LDS by waves that do nothing else.
//
// Workgroup tile BM x (32 w): four MFMA waves (2 x 2, as in gemm_vw_kernel: the same MFMAs in the same k order, so the same
// bits as the binary16 kernels give on the expanded matrix) and eight producer waves, two per SIMD.  A producer
// brings its share of X and of the codes, global -> LDS directly, three K-steps of 64 ahead, turns its codes into binary16
// with the formula of the standalone dequantisation and leaves them where the MFMA waves read their fragments, one step
// ahead of them.  A wave dequantises the codes that it loaded itself, so only the finished step needs a barrier: one a step,
// for all twelve waves.  The sums go through LDS to the epilogue, which all of them share.
//
// What bounds it: a wave issues an instruction every 6 to 10 cycles here, whatever the other waves of its SIMD do, so what
// counts is the producer's instructions from barrier to barrier (110 for one block of 16 columns, 182 for two: 64 a block for
// its codes, 4 a code).  512 x 2560 x (4 x 2560), us: four producers 55, eight 61 (1100 spilled registers in an epilogue of the
// four MFMA waves) -> 50 with the sums through LDS -> 46 with the loop free of branches and address arithmetic; the
// expansion of the codes and the binary16 product 59.  Products of a layer, expansion and binary16 kernels -> this one:
//   13 rows (codes dequantised in registers, 64 x 128 tiles): 2560 x (4 x 2560) 25.7 -> 18.6, 8192 x 2048 17.5 -> 14.9
//   128 rows: 4096 x (4 x 4096) 73.5 -> 38.9, 14336 x 4096 71.6 -> 37.3;  300 rows: 2560 x (2560 + 8960) 62.8 -> 41.9
//   512 rows: 2560 x 2560 28.1 -> 22.6, 2560 x (2560 + 8960) 56.7 -> 49.1, 8960 x 2560 63.2 -> 45.4
#include <climits>
#include <cmath>
#include <cstring>
#include <type_traits>

#include "gemm_device.h"

#pragma clang fp contract(off)

namespace frhip {

constexpr int kQ8Stages = 4;  // K-steps of X in LDS: one multiplied, three in flight
constexpr int kQ8Codes = 3;   // K-steps of codes, per producer
constexpr int q8_max_blocks(int bm) { return bm == 128 ? 6 : 8; }  // of 32 columns: what 160 KB hold
constexpr int kQ8Producers = 8;
// A producer's codes, ry and my of a step; its rx and mx behind the slots.  Tiles of up to w blocks of 32 columns.
__host__ __device__ constexpr int q8_blocks_before(int p, int w) {
  const int r = 2 * w % kQ8Producers;
  return p * (2 * w / kQ8Producers) + (p < r ? p : r);
}
__host__ __device__ constexpr int q8_producer_at(int p, int w) { return kQ8Codes * (q8_blocks_before(p, w) * 1024 + p * 256) + p * 256; }
constexpr int q8_lds_bytes(int bm, int w) { return kQ8Stages * bm * 128 + 2 * w * 4096 + q8_producer_at(kQ8Producers, w); }
static_assert(128 * sums_pitch(6) * 4 <= q8_lds_bytes(128, 6) && 128 * sums_pitch(2) * 4 <= q8_lds_bytes(128, 2) &&
                  64 * sums_pitch(8) * 4 <= q8_lds_bytes(64, 8) && 64 * sums_pitch(2) * 4 <= q8_lds_bytes(64, 2), "the sums fit");
static_assert(q8_lds_bytes(128, q8_max_blocks(128)) <= 160 * 1024 && q8_lds_bytes(64, q8_max_blocks(64)) <= 160 * 1024, "LDS of a compute unit");

// few_dequant's two values, the same bits, in 8 instructions: a code in the low byte of a binary16 is the subnormal q 2^-24, which
// v_fma_mix_f32 reads as it is; c24 is c 2^24 and the product the same real number (c ry is far from fp32's subnormals).
template <int HI>
__device__ __forceinline__ h2 q8_dequant(uint32_t word, float c24, float mx, h2 ry, h2 my) {
  const uint32_t q = __builtin_amdgcn_perm(0u, word, HI ? 0x0c030c02u : 0x0c010c00u);
  float w0, w1;
  asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel_hi:[1,0,0]" : "=v"(w0) : "v"(q), "v"(mul_h<0>(c24, ry)), "v"(add_h<0>(mx, my)));
  asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(w1) : "v"(q), "v"(mul_h<1>(c24, ry)), "v"(add_h<1>(mx, my)));
  return (h2){(h1)w0, (h1)w1};
}

// NB: blocks of 16 columns of this wave (p, p + 8)
template <int BM, int NB>
__device__ __forceinline__ void q8_producer(const GemmSeg& sg, unsigned char* smem, int maxw, int p, int m0, int n0, int M, int K,
                                            int kbase, int nk, int lane) {
  constexpr int NA = BM / 8 / kQ8Producers, NC = NB + 1;  // loads of a step: 8 rows of X each; 16 columns each, and the scales
  const int N = sg.N, lr = lane >> 3, row16 = lane & 15, grp = lane >> 4;
  unsigned char* const bsm = smem + kQ8Stages * BM * 128;
  const int slot_bytes = (q8_blocks_before(p + 1, maxw) - q8_blocks_before(p, maxw)) * 1024 + 256;
  unsigned char* const own = bsm + 2 * maxw * 4096 + q8_producer_at(p, maxw);
  const unsigned lds0 = (unsigned)(size_t)((__attribute__((address_space(3))) unsigned char*)smem);
  const unsigned own_lds = lds0 + (unsigned)(own - smem);
  unsigned va[NA], vb[NB + 1];
#pragma unroll
  for (int i = 0; i < NA; i++) {  // rows past the matrix repeat its last row and are never stored
    const int g = p * NA + i;
    va[i] = (unsigned)(min(m0 + g * 8 + lr, M - 1) - m0) * (unsigned)(K * 2) + (((lane & 7) ^ lr ^ (g & 1)) * 16);
  }
#pragma unroll
  for (int t = 0; t < NB; t++) {
    const int col = min(n0 + (p + kQ8Producers * t) * 16 + (lane >> 2), N - 1) - n0;
    vb[t] = (unsigned)col * (unsigned)K + (((lane & 3) ^ (lane >> 4)) * 16);
  }
  const unsigned char* const abase = uniform_ptr(reinterpret_cast<const unsigned char*>(sg.A) + ((size_t)m0 * K + kbase) * 2);
  const unsigned char* const bbase = uniform_ptr(sg.B + (size_t)n0 * K + kbase);
  const h1* scale_k = (lane < 32 ? sg.ry : sg.my) + kbase + (lane & 31) * 2;  // lanes 0..31 ry, 32..63 my, two each
  {
    // rx (lanes 0..31) and mx of the wave's up to 64 columns, two a lane
    const int c = min(n0 + (p + kQ8Producers * ((lane & 31) >> 3)) * 16 + (lane & 7) * 2, N - 2);
    load_lds_dword((lane < 32 ? sg.rx : sg.mx) + c, own_lds + kQ8Codes * slot_bytes);
  }
  // Where the next loads come from and go to, in the order of their steps
  const unsigned char *ak = abase, *bk = bbase;
  unsigned a_lds = lds0 + p * (NA * 1024), c_lds = own_lds;
  const unsigned a_end = a_lds + kQ8Stages * (BM * 128), c_end = own_lds + kQ8Codes * slot_bytes;
  auto issue_a = [&] {
#pragma unroll
    for (int i = 0; i < NA; i++) load_lds_saddr(va[i], ak, a_lds + i * 1024);
    ak += 128;
    a_lds += BM * 128;
    a_lds = a_lds == a_end ? a_end - kQ8Stages * (BM * 128) : a_lds;
  };
  auto issue_codes = [&] {
#pragma unroll
    for (int t = 0; t < NB; t++) load_lds_saddr(vb[t], bk, c_lds + 256 + t * 1024);
    load_lds_dword(scale_k, c_lds);
    bk += 64;
    scale_k += 64;
    c_lds += slot_bytes;
    c_lds = c_lds == c_end ? own_lds : c_lds;
  };
  struct Step {  // a lane's codes of one step, and the scales of their rows
    u32x4 q[NB + 1];
    h8 ry[2], my[2];
  };
  const unsigned char* from = own;  // the slot that is read next
  auto read = [&](Step& r) {
    const unsigned char* st = from;
    from += slot_bytes;
    from = from == own + kQ8Codes * slot_bytes ? own : from;
#pragma unroll
    for (int h = 0; h < 2; h++) {
      r.ry[h] = *reinterpret_cast<const h8*>(st + grp * 32 + h * 16);
      r.my[h] = *reinterpret_cast<const h8*>(st + 128 + grp * 32 + h * 16);
    }
#pragma unroll
    for (int t = 0; t < NB; t++)
      r.q[t] = *reinterpret_cast<const u32x4*>(st + 256 + t * 1024 + row16 * 64 + ((grp ^ (row16 >> 2)) * 16));
  };
  // Loads complete in order, and they are issued in the order codes 0, codes 1, X 0, codes 2, X 1, codes 3, X 2, ...: what
  // has to have landed is told by how many of the loads behind it are outstanding.
  issue_codes();
  if (nk > 1) issue_codes();
  issue_a();
  if (nk > 2) issue_codes();
  if (nk > 1) issue_a();
  if (nk > 2) wait_loads<2 * NA + 2 * NC>();
  else if (nk > 1) wait_loads<2 * NA + NC>();
  else wait_loads<NA>();
  float c[NB + 1], m[NB + 1];
  const h1* cols = reinterpret_cast<const h1*>(own + kQ8Codes * slot_bytes);
#pragma unroll
  for (int t = 0; t < NB; t++) {
    c[t] = dequant_c(cols[t * 16 + row16]) * 16777216.0f;  // q8_dequant
    m[t] = (float)cols[64 + t * 16 + row16];
  }
  __builtin_amdgcn_s_setprio(2);  // the step waits for its producers: 1-5 % of a launch
  Step s0, s1;
  read(s0);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  if (nk > 3) issue_codes();
  unsigned char* bst = bsm;
  int b_step = maxw * 4096;  // to the other stage, and back
  // Step j between barriers j - 1 and j: behind barrier j - 1 step j - 2 has been read by all, and its slots may be written.
  auto step = [&](const Step& cur, Step& next, int behind, auto all) {
    constexpr bool ALL = decltype(all)::value;  // four steps or more behind this one
    if (ALL || behind >= 2) issue_a();
    if (ALL || behind >= 3) wait_loads<3 * NA + 2 * NC>();
    else if (behind == 2) wait_loads<3 * NA + NC>();
    else if (behind == 1) wait_loads<2 * NA>();
    if (ALL || behind >= 1) read(next);  // arrives while this step's codes are dequantised
#pragma unroll
    for (int t = 0; t < NB; t++)
#pragma unroll
      for (int h = 0; h < 2; h++) {
        const uint32_t w0 = cur.q[t][2 * h], w1 = cur.q[t][2 * h + 1];
        const h2 p0 = q8_dequant<0>(w0, c[t], m[t], cur.ry[h].s01, cur.my[h].s01);
        const h2 p1 = q8_dequant<1>(w0, c[t], m[t], cur.ry[h].s23, cur.my[h].s23);
        const h2 p2 = q8_dequant<0>(w1, c[t], m[t], cur.ry[h].s45, cur.my[h].s45);
        const h2 p3 = q8_dequant<1>(w1, c[t], m[t], cur.ry[h].s67, cur.my[h].s67);
        // 16 lanes write 16 columns' k-segment: free of bank conflicts
        *reinterpret_cast<h8*>(bst + ldw_at((p + kQ8Producers * t) * 16 + row16, 2 * grp + h)) = (h8){p0.x, p0.y, p1.x, p1.y, p2.x, p2.y, p3.x, p3.y};
      }
    bst += b_step;
    b_step = -b_step;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the step is written, the next one read
    if (ALL || behind >= 4) issue_codes();
    if (ALL || behind >= 4) wait_loads<2 * NA + 3 * NC>();  // X j has landed
    else if (behind == 3) wait_loads<2 * NA + 2 * NC>();
    else if (behind == 2) wait_loads<2 * NA + NC>();
    else if (behind == 1) wait_loads<NA>();
    else wait_loads<0>();
    step_barrier();  // barrier j
  };
  int behind = nk - 1;
  for (; behind >= 5; behind -= 2) {
    step(s0, s1, behind, std::true_type());
    step(s1, s0, behind - 1, std::true_type());
  }
  for (; behind >= 0; behind -= 2) {
    step(s0, s1, behind, std::false_type());
    if (behind >= 1) step(s1, s0, behind - 1, std::false_type());
  }
  step_barrier();
}

template <int BM, int NJ>
__device__ __forceinline__ void q8_mma(unsigned char* smem, int maxw, int brow0, int nk, int lane, int wm) {
  constexpr int MI = BM / 64, KG = MI * NJ >= 6 ? 2 : 4;
  const unsigned char* const bsm = smem + kQ8Stages * BM * 128;
  f16v acc[MI][NJ];
#pragma unroll
  for (int i = 0; i < MI; i++)
#pragma unroll
    for (int j = 0; j < NJ; j++)
#pragma unroll
      for (int v = 0; v < 16; v++) acc[i][j][v] = 0.f;
  for (int k = 0; k < nk; k++) {
    step_barrier();
    const unsigned char* as = smem + (k % kQ8Stages) * (BM * 128);
    const unsigned char* bs = bsm + (k & 1) * (maxw * 4096);
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
  }
  step_barrier();  // all fragments have been read
  const int pitch = sums_pitch(maxw);
#pragma unroll
  for (int i = 0; i < MI; i++) sums_to_lds(acc[i], reinterpret_cast<float*>(smem) + (wm * (BM / 2) + i * 32) * pitch + brow0, pitch, lane);
}

template <int BM>
__global__ __launch_bounds__(64 * (4 + kQ8Producers)) void gemm_q8_kernel(GemmArgs a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char q8_smem[];
  int bx, by;
  xcd_tile(bx, by);
  int sidx = 0;
#pragma unroll
  for (int i = 1; i < kGemmMaxSeg; i++) sidx += (i < a.nseg && bx >= a.tile_start[i]) ? 1 : 0;
  GemmSeg sg = a.seg[sidx];
  const int ti = bx - a.tile_start[sidx], base = a.vw_base[sidx], wide = a.vw_wide[sidx];
  const int width = base + (ti < wide ? 1 : 0);  // 32-column blocks of this tile
  const int n0 = (ti * base + (ti < wide ? ti : wide)) * 32, m0 = by * BM;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // slice z of ksplit takes K-steps [z base + min(z, rem), ...): the first rem slices one step more
  const int ksplit = a.ksplit > 1 ? a.ksplit : 1, kz = blockIdx.z, ksteps = a.K / kLdwBK, kper = ksteps / ksplit, krem = ksteps % ksplit;
  const int nk = kper + (kz < krem ? 1 : 0), kbase = (kz * kper + (kz < krem ? kz : krem)) * kLdwBK;
  if (wave >= 4) {
    const int p = wave - 4;
    static_assert(2 * q8_max_blocks(BM) <= 2 * kQ8Producers, "a producer has at most two blocks of 16 columns");
    switch (p < 2 * width ? (2 * width - p + kQ8Producers - 1) / kQ8Producers : 0) {
      case 0: q8_producer<BM, 0>(sg, q8_smem, a.vw_maxw, p, m0, n0, a.M, a.K, kbase, nk, lane); break;
      case 1: q8_producer<BM, 1>(sg, q8_smem, a.vw_maxw, p, m0, n0, a.M, a.K, kbase, nk, lane); break;
      default: q8_producer<BM, 2>(sg, q8_smem, a.vw_maxw, p, m0, n0, a.M, a.K, kbase, nk, lane); break;
    }
  } else {
    const int wm = wave >> 1, nj0 = (width + 1) >> 1, nj = (wave & 1) ? width - nj0 : nj0, brow0 = (wave & 1) ? nj0 * 32 : 0;
    switch (nj) {  // every wave passes the same barriers, whatever its width
      case 1: q8_mma<BM, 1>(q8_smem, a.vw_maxw, brow0, nk, lane, wm); break;
      case 2: q8_mma<BM, 2>(q8_smem, a.vw_maxw, brow0, nk, lane, wm); break;
      case 3: q8_mma<BM, 3>(q8_smem, a.vw_maxw, brow0, nk, lane, wm); break;
      default: q8_mma<BM, q8_max_blocks(BM) / 2>(q8_smem, a.vw_maxw, brow0, nk, lane, wm); break;
    }
  }
  __syncthreads();
  if (a.ksplit > 1) {  // this slice's sums go out as fp32; the epilogue proper follows in gemm_splitk_reduce_kernel
    sg.out = a.partial + (size_t)kz * a.partial_stride + a.part_off[sidx];
    sg.epi = G_STORE_F32;
  }
  finish_tile<BM, 64 * (4 + kQ8Producers)>(a, sg, reinterpret_cast<const float*>(q8_smem), sums_pitch(a.vw_maxw), width, m0, n0, a.M, sg.N);
}

// What a launch of such tiles is expected to take, us: fitted to 1793 measured ones (13 to 1536 rows, widths 1024 to 4096, the
// products of a layer, weights from memory; 7 % rms, the tile chosen by it 0.6 % slower than the best of 11).  Per round a fixed
// part and its K-steps, and no faster than the codes arrive; slices of K and their reduction launch.
static double q8_us(const GemmArgs& a, int bm, int rounds, int w) {
  const int S = a.ksplit > 1 ? a.ksplit : 1, steps = (a.K / kLdwBK + S - 1) / S;
  double cols = 0;
  for (int s = 0; s < a.nseg; s++) cols += a.seg[s].N;
  const double x = rounds * (bm == 128 ? 3.17 + 0.102 * w + steps * (0.194 + 0.120 * w) : 2.41 + 0.261 * w + steps * (0.181 + 0.085 * w));
  const double y = cols * a.K / 3.44e6;
  return 4.2 + sqrt(sqrt(x * x * x * x + y * y * y * y)) + (S > 1 ? 1.6 + S * a.M * cols * 8 / 4.2e6 : 0);
}

TilePlan plan_q8(const GemmArgs& args, int cus) {
  TilePlan best;
  const int S = args.ksplit > 1 ? args.ksplit : 1;
  if ((size_t)args.K * 2 * 128 > 0xffffffffull) return best;  // 32-bit byte offsets within a tile
  for (int s = 0; s < args.nseg; s++)
    if (args.seg[s].N % 16 != 0) return best;
  for (int bm : {128, 64}) {
    const int strips = (args.M + bm - 1) / bm;
    for (int w = q8_max_blocks(bm); w >= 2; w--) {
      // as few tiles as this width allows, then as many as their rounds hold
      long need = 0;
      for (int s = 0; s < args.nseg; s++) need += ((args.seg[s].N + 31) / 32 + w - 1) / w;
      const int rounds = (int)((need * strips * S + cus - 1) / cus);
      TilePlan p;
      p.a = args;
      auto dealt = [&](long tiles) {  // the MFMA waves take two blocks or more of a tile
        if (!deal_tiles(p.a, (int)tiles) || p.a.vw_maxw > w) return false;
        for (int s = 0; s < args.nseg; s++)
          if (p.a.vw_base[s] < 2) return false;
        return true;
      };
      if (!dealt((long)rounds * cus / ((long)strips * S)) && !dealt(need)) continue;
      p.us = q8_us(args, bm, rounds, p.a.vw_maxw);
      p.rows = bm;
      p.rounds = rounds;
      p.grid = dim3(p.a.tile_start[p.a.nseg], strips, S);
      if (!best.rows || p.us < best.us) best = p;
    }
  }
  return best;
}

// codes are loaded 16 bytes at a time, rows' and columns' scales 4
bool q8_takes(const GemmArgs& a) {
  uintptr_t v16 = 0, v4 = 0;
  for (int s = 0; s < a.nseg; s++) {
    v16 |= reinterpret_cast<uintptr_t>(a.seg[s].A) | reinterpret_cast<uintptr_t>(a.seg[s].B);
    for (const h1* p : {a.seg[s].mx, a.seg[s].rx, a.seg[s].my, a.seg[s].ry}) v4 |= reinterpret_cast<uintptr_t>(p);
  }
  return (v16 & 15) == 0 && (v4 & 3) == 0;
}

int launch_gemm_q8(const TilePlan& p, hipStream_t st, const char* what) {
  static const bool raised = [] {
    for (const void* f : {reinterpret_cast<const void*>(&gemm_q8_kernel<128>), reinterpret_cast<const void*>(&gemm_q8_kernel<64>)})
      (void)hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    return true;
  }();
  (void)raised;
  const size_t lds = q8_lds_bytes(p.rows, p.a.vw_maxw);
  if (p.rows == 128)
    hipLaunchKernelGGL(gemm_q8_kernel<128>, p.grid, dim3(64 * (4 + kQ8Producers)), lds, st, p.a);
  else
    hipLaunchKernelGGL(gemm_q8_kernel<64>, p.grid, dim3(64 * (4 + kQ8Producers)), lds, st, p.a);
  return check_launch(what);
}

}  // namespace frhip
