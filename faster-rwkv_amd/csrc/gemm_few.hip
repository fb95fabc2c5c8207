// Products of a few rows (short prompts, short turns of a conversation) on the MFMA units: one launch, K split over the
// waves of a workgroup.
//
// With a handful of rows a product is its weights once from memory, and what counts is that all compute units pull at
// them.  A workgroup here owns NT x 16 columns and MT x 16 rows and its waves take the K-steps of 64 in turn (wave w the
// steps w, w + waves, ...), each through a ring of its own in LDS: tiles go global -> LDS directly
// (global_load_lds_dwordx4), a wave waits for nothing but its own loads, and there is no barrier until the waves' sums
// meet.  They are added in wave order, the epilogue is applied and the outputs are stored: no partial sums in memory and no
// second launch.
//
// The weights are the first operand of v_mfma_f32_16x16x32_f16 and the rows of X the second, so that a lane's four
// accumulators are four consecutive columns of one row of Y.  Lane group g (16 lanes) holds k = 16 g .. 16 g + 15 of a
// step, 8 per MFMA: the 16 codes that a lane reads of a uint8 weight.  uint8 codes go to LDS as they are and are
// dequantised by the lane that multiplies them, with the formula of the standalone dequantisation; the order of the sums
// depends on K and the number of waves only, so a uint8 weight and its binary16 image give the same bits.
//
// What bounds it: a compute unit has about 64 KB of loads in flight, some 50 GB/s from memory, and every workgroup reads all
// rows of X besides its columns; uint8 adds 4.5 vector instructions per code.  Per product in a chain of dependent launches, us,
// the forms with partial sums in memory and a reduction launch -> this one:
//   13 rows, uint8:    2048 x (3 x 2048) 17.1 -> 7.8, 2048 x 2048 11.4 -> 5.8, 2048 x (2048 + 8192) 22.0 -> 9.8, 8192 x 2048 17.9 -> 10.9
//   77 rows, binary16: 2048 x (3 x 2048) 17.3 -> 13.0, 2048 x 2048 11.5 -> 6.3, 2048 x (2048 + 8192) 29.5 -> 16.6
//   300 rows, binary16: 4096 x 4096 35.1 -> 23.1;  130 rows, uint8: 2560 x (4 x 2560) 71.7 -> 22.9
#include <climits>
#include <cmath>

#include "gemm_device.h"

#pragma clang fp contract(off)

namespace frhip {

constexpr int kFewScaleBytes = 512;  // uint8: rx, then mx of up to 128 columns, behind a wave's ring
// The waves decide the order of the sums: the same for both weight types.  The ring is as deep as 160 KB of LDS allow, up to
// four steps.
constexpr int few_waves(int mt, int nt) { return mt + nt <= 5 ? 8 : 4; }
constexpr int few_stage_bytes(int mt, int nt, bool u8) { return mt * 2048 + (u8 ? nt * 1024 + 256 : nt * 2048); }
constexpr int few_stages(int mt, int nt, bool u8) {
  const int s = (160 * 1024 / few_waves(mt, nt) - (u8 ? kFewScaleBytes : 0)) / few_stage_bytes(mt, nt, u8);
  return s > 4 ? 4 : s;
}
constexpr int few_wave_bytes(int mt, int nt, bool u8) { return few_stages(mt, nt, u8) * few_stage_bytes(mt, nt, u8) + (u8 ? kFewScaleBytes : 0); }

// A tile of 16 rows x 64 binary16: rows of 128 bytes, k-segment q (8 halves) of row r in slot q ^ (r % 8) ^ (r / 8)
// (the layout of the tiled kernels: fragment reads of 16 rows are free of bank conflicts)
__device__ __forceinline__ int few_at(int r, int q) { return r * 128 + ((q ^ (r & 7) ^ (r >> 3)) * 16); }

template <int MT, int NT, bool U8>
__global__ __launch_bounds__(few_waves(MT, NT) * 64) void gemm_few_kernel(GemmArgs a) {
  constexpr int NW = few_waves(MT, NT), S = few_stages(MT, NT, U8), kStage = few_stage_bytes(MT, NT, U8);
  constexpr int kBOff = MT * 2048, kScaleOff = kBOff + NT * (U8 ? 1024 : 2048);
  constexpr int kPer = 2 * MT + (U8 ? NT + 1 : 2 * NT);  // load instructions per step
  static_assert(S >= 2 && (S - 1) * kPer <= 63, "the wait counter's range");
  extern __shared__ __attribute__((aligned(16))) unsigned char few_smem[];

  // tiles are dealt to the XCDs in contiguous runs, strips of rows fastest: the strips that share weights share an L2
  const int n = gridDim.x, strips = a.few_strips, lin = blockIdx.x, xcd = lin & 7;
  const int id = xcd * (n >> 3) + min(xcd, n & 7) + (lin >> 3);
  const int tile = id / strips, strip = id - tile * strips;
  int sidx = 0;
#pragma unroll
  for (int i = 1; i < kGemmMaxSeg; i++) sidx += (i < a.nseg && tile >= a.tile_start[i]) ? 1 : 0;
  const GemmSeg& sg = a.seg[sidx];
  const int M = a.M, K = a.K, N = sg.N;
  const int n0 = (tile - a.tile_start[sidx]) * (NT * 16), m0 = strip * (MT * 16);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int row16 = lane & 15, grp = lane >> 4;

  unsigned char* const ring = few_smem + wave * few_wave_bytes(MT, NT, U8);
  const unsigned ring_lds = (unsigned)(size_t)((__attribute__((address_space(3))) unsigned char*)few_smem) + wave * few_wave_bytes(MT, NT, U8);

  // ---- this wave's loads; rows past the matrix repeat its last row and are never stored ----
  const int lr = lane >> 3;
  unsigned va[2 * MT], vb[U8 ? NT : 2 * NT];
#pragma unroll
  for (int b = 0; b < 2 * MT; b++) {
    const int row = min(m0 + b * 8 + lr, M - 1) - m0;
    va[b] = (unsigned)row * (unsigned)(K * 2) + (((lane & 7) ^ lr ^ (b & 1)) * 16);
  }
  if constexpr (U8) {
#pragma unroll
    for (int b = 0; b < NT; b++) {
      const int col = min(n0 + b * 16 + (lane >> 2), N - 1) - n0;
      vb[b] = (unsigned)col * (unsigned)K + (((lane & 3) ^ (lane >> 4)) * 16);
    }
  } else {
#pragma unroll
    for (int b = 0; b < 2 * NT; b++) {
      const int col = min(n0 + b * 8 + lr, N - 1) - n0;
      vb[b] = (unsigned)col * (unsigned)(K * 2) + (((lane & 7) ^ lr ^ (b & 1)) * 16);
    }
  }
  const unsigned char* const abase = uniform_ptr(reinterpret_cast<const unsigned char*>(sg.A) + (size_t)m0 * K * 2);
  const unsigned char* const bbase = uniform_ptr(sg.B + (size_t)n0 * K * (U8 ? 1 : 2));
  const h1* scale_k = nullptr;  // uint8: lanes 0..31 bring ry, lanes 32..63 my, two values each
  if constexpr (U8) scale_k = (lane < 32 ? sg.ry : sg.my) + (lane & 31) * 2;
  const int nk = K >> 6, mine = wave < nk ? (nk - wave + NW - 1) / NW : 0;
  auto issue = [&](int i) {
    const int k0 = (wave + i * NW) * 64;
    const unsigned st = ring_lds + (i % S) * kStage;
    const unsigned char* ak = abase + (size_t)k0 * 2;
    const unsigned char* bk = bbase + (size_t)k0 * (U8 ? 1 : 2);
#pragma unroll
    for (int b = 0; b < (U8 ? NT : 2 * NT); b++) load_lds_saddr(vb[b], bk, st + kBOff + b * 1024);
#pragma unroll
    for (int b = 0; b < 2 * MT; b++) load_lds_saddr(va[b], ak, st + b * 1024);
    if constexpr (U8) load_lds_dword(scale_k + k0, st + kScaleOff);
  };
  if constexpr (U8) {  // rx, mx of this workgroup's columns, two a lane
    static_assert(NT * 16 <= 128, "two columns a lane");
    const int c = min(n0 + lane * 2, N - 2);
    load_lds_dword(sg.rx + c, ring_lds + S * kStage);
    load_lds_dword(sg.mx + c, ring_lds + S * kStage + 256);
  }
#pragma unroll
  for (int i = 0; i < S; i++)
    if (i < mine) issue(i);

  f4v acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; i++)
#pragma unroll
    for (int j = 0; j < NT; j++) acc[i][j] = (f4v){0.f, 0.f, 0.f, 0.f};
  // loads complete in order: a step has landed when at most the loads of the steps behind it are outstanding
  auto landed = [&](int behind) {
    if (behind >= S - 1) wait_loads<(S - 1) * kPer>();
    else if (S > 3 && behind == 2) wait_loads<(S > 3 ? 2 : 0) * kPer>();
    else if (S > 2 && behind == 1) wait_loads<(S > 2 ? 1 : 0) * kPer>();
    else wait_loads<0>();
  };
  float c[NT], m[NT];  // uint8: rx / 255 and mx of the lane's columns
  if constexpr (U8) {
    landed(mine - 1);
#pragma unroll
    for (int t = 0; t < NT; t++) {
      const h1* sc = reinterpret_cast<const h1*>(ring + S * kStage) + t * 16 + row16;
      c[t] = dequant_c(sc[0]);
      m[t] = (float)sc[128];
    }
  }
  for (int i = 0; i < mine; i++) {
    landed(mine - 1 - i);
    const unsigned char* st = ring + (i % S) * kStage;
    h8 xa[2][MT], wb[2][NT];
#pragma unroll
    for (int t = 0; t < MT; t++)
#pragma unroll
      for (int h = 0; h < 2; h++) xa[h][t] = *reinterpret_cast<const h8*>(st + t * 2048 + few_at(row16, 2 * grp + h));
    if constexpr (U8) {
      u32x4 q[NT];
      h8 ry[2], my[2];
#pragma unroll
      for (int h = 0; h < 2; h++) {
        ry[h] = *reinterpret_cast<const h8*>(st + kScaleOff + grp * 32 + h * 16);
        my[h] = *reinterpret_cast<const h8*>(st + kScaleOff + 128 + grp * 32 + h * 16);
      }
#pragma unroll
      for (int t = 0; t < NT; t++)
        q[t] = *reinterpret_cast<const u32x4*>(st + kBOff + t * 1024 + row16 * 64 + ((grp ^ (row16 >> 2)) * 16));
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the slot has been read
      if (i + S < mine) issue(i + S);
#pragma unroll
      for (int t = 0; t < NT; t++)
#pragma unroll
        for (int h = 0; h < 2; h++) {
          const uint32_t w0 = q[t][2 * h], w1 = q[t][2 * h + 1];
          const h2 p0 = few_dequant<0>(w0, c[t], m[t], ry[h].s01, my[h].s01);
          const h2 p1 = few_dequant<1>(w0, c[t], m[t], ry[h].s23, my[h].s23);
          const h2 p2 = few_dequant<0>(w1, c[t], m[t], ry[h].s45, my[h].s45);
          const h2 p3 = few_dequant<1>(w1, c[t], m[t], ry[h].s67, my[h].s67);
          wb[h][t] = (h8){p0.x, p0.y, p1.x, p1.y, p2.x, p2.y, p3.x, p3.y};
        }
    } else {
#pragma unroll
      for (int t = 0; t < NT; t++)
#pragma unroll
        for (int h = 0; h < 2; h++) wb[h][t] = *reinterpret_cast<const h8*>(st + kBOff + t * 2048 + few_at(row16, 2 * grp + h));
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      if (i + S < mine) issue(i + S);
    }
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
      for (int t = 0; t < MT; t++)
#pragma unroll
        for (int j = 0; j < NT; j++) acc[t][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wb[h][j], xa[h][t], acc[t][j], 0, 0, 0);
  }

  // ---- the waves' sums meet: each leaves its tiles in its own ring (a tile is 1 KB; MT NT <= 2 S (MT + NT / 2) of them fit) ----
  static_assert(MT * NT * 1024 <= S * kStage, "the sums fit the ring");
#pragma unroll
  for (int t = 0; t < MT; t++)
#pragma unroll
    for (int j = 0; j < NT; j++) *reinterpret_cast<f4v*>(ring + ((t * NT + j) * 64 + lane) * 16) = acc[t][j];
  __syncthreads();
  for (int t = wave; t < MT * NT; t += NW) {
    const int i = t / NT, j = t - i * NT;
    const int r0 = m0 + i * 16, c0 = n0 + j * 16;
    if (r0 >= M || c0 >= N) continue;
    const int row = r0 + row16;
    const bool ok = row < M;
    const size_t o = (size_t)(ok ? row : M - 1) * N + c0 + grp * 4;
    h4 x = {}, r = {};
    if (sg.epi == G_RESIDUAL || sg.epi == G_FFN_OUT) x = *reinterpret_cast<const h4*>(a.res_x + o);
    if (sg.epi == G_FFN_OUT) r = *reinterpret_cast<const h4*>(a.res_r + o);
    f4v s = *reinterpret_cast<const f4v*>(few_smem + (t * 64 + lane) * 16);
#pragma unroll
    for (int w = 1; w < NW; w++) {
      const f4v p = *reinterpret_cast<const f4v*>(few_smem + w * few_wave_bytes(MT, NT, U8) + (t * 64 + lane) * 16);
#pragma unroll
      for (int v = 0; v < 4; v++) s[v] += p[v];
    }
    if (sg.epi == G_STORE_F32) {
      if (ok) *reinterpret_cast<f4v*>(static_cast<float*>(sg.out) + o) = s;
      continue;
    }
    h1 y[4];
    switch (sg.epi) {
      case G_SIGMOID: sigmoid_batch(s, y, ok ? 0xfu : 0u); break;
      case G_SILU: silu_batch(s, y, ok ? 0xfu : 0u); break;
      case G_RELU2:
#pragma unroll
        for (int v = 0; v < 4; v++) {
          const h1 q = (h1)s[v];
          y[v] = (q > (h1)0.0f) ? (q * q) : (h1)0.0f;
        }
        break;
      case G_RESIDUAL:
#pragma unroll
        for (int v = 0; v < 4; v++) y[v] = x[v] + (h1)s[v];
        break;
      case G_FFN_OUT:
#pragma unroll
        for (int v = 0; v < 4; v++) {
          h1 q = __builtin_fmaf16((h1)s[v], r[v], x[v]);
          if (a.div2) q = q / (h1)2.0f;
          y[v] = q;
        }
        break;
      default:
#pragma unroll
        for (int v = 0; v < 4; v++) y[v] = (h1)s[v];
        break;
    }
    if (ok) *reinterpret_cast<h4*>(static_cast<h1*>(sg.out) + o) = (h4){y[0], y[1], y[2], y[3]};
  }
}

template <int MT, int NT, bool U8>
static void few_launch(int grid, hipStream_t st, const GemmArgs& a) {
  constexpr size_t lds = (size_t)few_waves(MT, NT) * few_wave_bytes(MT, NT, U8);
  static_assert(lds <= 160 * 1024, "LDS of a compute unit");
  static const bool raised = [] {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_few_kernel<MT, NT, U8>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    return true;
  }();
  (void)raised;
  hipLaunchKernelGGL((gemm_few_kernel<MT, NT, U8>), dim3(grid), dim3(few_waves(MT, NT) * 64), lds, st, a);
}

// The tiles (16-row by 16-column blocks of a workgroup) that are built: within 2 % of the best of all 30 on 1360 measured products.
#define FR_FEW_TILES(X) \
  X(1, 1) X(1, 2) X(1, 3) X(1, 4) X(2, 1) X(2, 2) X(2, 3) X(2, 4) X(3, 1) X(3, 2) X(3, 3) X(3, 4) X(3, 5) \
  X(4, 2) X(4, 3) X(4, 4) X(5, 2) X(5, 3) X(5, 4) X(5, 5) X(6, 4)

// What a launch with these tiles is expected to take, us; fitted to the binary16 ones of those products (2 to 512 rows, K 768 to
// 20480, N 768 to 20480, weights from memory; 9 % rms, as on 476 others of 4 to 512 rows since, whose worst region, single narrow
// products of 17 to 64 rows, takes 13 % longer than expected).  Per round over the compute units: a fixed part that grows with
// the sums to be merged, then the K-steps beyond those that the rings hold at the start, each as long as its loads and
// products; and no faster than the weights arrive, which several strips of rows read more than once.
static double few_us(const GemmArgs& a, int mt, int nt, int cus) {
  long tiles = 0;
  double bytes = 0;
  for (int s = 0; s < a.nseg; s++) {
    tiles += (a.seg[s].N / 16 + nt - 1) / nt;
    bytes += 2.0 * a.seg[s].N * a.K;
  }
  const int strips = (a.M + 16 * mt - 1) / (16 * mt), nk = a.K / 64, nw = few_waves(mt, nt);
  const double rounds = (double)((tiles * strips + cus - 1) / cus), load = tiles * strips / (rounds * cus);
  const int held = nw * few_stages(mt, nt, false);
  double fixed, steps, bw;
  if (nw == 8) {
    fixed = 1.41 + 0.187 * mt * nt;
    steps = (nk - 0.59 * held > 0.3 * nk ? nk - 0.59 * held : 0.3 * nk) * (26.2 + 20.3 * mt + 24.6 * nt) * 1e-3;
    bw = 5.09e6 / (1 + 0.215 * (strips - 1));
  } else {
    fixed = 1.5 + 0.218 * mt * nt;
    steps = (nk - held > 0.3 * nk ? nk - held : 0.3 * nk) * (107 + 0.9 * mt + 6.54 * mt * nt) * 1e-3 * (0.883 + 0.117 * load);
    bw = 4.09e6 / (1 + 0.148 * (strips - 1));
  }
  const double x = rounds * steps, y = bytes / bw;
  return 1.4 + rounds * fixed + sqrt(sqrt(x * x * x * x + y * y * y * y));
}

FewPlan plan_few(const GemmArgs& a, int cus) {
  FewPlan p;
  if (a.M > kFewKernelRows || (size_t)a.K * 2 * 16 * 6 > 0xffffffffull) return p;  // 32-bit byte offsets within a tile
  for (int s = 0; s < a.nseg; s++)
    if (a.seg[s].N % 16 != 0) return p;
  const int blocks = (a.M + 15) / 16;
#define FR_FEW_TRY(MT_, NT_)                        \
  if (MT_ <= blocks) {                              \
    const double us = few_us(a, MT_, NT_, cus);     \
    if (!p.mt || us < p.us) p.mt = MT_, p.nt = NT_, p.us = us; \
  }
  FR_FEW_TILES(FR_FEW_TRY)
#undef FR_FEW_TRY
  return p;
}

bool few_takes(const GemmArgs& a, bool u8) {
  uintptr_t v16 = 0, v8 = reinterpret_cast<uintptr_t>(a.res_x) | reinterpret_cast<uintptr_t>(a.res_r), v4 = 0;
  for (int s = 0; s < a.nseg; s++) {
    const GemmSeg& g = a.seg[s];
    v16 |= reinterpret_cast<uintptr_t>(g.A) | reinterpret_cast<uintptr_t>(g.B);
    (g.epi == G_STORE_F32 ? v16 : v8) |= reinterpret_cast<uintptr_t>(g.out);
    if (u8)
      for (const h1* p : {g.mx, g.rx, g.my, g.ry}) v4 |= reinterpret_cast<uintptr_t>(p);
  }
  return (v16 & 15) == 0 && (v8 & 7) == 0 && (v4 & 3) == 0;
}

int launch_gemm_few(const GemmArgs& args, const FewPlan& p, bool u8, hipStream_t st, const char* what) {
  GemmArgs a = args;
  int tiles = 0;
  for (int s = 0; s < a.nseg; s++) {
    a.tile_start[s] = tiles;
    tiles += (a.seg[s].N / 16 + p.nt - 1) / p.nt;
  }
  for (int s = a.nseg; s <= kGemmMaxSeg; s++) a.tile_start[s] = INT_MAX;
  a.few_strips = (a.M + 16 * p.mt - 1) / (16 * p.mt);
  const int grid = tiles * a.few_strips;
#define FR_FEW_GO(MT_, NT_)                                             \
  if (p.mt == MT_ && p.nt == NT_) {                                     \
    if (u8) few_launch<MT_, NT_, true>(grid, st, a); else few_launch<MT_, NT_, false>(grid, st, a); \
  }
  FR_FEW_TILES(FR_FEW_GO)
#undef FR_FEW_GO
  return check_launch(what);
}

}  // namespace frhip
