// Argument structures of the MFMA GEMM shared by gemm.hip and seq.hip.
#pragma once

#include <cstddef>

#include "device_utils.h"
#include "frhip_internal.h"

namespace frhip {

constexpr int kGemmMaxSeg = 4;

enum GemmEpi : int {
  G_STORE_F16 = 0,
  G_STORE_F32 = 1,
  G_SIGMOID = 2,    // half(sigmoid(half(acc)))                        ffn_seq.cu:78-79, att.cu:203
  G_RELU2 = 3,      // relu(half(acc))^2                               ffn_seq.cu:80-81
  G_SILU = 4,       // silu(half(acc))                                 att_seq.cu:394-395
  G_RESIDUAL = 5,   // x + half(acc)                                   att_seq.cu:412-415
  G_FFN_OUT = 6     // fma(half(acc), r, x) [/ 2]                      ffn_seq.cu:82-85, model_forward_seq.cpp:163-165
};

struct GemmSeg {
  const h1* A;                       // [M][K]
  const unsigned char* B;            // [N][K] binary16 or uint8
  const h1 *mx, *rx, *my, *ry;       // uint8 only
  void* out;                         // [M][N]
  int N, epi;
};

struct GemmArgs {
  int M, K, nseg;
  // The sums over K stay in the order of the tiled forms (contiguous slices), at any number of rows: no gemm_few_kernel.  For
  // RWKV-5: from an empty state the group normalisation leaves of a head's first token only the sign of sum r u k, so where
  // that sum is near zero its last bits decide the logits.  With gemm_few_kernel's order, as good against float64 product by
  // product, the logits of 12 layers of 2560 moved by 5 % of their norm after a prompt of 16 tokens (4 tokens: 15 %).
  bool tiled_sums;
  int tile_start[kGemmMaxSeg + 1];  // first N-tile of each segment
  size_t part_off[kGemmMaxSeg + 1]; // split launches: where each segment's [M][N] block starts within a slice of `partial` (floats); [nseg] = all
  // tiles of a width chosen per launch: a segment's are vw_base (the first vw_wide of them vw_base + 1) blocks of 32 columns wide
  int vw_base[kGemmMaxSeg], vw_wide[kGemmMaxSeg], vw_maxw;
  int few_strips;  // gemm_few_kernel: strips of rows
  // A segment, and ksplit with all behind it, are one 64-byte line each of the kernel's arguments, counted from their beginning.  Over two,
  // 8 bytes earlier, a launch of gemm_ring_kernel took 0.2 us longer (1024 x 8192 x 2048 in two slices 37.84 -> 38.05, 77 rows in
  // slices 11.95 -> 12.2), the reduction launch of 1024 rows 0.25 (6.04 -> 6.28).
  alignas(16) GemmSeg seg[kGemmMaxSeg];
  // split K (ksplit >= 2; gemm_ring_kernel and gemm_q8_kernel): slice z of ksplit accumulates its K-steps of segment s into
  // partial + z * partial_stride + part_off[s] as fp32 [M][N]; gemm_splitk_reduce_kernel adds the slices and applies the epilogues
  int ksplit;
  float* partial;
  size_t partial_stride;
  const h1* res_x;  // [M][N] G_RESIDUAL, G_FFN_OUT
  const h1* res_r;  // [M][N] G_FFN_OUT
  int div2;
};
static_assert(sizeof(GemmSeg) == 64 && offsetof(GemmArgs, seg) % 64 == 0 && offsetof(GemmArgs, ksplit) / 64 == offsetof(GemmArgs, div2) / 64, "one line each");

// dq: optional scratch, 2 bytes per weight of the launch.  With it, uint8 weights of a launch with at least
// kDequantRows rows are expanded once to binary16 (the standalone dequantisation: the same bits as the
// in-kernel one) and the launch takes the binary16 kernel, unless it is one of gemm_few_kernel or is expected to be quicker as
// one of gemm_q8_kernel: those dequantise the codes themselves.
// partial: optional fp32 scratch of max_split slices of partial_stride floats (>= M * N each) for splitting K.
// few_rows: optional fp32 scratch of few_rows_floats floats; with it a launch of so few rows that 64 x 128 tiles leave
// at least half of the compute units idle is split over K across the idle units, whole or product by product.
constexpr size_t kFewRowsFloats = (size_t)512 * 64 * 128;  // two 64 x 128 tiles per compute unit of a 256-unit part
constexpr int kFewRowsMax = 360;                          // rows up to which the seq operators carry that scratch
constexpr int kSeqMaxSplit = 4;                           // slices of the [T][C] buffers that ffn value is given as `partial`
int launch_gemm(GemmArgs& a, bool u8, hipStream_t st, const char* what, void* dq = nullptr, float* partial = nullptr,
                size_t partial_stride = 0, int max_split = 0, float* few_rows = nullptr, size_t few_rows_floats = 0);
// Products of a few rows in one launch, K split over the waves of a workgroup (gemm_few.hip).  plan_few: the tile that is
// expected to be the quickest and its us; mt = 0: not a launch of this form.  It depends on the sizes alone, not on the
// weight type, so that a uint8 weight and its binary16 image take the same sums.  few_takes: the addresses allow it.
// Up to the rows that the times were fitted to; within them they decide.  Of 84 binary16 products of 384 to 512 rows (widths 768
// to 5120) they send 26 here, all of them the quicker for it (512 x 2048 x 2048: 14.9 us on tiles of 64 rows, 10.2 here; 512 x
// 3072 x 768: 20.6 and 9.0), and leave two behind that would have gained 5 % at most; a prompt of 512 tokens, 12 layers of 768:
// 1050 -> 794 us, 2048: 1714 -> 1647, 5120 (2 layers): 1118 -> 1126.
constexpr int kFewKernelRows = 512;
struct FewPlan {
  int mt = 0, nt = 0;  // blocks of 16 rows and 16 columns of a workgroup
  double us = 0;
};
FewPlan plan_few(const GemmArgs& a, int cus);
bool few_takes(const GemmArgs& a, bool u8);
int launch_gemm_few(const GemmArgs& a, const FewPlan& p, bool u8, hipStream_t st, const char* what);
// Deals `tiles` workgroups of a strip of rows to the segments by their columns: tile_start, vw_base, vw_wide, vw_maxw.  False: too few.
bool deal_tiles(GemmArgs& a, int tiles);
// A launch of tiles of `rows` rows and widths of its own per segment: with the cut that is expected to be the quickest; rows = 0: not
// a launch of the form.  a.ksplit, partial and part_off: slices of K, whose sums go there as fp32.
struct TilePlan {
  int rows = 0, rounds = 0;
  double us = 0;
  dim3 grid;
  GemmArgs a;
};
// binary16 weights, four loading waves (gemm_ring.hip)
TilePlan plan_ring(const GemmArgs& a, int cus);
int launch_gemm_ring(const TilePlan& p, hipStream_t st, const char* what);
// uint8 weights whose codes are dequantised on their way into LDS (gemm_q8.hip)
TilePlan plan_q8(const GemmArgs& a, int cus);
bool q8_takes(const GemmArgs& a);
int launch_gemm_q8(const TilePlan& p, hipStream_t st, const char* what);
constexpr int kDequantRows = FRHIP_SEQ_EXPAND_ROWS;
// uint8 [N][K] -> binary16 [N][K] with the frozen formula (ops.hip)
int dequant_u8_async(const unsigned char* q, const h1* mx, const h1* rx, const h1* my, const h1* ry, h1* dst, int K, int N,
                     hipStream_t st);
// the same for the nseg matrices of a grouped product (same K), one launch where the shapes allow it
int dequant_u8_group_async(int nseg, const unsigned char* const* q, const h1* const* mx, const h1* const* rx, const h1* const* my,
                           const h1* const* ry, h1* const* dst, int K, const int* N, hipStream_t st);
void gemm_add_seg(GemmArgs& a, const void* A, const frhip_weight* w, void* out, int epi);

}  // namespace frhip
