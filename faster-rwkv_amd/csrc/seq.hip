// Seq-mode (prompt) operators: layernorm + token shift + mix over T rows, the WKV scans of
// RWKV-4 and RWKV-5.2, and the att_seq / ffn_seq compositions around the MFMA GEMM.
//
// Both recurrences are linear in their state, so the scans run CHUNKED over time instead of
// as one serial loop of T steps on a handful of wavefronts (kernels/cuda/att_seq.cu:258-322
// runs 64 threads per head for T steps):
//   1. every chunk is scanned from an EMPTY state, all chunks in parallel -> local end states;
//   2. the local end states are turned into the true state at the start of every chunk
//      (state_in[c+1] = decay^len(state_in[c]) + local[c]): by doubling in LDS (RWKV-4, all in one
//      launch) or a short serial pass over the chunks (RWKV-5);
//   3. every chunk is scanned again from its true start state, all chunks in parallel,
//      producing the outputs; the last chunk leaves the final state.
// The arithmetic of pass 3 is the one-token recurrence (kernels/cuda/att.cu:30-62, :64-81);
// only the representation of the carried state differs from a serial scan, at fp32 rounding level.
#include <climits>
#include <cstring>
#include <type_traits>

#include "gemm.h"

#pragma clang fp contract(off)

namespace frhip {

// ---------------------------------------------------------------------------
// layernorm + token shift + mix for T rows: one workgroup (256 threads) per row.
//   xx_t = LN(x_t) ; sx_t = (t == 0) ? state : xx_{t-1} ; out_i[t] = mix(xx_t, sx_t, mix_i)
// (kernels/cuda/ffn_seq.cu:70-77, att_seq.cu:379-389).  LN(x_{t-1}) is recomputed by the
// workgroup of row t, which saves a [T, C] round trip.  Row T-1 also writes xx_{T-1}, the
// new shift state.
// ---------------------------------------------------------------------------
struct LnMixSeq {
  int T, C, nmix;
  const h1 *x, *state, *ln_w, *ln_b;
  const h1* mix[4];
  h1* out[4];
  h1* xx_last;
};

__device__ __forceinline__ void ln_row_to_lds(const h1* xr, const h1* g, const h1* b, int C, h1* dst, float* red) {
  float s = 0.f;
  for (int i = threadIdx.x; i < C; i += 256) s += (float)xr[i];
  const float mean = block_sum<4>(s, red) / (float)C;
  float q = 0.f;
  for (int i = threadIdx.x; i < C; i += 256) {
    float d = (float)xr[i] - mean;
    q += d * d;
  }
  float var = block_sum<4>(q, red) / (float)C;
  var = var > 0.f ? var : 0.f;
  const float inv = 1.0f / sqrtf(var + 1e-5f);
  for (int i = threadIdx.x; i < C; i += 256) {
    h1 n = (h1)(((float)xr[i] - mean) * inv);
    dst[i] = (n * g[i]) + b[i];
  }
}

__global__ __launch_bounds__(256) void ln_mix_seq_kernel(LnMixSeq a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  __shared__ float red[4];
  h1* cur = reinterpret_cast<h1*>(smem);
  h1* prev = cur + a.C;
  const int t = blockIdx.x, C = a.C;
  ln_row_to_lds(a.x + (size_t)t * C, a.ln_w, a.ln_b, C, cur, red);
  if (t == 0) {
    for (int i = threadIdx.x; i < C; i += 256) prev[i] = a.state[i];
  } else {
    ln_row_to_lds(a.x + (size_t)(t - 1) * C, a.ln_w, a.ln_b, C, prev, red);
  }
  __syncthreads();
  for (int i = threadIdx.x; i < C; i += 256) {
    const h1 xx = cur[i], sx = prev[i];
    for (int m = 0; m < a.nmix; m++) a.out[m][(size_t)t * C + i] = mix1(xx, sx, a.mix[m][i]);
    if (t == a.T - 1) a.xx_last[i] = xx;
  }
}

// The same for C % 8 == 0, C <= 8 * 256 * NG: a workgroup takes kLnRows consecutive rows plus the
// row before them (the token shift of its first row), every thread owns a group of 8 elements
// of every row in registers, all rows are loaded up front and their statistics reduced together
// (two barriers per workgroup), and the mixed rows leave as 16-byte stores.  The launch is a chain
// of one load, two reductions and one store per workgroup, so what counts is how many workgroups
// a compute unit has to overlap: at T = 1024, C = 2048 four rows per workgroup (one workgroup per
// CU, every row read 1.25 times) take 8.7 us, two 7.4 us, one (every row read twice) 7.0 us.
// For the same reason everything is requested at the start, the mixes too (one by one in the loop over the outputs each was a round
// trip of its own), and rows of more than 2048 elements have a thread per group: the first four waves take the sums of all of them,
// in the order of a thread with two groups, and each thread writes its own.  A launch is 0.7 us shorter for it (48 launches of a
// 77-token prompt of the 1.5B shape 2599 -> 2564 us, 13 tokens on a state 2626 -> 2546, 512 tokens of the 3B shape 3284 -> 3244).
constexpr int kLnRows = 1;

template <int NG, int NMIX>
__global__ __launch_bounds__(256 * NG) void ln_mix_rows_kernel(LnMixSeq a) {
  constexpr int NR = kLnRows + 1;  // row 0 is the row before the workgroup's first
  __shared__ float red[2][4][NR];
  const int C = a.C, ngrp = C >> 3;
  const int t0 = blockIdx.x * kLnRows;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, g = threadIdx.x;
  const bool own = g < ngrp, sums = NG == 1 || wv < 4, more = NG == 2 && sums && g + 256 < ngrp;
  const int gc = own ? g : 0, gm = more ? g + 256 : 0;
  h8 xr[NR], xm[NR], mx[NMIX];
#pragma unroll
  for (int r = 0; r < NR; r++) {
    int t = t0 - 1 + r;
    t = t < 0 ? 0 : (t < a.T ? t : a.T - 1);
    const h8* row = reinterpret_cast<const h8*>(a.x + (size_t)t * C);
    xr[r] = row[gc];
    if (NG == 2 && sums) xm[r] = row[gm];
  }
  const h8 gam = reinterpret_cast<const h8*>(a.ln_w)[gc], bet = reinterpret_cast<const h8*>(a.ln_b)[gc];
#pragma unroll
  for (int m = 0; m < NMIX; m++) mx[m] = reinterpret_cast<const h8*>(a.mix[m])[gc];
  h8 shift0;  // the shift state, used instead of LN(row -1) by the first workgroup
  if (t0 == 0) shift0 = reinterpret_cast<const h8*>(a.state)[gc];
  float mean[NR], inv[NR];
  {
    if (sums) {
#pragma unroll
      for (int r = 0; r < NR; r++) {
        float s = 0.f;
        if (own)
#pragma unroll
          for (int i = 0; i < 8; i++) s += (float)xr[r][i];
        if (NG == 2 && more)
#pragma unroll
          for (int i = 0; i < 8; i++) s += (float)xm[r][i];
        s = wave_sum(s);
        if (lane == 0) red[0][wv][r] = s;
      }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < NR; r++) mean[r] = (((red[0][0][r] + red[0][1][r]) + red[0][2][r]) + red[0][3][r]) / (float)C;
    if (sums) {
#pragma unroll
      for (int r = 0; r < NR; r++) {
        float q = 0.f;
        if (own)
#pragma unroll
          for (int i = 0; i < 8; i++) {
            const float d = (float)xr[r][i] - mean[r];
            q += d * d;
          }
        if (NG == 2 && more)
#pragma unroll
          for (int i = 0; i < 8; i++) {
            const float d = (float)xm[r][i] - mean[r];
            q += d * d;
          }
        q = wave_sum(q);
        if (lane == 0) red[1][wv][r] = q;
      }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < NR; r++) {
      float var = (((red[1][0][r] + red[1][1][r]) + red[1][2][r]) + red[1][3][r]) / (float)C;
      var = var > 0.f ? var : 0.f;
      inv[r] = 1.0f / sqrtf(var + 1e-5f);
    }
  }
  if (!own) return;
  h8 prev;
#pragma unroll
  for (int r = 0; r < NR; r++) {
    h8 xx;
#pragma unroll
    for (int i = 0; i < 8; i++) {  // kernels/cuda/layer_norm.cu:60-69: half, * gamma in half, + beta in half
      const h1 nrm = (h1)(((float)xr[r][i] - mean[r]) * inv[r]);
      xx[i] = (nrm * gam[i]) + bet[i];
    }
    if (r == 0) {
      prev = t0 == 0 ? shift0 : xx;
      continue;
    }
    const int t = t0 + r - 1;
    if (t < a.T) {
#pragma unroll
      for (int m = 0; m < NMIX; m++) {
        h8 o;
#pragma unroll
        for (int i = 0; i < 8; i++) o[i] = mix1(xx[i], prev[i], mx[m][i]);
        reinterpret_cast<h8*>(a.out[m] + (size_t)t * C)[g] = o;
      }
      if (t == a.T - 1) reinterpret_cast<h8*>(a.xx_last)[g] = xx;
    }
    prev = xx;
  }
}

template <int NMIX>
static void launch_ln_mix_rows(const LnMixSeq& a, int nwg, hipStream_t st) {
  const int ngrp = a.C >> 3;
  if (ngrp <= 256)
    hipLaunchKernelGGL((ln_mix_rows_kernel<1, NMIX>), dim3(nwg), dim3(256), 0, st, a);
  else
    hipLaunchKernelGGL((ln_mix_rows_kernel<2, NMIX>), dim3(nwg), dim3((ngrp + 63) / 64 * 64), 0, st, a);
}

// Rows beyond 4096 elements, up to 256 * NE: the row and the one before it stay in registers too, but
// thread t owns elements t, t + 256, ... as in ln_mix_seq_kernel, and every sum is taken in that kernel's order: the same
// bits as the general form, at any address.  (Groups of 8 consecutive elements, as above, would be another order of the
// same sums.)  Few rows are bound by the chain of loads, so
// each batch of them goes out together; many by the 2-byte loads and stores.  1000 x 5120: 14.5 us (13 rows: 5.7),
// ln_mix_seq_kernel 37.7 (29.9).
// The compiler unrolls the general form's last loop by two; a thread with an odd count of elements takes its last one in
// the remainder, where (x - mean) * inv is rounded once to binary16 (v_fma_mixlo_f16) instead of to fp32 and then to
// binary16.  Both roundings are written out here.
template <int NE>
__global__ __launch_bounds__(256) void ln_mix_wide_kernel(LnMixSeq a) {
  __shared__ float red[2][2][4];
  const int C = a.C, t = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  h1 xr[2][NE], gam[NE], bet[NE];  // [0]: the row before, [1]: this row
  const h1* row[2] = {a.x + (size_t)(t ? t - 1 : 0) * C, a.x + (size_t)t * C};
#pragma unroll
  for (int n = 0; n < NE; n++) {
    const int i = tid + n * 256, ic = i < C ? i : 0;
    xr[0][n] = row[0][ic];
    xr[1][n] = row[1][ic];
    gam[n] = a.ln_w[ic];
    bet[n] = a.ln_b[ic];
  }
  float mean[2], inv[2];
#pragma unroll
  for (int r = 0; r < 2; r++) {
    float s = 0.f;
#pragma unroll
    for (int n = 0; n < NE; n++)
      if (tid + n * 256 < C) s += (float)xr[r][n];
    s = wave_sum(s);
    if (lane == 0) red[0][r][wv] = s;
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 2; r++) {
    float s = 0.f;
#pragma unroll
    for (int w = 0; w < 4; w++) s += red[0][r][w];
    mean[r] = s / (float)C;
    float q = 0.f;
#pragma unroll
    for (int n = 0; n < NE; n++)
      if (tid + n * 256 < C) {
        const float d = (float)xr[r][n] - mean[r];
        q += d * d;
      }
    q = wave_sum(q);
    if (lane == 0) red[1][r][wv] = q;
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 2; r++) {
    float q = 0.f;
#pragma unroll
    for (int w = 0; w < 4; w++) q += red[1][r][w];
    float var = q / (float)C;
    var = var > 0.f ? var : 0.f;
    inv[r] = 1.0f / sqrtf(var + 1e-5f);
  }
#pragma unroll
  for (int n = 0; n < NE; n++) {
#pragma unroll
    for (int r = 0; r < 2; r++) {
      const float d = (float)xr[r][n] - mean[r];
      float p = d * inv[r];
      asm("" : "+v"(p));  // rounded to fp32 before the conversion
      h1 nrm = (h1)p;
      if (n >= 16 && n % 2 == 0) {  // C > 4096: every thread has 16 elements before its last
        uint32_t once;
        asm("v_fma_mixlo_f16 %0, %1, %2, 0" : "=v"(once) : "v"(d), "v"(inv[r]));
        if (tid + (n + 1) * 256 >= C) nrm = __builtin_bit_cast(h1, (uint16_t)once);
      }
      xr[r][n] = (nrm * gam[n]) + bet[n];
    }
  }
  if (t == 0) {
#pragma unroll
    for (int n = 0; n < NE; n++) xr[0][n] = a.state[tid + n * 256 < C ? tid + n * 256 : 0];
  }
  for (int m = 0; m < a.nmix; m++) {  // the loads of one vector together, then its stores
    h1 mx[NE];
#pragma unroll
    for (int n = 0; n < NE; n++) mx[n] = a.mix[m][tid + n * 256 < C ? tid + n * 256 : 0];
    h1* out = a.out[m] + (size_t)t * C;
#pragma unroll
    for (int n = 0; n < NE; n++)
      if (tid + n * 256 < C) out[tid + n * 256] = mix1(xr[1][n], xr[0][n], mx[n]);
  }
  if (t == a.T - 1) {
#pragma unroll
    for (int n = 0; n < NE; n++)
      if (tid + n * 256 < C) a.xx_last[tid + n * 256] = xr[1][n];
  }
}

// ---------------------------------------------------------------------------
// RWKV-4 WKV scan, one launch.  k, v [T][C] fp32; r [T][C] half (already through the sigmoid), overwritten with
// r * half(wkv).
//
// A workgroup owns CG channels and cuts time into blocks of nchunk chunks of Lc steps, a thread per (channel, chunk).
// Per block: every chunk is scanned from an empty state (k and v stay in registers); the local end states are
// composed into the states at the ends of the chunks by a doubling scan in LDS; every chunk is scanned again from its true
// start state, writing the outputs; the last chunk's end state starts the next block, whose k, v and r were requested step
// by step as the registers of this one became free.
// What bounds it: about 150 vector instructions per channel and step, most of them three expf (a six-instruction
// exponential within 2 ulp would save a tenth, but the outputs would no longer be those of the one-token kernel).  att_seq_v4
// as a whole (products included) against a launch for pass 1, one for passes 2 and 3, which read k and v twice and
// composed every chunk's start from all chunks before it, us: 2048 channels, T = 13: 22.2 -> 18.1, 77: 29.4 -> 25.1,
// 1024: 81.4 -> 73.3, 4099 (a serial pass 2 of its own): 240.9 -> 223.4; 5120 channels, T = 1024: 277 -> 273, 4099: 1010 -> 1019.
// Requests ahead: the scan alone, 5120 channels, T = 4099: 117 -> 109.  Registers for every second chunk length from 8 on, not
// for 16 only: 2048 channels, T = 4099 (11 steps): 230.5 -> 223.4.  What it still loses to: pieces of 8 to 14 channels are a
// part of a line, fetched once for each, so 2112 to 3072 channels and more than 4096 steps were 2 to 6 % quicker in the three
// launches (8192 x 2304: 522 against 555), whose states were two to six times further from float64.
// (A form with scalar bases for whole blocks and masked steps for the last one spilled registers: 1024: 75.)
// ---------------------------------------------------------------------------
constexpr int kWkv4MaxCg = 32;
struct Wkv4Seq {
  int T, C, Lc, nchunk, nblock, cg;
  const float *k, *v, *u, *w;
  h1* r;
  const float *aa, *bb, *pp;  // state before the sequence; may alias aa_out / bb_out / pp_out (a channel has one workgroup)
  float *aa_out, *bb_out, *pp_out;
};

// p = max(a, b) (b on ties), ea = exp(a - p), eb = exp(b - p) with one exponential instead of two: the
// argument of the other one is +0 and expf(+0) is exactly 1, so for finite a and b these are the bits
// of the two calls.
__device__ __forceinline__ void exp_pair(float a, float b, float& p, float& ea, float& eb) {
  const bool first = a > b;
  p = first ? a : b;
  const float e = expf(first ? b - a : a - b);
  ea = first ? 1.0f : e;
  eb = first ? e : 1.0f;
}

// a: state (aa, bb, pp) followed by `steps` (times the decay w: dw) that contribute (la, lb, lp)
__device__ __forceinline__ void wkv4_compose(float& aa, float& bb, float& pp, float dw, float la, float lb, float lp) {
  float p, e1, e2;
  exp_pair(pp + dw, lp, p, e1, e2);
  aa = e1 * aa + e2 * la;
  bb = e1 * bb + e2 * lb;
  pp = p;
}

template <int LMAX>
__global__ __launch_bounds__(1024) void wkv4_scan_kernel(Wkv4Seq a) {
  __shared__ float ends[2][3][1024];  // end states of the chunks, by thread; two copies in turn
  __shared__ float start[3][kWkv4MaxCg];  // state at the start of the block
  const int CG = a.cg;
  // neighbouring channels on one XCD: CG channels are 4 CG bytes of a row, a part of a line
  const int n = gridDim.x, xcd = blockIdx.x & 7, grp = xcd * (n >> 3) + min(xcd, n & 7) + (blockIdx.x >> 3);
  const int tid = threadIdx.x, cl = tid % CG, ch = tid / CG, c = min(grp * CG + cl, a.C - 1);
  const bool live = grp * CG + cl < a.C;  // the last workgroup's channels past the end follow the last one and store nothing
  const float w = a.w[c], u = a.u[c];
  if (ch == 0) {
    start[0][cl] = a.aa[c];
    start[1][cl] = a.bb[c];
    start[2][cl] = a.pp[c];
  }
  const float dw = (float)a.Lc * w;
  float kk[LMAX], vv[LMAX];
  h1 rr[LMAX];
  auto load = [&](int blk, int i) {
    const size_t j = (size_t)min((blk * a.nchunk + ch) * a.Lc + min(i, a.Lc - 1), a.T - 1) * a.C + c;
    kk[i] = a.k[j];
    vv[i] = a.v[j];
    rr[i] = a.r[j];
  };
#pragma unroll
  for (int i = 0; i < LMAX; i++) load(0, i);
  for (int blk = 0; blk < a.nblock; blk++) {
    const int t0 = (blk * a.nchunk + ch) * a.Lc, len = live ? min(a.Lc, a.T - t0) : 0;  // len <= 0: nothing left for this chunk
    // from an empty state, without the chain of running maxima: aa = sum exp(k_i + (len - 1 - i) w - pp) v_i, bb = the same without v
    float aa = 0.f, bb = 0.f, pp = -1e30f, q[LMAX], off = 0.f;
#pragma unroll
    for (int i = LMAX - 1; i >= 0; i--) {
      q[i] = i < len ? kk[i] + off : -1e30f;
      off = i < len ? off + w : off;
      pp = fmaxf(pp, q[i]);
    }
#pragma unroll
    for (int i = 0; i < LMAX; i++) {
      const float e = i < len ? expf(q[i] - pp) : 0.f;
      aa += e * vv[i];
      bb += e;
    }
    // after the step of distance s, a thread holds the contribution of its chunk and up to 2 s - 1 chunks before it
    int cur = 0;
    for (int s = 1; s < a.nchunk; s *= 2) {
      ends[cur][0][tid] = aa;
      ends[cur][1][tid] = bb;
      ends[cur][2][tid] = pp;
      __syncthreads();
      if (ch >= s) {
        float pa = ends[cur][0][tid - s * CG], pb = ends[cur][1][tid - s * CG], p = ends[cur][2][tid - s * CG];
        wkv4_compose(pa, pb, p, (float)s * dw, aa, bb, pp);
        aa = pa, bb = pb, pp = p;
      }
      cur ^= 1;
    }
    ends[cur][0][tid] = aa;
    ends[cur][1][tid] = bb;
    ends[cur][2][tid] = pp;
    __syncthreads();
    aa = start[0][cl], bb = start[1][cl], pp = start[2][cl];
    if (ch > 0)
      wkv4_compose(aa, bb, pp, (float)ch * dw, ends[cur][0][tid - CG], ends[cur][1][tid - CG], ends[cur][2][tid - CG]);
    // the registers of a step take the next block's step once they have been used
    auto apply = [&](auto more) {
#pragma unroll
      for (int i = 0; i < LMAX; i++) {
        if (i < len) {
          const float k = kk[i], v = vv[i];
          // kernels/cuda/att.cu:43-60
          float p, e1, e2;
          exp_pair(pp, u + k, p, e1, e2);
          const float wkv = (e1 * aa + e2 * v) / (e1 * bb + e2);
          a.r[(size_t)(t0 + i) * a.C + c] = rr[i] * (h1)wkv;
          wkv4_compose(aa, bb, pp, w, v, 1.0f, k);
        }
        if constexpr (decltype(more)::value) load(blk + 1, i);
      }
    };
    if (blk + 1 < a.nblock) apply(std::true_type{}); else apply(std::false_type{});
    if (len > 0 && t0 + len == a.T) {
      a.aa_out[c] = aa;
      a.bb_out[c] = bb;
      a.pp_out[c] = pp;
    }
    if (blk + 1 < a.nblock) {
      __syncthreads();  // everyone has read `start` and `ends`
      if (ch == a.nchunk - 1) start[0][cl] = aa, start[1][cl] = bb, start[2][cl] = pp;  // read behind the next block's barriers
    }
  }
}

// ---------------------------------------------------------------------------
// RWKV-5.2 scan, head size 64.  r, k, v [T][C] fp32; state [H][64 key][64 value] fp32.
// A workgroup of 256 threads serves one (head, chunk): thread t owns value index
// j = t % 64 and key rows i = (t / 64) * 16 .. +15 of the state (16 registers).
// Output row t: y_j = sum_i r_i (u_i k_i v_j + s_ij), then groupnorm over the head's 64
// values, rounding to half and the gate multiply (att_seq.cu:294-316, :406-411).
// The scan over a prompt regroups the sums by chunk anyway, so its multiply-adds are fused (four
// instructions per state element and step instead of seven); the one-token operator keeps the
// separately rounded products and sums.  The partial sums of 16 steps wait in LDS for one round
// of group norms shared by the four waves, instead of a barrier and one wave's group norm per step.
// ---------------------------------------------------------------------------
struct Wkv5Seq {
  int T, C, H, Lc, nchunk;
  int uw_head;       // 0: u, w are [H][64] (RWKV-5.2); 1: one value per head (RWKV-5.0)
  const float *r, *k, *v, *w, *u, *lx_w, *lx_b;
  const h1* g;       // [T][C] gate, already through silu; null for RWKV-5.0
  const float* s;    // state before the sequence
  float* loc;        // [nchunk][H][64][64] local end states
  float* sin;        // [nchunk][H][64][64] state at the start of each chunk
  float* s_out;
  h1* gated;         // [T][C]
};

constexpr int S5 = 64;

__global__ __launch_bounds__(256) void wkv5_local_kernel(Wkv5Seq a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  float* kk = reinterpret_cast<float*>(smem);  // [Lc][64]
  float* vv = kk + a.Lc * S5;
  __shared__ float wsh[S5];
  const int h = blockIdx.x, ch = blockIdx.y, t = threadIdx.x, j = t & 63, ig = t >> 6;
  const int t0 = ch * a.Lc, len = min(a.Lc, a.T - t0);
  for (int e = t; e < len * S5; e += 256) {
    const size_t src = (size_t)(t0 + e / S5) * a.C + h * S5 + (e % S5);
    kk[e] = a.k[src];
    vv[e] = a.v[src];
  }
  if (t < S5) wsh[t] = a.w[a.uw_head ? h : h * S5 + t];
  __syncthreads();
  float s[16];
#pragma unroll
  for (int ii = 0; ii < 16; ii++) s[ii] = 0.f;
  for (int tt = 0; tt < len; tt++) {
    const float vj = vv[tt * S5 + j];
#pragma unroll
    for (int ii = 0; ii < 16; ii++) {
      const int i = ig * 16 + ii;
      s[ii] = __builtin_fmaf(wsh[i], s[ii], kk[tt * S5 + i] * vj);
    }
  }
  float* dst = a.loc + ((size_t)ch * a.H + h) * S5 * S5;
#pragma unroll
  for (int ii = 0; ii < 16; ii++) dst[(ig * 16 + ii) * S5 + j] = s[ii];
}

// The serial pass over the chunks, one state element per thread.  The decay of the incoming state
// over a whole chunk is one multiplication by w^Lc (formed once by repeated multiplication), and the
// chunks' local end states are read eight at a time, the next eight while these are consumed.
__global__ __launch_bounds__(256) void wkv5_carry_kernel(Wkv5Seq a) {
  const size_t e = (size_t)blockIdx.x * 256 + threadIdx.x;  // element of [H][64][64]
  const size_t per = (size_t)a.H * S5 * S5;
  if (e >= per) return;
  constexpr int PF = 8;
  const int i = (int)((e / S5) % S5), h = (int)(e / (S5 * S5));
  const float w = a.w[a.uw_head ? h : h * S5 + i];
  float cur[PF], nxt[PF];
#pragma unroll
  for (int j = 0; j < PF; j++) cur[j] = a.loc[(size_t)(j < a.nchunk ? j : a.nchunk - 1) * per + e];
  float s = a.s[e];
  float wl = 1.0f;  // w^Lc; the last chunk may be shorter, but nothing is carried out of it here
  for (int q = 0; q < a.Lc; q++) wl *= w;
  for (int ch0 = 0; ch0 < a.nchunk; ch0 += PF) {
#pragma unroll
    for (int j = 0; j < PF; j++) {
      const int ch = ch0 + PF + j;
      nxt[j] = a.loc[(size_t)(ch < a.nchunk ? ch : a.nchunk - 1) * per + e];
    }
#pragma unroll
    for (int j = 0; j < PF; j++) {
      const int ch = ch0 + j;
      if (ch < a.nchunk) {
        a.sin[(size_t)ch * per + e] = s;
        s = __builtin_fmaf(wl, s, cur[j]);
      }
    }
#pragma unroll
    for (int j = 0; j < PF; j++) cur[j] = nxt[j];
  }
}

__global__ __launch_bounds__(256) void wkv5_apply_kernel(Wkv5Seq a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  float* rr = reinterpret_cast<float*>(smem);  // [Lc][64]
  float* kk = rr + a.Lc * S5;
  float* vv = kk + a.Lc * S5;
  __shared__ float wsh[S5], ush[S5];
  constexpr int kGroup = 16;  // steps whose partial sums wait in LDS for one round of group norms
  __shared__ float part[kGroup][4][S5];
  const int h = blockIdx.x, ch = blockIdx.y, t = threadIdx.x, j = t & 63, ig = t >> 6;
  const int t0 = ch * a.Lc, len = min(a.Lc, a.T - t0);
  for (int e = t; e < len * S5; e += 256) {
    const size_t src = (size_t)(t0 + e / S5) * a.C + h * S5 + (e % S5);
    rr[e] = a.r[src];
    kk[e] = a.k[src];
    vv[e] = a.v[src];
  }
  if (t < S5) {
    wsh[t] = a.w[a.uw_head ? h : h * S5 + t];
    ush[t] = a.u[a.uw_head ? h : h * S5 + t];
  }
  const float* src = a.sin + ((size_t)ch * a.H + h) * S5 * S5;
  float s[16];
#pragma unroll
  for (int ii = 0; ii < 16; ii++) s[ii] = src[(ig * 16 + ii) * S5 + j];
  const float gw = a.lx_w[h * S5 + j], gb = a.lx_b[h * S5 + j];
  __syncthreads();
  float wr[16], ur[16];
#pragma unroll
  for (int ii = 0; ii < 16; ii++) {
    wr[ii] = wsh[ig * 16 + ii];
    ur[ii] = ush[ig * 16 + ii];
  }
  for (int tb = 0; tb < len; tb += kGroup) {
    const int n = min(kGroup, len - tb);
    for (int q = 0; q < n; q++) {
      const int tt = tb + q;
      const float vj = vv[tt * S5 + j];
      float acc = 0.f;
#pragma unroll
      for (int ii = 0; ii < 16; ii++) {
        const int i = ig * 16 + ii;
        const float aij = kk[tt * S5 + i] * vj;
        const float tmp = __builtin_fmaf(ur[ii], aij, s[ii]);
        s[ii] = __builtin_fmaf(wr[ii], s[ii], aij);
        acc = __builtin_fmaf(rr[tt * S5 + i], tmp, acc);
      }
      part[q][ig][j] = acc;
    }
    __syncthreads();
    // wave ig: the group norms of steps ig, ig + 4, ... of this round
    for (int q = ig; q < n; q += 4) {
      const float o = ((part[q][0][j] + part[q][1][j]) + part[q][2][j]) + part[q][3][j];
      const float mean = wave_sum(o) / (float)S5;
      const float d = o - mean;
      float var = wave_sum(d * d) / (float)S5;
      var = var > 0.f ? var : 0.f;
      const float inv = 1.0f / sqrtf(var + 1e-5f);
      const float y = d * inv * gw + gb;
      const size_t oi = (size_t)(t0 + tb + q) * a.C + h * S5 + j;
      a.gated[oi] = a.g ? (h1)y * a.g[oi] : (h1)y;
    }
    __syncthreads();  // `part` is free for the next round
  }
  if (ch == a.nchunk - 1) {
    float* dst = a.s_out + (size_t)h * S5 * S5;
#pragma unroll
    for (int ii = 0; ii < 16; ii++) dst[(ig * 16 + ii) * S5 + j] = s[ii];
  }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
#define FR_TRY(expr)        \
  do {                      \
    int _e = (expr);        \
    if (_e != 0) return _e; \
  } while (0)

static size_t al256(size_t n) { return (n + 255) / 256 * 256; }

static int check_w(const frhip_weight* w, int K, int N, const char* what) {
  if (!w || !w->data) return set_error(FRHIP_EINVAL, what);
  if (w->dtype != FRHIP_F16 && w->dtype != FRHIP_U8) return set_error(FRHIP_EINVAL, what);
  if (w->K != K || w->N != N) return set_error(FRHIP_ESHAPE, what);
  if (w->dtype == FRHIP_U8 && (!w->mx || !w->rx || !w->my || !w->ry)) return set_error(FRHIP_EINVAL, what);
  return 0;
}

static int launch_ln_mix(int T, int C, const void* x, const void* state, const void* ln_w, const void* ln_b,
                         const void* const* mix, h1* const* out, int nmix, void* xx_last, hipStream_t st) {
  LnMixSeq a;
  a.T = T; a.C = C; a.nmix = nmix;
  a.x = (const h1*)x; a.state = (const h1*)state; a.ln_w = (const h1*)ln_w; a.ln_b = (const h1*)ln_b;
  for (int i = 0; i < nmix; i++) {
    a.mix[i] = (const h1*)mix[i];
    a.out[i] = out[i];
  }
  a.xx_last = (h1*)xx_last;
  const int nwg = (T + kLnRows - 1) / kLnRows;
  if (C % 8 == 0 && C <= 4096)
    nmix == 2 ? launch_ln_mix_rows<2>(a, nwg, st) : nmix == 3 ? launch_ln_mix_rows<3>(a, nwg, st) : launch_ln_mix_rows<4>(a, nwg, st);
  else if (C > 4096 && C <= 6144)
    hipLaunchKernelGGL(ln_mix_wide_kernel<24>, dim3(T), dim3(256), 0, st, a);
  else
    hipLaunchKernelGGL(ln_mix_seq_kernel, dim3(T), dim3(256), 4 * (size_t)C, st, a);
  return check_launch("ln_mix_seq");
}

// A workgroup's channels: one workgroup per compute unit (or as few rounds of them as 32 channels allow), at least 8 (32-byte
// pieces of a row); the last workgroup may have fewer (4736 channels: 250 workgroups of 19; as 148 of 32, which divides, T = 4099
// took 945 us of att_seq_v4 against 927).  Chunks of at least 4 steps (2 where that still is one wave's work), of at most 16, which
// a thread keeps in registers.  Up to 128 of them where 8 channels leave room; otherwise 64, of a prompt that they hold in one
// block, and as many as there are threads of a longer one (2112 channels, 113 chunks against 64: T = 1100 107 against 115,
// 2048 132.5 against 134; but T = 1024, ten steps a chunk against sixteen: 83 against 80.5).
// C = 5120, T = 2048: 484 with 20 channels, 501 with 16 (1.25 rounds), 492 with 8.
static void cut_wkv4_scan(Wkv4Seq& q, int cus) {
  constexpr int kMaxLc = 16;
  const int rounds = (q.C + cus * kWkv4MaxCg - 1) / (cus * kWkv4MaxCg);
  q.cg = (q.C + cus * rounds - 1) / (cus * rounds);
  if (q.cg < 8) q.cg = 8;
  const int most = 1024 / q.cg, chunks = q.cg == 8 ? 128 : most < 64 || q.T > 64 * kMaxLc ? most : 64;
  q.nblock = (q.T + chunks * kMaxLc - 1) / (chunks * kMaxLc);
  q.Lc = (q.T + chunks * q.nblock - 1) / (chunks * q.nblock);
  const int least = q.T <= 32 ? 2 : 4;
  if (q.Lc < least) q.Lc = least;
  q.nchunk = (q.T + q.Lc * q.nblock - 1) / (q.Lc * q.nblock);
}

static void launch_wkv4_scan(Wkv4Seq& q, hipStream_t st) {
  cut_wkv4_scan(q, compute_units());
  const dim3 grid((q.C + q.cg - 1) / q.cg), block(q.nchunk * q.cg);
  if (q.Lc <= 4)
    hipLaunchKernelGGL(wkv4_scan_kernel<4>, grid, block, 0, st, q);
  else if (q.Lc <= 8)
    hipLaunchKernelGGL(wkv4_scan_kernel<8>, grid, block, 0, st, q);
  else if (q.Lc <= 10)
    hipLaunchKernelGGL(wkv4_scan_kernel<10>, grid, block, 0, st, q);
  else if (q.Lc <= 12)
    hipLaunchKernelGGL(wkv4_scan_kernel<12>, grid, block, 0, st, q);
  else if (q.Lc <= 14)
    hipLaunchKernelGGL(wkv4_scan_kernel<14>, grid, block, 0, st, q);
  else
    hipLaunchKernelGGL(wkv4_scan_kernel<16>, grid, block, 0, st, q);
}

// chunk length for a scan of T steps when one chunk occupies `units` workgroup-sized units:
// enough chunks to fill the device (~4 units per CU), chunks of at least 16 steps (the serial pass
// over the chunks costs about 0.18 us per chunk: at T = 1024, 64 chunks of 16 beat 128 of 8)
constexpr int kMinChunk = 16;
static int pick_chunk(int T, int units) {
  int want = (4 * compute_units() + units - 1) / units;
  if (want < 1) want = 1;
  int Lc = (T + want - 1) / want;
  if (Lc < kMinChunk) Lc = kMinChunk;
  if (Lc > 64) Lc = 64;
  return Lc;
}

}  // namespace frhip

using namespace frhip;

static size_t seq_dequant_bytes(int C, int F) {
  const size_t cc = (size_t)C * C, cf = (size_t)C * F;
  const size_t att = 4 * cc, ffn = cc + cf;
  return 2 * (att > ffn ? att : ffn);
}

// RWKV-5: the chunks' end states and start states, [nchunk][C * 64] fp32 each, chunks of at least kMinChunk steps (pick_chunk)
static size_t scan_bytes(int T, int C) { return al256(4 * (((size_t)T + kMinChunk - 1) / kMinChunk) * C * 64); }

extern "C" size_t frhip_seq_workspace_bytes(int T, int C, int F) {
  if (T <= 0 || C <= 0 || F <= 0) return 0;
  const size_t tc = (size_t)T * C;
  // activations: 4 mixed inputs + g + gated (half), k v r y (fp32), vx [T][F] (half)
  size_t n = 6 * al256(2 * tc) + 4 * al256(4 * tc) + al256(2 * (size_t)T * F);
  // short prompts: partial sums of the products split over K (launch_gemm's few_rows scratch)
  if (T <= kFewRowsMax) n += al256(4 * kFewRowsFloats);
  n += 2 * scan_bytes(T, C);
  // binary16 expansion of the uint8 weights of one launch: the largest group is k,v,r,g or ffn r,k
  n += al256(seq_dequant_bytes(C, F));
  return n;
}

namespace {
struct SeqWs {
  h1 *m0, *m1, *m2, *m3, *g, *gated, *vx;
  float *f0, *f1, *f2, *f3;
  float* few;        // kFewRowsFloats floats when T <= kFewRowsMax, else null
  size_t few_floats;
  float* scan;
  h1* dq;  // binary16 expansion of one launch's uint8 weights
};
SeqWs carve_seq(void* ws, int T, int C, int F) {
  const size_t tc = (size_t)T * C;
  unsigned char* p = static_cast<unsigned char*>(ws);
  SeqWs w;
  h1** hs[6] = {&w.m0, &w.m1, &w.m2, &w.m3, &w.g, &w.gated};
  for (auto h : hs) {
    *h = reinterpret_cast<h1*>(p);
    p += al256(2 * tc);
  }
  float** fs[4] = {&w.f0, &w.f1, &w.f2, &w.f3};
  for (auto f : fs) {
    *f = reinterpret_cast<float*>(p);
    p += al256(4 * tc);
  }
  w.few = T <= kFewRowsMax ? reinterpret_cast<float*>(p) : nullptr;
  w.few_floats = T <= kFewRowsMax ? kFewRowsFloats : 0;
  if (w.few) p += al256(4 * kFewRowsFloats);
  w.vx = reinterpret_cast<h1*>(p);
  p += al256(2 * (size_t)T * F);
  w.scan = reinterpret_cast<float*>(p);
  p += 2 * scan_bytes(T, C);
  w.dq = reinterpret_cast<h1*>(p);
  return w;
}
}  // namespace

// ffn_seq (kernels/cuda/ffn_seq.cu:65-109).  x [T][C]; sx [C] shift state; xx_out [C] = LN(x)[T-1].
static int ffn_seq_impl(bool tiled_sums, int T, int C, int F, const void* x, const void* sx, const void* ln_w, const void* ln_b,
                        const void* k_mix, const void* r_mix, const frhip_weight* kw, const frhip_weight* vw,
                        const frhip_weight* rw, void* x_out, void* xx_out, int post_div2, void* workspace, frhip_stream s) {
  if (T <= 0) return set_error(FRHIP_ESHAPE, "ffn_seq: T must be positive");
  if (!x || !sx || !ln_w || !ln_b || !k_mix || !r_mix || !x_out || !xx_out || !workspace)
    return set_error(FRHIP_EINVAL, "ffn_seq: null pointer");
  if (C <= 0 || C % 64 != 0 || F <= 0 || F % 64 != 0) return set_error(FRHIP_ESHAPE, "ffn_seq: C and F must be multiples of 64");
  FR_TRY(check_w(kw, C, F, "ffn_seq: bad key weight"));
  FR_TRY(check_w(vw, F, C, "ffn_seq: bad value weight"));
  FR_TRY(check_w(rw, C, C, "ffn_seq: bad receptance weight"));
  hipStream_t st = static_cast<hipStream_t>(s);
  SeqWs w = carve_seq(workspace, T, C, F);
  const void* mixes[2] = {k_mix, r_mix};
  h1* outs[2] = {w.m0, w.m1};
  FR_TRY(launch_ln_mix(T, C, x, sx, ln_w, ln_b, mixes, outs, 2, xx_out, st));
  GemmArgs a;
  memset(&a, 0, sizeof(a));
  a.M = T; a.K = C; a.tiled_sums = tiled_sums;
  gemm_add_seg(a, w.m1, rw, w.m2, G_SIGMOID);  // r
  gemm_add_seg(a, w.m0, kw, w.vx, G_RELU2);    // vx
  if (kw->dtype != rw->dtype) return set_error(FRHIP_EINVAL, "ffn_seq: key/receptance dtypes differ");
  FR_TRY(launch_gemm(a, kw->dtype == FRHIP_U8, st, "ffn_seq r,k", w.dq, nullptr, 0, 0, w.few, w.few_floats));
  GemmArgs b;
  memset(&b, 0, sizeof(b));
  b.M = T; b.K = F; b.tiled_sums = tiled_sums;
  b.res_x = (const h1*)x; b.res_r = w.m2; b.div2 = post_div2 ? 1 : 0;
  gemm_add_seg(b, w.vx, vw, x_out, G_FFN_OUT);
  // the four fp32 [T][C] buffers of the workspace (unused by ffn) take the partial sums of a K-split launch
  return launch_gemm(b, vw->dtype == FRHIP_U8, st, "ffn_seq v", w.dq, w.f0, (size_t)(w.f1 - w.f0), kSeqMaxSplit, w.few,
                     w.few_floats);
}

extern "C" int frhip_ffn_seq(int T, int C, int F, const void* x, const void* sx, const void* ln_w, const void* ln_b,
                             const void* k_mix, const void* r_mix, const frhip_weight* kw, const frhip_weight* vw,
                             const frhip_weight* rw, void* x_out, void* xx_out, int post_div2, void* workspace,
                             frhip_stream s) {
  return ffn_seq_impl(true, T, C, F, x, sx, ln_w, ln_b, k_mix, r_mix, kw, vw, rw, x_out, xx_out, post_div2, workspace, s);
}

extern "C" int frhip_ffn_seq_v4(int T, int C, int F, const void* x, const void* sx, const void* ln_w, const void* ln_b,
                                const void* k_mix, const void* r_mix, const frhip_weight* kw, const frhip_weight* vw,
                                const frhip_weight* rw, void* x_out, void* xx_out, int post_div2, void* workspace,
                                frhip_stream s) {
  return ffn_seq_impl(false, T, C, F, x, sx, ln_w, ln_b, k_mix, r_mix, kw, vw, rw, x_out, xx_out, post_div2, workspace, s);
}

// RWKV-4 sequence attention.  The reference has no such operator
// (kernels/default/model_forward_seq.cpp:111-112); the result is defined by T one-token steps
// of kernels/cuda/att.cu:182-217 (model_forward_seq.cpp:34-46).
extern "C" int frhip_att_seq_v4(int T, int C, const void* x, const void* sx, const float* aa, const float* bb,
                                const float* pp, const void* ln_w, const void* ln_b, const void* k_mix,
                                const void* v_mix, const void* r_mix, const float* t_decay, const float* t_first,
                                const frhip_weight* kw, const frhip_weight* vw, const frhip_weight* rw,
                                const frhip_weight* ow, void* x_out, void* xx_out, float* aa_out, float* bb_out,
                                float* pp_out, void* workspace, frhip_stream s) {
  if (T <= 0) return set_error(FRHIP_ESHAPE, "att_seq_v4: T must be positive");
  if (!x || !sx || !aa || !bb || !pp || !ln_w || !ln_b || !k_mix || !v_mix || !r_mix || !t_decay || !t_first ||
      !x_out || !xx_out || !aa_out || !bb_out || !pp_out || !workspace)
    return set_error(FRHIP_EINVAL, "att_seq_v4: null pointer");
  if (C <= 0 || C % 64 != 0) return set_error(FRHIP_ESHAPE, "att_seq_v4: C must be a multiple of 64");
  FR_TRY(check_w(kw, C, C, "att_seq_v4: bad key weight"));
  FR_TRY(check_w(vw, C, C, "att_seq_v4: bad value weight"));
  FR_TRY(check_w(rw, C, C, "att_seq_v4: bad receptance weight"));
  FR_TRY(check_w(ow, C, C, "att_seq_v4: bad output weight"));
  if (kw->dtype != vw->dtype || kw->dtype != rw->dtype) return set_error(FRHIP_EINVAL, "att_seq_v4: k/v/r dtypes differ");
  hipStream_t st = static_cast<hipStream_t>(s);
  SeqWs w = carve_seq(workspace, T, C, 64);
  const void* mixes[3] = {k_mix, v_mix, r_mix};
  h1* outs[3] = {w.m0, w.m1, w.m2};
  FR_TRY(launch_ln_mix(T, C, x, sx, ln_w, ln_b, mixes, outs, 3, xx_out, st));
  GemmArgs a;
  memset(&a, 0, sizeof(a));
  a.M = T; a.K = C;
  gemm_add_seg(a, w.m0, kw, w.f0, G_STORE_F32);  // k
  gemm_add_seg(a, w.m1, vw, w.f1, G_STORE_F32);  // v
  gemm_add_seg(a, w.m2, rw, w.m3, G_SIGMOID);    // r
  FR_TRY(launch_gemm(a, kw->dtype == FRHIP_U8, st, "att_seq_v4 k,v,r", w.dq, nullptr, 0, 0, w.few, w.few_floats));

  Wkv4Seq q;
  q.T = T; q.C = C;
  q.k = w.f0; q.v = w.f1; q.u = t_first; q.w = t_decay; q.r = w.m3;
  q.aa = aa; q.bb = bb; q.pp = pp;
  q.aa_out = aa_out; q.bb_out = bb_out; q.pp_out = pp_out;
  launch_wkv4_scan(q, st);
  FR_TRY(check_launch("wkv4_seq"));

  GemmArgs b;
  memset(&b, 0, sizeof(b));
  b.M = T; b.K = C;
  b.res_x = (const h1*)x;
  gemm_add_seg(b, w.m3, ow, x_out, G_RESIDUAL);
  return launch_gemm(b, ow->dtype == FRHIP_U8, st, "att_seq_v4 out", w.dq, nullptr, 0, 0, w.few, w.few_floats);
}

extern "C" int frhip_wkv4_cut(int T, int C, int compute_units, int* out) {
  if (!out) return set_error(FRHIP_EINVAL, "wkv4_cut: null pointer");
  if (T <= 0 || C <= 0 || C % 64 != 0 || compute_units < 1) return set_error(FRHIP_ESHAPE, "wkv4_cut: no such scan");
  Wkv4Seq q = {};
  q.T = T; q.C = C;
  cut_wkv4_scan(q, compute_units);
  out[0] = q.cg; out[1] = (C + q.cg - 1) / q.cg; out[2] = q.nblock; out[3] = q.nchunk; out[4] = q.Lc;
  return 0;
}

// Shared by RWKV-5.0 (no gate, u and w per head) and RWKV-5.2.
static int att_seq_v5_impl(bool v50, int T, int C, int H, const void* x, const void* sx, const float* s_in,
                                  const void* ln_w, const void* ln_b, const float* lx_w, const float* lx_b,
                                  const void* k_mix, const void* v_mix, const void* r_mix, const void* g_mix,
                                  const float* t_decay, const float* t_first, const frhip_weight* kw,
                                  const frhip_weight* vw, const frhip_weight* rw, const frhip_weight* gw,
                                  const frhip_weight* ow, void* x_out, void* xx_out, float* s_out, void* workspace,
                                  frhip_stream s) {
  if (T <= 0) return set_error(FRHIP_ESHAPE, "att_seq_v5: T must be positive");
  if (!x || !sx || !s_in || !ln_w || !ln_b || !lx_w || !lx_b || !k_mix || !v_mix || !r_mix || (!v50 && !g_mix) || !t_decay ||
      !t_first || !x_out || !xx_out || !s_out || !workspace)
    return set_error(FRHIP_EINVAL, "att_seq_v5: null pointer");
  if (H <= 0 || C % H != 0 || C / H != 64) return set_error(FRHIP_ESHAPE, "att_seq_v5: head size must be 64");
  FR_TRY(check_w(kw, C, C, "att_seq_v5: bad key weight"));
  FR_TRY(check_w(vw, C, C, "att_seq_v5: bad value weight"));
  FR_TRY(check_w(rw, C, C, "att_seq_v5: bad receptance weight"));
  if (!v50) FR_TRY(check_w(gw, C, C, "att_seq_v5: bad gate weight"));
  FR_TRY(check_w(ow, C, C, "att_seq_v5: bad output weight"));
  if (kw->dtype != vw->dtype || kw->dtype != rw->dtype || (!v50 && kw->dtype != gw->dtype))
    return set_error(FRHIP_EINVAL, "att_seq_v5: k/v/r/g dtypes differ");
  hipStream_t st = static_cast<hipStream_t>(s);
  SeqWs w = carve_seq(workspace, T, C, 64);
  const void* mixes[4] = {k_mix, v_mix, r_mix, g_mix};
  h1* outs[4] = {w.m0, w.m1, w.m2, w.m3};
  FR_TRY(launch_ln_mix(T, C, x, sx, ln_w, ln_b, mixes, outs, v50 ? 3 : 4, xx_out, st));
  GemmArgs a;
  memset(&a, 0, sizeof(a));
  a.M = T; a.K = C; a.tiled_sums = true;
  gemm_add_seg(a, w.m0, kw, w.f0, G_STORE_F32);  // k
  gemm_add_seg(a, w.m1, vw, w.f1, G_STORE_F32);  // v
  gemm_add_seg(a, w.m2, rw, w.f2, G_STORE_F32);  // r
  if (!v50) gemm_add_seg(a, w.m3, gw, w.g, G_SILU);  // g
  FR_TRY(launch_gemm(a, kw->dtype == FRHIP_U8, st, "att_seq_v5 k,v,r,g", w.dq, nullptr, 0, 0, w.few, w.few_floats));

  Wkv5Seq q;
  q.T = T; q.C = C; q.H = H;
  q.uw_head = v50 ? 1 : 0;
  q.Lc = pick_chunk(T, H);
  q.nchunk = (T + q.Lc - 1) / q.Lc;
  q.r = w.f2; q.k = w.f0; q.v = w.f1; q.w = t_decay; q.u = t_first; q.lx_w = lx_w; q.lx_b = lx_b;
  q.g = v50 ? nullptr : w.g; q.s = s_in; q.s_out = s_out; q.gated = w.gated;
  const size_t per = al256(4 * (size_t)q.nchunk * C * 64) / 4;
  q.loc = w.scan;
  q.sin = q.loc + per;
  dim3 grid(H, q.nchunk);
  hipLaunchKernelGGL(wkv5_local_kernel, grid, dim3(256), 2 * sizeof(float) * q.Lc * S5, st, q);
  hipLaunchKernelGGL(wkv5_carry_kernel, dim3(((size_t)H * S5 * S5 + 255) / 256), dim3(256), 0, st, q);
  hipLaunchKernelGGL(wkv5_apply_kernel, grid, dim3(256), 3 * sizeof(float) * q.Lc * S5, st, q);
  FR_TRY(check_launch("wkv5_seq"));

  GemmArgs b;
  memset(&b, 0, sizeof(b));
  b.M = T; b.K = C; b.tiled_sums = true;
  b.res_x = (const h1*)x;
  gemm_add_seg(b, w.gated, ow, x_out, G_RESIDUAL);
  return launch_gemm(b, ow->dtype == FRHIP_U8, st, "att_seq_v5 out", w.dq, nullptr, 0, 0, w.few, w.few_floats);
}

// att_seq_v5_2 (kernels/cuda/att_seq.cu:368-423,464-493).
extern "C" int frhip_att_seq_v5_2(int T, int C, int H, const void* x, const void* sx, const float* s_in,
                                  const void* ln_w, const void* ln_b, const float* lx_w, const float* lx_b,
                                  const void* k_mix, const void* v_mix, const void* r_mix, const void* g_mix,
                                  const float* t_decay, const float* t_first, const frhip_weight* kw,
                                  const frhip_weight* vw, const frhip_weight* rw, const frhip_weight* gw,
                                  const frhip_weight* ow, void* x_out, void* xx_out, float* s_out, void* workspace,
                                  frhip_stream s) {
  return att_seq_v5_impl(false, T, C, H, x, sx, s_in, ln_w, ln_b, lx_w, lx_b, k_mix, v_mix, r_mix, g_mix, t_decay,
                         t_first, kw, vw, rw, gw, ow, x_out, xx_out, s_out, workspace, s);
}

// att_seq_v5 (RWKV-5.0): kernels/cuda/att_seq.cu:158-256,425-462.  The reference evaluates the
// recurrence in matrix form (decay powers times r k^T, att_seq.cu:181-243); here the same sums
// are taken by the chunked scan that serves RWKV-5.2, with u and w constant over a head.
extern "C" int frhip_att_seq_v5(int T, int C, int H, const void* x, const void* sx, const float* s_in,
                                const void* ln_w, const void* ln_b, const float* lx_w, const float* lx_b,
                                const void* k_mix, const void* v_mix, const void* r_mix, const float* t_decay,
                                const float* t_first, const frhip_weight* kw, const frhip_weight* vw,
                                const frhip_weight* rw, const frhip_weight* ow, void* x_out, void* xx_out,
                                float* s_out, void* workspace, frhip_stream s) {
  return att_seq_v5_impl(true, T, C, H, x, sx, s_in, ln_w, ln_b, lx_w, lx_b, k_mix, v_mix, r_mix, nullptr, t_decay,
                         t_first, kw, vw, rw, nullptr, ow, x_out, xx_out, s_out, workspace, s);
}
