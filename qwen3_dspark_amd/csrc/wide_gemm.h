// One 128-output-column "head" of a linear layer for 128 tokens, on gfx950:
//   C^T[dim][token] = W[dim][:] . x[token][:]      (dim < 128, token < 128)
// the tile of the projection kernels for many tokens (head_gemm.h has the
// 64-token tile that spreads a short call over the CUs).
//
// MFMA mapping (v_mfma_f32_32x32x16_bf16) as in head_gemm.h: A = 32 weight
// rows, B = 32 tokens.  4 waves, wave w taking tokens 64 (w & 1) .. + 63 and
// the dim tiles dh and dh + 2 (dh = w >> 1: dims 32 dh .. + 31 and their
// rotate-half partners + 64), so each wave reads 2 A and 2 B fragments per
// four MFMAs.  Every lane ends with, for two tokens (tt = 0, 1),
//   v[a][tt][r] = C^T[32 (dh + 2a) + 8 (r / 4) + 4 (l / 32) + r % 4][64 tg + 32 tt + l % 32],
// the RoPE partner of v[0] being v[1].
//
// Weights and token rows stream through two LDS slots of 64 hidden columns
// (32 KiB each, so that two workgroups fit a CU: one's start, stage waits and
// epilogue overlap the other's MFMAs), filled by direct-to-LDS loads one
// stage ahead.
//
// Bound: LDS reads (1 KiB per MFMA and wave, next to the loads' writes) and the
// workgroup's start and epilogue: 779 TFLOP/s at 8,192 tokens x 32 heads x
// hidden 1,024.  256 tokens on 8 waves with three slots (one workgroup per CU)
// took 98 us there against 88, and 22 against 17 us at 1,024 tokens.  Rotating
// the column order per head (the rows of a stage are a multiple of 2 KiB apart)
// changed nothing.
#pragma once
#include "head_gemm.h"

namespace dspark {

constexpr int WG_TOKENS = 128;                   // tokens per workgroup
constexpr int WG_WAVES = 4;
constexpr int WG_COLS = 64;                      // hidden columns per stage
constexpr int WG_PART = 128 * WG_COLS * 2;       // bytes of a stage's weight rows, or of its token rows
constexpr int WG_STAGE = 2 * WG_PART;
constexpr int WG_SMEM = 2 * WG_STAGE;            // 64 KiB

struct WideLane {
  int n, hl, tg, dh;
  __device__ __forceinline__ WideLane() {
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    n = lane & 31;
    hl = lane >> 5;
    tg = wave & 1;
    dh = wave >> 1;
  }
  // first of the 4 consecutive dims of v[a][..][4 q .. 4 q + 3]
  __device__ __forceinline__ int dim(int a, int q) const { return 32 * (dh + 2 * a) + 8 * q + 4 * hl; }
  __device__ __forceinline__ int token(int tt) const { return 64 * tg + 32 * tt + n; }
};

// w: first of the head's 128 weight rows; x: token rows, `tokens` of them;
// t0: the workgroup's first token; rows of both are `hidden` elements apart.
// Rows past `tokens` re-read the last token (their results are discarded by
// the caller).  The ring's LDS is free afterwards (the function ends with a
// barrier).
__device__ __forceinline__ void wide_tile_gemm(const bf16* __restrict__ w, const bf16* __restrict__ x, int tokens,
                                               int hidden, int t0, unsigned char* smem, f32x16 (&v)[2][2]) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const WideLane L;
  const int steps = hidden / WG_COLS;
  // Wave w loads rows 32w .. 32w+31 of both parts, 8 rows (1 KiB) per load:
  // lane L of load i fetches row 32w + 8i + L/8, 16-byte chunk (L%8) ^ swz(row).
  uint32_t off_w[4], off_x[4];
  #pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = 32 * wave + 8 * i + (lane >> 3);
    const uint32_t col = 16 * ((lane & 7) ^ hg_swz(row));
    off_w[i] = (uint32_t)(row * hidden * 2) + col;
    off_x[i] = (uint32_t)((min(t0 + row, tokens - 1) - t0) * hidden * 2) + col;
  }
  const bf16* xt = x + (size_t)t0 * hidden;
  const uint32_t smem_lds = lds_address(smem);
  auto issue = [&](int step) {
    const uint32_t slot = smem_lds + (uint32_t)((step & 1) * WG_STAGE + wave * 4096);
    #pragma unroll
    for (int i = 0; i < 4; ++i)
      lds_dma16_base(w + step * WG_COLS, off_w[i], __builtin_amdgcn_readfirstlane(slot + 1024u * i));
    #pragma unroll
    for (int i = 0; i < 4; ++i)
      lds_dma16_base(xt + step * WG_COLS, off_x[i], __builtin_amdgcn_readfirstlane(slot + WG_PART + 1024u * i));
  };
  #pragma unroll
  for (int a = 0; a < 2; ++a)
    #pragma unroll
    for (int tt = 0; tt < 2; ++tt) v[a][tt] = f32x16{};
  issue(0);
  for (int s = 0; s < steps; ++s) {
    // stage s has landed for every wave, whose LDS reads of stage s - 1 are done
    __builtin_amdgcn_sched_barrier(0);
    load_wait<0>();
    ring_barrier();
    if (s + 1 < steps) issue(s + 1);
    const unsigned char* wst = smem + (s & 1) * WG_STAGE;
    const unsigned char* xst = wst + WG_PART;
    #pragma unroll
    for (int ks = 0; ks < WG_COLS / 16; ++ks) {
      const int c = 2 * ks + L.hl;
      bf16x8 wa[2], xb[2];
      #pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int wr = 32 * (L.dh + 2 * i) + L.n, xr = L.token(i);
        wa[i] = *reinterpret_cast<const bf16x8*>(wst + wr * 128 + ((c ^ hg_swz(wr)) << 4));
        xb[i] = *reinterpret_cast<const bf16x8*>(xst + xr * 128 + ((c ^ hg_swz(xr)) << 4));
      }
      #pragma unroll
      for (int a = 0; a < 2; ++a)
        #pragma unroll
        for (int tt = 0; tt < 2; ++tt)
          v[a][tt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wa[a], xb[tt], v[a][tt], 0, 0, 0);
    }
  }
  __syncthreads();
}

// q/k RMSNorm over the 128 dims (y = w x / sqrt(mean(x^2) + eps)), then
// rotate-half RoPE, of both tokens of every lane.  angles(tt, dim, cos, sin)
// gives the rotary factors of dims dim .. dim + 3 (< 64) for token tt.  Holds a
// barrier: every wave of the workgroup calls it.
template <class Angles>
__device__ __forceinline__ void wide_norm_rope(f32x16 (&v)[2][2], const bf16* __restrict__ nw, float eps,
                                               unsigned char* smem, Angles angles) {
  const WideLane L;
  bf16x4 w[2][4];
  f32x4 c[2][4], s[2][4];
  #pragma unroll
  for (int q = 0; q < 4; ++q) {
    #pragma unroll
    for (int a = 0; a < 2; ++a) w[a][q] = *reinterpret_cast<const bf16x4*>(nw + L.dim(a, q));
    #pragma unroll
    for (int tt = 0; tt < 2; ++tt) angles(tt, L.dim(0, q), c[tt][q], s[tt][q]);
  }
  float* sums = reinterpret_cast<float*>(smem);        // [dh][token]
  float ss[2];
  #pragma unroll
  for (int tt = 0; tt < 2; ++tt) {
    ss[tt] = 0.f;
    #pragma unroll
    for (int a = 0; a < 2; ++a)
      #pragma unroll
      for (int r = 0; r < 16; ++r) ss[tt] += v[a][tt][r] * v[a][tt][r];
    ss[tt] += __shfl_xor(ss[tt], 32);
    if (L.hl == 0) sums[L.dh * WG_TOKENS + L.token(tt)] = ss[tt];
  }
  __syncthreads();
  #pragma unroll
  for (int tt = 0; tt < 2; ++tt) {
    const float r = rsqrtf((ss[tt] + sums[(L.dh ^ 1) * WG_TOKENS + L.token(tt)]) * (1.0f / HD) + eps);
    #pragma unroll
    for (int e = 0; e < 16; ++e) {
      const float lo = v[0][tt][e] * r * (float)w[0][e >> 2][e & 3];
      const float hi = v[1][tt][e] * r * (float)w[1][e >> 2][e & 3];
      v[0][tt][e] = lo * c[tt][e >> 2][e & 3] - hi * s[tt][e >> 2][e & 3];
      v[1][tt][e] = hi * c[tt][e >> 2][e & 3] + lo * s[tt][e >> 2][e & 3];
    }
  }
}

// Store the lane pair's 64 dims of token tt as bf16 (row = the token's 128-dim
// head): after swapping halves with its partner lane, a lane writes 8
// consecutive dims per 16 bytes.  Both lanes of the pair execute it; `valid`
// gates the stores only.
__device__ __forceinline__ void wide_store(const f32x16 (&v)[2][2], int tt, bf16* row, bool valid) {
  const WideLane L;
  #pragma unroll
  for (int a = 0; a < 2; ++a)
    #pragma unroll
    for (int q = 0; q < 4; q += 2) {
      uint32_t pk[2][2];                       // quads q and q + 1, two words each
      #pragma unroll
      for (int j = 0; j < 2; ++j) {
        bf16x4 b;
        #pragma unroll
        for (int i = 0; i < 4; ++i) b[i] = (bf16)v[a][tt][4 * (q + j) + i];
        __builtin_memcpy(pk[j], &b, 8);
      }
      // lanes < 32 end with the 8 dims of quad q, the others with those of quad q + 1
      const auto w0 = __builtin_amdgcn_permlane32_swap(pk[0][0], pk[1][0], false, false);
      const auto w1 = __builtin_amdgcn_permlane32_swap(pk[0][1], pk[1][1], false, false);
      const uint32_t o[4] = {(uint32_t)w0[0], (uint32_t)w1[0], (uint32_t)w0[1], (uint32_t)w1[1]};
      if (valid) {
        bf16x8 ov;
        __builtin_memcpy(&ov, o, 16);
        *reinterpret_cast<bf16x8*>(row + 32 * (L.dh + 2 * a) + 8 * (q + L.hl)) = ov;
      }
    }
}

}  // namespace dspark
