// Verify-layer prologue for gfx950: the Qwen3 attention steps that produce
// the kernel's inputs, in one launch per layer.
//
//   q = RoPE(RMSNorm_q(x Wq^T)),  k = RoPE(RMSNorm_k(x Wk^T)),  v = x Wv^T
//
// per 128-dim head (16 query heads, 8 KV heads), RMSNorm y = w x /
// sqrt(mean(x^2) + eps), RoPE in the rotate-half form with angles
// pos * inv_freq[d] (float32, the model's table).  This is what transformers'
// Qwen3Attention computes before the cache update / attention call used by
// dspark_qwen/persistent_qwen_target.py:45-95; the K/V rows can be written
// straight into the transaction scratch, replacing stage_layer's copy
// (dspark_qwen/persistent_target_kv.py:427-438).
//
// The rotary cos/sin either come from a table of the transaction's rows
// (dspark_rope_table: computed once and shared by every layer, as the
// model computes its position embeddings once per forward) or are formed
// in the epilogue from the positions; both give the same bits.
//
// Work: one workgroup per (head, 64- or 32-token tile) on the shared 32x32x16
// MFMA tile (head_gemm.h); all its waves run the epilogue on 16 dims of one
// token per lane.  Accumulation and the epilogue are FP32; outputs are
// rounded to bf16 once.
#include "wide_gemm.h"

namespace dspark {

struct PrologueArgs {
  const bf16* x;             // [T, hidden]
  const bf16* wq;            // [16*128, hidden]  (nn.Linear weight layout)
  const bf16* wk;            // [8*128, hidden]
  const bf16* wv;            // [8*128, hidden]
  const bf16* q_norm;        // [128]
  const bf16* k_norm;        // [128]
  const float* inv_freq;     // [64]
  const int64_t* positions;  // [T] absolute positions
  const float* rope;         // optional [T][128]: cos of the 64 angles, then their sin
  bf16* q_out;               // [T, 16, 128]
  bf16* k_out;               // token rows of 8*128, kv_row_stride apart
  bf16* v_out;
  int64_t kv_row_stride;     // elements
  int tokens;
  int hidden;
  float eps;
};

// grid: 32 heads (0-15 q, 16-23 k, 24-31 v) x ceil(T / (32 TG)) token tiles, one
// dimension (see the XCD mapping below); 4 TG waves.
template <int TG>
__global__ __launch_bounds__(4 * TG * WAVE) void qkv_prologue_kernel(PrologueArgs a) {
  __shared__ __attribute__((aligned(16))) unsigned char smem[HeadRing<TG>::SMEM];
  // XCD-aware placement: workgroups are dealt round-robin over the 8 XCDs
  // (each with its own L2), so the token tiles of one head are given ids
  // that share id % 8 - the head's weight slice is then fetched from HBM by
  // one L2 and served to all of its tiles from there.
  const int tiles = (a.tokens + 32 * TG - 1) / (32 * TG);
  const int xcd = blockIdx.x & 7;
  const int slot = blockIdx.x >> 3;
  const int head = xcd + 8 * (slot / tiles);
  const int t0 = (slot % tiles) * (32 * TG);
  const int kind = head < HQ ? 0 : (head < HQ + HKV ? 1 : 2);       // workgroup-uniform
  const int hh = kind == 0 ? head : (kind == 1 ? head - HQ : head - HQ - HKV);
  const bf16* w = (kind == 0 ? a.wq : (kind == 1 ? a.wk : a.wv)) + (size_t)hh * HD * a.hidden;

  const HeadLaneOf<TG> L;
  const int row = t0 + L.token();
  const int tok = min(row, a.tokens - 1);
  HeadNormWOf<TG> nw;
  HeadRopeOf<TG> rope;
  float pos = 0.f;
  float v[2][8];
  float ss;
  // the epilogue's operands are fetched while the K halves are exchanged
  head_tile_gemm<false, TG>(w, a.x, a.tokens, a.hidden, t0, smem, v, ss, [&]() {
    if (kind < 2) {
      nw.load(kind == 0 ? a.q_norm : a.k_norm);
      if (a.rope) rope.load(a.rope + (size_t)tok * 128);
      else pos = (float)a.positions[tok];
    }
  });
  if (kind < 2) {
    head_rms_norm(v, nw, a.eps, head_row_sumsq<TG>(v, smem));
    if (!a.rope) rope.compute(a.inv_freq, pos);
    head_rope(v, rope);
  }
  bf16* out = kind == 0 ? a.q_out + (size_t)tok * Q_ROW : (kind == 1 ? a.k_out : a.v_out) + (size_t)tok * a.kv_row_stride;
  head_store<TG>(v, out + (size_t)hh * HD, row < a.tokens);
}

// The same for many tokens: 128-token tiles (wide_gemm.h), two workgroups per CU.
template <bool TABLE>
__global__ __launch_bounds__(WG_WAVES * WAVE, 2) void qkv_prologue_wide_kernel(PrologueArgs a) {
  __shared__ __attribute__((aligned(16))) unsigned char smem[WG_SMEM];
  const int tiles = (a.tokens + WG_TOKENS - 1) / WG_TOKENS;
  const int xcd = blockIdx.x & 7;                // a head's tiles share id % 8 (see above)
  const int slot = blockIdx.x >> 3;
  const int head = xcd + 8 * (slot & 3);
  const int t0 = (slot >> 2) * WG_TOKENS;
  const int kind = head < HQ ? 0 : (head < HQ + HKV ? 1 : 2);       // workgroup-uniform
  const int hh = kind == 0 ? head : (kind == 1 ? head - HQ : head - HQ - HKV);
  const bf16* w = (kind == 0 ? a.wq : (kind == 1 ? a.wk : a.wv)) + (size_t)hh * HD * a.hidden;
  f32x16 v[2][2];
  wide_tile_gemm(w, a.x, a.tokens, a.hidden, t0, smem, v);
  const WideLane L;
  if (kind < 2) {
    int tok[2];
    float pos[2];
    #pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
      tok[tt] = min(t0 + L.token(tt), a.tokens - 1);
      pos[tt] = TABLE ? 0.f : (float)a.positions[tok[tt]];
    }
    wide_norm_rope(v, kind == 0 ? a.q_norm : a.k_norm, a.eps, smem, [&](int tt, int dim, f32x4& c, f32x4& s) {
      if (TABLE) {
        const float* row = a.rope + (size_t)tok[tt] * 128 + dim;
        c = *reinterpret_cast<const f32x4*>(row);
        s = *reinterpret_cast<const f32x4*>(row + 64);
      } else {
        #pragma unroll
        for (int i = 0; i < 4; ++i) {
          float sn, cs;
          sincosf(pos[tt] * a.inv_freq[dim + i], &sn, &cs);
          c[i] = cs;
          s[i] = sn;
        }
      }
    });
  }
  #pragma unroll
  for (int tt = 0; tt < 2; ++tt) {
    const int row = t0 + L.token(tt);
    const int tok = min(row, a.tokens - 1);
    bf16* out = kind == 0 ? a.q_out + (size_t)tok * Q_ROW : (kind == 1 ? a.k_out : a.v_out) + (size_t)tok * a.kv_row_stride;
    wide_store(v, tt, out + (size_t)hh * HD, row < a.tokens);
  }
}

// cos and sin of pos[t] * inv_freq[d] (FP32 angle, d < 64) for every row:
// table[t][d] = cos, table[t][64 + d] = sin.
__global__ __launch_bounds__(256) void rope_table_kernel(const float* __restrict__ inv_freq,
                                                         const int64_t* __restrict__ positions, int tokens,
                                                         float* __restrict__ table) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= tokens * 64) return;
  const int t = i >> 6, d = i & 63;
  float s, c;
  sincosf((float)positions[t] * inv_freq[d], &s, &c);
  table[(size_t)t * 128 + d] = c;
  table[(size_t)t * 128 + 64 + d] = s;
}

}  // namespace dspark

using namespace dspark;

// From here on the 64-token tiles (one workgroup per CU) need a second round of
// the 256 CUs.  64- against 128-token tiles, us per launch at hidden 1,024: 512
// tokens 10.3 / 14.8, 640 17.5 / 15.2, 1,024 19.0 / 16.8, 2,048 38.6 / 24.7,
// 4,096 73 / 45, 8,192 141 / 88.
constexpr int PROLOGUE_WIDE_TOKENS = 513;

// Up to here 32-token tiles are one round of the 256 CUs (one workgroup each)
// and stream a sixth fewer bytes per workgroup with more of them in flight than
// 64-token tiles on half of the CUs.  32- against 64-token tiles, us per
// launch at hidden 1,024 over the weights of 28 layers: 7 tokens 9.6 / 10.2, 64
// 10.4 / 12.1, 224 10.3 / 11.6, 256 10.3 / 11.8.
constexpr int PROLOGUE_NARROW_TOKENS = 256;

extern "C" int dspark_qkv_prologue(const void* x, const void* wq, const void* wk, const void* wv,
                                   const void* q_norm, const void* k_norm, const float* inv_freq,
                                   const int64_t* positions, const float* rope, int tokens, int hidden, float eps,
                                   void* q_out, void* k_out, void* v_out, int64_t kv_row_stride, void* stream) {
  clear_error();
  DSPARK_REQUIRE(x && wq && wk && wv && q_norm && k_norm && inv_freq && positions && q_out && k_out && v_out,
                 "null pointer argument");
  DSPARK_REQUIRE(tokens >= 1 && hidden >= HG_COLS && hidden % HG_COLS == 0, "need tokens >= 1 and hidden a multiple of %d",
                 HG_COLS);
  DSPARK_REQUIRE(kv_row_stride >= KV_ROW && kv_row_stride % 8 == 0, "kv_row_stride must be >= 1024 and a multiple of 8");
  DSPARK_REQUIRE(eps > 0.f, "eps must be positive");
  const uintptr_t any = (uintptr_t)x | (uintptr_t)wq | (uintptr_t)wk | (uintptr_t)wv | (uintptr_t)q_out |
                        (uintptr_t)k_out | (uintptr_t)v_out | (uintptr_t)inv_freq | (uintptr_t)rope;
  DSPARK_REQUIRE(any % 16 == 0, "tensors must be 16-byte aligned");
  DSPARK_REQUIRE(((uintptr_t)q_norm | (uintptr_t)k_norm) % 8 == 0, "norm weights must be 8-byte aligned");
  PrologueArgs a{static_cast<const bf16*>(x), static_cast<const bf16*>(wq), static_cast<const bf16*>(wk),
                 static_cast<const bf16*>(wv), static_cast<const bf16*>(q_norm), static_cast<const bf16*>(k_norm),
                 inv_freq, positions, rope, static_cast<bf16*>(q_out), static_cast<bf16*>(k_out),
                 static_cast<bf16*>(v_out), kv_row_stride, tokens, hidden, eps};
  if (tokens >= PROLOGUE_WIDE_TOKENS) {
    const dim3 grid((HQ + 2 * HKV) * ((tokens + WG_TOKENS - 1) / WG_TOKENS));
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (rope) hipLaunchKernelGGL(qkv_prologue_wide_kernel<true>, grid, dim3(WG_WAVES * WAVE), 0, s, a);
    else hipLaunchKernelGGL(qkv_prologue_wide_kernel<false>, grid, dim3(WG_WAVES * WAVE), 0, s, a);
    return launch_status("qkv_prologue_wide_kernel");
  }
  if (tokens <= PROLOGUE_NARROW_TOKENS) {
    hipLaunchKernelGGL(qkv_prologue_kernel<1>, dim3((HQ + 2 * HKV) * ((tokens + 31) / 32)), dim3(4 * WAVE), 0,
                       static_cast<hipStream_t>(stream), a);
    return launch_status("qkv_prologue_kernel");
  }
  hipLaunchKernelGGL(qkv_prologue_kernel<2>, dim3((HQ + 2 * HKV) * ((tokens + HG_TOKENS - 1) / HG_TOKENS)),
                     dim3(HG_WAVES * WAVE), 0, static_cast<hipStream_t>(stream), a);
  return launch_status("qkv_prologue_kernel");
}

extern "C" int dspark_rope_table(const float* inv_freq, const int64_t* positions, int tokens, float* table,
                                 void* stream) {
  clear_error();
  DSPARK_REQUIRE(inv_freq && positions && table, "null pointer argument");
  DSPARK_REQUIRE(tokens >= 1 && tokens <= (1 << 24), "tokens must be in [1, 2^24]");
  hipLaunchKernelGGL(rope_table_kernel, dim3((unsigned)((tokens * 64 + 255) / 256)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), inv_freq, positions, tokens, table);
  return launch_status("rope_table_kernel");
}
