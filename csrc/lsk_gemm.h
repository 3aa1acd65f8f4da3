// Shared by the GEMM tiers: the launch kinds' epilogues and the entry point of the many-token tier.
#pragma once

#include "lsk_common.h"

#define EPI_PARTIAL 3
#define EPI_ARGMAX 4
#define EPI_QKV 5

// Fused qkv epilogue (EPI_QKV): the qkv projection's output goes straight to RoPE and the caches instead of through
// K-slice partials and the RoPE + append kernel.  The weight is packed with its q and k row groups RoPE-paired
// (lsk_pack_weight_qkv): within each head of D rows (G = D / 16 groups) packed group 2 j holds dims 16 j .. 16 j + 15
// and packed group 2 j + 1 dims D / 2 + 16 j .. (the rotation partners), so a tile of two (or four) row groups holds
// whole rotation pairs and one lane owns both values of a pair.  v rows keep their order.
struct QkvRope {
  uint16_t* q;            // [N, Hq, D] RoPE-rotated queries
  uint16_t* kc;           // K cache, fragment-major 32-position blocks (k_cache_offset)
  uint16_t* vc;           // V cache, transposed 32-position blocks
  const float* cos_tab;   // [tab_len, D] fp32
  const float* sin_tab;
  const int32_t* rows;    // [N] cache row of each token
  const int32_t* pos;     // [N] position of each token
  int hq, hkv, d, max_batch, max_seq, tab_len;
};

// Token m's values x_lo, x_hi of packed row groups G (even) and G + 1, row w16 of each: a RoPE pair for q / k (stored
// rotated to q or the K cache), two v dims 16 apart otherwise (stored to the V cache), with the RoPE + append
// kernel's arithmetic (rope_pair) and indexing.
__device__ __forceinline__ void qkv_rope_store(const QkvRope& qa, int m, int G, int w16, float x_lo, float x_hi) {
  const int D = qa.d, GH = D >> 4, half = D >> 1;
  const int row = qa.rows[m], p = qa.pos[m];
  if (row < 0 || row >= qa.max_batch || p < 0 || p >= qa.max_seq || p >= qa.tab_len) return;  // host validates too
  const int kg = (qa.hq + qa.hkv) * GH;
  if (G < kg) {
    const int h = G / GH, d1 = 16 * ((G - h * GH) >> 1) + w16;
    float o1, o2;
    rope_pair<uint16_t>(x_lo, x_hi, qa.cos_tab + (long)p * D, qa.sin_tab + (long)p * D, d1, half, o1, o2);
    if (h < qa.hq) {
      uint16_t* dst = qa.q + ((long)m * qa.hq + h) * D;
      dst[d1] = f2bf(o1);
      dst[d1 + half] = f2bf(o2);
    } else {
      uint16_t* dst = qa.kc + ((long)row * qa.hkv + (h - qa.hq)) * (long)qa.max_seq * D;
      dst[k_cache_offset<uint16_t>(p, d1, D)] = f2bf(o1);
      dst[k_cache_offset<uint16_t>(p, d1 + half, D)] = f2bf(o2);
    }
  } else {
    const int gv = G - kg, h = gv / GH, d1 = 16 * (gv - h * GH) + w16;
    uint16_t* dst = qa.vc + ((long)row * qa.hkv + h) * (long)D * qa.max_seq + (long)(p >> 5) * 32 * D + (p & 31);
    dst[(long)d1 * 32] = f2bf(x_lo);
    dst[(long)(d1 + 16) * 32] = f2bf(x_hi);
  }
}

__device__ __forceinline__ float silu_f(float x) { return x / (1.0f + lsk_exp(-x)); }

#define LSK_DEEP_MIN_TOKENS 256     // below: the wide tier
#define LSK_DEEP_ALWAYS_TOKENS 900  // from here on the many-token tier unless its estimate is the higher one
// Many-token tier (lsk_gemm_deep.hip) over a fragment-major A: whether it takes a launch, and the launch.  Same sums as
// the other tiers.
struct DeepCfg {
  int mg, m_blocks, split;  // token groups per workgroup (0: not taken), token blocks, workgroups sharing a tile's slices
  double us;                // estimated time
};
DeepCfg lsk_deep_plan(int epi, int M, int N, int K, int ks);
void lsk_gemm_deep(const DeepCfg& cfg, int epi, hipStream_t s, const uint16_t* A, const uint16_t* W, uint16_t* C, long ldc,
                   int c_nks, const uint16_t* R, float* P, float* av, int* ai, int M, int N, int K, int ffn, int ks,
                   const QkvRope& qa);
