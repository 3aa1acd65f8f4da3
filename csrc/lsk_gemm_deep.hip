// Many-token tier of the bf16 GEMMs (prefill and large verify segments): C = epilogue(A W^T) with a fragment-major A.
//
// From a few hundred tokens on these products are bound by the matrix cores and by what feeds them, not by the weight
// stream.  The wide tier re-reads its activations from L2 for every 64 weight rows (400-800 TFLOP/s); here a workgroup of
// four waves owns 256 weight rows (64 per wave, read straight into registers three k-steps ahead: no other wave needs
// them) x MG 16-token groups (staged through LDS and shared by the four waves).  MG = 8 and 6 run one workgroup per CU
// (a wave holds up to 32 tiles in two accumulator sets), MG = 4 two.  MI355X, 4001 tokens of the 8B shape,
// cold weights, graph-timed (the wide tier first): qkv 403 -> 203 us, o with its norm 430 -> 188, w13 1198 -> 915 (1030
// TFLOP/s; the clock falls to 1.9 GHz there), w2 with its norm 1155 -> 450.
//
// Exactly the decode kernel's sums, as the wide tier: within a K slice the chunks of 128 k are visited class by class
// (0, 4, 8, ...; 1, 5, ...; ...), each class into a fresh accumulator `cur` that is added to the running `tot` at its end.
#include <type_traits>

#include "lsk_common.h"
#include "lsk_gemm.h"
#include "../include/lsk.h"

// Rounding through bf16 by the hardware conversion: f2bf's result for every number (a NaN stays one).
__device__ __forceinline__ float hbf(float f) { return (float)(__bf16)f; }
__device__ __forceinline__ lsk_u32x2_u pack4(const float* v) {
  typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
  const bf16x4 b = {(__bf16)v[0], (__bf16)v[1], (__bf16)v[2], (__bf16)v[3]};
  return __builtin_bit_cast(lsk_u32x2_u, b);
}

// qkv_rope_store for rows w16 .. w16 + 3 (w16 % 4 == 0) of the pair of row groups: four consecutive dims of a head, so
// the table rows are read and the q / K values stored 16 and 8 bytes at a time (at any address their elements align).
__device__ __forceinline__ void qkv_rope_store4(const QkvRope& qa, int m, int row, int p, int G, int w16, const float* lo,
                                                const float* hi) {
  const int D = qa.d, GH = D >> 4, half = D >> 1;
  if (row < 0 || row >= qa.max_batch || p < 0 || p >= qa.max_seq || p >= qa.tab_len) return;  // host validates too
  const int kg = (qa.hq + qa.hkv) * GH;
  if (G < kg) {
    const int h = G / GH, d1 = 16 * ((G - h * GH) >> 1) + w16;
    const float* ct = qa.cos_tab + (long)p * D + d1;
    const float* st = qa.sin_tab + (long)p * D + d1;
    const lsk_f32x4 cv1 = *(const lsk_f32x4_u*)ct, cv2 = *(const lsk_f32x4_u*)(ct + half);
    const lsk_f32x4 sv1 = *(const lsk_f32x4_u*)st, sv2 = *(const lsk_f32x4_u*)(st + half);
    float o1[4], o2[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {  // rope_pair's roundings
      o1[i] = hbf(lo[i] * hbf(cv1[i])) + hbf((-hi[i]) * hbf(sv1[i]));
      o2[i] = hbf(hi[i] * hbf(cv2[i])) + hbf(lo[i] * hbf(sv2[i]));
    }
    uint16_t *dst1, *dst2;
    if (h < qa.hq) {
      dst1 = qa.q + ((long)m * qa.hq + h) * D + d1;
      dst2 = dst1 + half;
    } else {
      uint16_t* base = qa.kc + ((long)row * qa.hkv + (h - qa.hq)) * (long)qa.max_seq * D;
      dst1 = base + k_cache_offset<uint16_t>(p, d1, D);
      dst2 = base + k_cache_offset<uint16_t>(p, d1 + half, D);
    }
    *(lsk_u32x2_u*)dst1 = pack4(o1);
    *(lsk_u32x2_u*)dst2 = pack4(o2);
  } else {
    const int gv = G - kg, h = gv / GH, d1 = 16 * (gv - h * GH) + w16;
    uint16_t* dst = qa.vc + ((long)row * qa.hkv + h) * (long)D * qa.max_seq + (long)(p >> 5) * 32 * D + (p & 31);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      dst[(long)(d1 + i) * 32] = f2bf(lo[i]);
      dst[(long)(d1 + i + 16) * 32] = f2bf(hi[i]);
    }
  }
}

template <int MG, int EPI>
__global__ __launch_bounds__(256, MG <= 4 ? 2 : 1) void gemm_deep_kernel(const uint16_t* __restrict__ A, const uint16_t* __restrict__ W,
                                                           uint16_t* C, long ldc, int c_nks,
                                                           const uint16_t* R, float* __restrict__ P,
                                                           float* __restrict__ amax_v, int* __restrict__ amax_i, int M, int N, int K, int ffn,
                                                           int kslice, int n_tiles, int m_blocks, int ks, int split,
                                                           QkvRope qa) {
  constexpr bool SILU = EPI == LSK_EPI_SILU_MUL;
  constexpr int NG = 4;                    // weight row groups per wave (silu-mul: 2 gate + 2 up)
  constexpr int WN = SILU ? 2 : 4;         // output row groups per wave
  constexpr bool SUM = EPI == LSK_EPI_RESIDUAL;  // the K slices are summed here (one workgroup walks all of them)
  constexpr int PU = MG / 2;               // 16-byte pieces per thread of half a staged chunk
  constexpr int UNIT = MG * 2 * 512;       // elements of half a chunk: MG groups x 2 k-steps
  static_assert(MG % 2 == 0 && MG <= 8, "staging split");
  __shared__ __attribute__((aligned(16))) uint16_t al0[UNIT], al1[UNIT];
  __shared__ __attribute__((aligned(16))) float slice_sum[SUM ? NG * MG * 1024 : 4];  // thread-private, 4 floats per (g, t)

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, lg = lane >> 4;
  // workgroup id -> (row tile, token block, slice range).  The launch's pieces are ordered 8 token blocks at a time, row
  // tiles within them, token blocks innermost, and each XCD takes one run of that order: its 32 concurrent workgroups
  // then share about 4 row tiles x 8 token blocks through its L2.
  const int total = n_tiles * m_blocks * split, run = (total + 7) >> 3;
  const int lin = (blockIdx.x & 7) * run + (blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= run || lin >= total) return;
  const int per = n_tiles * split;
  const int sup = lin / (8 * per), rem = lin - sup * 8 * per;
  const int mcount = min(8, m_blocks - 8 * sup);
  const int ni = rem / mcount, mb = 8 * sup + (rem - ni * mcount);
  const int tn = ni / split, sp = ni - tn * split;
  const int sl = ks / split;               // slices of this workgroup: [sp sl, (sp + 1) sl)
  const int s_first = sp * sl;
  const int nks = K >> 5, nfull = kslice >> 7;
  const int gtot = (M + 15) >> 4;
  // token groups of the block, dealt evenly
  const int gq = gtot / m_blocks, gr = gtot - gq * m_blocks;
  const int g0 = mb * gq + min(mb, gr), gn = gq + (mb < gr ? 1 : 0);

  const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(
      (void*)W, (short)0, (int)((unsigned)((SILU ? 2 * ffn : N) >> 4) * (unsigned)nks * 1024u), LSK_BUFFER_RSRC_WORD3);
  const __amdgpu_buffer_rsrc_t ar = __builtin_amdgcn_make_buffer_rsrc(
      (void*)A, (short)0, (int)((unsigned)gtot * (unsigned)nks * 1024u), LSK_BUFFER_RSRC_WORD3);
  const int r0 = tn * (SILU ? 8 : 16) + wave * WN;  // this wave's first output row group
  unsigned wofs[NG];
#pragma unroll
  for (int g = 0; g < NG; ++g)
    wofs[g] = (unsigned)((g < WN ? r0 + g : (ffn >> 4) + r0 + g - WN) * nks) * 1024u;
  // staging: half a chunk holds k-steps 2 u, 2 u + 1 of every group; its fragment f = wave + 4 p is group f / 2, k-step
  // 2 u + f % 2
  unsigned aofs[PU];
#pragma unroll
  for (int p = 0; p < PU; ++p)
    aofs[p] = (unsigned)(min(g0 + min((wave >> 1) + 2 * p, gn - 1), gtot - 1) * nks + (wave & 1)) * 1024u;
  const int lofs = 16 * lane;

  lsk_f32x4 cur[NG][MG], tot[NG][MG];
  lsk_bf16x8 wf[4][NG], af[2][MG];
  lsk_i32x4 st[2][PU];
  const lsk_f32x4 zero = {0.f, 0.f, 0.f, 0.f}, nzero = {-0.f, -0.f, -0.f, -0.f};
#pragma unroll
  for (int g = 0; g < NG; ++g)
#pragma unroll
    for (int t = 0; t < MG; ++t) {
      cur[g][t] = zero;
      tot[g][t] = nzero;  // -0 + x is x, bit for bit
    }
  lsk_f32x4* const sums = (lsk_f32x4*)slice_sum + tid;
  if constexpr (SUM) {
#pragma unroll
    for (int f = 0; f < NG * MG; ++f) sums[f * 256] = nzero;
  }
  // chunk sequence: slices in order; within a slice class q = 0..3 holds chunks q, q + 4, ...
  struct Seq {
    int s, q, c;
  };
  auto next = [&](Seq x) {
    x.c += 4;
    if (x.c >= nfull) {
      x.q += 1;
      x.c = x.q;
      if (x.q == 4 || x.c >= nfull) {
        x.q = 0;
        x.c = 0;
        x.s += 1;
      }
    }
    return x;
  };
  const int s_end = s_first + sl;
  // byte offset of a chunk's first k-step within a row group's fragments; past the last chunk (the loads that run ahead
  // of the loop's end): a chunk of the last slice again, loaded and never multiplied
  auto kofs = [&](const Seq& x) { return (unsigned)((min(x.s, s_end - 1) * (kslice >> 5)) + x.c * 4) * 1024u; };

  auto load_w = [&](lsk_bf16x8 (&w)[NG], unsigned ko, int ksi) {
#pragma unroll
    for (int g = 0; g < NG; ++g)
      w[g] = __builtin_bit_cast(lsk_bf16x8,
                                __builtin_amdgcn_raw_buffer_load_b128(wr, lofs + ksi * 1024, (int)(wofs[g] + ko), 0));
  };
  auto load_st = [&](unsigned ko, int u, int p) {
    st[u][p] = __builtin_bit_cast(
        lsk_i32x4, __builtin_amdgcn_raw_buffer_load_b128(ar, lofs + u * 2048, (int)(aofs[p] + ko), 0));
  };
  auto put_st = [&](int u, int p) {
    *(lsk_i32x4*)(&(u ? al1 : al0)[(wave + 4 * p) * 512 + 8 * lane]) = st[u][p];
  };
  auto read_a = [&](int ksi, int t) {
    return *(const lsk_bf16x8*)(&(ksi >= 2 ? al1 : al0)[(t * 2 + (ksi & 1)) * 512 + 8 * lane]);
  };
  auto fold = [&]() {  // closes a class
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
      for (int t = 0; t < MG; ++t) {
        tot[g][t] += cur[g][t];
        cur[g][t] = zero;
      }
  };

  Seq x0{s_first, 0, 0};
  Seq x1 = next(x0), x2 = next(x1);
  {
    const unsigned k0 = kofs(x0), k1 = kofs(x1);
#pragma unroll
    for (int p = 0; p < PU; ++p) load_st(k0, 0, p);
#pragma unroll
    for (int i = 0; i < 3; ++i) load_w(wf[i], k0, i);
#pragma unroll
    for (int p = 0; p < PU; ++p) put_st(0, p);
#pragma unroll
    for (int p = 0; p < PU; ++p) load_st(k0, 1, p);
#pragma unroll
    for (int p = 0; p < PU; ++p) load_st(k1, 0, p);
  }
  __syncthreads();
#pragma unroll
  for (int t = 0; t < MG; ++t) af[0][t] = read_a(0, t);
  // one k-step in MG slots of four MFMAs: a slot also reads one A fragment of the next step, issues the step's global
  // loads one or two at a time (a W fragment per row group; with LU >= 0 the pieces of half chunk LU) and, with
  // PUT >= 0, writes the pieces of half chunk PUT to LDS.  The order is fixed (the scheduler would bunch each kind
  // together): the four waves run in step, and bunched loads queue for the address unit.
  using std::integral_constant;
  auto step = [&](lsk_bf16x8 (&wn)[NG], unsigned kw, int wks, const lsk_bf16x8 (&w)[NG], const lsk_bf16x8 (&a)[MG],
                  lsk_bf16x8 (&an)[MG], int rks, unsigned kp, auto put_c, auto lu_c) {
    constexpr int PUT = decltype(put_c)::value, LU = decltype(lu_c)::value;
    auto mf = [&](int f) {
      const int g = f / MG, t = f - g * MG;
      cur[g][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[g], a[t], cur[g][t], 0, 0, 0);
    };
    auto ld = [&](int l) {
      if (l < NG)
        wn[l] = __builtin_bit_cast(
            lsk_bf16x8, __builtin_amdgcn_raw_buffer_load_b128(wr, lofs + wks * 1024, (int)(wofs[l] + kw), 0));
      else if (LU >= 0 && l < NG + PU)
        load_st(kp, LU, l - NG);
    };
#pragma unroll
    for (int i = 0; i < MG; ++i) {
      an[i] = read_a(rks, i);
      mf(4 * i);
      mf(4 * i + 1);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (MG < 8) {
        ld(2 * i);
        ld(2 * i + 1);
      } else {
        ld(i);
      }
      mf(4 * i + 2);
      if (PUT >= 0 && i >= MG - PU) put_st(PUT, i - (MG - PU));
      mf(4 * i + 3);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  auto chunk = [&]() {
    const unsigned k0 = kofs(x0), k1 = kofs(x1), k2 = kofs(x2);
    const integral_constant<int, 0> u0;
    const integral_constant<int, 1> u1;
    const integral_constant<int, -1> no;
    __builtin_amdgcn_sched_barrier(0);
    step(wf[3], k0, 3, wf[0], af[0], af[1], 1, 0, u1, no);
    __syncthreads();
    step(wf[0], k1, 0, wf[1], af[1], af[0], 2, k1, no, u1);
    step(wf[1], k1, 1, wf[2], af[0], af[1], 3, 0, u0, no);
    __syncthreads();
    step(wf[2], k1, 2, wf[3], af[1], af[0], 0, k2, no, u0);
  };
  const float empty = nfull < 4 ? 0.f : -0.f;  // classes without chunks add +0
  for (;;) {
    bool same;
    int s;
    do {  // the chunks of a class
      chunk();
      s = x0.s;
      same = x1.q == x0.q && x1.s == x0.s;
      x0 = x1;
      x1 = x2;
      x2 = next(x2);
    } while (same);
    fold();
    if (x0.s != s) {
      if constexpr (EPI == EPI_PARTIAL) {
#pragma unroll
        for (int t = 0; t < MG; ++t) {
          const int m = (g0 + t) * 16 + l16;
          if (t < gn && m < M) {
#pragma unroll
            for (int g = 0; g < NG; ++g)
              *(float4*)(P + ((long)s * M + m) * N + (r0 + g) * 16 + 4 * lg) =
                  make_float4(tot[g][t][0] + empty, tot[g][t][1] + empty, tot[g][t][2] + empty, tot[g][t][3] + empty);
          }
        }
      }
      if constexpr (SUM) {
#pragma unroll
        for (int f = 0; f < NG * MG; ++f) {
          sums[f * 256] = sums[f * 256] + (tot[f / MG][f % MG] + (lsk_f32x4){empty, empty, empty, empty});
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      if constexpr (EPI == EPI_PARTIAL || SUM) {
#pragma unroll
        for (int g = 0; g < NG; ++g)
#pragma unroll
          for (int t = 0; t < MG; ++t) tot[g][t] = nzero;
      }
      if (x0.s >= s_end) break;
    }
  }
  if constexpr (EPI == LSK_EPI_SILU_MUL) {
#pragma unroll
    for (int t = 0; t < MG; ++t) {
      const int m = (g0 + t) * 16 + l16;
      if (t >= gn || m >= M) continue;
#pragma unroll
      for (int g = 0; g < WN; ++g) {
        const int n = (r0 + g) * 16 + 4 * lg;
        float o[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
          o[i] = hbf(silu_f(hbf(tot[g][t][i] + empty))) * hbf(tot[g + WN][t][i] + empty);
        *(lsk_u32x2_u*)(C + (c_nks > 0 ? lsk_frag_off(m, n, c_nks) : (long)m * ldc + n)) = pack4(o);
      }
    }
  } else if constexpr (EPI == EPI_QKV) {
#pragma unroll
    for (int t = 0; t < MG; ++t) {
      const int m = (g0 + t) * 16 + l16;
      if (t >= gn || m >= M) continue;
      const int row = qa.rows[m], p = qa.pos[m];
#pragma unroll
      for (int pp = 0; pp < NG / 2; ++pp) {
        float lo[4], hi[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          lo[i] = hbf(tot[2 * pp][t][i] + empty);
          hi[i] = hbf(tot[2 * pp + 1][t][i] + empty);
        }
        qkv_rope_store4(qa, m, row, p, r0 + 2 * pp, 4 * lg, lo, hi);
      }
    }
  } else if constexpr (SUM) {
#pragma unroll
    for (int t = 0; t < MG; ++t) {
      const int m = (g0 + t) * 16 + l16;
      if (t >= gn || m >= M) continue;
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        const long off = (long)m * ldc + (r0 + g) * 16 + 4 * lg;
        const lsk_u32x2_u x = *(const lsk_u32x2_u*)(R + off);
        float o[4] = {__uint_as_float(x.x << 16), __uint_as_float(x.x & 0xffff0000u), __uint_as_float(x.y << 16),
                      __uint_as_float(x.y & 0xffff0000u)};
        const lsk_f32x4 v = sums[(g * MG + t) * 256];
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = o[i] + hbf(v[i]);
        *(lsk_u32x2_u*)(C + off) = pack4(o);
      }
    }
  } else if constexpr (EPI == EPI_ARGMAX) {
    const int nt64 = N >> 6, t64 = tn * 4 + wave;  // a wave's 64 rows are one argmax tile
#pragma unroll
    for (int t = 0; t < MG; ++t) {
      const int m = (g0 + t) * 16 + l16;
      const bool ok = t < gn && m < M;
      float best = -INFINITY;
      int bi = -1;
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        const int n = (r0 + g) * 16 + 4 * lg;
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          v[i] = rbf(tot[g][t][i] + empty);
          if (bi < 0 || v[i] > best) {
            best = v[i];
            bi = n + i;
          }
        }
        if (C != nullptr && ok) {
          uint2 pk;
          pk.x = (uint32_t)f2bf(v[0]) | ((uint32_t)f2bf(v[1]) << 16);
          pk.y = (uint32_t)f2bf(v[2]) | ((uint32_t)f2bf(v[3]) << 16);
          *(uint2*)(C + (long)m * ldc + n) = pk;
        }
      }
#pragma unroll
      for (int o = 16; o <= 32; o <<= 1) {
        const float ov = __shfl_xor(best, o, 64);
        const int oi = __shfl_xor(bi, o, 64);
        if (oi >= 0 && (bi < 0 || ov > best || (ov == best && oi < bi))) {
          best = ov;
          bi = oi;
        }
      }
      if (lg == 0 && ok) {
        amax_v[(long)m * nt64 + t64] = best;
        amax_i[(long)m * nt64 + t64] = bi;
      }
    }
  }
}

// Configuration of a launch (N: output columns, ffn for silu-mul) and its estimated time.  A workgroup of mg token groups
// walks c chunks of 128 k; the times below are of the busiest CU, fitted to MI355X measurements over the 1B, 7B and 8B
// projections at 256-4001 tokens:
//   mg = 8 / 6 (one workgroup per CU): 1.7 c + 12 (a single round: 6 with partials, else 14) / 1.25 c + 13 us each (mg = 6:
//     1.4 c up to 1024 tokens)
//   mg = 4 (two per CU): 2.1 c + 3 us per pair (2.5 c up to 1024 tokens and with partials), a lone one 1.3 c + 10 us (1.5 c +
//     9 summing its slices)
//   the LM head, whose logits and maxima cost more per workgroup: 1.8 c + 12, 1.66 c + 10, 2.45 c + 8 and 1.4 c + 9
// plus 3 us per slice summed, plus the stores of the partials.  Larger mg moves fewer bytes per product (24, 22 and 20 KiB
// per k-step for 8, 6 and 4 x 16 tokens of 256 rows), smaller mg splits a segment into more workgroups and overlaps one
// workgroup's epilogue with the other's products: w13 of the 8B shape at 4001 tokens 920 / 992 / 943 us, at 512 tokens
// 147 / 180 / 172 us, w13 of the 1B shape at 1517 tokens 122 / 124 / 104 us for mg = 8 / 6 / 4.
DeepCfg lsk_deep_plan(int epi, int M, int N, int K, int ks) {
  const DeepCfg none{0, 0, 0, 0.0};
  const bool silu = epi == LSK_EPI_SILU_MUL, partial = epi == EPI_PARTIAL, sum = epi == LSK_EPI_RESIDUAL;
  const bool head = epi == EPI_ARGMAX;
  const int cols = silu ? 128 : 256;
  if (M < LSK_DEEP_MIN_TOKENS || ks < 1 || N % cols != 0 || K % ks != 0 || (K / ks) % 128 != 0) return none;
  // 32-bit byte offsets into both operands
  if ((silu ? 2.0 : 1.0) * N * K * 2.0 >= 4294967296.0 || (M + 15.0) * K * 2.0 >= 4294967296.0) return none;
  const int gtot = (M + 15) / 16, nt = N / cols;
  const double slice_us = (double)M * N * 4.0 / 4.5e6;  // one K slice's fp32 partials to or from memory
  DeepCfg best = none;
  for (int mg = 8; mg >= 4; mg -= 2) {
    const int mb = (gtot + mg - 1) / mg;
    for (int split = 1; split <= (partial ? ks : 1); split *= 2) {
      if (ks % split != 0) continue;
      const int n = (int)(((long)nt * mb * split + 255) / 256);     // workgroups of the busiest CU
      const double c = (double)(ks / split) * (K / ks / 128);
      double us;
      if (mg == 4) {
        const double lone = head ? 1.4 * c + 9.0 : (sum ? 1.5 * c + 9.0 : 1.3 * c + 10.0);
        const double pair = head ? 2.45 * c + 8.0 : (partial || M <= 1024 ? 2.5 : 2.1) * c + 3.0 + (sum ? 2.5 * ks : 0.0);
        us = (n / 2) * pair + (n & 1 ? lone : 0.0);
      } else {
        const double each = head ? (mg == 8 ? 1.8 * c + 12.0 : 1.66 * c + 10.0)
                                 : (mg == 8 ? 1.7 * c + (n > 1 ? 12.0 : (partial ? 6.0 : 14.0))
                                            : (M <= 1024 ? 1.4 : 1.25) * c + 13.0);
        us = n * (each + (sum ? 3.0 * ks : 0.0));
      }
      if (partial) us += 1.3 * ks * slice_us;
      if (best.mg == 0 || us < best.us) best = DeepCfg{mg, mb, split, us};
    }
  }
  return best;
}

void lsk_gemm_deep(const DeepCfg& cfg, int epi, hipStream_t s, const uint16_t* A, const uint16_t* W, uint16_t* C, long ldc,
                   int c_nks, const uint16_t* R, float* P, float* av, int* ai, int M, int N, int K, int ffn, int ks,
                   const QkvRope& qa) {
  const int nt = N / (epi == LSK_EPI_SILU_MUL ? 128 : 256);
  const dim3 grid((unsigned)((nt * cfg.m_blocks * cfg.split + 7) / 8 * 8));
#define LSK_DEEP(MG_, EPI_)                                                                                          \
  gemm_deep_kernel<MG_, EPI_><<<grid, 256, 0, s>>>(A, W, C, ldc, c_nks, R, P, av, ai, M, N, K, ffn, K / ks, nt,         \
                                                   cfg.m_blocks, ks, cfg.split, qa)
#define LSK_DEEP_MG(EPI_)                 \
  do {                                    \
    if (cfg.mg == 8) LSK_DEEP(8, EPI_);   \
    else if (cfg.mg == 6) LSK_DEEP(6, EPI_); \
    else LSK_DEEP(4, EPI_);               \
  } while (0)
  if (epi == LSK_EPI_SILU_MUL) LSK_DEEP_MG(LSK_EPI_SILU_MUL);
  else if (epi == EPI_PARTIAL) LSK_DEEP_MG(EPI_PARTIAL);
  else if (epi == EPI_QKV) LSK_DEEP_MG(EPI_QKV);
  else if (epi == LSK_EPI_RESIDUAL) LSK_DEEP_MG(LSK_EPI_RESIDUAL);
  else LSK_DEEP_MG(EPI_ARGMAX);
#undef LSK_DEEP_MG
#undef LSK_DEEP
}
