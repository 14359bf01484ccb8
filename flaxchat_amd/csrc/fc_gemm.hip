// Skinny GEMMs with fused epilogues: out = epi(A[M][K] . W[N][K]^T).
//
// Replaces the nnx.Linear matmuls of the per-token forward
// (flaxchat/engine.py:106-108, 158, 161, 172; flaxchat/gpt.py:93-99, 154-163)
// and fuses what the reference does right after them: the residual add
// (engine.py:160-161), ReLU^2 (gpt.py:161), resid/x0 lambda mix of the next
// layer (engine.py:94), the backout capture and subtraction
// (engine.py:164-166) and the 15*tanh(z/15) softcap (engine.py:173-174).
//
// Kernels:
//   k_gemv     VALU dot products (fp32 weights, the parity mode): up to 16 rows,
//              few tiles of a long K, operands off the 16-byte boundary.
//   k_gemm_f32 fp32 MFMA, 64 x 64 or K-split 32 x 32 tiles (fp32, more rows).
//   k_gemm_ks  bf16 MFMA 16x16x32, workgroup tile of 16-32 rows x 16-64
//              columns, the four waves split K, register pipeline; draft
//              steps and the split-K residual GEMMs.
//   k_gemm_la  bf16 MFMA, 32-128 rows x 128 columns, the four waves split
//              the columns and share the activation tile through LDS;
//              verify row counts, the QKV GEMM with its fused attention
//              prologue (also at one-row decode sizes) and the draft lm_head.
//   k_gemm_dma bf16 MFMA, 64 x 64 tiles fed by direct global-to-LDS loads
//              into a 4-stage ring; verify c_fc.
//   k_gemm_ring bf16 MFMA, 64 x 96 tiles, a 5-stage direct-load LDS ring;
//              the verify MLP c_proj (K split 4).
//   k_gemm_big bf16 MFMA, 128 x 128 to 256 x 256 tiles, 4-stage LDS ring of
//              direct loads; prompt and whole-sequence chunks, large-batch
//              verify chunks, and the lm_head from 200 rows.
// The row count may be a device value (packed token chunks whose size is
// only known on the GPU): the grid covers the capacity and tiles past the
// actual count exit at once.
// When N alone gives too few workgroups to occupy 256 CUs, a GEMM whose
// output is the fp32 residual stream may split K across workgroups: each
// split writes its partial product with plain stores and the RMSNorm kernel
// that consumes x next sums the splits in fixed order and applies the
// epilogue (a kernel boundary is the only synchronisation; on MI355X the
// eight XCD L2 caches are not coherent, so an in-kernel device-scope fence
// would write back a whole L2 per workgroup).
#include "fc_common.h"
#include "fc_internal.h"

// 15 tanh(v / 15) in the bf16 kernels' epilogues: with the sign of v,
// 15 - 30 / (e^{2|v|/15} + 1) by the hardware base-2 exponential and reciprocal
// (about 1 ulp each; at their limits the form gives 15 by itself); below
// |v| = 15/16, where it cancels, the series v (1 - x^2/3 + 2x^4/15) of
// x = v / 15 (truncation < 3e-9). Of |v|, because a negative exponent's
// reciprocal lies in (0.5, 1), whose roundings are twice as large. The capped
// value is within 4e-6 of 15 tanhf(v / 15), rms 0.6e-6, far below the bf16
// GEMM's own rounding, in 12 instructions. The fp32 kernels keep the exact form.
__device__ __forceinline__ float softcap15_fast(float v) {
  const float v2 = v * v;
  const float ts = v * fmaf(v2, fmaf(v2, 2.f / (15.f * 50625.f), -1.f / (3.f * 225.f)), 1.f);
  const float ex = __builtin_amdgcn_exp2f(fabsf(v) * (2.8853900817779268f / 15.f));  // e^{2|v|/15}
  const float tl = copysignf(fmaf(-30.f, __builtin_amdgcn_rcpf(ex + 1.f), 15.f), v);
  return fabsf(v) < 0.9375f ? ts : tl;
}

// FAST: the bf16 kernels' softcap (softcap15_fast); the fp32 kernel uses tanhf.
template <int EPI, bool FAST = false>
__device__ __forceinline__ void epi_apply(const Epi e, int m, int n, float acc) {
  if constexpr (EPI == EPI_STORE) {
    ((float*)e.out)[(int64_t)m * e.ldo + n] = acc;
  } else if constexpr (EPI == EPI_ADD) {
    float* o = (float*)e.out + (int64_t)m * e.ldo + n;
    *o = *o + acc;
  } else if constexpr (EPI == EPI_RELU2) {  // the next GEMM's operand: fragment order in bf16
    float r = fmaxf(acc, 0.f);
    r = r * r;
    if (e.out_dtype == FC_BF16) ((bf16_t*)e.out)[frag_idx(m, n, (int)e.ldo)] = f2bf(r);
    else ((float*)e.out)[(int64_t)m * e.ldo + n] = r;
  } else if constexpr (EPI == EPI_MLPOUT) {
    const int64_t i = (int64_t)m * e.ldo + n;
    float* x = (float*)e.out;
    const float t = x[i] + acc;  // x + mlp(...)                 engine.py:161
    float xb_v = 0.f;
    if (e.capture) {             // x_backout                    engine.py:164
      e.xb[i] = t;
      xb_v = t;
    } else if (e.last) {
      xb_v = e.xb[i];
    }
    if (e.last) x[i] = t - e.lb * xb_v;      // x - lambda * x_b  engine.py:166
    else x[i] = e.r * t + e.a * e.x0[i];     // next layer's mix  engine.py:94
  } else if constexpr (EPI == EPI_PARTIAL) {  // split-K partial, finished by the next RMSNorm
    e.part[((int64_t)e.split * e.part_rows + m) * e.ldo + n] = acc;
  } else {                                   // EPI_SOFTCAP
    if (n < e.V) {
      const int b = m / e.n_out, rr = m - b * e.n_out;
      ((float*)e.out)[(int64_t)b * e.row_stride + (int64_t)rr * e.V + n] =
          FAST ? softcap15_fast(acc) : 15.f * tanhf(acc / 15.f);
    }
  }
}

// Folded RMSNorm, consumer side: the 256 / MT threads of each output row
// (consecutive lanes) each load up to FC_RMS_REG of the row's per-tile sums
// of squares at kernel start (clamped, unconditional: one batch of loads in
// flight together) and keep them in registers through the K loop, whose
// loads they precede; the epilogue adds them up over those lanes (a fixed
// shuffle tree: deterministic).
#define FC_RMS_REG 16
struct RmsPre {
  float v[FC_RMS_REG];
};
template <int MT>
__device__ __forceinline__ void rms_load(RmsPre& r, const Epi& e, int m0, int M) {
  constexpr int TPR = 256 / MT;
  const int m = min(m0 + (int)threadIdx.x / TPR, M - 1), sub = (int)threadIdx.x % TPR;
#pragma unroll
  for (int j = 0; j < FC_RMS_REG; ++j) r.v[j] = e.rms_in[(int64_t)min(sub + j * TPR, e.rms_n - 1) * e.ssq_ld + m];
}
template <int MT>
__device__ __forceinline__ float rms_finish(const RmsPre& r, const Epi& e, int K) {
  constexpr int TPR = 256 / MT;
  const int sub = (int)threadIdx.x % TPR;
  float p = 0.f;
#pragma unroll
  for (int j = 0; j < FC_RMS_REG; ++j) p += sub + j * TPR < e.rms_n ? r.v[j] : 0.f;
#pragma unroll
  for (int o = TPR / 2; o > 0; o >>= 1) p += __shfl_xor(p, o, WAVE);
  return 1.f / sqrtf(p / (float)K + 1e-6f);
}

// ---------------------------------------------------------------------------
// VALU GEMV / small GEMM. 256 threads = 4 waves; each wave owns 4 columns
// and MB rows; lanes split K in 16-byte vectors.
// ---------------------------------------------------------------------------
template <typename T, int VEC>
__device__ __forceinline__ void load_vec(const T* p, float* o);
template <>
__device__ __forceinline__ void load_vec<float, 4>(const float* p, float* o) {
  float4 v = *(const float4*)p;
  o[0] = v.x; o[1] = v.y; o[2] = v.z; o[3] = v.w;
}
template <>
__device__ __forceinline__ void load_vec<bf16_t, 8>(const bf16_t* p, float* o) {
  uint4 v = *(const uint4*)p;
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    o[2 * i] = __uint_as_float(w[i] << 16);
    o[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
  }
}

template <typename T, int MB, int EPI>
__global__ __launch_bounds__(256) void k_gemv(const T* __restrict__ A, const T* __restrict__ W, int Mcap,
                                              const int* __restrict__ Mdev, int N, int K, Epi e) {
  constexpr int VEC = 16 / sizeof(T);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int n0 = (blockIdx.x * 4 + wave) * 4;
  const int m0 = blockIdx.y * MB;
  const int M = Mdev ? min(*Mdev, Mcap) : Mcap;
  if (m0 >= M) return;
  float acc[MB][4];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[i][c] = 0.f;
  for (int k = lane * VEC; k < K; k += 64 * VEC) {
    float w[4][VEC];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      if (n0 + c < N) load_vec<T, VEC>(W + (int64_t)(n0 + c) * K + k, w[c]);
      else
#pragma unroll
        for (int j = 0; j < VEC; ++j) w[c][j] = 0.f;
    }
#pragma unroll
    for (int i = 0; i < MB; ++i) {
      if (m0 + i < M) {
        float a[VEC];
        load_vec<T, VEC>(A + (int64_t)(m0 + i) * K + k, a);
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
          for (int j = 0; j < VEC; ++j) acc[i][c] += a[j] * w[c][j];
      }
    }
  }
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[i][c] = wave_sum(acc[i][c]);
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int c = 0; c < 4; ++c)
      if (lane == ((i * 4 + c) & 63) && m0 + i < M && n0 + c < N) epi_apply<EPI>(e, m0 + i, n0 + c, acc[i][c]);
}

// ---------------------------------------------------------------------------
// fp32 GEMM on the fp32 matrix cores (32x32x2: true fp32 products and sums at
// twice the rate of unpacked VALU FMAs), for more than GEMV_MAX_M rows.
//
// KW = 1: a workgroup owns 64 x 64 outputs, its 2 x 2 waves 32 x 32 each;
// KW = 4, 8: 32 x 32 outputs, the KW waves take every KW-th 32-deep k chunk
// and are summed in LDS (outputs too few for 64 x 64 tiles to fill the CUs).
// A chunk's rows (128 bytes of 32 rows per operand) go to LDS by direct loads,
// whole lines, two stages. Lane l takes its operands 16 bytes at a time: row
// l % 32, k 8 j + 4 (l / 32) .. +3, whose component x is MFMA x of group j (the
// order of k within a chunk is free). For that the 16-byte piece p of row r
// lies at place p ^ (r % 8), so that eight rows' pieces do not share banks.
//
// Rounding: a group of 8 k is summed from zero, four groups pairwise, and the
// chunks with TwoSum (the error terms in a second accumulator), so the error
// does not grow with K: against 64 bits 7.1e-8 at K = 256 and 3072 where k_gemv,
// whose lanes sum K / 64 products each, has 7.8e-8 and 1.4e-7. Row-major
// operands, K % 8 == 0.
//
// 1000 rows x 8192 x 256: 493 -> 63 us, x 1024 x 256: 68 -> 13.7, x 256 x 1024:
// 32 -> 12.7 (k_gemv re-reads the weights every 8 rows and does 4 FMAs per
// load). Bound by the MFMAs (1024 cycles a chunk) and, not overlapped with them
// within a wave, the 16 x 10 VALU operations of its sums.
// ---------------------------------------------------------------------------
#define GEMV_MAX_M 16
__device__ __forceinline__ f32x16 mfma32f(float a, float b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}
struct F32Stage {
  float4 a[32][8], w[32][8];  // 32 rows x 32 k per operand, pieces swizzled
};
// TwoSum: tot + low += t, exactly in tot and its error term (NaN once tot is infinite: f32_round2)
__device__ __forceinline__ void f32_add2(float& tot, float& low, float t) {
  const float s = tot + t, b = s - tot;
  low += (tot - (s - b)) + (t - b);
  tot = s;
}
__device__ __forceinline__ float f32_round2(float tot, float low) {
  return fabsf(tot) < INFINITY ? tot + low : tot;
}
template <int KW, int EPI>
__global__ __launch_bounds__(KW == 8 ? 512 : 256, 2) void k_gemm_f32(const float* __restrict__ A, const float* __restrict__ W,
                                                     int Mcap, const int* __restrict__ Mdev, int N, int K, int ntiles,
                                                     Epi e) {
  constexpr int T = KW == 1 ? 64 : 32;
  // KW = 1: a row half of A and W each; else a wave each
  __shared__ F32Stage st0[KW == 1 ? 2 : KW], st1[KW == 1 ? 2 : KW];
  const int M = Mdev ? min(*Mdev, Mcap) : Mcap;
  const int nt = blockIdx.x % ntiles, mt = blockIdx.x / ntiles;
  const int m0 = mt * T, n0 = nt * T;
  if (m0 >= M) return;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = KW == 1 ? wave >> 1 : 0, wn = KW == 1 ? wave & 1 : 0;
  const int C = (K + 31) >> 5;                              // chunks; a wave takes chunks wave, wave + KW, ...
  const int nch = (C + KW - 1) / KW;
  // direct loads: lane l fetches the piece that lies at place l % 8 of row
  // l / 8 of a group of eight rows. KW = 1: wave w loads operand w / 2's half
  // w % 2 (rows 32 (w % 2) .. +31); KW > 1: both operands of its own chunk
  const int lr = lane >> 3, lp = (lane & 7) ^ lr;
  auto issue = [&](F32Stage* st, int ci) {
    const int c = min(KW == 1 ? ci : KW * ci + wave, C - 1);  // past the end: harmless re-reads
    const uint32_t koff = (uint32_t)min(32 * c + 4 * lp, K - 4) * 4u;    // past the row's end: its last piece again
    auto rows = [&](const float* P, int r0, int R, uint32_t lds) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {  // rows r0 + 8 u .. +7, clamped to the last one
        const uint32_t row = (uint32_t)min(8 * u + lr, R - 1 - r0);
        lds_load_1k(P + (int64_t)r0 * K, row * (uint32_t)K * 4u + koff, lds + 1024 * u);
      }
    };
    if constexpr (KW == 1) {
      const int h = wave & 1;
      if (wave < 2) rows(A, min(m0 + 32 * h, M - 1), M, LDS_ADDR(st[0].a) + (uint32_t)sizeof(F32Stage) * h);
      else rows(W, min(n0 + 32 * h, N - 1), N, LDS_ADDR(st[0].w) + (uint32_t)sizeof(F32Stage) * h);
    } else {
      rows(A, m0, M, LDS_ADDR(st[0].a) + (uint32_t)sizeof(F32Stage) * wave);
      rows(W, n0, N, LDS_ADDR(st[0].w) + (uint32_t)sizeof(F32Stage) * wave);
    }
  };
  float tot[16], low[16];
#pragma unroll
  for (int x = 0; x < 16; ++x) tot[x] = low[x] = 0.f;
  const int r = lane & 31, hl = lane >> 5;
  auto chunk = [&](const F32Stage* st, int ci) {
    const int c = KW == 1 ? ci : KW * ci + wave;
    if (c >= C) return;
    const F32Stage& sa = st[KW == 1 ? wm : wave];
    const F32Stage& sw = st[KW == 1 ? wn : wave];
    const int jn = min(4, (K - 32 * c) >> 3);  // groups of 8 k in the chunk
    f32x16 g[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
#pragma unroll
      for (int x = 0; x < 16; ++x) g[j][x] = 0.f;
      if (j < jn) {
        const float4 av = sa.a[r][(2 * j + hl) ^ (r & 7)], wv = sw.w[r][(2 * j + hl) ^ (r & 7)];
        g[j] = mfma32f(av.x, wv.x, g[j]);
        g[j] = mfma32f(av.y, wv.y, g[j]);
        g[j] = mfma32f(av.z, wv.z, g[j]);
        g[j] = mfma32f(av.w, wv.w, g[j]);
      }
    }
#pragma unroll
    for (int x = 0; x < 16; ++x) f32_add2(tot[x], low[x], (g[0][x] + g[1][x]) + (g[2][x] + g[3][x]));
  };
  auto sync = [&]() {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0);  // the chunk's loads, issued a chunk ago, and this wave's LDS reads
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
  };
  issue(st0, 0);
  for (int i = 0; i < nch; i += 2) {
    sync();
    issue(st1, i + 1);
    chunk(st0, i);
    if (i + 1 < nch) {
      sync();
      issue(st0, i + 2);
      chunk(st1, i + 1);
    }
  }
  __builtin_amdgcn_s_waitcnt(0);  // no direct load outlives the workgroup's LDS
  if constexpr (KW == 1) {
#pragma unroll
    for (int x = 0; x < 16; ++x) {
      const int m = m0 + 32 * wm + 8 * (x >> 2) + 4 * hl + (x & 3), n = n0 + 32 * wn + r;
      if (m < M && n < N) epi_apply<EPI>(e, m, n, f32_round2(tot[x], low[x]));
    }
  } else {
    __syncthreads();  // the stages become the waves' partial tiles
    typedef float Part[32][33];
    Part *hi = (Part*)&st0[0], *lo = (Part*)&st1[0];
    static_assert(sizeof(F32Stage) >= sizeof(Part), "a wave's partial tile");
#pragma unroll
    for (int x = 0; x < 16; ++x) {
      hi[wave][8 * (x >> 2) + 4 * hl + (x & 3)][r] = tot[x];
      lo[wave][8 * (x >> 2) + 4 * hl + (x & 3)][r] = low[x];
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 16 / KW; ++u) {
      const int rr = (threadIdx.x >> 5) + 2 * KW * u, cc = threadIdx.x & 31;
      float v = hi[0][rr][cc], c = lo[0][rr][cc];
#pragma unroll
      for (int w = 1; w < KW; ++w) {
        f32_add2(v, c, hi[w][rr][cc]);
        c += lo[w][rr][cc];
      }
      if (m0 + rr < M && n0 + cc < N) epi_apply<EPI>(e, m0 + rr, n0 + cc, f32_round2(v, c));
    }
  }
}

// ---------------------------------------------------------------------------
// bf16 MFMA 16x16x32. Operand layout (wave64): lane l holds row (l % 16) of
// A / column (l % 16) of B and 8 consecutive k values 8*(l/16)..+7 of a
// 32-wide k step; the f32x4 result holds rows 4*(l/16)+i of column l % 16.
// ---------------------------------------------------------------------------
// weight fragment loads: plain (they are re-read across M tiles through L2)
#define W_LD(p) (*(p))
// lm_head weights (the softcap epilogue) always stream non-temporally: the
// matrix (201 MB at cfg4) is about the size of the 256 MB Infinity Cache,
// and both the verify and the draft lm_head reading it non-temporally made
// the speculative round 2.2% faster (5.01 -> 4.91 ms) than either one alone
// or neither (the other reads of the round keep their cache lines). The
// other GEMMs re-read weight tiles across M tiles through L2 and lose more
// than they gain from it (5.0 -> 5.3 ms).
#define LM_LD(p) __builtin_nontemporal_load(p)
// The same for the lm_head on the K-split kernel (one-row decode: cfg2's
// 100 MB head read five times a round; 0.917-0.918 vs 0.924 ms per round)
// and on k_gemm_big's direct loads (the cfg4 verify head:
// 4.835-4.837 vs 4.840-4.845 ms per round; with more than two M tiles the
// tiles share the weights through the caches instead), alternating builds.
#ifndef FC_KS_LM_NT
#define FC_KS_LM_NT 1
#endif
__device__ __forceinline__ f32x4 mfma16(uint4 a, uint4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                  0, 0);
}
__device__ __forceinline__ f32x4 mfma16(v4u a, v4u b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                  0, 0);
}

// Epilogue on finished sums laid out row-major: thread t owns OPT = MT NT /
// 256 consecutive columns col0 .. of tile row `row` = t / (NT / OPT) (the
// threads of a row are consecutive lanes). Used by the kernels that stage
// their tile in LDS first (k_gemm_ks, k_gemm_ring): the folded-norm
// epilogues need whole row segments per thread.
template <int EPI, int MT, int NT>
__device__ __forceinline__ void row_epilogue(const Epi& e, float (&v)[MT * NT / 256], int row, int col0, int m0,
                                             int n0, int nt, int s, int M, int K, const RmsPre& rpre) {
  constexpr int OPT = MT * NT / 256, TPR = NT / OPT;
  const int m = m0 + row;
  const bool live = m < M;
  if constexpr (EPI == EPI_RELU2) {
    if (e.rms_in != nullptr) {  // thread t's epilogue row is its prefetch row (t / TPR)
      static_assert(TPR == 256 / MT, "row mapping");
      const float sc = rms_finish<MT>(rpre, e, K);
#pragma unroll
      for (int c = 0; c < OPT; ++c) v[c] *= sc;
    }
  }
  if constexpr (EPI == EPI_ADD) {
    if (e.xa != nullptr) {
      // residual add, bf16 copy of the new x (OPT consecutive columns: whole
      // bf16 pairs in fragment order) and the row's sum of squares over this
      // tile (the TPR threads of a row are consecutive lanes)
      static_assert(OPT % 2 == 0 && 64 % TPR == 0, "folded-norm epilogue tiling");
      float ss = 0.f;
      if (live) {
        float* o = (float*)e.out + (int64_t)m * e.ldo + n0 + col0;
#pragma unroll
        for (int c = 0; c < OPT; c += 2) {
          const float a0 = o[c] + v[c], a1 = o[c + 1] + v[c + 1];
          o[c] = a0;
          o[c + 1] = a1;
          ss += a0 * a0 + a1 * a1;
          *(uint32_t*)(e.xa + frag_idx(m, n0 + col0 + c, (int)e.ldo)) =
              pack2bf(a0, a1);
        }
      }
#pragma unroll
      for (int o = TPR / 2; o > 0; o >>= 1) ss += __shfl_xor(ss, o, WAVE);
      if (live && col0 == 0) e.ssq[(int64_t)nt * e.ssq_ld + m] = ss;
      return;
    }
  }
  if (!live) return;
  Epi ee = e;
  ee.split = s;
#pragma unroll
  for (int c = 0; c < OPT; ++c) epi_apply<EPI, true>(ee, m, n0 + col0 + c, v[c]);
}

// bf16 MFMA GEMM, K split over the four waves of a workgroup.
//
// A workgroup owns an MT x NT output tile (MT = 16 MB rows, NT = 16 NB
// columns) over its split's K range; its four waves take interleaved
// 64-wide k chunks, so every weight and activation byte reaches the CU once
// and no LDS traffic or barrier sits in the main loop. Each wave keeps NS
// chunks of A and W fragments in flight in registers (the loads of chunk
// i + NS are issued right after chunk i is consumed). The four partial
// tiles are summed in LDS at the end and the epilogue runs on a coalesced
// row-major layout.
//
// Grid: 1-D over (N tile, K split, M tile), the N tile count padded to a
// multiple of 8. Workgroups are dealt to the eight XCDs round robin and both
// tile orders keep N tile n on XCD n % 8, so the M tiles that share its
// weight slab read it from HBM once and hit in that XCD's L2:
//   mfast = 1: within an XCD the M tiles of one N tile run back to back
//              (wide N, e.g. lm_head: the slab is reused while still in L2);
//   mfast = 0: M tile slowest; with a device row count (`Mdev`, at most
//              Mcap) the tiles past it come last in dispatch order and exit
//              at once.
template <int MB, int NB, int NS, int EPI, bool PK = false>
__global__ __launch_bounds__(256) void k_gemm_ks(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W,
                                                 int Mcap, const int* __restrict__ Mdev, int N, int K, int ntiles,
                                                 int S, int mtiles, int mfast, Epi e) {
  constexpr int MT = 16 * MB, NT = 16 * NB;
  const int id = blockIdx.x;
  const int ntiles8 = (ntiles + 7) & ~7;
  int nt, s, mt;
  if (mfast) {  // per XCD: the M tiles of one N tile back to back
    const int xcd = id & 7, loc = id >> 3, per = S * mtiles;
    const int nl = loc / per, rem = loc - nl * per;
    s = rem / mtiles;
    mt = rem - s * mtiles;
    nt = nl * 8 + xcd;
  } else {      // M tile slowest
    nt = id % ntiles8;
    const int rest = id / ntiles8;
    s = rest % S;
    mt = rest / S;
  }
  if (nt >= ntiles) return;
  const int M = Mdev ? min(*Mdev, Mcap) : Mcap;
  const int m0 = mt * MT;
  if (m0 >= M) return;
  const int n0 = nt * NT;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int C = K >> 6;
  const int c_beg = (int)((int64_t)s * C / S), c_end = (int)((int64_t)(s + 1) * C / S);
  const int nch = c_end - c_beg > wave ? (c_end - c_beg - wave + 3) >> 2 : 0;
  RmsPre rpre;  // folded RMSNorm: this thread's share of its output row's sums of squares
  if constexpr (EPI == EPI_RELU2) {
    if (e.rms_in != nullptr) rms_load<MT>(rpre, e, m0, M);
  }

  f32x4 acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  // operand addresses at k = 0. Row-major: lane l reads row (l % 16), 16 B
  // at k = 8 (l / 16). Fragment order (PK): 16-row x 32-k blocks of 1 KB in
  // [row block][k step] order, lane l's 16 B at offset 16 l of its block,
  // so each load instruction reads 1 KB contiguous. Either way the chunk
  // offset of k step t is `kstep_elems * t`.
  const bf16_t* wrow[NB];
  const bf16_t* arow[MB];
  int64_t kstep_elems;
  if constexpr (PK) {
    const int64_t KS32 = K >> 5;
#pragma unroll
    for (int j = 0; j < NB; ++j) wrow[j] = W + (int64_t)(n0 / 16 + j) * KS32 * 512 + lane * 8;
    const int last_blk = (M - 1) >> 4;
#pragma unroll
    for (int i = 0; i < MB; ++i) arow[i] = A + (int64_t)min(m0 / 16 + i, last_blk) * KS32 * 512 + lane * 8;
    kstep_elems = 512;
  } else {
#pragma unroll
    for (int j = 0; j < NB; ++j) wrow[j] = W + (int64_t)(n0 + 16 * j + r) * K + 8 * g;
#pragma unroll
    for (int i = 0; i < MB; ++i) arow[i] = A + (int64_t)min(m0 + 16 * i + r, M - 1) * K + 8 * g;
    kstep_elems = 32;
  }

  if (nch > 0) {
    static_assert(NS >= 2 && NS <= 4, "register ring of 2-4 chunks");
    v4u wb[NS][NB][2], ab[NS][MB][2];
    // chunk index of the wave's i-th chunk, clamped so the tail loads are
    // harmless re-reads and the loop body has no branch
#define KS_LOAD(slot, i)                                                            \
  {                                                                                 \
    const int c_ = c_beg + wave + 4 * min((i), nch - 1);                            \
    _Pragma("unroll") for (int j = 0; j < NB; ++j)                                  \
      _Pragma("unroll") for (int ks = 0; ks < 2; ++ks)                              \
        wb[slot][j][ks] = EPI == EPI_SOFTCAP && FC_KS_LM_NT ? LM_LD((const v4u*)(wrow[j] + (2 * c_ + ks) * kstep_elems)) \
                                                             : W_LD((const v4u*)(wrow[j] + (2 * c_ + ks) * kstep_elems)); \
    _Pragma("unroll") for (int mb = 0; mb < MB; ++mb)                               \
      _Pragma("unroll") for (int ks = 0; ks < 2; ++ks)                              \
        ab[slot][mb][ks] = *(const v4u*)(arow[mb] + (2 * c_ + ks) * kstep_elems);   \
  }
#define KS_MMA(slot)                                                                \
  {                                                                                 \
    _Pragma("unroll") for (int ks = 0; ks < 2; ++ks)                                \
      _Pragma("unroll") for (int mb = 0; mb < MB; ++mb)                             \
        _Pragma("unroll") for (int j = 0; j < NB; ++j)                              \
          acc[mb][j] = mfma16(ab[slot][mb][ks], wb[slot][j][ks], acc[mb][j]);       \
  }
#pragma unroll
    for (int p = 0; p < NS; ++p) KS_LOAD(p, p);
    int i = 0;
    // the scheduling barriers keep each chunk's loads together and after the
    // MFMAs that free its registers, so the other slots' loads stay in flight
    // while a slot computes (the waits become vmcnt(NS - 1 slots))
    for (; i + NS - 1 < nch; i += NS) {
#pragma unroll
      for (int p = 0; p < NS; ++p) {
        KS_MMA(p);
        __builtin_amdgcn_sched_barrier(0);
        KS_LOAD(p, i + NS + p);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    // the last nch - i < NS chunks sit in slots 0 .. nch - i - 1
#pragma unroll
    for (int p = 0; p < NS - 1; ++p)
      if (i + p < nch) KS_MMA(p);
#undef KS_LOAD
#undef KS_MMA
  }

  // sum the four waves' tiles; thread t then owns OPT consecutive columns
  // of one row
  constexpr int LDR = NT + 4, OPT = MT * NT / 256, TPR = NT / OPT;
  static_assert(OPT >= 1 && NT % OPT == 0, "epilogue tiling");
  __shared__ float red[4][MT][LDR];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) red[wave][16 * mb + 4 * g + i][16 * j + r] = acc[mb][j][i];
  __syncthreads();
  const int t = threadIdx.x;
  const int row = t / TPR, col0 = (t - row * TPR) * OPT;
  float v[OPT];
#pragma unroll
  for (int c = 0; c < OPT; ++c)
    v[c] = red[0][row][col0 + c] + red[1][row][col0 + c] + red[2][row][col0 + c] + red[3][row][col0 + c];
  row_epilogue<EPI, MT, NT>(e, v, row, col0, m0, n0, nt, s, M, K, rpre);
}

// Attention prologue of one token and one head slot from its fp32 GEMM
// output row x (128 values; flaxchat/engine.py:96-126, flaxchat/gpt.py:65-71):
// q / k heads get RoPE (pairs d, d + 64) and 1.2 * RMSNorm, v heads the
// value-embedding gate; q goes to q[m][head], k / v to the cache at the
// token's position. Eight consecutive lanes share a token (`part` = which
// 8 rotary pairs); all 8 take part in the norm's shuffles.
//
// The inputs that do not depend on the GEMM result are loaded first, in two
// steps that callers issue ahead of the accumulator staging so the loads of
// several tokens are in flight together: qkv_pre_row (the token's cache row,
// position and id) and qkv_pre_tab (the rotary table entries of the q / k
// heads; the value-embedding slice and the gate inputs of the v heads).
struct QkvPre {
  int b, pos, tok;
  float c[8], s[8];  // q / k heads: cos / sin of the lane's 8 rotary pairs
  uint4 h0, ve0, ve1;  // v heads: A row k 0..7, ve dims 8 part .. +7 and 64 + 8 part .. +7
  uint2 h1;            // v heads: A row k 8..11
};

__device__ __forceinline__ void qkv_pre_row(const QkvEpi& Q, int m, int M, int hh, QkvPre& p) {
  p.b = 0;
  p.pos = 0;
  p.tok = 0;
  if (m < M) {
    p.b = Q.tok_row[m];
    p.pos = Q.tok_pos[m];
    if (hh >= Q.H + Q.G && Q.ve != nullptr) p.tok = Q.tokens[m];
  }
}

__device__ __forceinline__ void qkv_pre_tab(const QkvEpi& Q, int m, int M, int hh, int part, QkvPre& p) {
  if (hh < Q.H + Q.G) {
    const int pc = min(max(p.pos, 0), Q.rope_len - 1);
    const float4* cp = (const float4*)(Q.rcos + (int64_t)pc * 64 + 8 * part);
    const float4* sp = (const float4*)(Q.rsin + (int64_t)pc * 64 + 8 * part);
    const float4 c0 = cp[0], c1 = cp[1], s0 = sp[0], s1 = sp[1];
    p.c[0] = c0.x; p.c[1] = c0.y; p.c[2] = c0.z; p.c[3] = c0.w;
    p.c[4] = c1.x; p.c[5] = c1.y; p.c[6] = c1.z; p.c[7] = c1.w;
    p.s[0] = s0.x; p.s[1] = s0.y; p.s[2] = s0.z; p.s[3] = s0.w;
    p.s[4] = s1.x; p.s[5] = s1.y; p.s[6] = s1.z; p.s[7] = s1.w;
  } else if (Q.ve != nullptr && m < M) {
    // A row m, k 0..7 then 8..11: 16 contiguous bytes each in fragment order
    const uint16_t* hr = Q.h + frag_idx(m, 0, Q.D);
    p.h0 = *(const uint4*)hr;
    p.h1 = *(const uint2*)(hr + 128);
    const uint16_t* vr = Q.ve + ((int64_t)p.tok * Q.G + (hh - Q.H - Q.G)) * 128;
    p.ve0 = *(const uint4*)(vr + 8 * part);
    p.ve1 = *(const uint4*)(vr + 64 + 8 * part);
  }
}

__device__ __forceinline__ float bf_lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float bf_hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }

__device__ __forceinline__ void qkv_finish(const QkvEpi& Q, const float* x, int m, int M, int hh, int part,
                                           const QkvPre& p) {
  const bool live = m < M;
  float x1[8], x2[8];
  {
    const float4* xa = (const float4*)(x + 8 * part);
    const float4* xb = (const float4*)(x + 64 + 8 * part);
    const float4 a0 = xa[0], a1 = xa[1], b0 = xb[0], b1 = xb[1];
    x1[0] = a0.x; x1[1] = a0.y; x1[2] = a0.z; x1[3] = a0.w; x1[4] = a1.x; x1[5] = a1.y; x1[6] = a1.z; x1[7] = a1.w;
    x2[0] = b0.x; x2[1] = b0.y; x2[2] = b0.z; x2[3] = b0.w; x2[4] = b1.x; x2[5] = b1.y; x2[6] = b1.z; x2[7] = b1.w;
  }
  const int b = p.b, pos = p.pos;
  // a token whose row lies outside [0, B) (an empty or rejected chunk row)
  // writes nothing, q included, like the unfused prologue
  const bool in_row = live && (unsigned)b < (unsigned)Q.B;
  const bool in_cache = in_row && pos >= 0 && pos < Q.cap;
  if (hh < Q.H + Q.G) {
    float ss = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float c = p.c[e], s = p.s[e];
      const float y1 = x1[e] * c + x2[e] * s;
      const float y2 = x1[e] * (-s) + x2[e] * c;
      x1[e] = y1;
      x2[e] = y2;
      ss += y1 * y1 + y2 * y2;
    }
    ss += __shfl_xor(ss, 1, WAVE);
    ss += __shfl_xor(ss, 2, WAVE);
    ss += __shfl_xor(ss, 4, WAVE);
    const float inv = 1.f / sqrtf(ss / 128.f + 1e-6f);
    uint4 p1, p2;
    uint32_t* w1 = (uint32_t*)&p1;
    uint32_t* w2 = (uint32_t*)&p2;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      w1[e] = pack2bf(x1[2 * e] * inv * 1.2f, x1[2 * e + 1] * inv * 1.2f);
      w2[e] = pack2bf(x2[2 * e] * inv * 1.2f, x2[2 * e + 1] * inv * 1.2f);
    }
    if (hh < Q.H) {
      if (in_row) {
        bf16_t* qo = Q.q + ((int64_t)m * Q.H + hh) * 128;
        *(uint4*)(qo + 8 * part) = p1;
        *(uint4*)(qo + 64 + 8 * part) = p2;
      }
    } else if (in_cache) {
      bf16_t* kg = Q.kc + ((int64_t)b * Q.G + (hh - Q.H)) * Q.cap * 128;
      *(uint4*)(kg + kblk_idx(pos, 8 * part)) = p1;       // 8 consecutive dims stay contiguous
      *(uint4*)(kg + kblk_idx(pos, 64 + 8 * part)) = p2;
    }
  } else {
    const int gv = hh - Q.H - Q.G;
    if (Q.ve != nullptr && live) {
      const uint32_t hw[6] = {p.h0.x, p.h0.y, p.h0.z, p.h0.w, p.h1.x, p.h1.y};
      const float* wg = Q.ve_gate + gv * 12;
      float z = 0.f;
#pragma unroll
      for (int i = 0; i < 6; ++i) {
        z += bf_lo(hw[i]) * wg[2 * i];
        z += bf_hi(hw[i]) * wg[2 * i + 1];
      }
      const float gate = 3.f * (1.f / (1.f + expf(-z)));
      const uint32_t va[4] = {p.ve0.x, p.ve0.y, p.ve0.z, p.ve0.w}, vb[4] = {p.ve1.x, p.ve1.y, p.ve1.z, p.ve1.w};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        x1[2 * e] = x1[2 * e] + gate * bf_lo(va[e]);
        x1[2 * e + 1] = x1[2 * e + 1] + gate * bf_hi(va[e]);
        x2[2 * e] = x2[2 * e] + gate * bf_lo(vb[e]);
        x2[2 * e + 1] = x2[2 * e + 1] + gate * bf_hi(vb[e]);
      }
    }
    if (in_cache) {
      bf16_t* vb = Q.vc + (((int64_t)b * Q.G + gv) * (Q.cap / 32) + pos / 32) * 128 * 32 + (pos & 31);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        vb[(8 * part + e) * 32] = f2bf(x1[e]);
        vb[(64 + 8 * part + e) * 32] = f2bf(x2[e]);
      }
    }
  }
}

// The draw's Gumbel noise for this thread's epilogue columns (row m0 + t / 8,
// NT / 8 columns from n0 + (t % 8) NT / 8), which depends only on the Philox
// counter: where the tile has a single 32-row pass (MB = 2) k_gemm_la computes
// it before its K loop, while the first chunks load, instead of in the tail.
template <int MB, int NBW>
struct VpNoise {
  float g[MB == 2 ? 8 * NBW : 1];
  bool ok;
};
template <int MB, int NBW>
__device__ __forceinline__ bool vp_noise_wanted(const Epi& e) {
  return MB == 2 && e.vp != nullptr && e.vp_draw && e.vp_T > 0.f;
}
template <int MB, int NBW>
__device__ __forceinline__ void vp_noise(const Epi& e, int m0, int n0, int rnd, VpNoise<MB, NBW>& nz) {
  nz.ok = false;
  if constexpr (MB == 2) {
    if (!vp_noise_wanted<MB, NBW>(e)) return;
    constexpr int PER = 8 * NBW;
    const int m = m0 + (threadIdx.x >> 3), c0 = n0 + (threadIdx.x & 7) * PER;
#pragma unroll
    for (int w0 = 0; w0 < PER; w0 += 4) {
      const u32x4 rr = philox4x32_10(u32x4{(uint32_t)((c0 + w0) >> 2), (uint32_t)m, (uint32_t)rnd,
                                           (uint32_t)e.vp_slot},
                                     (uint32_t)e.vp_seed, (uint32_t)(e.vp_seed >> 32));
#pragma unroll
      for (int w = 0; w < 4; ++w) nz.g[w0 + w] = gumbel_of(pick(rr, w));
    }
    nz.ok = true;
  }
}

// Vocab-pass partials of the logits tile (EPI_SOFTCAP with e.vp): the same
// terms as the separate pass (k_vpart) over the tile's columns instead of a
// 1024-entry chunk, so the draft step needs no second pass over its logits.
// Per 32 rows the capped values are staged in LDS; then 8 consecutive lanes
// own a row, NT / 8 columns each (whole Philox groups of 4), and reduce with
// shuffles; lane 0 of the 8 writes the row's VPart.
// The capped logits are stored here too, from the same values the partials
// are computed from (acc is overwritten with them).
template <int MB, int NBW>
__device__ __forceinline__ void vocab_tile_parts(const Epi& e, f32x4 (&acc)[MB][NBW], int m0, int n0, int nt,
                                                 int M, const VpNoise<MB, NBW>* nz) {
  constexpr int NT = 64 * NBW, PER = NT / 8, LD = NT + 4;
  static_assert(MB % 2 == 0, "32-row passes");
  __shared__ __align__(16) float T[32 * LD];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int row = threadIdx.x >> 3, q = threadIdx.x & 7;
  const int c0 = n0 + q * PER;  // this thread's first column
  const float Tt = e.vp_T;
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int j = 0; j < NBW; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float z = softcap15_fast(acc[mb][j][i]);
        acc[mb][j][i] = z;
        const int m = m0 + 16 * mb + 4 * g + i, n = n0 + 16 * (wave * NBW + j) + r;
        if (m < M && n < e.V) {
          const int b = m / e.n_out, rr = m - b * e.n_out;
          ((float*)e.out)[(int64_t)b * e.row_stride + (int64_t)rr * e.V + n] = z;
        }
      }
#pragma unroll
  for (int p = 0; p < MB / 2; ++p) {
    if (p > 0) __syncthreads();  // the previous pass's readers are done with T
#pragma unroll
    for (int mh = 0; mh < 2; ++mh)
#pragma unroll
      for (int j = 0; j < NBW; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) T[(16 * mh + 4 * g + i) * LD + 16 * (wave * NBW + j) + r] = acc[2 * p + mh][j][i];
    __syncthreads();
    const int m = m0 + 32 * p + row;
    float v[PER];
#pragma unroll
    for (int w = 0; w < PER; w += 4) {
      const float4 t4 = *reinterpret_cast<const float4*>(&T[row * LD + q * PER + w]);
      v[w] = t4.x;
      v[w + 1] = t4.y;
      v[w + 2] = t4.z;
      v[w + 3] = t4.w;
    }
    float bz = -INFINITY;
    int bzi = 0x7fffffff;
#pragma unroll
    for (int w = 0; w < PER; ++w)
      if (c0 + w < e.V) argmax_merge(bz, bzi, v[w], c0 + w);
#pragma unroll
    for (int o = 1; o < 8; o <<= 1) argmax_merge(bz, bzi, __shfl_xor(bz, o, WAVE), __shfl_xor(bzi, o, WAVE));
    VPart pt;
    pt.zmax = bz;
    pt.zarg = bzi;
    pt.m = 0.f;
    pt.s = 1.f;
    pt.a = -INFINITY;
    pt.ai = 0x7fffffff;
    pt.g = -INFINITY;
    pt.gi = 0x7fffffff;
    if (Tt > 0.f) {
      const float mx = bz / Tt;
#pragma unroll
      for (int w = 0; w < PER; ++w) v[w] = v[w] / Tt;
      float sum = 0.f;
#pragma unroll
      for (int w = 0; w < PER; ++w)
        if (c0 + w < e.V) sum += expf(v[w] - mx);
#pragma unroll
      for (int o = 1; o < 8; o <<= 1) sum += __shfl_xor(sum, o, WAVE);
      pt.m = mx;
      pt.s = sum;
      if (e.vp_draw) {
        const int rnd = m < M ? e.vp_round[m] : 0;
        float ba = -INFINITY, bg = -INFINITY;
        int bai = 0x7fffffff, bgi = 0x7fffffff;
        bool pre = false;
        if constexpr (MB == 2) {
          if (nz != nullptr && nz->ok) {  // the noise computed before the K loop
            pre = true;
#pragma unroll
            for (int w = 0; w < PER; ++w) {
              const int i = c0 + w;
              if (i >= e.V) break;
              argmax_merge(ba, bai, (v[w] - mx) + nz->g[w], i);
              argmax_merge(bg, bgi, nz->g[w], i);
            }
          }
        }
        if (!pre) {
#pragma unroll
          for (int w0 = 0; w0 < PER; w0 += 4) {
            if (c0 + w0 >= e.V) break;
            const u32x4 rr = philox4x32_10(u32x4{(uint32_t)((c0 + w0) >> 2), (uint32_t)m, (uint32_t)rnd,
                                                 (uint32_t)e.vp_slot},
                                           (uint32_t)e.vp_seed, (uint32_t)(e.vp_seed >> 32));
#pragma unroll
            for (int w = 0; w < 4; ++w) {
              const int i = c0 + w0 + w;
              if (i >= e.V) break;
              const float G = gumbel_of(pick(rr, w));
              argmax_merge(ba, bai, (v[w0 + w] - mx) + G, i);
              argmax_merge(bg, bgi, G, i);
            }
          }
        }
#pragma unroll
        for (int o = 1; o < 8; o <<= 1) {
          argmax_merge(ba, bai, __shfl_xor(ba, o, WAVE), __shfl_xor(bai, o, WAVE));
          argmax_merge(bg, bgi, __shfl_xor(bg, o, WAVE), __shfl_xor(bgi, o, WAVE));
        }
        pt.a = ba;
        pt.ai = bai;
        pt.g = bg;
        pt.gi = bgi;
      }
    }
    if (q == 0 && m < M) {
      float4* dst = reinterpret_cast<float4*>(e.vp + (int64_t)m * e.vp_ld + nt);
      dst[0] = make_float4(pt.zmax, __int_as_float(pt.zarg), pt.m, pt.s);
      dst[1] = make_float4(pt.a, __int_as_float(pt.ai), pt.g, __int_as_float(pt.gi));
    }
  }
}

// Epilogue of the column-split kernels (k_gemm_la, k_gemm_dma): acc[mb][j]
// holds rows 16 mb + 4 g + i, column 16 (wave NBW + j) + r of the tile. VP:
// the kernel can write the vocab-pass partials (k_gemm_la).
template <int MB, int NBW, int EPI, bool VP = false>
__device__ __forceinline__ void tile_epilogue(const Epi& e, const f32x4 (&acc)[MB][NBW], const RmsPre& rpre,
                                              QkvPre (&qpre)[(MB + 1) / 2], int m0, int n0, int nt, int s, int M,
                                              int K, const VpNoise<MB, NBW>* nz = nullptr) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, g = lane >> 4;
  if constexpr (EPI == EPI_QKV) {
    // the tile is one head (column tile nt = head slot) for 32 or 64 tokens:
    // per 32 tokens, stage them in LDS, then 8 threads per token finish them
    // (16 dims each: d and d + 64 of 8 rotary pairs)
    static_assert((MB == 2 || MB == 4) && NBW == 2, "EPI_QKV needs 32 x 128 or 64 x 128 tiles");
    __shared__ float T[32][128 + 4];
#pragma unroll
    for (int p = 0; p < MB / 2; ++p) {
      const int mt = m0 + 32 * p + (threadIdx.x >> 3);
      qkv_pre_tab(e.qkv, mt, M, nt, threadIdx.x & 7, qpre[p]);  // in flight while staging
      if (p > 0) __syncthreads();  // the previous pass's readers are done with T
#pragma unroll
      for (int mh = 0; mh < 2; ++mh)
#pragma unroll
        for (int j = 0; j < NBW; ++j)
#pragma unroll
          for (int i = 0; i < 4; ++i) T[16 * mh + 4 * g + i][16 * (wave * NBW + j) + r] = acc[2 * p + mh][j][i];
      __syncthreads();
      qkv_finish(e.qkv, T[threadIdx.x >> 3], mt, M, nt, threadIdx.x & 7, qpre[p]);
    }
  } else {
    // folded RMSNorm (RELU2 reading the bf16 copy of x): acc row
    // 16 mb + 4 g + i takes the factor lane 4 g + i computed for its row
    float rsc[MB][4];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int i = 0; i < 4; ++i) rsc[mb][i] = 1.f;
    if constexpr (EPI == EPI_RELU2) {
      if (e.rms_in != nullptr) {
        constexpr int MT = 16 * MB;
        __shared__ float rowinv[MT];
        const float inv = rms_finish<MT>(rpre, e, K);
        if (threadIdx.x % (256 / MT) == 0) rowinv[threadIdx.x / (256 / MT)] = inv;
        __syncthreads();
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
#pragma unroll
          for (int i = 0; i < 4; ++i) rsc[mb][i] = rowinv[16 * mb + 4 * g + i];
      }
    }
    if constexpr (VP && EPI == EPI_SOFTCAP && MB % 2 == 0) {
      if (e.vp != nullptr) {
        f32x4 z[MB][NBW];
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
#pragma unroll
          for (int j = 0; j < NBW; ++j) z[mb][j] = acc[mb][j];
        vocab_tile_parts<MB, NBW>(e, z, m0, n0, nt, M, nz);
        return;
      }
    }
    Epi ee = e;
    ee.split = s;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int j = 0; j < NBW; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int m = m0 + 16 * mb + 4 * g + i;
          if (m < M) epi_apply<EPI, true>(ee, m, n0 + 16 * (wave * NBW + j) + r, acc[mb][j][i] * rsc[mb][i]);
        }
  }
}

// bf16 MFMA GEMM for larger row counts, A shared through LDS.
//
// A workgroup owns an MT x NT tile (MT = 16 MB rows, NT = 64 NBW columns);
// its four waves split the columns (each 16 NBW of them, all MT rows), so
// each wave streams only its own weight fragments, straight into registers,
// while the activation tile of a 64-wide k chunk (2 MB blocks of 1 KB in
// fragment order) is fetched once per workgroup and shared in LDS. Per
// output this moves (MT + NT) / (MT NT) of the operand bytes through L2,
// half of what the K-split kernel's 32 x 64 tile moves at MT = 64, NT = 128.
// Both operands are loaded NS chunks ahead in a register ring; the A chunk
// is written to the LDS double buffer one chunk before it is used.
// Grid and tile order as in k_gemm_ks.
template <int MB, int NBW, int NS, int EPI>
__global__ __launch_bounds__(256) void k_gemm_la(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W,
                                                 int Mcap, const int* __restrict__ Mdev, int N, int K, int ntiles,
                                                 int S, int mtiles, int mfast, Epi e) {
  static_assert(MB == 2 || MB == 4 || MB == 8 || MB == 16, "MB in {2, 4, 8, 16}");
  constexpr int MT = 16 * MB, NT = 64 * NBW, AB = 2 * MB / 4;  // A blocks per wave per chunk
  __shared__ uint4 As[2][2 * MB][64];
  const int id = blockIdx.x;
  const int ntiles8 = (ntiles + 7) & ~7;
  int nt, s, mt;
  if (mfast) {
    const int xcd = id & 7, loc = id >> 3, per = S * mtiles;
    const int nl = loc / per, rem = loc - nl * per;
    s = rem / mtiles;
    mt = rem - s * mtiles;
    nt = nl * 8 + xcd;
  } else {
    nt = id % ntiles8;
    const int rest = id / ntiles8;
    s = rest % S;
    mt = rest / S;
  }
  if (nt >= ntiles) return;
  const int M = Mdev ? min(*Mdev, Mcap) : Mcap;
  const int m0 = mt * MT;
  if (m0 >= M) return;
  const int n0 = nt * NT;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int C = K >> 6;
  const int c_beg = (int)((int64_t)s * C / S), c_end = (int)((int64_t)(s + 1) * C / S);
  const int n = c_end - c_beg;
  const int64_t KS32 = K >> 5;
  // this wave's A blocks of a chunk: q = wave + 4 u, row block q / 2, k step q % 2
  const int last_blk = (M - 1) >> 4;
  const bf16_t* abase[AB];
#pragma unroll
  for (int u = 0; u < AB; ++u) {
    const int q = wave + 4 * u;
    abase[u] = A + ((int64_t)min(m0 / 16 + q / 2, last_blk) * KS32 + (q & 1)) * 512 + lane * 8;
  }
  const bf16_t* wbase[NBW];
#pragma unroll
  for (int j = 0; j < NBW; ++j) wbase[j] = W + (int64_t)(n0 / 16 + wave * NBW + j) * KS32 * 512 + lane * 8;

  RmsPre rpre;  // folded RMSNorm: this thread's share of row m0 + t / (256 / MT)
  if constexpr (EPI == EPI_RELU2) {
    if (e.rms_in != nullptr) rms_load<16 * MB>(rpre, e, m0, M);
  }
  QkvPre qpre[(MB + 1) / 2];  // EPI_QKV: cache row / position of this thread's token in each 32-row pass
  if constexpr (EPI == EPI_QKV) {
#pragma unroll
    for (int p = 0; p < MB / 2; ++p) qkv_pre_row(e.qkv, m0 + 32 * p + (threadIdx.x >> 3), M, nt, qpre[p]);
  }
  // EPI_SOFTCAP draw noise: the row's round counter loads ahead of the
  // operands, so waiting for it does not wait for them
  VpNoise<MB, NBW> nz;
  nz.ok = false;
  int vp_rnd = 0;
  if constexpr (EPI == EPI_SOFTCAP && MB == 2) {
    const int mrow = m0 + (threadIdx.x >> 3);
    if (vp_noise_wanted<MB, NBW>(e) && mrow < M) vp_rnd = e.vp_round[mrow];
  }
  f32x4 acc[MB][NBW];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NBW; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  if (n > 0) {
    v4u wr[NS][NBW][2], ar[NS][AB];
#define LA_LOAD(slot, i)                                                              \
  {                                                                                   \
    const int c_ = c_beg + min((i), n - 1);                                           \
    _Pragma("unroll") for (int j = 0; j < NBW; ++j)                                   \
      _Pragma("unroll") for (int ks = 0; ks < 2; ++ks)                                \
        wr[slot][j][ks] = EPI == EPI_SOFTCAP ? LM_LD((const v4u*)(wbase[j] + (2 * c_ + ks) * 512)) \
                                             : W_LD((const v4u*)(wbase[j] + (2 * c_ + ks) * 512));   \
    _Pragma("unroll") for (int u = 0; u < AB; ++u)                                    \
      ar[slot][u] = *(const v4u*)(abase[u] + (int64_t)c_ * 1024);                     \
  }
#define LA_STAGE_A(slot, buf)                                                         \
  {                                                                                   \
    _Pragma("unroll") for (int u = 0; u < AB; ++u)                                    \
      As[buf][wave + 4 * u][lane] = __builtin_bit_cast(uint4, ar[slot][u]);           \
  }
#pragma unroll
    for (int p = 0; p < NS; ++p) LA_LOAD(p, p);
    if constexpr (EPI == EPI_SOFTCAP && MB == 2) vp_noise<MB, NBW>(e, m0, n0, vp_rnd, nz);
    LA_STAGE_A(0, 0);
    __syncthreads();
    for (int i0 = 0; i0 < n; i0 += NS) {
#pragma unroll
      for (int p = 0; p < NS; ++p) {
        const int i = i0 + p;
        const int buf = i & 1;
        if (i < n) {
#pragma unroll
          for (int ks = 0; ks < 2; ++ks)
#pragma unroll
            for (int mb = 0; mb < MB; ++mb) {
              const v4u a = __builtin_bit_cast(v4u, As[buf][2 * mb + ks][lane]);
#pragma unroll
              for (int j = 0; j < NBW; ++j) acc[mb][j] = mfma16(a, wr[p][j][ks], acc[mb][j]);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        // next chunk's A into the other LDS buffer (its last reader was
        // chunk i - 1, finished before the previous barrier), then refill
        // the freed ring slots
        LA_STAGE_A((p + 1) % NS, buf ^ 1);
        __builtin_amdgcn_sched_barrier(0);
        LA_LOAD(p, i + NS);
        __syncthreads();
      }
    }
#undef LA_LOAD
#undef LA_STAGE_A
  }

  tile_epilogue<MB, NBW, EPI, true>(e, acc, rpre, qpre, m0, n0, nt, s, M, K, &nz);
}

// bf16 MFMA GEMM for verify-size row counts with both operands staged in an
// LDS ring by direct global-to-LDS loads.
//
// Same tile and column split as k_gemm_la (MT = 16 MB rows, NT = 64 NBW
// columns, each wave owns 16 NBW columns), but the activation blocks and the
// wave's own weight blocks of a 64-wide k chunk go straight from global
// memory into one of four LDS stages (no registers held by loads in flight):
// while chunk i computes, chunks i+1 and i+2 are loading. The compiler does not
// see the loads (lds_load_1k), so each step waits itself for the chunk it needs
// (vmcnt(two chunks' loads)), then a plain barrier makes every wave's part of
// the stage visible. The stage refilled at step i is the one
// read at step i-1, which every wave has finished by the barrier of step i.
// Grid and tile order as in k_gemm_la.
template <int MB, int NBW>
struct DmaStage {
  uint4 a[2 * MB][64];
  uint4 w[4][2 * NBW][64];
};
template <int MB, int NBW, int EPI>
__global__ __launch_bounds__(256) void k_gemm_dma(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W,
                                                  int Mcap, const int* __restrict__ Mdev, int N, int K, int ntiles,
                                                  int mtiles, int mfast, Epi e) {
  constexpr int WAVES = 4, AB = 2 * MB, NSTG = 4;
  static_assert(AB % WAVES == 0, "the A blocks of a chunk split evenly over the waves");
  __shared__ DmaStage<MB, NBW> s0, s1, s2, s3;
  const int id = blockIdx.x;
  const int ntiles8 = (ntiles + 7) & ~7;
  int nt, mt;
  if (mfast) {
    const int xcd = id & 7, loc = id >> 3;
    const int nl = loc / mtiles;
    mt = loc - nl * mtiles;
    nt = nl * 8 + xcd;
  } else {
    nt = id % ntiles8;
    mt = id / ntiles8;
  }
  if (nt >= ntiles) return;
  const int M = Mdev ? min(*Mdev, Mcap) : Mcap;
  const int m0 = mt * 16 * MB;
  if (m0 >= M) return;
  const int n0 = nt * 64 * NBW;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t KS32 = K >> 5;
  const int C = K >> 6;
  const int last_blk = (M - 1) >> 4;
  const bf16_t* wbase = W + ((int64_t)(n0 / 16 + wave * NBW)) * KS32 * 512;
  const bf16_t* abase[AB / WAVES];
#pragma unroll
  for (int u = 0; u < AB / WAVES; ++u) {
    const int q = wave + WAVES * u;  // row block q / 2, k step q % 2
    abase[u] = A + ((int64_t)min(m0 / 16 + (q >> 1), last_blk) * KS32 + (q & 1)) * 512;
  }
  RmsPre rpre;  // folded RMSNorm: this thread's share of row m0 + t / (256 / MT)
  if constexpr (EPI == EPI_RELU2) {
    if (e.rms_in != nullptr) rms_load<16 * MB>(rpre, e, m0, M);
  }
  QkvPre qpre[(MB + 1) / 2];  // unused: the fused QKV epilogue runs on k_gemm_la and k_gemm_big
  f32x4 acc[MB][NBW];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NBW; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  // loads per chunk and wave: 2 NBW weight blocks + AB / WAVES activation blocks
  constexpr int PER = 2 * NBW + AB / WAVES;
  constexpr int NV = PER * (NSTG - 2);
  static_assert(NV < 64, "vmcnt range");
  const uint32_t voff = lane * 16;
#define DMA_ISSUE(S, c_)                                                                             \
  {                                                                                                  \
    const int c = min((c_), C - 1); /* past the end: harmless re-reads into an unread stage */       \
    const uint32_t lw_ = LDS_ADDR(S.w[0]) + 2048 * NBW * wave, la_ = LDS_ADDR(S.a[0]) + 1024 * wave; \
    _Pragma("unroll") for (int j = 0; j < NBW; ++j)                                                  \
      _Pragma("unroll") for (int ks = 0; ks < 2; ++ks)                                               \
        lds_load_1k(wbase + ((int64_t)j * KS32 + 2 * c + ks) * 512, voff, lw_ + 1024 * (2 * j + ks)); \
    _Pragma("unroll") for (int u = 0; u < AB / WAVES; ++u)                                           \
      lds_load_1k(abase[u] + (int64_t)c * 1024, voff, la_ + 1024 * WAVES * u);                       \
  }
#define DMA_STEP(S, SN, i_)                                                                          \
  {                                                                                                  \
    __builtin_amdgcn_s_waitcnt((NV & 15) | ((NV >> 4) << 14) | (7 << 4) | (15 << 8));                \
    __atomic_signal_fence(__ATOMIC_SEQ_CST);                                                         \
    __builtin_amdgcn_sched_barrier(0);                                                               \
    __builtin_amdgcn_s_barrier();                                                                    \
    __builtin_amdgcn_sched_barrier(0);                                                               \
    __atomic_signal_fence(__ATOMIC_SEQ_CST);                                                         \
    _Pragma("unroll") for (int ks = 0; ks < 2; ++ks) {                                               \
      v4u w[NBW];                                                                                    \
      _Pragma("unroll") for (int j = 0; j < NBW; ++j) w[j] = __builtin_bit_cast(v4u, S.w[wave][2 * j + ks][lane]); \
      _Pragma("unroll") for (int mb = 0; mb < MB; ++mb) {                                            \
        const v4u a = __builtin_bit_cast(v4u, S.a[2 * mb + ks][lane]);                               \
        _Pragma("unroll") for (int j = 0; j < NBW; ++j) acc[mb][j] = mfma16(a, w[j], acc[mb][j]);    \
      }                                                                                              \
    }                                                                                                \
    DMA_ISSUE(SN, (i_) + NSTG - 1);                                                                  \
  }
  DMA_ISSUE(s0, 0);
  DMA_ISSUE(s1, 1);
  DMA_ISSUE(s2, 2);
  int i = 0;
  for (; i + 3 < C; i += 4) {
    DMA_STEP(s0, s3, i);
    DMA_STEP(s1, s0, i + 1);
    DMA_STEP(s2, s1, i + 2);
    DMA_STEP(s3, s2, i + 3);
  }
  if (i < C) DMA_STEP(s0, s3, i);
  if (i + 1 < C) DMA_STEP(s1, s0, i + 1);
  if (i + 2 < C) DMA_STEP(s2, s1, i + 2);
#undef DMA_STEP
#undef DMA_ISSUE
  __builtin_amdgcn_s_waitcnt(0);  // no direct load outlives the workgroup's LDS
  __syncthreads();                // the epilogue may reuse LDS
  tile_epilogue<MB, NBW, EPI>(e, acc, rpre, qpre, m0, n0, nt, 0, M, K);
}

// bf16 MFMA GEMM for verify-size row counts with every operand block in a
// deep LDS ring fed by direct global-to-LDS loads.
//
// A workgroup owns an MT x NT tile (MT = 16 MB rows, NT = 16 NB columns) of
// one K split; its four waves form a WM x (4 / WM) grid over (row blocks,
// column blocks). Per 64-wide k chunk the tile needs 2 MB activation and
// 2 NB weight blocks of 1 KB (fragment order); they go straight into stage
// chunk % NSTG of the ring, PER per wave, with no registers held by loads in
// flight. Step i waits until the wave's own loads of chunk i have landed
// (vmcnt: the NSTG - 2 later chunks may still be in flight), meets the other
// waves at a barrier (so every wave's part of the stage is visible and every
// wave has finished reading stage i - 1), refills stage i - 1 with chunk
// i + NSTG - 1, then reads its fragments of stage i and runs its MFMAs.
// The compiler does not see the loads (lds_load_1k): that wait is the kernel's
// own, and the loop is unrolled over the ring's stages.
// Against the register-staged kernels this keeps NSTG - 1 chunks in flight
// per workgroup instead of one or two: at the cfg4 verify MLP c_proj shape
// (224 rows, N 1536, K 6144, 64 x 96 tiles, K split 4: 256 workgroups) it
// takes 13.4-13.8 us against 15.4 us for the 32 x 64 split-3 tiles of
// k_gemm_ks (weights cycled from HBM). Measured limits: with the weights
// resident in L2 its loads alone run at ~120 GB/s per CU (the L2-resident
// read ceiling), and its LDS traffic (stage writes plus fragment reads,
// 3x the global bytes at a 2 x 2 wave grid) then bounds it; streaming the
// weights from HBM adds ~3 us per launch that the ring depth does not hide.
// Grid: N tile fastest (tile n on XCD n % 8: the M tiles and splits of one
// weight slab share that XCD's L2), then split, then M tile; tiles past the
// device row count exit at once.
template <int TOT>
struct RingStage {
  uint4 blk[TOT][64];
};
template <int MB, int NB, int NSTG, int WM, int EPI>
__global__ __launch_bounds__(256) void k_gemm_ring(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W,
                                                   int Mcap, const int* __restrict__ Mdev, int N, int K, int ntiles,
                                                   int S, Epi e) {
  constexpr int WN = 4 / WM, MBW = MB / WM, NBW = NB / WN;
  static_assert(MB % WM == 0 && NB % WN == 0, "wave grid");
  constexpr int TOT = 2 * MB + 2 * NB, PER = (TOT + 3) / 4, NV = PER * (NSTG - 2);
  static_assert(NV < 64 && NSTG >= 3 && NSTG <= 8, "ring depth / vmcnt range");
  __shared__ RingStage<TOT> s0, s1, s2, s3, s4, s5, s6, s7;  // the first NSTG are used
  const int id = blockIdx.x;
  const int ntiles8 = (ntiles + 7) & ~7;
  const int nt = id % ntiles8;
  const int rest = id / ntiles8;
  const int s = rest % S, mt = rest / S;
  if (nt >= ntiles) return;
  const int M = Mdev ? min(*Mdev, Mcap) : Mcap;
  const int m0 = mt * 16 * MB;
  if (m0 >= M) return;
  const int n0 = nt * 16 * NB;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / WN, wn = wave % WN;
  const int r = lane & 15, g = lane >> 4;
  const int C = K >> 6;
  const int c_beg = (int)((int64_t)s * C / S), c_end = (int)((int64_t)(s + 1) * C / S);
  const int n = c_end - c_beg;
  const int64_t KS32 = K >> 5;
  const int last_blk = (M - 1) >> 4;
  // this wave's blocks of a chunk: q < 2 MB activation row block q / 2, else
  // weight column block (q - 2 MB) / 2; k step q % 2. A wave with fewer than
  // PER distinct blocks repeats the last one (the same bytes into the same
  // LDS slot, harmless).
  const bf16_t* src[PER];
  int dst[PER];
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int q = min(wave + 4 * u, TOT - 1);
    dst[u] = q;
    if (q < 2 * MB) {
      src[u] = A + ((int64_t)min(m0 / 16 + (q >> 1), last_blk) * KS32 + (q & 1)) * 512;
    } else {
      const int j2 = q - 2 * MB;
      src[u] = W + ((int64_t)(n0 / 16 + (j2 >> 1)) * KS32 + (j2 & 1)) * 512;
    }
  }
  RmsPre rpre;  // folded RMSNorm: this thread's share of row m0 + t / (256 / MT)
  if constexpr (EPI == EPI_RELU2) {
    if (e.rms_in != nullptr) rms_load<16 * MB>(rpre, e, m0, M);
  }
  f32x4 acc[MBW][NBW];
#pragma unroll
  for (int i = 0; i < MBW; ++i)
#pragma unroll
    for (int j = 0; j < NBW; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const uint32_t voff = lane * 16;
#define RING_STG(k) (k == 0 ? s0 : k == 1 ? s1 : k == 2 ? s2 : k == 3 ? s3 : k == 4 ? s4 : k == 5 ? s5 : k == 6 ? s6 : s7)
#define RING_ISSUE(k, c_)                                                                                  \
  {                                                                                                        \
    const int64_t cc_ = (int64_t)(c_beg + min((c_), n - 1)) * 1024; /* past the end: harmless re-reads */  \
    const uint32_t l_ = LDS_ADDR(RING_STG(k).blk[0]);                                                      \
    _Pragma("unroll") for (int u = 0; u < PER; ++u) lds_load_1k(src[u] + cc_, voff, l_ + 1024 * dst[u]);   \
  }
#define RING_STEP(k, i_)                                                                                   \
  {                                                                                                        \
    __builtin_amdgcn_sched_barrier(0);                                                                     \
    __builtin_amdgcn_s_waitcnt((NV & 15) | ((NV >> 4) << 14) | (7 << 4) | (15 << 8));                      \
    __atomic_signal_fence(__ATOMIC_SEQ_CST);                                                               \
    __builtin_amdgcn_sched_barrier(0);                                                                     \
    __builtin_amdgcn_s_barrier();                                                                          \
    __builtin_amdgcn_sched_barrier(0);                                                                     \
    __atomic_signal_fence(__ATOMIC_SEQ_CST);                                                               \
    RING_ISSUE(((k) + NSTG - 1) % NSTG, (i_) + NSTG - 1);                                                  \
    _Pragma("unroll") for (int ks = 0; ks < 2; ++ks) {                                                     \
      v4u af[MBW], wf[NBW];                                                                                \
      _Pragma("unroll") for (int i = 0; i < MBW; ++i)                                                      \
        af[i] = __builtin_bit_cast(v4u, RING_STG(k).blk[2 * (wm * MBW + i) + ks][lane]);                   \
      _Pragma("unroll") for (int j = 0; j < NBW; ++j)                                                      \
        wf[j] = __builtin_bit_cast(v4u, RING_STG(k).blk[2 * MB + 2 * (wn * NBW + j) + ks][lane]);          \
      _Pragma("unroll") for (int i = 0; i < MBW; ++i)                                                      \
        _Pragma("unroll") for (int j = 0; j < NBW; ++j) acc[i][j] = mfma16(af[i], wf[j], acc[i][j]);       \
    }                                                                                                      \
  }
  if (n > 0) {
#pragma unroll
    for (int c = 0; c < NSTG - 1; ++c) RING_ISSUE(c, c);
    int i = 0;
    for (; i + NSTG <= n; i += NSTG) {
      RING_STEP(0, i);
      RING_STEP(1, i + 1);
      RING_STEP(2, i + 2);
      if (NSTG > 3) RING_STEP(3 % NSTG, i + 3);
      if (NSTG > 4) RING_STEP(4 % NSTG, i + 4);
      if (NSTG > 5) RING_STEP(5 % NSTG, i + 5);
      if (NSTG > 6) RING_STEP(6 % NSTG, i + 6);
      if (NSTG > 7) RING_STEP(7 % NSTG, i + 7);
    }
    // the last n - i < NSTG chunks sit in stages 0 .. n - i - 1
    if (i < n) RING_STEP(0, i);
    if (i + 1 < n) RING_STEP(1, i + 1);
    if (NSTG > 3 && i + 2 < n) RING_STEP(2, i + 2);
    if (NSTG > 4 && i + 3 < n) RING_STEP(3 % NSTG, i + 3);
    if (NSTG > 5 && i + 4 < n) RING_STEP(4 % NSTG, i + 4);
    if (NSTG > 6 && i + 5 < n) RING_STEP(5 % NSTG, i + 5);
    if (NSTG > 7 && i + 6 < n) RING_STEP(6 % NSTG, i + 6);
  }
#undef RING_STEP
#undef RING_ISSUE
#undef RING_STG
  __builtin_amdgcn_s_waitcnt(0);  // no direct load outlives the workgroup's LDS
  if constexpr (EPI == EPI_RELU2 || EPI == EPI_ADD) {
    // ReLU^2 and the residual add go through the row-major epilogue (the
    // folded RMSNorm works on whole row segments): stage the tile in LDS
    constexpr int MT = 16 * MB, NT = 16 * NB, OPT = MT * NT / 256, TPR = NT / OPT;
    static_assert(OPT >= 1 && NT % OPT == 0, "epilogue tiling");
    __shared__ float red[MT][NT + 4];
#pragma unroll
    for (int mb = 0; mb < MBW; ++mb)
#pragma unroll
      for (int j = 0; j < NBW; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) red[16 * (wm * MBW + mb) + 4 * g + i][16 * (wn * NBW + j) + r] = acc[mb][j][i];
    __syncthreads();
    const int t = threadIdx.x;
    const int row = t / TPR, col0 = (t - row * TPR) * OPT;
    float v[OPT];
#pragma unroll
    for (int c = 0; c < OPT; ++c) v[c] = red[row][col0 + c];
    row_epilogue<EPI, MT, NT>(e, v, row, col0, m0, n0, nt, s, M, K, rpre);
  } else {
    Epi ee = e;
    ee.split = s;
#pragma unroll
    for (int mb = 0; mb < MBW; ++mb)
#pragma unroll
      for (int j = 0; j < NBW; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int m = m0 + 16 * (wm * MBW + mb) + 4 * g + i;
          if (m < M) epi_apply<EPI, true>(ee, m, n0 + 16 * (wn * NBW + j) + r, acc[mb][j][i]);
        }
  }
}

// bf16 MFMA GEMM for prompt and whole-sequence row counts.
//
// A workgroup owns a 64 MB x 64 NB output tile; each of its 2 x 2 waves owns
// MB x NB blocks of 32 x 32 (the 32x32x16 MFMA: with one wave per SIMD it
// keeps the matrix unit ~86% busy, where 16x16x32 chains reach about half).
// Per 32-wide k step the tile needs 4 MB activation and 4 NB weight blocks of
// 1 KB (16 rows x 32 k, fragment order); they go straight from global memory
// into one of four LDS stages by direct loads, MB + NB per wave. The
// 32x32x16 operand of lane l is row l % 32, k 8 (l / 32) .. +7 of a 16-k half:
// 16 bytes that sit in 16-row block (l % 32) / 16 at lane slot
// l % 16 + 16 (2 half + l / 32), so the stored layout feeds it unchanged.
//
// Per step i: wait until stage i+1 has landed (own loads: vmcnt, the two
// later stages may still be in flight) and every wave has finished reading
// stage i into registers (lgkmcnt(0)); one barrier; start reading stage i+1
// into the other fragment set; refill stage i with chunk i+4; then the MFMAs
// of step i run on fragments already in registers.
//
// What bounds a tile: the L2-to-LDS bytes and the LDS reads per MFMA fall with
// the tile's sides (a k step of 32 takes 0.16 us on 128 x 128 tiles, of them
// 0.11 us MFMA at 2.4 GHz, and 0.62 us on 256 x 256, 0.43 us MFMA), against
// how evenly the tiles fill the CUs and how long a tile's fill and epilogue
// stand alone (4.9 against 11.7 us; the smaller tiles share a CU in twos).
// Hence the four tiles and the cost model that picks one (big_tile). Measured,
// us, 256-row tiles alone before: 3056 x 6144 x 1536 91 -> 62 (128 x 192),
// 3056 x 1536 x 6144 128 -> 61 (was 64 x 64), 4096 x 768 x 3072 57 -> 24
// (128 x 128), 8192 x 1536 x 6144 165 -> 128 (1.2 PFLOP/s).
//
// The MFMA takes the weight block as its first operand, so a lane's result
// is row m0 + l % 32 and, per group of four registers, four consecutive
// columns: fp32 outputs are written as float4, and the bf16 fragment-order
// output (ReLU^2, the next GEMM's operand) goes through a 32 x 32 LDS
// transpose per wave (8-byte writes, 16-byte reads). The QKV projection takes
// 128 x 128 tiles, one head each (1904-8192 rows x 4608 x 1536, with its
// attention prologue: 49-126 us, 59-167 us on 256 x 256).
//
// Tile order: tiles are grouped by 1024 rows of M tiles (N tile slower within
// a group) and dealt to the eight XCDs in contiguous ranges, so that the
// workgroups an XCD runs at once share their operand slabs in its L2.
#ifndef FC_BIG_M
#define FC_BIG_M 1024
#endif
#ifndef FC_BIG_MIN_TILES
#define FC_BIG_MIN_TILES 224
#endif
// Wide outputs (the lm_head, N >= 16384) of fewer than FC_BIG_M rows take the
// 256 x 256 tiles from this many rows: the cfg4 verify head (224 rows, 256 tiles) runs 78.7 us on them
// against 92.7 us on the LDS-shared 128 x 128 tiles (kernel trace); the
// round gains ~3 us of it (4.814-4.818 vs 4.817-4.820 ms, alternating builds).
#ifndef FC_BIG_HEAD_M
#define FC_BIG_HEAD_M 200
#endif
template <int MB, int NB>
struct BigStage {
  uint4 a[4 * MB][64];
  uint4 w[4 * NB][64];
};
// Epilogue inputs of a 32 x 32 output block: the lane's four float4 of x and
// of the second operand (EPI_MLPOUT: x0, or the backout capture at the end).
struct BigIn {
  float4 x[4], z[4];
};
template <int EPI>
__device__ __forceinline__ void big_load(const Epi& e, int m, int n, int M, BigIn& in) {
  if constexpr (EPI == EPI_ADD || EPI == EPI_MLPOUT) {
#pragma unroll
    for (int it = 0; it < 4; ++it) {
      const int64_t i = (int64_t)min(m + 8 * it, M - 1) * e.ldo + n;
      in.x[it] = *(const float4*)((const float*)e.out + i);
      if constexpr (EPI == EPI_MLPOUT)
        if (!e.last || !e.capture) in.z[it] = *(const float4*)((e.last ? e.xb : e.x0) + i);
    }
  }
}
template <int EPI>
__device__ __forceinline__ void big_store4(const Epi& e, int m, int n, float4 v, float4 x, float4 z, int split,
                                           float* logit_row) {
  if constexpr (EPI == EPI_STORE) {
    *(float4*)((float*)e.out + (int64_t)m * e.ldo + n) = v;
  } else if constexpr (EPI == EPI_ADD) {
    *(float4*)((float*)e.out + (int64_t)m * e.ldo + n) = float4{x.x + v.x, x.y + v.y, x.z + v.z, x.w + v.w};
  } else if constexpr (EPI == EPI_MLPOUT) {
    const int64_t i = (int64_t)m * e.ldo + n;
    float4* xp = (float4*)((float*)e.out + i);
    const float4 t = float4{x.x + v.x, x.y + v.y, x.z + v.z, x.w + v.w};  // engine.py:161
    if (e.capture) *(float4*)(e.xb + i) = t;                               // engine.py:164
    if (e.last) {                                                          // engine.py:166
      const float4 xb = e.capture ? t : z;
      *xp = float4{t.x - e.lb * xb.x, t.y - e.lb * xb.y, t.z - e.lb * xb.z, t.w - e.lb * xb.w};
    } else {                                                               // engine.py:94
      *xp = float4{e.r * t.x + e.a * z.x, e.r * t.y + e.a * z.y, e.r * t.z + e.a * z.z, e.r * t.w + e.a * z.w};
    }
  } else if constexpr (EPI == EPI_PARTIAL) {  // split-K partial, finished by the next RMSNorm
    *(float4*)(e.part + ((int64_t)split * e.part_rows + m) * e.ldo + n) = v;
  } else if constexpr (EPI == EPI_SOFTCAP) {  // logits row (m / n_out, m % n_out), columns past V dropped
    float* o = logit_row + n;
    const float4 t = float4{softcap15_fast(v.x), softcap15_fast(v.y), softcap15_fast(v.z), softcap15_fast(v.w)};
    if (n + 3 < e.V && (((uintptr_t)o) & 15) == 0) {
      *(float4*)o = t;
    } else {
      if (n < e.V) o[0] = t.x;
      if (n + 1 < e.V) o[1] = t.y;
      if (n + 2 < e.V) o[2] = t.z;
      if (n + 3 < e.V) o[3] = t.w;
    }
  }
}
// NTW: the weights stream non-temporally (one or two M tiles).
template <int EPI, int MB, int NB, bool NTW = false>
__global__ __launch_bounds__(256, MB == 2 ? 2 : 1) void k_gemm_big(
    const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, int Mcap, const int* __restrict__ Mdev, int N, int K,
    int ntiles, int S, Epi e) {
  // MB 32-row by NB 32-column blocks per wave, 2 x 2 waves: tile 64 MB x 64 NB
  constexpr int NSTG = 4, GM = 16 / MB, MT = 64 * MB, NT = 64 * NB;
  static_assert((MB == 2 || MB == 4) && NB >= 2 && NB <= 4, "tile shapes");
  static_assert(EPI != EPI_QKV || NB == 2, "the QKV epilogue takes one head (128 columns) per tile");
  typedef BigStage<MB, NB> Stage;
  __shared__ Stage s0, s1, s2, s3;
  // tile of this workgroup: XCD id % 8 takes an eighth of the live tiles (below
  // the device row count) of all splits, split-major, so that the workgroups
  // of a split share their A and W slabs in few XCDs' L2 (S = 8: split x on
  // XCD x). Within a split, groups of GM M tiles, N tile slower in a group.
  const int M = Mdev ? min(*Mdev, Mcap) : Mcap;
  const int mtiles = (M + MT - 1) / MT, tiles = ntiles * mtiles;
  const int per_xcd = (tiles * S + 7) / 8;
  const int t = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per_xcd || t >= tiles * S) return;
  const int sp = t / tiles, tt = t - sp * tiles;
  const int grp = tt / (GM * ntiles), rr = tt - grp * GM * ntiles;
  const int gm = min(GM, mtiles - grp * GM);
  const int nt = rr / gm, mt = grp * GM + rr % gm;
  const int m0 = mt * MT;
  const int n0 = nt * NT;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int64_t KS32 = K >> 5;
  // this split's 32-deep k steps [c0, c0 + C)
  const int c0 = (int)(sp * KS32 / S), C = (int)((sp + 1) * KS32 / S) - c0;
  const int last_blk = (M - 1) >> 4;
  // this wave's loads: activation row blocks MB wave .. +MB-1 and weight column blocks NB wave .. +NB-1
  const bf16_t* ab[MB];
  const bf16_t* wb[NB];
#pragma unroll
  for (int u = 0; u < MB; ++u)
    ab[u] = A + ((int64_t)min(m0 / 16 + MB * wave + u, last_blk) * KS32 + c0) * 512;
#pragma unroll
  for (int u = 0; u < NB; ++u) wb[u] = W + ((int64_t)(n0 / 16 + NB * wave + u) * KS32 + c0) * 512;
  // this lane's 32x32x16 operand slot: 16-row block offset and lane slot (half 0; +32 for half 1)
  const int sub = (lane & 31) >> 4, slot = (lane & 15) + 16 * (lane >> 5);
  f32x16 acc[MB][NB];
#pragma unroll
  for (int p = 0; p < MB; ++p)
#pragma unroll
    for (int q = 0; q < NB; ++q)
#pragma unroll
      for (int x = 0; x < 16; ++x) acc[p][q][x] = 0.f;
  constexpr int NV = (MB + NB) * (NSTG - 2);
  static_assert(NV < 64, "vmcnt range");
  const uint32_t voff = lane * 16;
#define BIG_ISSUE(S, c_)                                                                                      \
  {                                                                                                           \
    const int c = min((c_), C - 1); /* past the end: harmless re-reads into an unread stage */                \
    const uint32_t la_ = LDS_ADDR(S) + MB * 1024 * wave, lw_ = LDS_ADDR(S) + 4096 * MB + NB * 1024 * wave;    \
    _Pragma("unroll") for (int u = 0; u < MB; ++u)                                                            \
      lds_load_1k(ab[u] + (int64_t)c * 512, voff, la_ + 1024 * u);                                            \
    _Pragma("unroll") for (int u = 0; u < NB; ++u)                                                            \
      lds_load_1k<NTW>(wb[u] + (int64_t)c * 512, voff, lw_ + 1024 * u);        \
  }
#define BIG_SYNC(NVW)                                                                                         \
  {                                                                                                           \
    __builtin_amdgcn_sched_barrier(0); /* the wait must not rise above the previous step's MFMAs */           \
    __builtin_amdgcn_s_waitcnt(((NVW) & 15) | (((NVW) >> 4) << 14) | (7 << 4) | (0 << 8));                  \
    __atomic_signal_fence(__ATOMIC_SEQ_CST);                                                                  \
    __builtin_amdgcn_sched_barrier(0);                                                                        \
    __builtin_amdgcn_s_barrier();                                                                             \
    __builtin_amdgcn_sched_barrier(0);                                                                        \
    __atomic_signal_fence(__ATOMIC_SEQ_CST);                                                                  \
  }
  // fragments of one k step: [half][32-row / 32-column block]
#define BIG_READ(S, WF, AF)                                                                                   \
  {                                                                                                           \
    _Pragma("unroll") for (int h = 0; h < 2; ++h) {                                                           \
      _Pragma("unroll") for (int b = 0; b < NB; ++b)                                                          \
        WF[h][b] = __builtin_bit_cast(v4u, S.w[2 * NB * wn + 2 * b + sub][slot + 32 * h]);                    \
      _Pragma("unroll") for (int b = 0; b < MB; ++b)                                                          \
        AF[h][b] = __builtin_bit_cast(v4u, S.a[2 * MB * wm + 2 * b + sub][slot + 32 * h]);                    \
    }                                                                                                         \
  }
#define BIG_MMA(WF, AF)                                                                                       \
  {                                                                                                           \
    _Pragma("unroll") for (int h = 0; h < 2; ++h)                                                             \
      _Pragma("unroll") for (int p = 0; p < MB; ++p)                                                          \
        _Pragma("unroll") for (int q = 0; q < NB; ++q) acc[p][q] = mfma32(WF[h][q], AF[h][p], acc[p][q]);     \
  }
  // step i: SN = stage of chunk i + 1 (read now; past the last chunk a
  // re-read that nothing uses), SI = stage of chunk i (refilled with chunk i + 4)
#define BIG_STEP(SI, SN, WFC, AFC, WFN, AFN, i_)                                                              \
  if ((i_) < C) {                                                                                             \
    BIG_SYNC(NV);                                                                                             \
    BIG_READ(SN, WFN, AFN);                                                                                   \
    BIG_ISSUE(SI, (i_) + NSTG);                                                                               \
    BIG_MMA(WFC, AFC);                                                                                        \
  }
  v4u wf0[2][NB], af0[2][MB], wf1[2][NB], af1[2][MB];
  BIG_ISSUE(s0, 0);
  BIG_ISSUE(s1, 1);
  BIG_ISSUE(s2, 2);
  BIG_ISSUE(s3, 3);
  BIG_SYNC(3 * (MB + NB));  // chunk 0 landed: at most the 3 later chunks' loads outstanding
  BIG_READ(s0, wf0, af0);
  for (int i = 0; i < C; i += NSTG) {
    BIG_STEP(s0, s1, wf0, af0, wf1, af1, i);
    BIG_STEP(s1, s2, wf1, af1, wf0, af0, i + 1);
    BIG_STEP(s2, s3, wf0, af0, wf1, af1, i + 2);
    BIG_STEP(s3, s0, wf1, af1, wf0, af0, i + 3);
  }
#undef BIG_STEP
#undef BIG_MMA
#undef BIG_READ
#undef BIG_SYNC
#undef BIG_ISSUE
  __builtin_amdgcn_s_waitcnt(0);  // no direct load outlives the workgroup's LDS
  __syncthreads();                // stage s0 becomes the epilogue's scratch
  // lane l holds row 32 p + l % 32 of the quadrant; register 4 j + x holds
  // column 32 q + 8 j + 4 (l / 32) + x
  const int rl = lane & 31, ch = 4 * (lane >> 5);
  if constexpr (EPI == EPI_QKV) {
    // the tile is one head slot: the two waves of a row half stage 16 tokens
    // at a time in one LDS stage and finish them, eight lanes per token
    float(*T)[128 + 4] = wm == 0 ? (float(*)[128 + 4])&s0 : (float(*)[128 + 4])&s1;
    static_assert(sizeof(Stage) >= 16 * 132 * 4, "16 staging rows");
    const int hh = n0 >> 7, tk = 8 * wn + (lane >> 3);
    QkvPre pre[2 * MB];
#pragma unroll
    for (int u = 0; u < 2 * MB; ++u) qkv_pre_row(e.qkv, m0 + 32 * MB * wm + 16 * u + tk, M, hh, pre[u]);
#pragma unroll
    for (int u = 0; u < 2 * MB; ++u) {
      const int m = m0 + 32 * MB * wm + 16 * u + tk;
      qkv_pre_tab(e.qkv, m, M, hh, lane & 7, pre[u]);
      if ((lane & 31) >> 4 == (u & 1)) {
#pragma unroll
        for (int q = 0; q < NB; ++q)
#pragma unroll
          for (int j = 0; j < 4; ++j)
            *(float4*)&T[lane & 15][64 * wn + 32 * q + 8 * j + ch] =
                float4{acc[u >> 1][q][4 * j], acc[u >> 1][q][4 * j + 1], acc[u >> 1][q][4 * j + 2],
                       acc[u >> 1][q][4 * j + 3]};
      }
      __syncthreads();
      qkv_finish(e.qkv, T[tk], m, M, hh, lane & 7, pre[u]);
      __syncthreads();
    }
  } else if constexpr (EPI == EPI_RELU2) {
    // bf16 fragment order: per 32 x 32 block, lane l writes row l % 32,
    // columns 8 j + 4 (l / 32) .. +3 into a 32 x 80 B scratch; then per
    // 16-row half, lane L reads row L % 16, columns 8 (L / 16) .. +7
    char* scr = (char*)&s0 + wave * 32 * 80;
    bf16_t* out = (bf16_t*)e.out;
    const int KB = e.ldo >> 5;
#pragma unroll
    for (int p = 0; p < MB; ++p) {
#pragma unroll
      for (int q = 0; q < NB; ++q) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          uint32_t pk[2];
#pragma unroll
          for (int hh = 0; hh < 2; ++hh) {
            const float x0 = fmaxf(acc[p][q][4 * j + 2 * hh], 0.f), x1 = fmaxf(acc[p][q][4 * j + 2 * hh + 1], 0.f);
            pk[hh] = pack2bf(x0 * x0, x1 * x1);
          }
          *(uint2*)(scr + rl * 80 + (8 * j + ch) * 2) = uint2{pk[0], pk[1]};
        }
        const int kb = (n0 + 32 * NB * wn + 32 * q) >> 5;
#pragma unroll
        for (int hs = 0; hs < 2; ++hs) {
          const uint4 val = *(const uint4*)(scr + (16 * hs + (lane & 15)) * 80 + 16 * (lane >> 4));
          const int rb = (m0 + 32 * MB * wm + 32 * p + 16 * hs) >> 4;
          if (16 * rb < M) *(uint4*)(out + ((int64_t)rb * KB + kb) * 512 + lane * 8) = val;
        }
      }
    }
  } else {
    // per 32 x 32 block through this wave's LDS scratch (rows of 36 floats): a
    // lane then holds row lane / 8 + 8 it, columns 4 (lane % 8) .. +3, so each
    // access covers whole 128-byte lines of 8 rows. From the accumulators it
    // would be 32 bytes of 32 rows: with rows a power of two apart (logits of
    // 65536 entries) the lines left the L2 in pieces (4096 x 65536 x 768 with
    // the softcap: 970 us, 727 so, 640 with the softcap's shorter form; the MLP
    // c_proj's residual update 3056 x 1536 x 6144 87 -> 65). The next block's residual inputs are loaded
    // before this block's stores, which would otherwise stand ahead of them.
    // Block k + 1 is read back while block k is finished, k + 2 written.
    float* scr = (float*)(wave == 0 ? &s0 : wave == 1 ? &s1 : wave == 2 ? &s2 : &s3);
    constexpr int NBLK = MB * NB, SCR = 32 * 36;
    static_assert(sizeof(Stage) >= 2 * SCR * 4, "a wave's two scratch blocks");
    const int mr = m0 + 32 * MB * wm + (lane >> 3), nc = n0 + 32 * NB * wn + 4 * (lane & 7);
    BigIn in[2];
    float4 v[2][4];
    float* lrow[4] = {nullptr, nullptr, nullptr, nullptr};  // EPI_SOFTCAP: the lane's four logits rows
    auto put = [&](int k) {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        *(float4*)(scr + (k & 1) * SCR + rl * 36 + 8 * j + ch) =
            float4{acc[k / NB][k % NB][4 * j], acc[k / NB][k % NB][4 * j + 1], acc[k / NB][k % NB][4 * j + 2],
                   acc[k / NB][k % NB][4 * j + 3]};
    };
    auto get = [&](int k) {
#pragma unroll
      for (int it = 0; it < 4; ++it)
        v[k & 1][it] = *(const float4*)(scr + (k & 1) * SCR + (8 * it + (lane >> 3)) * 36 + 4 * (lane & 7));
      big_load<EPI>(e, mr + 32 * (k / NB), nc + 32 * (k % NB), M, in[k & 1]);
    };
    put(0);
    __builtin_amdgcn_wave_barrier();
    get(0);
    put(1);
#pragma unroll
    for (int k = 0; k < NBLK; ++k) {
      const int p = k / NB, q = k % NB;
      if (q == 0 && m0 + 32 * MB * wm + 32 * p >= M) return;  // no rows from here on
      __builtin_amdgcn_wave_barrier();
      if (k + 1 < NBLK) get(k + 1);
      __builtin_amdgcn_wave_barrier();
      if (k + 2 < NBLK) put(k + 2);
      if constexpr (EPI == EPI_SOFTCAP) {
        if (q == 0)
#pragma unroll
          for (int it = 0; it < 4; ++it) {
            const int m = mr + 32 * p + 8 * it, b = m / e.n_out;
            lrow[it] = (float*)e.out + (int64_t)b * e.row_stride + (int64_t)(m - b * e.n_out) * e.V;
          }
      }
#pragma unroll
      for (int it = 0; it < 4; ++it) {
        const int m = mr + 32 * p + 8 * it;
        if (m < M) big_store4<EPI>(e, m, nc + 32 * q, v[k & 1][it], in[k & 1].x[it], in[k & 1].z[it], sp, lrow[it]);
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Dispatch
// ---------------------------------------------------------------------------
#define FC_EPI_SWITCH(mode, CALL)                              \
  switch (mode) {                                              \
    case EPI_STORE: { constexpr int E = EPI_STORE; CALL; break; }     \
    case EPI_ADD: { constexpr int E = EPI_ADD; CALL; break; }         \
    case EPI_RELU2: { constexpr int E = EPI_RELU2; CALL; break; }     \
    case EPI_MLPOUT: { constexpr int E = EPI_MLPOUT; CALL; break; }   \
    case EPI_PARTIAL: { constexpr int E = EPI_PARTIAL; CALL; break; } \
    default: { constexpr int E = EPI_SOFTCAP; CALL; break; }          \
  }

template <typename T, int MB>
static void launch_gemv_mb(const void* A, const void* W, int M, const int* Mdev, int N, int K, const Epi& e,
                           hipStream_t s) {
  const dim3 grid((N + 15) / 16, (M + MB - 1) / MB);
  FC_EPI_SWITCH(e.mode, hipLaunchKernelGGL((k_gemv<T, MB, E>), grid, dim3(256), 0, s, (const T*)A, (const T*)W, M,
                                           Mdev, N, K, e));
}
template <typename T>
static void launch_gemv(const void* A, const void* W, int M, const int* Mdev, int N, int K, const Epi& e,
                        hipStream_t s) {
  if (M <= 1) launch_gemv_mb<T, 1>(A, W, M, Mdev, N, K, e, s);
  else if (M <= 2) launch_gemv_mb<T, 2>(A, W, M, Mdev, N, K, e, s);
  else if (M <= 4) launch_gemv_mb<T, 4>(A, W, M, Mdev, N, K, e, s);
  else launch_gemv_mb<T, 8>(A, W, M, Mdev, N, K, e, s);
}

static void launch_f32(const void* A, const void* W, int Mcap, const int* Mdev, int Mtyp, int N, int K, const Epi& e,
                       hipStream_t s) {
  // 64 x 64 tiles once they give every CU two (a wave per SIMD each); eight
  // waves where a CU has no more than one tile and each has two chunks at least
  const bool wide = (int64_t)((Mtyp + 63) / 64) * ((N + 63) / 64) >= 512;
  const bool few = (int64_t)((Mtyp + 31) / 32) * ((N + 31) / 32) <= 256 && K >= 512;
  const int T = wide ? 64 : 32, ntiles = (N + T - 1) / T, mtiles = (Mcap + T - 1) / T;
  const dim3 grid((unsigned)(ntiles * mtiles));
  const float *a = (const float*)A, *w = (const float*)W;
  if (wide)
    FC_EPI_SWITCH(e.mode,
                  hipLaunchKernelGGL((k_gemm_f32<1, E>), grid, dim3(256), 0, s, a, w, Mcap, Mdev, N, K, ntiles, e))
  else if (few)
    FC_EPI_SWITCH(e.mode,
                  hipLaunchKernelGGL((k_gemm_f32<8, E>), grid, dim3(512), 0, s, a, w, Mcap, Mdev, N, K, ntiles, e))
  else
    FC_EPI_SWITCH(e.mode,
                  hipLaunchKernelGGL((k_gemm_f32<4, E>), grid, dim3(256), 0, s, a, w, Mcap, Mdev, N, K, ntiles, e))
}

// register ring depth of the K-split kernel: 4 chunks for the 32 x 16 and
// 32 x 32 tiles (the draft's weight streams: few columns per wave), else 3
template <int MB, int NB, bool PK = false, int NS = (MB == 2 && NB <= 2) ? 4 : 3>
static void launch_ks(const void* A, const void* W, int Mcap, const int* Mdev, int N, int K, int S, const Epi& e,
                      hipStream_t s) {
  const int ntiles = N / (16 * NB), mtiles = (Mcap + 16 * MB - 1) / (16 * MB);
  const int nwg = (ntiles + 7) / 8 * 8 * S * mtiles;
  const int mfast = Mdev == nullptr ? 1 : 0;
  FC_EPI_SWITCH(e.mode, hipLaunchKernelGGL((k_gemm_ks<MB, NB, NS, E, PK>), dim3(nwg), dim3(256), 0, s,
                                           (const bf16_t*)A, (const bf16_t*)W, Mcap, Mdev, N, K, ntiles, S, mtiles,
                                           mfast, e));
}

#define FC_GEMM_LA_NS 3
template <int MB, int NBW>
static void launch_la(const void* A, const void* W, int Mcap, const int* Mdev, int N, int K, int S, const Epi& e,
                      hipStream_t s) {
  const int ntiles = N / (64 * NBW), mtiles = (Mcap + 16 * MB - 1) / (16 * MB);
  const int nwg = (ntiles + 7) / 8 * 8 * S * mtiles;
  const int mfast = Mdev == nullptr ? 1 : 0;
  FC_EPI_SWITCH(e.mode, hipLaunchKernelGGL((k_gemm_la<MB, NBW, FC_GEMM_LA_NS, E>), dim3(nwg), dim3(256), 0, s,
                                           (const bf16_t*)A, (const bf16_t*)W, Mcap, Mdev, N, K, ntiles, S, mtiles,
                                           mfast, e));
}

template <int MB, int NBW>
static void launch_dma(const void* A, const void* W, int Mcap, const int* Mdev, int N, int K, const Epi& e,
                       hipStream_t s) {
  const int ntiles = N / (64 * NBW), mtiles = (Mcap + 16 * MB - 1) / (16 * MB);
  const int nwg = (ntiles + 7) / 8 * 8 * mtiles;
  const int mfast = Mdev == nullptr ? 1 : 0;
  FC_EPI_SWITCH(e.mode, hipLaunchKernelGGL((k_gemm_dma<MB, NBW, E>), dim3(nwg), dim3(256), 0, s, (const bf16_t*)A,
                                           (const bf16_t*)W, Mcap, Mdev, N, K, ntiles, mtiles, mfast, e));
}

// the ring tiles: 64 x 96 with 5 stages (verify c_fc and MLP c_proj), 32 x 32
// with 4 (verify attention c_proj); 2 x 2 waves
template <int MB, int NB, int NSTG, int WM>
static void launch_ring(const void* A, const void* W, int Mcap, const int* Mdev, int N, int K, int S, const Epi& e,
                        hipStream_t s) {
  const int ntiles = N / (16 * NB), mtiles = (Mcap + 16 * MB - 1) / (16 * MB);
  const int nwg = (ntiles + 7) / 8 * 8 * S * mtiles;
  FC_EPI_SWITCH(e.mode, hipLaunchKernelGGL((k_gemm_ring<MB, NB, NSTG, WM, E>), dim3(nwg), dim3(256), 0, s,
                                           (const bf16_t*)A, (const bf16_t*)W, Mcap, Mdev, N, K, ntiles, S, e));
}

template <int EPI, int MB, int NB, bool NTW = false>
static void launch_big_e(const void* A, const void* W, int Mcap, const int* Mdev, int N, int K, int S, const Epi& e,
                         hipStream_t s) {
  const int ntiles = N / (64 * NB), mtiles = (Mcap + 64 * MB - 1) / (64 * MB);
  const int per_xcd = (ntiles * mtiles * S + 7) / 8;
  hipLaunchKernelGGL((k_gemm_big<EPI, MB, NB, NTW>), dim3(8 * per_xcd), dim3(256), 0, s, (const bf16_t*)A,
                     (const bf16_t*)W, Mcap, Mdev, N, K, ntiles, S, e);
}
// 64 mb x 64 nb tiles; S > 1 only with EPI_PARTIAL
static void launch_big(const void* A, const void* W, int Mcap, const int* Mdev, int N, int K, int mb, int nb, int S,
                       const Epi& e, hipStream_t s) {
#define BIG_TILE(E)                                                                      \
  {                                                                                      \
    if (mb == 4 && nb == 4) launch_big_e<E, 4, 4>(A, W, Mcap, Mdev, N, K, S, e, s);      \
    else if (mb == 4) launch_big_e<E, 4, 3>(A, W, Mcap, Mdev, N, K, S, e, s);            \
    else if (nb == 3) launch_big_e<E, 2, 3>(A, W, Mcap, Mdev, N, K, S, e, s);            \
    else launch_big_e<E, 2, 2>(A, W, Mcap, Mdev, N, K, S, e, s);                         \
  }
  switch (e.mode) {
    case EPI_STORE: BIG_TILE(EPI_STORE); break;
    case EPI_ADD: BIG_TILE(EPI_ADD); break;
    case EPI_RELU2: BIG_TILE(EPI_RELU2); break;
    case EPI_MLPOUT: BIG_TILE(EPI_MLPOUT); break;
    case EPI_PARTIAL: BIG_TILE(EPI_PARTIAL); break;
    case EPI_QKV: launch_big_e<EPI_QKV, 2, 2>(A, W, Mcap, Mdev, N, K, 1, e, s); break;  // one head per tile
    default:
      // the lm_head: its weights go past the caches up to two M tiles, which run
      // side by side on an XCD (us, past / through them: 65536 x 768 300 rows 78.0 /
      // 80.4, 512 rows 85.1 / 86.1; 32768 x 768 40.7 / 41.2, 44.1 / 44.9; x 1536 the
      // same); more M tiles share them there (65536 x 1536, 1000 rows: 234 / 232)
      if (mb == 4 && nb == 4 && Mcap <= 512) launch_big_e<EPI_SOFTCAP, 4, 4, true>(A, W, Mcap, Mdev, N, K, S, e, s);
      else BIG_TILE(EPI_SOFTCAP);
      break;
  }
#undef BIG_TILE
}

template <int MB>
static void launch_la_qkv(const void* A, const void* W, int Mcap, const int* Mdev, int N, int K, const Epi& e,
                          hipStream_t s) {
  const int ntiles = N / 128, mtiles = (Mcap + 16 * MB - 1) / (16 * MB);
  const int nwg = (ntiles + 7) / 8 * 8 * mtiles;
  hipLaunchKernelGGL((k_gemm_la<MB, 2, FC_GEMM_LA_NS, EPI_QKV>), dim3(nwg), dim3(256), 0, s, (const bf16_t*)A,
                     (const bf16_t*)W, Mcap, Mdev, N, K, ntiles, 1, mtiles, Mdev == nullptr ? 1 : 0, e);
}

// One plan drives the workspace sizing and the launch. The tile shape and
// the K split are chosen for the typical row count Mtyp (the grid covers
// Mcap rows; tiles past the device-side count exit at once).
struct GemmPlan {
  bool gemv, la, dma, big;  // VALU GEMV (fp32) / LDS-shared-A / LDS-ring / k_gemm_big (else the K-split kernel)
  bool ring;                // deep direct-load ring, 64 x 96 tiles (k_gemm_ring)
  int mb, nb, S;       // k_gemm_ks: 16 mb x 16 nb tile; k_gemm_la, k_gemm_dma: 16 mb x 64 nb; k_gemm_big: 64 mb x 64 nb
};
#ifndef FC_GEMM_DMA
#define FC_GEMM_DMA 1
#endif
#ifndef FC_GEMM_RING
#define FC_GEMM_RING 1
#endif
// The ring tiles for the verify c_fc (64 x 96, ReLU^2 with the folded
// RMSNorm) and the folded-norm attention c_proj (32 x 32): correct (the GPU
// suite passes with them) but not faster in the cfg4 round (alternating
// builds, three runs each: c_fc 4.868-4.881 vs 4.837-4.840 ms, attention
// c_proj 4.833-4.838 ms), so both stay on k_gemm_dma / k_gemm_ks.
#ifndef FC_RING_FC
#define FC_RING_FC 0
#endif
#ifndef FC_RING_APROJ
#define FC_RING_APROJ 0
#endif
// Row counts from which the layer GEMMs that k_gemm_big does not take yet
// (big_rows) use larger tiles (large-batch verify chunks, e.g. 128 rows x 9
// tokens): c_fc on the LDS-shared 128 x 128 tile, QKV with its fused prologue
// on 64 x 128, the folded-norm attention c_proj on 32 x 64, and residual GEMMs
// unsplit on the LDS-ring 64 x 64 tile unless K is deep (big_deep: the MLP
// c_proj). A sweep of the layer shapes at 224 / 448 / 672 / 896 / 1152 rows put
// the crossover between 672 and 896 rows.
#ifndef FC_MID_M
#define FC_MID_M 832
#endif
// column blocks of 64 per tile of the draft lm_head (up to 32 rows): with the
// vocab pass in its epilogue, 32 x 128 tiles (2) measured 4.780-4.788 vs
// 4.773-4.775 ms per cfg4 round (alternating builds)
#ifndef FC_DRAFT_HEAD_NB
#define FC_DRAFT_HEAD_NB 1
#endif
// The k_gemm_big tiles and what one of them costs a CU: fixed + per 32-deep k
// step, in us, from sweeps of 160-8192 rows over N = 768-6144, K = 768-6144.
// A launch takes about the tiles of the busiest CU times that, whether one or
// two workgroups share the CU.
struct BigTile {
  int mb, nb;
  float fixed, step;
};
static const BigTile kBigTiles[] = {{2, 2, 4.9f, 0.16f}, {2, 3, 5.9f, 0.243f}, {4, 3, 9.f, 0.48f}, {4, 4, 11.7f, 0.62f}};

// From more 64 x 64 tiles than two per CU, k_gemm_big is the faster kernel
// (us at N x K: 4608 x 1536 448 rows 11.9 vs 13.8, 640 rows 16.5 vs 15.0;
// 1536 x 1536 1300 rows 12.6 vs 14.4, 1904 rows 20.9 vs 15.2; 768 x 768 1904
// rows 7.9 vs 9.4, 3056 rows 13.4 vs 10.0; at 3056 rows of 6144 x 1536 134 vs 62).
static bool big_rows(int M, int N) {
  if (N >= 16384) return M >= FC_BIG_M && N % 128 == 0;
  return N % 128 == 0 && (int64_t)((M + 63) / 64) * (N / 64) > 512;
}

// A residual GEMM with a deep K (the MLP c_proj) that may split it is the
// faster there from FC_MID_M rows on: with the split its tiles fill the CUs,
// while a 64 x 64 tile of k_gemm_dma walks all of K alone.
// Whole chunks, us, without and with: 4 layers of 1536 at 900 rows 880 / 812, at
// 1152 rows (4 KV heads) 1064 / 1007; of 768 at 1080 rows 611 / 548.
static bool big_deep(int M, int N, int K) { return M >= FC_MID_M && N % 128 == 0 && K >= 2048; }

// The same product without the split (the linear operator). k_gemm_dma's tiles
// go to the XCDs by column (tile n on XCD n % 8), and from 48 of them for an XCD's
// 32 CUs on its rings of two workgroups a CU get in each other's way; where K is
// as deep as c_proj's the large tiles' one round is the faster (us, N x K, at
// 64 x 64 / large): 1536 x 6144 900 rows 31.2 / 35.9, 1000 rows 38.5 / 36.0, 1300
// rows 41.3 / 36.4; 768 x 3072 1365 rows 19.3 / 20.0, 1500 rows 20.7 / 19.8, 2000
// rows 27.4 / 20.2; at K = 2 N 1536 x 3072 1000 rows 17.9 / 20.2.
static bool big_deep_unsplit(int M, int N, int K) {
  return N % 128 == 0 && K >= 2048 && K >= 4 * N && ((N / 64 + 7) / 8) * ((M + 63) / 64) >= 48;
}

// The cheapest tile and K split (S of at most s_max, each split's partials
// written and read back once by the RMSNorm that sums them, at ~4 TB/s). A
// split needs at least 8 k steps. Below 8 k steps (K < 256) the sweeps say
// nothing and it is the 128 x 128 tile: by the prices 1025 x 65536 x 192 would
// take 75 us for 64 and 8192 x 1536 x 192 15.0 for 14.3, against 7.6 for 8.3 at
// 3056 x 1536 x 128.
static void big_tile(int M, int N, int K, int s_max, int& mb, int& nb, int& S) {
  mb = nb = 2;
  S = 1;
  float best = 1e30f;
  for (const BigTile& t : kBigTiles) {
    if (N % (64 * t.nb) != 0) continue;
    const int64_t tiles = (int64_t)((M + 64 * t.mb - 1) / (64 * t.mb)) * (N / (64 * t.nb));
    for (int sp = 1; sp <= s_max && K / 32 >= 8 * sp; sp *= 2) {
      const float part = sp > 1 ? (float)sp * M * N * 8.f / 4e6f : 0.f;
      const float us = (float)((tiles * sp + 255) / 256) * (t.fixed + t.step * (float)(K / 32) / sp) + part;
      if (us < best) {
        best = us;
        mb = t.mb;
        nb = t.nb;
        S = sp;
      }
    }
  }
}

// Tile shape and K split by typical row count, from sweeps on MI355X at the
// engine's shapes (N = 1536 / 4608 / 6144 / 65536, K = 1536 / 6144).
static GemmPlan plan_gemm(int Mtyp, int N, int K, int dtype, bool can_split) {
  GemmPlan p{};
  p.S = 1;
  if (dtype == FC_F32) {
    p.gemv = true;
    return p;
  }
  if (N >= 16384 && Mtyp >= FC_BIG_HEAD_M && N % 256 == 0 && Mtyp < FC_BIG_M) {  // the verify head
    const int mt = (Mtyp + 255) / 256;
    if (mt * (N / 256) >= FC_BIG_MIN_TILES) {
      p.big = true;
      p.mb = p.nb = 4;
      return p;
    }
  }
  if (big_rows(Mtyp, N) || (can_split ? big_deep(Mtyp, N, K) : big_deep_unsplit(Mtyp, N, K))) {
    p.big = true;
    big_tile(Mtyp, N, K, can_split ? FC_MAX_SPLIT : 1, p.mb, p.nb, p.S);
    return p;
  }
  const int C = K / 64;
  const int s_max = std::max(1, std::min(C / 4, FC_MAX_SPLIT));  // >= 1 chunk per wave
  if (Mtyp <= 16) {
    // one 16-row tile: fill the GPU with column tiles and K splits
    p.mb = 1;
    p.nb = 4;
    const int wgs = std::max(1, N / 64);
    if (can_split && wgs < 256) p.S = std::min((256 + wgs - 1) / wgs, s_max);
  } else if (Mtyp <= 32) {
    if (!can_split && N >= 16384 && N % (64 * FC_DRAFT_HEAD_NB) == 0) {  // draft lm_head: LDS-shared rows
      p.la = true;
      p.mb = 2;
      p.nb = FC_DRAFT_HEAD_NB;  // 64-column tiles (or 128)
      return p;
    }
    p.mb = 2;
    p.nb = 2;
    if (can_split) {  // n_embd columns: 16-column tiles and a K split fill the GPU
      p.nb = 1;
      p.S = std::min(K > 2048 ? 8 : 3, s_max);
    }
  } else if (can_split) {
    if (Mtyp >= FC_MID_M && N % 64 == 0 && FC_GEMM_DMA) {  // enough 64 x 64 tiles: no K split
      p.dma = true;
      p.mb = 4;
      p.nb = 1;
      return p;
    }
    // verify chunks below FC_MID_M rows whose residual GEMM has n_embd = a
    // multiple of 96 columns: the deep-ring 64 x 96 tiles with a 4-way split
    // (cfg4's MLP c_proj: 16 x 4 tiles x 4 splits = 256 workgroups)
    if (FC_GEMM_RING && Mtyp > 160 && N % 96 == 0 && C % 4 == 0 && s_max >= 4) {
      p.ring = true;
      p.mb = 4;
      p.nb = 6;
      p.S = 4;
      return p;
    }
    // 33-160 rows (large-batch draft steps): 32 x 32 tiles, 4-way split;
    // from there (verify chunks) 32 x 64, 3-way
    p.mb = 2;
    p.nb = Mtyp <= 160 ? 2 : 4;
    p.S = std::min(Mtyp <= 160 ? 4 : 3, s_max);
  } else if (Mtyp >= 128 && N % 128 == 0) {
    // verify / prefill rows: a wide output (lm_head) takes the LDS-shared
    // kernel's 128 x 128 tiles; the layer GEMMs the LDS-ring kernel's 64 x 64
    // (the fused QKV epilogue takes its 32 x 128: one head per tile)
    if (N >= 16384 || !FC_GEMM_DMA) {
      p.la = true;
      p.mb = N >= 16384 ? 8 : 2;
      p.nb = 2;
    } else {
      p.dma = true;
      p.mb = 4;
      p.nb = 1;
    }
    return p;
  } else {
    p.mb = 2;
    p.nb = 4;
  }
  while (p.nb > 1 && N % (16 * p.nb) != 0) p.nb /= 2;
  if (p.nb == 1 && p.mb != 2) p.nb = 2;  // instantiated shapes: (1,2|4), (2,1|2|4)
  return p;
}

// c_fc (the ReLU^2 epilogue): verify rows (161 .. FC_MID_M - 1) on the ring's
// 64 x 96 tiles; from FC_MID_M rows the LDS-shared 128 x 128 tile
// `fold`: with the folded RMSNorm, which k_gemm_big does not have
static GemmPlan plan_relu2(int Mtyp, int N, int K, int dtype, bool fold) {
  GemmPlan p = plan_gemm(Mtyp, N, K, dtype, false);
  if (fold && p.big) {  // the next best tiles of these row counts: 64 x 64
    p = GemmPlan{};
    p.S = 1;
    p.dma = true;
    p.mb = 4;
    p.nb = 1;
  }
  if (FC_GEMM_RING && FC_RING_FC && dtype == FC_BF16 && !p.big && Mtyp > 160 && Mtyp < FC_MID_M && N % 96 == 0) {
    p = GemmPlan{};
    p.S = 1;
    p.ring = true;
    p.mb = 4;
    p.nb = 6;
    return p;
  }
  if (dtype == FC_BF16 && !p.big && Mtyp >= FC_MID_M && N % 128 == 0) {
    p = GemmPlan{};
    p.S = 1;
    p.la = true;
    p.mb = 8;
    p.nb = 2;
  }
  return p;
}

// Up to this many typical rows (one-row decode: cfg2's 5-token verify and
// 1-token draft steps) the QKV GEMM takes one-head 32 x 128 tiles and
// finishes the attention prologue itself, saving the k_prologue dispatch:
// cfg2 0.923-0.927 vs 0.952-0.956 ms per round (alternating builds). At 32
// rows (cfg4's draft steps: 36 workgroups over 14 MB) the separate
// prologue is faster.
#ifndef FC_QKV_TINY_M
#define FC_QKV_TINY_M 16
#endif
bool fc_gemm_fuses_qkv(int Mtyp, int N, int K, int dtype, int head_dim) {
  if (dtype != FC_BF16 || head_dim != 128 || N % 128 != 0 || K % 64 != 0) return false;
  if (Mtyp <= FC_QKV_TINY_M) return true;
  const GemmPlan p = plan_gemm(Mtyp, N, K, dtype, false);
  // the QKV tile itself is k_gemm_la's 32 x 128 (64 x 128 from FC_MID_M rows), or k_gemm_big's 128 x 128
  return p.big || p.dma || (p.la && p.mb == 2 && p.nb == 2);
}

// The EPI_ADD GEMM that writes the bf16 copy of x (attention c_proj, bf16):
// unsplit K-split kernel, 32 x 16 tiles for draft rows, 32 x 32 for verify rows.
static GemmPlan plan_fold_add(int Mtyp, int N) {
  GemmPlan p{};
  p.S = 1;
  if (FC_GEMM_RING && FC_RING_APROJ && Mtyp > 160 && Mtyp < FC_MID_M && N % 32 == 0) {  // verify rows: the ring's 32 x 32 tiles
    p.ring = true;
    p.mb = 2;
    p.nb = 2;
    return p;
  }
  p.mb = Mtyp <= 16 ? 1 : 2;
  p.nb = Mtyp <= 16 ? 2 : (Mtyp <= 32 ? 1 : (Mtyp < FC_MID_M ? 2 : 4));
  while (p.nb > 1 && N % (16 * p.nb) != 0) p.nb /= 2;
  if (p.nb == 1 && p.mb != 2) p.nb = 2;
  return p;
}
int fc_gemm_fold_tiles(int Mtyp, int N) { return N / (16 * plan_fold_add(Mtyp, N).nb); }
// The consumer (c_fc: N = 4 D, K = D) prefetches FC_RMS_REG tiles per thread
// with 256 / MT threads per row. c_fc on k_gemm_big gives the fold up: an RMSNorm
// launch and a split attention c_proj more per layer (about 8 us), which pays
// where c_fc gains more, from 2^31 multiply-adds, or where the MLP c_proj has
// the large tiles too (FC_MID_M rows, big_deep). Whole steps of 8 layers, us,
// folded / not: n_embd 768, 648 rows 557 / 583, 810 rows 645 / 665, 837 rows 683 / 650;
// n_embd 1024, 648 rows 774 / 761; 1536, 324 rows 773 / 770, 648 rows 1156 / 1124.
bool fc_gemm_fold_ok(int Mtyp, int D) {
  const bool big_pays = Mtyp >= FC_MID_M || (int64_t)Mtyp * 4 * D * D >= (int64_t)1 << 31;
  const GemmPlan c = plan_relu2(Mtyp, 4 * D, D, FC_BF16, !big_pays);
  return !c.gemv && !c.big && fc_gemm_fold_tiles(Mtyp, D) <= FC_RMS_REG * (256 / (16 * c.mb));
}

int64_t fc_gemm_part_bytes(int Mtyp, int Mcap, int N, int K, int dtype) {
  if (Mtyp <= 0 || Mcap <= 0 || N <= 0 || K <= 0) return 0;
  GemmPlan p = plan_gemm(Mtyp, N, K, dtype, true);  // fp32 GEMMs never split
  return p.S > 1 ? fc_align((int64_t)p.S * Mcap * N * 4) : 0;
}

int fc_launch_gemm(const void* A, const void* W, int Mcap, const int* Mdev, int Mtyp, int N, int K, int dtype,
                   const Epi& e, const GemmWork& gw, hipStream_t s, int* splits) {
  if (splits) *splits = 1;
  if (Mcap <= 0 || N <= 0) return FC_OK;
  FC_CHECK_ARG(K > 0 && K % 8 == 0, "gemm K must be a positive multiple of 8");
  if (Mtyp <= 0 || Mtyp > Mcap) Mtyp = Mcap;
  FC_CHECK_ARG(dtype == FC_F32 || (K % 64 == 0 && N % 32 == 0),
               "bf16 GEMM needs K % 64 == 0 and N % 32 == 0 (fragment-order operands)");
  if (e.mode == EPI_QKV) {
    FC_CHECK_ARG(fc_gemm_fuses_qkv(Mtyp, N, K, dtype, 128),
                 "EPI_QKV needs bf16, head_dim 128 and a plan with one head (128 columns) per tile");
    const GemmPlan q = plan_gemm(Mtyp, N, K, dtype, false);
    if (q.big) launch_big(A, W, Mcap, Mdev, N, K, q.mb, q.nb, 1, e, s);
    else if (Mtyp >= FC_MID_M) launch_la_qkv<4>(A, W, Mcap, Mdev, N, K, e, s);  // 64 x 128 tiles
    else launch_la_qkv<2>(A, W, Mcap, Mdev, N, K, e, s);
    FC_LAUNCH_CHECK();
    return FC_OK;
  }
  const bool can_split = splits != nullptr && gw.part != nullptr;
  GemmPlan p = e.mode == EPI_RELU2 && !can_split ? plan_relu2(Mtyp, N, K, dtype, e.rms_in != nullptr)
                                                  : plan_gemm(Mtyp, N, K, dtype, can_split);
  if (e.mode == EPI_ADD && e.xa != nullptr) {
    FC_CHECK_ARG(dtype == FC_BF16 && e.ssq != nullptr && !can_split, "folded-norm GEMM: bf16, ssq, no split");
    p = plan_fold_add(Mtyp, N);
  }
  if (p.S > 1 && (int64_t)p.S * Mcap * N * 4 > gw.part_bytes) p.S = 1;
  FC_CHECK_ARG(e.vp == nullptr || (e.mode == EPI_SOFTCAP && p.la && p.S == 1 && p.mb % 2 == 0 &&
                                   e.vp_ld == N / (64 * (p.mb == 8 || p.nb != 1 ? 2 : 1))),
               "vocab-pass partials: an unsplit EPI_SOFTCAP GEMM on the LDS-shared kernel, vp_ld = its column tiles");
  Epi ee = e;
  if (p.S > 1) {
    ee.mode = EPI_PARTIAL;
    ee.part = gw.part;
    ee.part_rows = Mcap;
    ee.ldo = N;
    *splits = p.S;
  }
  if (p.gemv) {
    // Up to 16 rows k_gemv reads the weights twice at most (16 x 256 x 1024: 11.5 us
    // against 12); where the 32 x 32 tiles leave three CUs in four without one
    // and K is long, its column per wave spreads the work better (24 x 768 x 3072:
    // 22.5 against 28). The tiles' 16-byte loads want their operands on that boundary.
    const bool starved = (int64_t)((Mtyp + 31) / 32) * ((N + 31) / 32) <= 64 && K > 1024;
    if (Mtyp <= GEMV_MAX_M || starved || (((uintptr_t)A | (uintptr_t)W) & 15) != 0)
      launch_gemv<float>(A, W, Mcap, Mdev, N, K, ee, s);
    else launch_f32(A, W, Mcap, Mdev, Mtyp, N, K, ee, s);
  } else if (p.big) {
    FC_CHECK_ARG(ee.rms_in == nullptr && ee.xa == nullptr, "k_gemm_big has no folded-norm epilogue");
    launch_big(A, W, Mcap, Mdev, N, K, p.mb, p.nb, p.S, ee, s);
  } else if (p.ring) {
    if (p.mb == 2) launch_ring<2, 2, 4, 2>(A, W, Mcap, Mdev, N, K, p.S, ee, s);  // 32 x 32, 4 stages
    else launch_ring<4, 6, 5, 2>(A, W, Mcap, Mdev, N, K, p.S, ee, s);           // 64 x 96, 5 stages
  } else if (p.dma) {
    launch_dma<4, 1>(A, W, Mcap, Mdev, N, K, ee, s);
  } else if (p.la) {
    if (p.mb == 8) launch_la<8, 2>(A, W, Mcap, Mdev, N, K, p.S, ee, s);
    else if (p.nb == 1) launch_la<2, 1>(A, W, Mcap, Mdev, N, K, p.S, ee, s);
    else launch_la<2, 2>(A, W, Mcap, Mdev, N, K, p.S, ee, s);
  } else if (p.mb == 1) {
    if (p.nb == 4) launch_ks<1, 4, true>(A, W, Mcap, Mdev, N, K, p.S, ee, s);
    else launch_ks<1, 2, true>(A, W, Mcap, Mdev, N, K, p.S, ee, s);
  } else {
    if (p.nb == 4) launch_ks<2, 4, true>(A, W, Mcap, Mdev, N, K, p.S, ee, s);
    else if (p.nb == 2) launch_ks<2, 2, true>(A, W, Mcap, Mdev, N, K, p.S, ee, s);
    else launch_ks<2, 1, true>(A, W, Mcap, Mdev, N, K, p.S, ee, s);
  }
  FC_LAUNCH_CHECK();
  return FC_OK;
}

int fc_gemm_vocab_tiles(int M, int N, int K, int dtype) {
  if (M <= 0 || N <= 0 || dtype != FC_BF16 || K % 64 != 0 || N % 32 != 0) return 0;
  const GemmPlan p = plan_gemm(M, N, K, dtype, false);
  if (!p.la || p.S != 1 || p.mb % 2 != 0) return 0;
  return N / (64 * (p.mb == 8 || p.nb != 1 ? 2 : 1));  // launch_la<8, 2>, <2, 1> or <2, 2>
}

extern "C" int32_t fc_gemm(const void* A, const void* W, void* out, int32_t M, int32_t N, int32_t K, int32_t dtype,
                           int32_t epi, void* stream) {
  FC_CHECK_ARG(A && W && out, "null pointer");
  FC_CHECK_ARG(dtype == FC_F32 || dtype == FC_BF16, "dtype");
  FC_CHECK_ARG(epi == EPI_STORE || epi == EPI_ADD || epi == EPI_RELU2 || epi == EPI_SOFTCAP, "epilogue");
  Epi e{};
  e.mode = epi;
  e.out = out;
  e.ldo = N;
  e.out_dtype = dtype;
  e.n_out = 1;
  e.row_stride = N;
  e.V = N;
  return fc_launch_gemm(A, W, M, nullptr, M, N, K, dtype, e, GemmWork{}, (hipStream_t)stream, nullptr);
}

// Fragment-order copy of a row-major bf16 matrix src[rows][K] into
// dst[round16(rows)][K] (padding rows zero); one thread per 16-byte group.
__global__ __launch_bounds__(256) void k_pack_frag(const bf16_t* __restrict__ src, bf16_t* __restrict__ dst,
                                                   int rows, int K) {
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t groups = round16(rows) * (K / 8);
  if (t >= groups) return;
  const int64_t blk = t >> 6;  // 64 groups per 16 x 32 block
  const int lane = (int)(t & 63);
  const int KS = K >> 5;
  const int64_t rb = blk / KS;
  const int ks = (int)(blk - rb * KS);
  const int64_t r = rb * 16 + (lane & 15);
  const int k = ks * 32 + (lane >> 4) * 8;
  uint4 v = {0u, 0u, 0u, 0u};
  if (r < rows) v = *(const uint4*)(src + r * K + k);
  *(uint4*)(dst + t * 8) = v;
}

extern "C" int32_t fc_pack_operand(const void* src, void* dst, int32_t rows, int32_t K, void* stream) {
  FC_CHECK_ARG(src && dst && src != dst, "pointers (distinct, non-null)");
  FC_CHECK_ARG(rows > 0 && K > 0 && K % 32 == 0, "rows > 0 and K % 32 == 0");
  const int64_t groups = round16(rows) * (K / 8);
  hipLaunchKernelGGL(k_pack_frag, dim3((unsigned)((groups + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                     (const bf16_t*)src, (bf16_t*)dst, rows, K);
  FC_LAUNCH_CHECK();
  return FC_OK;
}
