// Per-token attention prologue and split-KV flash-decode attention.
//
// Prologue (flaxchat/engine.py:96-126, flaxchat/gpt.py:65-71): value
// embedding gate on the V heads, RoPE (base 100000) and 1.2 * RMSNorm on
// the Q and K heads, then the K/V append at each valid slot's position.
//
// Attention (flaxchat/engine.py:128-156): for query position p and KV
// group g = h / (H / G), softmax over keys j with j <= p and, for layers
// with a window W > 0, p - j <= W (W + 1 keys, inclusive). The reference
// scores every cached position and masks with -1e9; the masked terms are
// exact zeros in fp32, so reading only the visible keys is the same sum.
//
// bf16 path (head_dim 128): one workgroup per (row, KV group, query block of
// 16 columns, key split). Columns are (token, head-in-group) pairs of the
// row's packed tokens, so a verify chunk's tokens and the GQA heads of a
// group share every K/V tile read. Each wave walks 32-key tiles with two matrix-core products:
//   S^T = K Q^T   (16 keys x 16 columns per MFMA; two MFMAs per tile, with
//                  the key rows interleaved so each lane ends up holding 8
//                  consecutive keys of its column), then online softmax in
//                  registers with wave shuffles,
//   O^T += V^T P^T (P taken straight from registers as the B operand; V^T
//                  read from the 32-key blocked-transposed V cache as one
//                  16-byte load per lane).
// The four waves merge in LDS; splits merge in k_attn_combine.
// Prefill-width chunks (>= 128 query columns per row) take k_attn_pf: 128
// columns per workgroup on the 32x32x16 MFMA, K/V tiles shared through LDS.
// fp32 path (parity mode): k_attn_f32 on the fp32 matrix cores. Other head
// sizes, arrays off the 16-byte boundary: k_attn_valu, one workgroup per query
// with the reference's operation order (scores, max, exp, normalise, weighted
// sum).
#include "fc_common.h"
#include "fc_internal.h"
#include <mutex>
#include <string>

// K/V cache loads are streamed once per call: non-temporal loads keep them
// from displacing reusable lines in the caches (measured ~8% faster at cfg4)
#ifndef FC_ATTN_NT
#define FC_ATTN_NT 1
#endif
#if FC_ATTN_NT
typedef uint32_t kv_u32x4 __attribute__((ext_vector_type(4)));
#define KV_LD(p) __builtin_bit_cast(uint4, __builtin_nontemporal_load((const kv_u32x4*)(p)))
#else
#define KV_LD(p) (*(p))
#endif

// ---------------------------------------------------------------------------
// Prologue: one wave per (packed token m, head slot hh in [0, H + 2G)).
// ---------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(256) void k_prologue(const float* __restrict__ qkv, const T* __restrict__ h,
                                                  const int* __restrict__ tokens, const float* __restrict__ rcos,
                                                  const float* __restrict__ rsin, int rope_len,
                                                  const T* __restrict__ ve, const float* __restrict__ ve_gate,
                                                  int D, T* __restrict__ kc, T* __restrict__ vc, int B, int Mcap,
                                                  const int* __restrict__ Mdev, int H, int G, int hd, int cap,
                                                  const int* __restrict__ tok_row, const int* __restrict__ tok_pos,
                                                  T* __restrict__ q, int kblk) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int NH = H + 2 * G;
  const int64_t item = (int64_t)blockIdx.x * 4 + wave;
  if (item >= (int64_t)Mcap * NH) return;
  const int m = (int)(item / NH), hh = (int)(item % NH);
  const int half = hd >> 1;
  const bool act = lane < half;
  const bool vhead = hh >= H + G;
  // every load that needs neither the token's row nor its position (the
  // device total included: a launch covers the chunk's capacity, and the
  // loads of a token past the total stay inside it) is issued before any of
  // them is waited for; tokens past the total then exit, and the rotary table
  // and the value-embedding row follow as one second batch
  const int mdev = Mdev != nullptr ? *Mdev : Mcap;
  const int b = tok_row[m], pos = tok_pos[m];
  const float* row = qkv + ((int64_t)m * NH + hh) * hd;
  float x1 = act ? row[lane] : 0.f, x2 = act ? row[lane + half] : 0.f;
  int tok = 0;
  float part = 0.f;
  if (vhead && ve != nullptr) {
    tok = tokens[m];
    part = lane < 12 ? ld<T>(h, act_idx<T>(m, lane, D)) * ve_gate[(hh - H - G) * 12 + lane] : 0.f;
  }
  if (m >= mdev) return;
  if ((unsigned)b >= (unsigned)B) return;
  if (!vhead) {
    const int pc = min(max(pos, 0), rope_len - 1);
    const float c = act ? rcos[(int64_t)pc * half + lane] : 0.f;
    const float s = act ? rsin[(int64_t)pc * half + lane] : 0.f;
    float y1 = x1 * c + x2 * s;
    float y2 = x1 * (-s) + x2 * c;
    const float ss = wave_sum(y1 * y1 + y2 * y2);
    const float inv = 1.f / sqrtf(ss / (float)hd + 1e-6f);
    y1 = y1 * inv * 1.2f;
    y2 = y2 * inv * 1.2f;
    if (hh < H) {
      if (act) {
        T* qo = q + ((int64_t)m * H + hh) * hd;
        st<T>(qo, lane, y1);
        st<T>(qo, lane + half, y2);
      }
    } else if (act && pos >= 0 && pos < cap) {
      const int g = hh - H;
      T* kg = kc + ((int64_t)b * G + g) * cap * hd;
      if (kblk) {
        st<T>(kg, kblk_idx(pos, lane), y1);
        st<T>(kg, kblk_idx(pos, lane + half), y2);
      } else {
        st<T>(kg, (int64_t)pos * hd + lane, y1);
        st<T>(kg, (int64_t)pos * hd + lane + half, y2);
      }
    }
  } else {
    const int g = hh - H - G;
    if (ve != nullptr) {
      float v1 = 0.f, v2 = 0.f;
      if (act) {
        const T* vr = ve + ((int64_t)tok * G + g) * hd;
        v1 = ld<T>(vr, lane);
        v2 = ld<T>(vr, lane + half);
      }
      const float z = wave_sum(part);
      const float gate = 3.f * (1.f / (1.f + expf(-z)));
      x1 = x1 + gate * v1;
      x2 = x2 + gate * v2;
    }
    if (act && pos >= 0 && pos < cap) {
      T* vb = vc + ((((int64_t)b * G + g) * (cap / 32) + pos / 32) * hd) * 32;
      st<T>(vb, (int64_t)lane * 32 + (pos & 31), x1);
      st<T>(vb, (int64_t)(lane + half) * 32 + (pos & 31), x2);
    }
  }
}

int fc_launch_prologue(const float* qkv, const void* h, const int* tokens, const fc_model* m, int layer,
                       const fc_cache* c, const int* tok_row, const int* tok_pos, int Mcap, const int* Mdev, void* q,
                       hipStream_t s) {
  const fc_layer& L = m->layers[layer];
  const int H = m->n_head, G = m->n_kv_head, hd = m->head_dim;
  FC_CHECK_ARG(hd <= 128 && hd % 2 == 0, "head_dim must be even and <= 128");
  const int64_t layer_elems = (int64_t)c->batch * G * c->cap * hd;
  const int64_t items = (int64_t)Mcap * (H + 2 * G);
  const dim3 grid((unsigned)((items + 3) / 4));
  if (m->dtype == FC_BF16) {
    bf16_t* kc = (bf16_t*)c->k + layer_elems * layer;
    bf16_t* vc = (bf16_t*)c->v + layer_elems * layer;
    hipLaunchKernelGGL(k_prologue<bf16_t>, grid, dim3(256), 0, s, qkv, (const bf16_t*)h, tokens, m->rope_cos,
                       m->rope_sin, m->rope_len, (const bf16_t*)L.ve, L.ve_gate, m->n_embd, kc, vc, c->batch, Mcap, Mdev, H, G,
                       hd, c->cap, tok_row, tok_pos, (bf16_t*)q, hd == 128 ? 1 : 0);
  } else {
    float* kc = (float*)c->k + layer_elems * layer;
    float* vc = (float*)c->v + layer_elems * layer;
    hipLaunchKernelGGL(k_prologue<float>, grid, dim3(256), 0, s, qkv, (const float*)h, tokens, m->rope_cos,
                       m->rope_sin, m->rope_len, (const float*)L.ve, L.ve_gate, m->n_embd, kc, vc, c->batch, Mcap, Mdev, H, G,
                       hd, c->cap, tok_row, tok_pos, (float*)q, 0);
  }
  FC_LAUNCH_CHECK();
  return FC_OK;
}

extern "C" int32_t fc_attn_prologue(const fc_model* m, int32_t layer, const fc_cache* c, const float* qkv,
                                    const void* h, const int32_t* tokens, const int32_t* tok_row,
                                    const int32_t* tok_pos, int32_t M, void* q, void* stream) {
  FC_CHECK_ARG(m && c && qkv && h && tokens && tok_row && tok_pos && q, "null pointer");
  FC_CHECK_ARG(layer >= 0 && layer < m->n_layer && m->layers != nullptr, "layer out of range");
  FC_CHECK_ARG(m->dtype == FC_F32 || m->dtype == FC_BF16, "dtype");
  FC_CHECK_ARG(m->n_head > 0 && m->n_kv_head > 0 && m->n_head % m->n_kv_head == 0, "head counts");
  FC_CHECK_ARG(c->k && c->v && c->batch > 0 && c->cap > 0 && c->cap % 32 == 0, "cache");
  FC_CHECK_ARG(M >= 0, "M");
  if (M == 0) return FC_OK;
  return fc_launch_prologue(qkv, h, tokens, m, layer, c, tok_row, tok_pos, M, nullptr, q, (hipStream_t)stream);
}

// ---------------------------------------------------------------------------
// bf16 MFMA split-KV attention (head_dim 128)
// ---------------------------------------------------------------------------
__device__ __forceinline__ f32x4 mfma16a(uint4 a, uint4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                  0, 0);
}

// Where the attention kernels put 8 consecutive values (dims d .. +7 of a
// head) of token m: c_proj's operand order, or row-major (`rows`).
__device__ __forceinline__ int64_t y_idx(int64_t m, int k, int K, int rows) {
  return rows ? m * K + k : frag_idx(m, k, K);
}

// One 32-key tile of one wave: scores S^T = K Q^T, online softmax update,
// O^T += V^T P^T (see the kernel comment).
__device__ __forceinline__ void attn_tile(const uint4 (&kf)[2][4], const uint4 (&vf)[8], const uint4 (&qf)[4],
                                          int kb, int g4, bool cvalid, int kbeg, int kend, int lo_c, int pos_c,
                                          float scale_log2, float& m_run, float& l_run, f32x4 (&O)[8]) {
  f32x4 sc[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
  for (int cc = 0; cc < 2; ++cc)
#pragma unroll
    for (int s = 0; s < 4; ++s) sc[cc] = mfma16a(kf[cc][s], qf[s], sc[cc]);
  float p[8];
  float mt = -INFINITY;
#pragma unroll
  for (int cc = 0; cc < 2; ++cc)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int jj = i + 4 * cc;
      const int key = kb + 8 * g4 + jj;
      const bool ok = cvalid && key >= kbeg && key < kend && key >= lo_c && key <= pos_c;
      p[jj] = ok ? sc[cc][i] * scale_log2 : -INFINITY;
      mt = fmaxf(mt, p[jj]);
    }
  mt = fmaxf(mt, __shfl_xor(mt, 16, WAVE));
  mt = fmaxf(mt, __shfl_xor(mt, 32, WAVE));
  const float m_new = fmaxf(m_run, mt);
  float alpha = 1.f, psum = 0.f;
  if (m_new == -INFINITY) {
#pragma unroll
    for (int jj = 0; jj < 8; ++jj) p[jj] = 0.f;
  } else {
    alpha = exp2f(m_run - m_new);
#pragma unroll
    for (int jj = 0; jj < 8; ++jj) {
      p[jj] = exp2f(p[jj] - m_new);
      psum += p[jj];
    }
  }
  l_run = l_run * alpha + psum;
  m_run = m_new;
  uint4 pf;
  pf.x = pack2bf(p[0], p[1]);
  pf.y = pack2bf(p[2], p[3]);
  pf.z = pack2bf(p[4], p[5]);
  pf.w = pack2bf(p[6], p[7]);
#pragma unroll
  for (int db = 0; db < 8; ++db) {
    O[db] *= alpha;
    O[db] = mfma16a(vf[db], pf, O[db]);
  }
}

// grid (key split, row x KV group, query block): the query block is the
// slowest dimension, so blocks with no query (a row's second block is
// usually empty) are dispatched last and exit at once.
template <int NW>
__global__ __launch_bounds__(64 * NW) void k_attn_mfma(const bf16_t* __restrict__ q, const bf16_t* __restrict__ kc,
                                                       const bf16_t* __restrict__ vc, float* __restrict__ part_o,
                                                       float* __restrict__ part_ml, bf16_t* __restrict__ y, int H,
                                                       int G, int cap, const int* __restrict__ row_off,
                                                       const int* __restrict__ start, int max_per_row, int Mcap,
                                                       int window, int split_keys, int nsplit, int nqblk,
                                                       float scale_log2, int rows) {
  constexpr int HD = 128;
  const int split = blockIdx.x, bg = blockIdx.y, qb = blockIdx.z;
  const int b = bg / G, g = bg - b * G, rep = H / G;
  const RowSpan sp = row_span(row_off, b, max_per_row, Mcap);
  const int base = sp.base, n = sp.n, s0 = start[b];
  const int ncol = n * rep;
  if (qb * 16 >= ncol) return;  // no query of this row in the block: combine reads nothing here
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int c = lane & 15, g4 = lane >> 4;
  const int64_t pidx = ((int64_t)bg * nqblk + qb) * nsplit + split;

  // key range of the whole query block
  const int f = qb * 16, lcol = min(qb * 16 + 15, ncol - 1);
  int kbeg = 0, kend = 0;
  {
    const int pf = s0 + f / rep, pl = s0 + lcol / rep;
    const int klo = window > 0 ? max(0, pf - window) : 0;
    const int khi = min(pl + 1, cap);
    kbeg = klo + split * split_keys;
    kend = min(khi, kbeg + split_keys);
  }
  if (kbeg >= kend) {  // only with several splits: a query always sees itself
    if (threadIdx.x < 16) {
      part_ml[(pidx * 16 + threadIdx.x) * 2 + 0] = -INFINITY;
      part_ml[(pidx * 16 + threadIdx.x) * 2 + 1] = 0.f;
    }
    return;
  }
  // this lane's query column
  const int col = qb * 16 + c;
  const int j = col / rep, head = g * rep + (col - j * rep);
  const bool cvalid = col < ncol;
  const int pos_c = s0 + j;
  const int lo_c = window > 0 ? max(0, pos_c - window) : 0;

  const uint4 zero = {0u, 0u, 0u, 0u};
  uint4 qf[4];
  {
    const bf16_t* qr = q + ((int64_t)(base + (cvalid ? j : 0)) * H + head) * HD + 8 * g4;
#pragma unroll
    for (int s = 0; s < 4; ++s) qf[s] = cvalid ? *(const uint4*)(qr + 32 * s) : zero;
  }
  const bf16_t* kbase = kc + (int64_t)bg * cap * HD;
  const bf16_t* vbase = vc + (int64_t)bg * (cap / 32) * HD * 32;
  const int r = c;

  float m_run = -INFINITY, l_run = 0.f;
  f32x4 O[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) O[i] = f32x4{0.f, 0.f, 0.f, 0.f};

  // K blocks of 32 keys in fragment order: load (cc, s) of a tile is 1 KB
  // contiguous; V blocks are [128 dims][32 keys], one 1 KB load per db
  const int t0 = kbeg & ~31;
  const int ntiles = (kend - t0 + 31) >> 5;
#define ATT_LOAD(kf, vf, kb_)                                                                      \
  {                                                                                                \
    const bf16_t* kt = kbase + (int64_t)((kb_) >> 5) * 32 * HD + lane * 8;                         \
    _Pragma("unroll") for (int cc = 0; cc < 2; ++cc)                                               \
      _Pragma("unroll") for (int s = 0; s < 4; ++s) kf[cc][s] = KV_LD((const uint4*)(kt + (s * 2 + cc) * 512)); \
    const bf16_t* vt = vbase + (int64_t)((kb_) >> 5) * HD * 32 + r * 32 + 8 * g4;                  \
    _Pragma("unroll") for (int db = 0; db < 8; ++db) vf[db] = KV_LD((const uint4*)(vt + db * 16 * 32));  \
  }
  for (int t = wave; t < ntiles; t += NW) {
    const int kb = t0 + 32 * t;
    uint4 kf[2][4], vf[8];
    ATT_LOAD(kf, vf, kb);
    attn_tile(kf, vf, qf, kb, g4, cvalid, kbeg, kend, lo_c, pos_c, scale_log2, m_run, l_run, O);
  }
#undef ATT_LOAD
  // merge the NW waves in LDS; thread t < 256 then owns column t / 16 and
  // dims 8 (t % 16) .. +7. A single key split writes y directly (normalised,
  // in the c_proj operand layout); otherwise the unnormalised partial and its
  // (max, sum) go to k_attn_combine.
  float l_tot = l_run + __shfl_xor(l_run, 16, WAVE);
  l_tot = l_tot + __shfl_xor(l_tot, 32, WAVE);
  __shared__ float sm[NW][16], sl[NW][16];
  __shared__ float so[NW][16][HD + 4];
  if (g4 == 0) {
    sm[wave][c] = m_run;
    sl[wave][c] = l_tot;
  }
#pragma unroll
  for (int db = 0; db < 8; ++db)
#pragma unroll
    for (int i = 0; i < 4; ++i) so[wave][c][16 * db + 4 * g4 + i] = O[db][i];
  __syncthreads();
  if (threadIdx.x >= 256) return;
  const int qc = threadIdx.x >> 4, d0 = (threadIdx.x & 15) * 8;
  float M = -INFINITY;
#pragma unroll
  for (int w = 0; w < NW; ++w) M = fmaxf(M, sm[w][qc]);
  float o[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  float L = 0.f;
  if (M != -INFINITY) {
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float a = exp2f(sm[w][qc] - M);
      L += a * sl[w][qc];
#pragma unroll
      for (int i = 0; i < 8; ++i) o[i] += a * so[w][qc][d0 + i];
    }
  }
  if (nsplit == 1) {
    const int colq = qb * 16 + qc;
    if (colq >= ncol) return;
    const int jq = colq / rep, hq = g * rep + (colq - jq * rep);
    const float inv = L > 0.f ? 1.f / L : 0.f;
    uint4 pk;
    pk.x = pack2bf(o[0] * inv, o[1] * inv);
    pk.y = pack2bf(o[2] * inv, o[3] * inv);
    pk.z = pack2bf(o[4] * inv, o[5] * inv);
    pk.w = pack2bf(o[6] * inv, o[7] * inv);
    *(uint4*)(y + y_idx(base + jq, hq * HD + d0, H * HD, rows)) = pk;
    return;
  }
  float4* po = (float4*)(part_o + (pidx * 16 + qc) * HD + d0);
  po[0] = make_float4(o[0], o[1], o[2], o[3]);
  po[1] = make_float4(o[4], o[5], o[6], o[7]);
  if (d0 == 0) {
    part_ml[(pidx * 16 + qc) * 2 + 0] = M;
    part_ml[(pidx * 16 + qc) * 2 + 1] = L;
  }
}

// The same for QB query blocks per workgroup (GQA verify chunks: tokens x
// heads-per-group > 16 columns): each wave applies every K/V tile it loads
// to all QB blocks, so the key range is read once per QB blocks instead of
// once per block; the waves are merged block by block. grid (key split,
// row x KV group, group of QB query blocks).
template <int NW, int QB>
__global__ __launch_bounds__(64 * NW, 2) void k_attn_mfma_qb(const bf16_t* __restrict__ q, const bf16_t* __restrict__ kc,
                                                       const bf16_t* __restrict__ vc, float* __restrict__ part_o,
                                                       float* __restrict__ part_ml, bf16_t* __restrict__ y, int H,
                                                       int G, int cap, const int* __restrict__ row_off,
                                                       const int* __restrict__ start, int max_per_row, int Mcap,
                                                       int window, int split_keys, int nsplit, int nqblk,
                                                       float scale_log2, int rows) {
  constexpr int HD = 128;
  const int split = blockIdx.x, bg = blockIdx.y, qb0 = blockIdx.z * QB;
  const int b = bg / G, g = bg - b * G, rep = H / G;
  const RowSpan sp = row_span(row_off, b, max_per_row, Mcap);
  const int base = sp.base, n = sp.n, s0 = start[b];
  const int ncol = n * rep;
  if (qb0 * 16 >= ncol) return;  // no query of this row in the group: combine reads nothing here
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int c = lane & 15, g4 = lane >> 4;
  const int nblk = min(QB, (ncol - qb0 * 16 + 15) / 16);  // blocks of the group holding a query

  // key range of the whole group of query blocks
  const int f = qb0 * 16, lcol = min(qb0 * 16 + 16 * QB - 1, ncol - 1);
  int kbeg = 0, kend = 0;
  {
    const int pf = s0 + f / rep, pl = s0 + lcol / rep;
    const int klo = window > 0 ? max(0, pf - window) : 0;
    const int khi = min(pl + 1, cap);
    kbeg = klo + split * split_keys;
    kend = min(khi, kbeg + split_keys);
  }
  if (kbeg >= kend) {  // only with several splits: a query always sees itself
    if (threadIdx.x < 16) {
      for (int u = 0; u < nblk; ++u) {
        const int64_t pidx = ((int64_t)bg * nqblk + qb0 + u) * nsplit + split;
        part_ml[(pidx * 16 + threadIdx.x) * 2 + 0] = -INFINITY;
        part_ml[(pidx * 16 + threadIdx.x) * 2 + 1] = 0.f;
      }
    }
    return;
  }
  // this lane's query column in each block
  bool cvalid[QB];
  int pos_c[QB], lo_c[QB];
  uint4 qf[QB][4];
#pragma unroll
  for (int u = 0; u < QB; ++u) {
    const int col = (qb0 + u) * 16 + c;
    const int j = col / rep, head = g * rep + (col - j * rep);
    cvalid[u] = col < ncol;
    pos_c[u] = s0 + j;
    lo_c[u] = window > 0 ? max(0, pos_c[u] - window) : 0;
    const bf16_t* qr = q + ((int64_t)(base + (cvalid[u] ? j : 0)) * H + (cvalid[u] ? head : 0)) * HD + 8 * g4;
    // load from the (always valid, clamped) address, then mask the value: a
    // select between the load and `zero` becomes a select of pointers, one of
    // them to a private copy of `zero`, and the loads turn into flat loads
    const uint32_t keep = cvalid[u] ? 0xffffffffu : 0u;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const uint4 v = *(const uint4*)(qr + 32 * s);
      qf[u][s] = uint4{v.x & keep, v.y & keep, v.z & keep, v.w & keep};
    }
  }
  const bf16_t* kbase = kc + (int64_t)bg * cap * HD;
  const bf16_t* vbase = vc + (int64_t)bg * (cap / 32) * HD * 32;
  const int r = c;

  float m_run[QB], l_run[QB];
  f32x4 O[QB][8];
#pragma unroll
  for (int u = 0; u < QB; ++u) {
    m_run[u] = -INFINITY;
    l_run[u] = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) O[u][i] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

  // K blocks of 32 keys in fragment order: load (cc, s) of a tile is 1 KB
  // contiguous; V blocks are [128 dims][32 keys], one 1 KB load per db
  const int t0 = kbeg & ~31;
  const int ntiles = (kend - t0 + 31) >> 5;
  for (int t = wave; t < ntiles; t += NW) {
    const int kb = t0 + 32 * t;
    uint4 kf[2][4], vf[8];
    const bf16_t* kt = kbase + (int64_t)(kb >> 5) * 32 * HD + lane * 8;
#pragma unroll
    for (int cc = 0; cc < 2; ++cc)
#pragma unroll
      for (int s = 0; s < 4; ++s) kf[cc][s] = KV_LD((const uint4*)(kt + (s * 2 + cc) * 512));
    const bf16_t* vt = vbase + (int64_t)(kb >> 5) * HD * 32 + r * 32 + 8 * g4;
#pragma unroll
    for (int db = 0; db < 8; ++db) vf[db] = KV_LD((const uint4*)(vt + db * 16 * 32));
#pragma unroll
    for (int u = 0; u < QB; ++u)
      if (u < nblk)
        attn_tile(kf, vf, qf[u], kb, g4, cvalid[u], kbeg, kend, lo_c[u], pos_c[u], scale_log2, m_run[u], l_run[u],
                  O[u]);
  }
  // merge the NW waves in LDS, block by block; thread t < 256 then owns
  // column t / 16 and dims 8 (t % 16) .. +7. A single key split writes y
  // directly (normalised, in the c_proj operand layout); otherwise the
  // unnormalised partial and its (max, sum) go to k_attn_combine.
  __shared__ float sm[NW][16], sl[NW][16];
  __shared__ float so[NW][16][HD + 4];
  // (a guard instead of a break keeps the loop unrolled, so m_run / l_run / O
  // stay in registers: a runtime index would put them in scratch memory)
#pragma unroll
  for (int u = 0; u < QB; ++u) {
    if (u < nblk) {  // uniform over the workgroup
      const int qb = qb0 + u;
      const int64_t pidx = ((int64_t)bg * nqblk + qb) * nsplit + split;
      float l_tot = l_run[u] + __shfl_xor(l_run[u], 16, WAVE);
      l_tot = l_tot + __shfl_xor(l_tot, 32, WAVE);
      if (u > 0) __syncthreads();  // the previous block's readers are done with the LDS
      if (g4 == 0) {
        sm[wave][c] = m_run[u];
        sl[wave][c] = l_tot;
      }
  #pragma unroll
      for (int db = 0; db < 8; ++db)
  #pragma unroll
        for (int i = 0; i < 4; ++i) so[wave][c][16 * db + 4 * g4 + i] = O[u][db][i];
      __syncthreads();
      if (threadIdx.x < 256) {
        const int qc = threadIdx.x >> 4, d0 = (threadIdx.x & 15) * 8;
        float M = -INFINITY;
  #pragma unroll
        for (int w = 0; w < NW; ++w) M = fmaxf(M, sm[w][qc]);
        float o[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        float L = 0.f;
        if (M != -INFINITY) {
  #pragma unroll
          for (int w = 0; w < NW; ++w) {
            const float a = exp2f(sm[w][qc] - M);
            L += a * sl[w][qc];
  #pragma unroll
            for (int i = 0; i < 8; ++i) o[i] += a * so[w][qc][d0 + i];
          }
        }
        const int colq = qb * 16 + qc;
        if (nsplit == 1) {
          if (colq < ncol) {
            const int jq = colq / rep, hq = g * rep + (colq - jq * rep);
            const float inv = L > 0.f ? 1.f / L : 0.f;
            uint4 pk;
            pk.x = pack2bf(o[0] * inv, o[1] * inv);
            pk.y = pack2bf(o[2] * inv, o[3] * inv);
            pk.z = pack2bf(o[4] * inv, o[5] * inv);
            pk.w = pack2bf(o[6] * inv, o[7] * inv);
            *(uint4*)(y + y_idx(base + jq, hq * HD + d0, H * HD, rows)) = pk;
          }
        } else {
          float4* po = (float4*)(part_o + (pidx * 16 + qc) * HD + d0);
          po[0] = make_float4(o[0], o[1], o[2], o[3]);
          po[1] = make_float4(o[4], o[5], o[6], o[7]);
          if (d0 == 0) {
            part_ml[(pidx * 16 + qc) * 2 + 0] = M;
            part_ml[(pidx * 16 + qc) * 2 + 1] = L;
          }
        }
      }
    }
  }
}

// Prefill attention on the 32x32x16 MFMA. A workgroup owns 128 query
// columns of one (row, KV group), 32 per wave, and walks the group's key range
// in steps of 64 keys through two LDS stages: the next step's K and V load
// while this one computes, so a key is read once per 128 columns and a step
// has one barrier. Per step a wave computes S^T = K Q^T (two 32-key tiles x
// its 32 columns), one online softmax update in registers, then O^T += V^T P^T
// (4 x 32 dims).
//
// Operand order: the direct loads put every matrix-core operand into LDS in
// lane order (64 lanes x 16 bytes), each lane fetching its own 16 bytes, so
// that every LDS read is 1 KB in a row, free of bank conflicts (in the caches'
// own order the V reads met four to a bank). The rows of the K operand are
// taken in the order that leaves lane l with keys 16 kh + 8 (l / 32) .. +7 of
// its column in registers 8 kh .. +7: the P operand of a 16-key half as it
// stands, with no exchange between lanes.
//
// What bounds it: per 32 keys x 32 columns 512 MFMA cycles against ~540 VALU
// (256 of them the exponentials), overlapped by the two waves of a SIMD; hence
// the output is rescaled only in steps that raise some column's maximum.
// (Rescaling only past a rise of 2^8 took 2% less, but then the largest term
// is no longer exactly 1 and its rounding to bf16 shows: error against 64 bits
// 0.0023 for 0.0020.)
// 8 rows x 500-1000 queries, 12 heads, window 1024: 112 -> 70 us (before: 32 keys
// per barrier, operands in the caches' order, an exchange per P operand).
//
// Workgroups: all column blocks of a (row, group) on one XCD (its K and V in
// one L2), the last blocks, which see the most keys, first.
struct PfStage {
  uint4 k[2][8][64];  // [32-key tile][16-dim slice][lane]
  uint4 v[2][8][64];  // [32-key tile][2 (dim / 32) + key half][lane]
};
// KS = 2: eight waves, the second four taking every other step of the same
// columns with stages of their own, the halves merged in LDS at the end. For
// launches of at most one workgroup per CU, where a wave otherwise has its
// SIMD to itself and walks all keys (4 x 476 queries on 1024-1500 keys, 6
// heads, 96 workgroups: 38 -> 31 us; at 384 workgroups one group is the faster,
// 30 against 39).
template <int KS>
__global__ __launch_bounds__(256 * KS, 2) void k_attn_pf(const bf16_t* __restrict__ q, const bf16_t* __restrict__ kc,
                                                 const bf16_t* __restrict__ vc, bf16_t* __restrict__ y, int H, int G,
                                                 int cap, const int* __restrict__ row_off,
                                                 const int* __restrict__ start, int max_per_row, int Mcap,
                                                 int window, float scale_log2, int nbg, int nblk, int rows) {
  constexpr int HD = 128;
  __shared__ PfStage stg0[KS], stg1[KS];
  const int nbgl = (nbg + 7) >> 3, jj = blockIdx.x >> 3;
  const int bg = (jj % nbgl) * 8 + (blockIdx.x & 7);
  if (bg >= nbg) return;
  const int b = bg / G, g = bg - b * G, rep = H / G;
  const RowSpan sp = row_span(row_off, b, max_per_row, Mcap);
  const int base = sp.base, n = sp.n, s0 = start[b];
  const int ncol = n * rep;
  const int c0 = (nblk - 1 - jj / nbgl) * 128;
  if (c0 >= ncol) return;  // the whole workgroup
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wave = wid & 3, grp = KS > 1 ? wid >> 2 : 0;
  const int hl = lane >> 5, kk = lane & 31;
  // the workgroup's key range
  const int lcol = min(c0 + 127, ncol - 1);
  const int kbeg = window > 0 ? max(0, s0 + c0 / rep - window) : 0;
  const int kend = min(s0 + lcol / rep + 1, cap);
  const int t0 = kbeg & ~31;
  const int ntiles = (kend - t0 + 31) >> 5, nstep = (ntiles + 1) >> 1;  // group grp takes steps grp, grp + KS, ..
  // this wave's columns and key range; positions past the cache end with the
  // range (kend), behind which a step holds the last tile once more
  const int wc0 = c0 + 32 * wave;
  const bool wact = wc0 < ncol;
  const int w_hi = wact ? min(s0 + min(wc0 + 31, ncol - 1) / rep, kend - 1) : -1;
  const int w_lo = window > 0 ? max(0, s0 + wc0 / rep - window) : 0;
  // keys inside [w_full_lo, w_full_hi] are visible to every column of the wave (no masks)
  const bool wfull = wc0 + 31 < ncol;
  const int w_full_hi = min(s0 + wc0 / rep, kend - 1);  // the first column's position
  const int w_full_lo = window > 0 ? max(0, s0 + (wc0 + 31) / rep - window) : 0;
  // this lane's column (query)
  const int col = wc0 + kk;
  const bool cvalid = col < ncol;
  const int j = cvalid ? col / rep : 0;
  const int head = g * rep + (cvalid ? col - (col / rep) * rep : 0);
  const int hi_c = min(s0 + j, kend - 1), lo_c = window > 0 ? max(0, s0 + j - window) : 0;
  v4u qf[8];  // dims 16 h + 8 hl .. +7 of this lane's query
  {
    const bf16_t* qr = q + ((int64_t)(base + j) * H + head) * HD + 8 * hl;
#pragma unroll
    for (int h = 0; h < 8; ++h) qf[h] = cvalid ? *(const v4u*)(qr + 16 * h) : v4u{0u, 0u, 0u, 0u};
  }
  // byte offsets of this lane's 16 bytes: K operand row kk is key
  // 16 (kk / 16) + 8 ((kk / 4) % 2) + 4 ((kk / 8) % 2) + kk % 4 of the tile (its
  // place in a K block: see kblk_idx), V operand row kk is dim kk of 32
  const int key = ((kk >> 4) << 4) | (((kk >> 2) & 1) << 3) | (((kk >> 3) & 1) << 2) | (kk & 3);
  const uint32_t koff = 16u * (uint32_t)((((key >> 2) & 1) << 6) + ((key >> 3) << 2) + (key & 3) + 16 * hl);
  const uint32_t voff = 16u * (uint32_t)(4 * kk + hl);
  const bf16_t* kbase = kc + (int64_t)bg * cap * HD;
  const bf16_t* vbase = vc + (int64_t)bg * (cap / 32) * HD * 32;
  f32x16 O[4];
#pragma unroll
  for (int dd = 0; dd < 4; ++dd)
#pragma unroll
    for (int x = 0; x < 16; ++x) O[dd][x] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;
  // the wave's eight loads of a step: 16-dim slices 2 wave, 2 wave + 1 of K and
  // dims 32 wave .. +31 of V, of both tiles
#define PF_ISSUE(S, i_)                                                                                    \
  {                                                                                                        \
    _Pragma("unroll") for (int u = 0; u < 2; ++u) {                                                        \
      const int64_t blk = (int64_t)((t0 >> 5) + min(2 * (i_) + u, ntiles - 1)) * 32 * HD; /* past the end: harmless re-reads */ \
      const bf16_t* kt = kbase + blk + 1024 * wave;                                                        \
      const bf16_t* vt = vbase + blk + 1024 * wave;                                                        \
      const uint32_t lk = LDS_ADDR(S.k[u][0]) + 2048 * wave, lv = LDS_ADDR(S.v[u][0]) + 2048 * wave;       \
      lds_load_1k(kt, koff, lk);                                                                           \
      lds_load_1k(kt + 256, koff, lk + 1024);                                                              \
      lds_load_1k(vt, voff, lv);                                                                           \
      lds_load_1k(vt + 16, voff, lv + 1024);                                                               \
    }                                                                                                      \
  }
#define PF_SYNC()                                                                                          \
  {                                                                                                        \
    __builtin_amdgcn_sched_barrier(0);                                                                     \
    __builtin_amdgcn_s_waitcnt(0); /* this step's loads, issued a step ago, and this wave's LDS reads */   \
    __atomic_signal_fence(__ATOMIC_SEQ_CST);                                                               \
    __builtin_amdgcn_sched_barrier(0);                                                                     \
    __builtin_amdgcn_s_barrier();                                                                          \
    __builtin_amdgcn_sched_barrier(0);                                                                     \
    __atomic_signal_fence(__ATOMIC_SEQ_CST);                                                               \
  }
  auto step = [&](const PfStage& S, int i) {
    const int kb = t0 + 64 * i;
    if (!(wact && kb <= w_hi && kb + 63 >= w_lo)) return;
    f32x16 sc[2];
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int x = 0; x < 16; ++x) sc[u][x] = 0.f;
    // all K operands are read ahead of the first product, V's behind the last
    // one and ahead of the softmax (read one or two ahead of their use, as the
    // compiler places them, each product waits out an LDS latency)
    v4u kf[8][2], vf[2][8];
#pragma unroll
    for (int h = 0; h < 8; ++h)
#pragma unroll
      for (int u = 0; u < 2; ++u) kf[h][u] = __builtin_bit_cast(v4u, S.k[u][h][lane]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int h = 0; h < 8; ++h)
#pragma unroll
      for (int u = 0; u < 2; ++u) sc[u] = mfma32(kf[h][u], qf[h], sc[u]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int f = 0; f < 8; ++f) vf[u][f] = __builtin_bit_cast(v4u, S.v[u][f][lane]);
    __builtin_amdgcn_sched_barrier(0);
    if (!(wfull && kb >= w_full_lo && kb + 63 <= w_full_hi)) {
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int x = 0; x < 16; ++x) {
          const int kx = kb + 32 * u + 16 * (x >> 3) + 8 * hl + (x & 7);
          if (!(cvalid && kx >= lo_c && kx <= hi_c)) sc[u][x] = -INFINITY;
        }
      // a tile that no column of the wave sees: P is 0 there, and so has V to be, whose slots hold anything
#pragma unroll
      for (int u = 0; u < 2; ++u)
        if (kb + 32 * u > w_hi || kb + 32 * u + 31 < w_lo) {
#pragma unroll
          for (int f = 0; f < 8; ++f) vf[u][f] = v4u{0u, 0u, 0u, 0u};
        }
    }
    float m4[4];  // four chains each: one or two waves per SIMD leave latencies in sight
#pragma unroll
    for (int x = 0; x < 4; ++x) m4[x] = fmaxf(sc[0][x], sc[1][x]);
#pragma unroll
    for (int x = 4; x < 16; ++x) m4[x & 3] = fmaxf(m4[x & 3], fmaxf(sc[0][x], sc[1][x]));
    float mt = fmaxf(fmaxf(m4[0], m4[1]), fmaxf(m4[2], m4[3]));
    {
      const auto h2 = __builtin_amdgcn_permlane32_swap(__float_as_uint(mt), __float_as_uint(mt), false, false);
      mt = fmaxf(__uint_as_float(h2[0]), __uint_as_float(h2[1]));  // lanes l and l ^ 32: the column's two key halves
    }
    const float m_new = fmaxf(m_run, mt * scale_log2);
    if (__any(m_new > m_run)) {
      const float alpha = __builtin_amdgcn_exp2f(m_run - (m_new == -INFINITY ? 0.f : m_new));
      l_run *= alpha;
#pragma unroll
      for (int dd = 0; dd < 4; ++dd) O[dd] *= alpha;
      m_run = m_new;
    }
    const float m_use = m_run == -INFINITY ? 0.f : m_run;  // no key yet: every term exp2(-inf) = 0
    float ps[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int kh = 0; kh < 2; ++kh) {
        float pv[8];
#pragma unroll
        for (int x = 0; x < 8; ++x) {
          pv[x] = __builtin_amdgcn_exp2f(fmaf(sc[u][8 * kh + x], scale_log2, -m_use));
          ps[x & 3] += pv[x];
        }
        const v4u pb = v4u{pack2bf(pv[0], pv[1]), pack2bf(pv[2], pv[3]), pack2bf(pv[4], pv[5]), pack2bf(pv[6], pv[7])};
#pragma unroll
        for (int dd = 0; dd < 4; ++dd)
          O[dd] = mfma32(vf[u][2 * dd + kh], pb, O[dd]);
      }
    l_run += (ps[0] + ps[1]) + (ps[2] + ps[3]);
  };
  if (ntiles > 0) PF_ISSUE(stg0[grp], grp);  // (a row past the cache's end has no key to read)
  for (int i = 0; i < nstep; i += 2 * KS) {
    PF_SYNC();
    PF_ISSUE(stg1[grp], i + KS + grp);
    step(stg0[grp], i + grp);
    if (i + KS < nstep) {
      PF_SYNC();
      PF_ISSUE(stg0[grp], i + 2 * KS + grp);
      step(stg1[grp], i + KS + grp);
    }
  }
#undef PF_SYNC
#undef PF_ISSUE
  __builtin_amdgcn_s_waitcnt(0);  // no direct load outlives its stage
  __syncthreads();                // the stages become scratch
  if constexpr (KS == 2) {
    // the second group's O, maximum and sum, lane for lane
    float(*xo)[64][64] = (float(*)[64][64])&stg0[0];  // [wave][value][lane], 64 KB
    float(*xm)[2][64] = (float(*)[2][64])&stg1[0];
    static_assert(sizeof(stg0) >= 4 * 64 * 64 * 4, "the second group's output");
    if (grp == 1) {
#pragma unroll
      for (int dd = 0; dd < 4; ++dd)
#pragma unroll
        for (int x = 0; x < 16; ++x) xo[wave][16 * dd + x][lane] = O[dd][x];
      xm[wave][0][lane] = m_run;
      xm[wave][1][lane] = l_run;
    }
    __syncthreads();
    if (grp == 0) {
      const float m1 = xm[wave][0][lane], m = fmaxf(m_run, m1), mu = m == -INFINITY ? 0.f : m;
      const float a0 = __builtin_amdgcn_exp2f(m_run - mu), a1 = __builtin_amdgcn_exp2f(m1 - mu);
      l_run = l_run * a0 + xm[wave][1][lane] * a1;
#pragma unroll
      for (int dd = 0; dd < 4; ++dd)
#pragma unroll
        for (int x = 0; x < 16; ++x) O[dd][x] = O[dd][x] * a0 + xo[wave][16 * dd + x][lane] * a1;
    }
    __syncthreads();
    if (grp == 1) return;
  }
  const float l_tot = l_run + __shfl_xor(l_run, 32, WAVE);
  const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
  // lane: column l % 32; register 4 i4 + x of O[dd] is dim 32 dd + 8 i4 + 4 hl + x.
  // Through LDS (rows of 136 values) so that a lane writes 8 dims of a column:
  // 16 columns x 4 groups per store in operand order (1 KB in a row where the
  // columns are 16 tokens), 4 columns of 256 bytes in row-major order.
  bf16_t* T = (bf16_t*)(wave < 2 ? &stg0[0] : &stg1[0]) + (wave & 1) * 32 * 136;
  static_assert(sizeof(PfStage) >= 2 * 32 * 136 * 2, "two waves' scratch");
#pragma unroll
  for (int dd = 0; dd < 4; ++dd)
#pragma unroll
    for (int i4 = 0; i4 < 4; ++i4) {
      uint2 pk;
      pk.x = pack2bf(O[dd][4 * i4] * inv, O[dd][4 * i4 + 1] * inv);
      pk.y = pack2bf(O[dd][4 * i4 + 2] * inv, O[dd][4 * i4 + 3] * inv);
      *(uint2*)(T + kk * 136 + 32 * dd + 8 * i4 + 4 * hl) = pk;
    }
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int it = 0; it < 8; ++it) {
    const int cc = rows ? 4 * it + (lane >> 4) : (lane & 15) + 16 * (it & 1);
    const int d0 = 8 * (rows ? lane & 15 : (lane >> 4) + 4 * (it >> 1));
    const uint4 val = *(const uint4*)(T + cc * 136 + d0);
    const int co = wc0 + cc, jo = co / rep;
    if (co < ncol) *(uint4*)(y + y_idx(base + jo, (g * rep + co - jo * rep) * HD + d0, H * HD, rows)) = val;
  }
}

// One workgroup per (row, KV group, query block): merge the key splits of
// its 16 columns and normalise; thread t owns column t / 16 and 8
// consecutive dimensions. Bound by load latency alone (a few KB), so the loads
// of CB splits are in flight together, the first CB ahead of the row's span and
// the maximum, whose terms the column's 16 threads load side by side; split by
// split, every one waited for the one before (one row, 6 heads, 6 splits: a step of
// 12 layers 499 -> 486 us; 7 queries, 4 groups, 48 splits: the whole call 38 -> 21).
// CB follows the number of splits (2, 4 or 8): 8 for the 2 splits of 192 row x
// group pairs reads each of them four times, 4.75 us a launch instead of 3.7.
template <typename T, int CB>
__global__ __launch_bounds__(256) void k_attn_combine(const float* __restrict__ part_o,
                                                      const float* __restrict__ part_ml, T* __restrict__ y, int H,
                                                      int G, int nqblk, int nsplit, const int* __restrict__ row_off,
                                                      int max_per_row, int Mcap, int rows) {
  constexpr int HD = 128;
  const int bg = blockIdx.x, qb = blockIdx.y;
  const int c = threadIdx.x >> 4, d0 = (threadIdx.x & 15) * 8;
  const int64_t pb = ((int64_t)bg * nqblk + qb) * nsplit;
  const float2* ml = (const float2*)part_ml + pb * 16 + c;            // split s: ml[16 s]
  const float* po = part_o + (pb * 16 + c) * HD + d0;                 // split s: po + 16 HD s
  float2 e[CB];
  float4 u[CB][2];
  auto load = [&](int s0) {
#pragma unroll
    for (int k = 0; k < CB; ++k) {
      const int s = min(s0 + k, nsplit - 1);
      e[k] = ml[(int64_t)s * 16];
      u[k][0] = *(const float4*)(po + (int64_t)s * (16 * HD));
      u[k][1] = *(const float4*)(po + (int64_t)s * (16 * HD) + 4);
    }
  };
  load(0);
  float M = -INFINITY;
  for (int s = threadIdx.x & 15; s < nsplit; s += 16) M = fmaxf(M, ml[(int64_t)s * 16].x);
#pragma unroll
  for (int m = 8; m > 0; m >>= 1) M = fmaxf(M, __shfl_xor(M, m, WAVE));  // the 16 threads of a column
  const int b = bg / G, g = bg - b * G, rep = H / G;
  const RowSpan sp = row_span(row_off, b, max_per_row, Mcap);
  const int base = sp.base, ncol = sp.n * rep;
  const int col = qb * 16 + c;
  if (col >= ncol) return;
  const int j = col / rep, head = g * rep + (col - j * rep);
  float o[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  float L = 0.f;
  for (int s0 = 0; s0 < nsplit && M != -INFINITY; s0 += CB) {
    if (s0 > 0) load(s0);
#pragma unroll
    for (int k = 0; k < CB; ++k) {
      // a split without visible keys holds (-inf, 0) and no output
      if (s0 + k >= nsplit || e[k].x == -INFINITY) continue;
      const float a = exp2f(e[k].x - M);
      L += a * e[k].y;
      o[0] += a * u[k][0].x; o[1] += a * u[k][0].y; o[2] += a * u[k][0].z; o[3] += a * u[k][0].w;
      o[4] += a * u[k][1].x; o[5] += a * u[k][1].y; o[6] += a * u[k][1].z; o[7] += a * u[k][1].w;
    }
  }
  const float inv = L > 0.f ? 1.f / L : 0.f;
  // y is the c_proj GEMM's operand [token][H * 128]: 8 consecutive k are one
  // contiguous 16-byte group in both layouts
  T* yo = y + (sizeof(T) == 2 ? y_idx(base + j, head * HD + d0, H * HD, rows)
                              : (int64_t)(base + j) * H * HD + head * HD + d0);
  if constexpr (sizeof(T) == 2) {
    uint4 pk;
    pk.x = pack2bf(o[0] * inv, o[1] * inv);
    pk.y = pack2bf(o[2] * inv, o[3] * inv);
    pk.z = pack2bf(o[4] * inv, o[5] * inv);
    pk.w = pack2bf(o[6] * inv, o[7] * inv);
    *(uint4*)yo = pk;
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) st<T>(yo, i, o[i] * inv);
  }
}

// ---------------------------------------------------------------------------
// fp32 attention on the fp32 matrix cores (head_dim 128, the parity mode): a
// workgroup owns 32 query columns (token, head in group) of one (row, KV
// group); its eight waves take every eighth 32-key tile, each with its own
// online softmax, and are merged in LDS. Per tile and wave S^T = K Q^T and
// O^T += V^T P^T are 64 32x32x2 MFMAs each; lane l holds column l % 32 and its
// operands come 16 bytes at a time, 4 k of half l / 32 (the order of dims and
// of keys is free), which makes the scores' registers the P operand as they
// stand. k_attn_valu gives one query to a workgroup, whose threads each walk
// whole key rows: 2 x 500 queries, 2 heads, window 256: 132 -> 27 us; one query
// of 1000 keys 76 -> 50, of 10 18.6 -> 18.4. Bound by the latency of one wave's
// tiles (its loads wait for each other: 256 VGPRs hold no second tile).
// ---------------------------------------------------------------------------
__device__ __forceinline__ f32x16 mfma32fa(float a, float b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}
#define AF_WAVES 8
__global__ __launch_bounds__(64 * AF_WAVES, 2) void k_attn_f32(const float* __restrict__ q,
                                                               const float* __restrict__ kc,
                                                               const float* __restrict__ vc, float* __restrict__ y,
                                                               int H, int G, int cap, const int* __restrict__ row_off,
                                                               const int* __restrict__ start, int max_per_row,
                                                               int Mcap, int window, float scale) {
  constexpr int HD = 128;
  const int bg = blockIdx.y, b = bg / G, g = bg - b * G, rep = H / G;
  const RowSpan sp = row_span(row_off, b, max_per_row, Mcap);
  const int base = sp.base, n = sp.n, s0 = start[b];
  const int ncol = n * rep, c0 = blockIdx.x * 32;
  if (c0 >= ncol) return;  // the whole workgroup
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, hl = lane >> 5;
  const int col = c0 + (lane & 31);
  const bool cvalid = col < ncol;
  const int j = cvalid ? col / rep : 0, head = g * rep + (cvalid ? col - j * rep : 0);
  // a position past the cache sees what its last position sees
  const int pos_c = min(s0 + j, cap - 1), lo_c = window > 0 ? max(0, pos_c - window) : 0;
  const int p_hi = min(s0 + min(c0 + 31, ncol - 1) / rep, cap - 1);
  const int p_lo = min(s0 + c0 / rep, cap - 1);
  const int t0 = (window > 0 ? max(0, p_lo - window) : 0) & ~31;
  const int ntiles = (p_hi - t0 + 32) >> 5;
  float4 qf[16];  // dims 8 j + 4 hl .. +3 of this lane's query
  {
    const float* qr = q + ((int64_t)(base + j) * H + head) * HD + 4 * hl;
#pragma unroll
    for (int d = 0; d < 16; ++d) qf[d] = *(const float4*)(qr + 8 * d);
  }
  const float* kb = kc + (int64_t)bg * cap * HD;
  const float* vb = vc + (int64_t)bg * cap * HD;
  __shared__ float xo[AF_WAVES / 2][64][64], xm[AF_WAVES / 2][2][64];
  float m_run = -INFINITY, l_run = 0.f;
  f32x16 O[4];  // dims 32 dd + 8 (x / 4) + 4 hl + x % 4 of this lane's column
#pragma unroll
  for (int dd = 0; dd < 4; ++dd)
#pragma unroll
    for (int x = 0; x < 16; ++x) O[dd][x] = 0.f;
  for (int t = wave; t < ntiles; t += AF_WAVES) {
    const int k0 = t0 + 32 * t;  // a multiple of 32 below cap
    float4 kf[16];
    const float* kr = kb + (int64_t)(k0 + (lane & 31)) * HD + 4 * hl;
#pragma unroll
    for (int d = 0; d < 16; ++d) kf[d] = *(const float4*)(kr + 8 * d);
    f32x16 s2[2];
#pragma unroll
    for (int x = 0; x < 16; ++x) s2[0][x] = s2[1][x] = 0.f;
#pragma unroll
    for (int d = 0; d < 16; ++d) {
      s2[d & 1] = mfma32fa(kf[d].x, qf[d].x, s2[d & 1]);
      s2[d & 1] = mfma32fa(kf[d].y, qf[d].y, s2[d & 1]);
      s2[d & 1] = mfma32fa(kf[d].z, qf[d].z, s2[d & 1]);
      s2[d & 1] = mfma32fa(kf[d].w, qf[d].w, s2[d & 1]);
    }
    float p[16], mt = -INFINITY;
#pragma unroll
    for (int x = 0; x < 16; ++x) {
      const int key = k0 + 8 * (x >> 2) + 4 * hl + (x & 3);
      const bool ok = cvalid && key >= lo_c && key <= pos_c;
      p[x] = ok ? (s2[0][x] + s2[1][x]) * scale : -INFINITY;
      mt = fmaxf(mt, p[x]);
    }
    mt = fmaxf(mt, __shfl_xor(mt, 32, WAVE));
    const float m_new = fmaxf(m_run, mt), m_use = m_new == -INFINITY ? 0.f : m_new;
    if (__any(m_new > m_run)) {
      const float alpha = expf(m_run - m_use);
      l_run *= alpha;
#pragma unroll
      for (int dd = 0; dd < 4; ++dd) O[dd] *= alpha;
      m_run = m_new;
    }
#pragma unroll
    for (int x = 0; x < 16; ++x) {
      p[x] = expf(p[x] - m_use);
      l_run += p[x];
    }
    // V blocks of 32 keys are [128 dims][32]: keys 8 jj + 4 hl .. +3 of dim 32 dd + l % 32
    const float* vt = vb + (int64_t)k0 * HD;
    // a key that some column does not see counts as 0 there even where its V
    // is not finite (slots past the row's end hold anything): key by key then
    bool odd = false;
    if (k0 + 31 > p_lo || (window > 0 && k0 < p_hi - window)) {
#pragma unroll 4
      for (int i = 0; i < 16; ++i) {
        const float4 f = *(const float4*)(vt + 256 * i + 4 * lane);
        const float z = (f.x * 0.f + f.y * 0.f) + (f.z * 0.f + f.w * 0.f);  // NaN unless all are finite
        odd |= z != z;
      }
    }
    if (__any(odd)) {
      float(*pw)[32] = (float(*)[32])((float*)xo + wave * 1024);  // this wave's P, [key][column]
#pragma unroll
      for (int x = 0; x < 16; ++x) pw[8 * (x >> 2) + 4 * hl + (x & 3)][lane & 31] = p[x];
      __builtin_amdgcn_wave_barrier();
      for (int kk = 0; kk < 32; ++kk) {
        const bool sees = k0 + kk >= lo_c && k0 + kk <= pos_c;
        const float pk = pw[kk][lane & 31];
#pragma unroll
        for (int dd = 0; dd < 4; ++dd)
#pragma unroll
          for (int x = 0; x < 16; ++x) {
            const float v = vt[(32 * dd + 8 * (x >> 2) + 4 * hl + (x & 3)) * 32 + kk];
            O[dd][x] = sees ? fmaf(pk, v, O[dd][x]) : O[dd][x];
          }
      }
      __builtin_amdgcn_wave_barrier();
      continue;
    }
#pragma unroll
    for (int dd = 0; dd < 4; ++dd) {
      float4 vf[4];
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) vf[jj] = *(const float4*)(vt + dd * 1024 + (lane & 31) * 32 + 8 * jj + 4 * hl);
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) {
        O[dd] = mfma32fa(vf[jj].x, p[4 * jj], O[dd]);
        O[dd] = mfma32fa(vf[jj].y, p[4 * jj + 1], O[dd]);
        O[dd] = mfma32fa(vf[jj].z, p[4 * jj + 2], O[dd]);
        O[dd] = mfma32fa(vf[jj].w, p[4 * jj + 3], O[dd]);
      }
    }
  }
  // merge the waves, half of the rest giving its O, maximum and sum to the other half each time
  l_run += __shfl_xor(l_run, 32, WAVE);
#pragma unroll
  for (int half = AF_WAVES / 2; half >= 1; half >>= 1) {
    __syncthreads();
    if (wave >= half && wave < 2 * half) {
#pragma unroll
      for (int dd = 0; dd < 4; ++dd)
#pragma unroll
        for (int x = 0; x < 16; ++x) xo[wave - half][16 * dd + x][lane] = O[dd][x];
      xm[wave - half][0][lane] = m_run;
      xm[wave - half][1][lane] = l_run;
    }
    __syncthreads();
    if (wave < half) {
      const float m1 = xm[wave][0][lane], m = fmaxf(m_run, m1), mu = m == -INFINITY ? 0.f : m;
      const float a0 = expf(m_run - mu), a1 = expf(m1 - mu);
      l_run = l_run * a0 + xm[wave][1][lane] * a1;
#pragma unroll
      for (int dd = 0; dd < 4; ++dd)
#pragma unroll
        for (int x = 0; x < 16; ++x) O[dd][x] = O[dd][x] * a0 + xo[wave][16 * dd + x][lane] * a1;
      m_run = m;
    }
  }
  if (wave != 0 || !cvalid) return;
  float* yr = y + (int64_t)(base + j) * H * HD + head * HD + 4 * hl;
  const bool none = pos_c < 0;  // a query before position 0 sees no key: 0, not 0 / 0
#pragma unroll
  for (int dd = 0; dd < 4; ++dd)
#pragma unroll
    for (int u = 0; u < 4; ++u)
      *(float4*)(yr + 32 * dd + 8 * u) =
          none ? make_float4(0.f, 0.f, 0.f, 0.f)
               : make_float4(O[dd][4 * u] / l_run, O[dd][4 * u + 1] / l_run, O[dd][4 * u + 2] / l_run,
                             O[dd][4 * u + 3] / l_run);
}

// ---------------------------------------------------------------------------
// VALU attention, reference operation order (any hd <= 128)
// ---------------------------------------------------------------------------
#define VALU_MAXK 8192
template <typename T>
__global__ __launch_bounds__(256) void k_attn_valu(const T* __restrict__ q, const T* __restrict__ kc,
                                                   const T* __restrict__ vc, T* __restrict__ y, int H, int G, int hd,
                                                   int cap, const int* __restrict__ row_off,
                                                   const int* __restrict__ start, int max_per_row, int Mcap,
                                                   int window, float scale, int rows) {
  __shared__ float qs[128];
  __shared__ float sc[VALU_MAXK];
  __shared__ float red[16];
  const int j = blockIdx.x, h = blockIdx.y, b = blockIdx.z;
  const RowSpan sp = row_span(row_off, b, max_per_row, Mcap);
  const int base = sp.base;
  if (j >= sp.n) return;
  const int m = base + j;
  const int rep = H / G, g = h / rep;
  const int pos = min(start[b] + j, cap - 1);
  const int lo = window > 0 ? max(0, pos - window) : 0;
  const int nk = min(pos - lo + 1, VALU_MAXK);
  const int64_t bg = (int64_t)b * G + g;
  for (int d = threadIdx.x; d < hd; d += blockDim.x) qs[d] = ld<T>(q, ((int64_t)m * H + h) * hd + d);
  __syncthreads();
  for (int i = threadIdx.x; i < nk; i += blockDim.x) {
    const T* kr = kc + (bg * cap + lo + i) * hd;
    float s = 0.f;
    for (int d = 0; d < hd; ++d) s += qs[d] * ld<T>(kr, d);
    sc[i] = s * scale;
  }
  __syncthreads();
  float mx = -INFINITY;
  for (int i = threadIdx.x; i < nk; i += blockDim.x) mx = fmaxf(mx, sc[i]);
  mx = block_max(mx, red);
  float sum = 0.f;
  for (int i = threadIdx.x; i < nk; i += blockDim.x) {
    const float e = expf(sc[i] - mx);
    sc[i] = e;
    sum += e;
  }
  sum = block_sum(sum, red);
  for (int i = threadIdx.x; i < nk; i += blockDim.x) sc[i] = sc[i] / sum;
  __syncthreads();
  const T* vb = vc + bg * (cap / 32) * hd * 32;
  for (int d = threadIdx.x; d < hd; d += blockDim.x) {
    float acc = 0.f;
    for (int i = 0; i < nk; ++i) {
      const int key = lo + i;
      acc += sc[i] * ld<T>(vb, ((int64_t)(key >> 5) * hd + d) * 32 + (key & 31));
    }
    st<T>(y, sizeof(T) == 2 ? y_idx(m, h * hd + d, H * hd, rows) : (int64_t)m * H * hd + h * hd + d, acc);
  }
}

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------
// Workgroups a typical attention launch is split into (key splits x rows x
// KV groups x query blocks).
#ifndef FC_ATTN_TARGET_WG
#define FC_ATTN_TARGET_WG 256
#endif
// query columns per row from which a chunk takes the prefill kernel
#ifndef FC_ATTN_CHUNK_COLS
#define FC_ATTN_CHUNK_COLS 128
#endif
// waves per attention workgroup (they take the block's 32-key tiles round robin)
#ifndef FC_ATTN_WAVES
#define FC_ATTN_WAVES 4
#endif

AttnGrid fc_attn_grid(int batch, int max_per_row, int typ_per_row, int n_head, int n_kv_head, int max_keys) {
  AttnGrid a;
  const int rep = n_head / n_kv_head;
  a.nqblk = (max_per_row * rep + 15) / 16;
  // split the key range so that the blocks a typical chunk fills reach ~4
  // workgroups per CU
  const int typ_blk = std::min(a.nqblk, std::max(1, (typ_per_row * rep + 15) / 16));
  // two query blocks per workgroup when a typical row x group fills more than one
  a.qb = typ_blk >= 2 ? 2 : 1;
  const int64_t units = (int64_t)batch * n_kv_head * ((typ_blk + a.qb - 1) / a.qb);
  const int range = max(max_keys, 1);
  int want = (int)((FC_ATTN_TARGET_WG + units - 1) / units);
  want = max(1, min(want, (range + 127) / 128));
  int sk = (range + want - 1) / want;
  sk = max(128, (sk + 127) / 128 * 128);
  a.split_keys = sk;
  a.nsplit = (range + sk - 1) / sk;
  return a;
}

int64_t fc_attn_part_bytes(int batch, int max_per_row, int n_head, int n_kv_head, int head_dim, int max_keys) {
  if (head_dim != 128) return 0;
  // fc_attn_grid never makes more splits than ceil(FC_ATTN_TARGET_WG /
  // units), and one token per row gives the fewest units
  AttnGrid a = fc_attn_grid(batch, max_per_row, 1, n_head, n_kv_head, max_keys);
  const int64_t units1 = (int64_t)batch * n_kv_head;
  const int64_t nsplit = std::max<int64_t>(a.nsplit, (FC_ATTN_TARGET_WG + units1 - 1) / units1);
  const int64_t units = (int64_t)batch * n_kv_head * a.nqblk * nsplit * 16;
  return fc_align(units * 128 * 4) + fc_align(units * 2 * 4);
}

// Prefill-width chunks (bf16, head_dim 128, >= FC_ATTN_CHUNK_COLS query
// columns per row and KV group) take k_attn_pf, which writes no partials.
static bool attn_uses_pf(int dtype, int hd, int typ_per_row, int H, int G) {
  return dtype == FC_BF16 && hd == 128 && G > 0 && typ_per_row * (H / G) >= FC_ATTN_CHUNK_COLS;
}

int fc_launch_attention(const void* q, const void* kc, const void* vc, void* y, int B, int max_tokens,
                        int max_per_row, int typ_per_row, int H, int G, int hd, int cap, const int* row_off,
                        const int* start, int window, int max_keys, int dtype, void* part, int64_t part_bytes,
                        hipStream_t s, int rows) {
  FC_CHECK_ARG(H % G == 0, "n_head must be a multiple of n_kv_head");
  FC_CHECK_ARG(cap % 32 == 0, "cache capacity must be a multiple of 32");
  FC_CHECK_ARG(max_per_row > 0, "max_per_row");
  const float scale = 1.f / sqrtf((float)hd);
  if (attn_uses_pf(dtype, hd, typ_per_row, H, G)) {
    FC_CHECK_ARG(B * G <= 65535, "batch * n_kv_head must be <= 65535");
    const int ncolmax = max_per_row * (H / G);
    // prefill-width chunks: 128 query columns per workgroup, 32x32x16 MFMA
    const int nblk = (ncolmax + 127) / 128;
    const dim3 grid((unsigned)(8 * ((B * G + 7) / 8) * nblk));
    const float sl2 = scale * 1.4426950408889634f;
    // two key halves per workgroup up to about one workgroup per CU (272
    // workgroups: 50 -> 40 us, 384: 30 -> 39)
    if ((int64_t)B * G * nblk <= 288 && max_keys >= 256)
      hipLaunchKernelGGL(k_attn_pf<2>, grid, dim3(512), 0, s, (const bf16_t*)q, (const bf16_t*)kc, (const bf16_t*)vc,
                         (bf16_t*)y, H, G, cap, row_off, start, max_per_row, max_tokens, window, sl2, B * G, nblk, rows);
    else
      hipLaunchKernelGGL(k_attn_pf<1>, grid, dim3(256), 0, s, (const bf16_t*)q, (const bf16_t*)kc, (const bf16_t*)vc,
                         (bf16_t*)y, H, G, cap, row_off, start, max_per_row, max_tokens, window, sl2, B * G, nblk, rows);
  } else if (dtype == FC_BF16 && hd == 128) {
    AttnGrid a = fc_attn_grid(B, max_per_row, typ_per_row, H, G, max_keys);
    const int64_t units = (int64_t)B * G * a.nqblk * a.nsplit * 16;
    FC_CHECK_ARG(part != nullptr && part_bytes >= fc_align(units * 128 * 4) + fc_align(units * 2 * 4),
                 "attention workspace too small");
    float* po = (float*)part;
    float* pml = (float*)((char*)part + fc_align(units * 128 * 4));
    FC_CHECK_ARG(B * G <= 65535, "batch * n_kv_head must be <= 65535");
    const float sl2 = scale * 1.4426950408889634f;
    if (a.qb == 2)
      hipLaunchKernelGGL((k_attn_mfma_qb<FC_ATTN_WAVES, 2>), dim3(a.nsplit, B * G, (a.nqblk + 1) / 2),
                         dim3(64 * FC_ATTN_WAVES), 0, s, (const bf16_t*)q, (const bf16_t*)kc, (const bf16_t*)vc, po,
                         pml, (bf16_t*)y, H, G, cap, row_off, start, max_per_row, max_tokens, window, a.split_keys,
                         a.nsplit, a.nqblk, sl2, rows);
    else
      hipLaunchKernelGGL(k_attn_mfma<FC_ATTN_WAVES>, dim3(a.nsplit, B * G, a.nqblk), dim3(64 * FC_ATTN_WAVES),
                         0, s, (const bf16_t*)q, (const bf16_t*)kc, (const bf16_t*)vc, po, pml, (bf16_t*)y, H, G, cap,
                         row_off, start, max_per_row, max_tokens, window, a.split_keys, a.nsplit, a.nqblk, sl2, rows);
    if (a.nsplit > 1) {
      FC_LAUNCH_CHECK();
#define COMBINE(CB)                                                                                              \
  hipLaunchKernelGGL((k_attn_combine<bf16_t, CB>), dim3(B * G, a.nqblk), dim3(256), 0, s, po, pml, (bf16_t*)y, H, G, \
                     a.nqblk, a.nsplit, row_off, max_per_row, max_tokens, rows)
      if (a.nsplit <= 2) COMBINE(2);
      else if (a.nsplit <= 4) COMBINE(4);
      else COMBINE(8);
#undef COMBINE
    }
  } else {
    FC_CHECK_ARG(hd <= 128, "head_dim must be <= 128");
    FC_CHECK_ARG(max_keys <= VALU_MAXK, "VALU attention supports at most 8192 visible keys");
    const dim3 grid(max_per_row, H, B);
    // 16-byte operand loads: every array on its boundary (head_dim 128 keeps the rows on it)
    const bool vec = (((uintptr_t)q | (uintptr_t)kc | (uintptr_t)vc | (uintptr_t)y) & 15) == 0;
    if (dtype == FC_F32 && hd == 128 && vec && (int64_t)B * G <= 65535)
      hipLaunchKernelGGL(k_attn_f32, dim3((max_per_row * (H / G) + 31) / 32, B * G), dim3(64 * AF_WAVES), 0, s,
                         (const float*)q, (const float*)kc, (const float*)vc, (float*)y, H, G, cap, row_off, start,
                         max_per_row, max_tokens, window, scale);
    else if (dtype == FC_BF16)
      hipLaunchKernelGGL(k_attn_valu<bf16_t>, grid, dim3(256), 0, s, (const bf16_t*)q, (const bf16_t*)kc,
                         (const bf16_t*)vc, (bf16_t*)y, H, G, hd, cap, row_off, start, max_per_row, max_tokens,
                         window, scale, rows);
    else
      hipLaunchKernelGGL(k_attn_valu<float>, grid, dim3(256), 0, s, (const float*)q, (const float*)kc,
                         (const float*)vc, (float*)y, H, G, hd, cap, row_off, start, max_per_row, max_tokens, window,
                         scale, rows);
  }
  FC_LAUNCH_CHECK();
  return FC_OK;
}

extern "C" int64_t fc_attention_workspace_bytes(int32_t batch, int32_t max_per_row, int32_t n_head,
                                                int32_t n_kv_head, int32_t head_dim, int32_t max_keys) {
  return fc_attn_part_bytes(batch, max_per_row, n_head, n_kv_head, head_dim, max_keys);
}

extern "C" int32_t fc_attention(const void* q, const void* kc, const void* vc, void* y, int32_t batch,
                                int32_t max_tokens, int32_t max_per_row, int32_t n_head, int32_t n_kv_head,
                                int32_t head_dim, int32_t cap, const int32_t* row_off, const int32_t* start,
                                int32_t window, int32_t max_keys, int32_t dtype, void* work, int64_t work_bytes,
                                void* stream) {
  FC_CHECK_ARG(q && kc && vc && y && row_off && start, "null pointer");
  FC_CHECK_ARG(batch > 0 && max_tokens > 0 && max_per_row > 0 && n_head > 0 && n_kv_head > 0, "sizes");
  FC_CHECK_ARG(max_keys > 0 && max_keys <= cap, "max_keys must be in [1, cap]");
  return fc_launch_attention(q, kc, vc, y, batch, max_tokens, max_per_row, max_per_row, n_head, n_kv_head, head_dim,
                             cap, row_off, start, window, max_keys, dtype, work, work_bytes, (hipStream_t)stream, 0);
}

extern "C" int32_t fc_attention_rows(const void* q, const void* kc, const void* vc, void* y, int32_t batch,
                                     int32_t max_tokens, int32_t max_per_row, int32_t n_head, int32_t n_kv_head,
                                     int32_t head_dim, int32_t cap, const int32_t* row_off, const int32_t* start,
                                     int32_t window, int32_t max_keys, int32_t dtype, void* work, int64_t work_bytes,
                                     void* stream) {
  FC_CHECK_ARG(q && kc && vc && y && row_off && start, "null pointer");
  FC_CHECK_ARG(batch > 0 && max_tokens > 0 && max_per_row > 0 && n_head > 0 && n_kv_head > 0, "sizes");
  FC_CHECK_ARG(max_keys > 0 && max_keys <= cap, "max_keys must be in [1, cap]");
  return fc_launch_attention(q, kc, vc, y, batch, max_tokens, max_per_row, max_per_row, n_head, n_kv_head, head_dim,
                             cap, row_off, start, window, max_keys, dtype, work, work_bytes, (hipStream_t)stream, 1);
}

// ---------------------------------------------------------------------------
// fc_attention_noalloc: fc_attention for callers that cannot allocate (code
// under stream capture, serving loops that forbid allocation). The split-KV
// partials (unnormalised O and (max, sum) per query column and key split)
// live in `scratch`, a file-scope device array each GPU holds until the
// process ends. Nothing in it has to start at zero: a launch writes every
// partial its combine step reads (empty key splits write (-inf, 0)). All
// calls on one GPU share that GPU's array, so calls that overlap in time on
// one GPU (different streams, or host threads) race; calls ordered on one
// stream do not.
// ---------------------------------------------------------------------------
#ifndef FC_NOALLOC_SCRATCH_BYTES
#define FC_NOALLOC_SCRATCH_BYTES (32ll << 20)
#endif
static __device__ __align__(256) char scratch[FC_NOALLOC_SCRATCH_BYTES];

namespace {
constexpr int kScratchMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kScratchMaxDevices];  // device address of `scratch`, per device
}  // namespace

// The device address of `scratch` on the GPU `stream` runs on (the current
// device for the null stream), looked up once per device with that device
// current. Host code must use this address, never the array's name.
static int fc_scratch_ptr(hipStream_t stream, void** out) {
  int cur = 0;
  FC_HIP(hipGetDevice(&cur));
  int dev = cur;
  if (stream != nullptr) {
    hipDevice_t sd = 0;
    FC_HIP(hipStreamGetDevice(stream, &sd));
    dev = (int)sd;
  }
  FC_CHECK_ARG(dev >= 0 && dev < kScratchMaxDevices, "device ordinal beyond the scratch table");
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (g_scratch_ptr[dev] == nullptr) {
    if (dev != cur) FC_HIP(hipSetDevice(dev));
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (dev != cur) FC_HIP(hipSetDevice(cur));
    if (e != hipSuccess || p == nullptr) {
      fc_set_error(std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
      return FC_ERR_HIP;
    }
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return FC_OK;
}

// Resolves the scratch address of the stream's GPU ahead of time: fc_graph_begin
// calls it before capture starts, so a captured fc_attention_noalloc makes no
// runtime lookup inside the capture.
int fc_noalloc_prepare(hipStream_t stream) {
  void* p = nullptr;
  return fc_scratch_ptr(stream, &p);
}

extern "C" int64_t fc_attention_noalloc_max_bytes(void) { return FC_NOALLOC_SCRATCH_BYTES; }

extern "C" int32_t fc_attention_noalloc(const void* q, const void* kc, const void* vc, void* y, int32_t batch,
                                        int32_t max_tokens, int32_t max_per_row, int32_t n_head, int32_t n_kv_head,
                                        int32_t head_dim, int32_t cap, const int32_t* row_off, const int32_t* start,
                                        int32_t window, int32_t max_keys, int32_t dtype, void* stream) {
  FC_CHECK_ARG(q && kc && vc && y && row_off && start, "null pointer");
  FC_CHECK_ARG(batch > 0 && max_tokens > 0 && max_per_row > 0 && n_head > 0 && n_kv_head > 0, "sizes");
  FC_CHECK_ARG(max_keys > 0 && max_keys <= cap, "max_keys must be in [1, cap]");
  FC_CHECK_ARG(n_head % n_kv_head == 0, "n_head must be a multiple of n_kv_head");
  // the same kernel choice as fc_launch_attention (typical = max_per_row
  // here): only the split decode kernel (bf16, head_dim 128, below prefill
  // width) writes partials; the prefill and VALU kernels need none
  const bool split = dtype == FC_BF16 && head_dim == 128 &&
                     !attn_uses_pf(dtype, head_dim, max_per_row, n_head, n_kv_head);
  const int64_t need = split ? fc_attn_part_bytes(batch, max_per_row, n_head, n_kv_head, head_dim, max_keys) : 0;
  if (need > FC_NOALLOC_SCRATCH_BYTES) {
    fc_set_error("fc_attention_noalloc: these sizes need " + std::to_string(need) +
                 " bytes of split-KV partials; the static scratch holds " +
                 std::to_string((long long)FC_NOALLOC_SCRATCH_BYTES) + " (use fc_attention with a workspace)");
    return FC_ERR_CAPACITY;
  }
  void* part = nullptr;
  const int rc = fc_scratch_ptr((hipStream_t)stream, &part);
  if (rc != FC_OK) return rc;
  return fc_launch_attention(q, kc, vc, y, batch, max_tokens, max_per_row, max_per_row, n_head, n_kv_head, head_dim,
                             cap, row_off, start, window, max_keys, dtype, part, FC_NOALLOC_SCRATCH_BYTES,
                             (hipStream_t)stream, 0);
}
