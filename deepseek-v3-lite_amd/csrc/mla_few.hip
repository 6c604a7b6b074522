// (f4) MLA attention for a few queries over a long latent cache (decoding, a
// handful of speculated tokens): the attention of mla.hip (models/mla_triton.py:73-183,
// the same masks and scale) without materialising K and V.
//
// With k_nope = c W_k^T and v = c W_v^T for a latent row c, the score of a query
// is (q_nope W_k) . c + q_pe . pe and its output (sum_j p_j c_j) W_v^T, so a pass
// reads each latent row once for all heads instead of writing and reading
// 2 D_nope + D_rope + D_v columns of every (row, head).  Rows of the score matrix
// are (query, head) pairs, M = S_q H of them per batch.
//
//   mla_absorb_kernel   q_abs = q_nope W_k in fp32, stored as an exact pair of bf16
//                       parts (hi, lo: about 16 significant bits, as mla.hip keeps
//                       K_nope), followed by q_pe.
//   mla_few_kernel      flash attention of 32 rows over one range of keys per wave:
//                       scores from the latent rows in registers (the fragment of
//                       a latent row serves hi and lo), the same rows staged in the
//                       wave's own LDS tile and read transposed for sum_j p_j c_j.
//                       fp32 partial sums, maximum and normaliser per range.
//   mla_few_out_kernel  the ranges added by their weights, times W_v^T in fp32.
//
// p is rounded to bf16 for its MFMA as in mla.hip; c is exact there where mla.hip
// rounds v (relative error against float64 1.7e-3, mla.hip 2.1e-3).
//
// Measured at H 12, R 192, D_nope 48, D_rope 24, D_v 64 (us per call in a graph,
// K and V built against this path): B 8, S_q 1, S_kv 1537: 54, 18 (absorb 4.0,
// attention 9.5, sum 5.8; 5.7 MB of latent rows, 1.1 us at 5.2 TB/s: launch and
// load latencies bound it); B 32, S_q 1, S_kv 600: 77, 19; B 8, S_q 16, S_kv 1537: 54, 40;
// B 8, S_q 16, S_kv 300: 26, 28.  Where the line lies: _few in dsmoe/mla.py.
#include <algorithm>
#include <cstring>

#include "mla_tile.h"

namespace dsmoe {

constexpr int FEW_MAX_SPLITS = 128;

struct MlaFew {
  const bf16_t* q_nope;   // (B, H, S_q, Dn)
  const bf16_t* q_pe;     // (B, H, S_q, Dr)
  const bf16_t* ctx_kv;   // (B, S_kv, R)
  const bf16_t* ctx_pe;   // (B, S_kv, Dr)
  const bf16_t* w_k;      // head h's (Dn, R) rows at h wk_hs
  const bf16_t* w_v;      // head h's (Dv, R) rows at h wv_hs
  int64_t wk_hs, wv_hs;
  bf16_t* out;            // (B, S_q, H, Dv)
  float* lse;             // (B, H, S_q) base-2 log-sum-exp, or null
  bf16_t* qabs;           // (B, Mp, 2 Rq + Drp): [hi | lo | pe], zeros in the padding
  float* po;              // (B, nsplit, Mp, Rq) partial sums of p c
  float2* ml;             // (B, nsplit, Mp) {max of the scores, sum of p}
  int B, H, S_q, S_kv, R, Dn, Dr, Dv;
  int M, Mp;              // rows (s H + h) of a batch, rounded up to whole tiles of 32
  int Rq, Drp;            // R and Dr in whole MFMA steps
  int nsplit, cpw;        // key ranges, and 32-key chunks of one
  int causal, q_start;
  int neg;                // softmax_scale < 0: q is negated, c = |scale| log2(e)
  int wvec;               // 16-byte loads of weight rows
  float c;
};

// 8 bf16 at p (16 bytes), or those of p[0 .. n) one by one and zeros.
__device__ __forceinline__ bf16x8_t few_ld8(const bf16_t* p, int n, bool vec) {
  mla_u32x4 v;
  if (vec) {
    v = *reinterpret_cast<const mla_u32x4*>(p);
  } else {
    bf16_t e8[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) e8[e] = e < n ? p[e] : bf16_t(0);
    v = *reinterpret_cast<const mla_u32x4*>(e8);
  }
  return __builtin_bit_cast(bf16x8_t, v);
}

// The first key that no row of tile mt sees (at least 1).
__device__ __forceinline__ int few_kend(const MlaFew& a, int mt) {
  return a.causal ? min(a.S_kv, (min(a.M, 32 * mt + 32) - 1) / a.H + a.q_start + 1) : a.S_kv;
}

// Grid (M, B).  Thread (g, c): columns 8 c .. 8 c + 7 over the D_nope rows g,
// g + groups, ..., the groups added through LDS.
__global__ __launch_bounds__(256) void mla_absorb_kernel(const MlaFew a) {
  extern __shared__ __attribute__((aligned(16))) float few_sm[];
  const int tid = threadIdx.x, row = blockIdx.x, b = blockIdx.y;
  const int s = row / a.H, h = row - s * a.H;
  const int64_t q = ((int64_t)b * a.H + h) * a.S_q + s;
  const bf16_t* qn = a.q_nope + q * a.Dn;
  const bf16_t* qp = a.q_pe + q * a.Dr;
  bf16_t* dst = a.qabs + ((int64_t)b * a.Mp + row) * (2 * a.Rq + a.Drp);
  const int cols = a.Rq / 8, groups = 256 / cols;
  const int g = tid / cols, c = tid - g * cols;
  if (g < groups) {
    float acc[8] = {};
    const int n = min(8, a.R - 8 * c);
    const bf16_t* w = a.w_k + (int64_t)h * a.wk_hs + 8 * c;
    if (n > 0) {
#pragma unroll 4
      for (int d = g; d < a.Dn; d += groups) {
        const bf16x8_t v = few_ld8(w + (int64_t)d * a.R, n, a.wvec != 0);
        const float qd = bf2f(qn[d]);
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] = fmaf(qd, (float)v[e], acc[e]);
      }
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) few_sm[g * a.Rq + 8 * c + e] = acc[e];
  }
  __syncthreads();
  for (int r = tid; r < a.Rq; r += 256) {
    float v = few_sm[r];
    for (int i = 1; i < groups; ++i) v += few_sm[i * a.Rq + r];
    if (a.neg) v = -v;
    const bf16_t hi = f2bf(v);
    dst[r] = hi;
    dst[a.Rq + r] = f2bf(v - bf2f(hi));
  }
  for (int d = tid; d < a.Drp; d += 256)
    dst[2 * a.Rq + d] = d < a.Dr ? (bf16_t)(qp[d] ^ (a.neg ? 0x8000 : 0)) : bf16_t(0);
}

// One wave per (batch, row tile, key range), range fastest.  A range past few_kend
// writes nothing (mla_few_out_kernel does not read it).  NS = Rq / 16; VEC:
// 16-byte loads of latent and rope rows.
template <int NS, bool VEC>
__global__ __launch_bounds__(256) void mla_few_kernel(const MlaFew a) {
  constexpr int NV = NS / 2;                             // 32-column tiles of the latent row
  constexpr int RB = (NS * 16 + 127) / 128 * 256;        // LDS tile row bytes
  extern __shared__ __attribute__((aligned(16))) char few_tile[];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int hi = lane >> 5, l32 = lane & 31;
  const int mts = a.Mp / 32;
  const int unit = blockIdx.x * 4 + wave;
  const int split = unit % a.nsplit, bm = unit / a.nsplit;
  const int mt = bm % mts, b = bm / mts;
  if (b >= a.B) return;
  const int row = 32 * mt + l32;
  const int qpos = row / a.H + a.q_start;
  const int kb = split * a.cpw * 32, ke = min(few_kend(a, mt), kb + a.cpw * 32);
  const int64_t part = ((int64_t)b * a.nsplit + split) * a.Mp + row;
  if (kb >= ke) return;
  char* tile = few_tile + wave * 32 * RB;
  const MlbLane<RB> lk(lane);
  const bf16_t* qrow = a.qabs + ((int64_t)b * a.Mp + min(row, a.M - 1)) * (2 * a.Rq + a.Drp) + 8 * hi;
  bf16x8_t qh[NS], ql[NS];
#pragma unroll
  for (int st = 0; st < NS; ++st) {
    qh[st] = *reinterpret_cast<const bf16x8_t*>(qrow + 16 * st);
    ql[st] = *reinterpret_cast<const bf16x8_t*>(qrow + a.Rq + 16 * st);
  }
  mla_f32x16 o[NV];
#pragma unroll
  for (int v = 0; v < NV; ++v)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[v][i] = 0.0f;
  float m = -INFINITY, l = 0.0f;
  // the lane's latent row of a chunk, clamped to the last visible key; columns past
  // R: whole-chunk loads repeat the row's last ones (q_abs is zero there)
  const auto krow = [&](int k0) { return (int64_t)b * a.S_kv + min(k0 + l32, ke - 1); };
  bf16x8_t cf[NS];
  const auto load = [&](int k0) {
    const bf16_t* cr = a.ctx_kv + krow(k0) * a.R;
#pragma unroll
    for (int st = 0; st < NS; ++st) {
      const int col = 16 * st + 8 * hi;
      cf[st] = VEC ? few_ld8(cr + min(col, a.R - 8), 8, true) : few_ld8(cr + col, a.R - col, false);
    }
  };
  load(kb);
  for (int k0 = kb; k0 < ke; k0 += 32) {
#pragma unroll
    for (int st = 0; st < NS; ++st)
      *reinterpret_cast<bf16x8_t*>(tile + lk.f[st & 7] + 256 * (st >> 3)) = cf[st];
    // scores: register i -> key k0 + 8 (i / 4) + 4 hi + i % 4
    mla_f32x16 s;
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = 0.0f;
    const bf16_t* pr = a.ctx_pe + krow(k0) * a.Dr;
    for (int d = 8 * hi; d < a.Drp; d += 16) {
      const bf16x8_t pf = VEC ? few_ld8(pr + min(d, a.Dr - 8), 8, true) : few_ld8(pr + d, a.Dr - d, false);
      s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
          pf, *reinterpret_cast<const bf16x8_t*>(qrow + 2 * a.Rq + d - 8 * hi), s, 0, 0, 0);
    }
#pragma unroll
    for (int st = 0; st < NS; ++st) {
      s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(cf[st], ql[st], s, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(cf[st], qh[st], s, 0, 0, 0);
    }
    if (k0 + 32 < ke) load(k0 + 32);
    float mb = -INFINITY;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int key = k0 + 8 * (i >> 2) + 4 * hi + (i & 3);
      if (key >= ke || (a.causal && key > qpos)) s[i] = -INFINITY;
      mb = fmaxf(mb, s[i]);
    }
    mb = mla_pair_max(mb);
    const float mn = fmaxf(m, mb);
    const float mc = mn == -INFINITY ? 0.0f : mn * a.c;
    const float alpha = m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(fmaf(m, a.c, -mc));
    const bool moved = m != mn;
    m = mn;
    float ls = 0.0f;
    bf16x8_t pf[2];
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      bf16x2_t w[4];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float p = __builtin_amdgcn_exp2f(fmaf(s[8 * half + e], a.c, -mc));
        ls += p;
        w[e >> 1][e & 1] = (__bf16)p;
      }
      pf[half] = __builtin_bit_cast(bf16x8_t, w);
    }
    l = l * alpha + ls;
    if (__builtin_amdgcn_ballot_w64(moved)) {
#pragma unroll
      for (int v = 0; v < NV; ++v)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[v][i] *= alpha;
    }
    // the tile's writes (this wave's own, completed in order) before its transposed reads
    wait_lgkm0();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int ps = 0; ps < 2; ++ps)
#pragma unroll
      for (int v = 0; v < NV; ++v)
        o[v] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(lk.tfrag(tile, 16 * ps, v), pf[ps], o[v], 0, 0, 0);
    wait_lgkm0();
    asm volatile("" ::: "memory");
  }
  l = mla_pair_sum(l);
  if (row >= a.M) return;
  if (hi == 0) a.ml[part] = make_float2(m, l);
  float* po = a.po + part * a.Rq;
#pragma unroll
  for (int v = 0; v < NV; ++v)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *reinterpret_cast<float4*>(po + 32 * v + 8 * g + 4 * hi) =
          make_float4(o[v][4 * g], o[v][4 * g + 1], o[v][4 * g + 2], o[v][4 * g + 3]);
}

// The ranges of a row added by their weights.  Every range that mla_few_kernel
// wrote takes part, whatever it holds: a NaN in one key, or in the query, reaches
// the sum as in mla.hip, also through a weight of 0 (a range whose scores are all
// NaN has no maximum).
// Grid (M, B).  LDS (floats): weights of the ranges [FEW_MAX_SPLITS] | group sums
// [groups][Rq] (the first row then holds the normalised sum).
__global__ __launch_bounds__(256) void mla_few_out_kernel(const MlaFew a) {
  extern __shared__ __attribute__((aligned(16))) float few_sm[];
  float* wt = few_sm;
  float* sum = few_sm + FEW_MAX_SPLITS;
  const int tid = threadIdx.x, row = blockIdx.x, b = blockIdx.y;
  const int s = row / a.H, h = row - s * a.H;
  const int64_t p0 = (int64_t)b * a.nsplit * a.Mp + row;
  const int nr = min(a.nsplit, (few_kend(a, row / 32) + 32 * a.cpw - 1) / (32 * a.cpw));   // ranges written
  // every wave reduces the ranges' maxima and normalisers, two ranges per lane
  const int lane = tid & 63;
  static_assert(FEW_MAX_SPLITS == 128, "two ranges per lane");
  float2 r2[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int i = lane + 64 * u;
    r2[u] = a.ml[p0 + (int64_t)min(i, nr - 1) * a.Mp];
    if (i >= nr) r2[u] = make_float2(-INFINITY, 0.0f);
  }
  float m = fmaxf(r2[0].x, r2[1].x);
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) m = fmaxf(m, __shfl_xor(m, d));
  float lt = 0.0f;
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const float w = r2[u].x != -INFINITY ? __builtin_amdgcn_exp2f((r2[u].x - m) * a.c) : 0.0f;
    lt = fmaf(w, r2[u].y, lt);
    if (tid < 64) wt[lane + 64 * u] = w;
  }
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) lt += __shfl_xor(lt, d);
  __syncthreads();
  const int cols = a.Rq / 4, groups = 256 / cols;
  const int g = tid / cols, c = tid - g * cols;
  if (g < groups) {
    float4 acc = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    const float* po = a.po + p0 * a.Rq + 4 * c;
    const int64_t step = (int64_t)a.Mp * a.Rq;
    constexpr int U = 6;   // loads in flight
    for (int i = g; i < nr; i += U * groups) {
      float4 v[U];
#pragma unroll
      for (int u = 0; u < U; ++u)
        v[u] = *reinterpret_cast<const float4*>(po + min(i + u * groups, nr - 1) * step);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const bool on = i + u * groups < nr;
        const float w = wt[min(i + u * groups, FEW_MAX_SPLITS - 1)];
        acc.x = fmaf(w, on ? v[u].x : 0.0f, acc.x);
        acc.y = fmaf(w, on ? v[u].y : 0.0f, acc.y);
        acc.z = fmaf(w, on ? v[u].z : 0.0f, acc.z);
        acc.w = fmaf(w, on ? v[u].w : 0.0f, acc.w);
      }
    }
    *reinterpret_cast<float4*>(sum + g * a.Rq + 4 * c) = acc;
  }
  __syncthreads();
  const float inv = lt > 0.0f ? 1.0f / lt : 0.0f;
  for (int r = tid; r < a.Rq; r += 256) {
    float v = sum[r];
    for (int i = 1; i < groups; ++i) v += sum[i * a.Rq + r];
    sum[r] = v * inv;
  }
  __syncthreads();
  if (a.lse && tid == 0) a.lse[((int64_t)b * a.H + h) * a.S_q + s] = lt > 0.0f ? m * a.c + log2f(lt) : INFINITY;
  // four lanes per output column, every fourth chunk of 8 latent columns each
  bf16_t* orow = a.out + (((int64_t)b * a.S_q + s) * a.H + h) * a.Dv;
  const int q4 = tid & 3;
  for (int dv = tid >> 2; dv < a.Dv; dv += 64) {
    const bf16_t* w = a.w_v + (int64_t)h * a.wv_hs + (int64_t)dv * a.R;
    float acc = 0.0f;
#pragma unroll 4
    for (int r = 8 * q4; r < a.R; r += 32) {
      const bf16x8_t v = few_ld8(w + r, a.R - r, a.wvec != 0);
#pragma unroll
      for (int e = 0; e < 8; ++e) acc = fmaf(sum[min(r + e, a.Rq - 1)], (float)v[e], acc);
    }
    acc += __shfl_xor(acc, 1);
    acc += __shfl_xor(acc, 2);
    if (q4 == 0) orow[dv] = f2bf(acc);
  }
}

// ------------------------------------------------------------------ host
static MlaFew few_args(const dsmoe_mla_dims* d) {
  MlaFew a;
  std::memset(static_cast<void*>(&a), 0, sizeof(a));
  a.B = d->B; a.H = d->H; a.S_q = d->S_q; a.S_kv = d->S_kv;
  a.R = d->R; a.Dn = d->D_nope; a.Dr = d->D_rope; a.Dv = d->D_v;
  a.M = d->S_q * d->H;
  a.Mp = (int)align_up(a.M, 32);
  for (int ns : {2, 4, 8, 12, 16})
    if (a.Rq == 0 && d->R <= 16 * ns) a.Rq = 16 * ns;
  a.Drp = (int)align_up(d->D_rope, 16);
  // about 1024 waves (four for each CU), ranges of whole 32-key chunks
  const int64_t chunks = cdiv(d->S_kv, 32), tiles = (int64_t)a.B * (a.Mp / 32);
  a.cpw = (int)std::max(std::max<int64_t>(1, tiles * chunks / 1024), cdiv(chunks, FEW_MAX_SPLITS));
  a.nsplit = (int)cdiv(chunks, a.cpw);
  a.causal = d->is_causal ? 1 : 0;
  a.q_start = d->q_start;
  a.neg = d->softmax_scale < 0.0f ? 1 : 0;
  a.c = (d->softmax_scale < 0.0f ? -d->softmax_scale : d->softmax_scale) * MLA_LOG2E;
  return a;
}

static size_t few_carve(MlaFew& a, void* ws) {
  Carver c(ws);
  a.qabs = c.take<bf16_t>((size_t)a.B * a.Mp * (2 * a.Rq + a.Drp));
  a.ml = c.take<float2>((size_t)a.B * a.nsplit * a.Mp);
  a.po = c.take<float>((size_t)a.B * a.nsplit * a.Mp * a.Rq);
  return c.used();
}

template <int NS>
static int launch_few(const MlaFew& a, bool vec, hipStream_t st) {
  constexpr size_t lds = 4 * 32 * ((NS * 16 + 127) / 128 * 256);
  const int64_t units = (int64_t)a.B * (a.Mp / 32) * a.nsplit;
  auto kern = vec ? mla_few_kernel<NS, true> : mla_few_kernel<NS, false>;
  hipLaunchKernelGGL(kern, dim3((unsigned)cdiv(units, 4)), dim3(256), lds, st, a);
  return check_launch("mla_few");
}

}  // namespace dsmoe

using namespace dsmoe;

extern "C" size_t dsmoe_mla_attn_few_workspace_size(const dsmoe_mla_dims* dims) {
  if (dsmoe_mla_attn_workspace_size(dims) == 0) return 0;
  MlaFew a = few_args(dims);
  return few_carve(a, nullptr);
}

extern "C" int dsmoe_mla_attn_few(const void* q_nope, const void* q_pe, const void* ctx_kv, const void* ctx_pe,
                                  const void* wkv_b_k, int64_t wk_head_stride, const void* wkv_b_v,
                                  int64_t wv_head_stride, const dsmoe_mla_dims* dims, void* out, float* lse,
                                  void* workspace, size_t workspace_bytes, void* stream) {
  const size_t need = dsmoe_mla_attn_few_workspace_size(dims);
  if (need == 0)   // dims no attention call takes: that call's error
    return dsmoe_mla_attn_fwd(nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, dims, nullptr, nullptr, 0, nullptr);
  DSMOE_REQUIRE(q_nope && q_pe && ctx_kv && ctx_pe && wkv_b_k && wkv_b_v && out, DSMOE_ERR_INVALID,
                "mla_few: NULL tensor pointer");
  DSMOE_REQUIRE(wk_head_stride >= 0 && wv_head_stride >= 0, DSMOE_ERR_INVALID, "mla_few: negative weight stride");
  DSMOE_REQUIRE(workspace && workspace_bytes >= need, DSMOE_ERR_WORKSPACE, "mla_few: workspace too small");
  DSMOE_REQUIRE((reinterpret_cast<uintptr_t>(workspace) & 15) == 0, DSMOE_ERR_INVALID,
                "mla_few: workspace must be 16-byte aligned");
  MlaFew a = few_args(dims);
  few_carve(a, workspace);
  a.q_nope = static_cast<const bf16_t*>(q_nope);
  a.q_pe = static_cast<const bf16_t*>(q_pe);
  a.ctx_kv = static_cast<const bf16_t*>(ctx_kv);
  a.ctx_pe = static_cast<const bf16_t*>(ctx_pe);
  a.w_k = static_cast<const bf16_t*>(wkv_b_k);
  a.w_v = static_cast<const bf16_t*>(wkv_b_v);
  a.wk_hs = wk_head_stride;
  a.wv_hs = wv_head_stride;
  a.out = static_cast<bf16_t*>(out);
  a.lse = lse;
  const auto al = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
  a.wvec = (a.R % 8 == 0 && wk_head_stride % 8 == 0 && wv_head_stride % 8 == 0 && al(wkv_b_k) && al(wkv_b_v)) ? 1 : 0;
  const bool vec = a.R % 8 == 0 && a.Dr % 8 == 0 && al(ctx_kv) && al(ctx_pe);
  hipStream_t st = static_cast<hipStream_t>(stream);
  const dim3 grid((unsigned)a.M, (unsigned)a.B);
  hipLaunchKernelGGL(mla_absorb_kernel, grid, dim3(256), sizeof(float) * (256 / (a.Rq / 8)) * a.Rq, st, a);
  int rc = check_launch("mla_absorb");
  if (rc) return rc;
  switch (a.Rq / 16) {
    case 2: rc = launch_few<2>(a, vec, st); break;
    case 4: rc = launch_few<4>(a, vec, st); break;
    case 8: rc = launch_few<8>(a, vec, st); break;
    case 12: rc = launch_few<12>(a, vec, st); break;
    default: rc = launch_few<16>(a, vec, st); break;
  }
  if (rc) return rc;
  hipLaunchKernelGGL(mla_few_out_kernel, grid, dim3(256),
                     sizeof(float) * (FEW_MAX_SPLITS + (size_t)(256 / (a.Rq / 4)) * a.Rq), st, a);
  return check_launch("mla_few_out");
}
