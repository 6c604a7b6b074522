// Grouped GEMMs of the fp32 layer, both directions, on the fp32 matrix cores.
//
// Forward (GemmDesc): x W1^T | x W3^T with the SwiGLU epilogue and h W2^T, as
// models/moe.py:127-131,166-179; backward (XGemm): dh, dx and the weight
// gradients, operand layouts as listed in gemm_x.hip.  Every product is an
// fp32 product accumulated in fp32 (v_mfma_f32_32x32x2_f32), the K range in
// ascending slabs by one workgroup per output tile, no atomics.  The shared experts'
// weight gradients, whose K is all tokens, are cut along K into 1 to 8 parts by shape
// (xgemm_f32_ksplit); wgrad_reduce_kernel adds the parts in ascending order.
//
// What bounds it: the fp32 matrix rate, 64 cycles per 32x32x2 MFMA and SIMD
// (157 TFLOP/s; the vector FMA units without packed instructions reach half of
// that).  A wave reads two 16-byte fragments per 8 K values for four MFMAs (256
// cycles), so LDS is busy an eighth of the time.  The next slab's loads are in
// registers while the current one computes; one LDS buffer and two barriers per
// slab, so that 4 to 6 workgroups share a CU and cover each other's barriers and
// load latency.  Measured at D 768, E 20, k 4, I 384, T 2048 (us; the FMA kernels
// this replaces, then this one): gate/up 681, 145 (84 TFLOP/s); down 279, 70; dh
// 229, 69; dx 300, 115; dW1|dW3 247, 107; dW2 143, 68; the shared experts' three
// 175 + 177 + 893, 29 + 35 + 69.  Two buffers and one barrier, at half the
// workgroups per CU: 163, 78, 73, 126, 110, 68.  128 x 128 tiles with two buffers:
// 193, 102, 114, 149, 164, 102 (the last round of tiles is emptier).
//
// K order inside a slab: lane half h of MFMA i of group j takes k = 8 j + 4 h
// + i, which lets a lane read four K values of a row with one ds_read_b128.
// LDS tiles: "row form" [row][32 k + 4 pad] for operands contiguous in K (16
// rows' 16-byte reads cover all 64 banks once), "K form" [32 k][cols + 8 pad]
// for operands contiguous in M or N (the two lane halves read rows k and k + 4,
// half the banks apart).
#include <algorithm>

#include "gemm_tile.h"
#include "mfma.h"

namespace dsmoe {

constexpr int F_FK_ROWS = 32;   // K slab of the kernels with a row-form operand
constexpr int F_FK_WGRAD = 16;  // K slab of the weight gradients (32: dW1|dW3 144 against 125 us at the shape above)
constexpr int FB = 64;          // output tile: FB x FB (SwiGLU: of each operand), a wave 32 x 32 of it

typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(1))) const f32x4_t gf32x4_t;
typedef __attribute__((address_space(1))) const float gf32_t;
__device__ __forceinline__ f32x4_t ldg_f4(const float* p) { return *(gf32x4_t*)(p); }
__device__ __forceinline__ float ldg_f(const float* p) { return *(gf32_t*)(p); }

// An operand tile of FB rows (row form) or columns (K form) by FK of K in LDS,
// staged by 256 threads in 16-byte chunks.
template <int FK, bool KF>
struct FTile {
  static constexpr int LD = KF ? FB + 8 : FK + 4;              // leading dimension
  static constexpr int FLOATS = (KF ? FK : FB) * LD;
  static constexpr int N = FB * FK / 4 / 256;                  // chunks per thread
  static constexpr int L = (KF ? FB : FK) / 4;                 // chunks of a line
  // line (row, or K row) and column (K, or column) of a thread's chunk i
  static __device__ __forceinline__ int row(int tid, int i) { return tid / L + 256 / L * i; }
  static __device__ __forceinline__ int col(int tid) { return 4 * (tid % L); }
  static __device__ __forceinline__ void put(float* s, int tid, const f32x4_t (&v)[N]) {
#pragma unroll
    for (int i = 0; i < N; ++i) *reinterpret_cast<f32x4_t*>(s + row(tid, i) * LD + col(tid)) = v[i];
  }
  // Fragment of rows (columns) c0 .. c0 + 31: the lane's is c0 + (lane & 31), K
  // values 8 j + 4 (lane >> 5) + {0..3}.
  static __device__ __forceinline__ f32x4_t frag(const float* s, int c0, int j, int lane) {
    if constexpr (KF) {
      const float* p = s + (8 * j + 4 * (lane >> 5)) * LD + c0 + (lane & 31);
      return f32x4_t{p[0], p[LD], p[2 * LD], p[3 * LD]};
    } else {
      return *reinterpret_cast<const f32x4_t*>(s + (c0 + (lane & 31)) * LD + 8 * j + 4 * (lane >> 5));
    }
  }
};

// acc[b] += A B_b^T over one slab; the B fragment is the first MFMA operand, so a
// lane holds one row m and per q the columns 8 q + 4 (lane >> 5) + {0..3}.
template <int FK, int NB, bool AK, bool BK>
__device__ __forceinline__ void f_slab(const float* sA, const float* sB, int m0, int n0, int lane,
                                       f32x16_t (&acc)[NB]) {
#pragma unroll
  for (int j = 0; j < FK / 8; ++j) {
    const f32x4_t af = FTile<FK, AK>::frag(sA, m0, j, lane);
    f32x4_t bf[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) bf[b] = FTile<FK, BK>::frag(sB + b * FTile<FK, BK>::FLOATS, n0, j, lane);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int b = 0; b < NB; ++b) acc[b] = __builtin_amdgcn_mfma_f32_32x32x2f32(bf[b][i], af[i], acc[b], 0, 0, 0);
  }
}

// Four consecutive floats of a row of `n` (the first at column c): whole when
// VEC (n and every stride and base a multiple of four floats), else one by one.
// Columns past the row read its last ones and are given 0 when ZERO.
template <bool VEC, bool ZERO>
__device__ __forceinline__ f32x4_t f_row4(const float* row, int c, int n) {
  f32x4_t v;
  if constexpr (VEC) {
    v = ldg_f4(row + min(c, n - 4));
    if (ZERO && c >= n) v = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  } else {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      v[q] = ldg_f(row + min(c + q, n - 1));
      if (ZERO && c + q >= n) v[q] = 0.0f;
    }
  }
  return v;
}

// Columns c .. c + 3 of row `row` of an (N x K) weight whose K columns lie in
// segments of kseg columns, one block each (tab[segment]).
template <bool VEC>
__device__ __forceinline__ f32x4_t f_seg4(const void* const* tab, int64_t row_off, int c, int K, int kseg) {
  f32x4_t v;
  if constexpr (VEC) {
    const int cc = min(c, K - 4), seg = cc / kseg;
    v = ldg_f4(static_cast<const float*>(tab[seg]) + row_off + (cc - seg * kseg));
    if (c >= K) v = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  } else {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int cc = min(c + q, K - 1), seg = cc / kseg;
      v[q] = ldg_f(static_cast<const float*>(tab[seg]) + row_off + (cc - seg * kseg));
      if (c + q >= K) v[q] = 0.0f;
    }
  }
  return v;
}

__device__ __forceinline__ void f_put4(float* p, const f32x4_t& v, int left, bool vec) {
  if (vec) {
    *reinterpret_cast<f32x4_t*>(p) = v;
  } else {
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (q < left) p[q] = v[q];
  }
}

// The tile of block j of XCD x in one problem (routed or dense): tiles of FB rows
// (the schedule's entries are cut into bm / FB), N fastest, XCD x taking the x-th
// eighth of the list.
__device__ __forceinline__ bool f_tile_at(const GemmDesc& g, int64_t j, int x, int64_t& per_xcd, int& grp, int& row0,
                                          int& rows, int& n_tile) {
  const int n_tiles = (int)cdiv(g.N, FB);
  const int sub = g.sched ? g.bm / FB : 1;
  const int tpg = g.sched ? 0 : (int)cdiv(g.dense_rows, FB);
  const int64_t total = (g.sched ? (int64_t)(*g.sched_count) * sub : (int64_t)tpg * g.groups) * n_tiles;
  per_xcd = cdiv(total, 8);
  const int64_t lin = x * per_xcd + j;
  if (j >= per_xcd || lin >= total) return false;
  const int64_t mt = lin / n_tiles;
  n_tile = (int)(lin - mt * n_tiles);
  if (g.sched) {
    const MTile t = g.sched[mt / sub];
    const int s = (int)(mt % sub);
    grp = t.group;
    row0 = t.row0 + s * FB;
    rows = min(FB, t.rows - s * FB);
    return rows > 0;
  }
  grp = (int)(mt / tpg);
  row0 = (int)(mt - (int64_t)grp * tpg) * FB;
  rows = min(FB, g.dense_rows - row0);
  return true;
}

// gd's fields for a dense tile, else gr's, one by one (a reference or a struct
// copy chosen at run time would put both arguments in scratch memory).
__device__ __forceinline__ GemmDesc f_pick(const GemmDesc& gr, const GemmDesc& gd, bool dense) {
  GemmDesc g;
  g.A = dense ? gd.A : gr.A;
  g.lda = dense ? gd.lda : gr.lda;
  g.a_map = dense ? gd.a_map : gr.a_map;
  g.B0 = dense ? gd.B0 : gr.B0;
  g.B1 = dense ? gd.B1 : gr.B1;
  g.ldb = dense ? gd.ldb : gr.ldb;
  g.kseg = dense ? gd.kseg : gr.kseg;
  g.nseg = dense ? gd.nseg : gr.nseg;
  g.N = dense ? gd.N : gr.N;
  g.K = dense ? gd.K : gr.K;
  g.C = dense ? gd.C : gr.C;
  g.ldc = dense ? gd.ldc : gr.ldc;
  g.c_map = dense ? gd.c_map : gr.c_map;
  g.c_group_col = dense ? gd.c_group_col : gr.c_group_col;
  g.Gs = dense ? gd.Gs : gr.Gs;
  g.Us = dense ? gd.Us : gr.Us;
  return g;
}

// ------------------------------------------------------------------ forward
template <int EPI, bool VEC>
__global__ __launch_bounds__(256) void gemm_f32_kernel(const GemmDesc gr, const GemmDesc gd, int has_gd,
                                                       const float* __restrict__ row_scale) {
  constexpr int NB = EPI == EPI_SWIGLU ? 2 : 1;
  constexpr int FK = F_FK_ROWS;
  using Tile = FTile<FK, false>;
  extern __shared__ __attribute__((aligned(16))) float fsm[];
  const int x = blockIdx.x & 7;
  int64_t j = blockIdx.x >> 3, per_xcd;
  int grp, row0, rows, n_tile;
  bool dense = false;
  if (!f_tile_at(gr, j, x, per_xcd, grp, row0, rows, n_tile)) {
    j -= per_xcd;
    if (!has_gd || j < 0 || !f_tile_at(gd, j, x, per_xcd, grp, row0, rows, n_tile)) return;
    dense = true;
  }
  const GemmDesc g = f_pick(gr, gd, dense);
  const int n0 = n_tile * FB;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int m_w = (wave >> 1) * 32, n_w = (wave & 1) * 32, c0 = Tile::col(tid);

  const float* arow[Tile::N];
  int64_t brow[Tile::N];
#pragma unroll
  for (int i = 0; i < Tile::N; ++i) {
    const int r = row0 + min(Tile::row(tid, i), rows - 1);
    arow[i] = static_cast<const float*>(g.A) + (g.a_map ? (int64_t)g.a_map[r] : (int64_t)r) * g.lda;
    brow[i] = (int64_t)min(n0 + Tile::row(tid, i), g.N - 1) * g.ldb;
  }
  const void* const* tab0 = g.B0 + (int64_t)grp * g.nseg;
  const void* const* tab1 = NB == 2 ? g.B1 + (int64_t)grp * g.nseg : nullptr;

  f32x4_t ra[Tile::N], rb[NB][Tile::N];
  // a slab inside K and inside one segment needs neither masks nor a segment per chunk
  const bool whole = VEC && g.kseg % FK == 0;
  const auto load = [&](int k0) {
    const int c = k0 + c0;
    if (whole) {
      const int seg = k0 / g.kseg;
#pragma unroll
      for (int i = 0; i < Tile::N; ++i) ra[i] = ldg_f4(arow[i] + c);
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const float* base = static_cast<const float*>((b ? tab1 : tab0)[seg]) + (k0 - seg * g.kseg) + c0;
#pragma unroll
        for (int i = 0; i < Tile::N; ++i) rb[b][i] = ldg_f4(base + brow[i]);
      }
    } else {
#pragma unroll
      for (int i = 0; i < Tile::N; ++i) ra[i] = f_row4<VEC, true>(arow[i], c, g.K);
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int i = 0; i < Tile::N; ++i) rb[b][i] = f_seg4<VEC>(b ? tab1 : tab0, brow[i], c, g.K, g.kseg);
    }
  };
  const auto put = [&](float* s) {
    Tile::put(s, tid, ra);
#pragma unroll
    for (int b = 0; b < NB; ++b) Tile::put(s + (1 + b) * Tile::FLOATS, tid, rb[b]);
  };

  f32x16_t acc[NB] = {};
  const int nk = (int)cdiv(g.K, FK);
  load(0);
  for (int kb = 0; kb < nk; ++kb) {
    put(fsm);
    __syncthreads();
    if (kb + 1 < nk) load((kb + 1) * FK);
    f_slab<FK, NB, false, false>(fsm, fsm + Tile::FLOATS, m_w, n_w, lane, acc);
    __syncthreads();
  }

  float* C = static_cast<float*>(g.C) + (int64_t)grp * g.c_group_col;
  float* Gs = g.Gs ? static_cast<float*>(g.Gs) + (int64_t)grp * g.c_group_col : nullptr;
  float* Us = g.Us ? static_cast<float*>(g.Us) + (int64_t)grp * g.c_group_col : nullptr;
  const bool vec = ((g.N | g.ldc | g.c_group_col) & 3) == 0 &&
                   ((reinterpret_cast<uintptr_t>(g.C) | reinterpret_cast<uintptr_t>(g.Gs) |
                     reinterpret_cast<uintptr_t>(g.Us)) & 15) == 0;
  const int m = m_w + (lane & 31);
  if (m >= rows) return;
  const int64_t crow = g.c_map ? (int64_t)g.c_map[row0 + m] : (int64_t)(row0 + m);
  const float scale = (EPI == EPI_STORE && row_scale && !dense) ? row_scale[row0 + m] : 1.0f;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int n = n0 + n_w + 8 * q + 4 * (lane >> 5);
    if (n >= g.N) continue;
    const int64_t o = crow * g.ldc + n;
    f32x4_t v0, v1, v2;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      v0[r] = acc[0][4 * q + r];
      if constexpr (EPI == EPI_SWIGLU) {
        v1[r] = acc[NB - 1][4 * q + r];
        v2[r] = silu_f(v0[r]) * v1[r];
      } else {
        v2[r] = v0[r] * scale;
      }
    }
    f_put4(C + o, v2, g.N - n, vec);
    if constexpr (EPI == EPI_SWIGLU) {
      if (Gs) f_put4(Gs + o, v0, g.N - n, vec);
      if (Us) f_put4(Us + o, v1, g.N - n, vec);
    }
  }
}

// ------------------------------------------------------------------ backward
// MAP: A's K-major rows come through a_map, scaled by a_kscale (one chunk of a slab
// per thread: its row index and scale are loaded one slab ahead).
template <int EPI, bool VEC, bool MAP>
__global__ __launch_bounds__(256) void xgemm_f32_kernel(const XGemm g) {
  constexpr bool AK = EPI == XE_WGRAD;    // both operands K-major; else A rows, B weights N-contiguous
  constexpr int FK = AK ? F_FK_WGRAD : F_FK_ROWS;
  using TA = FTile<FK, AK>;
  using TB = FTile<FK, true>;
  extern __shared__ __attribute__((aligned(16))) float fsm[];
  int grp, row0, rows, n_tile, kbeg, kend, split;
  if (!xtile<FB, FB>(g, grp, row0, rows, n_tile, kbeg, kend, split)) return;
  const int n0 = n_tile * FB;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int m_w = (wave >> 1) * 32, n_w = (wave & 1) * 32;
  const float* A = static_cast<const float*>(g.A);

  const float* arow[TA::N];   // row form: the thread's rows
  if constexpr (!AK) {
#pragma unroll
    for (int i = 0; i < TA::N; ++i) {
      const int r = row0 + min(TA::row(tid, i), rows - 1);
      arow[i] = A + (g.a_map ? (int64_t)g.a_map[r] : (int64_t)r) * g.lda;
    }
  }
  const void* const* tab = AK ? nullptr : g.Btab + (int64_t)grp * g.nseg;
  f32x4_t ra[TA::N], rb[TB::N];
  int map_row = 0;
  float map_scale = 1.0f;
  const auto map_next = [&](int k0) {
    if constexpr (MAP) {
      static_assert(!MAP || TA::N == 1, "one row of a slab per thread");
      const int kc = min(k0 + TA::row(tid, 0), kend - 1);
      map_row = g.a_map[kc];
      map_scale = g.a_kscale ? g.a_kscale[kc] : 1.0f;
    }
  };
  const auto load = [&](int k0) {
    const bool whole = VEC && k0 + FK <= kend && (AK || g.kseg % FK == 0);   // no masks, one segment
    if constexpr (AK) {
      const float* ab = A + (int64_t)grp * g.a_col;
      const float* bb = static_cast<const float*>(g.Bact) + (int64_t)grp * g.b_col;
      const int ac = row0 + TA::col(tid), bc = n0 + TB::col(tid);
      if (whole) {
#pragma unroll
        for (int i = 0; i < TA::N; ++i)
          ra[i] = f_row4<VEC, false>(ab + (MAP ? (int64_t)map_row : (int64_t)(k0 + TA::row(tid, i))) * g.lda, ac, g.M);
#pragma unroll
        for (int i = 0; i < TB::N; ++i)
          rb[i] = f_row4<VEC, false>(bb + (int64_t)(k0 + TB::row(tid, i)) * g.ldb, bc, g.N);
        if constexpr (MAP) ra[0] *= map_scale;
      } else {
#pragma unroll
        for (int i = 0; i < TA::N; ++i) {
          const int k = k0 + TA::row(tid, i);
          ra[i] = f_row4<VEC, false>(ab + (MAP ? (int64_t)map_row : (int64_t)min(k, kend - 1)) * g.lda, ac, g.M);
          if constexpr (MAP) ra[i] *= map_scale;
          if (k >= kend) ra[i] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
        }
#pragma unroll
        for (int i = 0; i < TB::N; ++i) {
          const int k = k0 + TB::row(tid, i);
          rb[i] = f_row4<VEC, false>(bb + (int64_t)min(k, kend - 1) * g.ldb, bc, g.N);
          if (k >= kend) rb[i] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
        }
      }
    } else if (whole) {
      const int seg = k0 / g.kseg;
      const float* base = static_cast<const float*>(tab[seg]) + (int64_t)(k0 - seg * g.kseg) * g.ldb;
#pragma unroll
      for (int i = 0; i < TA::N; ++i) ra[i] = ldg_f4(arow[i] + k0 + TA::col(tid));
#pragma unroll
      for (int i = 0; i < TB::N; ++i)
        rb[i] = f_row4<VEC, false>(base + (int64_t)TB::row(tid, i) * g.ldb, n0 + TB::col(tid), g.N);
    } else {
#pragma unroll
      for (int i = 0; i < TA::N; ++i) ra[i] = f_row4<VEC, true>(arow[i], k0 + TA::col(tid), kend);
#pragma unroll
      for (int i = 0; i < TB::N; ++i) {
        const int k = k0 + TB::row(tid, i), kc = min(k, kend - 1), seg = kc / g.kseg;
        rb[i] = f_row4<VEC, false>(static_cast<const float*>(tab[seg]) + (int64_t)(kc - seg * g.kseg) * g.ldb,
                                   n0 + TB::col(tid), g.N);
        if (k >= kend) rb[i] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
      }
    }
  };
  const auto put = [&](float* s) {
    TA::put(s, tid, ra);
    TB::put(s + TA::FLOATS, tid, rb);
  };

  f32x16_t acc[1] = {};
  const int nk = (int)cdiv(max(kend - kbeg, 0), FK);
  if (nk > 0) {
    map_next(kbeg);
    load(kbeg);
    map_next(kbeg + FK);
  }
  for (int kb = 0; kb < nk; ++kb) {
    put(fsm);
    __syncthreads();
    if (kb + 1 < nk) {
      load(kbeg + (kb + 1) * FK);
      map_next(kbeg + (kb + 2) * FK);
    }
    f_slab<FK, 1, AK, true>(fsm, fsm + TA::FLOATS, m_w, n_w, lane, acc);
    __syncthreads();
  }

  const int m = m_w + (lane & 31);
  if (m >= rows) return;
  const int r = row0 + m;
  float* C;          // the row's first element
  int64_t ogu = 0;
  float w = 1.0f;
  if constexpr (EPI == XE_WGRAD) {
    if (g.ksplit > 1)
      C = g.part + (((int64_t)split * g.groups + grp) * g.M + r) * g.N;
    else
      C = r < g.msplit ? static_cast<float*>(g.Ctab0[grp]) + (int64_t)r * g.ldc
                       : static_cast<float*>(g.Ctab1[grp]) + (int64_t)(r - g.msplit) * g.ldc;
  } else {
    C = static_cast<float*>(g.C) + (g.c_map ? (int64_t)g.c_map[r] : (int64_t)r) * g.ldc + (int64_t)grp * g.c_group_col;
    if constexpr (EPI == XE_SWIGLU_BWD) {
      ogu = (int64_t)r * g.ld_gu + (int64_t)grp * g.gu_group_col;
      w = g.row_w ? g.row_w[r] : 1.0f;
    }
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int n = n0 + n_w + 8 * q + 4 * (lane >> 5);
    if (n >= g.N) continue;
    f32x4_t v, u;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = acc[0][4 * q + e];
    if constexpr (EPI == XE_SWIGLU_BWD) {
      // h = silu(gv) * uv, dh = w * acc
      const f32x4_t gv = f_row4<VEC, false>(static_cast<const float*>(g.Gs) + ogu, n, g.N);
      const f32x4_t uv = f_row4<VEC, false>(static_cast<const float*>(g.Us) + ogu, n, g.N);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float dh = w * v[e], sg = sigmoid_f(gv[e]);
        v[e] = dh * uv[e] * sg * (1.0f + gv[e] * (1.0f - sg));
        u[e] = dh * gv[e] * sg;
      }
      f_put4(C + g.du_off + n, u, g.N - n, VEC);
    }
    f_put4(C + n, v, g.N - n, VEC);
  }
}

// ------------------------------------------------------------------ launch
static bool al16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

template <auto Kern, class... Args>
static int f_launch(int64_t grid, size_t lds, hipStream_t st, const char* what, const Args&... args) {
  if (grid <= 0) return DSMOE_OK;
  hipLaunchKernelGGL(Kern, dim3((unsigned)grid), dim3(256), lds, st, args...);
  return check_launch(what);
}

// 16-byte loads of both operands: K and its segments, strides and the A base
// whole chunks (the caller vouches for the weight pointers).
static bool f_vec(const GemmDesc& g) {
  return ((g.K | g.kseg | g.lda | g.ldb) & 3) == 0 && al16(g.A);
}

// Workgroups of an XCD for one problem (bound).
static int64_t f_share(const GemmDesc& g) {
  const int64_t m = g.sched ? (int64_t)g.m_tiles_bound * (g.bm / FB) : cdiv(g.dense_rows, FB) * g.groups;
  return cdiv(m * cdiv(g.N, FB), 8);
}

int launch_gemm_f32(const GemmDesc& gr, const GemmDesc* gd, int epi, const float* row_scale, bool tables_aligned,
                    hipStream_t st) {
  if (gr.sched && gr.bm % FB != 0)
    return fail(DSMOE_ERR_INVALID, "gemm_f32: schedule height must be a multiple of 64");
  const bool vec = tables_aligned && f_vec(gr) && (!gd || f_vec(*gd));
  const int64_t grid = 8 * (f_share(gr) + (gd ? f_share(*gd) : 0));
  constexpr size_t tile = sizeof(float) * FTile<F_FK_ROWS, false>::FLOATS;
  static_assert(3 * tile <= 64 * 1024, "default LDS limit");
  const GemmDesc& d = gd ? *gd : gr;
  const int has = gd ? 1 : 0;
  if (epi == EPI_SWIGLU)
    return vec ? f_launch<&gemm_f32_kernel<EPI_SWIGLU, true>>(grid, 3 * tile, st, "gemm_f32", gr, d, has, row_scale)
               : f_launch<&gemm_f32_kernel<EPI_SWIGLU, false>>(grid, 3 * tile, st, "gemm_f32", gr, d, has, row_scale);
  return vec ? f_launch<&gemm_f32_kernel<EPI_STORE, true>>(grid, 2 * tile, st, "gemm_f32", gr, d, has, row_scale)
             : f_launch<&gemm_f32_kernel<EPI_STORE, false>>(grid, 2 * tile, st, "gemm_f32", gr, d, has, row_scale);
}

static bool f_xvec(const XGemm& g, int epi) {
  const int64_t mk = g.a_mode == XA_KMAJOR ? g.M | g.a_col : g.K;
  const int64_t b = g.b_mode == XB_ACT_KMAJOR ? g.b_col : 0;
  const int64_t c = epi == XE_WGRAD ? g.ldc : g.ldc | g.c_group_col;
  const int64_t s = epi == XE_SWIGLU_BWD ? g.ld_gu | g.gu_group_col | g.du_off : 0;
  return ((mk | b | c | s | g.lda | g.ldb | g.N) & 3) == 0 && al16(g.A) &&
         (g.b_mode != XB_ACT_KMAJOR || al16(g.Bact)) && (epi == XE_WGRAD || al16(g.C)) &&
         (epi != XE_SWIGLU_BWD || (al16(g.Gs) && al16(g.Us)));
}

template <int EPI, bool MAP = false>
static int f_bwd(const XGemm& g, bool vec, hipStream_t st) {
  constexpr bool AK = EPI == XE_WGRAD;
  constexpr int FK = AK ? F_FK_WGRAD : F_FK_ROWS;
  constexpr size_t lds = sizeof(float) * (FTile<FK, AK>::FLOATS + FTile<FK, true>::FLOATS);
  static_assert(lds <= 64 * 1024, "default LDS limit");
  int64_t m;
  if (g.sched_mode == XS_ROUTED)
    m = (int64_t)g.m_tiles_bound * (g.bm / FB);
  else
    m = cdiv(g.sched_mode == XS_DENSE ? g.dense_rows : g.M, FB) * g.groups * std::max(g.ksplit, 1);
  const int64_t grid = 8 * cdiv(m * cdiv(g.N, FB), 8);
  return vec ? f_launch<&xgemm_f32_kernel<EPI, true, MAP>>(grid, lds, st, "xgemm_f32", g)
             : f_launch<&xgemm_f32_kernel<EPI, false, MAP>>(grid, lds, st, "xgemm_f32", g);
}

int launch_xgemm_f32(const XGemm& g_in, int epi, bool tables_aligned, hipStream_t st) {
  XGemm g = g_in;
  if (g.sched_mode == XS_ROUTED && g.bm % FB != 0)
    return fail(DSMOE_ERR_INVALID, "xgemm_f32: schedule height must be a multiple of 64");
  const bool wgrad = epi == XE_WGRAD;
  if (wgrad != (g.a_mode == XA_KMAJOR) || wgrad != (g.b_mode == XB_ACT_KMAJOR) || g.b_mode == XB_W_NT || g.b_map ||
      (wgrad && g.a_kscale && !g.a_map))
    return fail(DSMOE_ERR_INVALID, "xgemm_f32: operand layout");
  const bool vec = tables_aligned && f_xvec(g, epi);
  if (!wgrad || !vec) g.ksplit = 1;   // the reduction reads and writes 16-byte vectors
  if (epi == XE_STORE) return f_bwd<XE_STORE>(g, vec, st);
  if (epi == XE_SWIGLU_BWD) return f_bwd<XE_SWIGLU_BWD>(g, vec, st);
  const int rc = g.a_map ? f_bwd<XE_WGRAD, true>(g, vec, st) : f_bwd<XE_WGRAD>(g, vec, st);
  if (rc || g.ksplit <= 1) return rc;
  g.c_f32 = 1;
  return launch_wgrad_reduce(g, st);
}

// Two workgroups or more for each CU, parts of 128 rows or more.
int xgemm_f32_ksplit(int64_t M, int64_t N, int groups, int64_t k_len) {
  const int64_t tiles = cdiv(M, FB) * cdiv(N, FB) * groups;
  int ks = 1;
  while (ks < 8 && tiles * ks < 512 && k_len >= 256 * ks) ks *= 2;
  return ks;
}

}  // namespace dsmoe
