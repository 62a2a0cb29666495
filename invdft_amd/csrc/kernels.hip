// Device kernels of the MI355X inverse-DFT hot path (gfx950 / CDNA4).
//
// Layouts
//   multivectors  node-major X[node * B + col]
//   quad data     [cell][q], q = (qz*Q + qy)*Q + qx
//   H tiles       H_e is symmetric, so per cell only the 16x16 tiles (rt, kg)
//                 with rt <= kg of the NEP x NEP matrix (NEP = ne rounded up
//                 to 16) are stored, row-major over the upper triangle
//                 (tile_index), each as [lane][s] so that lane l of a wave
//                 holds the A operand of v_mfma_*_16x16x4 for four
//                 consecutive k-steps: H[rt*16 + l%16][kg*16 + s*4 + l/16].
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <mutex>
#include <type_traits>

#include "common.h"
#include "sf_tables.h"

namespace idft {

namespace {

constexpr int kThreads = 256;

// Total of one value per thread over a work-group of NT threads (fixed
// order: each wave by shuffles, then the NT / 64 wave sums in order), returned
// to every thread.  red holds NT / 64 doubles; a caller that reuses red for a
// second total synchronises in between.
template <int NT>
__device__ inline double block_total(double t, double* red) {
  const int tid = threadIdx.x;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) t += __shfl_xor(t, o, 64);
  if ((tid & 63) == 0) red[tid >> 6] = t;
  __syncthreads();
  double s = 0.0;
#pragma unroll
  for (int w = 0; w < NT / 64; ++w) s += red[w];
  return s;
}

// Sum of partial[b * B + j] over b < nblk by one work-group of NT threads
// (fixed order: strided per-thread sums, then block_total).
template <int NT = kThreads>
__device__ inline double block_sum_col(const double* __restrict__ partial, int nblk, int B, int j,
                                       double* red) {
  const int tid = threadIdx.x;
  double s = 0.0;
  for (int b = tid; b < nblk; b += NT) s += partial[(int64_t)b * B + j];
  return block_total<NT>(s, red);
}

// Sum of n contiguous values by one work-group of NT threads (all threads
// call it).
template <int NT = kThreads>
__device__ inline double block_sum_contig(const double* __restrict__ v, int n, double* red) {
  const int tid = threadIdx.x;
  // four independent partial sums, so that four loads are in flight
  double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
  int b = tid;
  for (; b + 3 * NT < n; b += 4 * NT) {
    s0 += v[b];
    s1 += v[b + NT];
    s2 += v[b + 2 * NT];
    s3 += v[b + 3 * NT];
  }
  for (; b < n; b += NT) s0 += v[b];
  return block_total<NT>((s0 + s1) + (s2 + s3), red);
}

// Sums over k < per of red[k B + c] into red[c] for every c < B, by the
// threads tid = k B + c (off = tid / B, tid < per B): a tree of ceil(log2 per)
// steps in a fixed order, all threads call it.
__device__ inline void tree_cols(double* red, int per, int B, int tid, int off) {
  __syncthreads();
  for (int n = per; n > 1;) {
    const int h = (n + 1) / 2;
    if (off < n - h) red[tid] += red[tid + h * B];
    __syncthreads();
    n = h;
  }
}
// The same for NQ sums of VW columns per thread at once: thread tid = k nb + g holds
// q[n][v] of column g VW + v (threads past per nb hold nothing), and the sums over k < per
// arrive in red[n][g VW + v].  A tree: one thread per column adding `per` values in turn
// took half of the gather's time at 2 columns (per = 256).
template <int NQ, int VW>
__device__ inline void tree_groups(double (&red)[NQ][kThreads * VW], const double (&q)[NQ][VW],
                                   uint32_t per, uint32_t nb, uint32_t tid, uint32_t off) {
#pragma unroll
  for (int n = 0; n < NQ; ++n)
#pragma unroll
    for (int v = 0; v < VW; ++v) red[n][tid * VW + v] = q[n][v];
  for (uint32_t n = per; n > 1;) {
    __syncthreads();
    const uint32_t h = (n + 1) / 2;
    if (off < n - h)
#pragma unroll
      for (int k = 0; k < NQ; ++k)
#pragma unroll
        for (int v = 0; v < VW; ++v) red[k][tid * VW + v] += red[k][(tid + h * nb) * VW + v];
    n = h;
  }
  __syncthreads();
}

// The same sums in the order of the positions k = 0, 1, .. per - 1, all NQ VW nb <= 256
// of them at once: returns sum c (column c % (VW nb) of quantity c / (VW nb)) to the
// thread that asks for it.  For the dots of a MINRES step, whose order is fixed (see
// k_cell_line).
template <int NQ, int VW>
__device__ inline double ordered_groups(double (&red)[NQ][kThreads * VW],
                                        const double (&q)[NQ][VW], uint32_t per, uint32_t nb,
                                        uint32_t tid, uint32_t c) {
#pragma unroll
  for (int n = 0; n < NQ; ++n)
#pragma unroll
    for (int v = 0; v < VW; ++v) red[n][tid * VW + v] = q[n][v];
  __syncthreads();
  const uint32_t B = nb * VW;
  double t = 0.0;
  if (c < NQ * B) {
    const double* row = red[c / B] + c % B;
    for (uint32_t k = 0; k < per; ++k) t += row[k * B];
  }
  return t;
}

// Work-group size of the per-column reductions of long partial rows (cell
// dots, gather partials, Gram partials): 16 waves, about 12 values per thread
// for the 12-16 k values of a column.
constexpr int kRedThreads = 1024;

inline void check_u32(int64_t n) {
  if (n >= (int64_t)0xffffffffLL) throw Error(IDFT_EINVAL, "multivector too large for 32-bit indexing");
}

__host__ __device__ constexpr int ne_of(int p) { return (p + 1) * (p + 1) * (p + 1); }
__host__ __device__ constexpr int nep_of(int p) { return (ne_of(p) + 15) / 16 * 16; }
// stored tiles per cell and the position of tile (r, k), r <= k, among them
__host__ __device__ constexpr int ntiles_of(int p) { return (nep_of(p) / 16) * (nep_of(p) / 16 + 1) / 2; }
__host__ __device__ constexpr int tile_index(int rt_count, int r, int k) {
  return r * rt_count - r * (r - 1) / 2 + (k - r);
}

__device__ inline int64_t cell_node(const Geo& g, int64_t cx, int64_t cy, int64_t cz, int l) {
  const int a = l % g.n1, b = (l / g.n1) % g.n1, c = l / (g.n1 * g.n1);
  return ((cz * g.p + c) * g.N1 + (cy * g.p + b)) * (int64_t)g.N1 + (cx * g.p + a);
}

// Cell of colour `colour` handled by work-group w.  The 8 XCDs receive
// work-groups round-robin; each XCD is given a contiguous run of cells so its
// L2 sees spatially adjacent cells.
// The grid has 8 * ceil(nw / 8) work-groups, so (xcd, slot) covers every k.
__device__ inline int64_t colour_cell(const Geo& g, int colour, int64_t w, int64_t nw) {
  const int64_t per = (nw + 7) / 8;
  const int64_t xcd = w % 8, slot = w / 8;
  const int64_t k = xcd * per + slot;  // position inside the colour
  if (k >= nw) return -1;
  const int64_t hc = (g.nc + 1 - (colour & 1)) / 2;
  const int64_t hy = (g.nc + 1 - ((colour >> 1) & 1)) / 2;
  const int64_t kx = k % hc, ky = (k / hc) % hy, kz = k / (hc * hy);
  const int64_t cx = 2 * kx + (colour & 1), cy = 2 * ky + ((colour >> 1) & 1),
                cz = 2 * kz + ((colour >> 2) & 1);
  return (cz * g.nc + cy) * g.nc + cx;
}

inline unsigned colour_grid(int64_t nw) { return (unsigned)(8 * ((nw + 7) / 8)); }

inline int64_t colour_count(const Geo& g, int colour) {
  const int64_t hx = (g.nc + 1 - (colour & 1)) / 2;
  const int64_t hy = (g.nc + 1 - ((colour >> 1) & 1)) / 2;
  const int64_t hz = (g.nc + 1 - ((colour >> 2) & 1)) / 2;
  return hx * hy * hz;
}

// ------------------------------------------------------------ MFMA apply
typedef float v4f __attribute__((ext_vector_type(4)));
typedef double v4d __attribute__((ext_vector_type(4)));

template <typename T> struct Mfma;
// Output rows held by lane group lk (= lane / 16), item i, of the 16x16x4 MFMA:
// f32 keeps 4 consecutive rows per group, f64 interleaves them (measured on gfx950).
template <> struct Mfma<float> {
  typedef v4f acc_t;
  static __device__ inline int row(int lk, int i) { return 4 * lk + i; }
  static __device__ inline acc_t run(float a, float b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
};
template <> struct Mfma<double> {
  typedef v4d acc_t;
  static __device__ inline int row(int lk, int i) { return lk + 4 * i; }
  static __device__ inline acc_t run(double a, double b, acc_t c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
};

template <typename T> struct Vec4;
template <> struct Vec4<float> { typedef float4 type; };
template <> struct Vec4<double> { typedef double4 type; };

__host__ __device__ constexpr int ldb_of(int bt) { return (bt % 32 == 16) ? bt : bt + 16; }

// Stored tile of block row i, k-group k of H_e (Hc = the cell's stored
// tiles), one vector load per lane: tile (i, k) for k >= i, else its mirror
// (k, i), which the caller transposes (lds_transpose).
template <typename T, int RT>
__device__ inline typename Vec4<T>::type fetch_tile(const T* __restrict__ Hc, int i, int k,
                                                     int lane) {
  typedef typename Vec4<T>::type vec_t;
  const int t = k >= i ? tile_index(RT, i, k) : tile_index(RT, k, i);
  return reinterpret_cast<const vec_t*>(Hc)[t * 64 + lane];
}

// The transposed tile read straight from memory: lane l needs
// T[4s + l/16][l%16], which sits in lane (4s + l/16) + 16 (l%4), slot
// (l%16)/4 of the mirror tile (k, i) -- four scalar loads of the same 1 KiB
// (FP32) tile.  Used where the LDS square would cost occupancy.
template <typename T, int RT>
__device__ inline typename Vec4<T>::type fetch_tile_transposed(const T* __restrict__ Hc, int i,
                                                                int k, int lane) {
  typedef typename Vec4<T>::type vec_t;
  const T* t = Hc + tile_index(RT, k, i) * 256 + ((lane & 15) >> 2);
  const int lb = (lane >> 4) + 16 * (lane & 3);
  vec_t v;
  v.x = t[lb * 4];
  v.y = t[(lb + 4) * 4];
  v.z = t[(lb + 8) * 4];
  v.w = t[(lb + 12) * 4];
  return v;
}

// A operand of the transposed tile: lane l holds m = T[l%16][4s + l/16]
// (s = 0..3) and needs T[4s + l/16][l%16].  Through a per-wave 16 x 17
// (padded) LDS square: write row-major, read column-major.  LDS operations of
// one wave execute in order; the wavefront fences keep the compiler from
// moving the reads above the writes.
template <typename T>
__device__ inline typename Vec4<T>::type lds_transpose(typename Vec4<T>::type m, T* sq,
                                                        int lane) {
  typedef typename Vec4<T>::type vec_t;
  const int a = lane & 15, b = lane >> 4;
  sq[a * 17 + b] = m.x;
  sq[a * 17 + 4 + b] = m.y;
  sq[a * 17 + 8 + b] = m.z;
  sq[a * 17 + 12 + b] = m.w;
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  vec_t t;
  t.x = sq[b * 17 + a];
  t.y = sq[(4 + b) * 17 + a];
  t.z = sq[(8 + b) * 17 + a];
  t.w = sq[(12 + b) * 17 + a];
  return t;
}

// The cell's input tile in LDS: xs[l][j] = S[n] xn[n] X[n][c0 + j] xcol[c0 + j]
// (node n of local index l; rows l >= NE and columns j >= bw are zero).
template <typename T, typename TV, int P, int BT, int LDB, int NTH = kThreads>
__device__ inline void load_cell_input(const Geo& g, int64_t cx, int64_t cy, int64_t cz,
                                       const T* __restrict__ S, const TV* __restrict__ X,
                                       const double* __restrict__ xn,
                                       const double* __restrict__ xcol, int B, int c0, int bw,
                                       T* xs) {
  constexpr int NE = ne_of(P), NEP = nep_of(P), TOT = NEP * BT;
  // U entries per thread per round, all loads of a round issued before the
  // first product: the optional scales are loaded inside uniform branches
  // that hold nothing else, so no product is pulled in after its own load
  constexpr int U = 4;
  for (int i0 = threadIdx.x; i0 < TOT; i0 += NTH * U) {
    int64_t n[U];
    int col[U];
    bool ok[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = i0 + u * NTH;
      const int l = i / BT, j = i % BT;
      ok[u] = i < TOT && l < NE && j < bw;
      n[u] = ok[u] ? cell_node(g, cx, cy, cz, l) : 0;
      col[u] = ok[u] ? c0 + j : 0;
    }
    T sv[U];
    TV xv[U];
    double nv[U], cv[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      sv[u] = S[n[u]];
      xv[u] = X[n[u] * B + col[u]];
    }
    if (xn) {
#pragma unroll
      for (int u = 0; u < U; ++u) nv[u] = xn[n[u]];
    } else {
#pragma unroll
      for (int u = 0; u < U; ++u) nv[u] = 1.0;
    }
    if (xcol) {
#pragma unroll
      for (int u = 0; u < U; ++u) cv[u] = xcol[col[u]];
    } else {
#pragma unroll
      for (int u = 0; u < U; ++u) cv[u] = 1.0;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = i0 + u * NTH;
      if (i < TOT) {
        T v = T(0);
        if (ok[u]) {
          if constexpr (std::is_same<T, TV>::value) {
            v = sv[u] * xv[u] * (T)nv[u] * (T)cv[u];
          } else {  // wider input vectors: scale in FP64, round once
            v = (T)((double)sv[u] * (double)xv[u] * nv[u] * cv[u]);
          }
        }
        xs[(i / BT) * LDB + i % BT] = v;
      }
    }
  }
}

// Phase 1 of the cell operator.  One work-group handles `cpw` consecutive
// cells and the column tile [blockIdx.y * 16 NCT, +16 NCT) of the block.  Per
// cell the tile of (S X)_e is gathered into LDS and each wave computes whole
// 16-row blocks of H_e (S X)_e, streaming the tiles of its block row from
// HBM (upper-triangle tiles as stored, lower-triangle ones as LDS transposes
// of their mirror tiles, which the mirror's own row pass reads too, so the
// second read is mostly served by the caches), KPF k-groups in flight per
// wave.
// Output: Yc[e][l][j] = (H_e (S X)_e)[l][j].  Work-groups are dealt to the 8
// XCDs in contiguous runs of cells.
template <typename T, typename TV, int P, int NCT>
__global__ __launch_bounds__(kThreads) void k_cell_gemm(Geo g, const T* __restrict__ H,
                                                        const T* __restrict__ S,
                                                        const TV* __restrict__ X,
                                                        const double* __restrict__ xn,
                                                        const double* __restrict__ xcol,
                                                        T* __restrict__ Yc, int B, int cpw) {
  constexpr int NE = ne_of(P), NEP = nep_of(P), RT = NEP / 16, BT = NCT * 16;
  constexpr int NTILE = ntiles_of(P);
  constexpr int LDB = ldb_of(BT);
  // k-groups of H_e in flight per wave (deeper prefetch costs occupancy and
  // measured slower at p = 4, 5)
  constexpr int KPF = 3;
  // lower-triangle tiles through per-wave LDS transpose squares, unless
  // these would push the work-group past half the 160 KiB LDS (two
  // work-groups per CU), as for FP64 with 80-column tiles
  constexpr bool kLdsT = (NEP * LDB + 4 * 272) * (int)sizeof(T) <= 81920 ||
                         NEP * LDB * (int)sizeof(T) > 81920;
  __shared__ T xs[NEP * LDB];
  __shared__ T tsq[kLdsT ? 4 : 1][kLdsT ? 16 * 17 : 1];
  typedef typename Vec4<T>::type vec_t;
  // stored tile (transposed by the caller) or the transposed tile itself
  auto fetch = [](auto ldsT, const T* Hc, int i, int k, int lane) -> vec_t {
    if constexpr (decltype(ldsT)::value) return fetch_tile<T, RT>(Hc, i, k, lane);
    else return k >= i ? fetch_tile<T, RT>(Hc, i, k, lane)
                       : fetch_tile_transposed<T, RT>(Hc, i, k, lane);
  };
  const int64_t nwg = (g.ncell + cpw - 1) / cpw;
  const int64_t per = (nwg + 7) / 8;
  const int64_t wg = (blockIdx.x % 8) * per + blockIdx.x / 8;
  if (wg >= nwg) return;
  const int c0 = blockIdx.y * BT;
  const int bw = min(BT, B - c0);  // columns of this tile
  const int tid = threadIdx.x;
  const int wave = tid / 64, lane = tid % 64;
  const int lr = lane % 16, lk = lane / 16;
  typedef typename Mfma<T>::acc_t acc_t;
  const int64_t e0 = wg * cpw, e1 = min((int64_t)g.ncell, e0 + cpw);
  for (int64_t e = e0; e < e1; ++e) {
    const int64_t cx = e % g.nc, cy = (e / g.nc) % g.nc, cz = e / ((int64_t)g.nc * g.nc);
    if (e > e0) __syncthreads();  // previous cell's tiles fully consumed
    load_cell_input<T, TV, P, BT, LDB>(g, cx, cy, cz, S, X, xn, xcol, B, c0, bw, xs);
    __syncthreads();
    const T* Hc = H + (size_t)e * NTILE * 256;
    T* yc = Yc + (size_t)e * NE * B + c0;
    for (int rt = wave; rt < RT; rt += 4) {
      acc_t acc[NCT];
#pragma unroll
      for (int ct = 0; ct < NCT; ++ct) acc[ct] = acc_t{0, 0, 0, 0};
      vec_t buf[KPF];
#pragma unroll
      for (int kk = 0; kk < KPF; ++kk)
        buf[kk] = kk < RT ? fetch(std::integral_constant<bool, kLdsT>{}, Hc, rt, kk, lane) : vec_t{};
#pragma unroll 1
      for (int kg0 = 0; kg0 < RT; kg0 += KPF) {
#pragma unroll
        for (int kk = 0; kk < KPF; ++kk) {
          const int kg = kg0 + kk;
          if (kg < RT) {
            vec_t a = buf[kk];
            if (kg + KPF < RT) buf[kk] = fetch(std::integral_constant<bool, kLdsT>{}, Hc, rt, kg + KPF, lane);
            if constexpr (kLdsT) {
              if (kg < rt) a = lds_transpose<T>(a, tsq[wave], lane);
            }
            const T* xk = xs + (kg * 16 + lk) * LDB + lr;
            const T av[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
            for (int s = 0; s < 4; ++s) {
#pragma unroll
              for (int ct = 0; ct < NCT; ++ct)
                acc[ct] = Mfma<T>::run(av[s], xk[s * 4 * LDB + ct * 16], acc[ct]);
            }
          }
        }
      }
      // lane holds rows rt*16 + Mfma<T>::row(lk, i), column ct*16 + lr
#pragma unroll
      for (int ct = 0; ct < NCT; ++ct) {
        const int col = ct * 16 + lr;
        if (col >= bw) continue;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int r = rt * 16 + Mfma<T>::row(lk, i);
          if (r < NE) yc[(size_t)r * B + col] = acc[ct][i];
        }
      }
    }
  }
}

// Compile-time row / column of stored tile t (row-major upper triangle).
__host__ __device__ constexpr int tile_row(int rt_count, int t) {
  int r = 0;
  while (r + 1 < rt_count && tile_index(rt_count, r + 1, r + 1) <= t) ++r;
  return r;
}
__host__ __device__ constexpr int tile_col(int rt_count, int t) {
  return tile_row(rt_count, t) + (t - tile_index(rt_count, tile_row(rt_count, t),
                                                 tile_row(rt_count, t)));
}

template <int I>
using ic = std::integral_constant<int, I>;
template <int B0, int E0, typename F>
__device__ inline void static_for(F&& f) {
  if constexpr (B0 < E0) {
    f(ic<B0>{});
    static_for<B0 + 1, E0>(f);
  }
}

// Tiles of the stored upper triangle that touch block rows [r0, r1): the
// j-th (in storage order) of those with r or k in the range, and their count.
__host__ __device__ constexpr int half_tile_count(int rt_count, int r0, int r1) {
  int n = 0;
  for (int t = 0; t < rt_count * (rt_count + 1) / 2; ++t) {
    const int r = tile_row(rt_count, t), k = tile_col(rt_count, t);
    if ((r >= r0 && r < r1) || (k >= r0 && k < r1)) ++n;
  }
  return n;
}
__host__ __device__ constexpr int half_tile(int rt_count, int r0, int r1, int j) {
  for (int t = 0; t < rt_count * (rt_count + 1) / 2; ++t) {
    const int r = tile_row(rt_count, t), k = tile_col(rt_count, t);
    if ((r >= r0 && r < r1) || (k >= r0 && k < r1)) {
      if (j == 0) return t;
      --j;
    }
  }
  return -1;
}

constexpr int kSymmThreads = 512;

// Phase 1, tile pass (8 waves per work-group).  The block rows are split in
// two halves; waves 0-3 produce the rows of the first half, waves 4-7 those
// of the second.  A half's four waves split, in compile-time lists (every
// accumulator index static), the stored tiles (r, k) that touch the half:
// T (S X)_k is added to row r if r is in the half and, for r < k,
// T^T (S X)_r (LDS transpose) to row k if k is in the half.  A tile is read
// once per half it touches -- the two halves read the shared ones at the same
// time on the same CU, so the second read is a cache hit -- and each wave
// keeps partial sums of its half's rows only.  The four partials of each half
// are added in LDS in wave order (deterministic) and written to Yc.
template <typename T, typename TV, int P, int NCT>
__global__ __launch_bounds__(kSymmThreads) void k_cell_symm(Geo g, const T* __restrict__ H,
                                                            const T* __restrict__ S,
                                                            const TV* __restrict__ X,
                                                            const double* __restrict__ xn,
                                                            const double* __restrict__ xcol,
                                                            T* __restrict__ Yc, int B, int cpw) {
  constexpr int NE = ne_of(P), NEP = nep_of(P), RT = NEP / 16, BT = NCT * 16;
  constexpr int NTILE = ntiles_of(P);
  constexpr int LDB = ldb_of(BT);
  constexpr int KPF = 3;
  constexpr int RH = (RT + 1) / 2;  // block rows of the first half (and at most per half)
  __shared__ T xs[NEP * LDB];  // the input tile, then the partial-sum buffer
  __shared__ T tsq[8][16 * 17];
  typedef typename Vec4<T>::type vec_t;
  typedef typename Mfma<T>::acc_t acc_t;
  const int64_t nwg = (g.ncell + cpw - 1) / cpw;
  const int64_t per = (nwg + 7) / 8;
  const int64_t wg = (blockIdx.x % 8) * per + blockIdx.x / 8;
  if (wg >= nwg) return;
  const int c0 = blockIdx.y * BT;
  const int bw = min(BT, B - c0);
  const int tid = threadIdx.x;
  const int wave = tid / 64, lane = tid % 64;
  const int lr = lane % 16, lk = lane / 16;
  const int64_t e0 = wg * cpw, e1 = min((int64_t)g.ncell, e0 + cpw);
  for (int64_t e = e0; e < e1; ++e) {
    const int64_t cx = e % g.nc, cy = (e / g.nc) % g.nc, cz = e / ((int64_t)g.nc * g.nc);
    if (e > e0) __syncthreads();  // previous cell's output read from xs
    load_cell_input<T, TV, P, BT, LDB, kSymmThreads>(g, cx, cy, cz, S, X, xn, xcol, B, c0, bw,
                                                     xs);
    __syncthreads();
    const vec_t* Hc = reinterpret_cast<const vec_t*>(H + (size_t)e * NTILE * 256) + lane;
    acc_t acc[RH][NCT];
#pragma unroll
    for (int r = 0; r < RH; ++r)
#pragma unroll
      for (int ct = 0; ct < NCT; ++ct) acc[r][ct] = acc_t{0, 0, 0, 0};
    // tiles [J0, J1) of the list of half [R0, R1)
    auto run = [&](auto r0c, auto r1c, auto j0c, auto j1c) {
      constexpr int R0 = decltype(r0c)::value, R1 = decltype(r1c)::value;
      constexpr int J0 = decltype(j0c)::value, CNT = decltype(j1c)::value - J0;
      vec_t buf[KPF];
      static_for<0, (KPF < CNT ? KPF : CNT)>([&](auto jc) {
        constexpr int tp = half_tile(RT, R0, R1, J0 + decltype(jc)::value);
        buf[decltype(jc)::value] = Hc[tp * 64];
      });
      static_for<0, CNT>([&](auto jc) {
        constexpr int J = decltype(jc)::value, t = half_tile(RT, R0, R1, J0 + J);
        constexpr int r = tile_row(RT, t), k = tile_col(RT, t);
        const vec_t a = buf[J % KPF];
        if constexpr (J + KPF < CNT) {
          constexpr int tn = half_tile(RT, R0, R1, J0 + J + KPF);
          buf[J % KPF] = Hc[tn * 64];
        }
        if constexpr (r >= R0 && r < R1) {  // row r += T (S X)_k
          const T* xk = xs + (k * 16 + lk) * LDB + lr;
          const T av[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
          for (int s4 = 0; s4 < 4; ++s4)
#pragma unroll
            for (int ct = 0; ct < NCT; ++ct)
              acc[r - R0][ct] = Mfma<T>::run(av[s4], xk[s4 * 4 * LDB + ct * 16], acc[r - R0][ct]);
        }
        if constexpr (r < k && k >= R0 && k < R1) {  // row k += T^T (S X)_r
          const vec_t at = lds_transpose<T>(a, tsq[wave], lane);
          const T* xr = xs + (r * 16 + lk) * LDB + lr;
          const T av[4] = {at.x, at.y, at.z, at.w};
#pragma unroll
          for (int s4 = 0; s4 < 4; ++s4)
#pragma unroll
            for (int ct = 0; ct < NCT; ++ct)
              acc[k - R0][ct] = Mfma<T>::run(av[s4], xr[s4 * 4 * LDB + ct * 16], acc[k - R0][ct]);
        }
      });
    };
    constexpr int C0 = half_tile_count(RT, 0, RH), C1 = half_tile_count(RT, RH, RT);
    switch (wave) {
      case 0: run(ic<0>{}, ic<RH>{}, ic<0>{}, ic<C0 / 4>{}); break;
      case 1: run(ic<0>{}, ic<RH>{}, ic<C0 / 4>{}, ic<C0 / 2>{}); break;
      case 2: run(ic<0>{}, ic<RH>{}, ic<C0 / 2>{}, ic<(3 * C0) / 4>{}); break;
      case 3: run(ic<0>{}, ic<RH>{}, ic<(3 * C0) / 4>{}, ic<C0>{}); break;
      case 4: run(ic<RH>{}, ic<RT>{}, ic<0>{}, ic<C1 / 4>{}); break;
      case 5: run(ic<RH>{}, ic<RT>{}, ic<C1 / 4>{}, ic<C1 / 2>{}); break;
      case 6: run(ic<RH>{}, ic<RT>{}, ic<C1 / 2>{}, ic<(3 * C1) / 4>{}); break;
      default: run(ic<RH>{}, ic<RT>{}, ic<(3 * C1) / 4>{}, ic<C1>{}); break;
    }
    // partial sums of each half's four waves, added in wave order through xs
    // (the halves own disjoint rows, so they reduce side by side)
    const int r0 = wave < 4 ? 0 : RH, nr = wave < 4 ? RH : RT - RH;
    for (int w = 0; w < 4; ++w) {
      __syncthreads();
      if (wave % 4 == w) {
#pragma unroll
        for (int r = 0; r < RH; ++r) {
          if (r >= nr) break;
#pragma unroll
          for (int ct = 0; ct < NCT; ++ct)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              T* p = xs + ((r0 + r) * 16 + Mfma<T>::row(lk, i)) * LDB + ct * 16 + lr;
              *p = w == 0 ? acc[r][ct][i] : *p + acc[r][ct][i];
            }
        }
      }
    }
    __syncthreads();
    T* yc = Yc + (size_t)e * NE * B + c0;
    for (int i = tid; i < NE * BT; i += kSymmThreads) {
      const int l = i / BT, j = i % BT;
      if (j < bw) yc[(size_t)l * B + j] = xs[l * LDB + j];
    }
  }
}

// ----------------------------------------------- sum-factorised cell product
// Phase 1 without stored cell matrices.  On the uniform mesh
//   H_e = (h/4)(D(x)M(x)M + M(x)D(x)M + M(x)M(x)D) + L^T diag(w_e) L,  L = Lq(x)Lq(x)Lq,
// so H_e X_e is a chain of 1D contractions along x, y and z, each in the
// even-odd form below: 11.9 k FMA and 6.6 k adds per column at p = 5 (23 k FMA
// without the even-odd split, 47 k for the dense product), and per cell only
// the (p+3)^3 weights w_e are read from HBM instead of n_e(n_e+1)/2 entries of
// H_e.  The 1D tables are compile-time constants (SfC<P>): after unrolling
// every FP32 coefficient is an immediate operand, and the FP64 ones come from
// a constant-memory table (PlCoef below); h/4 scales the kinetic sum once.
//
// Layout.  A lane owns one (cell, column) slot and one of its Q = p + 3 Gauss
// planes along z; a wave holds NS = 64 / Q slots and works alone (no barriers).
// Along x and y everything happens in the lane's registers, so the tensor crosses
// LDS only where z mixes the planes:
//   1  z lines of the scaled input (from HBM): u[q] = Lq x, to LDS
//   2  the lane's plane u: m = (M (x) M) u and
//      p = (h/4) g_q (D (x) M + M (x) D) u + (Lq (x) Lq)^T diag(w) (Lq (x) Lq) u
//      with g_q the Gauss weight, since M = Lq^T diag(g) Lq along z
//   3  z lines back: y = Lq^T p + (h/4) E m, E Lq = D, to the cell scratch
// That is about 2000 LDS entries per cell and column at p = 5 where the same chain
// taken line by line (one work-group per cell and 4 columns, eight stages with a
// barrier each) moved 4850 and left a quarter of its lanes idle in most stages.
// Slots are numbered cell B + column over the whole mesh, so that a wave is full at
// every block width.
// It takes every FP32 product and the FP64 ones of the operator, the filter and the
// quadrature operator; the FP64 steps of MINRES keep the line-by-line kernel below.
// Bound by VALU issue: about 60 % of it in FP64, 80 % in FP32 (2 to 5 waves per
// SIMD; FP64 at p = 5 takes 246 registers).  Measured against the line-by-line
// kernel, us of the cell product alone: FP64 27 cells p = 3 B = 12 135 -> 96,
// 19 p = 4 B = 21 171 -> 111, 30 p = 4 B = 64 1383 -> 1139, 24 p = 5 B = 1 65 -> 26
// and B = 12 261 -> 233, 40 p = 2 B = 8 190 -> 73; FP32 87 -> 42, 93 -> 57,
// 921 -> 735, 39 -> 18, 154 -> 138 and 136 -> 34; 8 p = 3 B = 5, where one wave's
// latency is the time, 5.4 -> 5.3 and (FP32) 4.1 -> 4.6.
// The 1D tables as operators A (R x C): K = 0 Lq (Gauss points from nodes),
// 1 Lq^T, 2 M, 3 D, 4 E (D from the Gauss points, E Lq = D).  The GLL nodes and the Gauss points lie symmetrically
// about the cell centre, so each A is centro-symmetric,
// A[R-1-i][C-1-j] = A[i][j] (to rounding of the tables).
template <int P, int K>
struct SfTab {
  static constexpr int kP = P, kK = K;
  static constexpr int N1 = P + 1, Q = P + 3;
  static constexpr int R = K == 0 ? Q : N1;
  static constexpr int C = K == 1 || K == 4 ? Q : N1;
  __host__ __device__ static constexpr double at(int i, int j) {
    return K == 0   ? SfC<P>::v.L[i * N1 + j]
           : K == 1 ? SfC<P>::v.L[j * N1 + i]
           : K == 2 ? SfC<P>::v.M[i * N1 + j]
           : K == 3 ? SfC<P>::v.D[i * N1 + j]
                    : SfC<P>::v.E[i * Q + j];
  }
};
// Even-odd form of y = A x (Kopriva's even-odd decomposition).  With
// x+_j = x_j + x_{C-1-j} and x-_j = x_j - x_{C-1-j} for j < C/2 (the middle
// entry of an odd C kept alone as x+_{C/2}), row i < R/2 takes
//   e_i = sum_j (A_ij + A_i,C-1-j)/2 x+_j [+ A_i,mid x_mid]
//   o_i = sum_j (A_ij - A_i,C-1-j)/2 x-_j
// and y_i = e_i + o_i, y_{R-1-i} = e_i - o_i; the middle row of an odd R is
// e alone.  R C / 2 multiply-adds instead of R C.  The coefficients are
// constant expressions, so each is an immediate operand after unrolling.
template <typename T, class A, int I, int J>
__device__ constexpr T eo_even() {
  constexpr double c = 0.5 * (A::at(I, J) + A::at(I, A::C - 1 - J));
  return (T)c;
}
template <typename T, class A, int I, int J>
__device__ constexpr T eo_odd() {
  constexpr double c = 0.5 * (A::at(I, J) - A::at(I, A::C - 1 - J));
  return (T)c;
}
template <typename T, class A, int I>
__device__ constexpr T eo_mid() {
  constexpr double c = A::at(I, A::C / 2);
  return (T)c;
}
// FP64 coefficients from constant memory.  A double has no literal operand,
// so an immediate FP64 coefficient costs two scalar moves per use; the FP64
// kernels instead read the even-odd coefficients of all four operators from
// one table in constant memory, which the compiler fetches with wide scalar
// loads (4 doubles per load).  Per operator K (R x C) and row I < ceil(R/2):
// the floor(C/2) even coefficients, the floor(C/2) odd ones, then the middle
// one if C is odd.
template <int P>
struct EoTable {
  static constexpr int R(int k) { return k == 0 ? P + 3 : P + 1; }
  static constexpr int C(int k) { return k == 1 || k == 4 ? P + 3 : P + 1; }
  static constexpr int stride(int k) { return 2 * (C(k) / 2) + C(k) % 2; }
  static constexpr int base(int k) {
    int b = 0;
    for (int j = 0; j < k; ++j) b += ((R(j) + 1) / 2) * stride(j);
    return b;
  }
  static constexpr int kWeights = base(5);  // then the p + 3 Gauss weights
  static constexpr int kSize = kWeights + P + 3;
  double v[kSize];
};
template <int P>
constexpr EoTable<P> make_eo_table() {
  EoTable<P> t{};
  for (int q = 0; q < P + 3; ++q) t.v[EoTable<P>::kWeights + q] = SfC<P>::v.w[q];
  for (int k = 0; k < 5; ++k) {
    const int r = EoTable<P>::R(k), c = EoTable<P>::C(k), st = EoTable<P>::stride(k);
    for (int i = 0; i < (r + 1) / 2; ++i) {
      double* row = t.v + EoTable<P>::base(k) + i * st;
      auto at = [&](int ii, int jj) {
        return k == 0   ? SfC<P>::v.L[ii * (P + 1) + jj]
               : k == 1 ? SfC<P>::v.L[jj * (P + 1) + ii]
               : k == 2 ? SfC<P>::v.M[ii * (P + 1) + jj]
               : k == 3 ? SfC<P>::v.D[ii * (P + 1) + jj]
                        : SfC<P>::v.E[ii * (P + 3) + jj];
      };
      for (int j = 0; j < c / 2; ++j) {
        row[j] = 0.5 * (at(i, j) + at(i, c - 1 - j));
        row[c / 2 + j] = 0.5 * (at(i, j) - at(i, c - 1 - j));
      }
      if (c % 2) row[2 * (c / 2)] = at(i, c / 2);
    }
  }
  return t;
}
// Written from the host once per device (upload_sf_constants): with an
// initialiser the compiler would fold the values back into immediates.  The
// kernels take the table's device address as an argument (sf_eo_table): an
// access through the symbol itself goes through the global offset table, one
// more dependent scalar load wherever the compiler reloads the coefficients.
__constant__ EoTable<2> kEo2;
__constant__ EoTable<3> kEo3;
__constant__ EoTable<4> kEo4;
__constant__ EoTable<5> kEo5;
// Unsigned 32-bit division by a run-time constant d >= 2 through a
// multiplier computed on the host (Granlund-Montgomery): with
// s = ceil(log2 d) and m = floor(2^32 (2^s - d) / d) + 1,
// n / d = (t + ((n - t) >> 1)) >> (s - 1), t = mulhi(n, m), for every n.
struct FastDiv {
  uint32_t m, s;
};
inline FastDiv make_fastdiv(uint32_t d) {
  uint32_t s = 0;
  while ((uint64_t(1) << s) < d) ++s;
  const uint64_t m = ((uint64_t(1) << 32) * ((uint64_t(1) << s) - d)) / d + 1;
  return FastDiv{(uint32_t)m, s};
}
__device__ inline uint32_t fast_div(uint32_t n, FastDiv f) {
  const uint32_t t = __umulhi(n, f.m);
  return (t + ((n - t) >> 1)) >> (f.s - 1);
}

// x+ and x- of a line (see the even-odd form above).
template <int C, typename T>
__device__ inline void pl_split(const T (&x)[C], T (&p)[(C + 1) / 2], T (&m)[C / 2]) {
#pragma unroll
  for (int j = 0; j < C / 2; ++j) {
    p[j] = x[j] + x[C - 1 - j];
    m[j] = x[j] - x[C - 1 - j];
  }
  if constexpr (C % 2 == 1) p[C / 2] = x[C / 2];
}
// The even-odd coefficients of operator A for one phase: immediates in FP32; in
// FP64 one block of scalar registers, loaded together at the phase's start and
// kept (the empty asm stops the compiler from loading a coefficient again at each
// use: at 2 waves per SIMD nothing hides those waits).
template <typename T, class A>
struct PlCoef {
  typedef EoTable<A::kP> E;
  static constexpr bool kTab = sizeof(T) == 8;
  static constexpr int kMid = A::C % 2 == 1 ? A::C / 2 : -1;  // the middle column
  static constexpr int kN = ((A::R + 1) / 2) * E::stride(A::kK);
  T c[kTab ? kN : 1];
  // after: a value of the phase before.  The offset, a 0 that the compiler does not
  // see, is tied to it, so that the loads stay behind it: two phases' coefficients
  // do not fit the scalar registers.
  __device__ inline PlCoef(const double* __restrict__ eo, T after) {
    if constexpr (kTab) {
      int zero = 0;
      asm("" : "+s"(zero) : "v"(after));
      static_for<0, kN>([&](auto i) { c[decltype(i)::value] = eo[zero + E::base(A::kK) + decltype(i)::value]; });
      if constexpr (A::kK != 4)
        static_for<0, kN>([&](auto i) { asm("" : "+s"(c[decltype(i)::value])); });
    }
  }
  // coefficient W (0 even, 1 odd, 2 middle) of row I, column J
  template <int I, int J, int W>
  __device__ inline T at() const {
    if constexpr (kTab) {
      constexpr int cc = A::C;
      return c[I * E::stride(A::kK) + (W == 0 ? J : W == 1 ? cc / 2 + J : 2 * (cc / 2))];
    } else if constexpr (W == 0) {
      return eo_even<T, A, I, J>();
    } else if constexpr (W == 1) {
      return eo_odd<T, A, I, J>();
    } else {
      return eo_mid<T, A, I>();
    }
  }
};
// The same coefficients read as the transposed operator's (Lq^T from Lq, equal by
// centro-symmetry).
template <class CF, int C>
struct PlTransposed {
  const CF& f;
  template <int I, int J, int W>
  __device__ inline auto at() const {
    constexpr int row = W == 2 ? C / 2 : J;
    if constexpr (CF::kMid == I) return f.template at<row, 0, 2>();
    else return f.template at<row, I, W == 1 ? 1 : 0>();
  }
};
// The even (i < ceil(R/2)) and odd (i < floor(R/2)) halves of A x from x's split:
// y_i = e_i + o_i, y_{R-1-i} = e_i - o_i, the middle row of an odd R is e alone.
// ADD: added to what e and o hold.
template <class A, bool ADD, typename T, class CF>
__device__ inline void pl_halves(const CF& cf, const T (&p)[(A::C + 1) / 2],
                                 const T (&m)[A::C / 2], T (&e)[(A::R + 1) / 2],
                                 T (&o)[A::R / 2]) {
  static_for<0, (A::R + 1) / 2>([&](auto i) {
    constexpr int I = decltype(i)::value;
    T ei = ADD ? e[I] : T(0), oi = T(0);
    if constexpr (ADD && I < A::R / 2) oi = o[I];
    static_for<0, A::C / 2>([&](auto j) {
      constexpr int J = decltype(j)::value;
      if (!ADD && J == 0) ei = cf.template at<I, J, 0>() * p[J];
      else ei += cf.template at<I, J, 0>() * p[J];
      if constexpr (I < A::R / 2) {
        if (!ADD && J == 0) oi = cf.template at<I, J, 1>() * m[J];
        else oi += cf.template at<I, J, 1>() * m[J];
      }
    });
    if constexpr (A::C % 2 == 1) ei += cf.template at<I, 0, 2>() * p[A::C / 2];
    e[I] = ei;
    if constexpr (I < A::R / 2) o[I] = oi;
  });
}
template <int R, typename T>
__device__ inline void pl_join(const T (&e)[(R + 1) / 2], const T (&o)[R / 2], T (&y)[R]) {
#pragma unroll
  for (int i = 0; i < R / 2; ++i) {
    y[i] = e[i] + o[i];
    y[R - 1 - i] = e[i] - o[i];
  }
  if constexpr (R % 2 == 1) y[R / 2] = e[R / 2];
}
// LDS accesses of one wave complete in order: between phases only the compiler
// has to be kept from moving them.
__device__ inline void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
  __builtin_amdgcn_wave_barrier();
}

// Lanes of a wave: NS (cell, column) slots x Q Gauss planes.
template <int P>
struct PlaneLanes {
  static constexpr int Q = P + 3, NS = 64 / Q;
};
// Plane stride in LDS: N1^2 lines of NS entries, padded so that plane r of slot s
// starts r NS + s banks on, as in the line phases.
template <typename T, int P>
struct PlaneStride {
  static constexpr int NS = PlaneLanes<P>::NS, L = (P + 1) * (P + 1) * NS;
  static constexpr int M = 256 / (int)sizeof(T);
  static constexpr int v = L + ((NS - L) % M + M) % M;
};
// The node scale of the input: S, or with a further node scale the product in FP64.
template <typename T, bool XN>
struct PlaneScale {
  typedef typename std::conditional<XN, double, T>::type type;
};
// KIN = false: the potential chain alone on the unscaled input (S unused):
// Yc = Lq^T diag(w_e) Lq X_e, the quadrature operator of a weight.  wstride: the
// weights' step from cell to cell (0: the same weights in every cell); ldx: the row
// length of X (B, or more for a block of columns).  XN: node-scaled input, and with
// dotp also each slot's x.(H_e x), dotp[column * ncell + cell] (FP32 products alone).
template <typename T, typename TV, int P, bool XN, bool KIN>
__global__ __launch_bounds__(64, 2) void k_cell_plane(
    Geo g, T hq, const T* __restrict__ W, uint32_t wstride,
    const typename PlaneScale<T, XN>::type* __restrict__ S, const TV* __restrict__ X, uint32_t ldx,
    const double* __restrict__ xcol, T* __restrict__ Yc, uint32_t B, FastDiv divB, uint32_t nslot,
    double* __restrict__ dotp, const double* __restrict__ eo) {
  typedef typename PlaneScale<T, XN>::type SN;
  constexpr int N1 = P + 1, Q = P + 3, N2 = N1 * N1, NE = N2 * N1, Q2 = Q * Q;
  constexpr int NS = PlaneLanes<P>::NS, PS = PlaneStride<T, P>::v;
  constexpr int K3 = (N2 + Q - 1) / Q;  // lines per lane in the line phases
  constexpr int HE = (N1 + 1) / 2, HO = N1 / 2, QE = (Q + 1) / 2, QO = Q / 2;
  typedef SfTab<P, 0> TL;
  typedef SfTab<P, 1> TLt;
  typedef SfTab<P, 2> TM;
  typedef SfTab<P, 3> TD;
  typedef SfTab<P, 4> TE;
  __shared__ __align__(16) T lds[Q * PS];
  const uint32_t lane = threadIdx.x;
  if (lane >= NS * Q) return;
  const uint32_t r = lane / NS, slot = lane % NS;
  const uint32_t nwave = (nslot + NS - 1) / NS, per = (nwave + 7) / 8;
  const uint32_t kw = (blockIdx.x % 8) * per + blockIdx.x / 8;
  if (kw >= nwave) return;
  const bool live = kw * NS + slot < nslot;
  const uint32_t sid = live ? kw * NS + slot : nslot - 1;
  const uint32_t nc = (uint32_t)g.nc, NN = (uint32_t)g.N1, NNN = NN * NN;
  const auto cell_of = [&](uint32_t s) { return B == 1 ? s : fast_div(s, divB); };
  const auto first_node = [&](uint32_t c) {
    const uint32_t cx = c % nc, cyz = c / nc, cy = cyz % nc, cz = cyz / nc;
    return (cz * P * NN + cy * P) * NN + cx * P;
  };
  const uint32_t e = cell_of(sid), j = sid - e * B, n00 = first_node(e);
  const T* we = W + (size_t)e * wstride + r * Q2;
  const double xc = xcol ? xcol[j] : 1.0;
  const T wg = KIN ? (T)eo[EoTable<P>::kWeights + r] : T(0);
  // the input of line l of this lane, scaled
  // (pointers stepped by uniform strides: a 64-bit product per entry would cost as
  // much as the entry's arithmetic)
  const size_t zx = (size_t)NNN * ldx;
  const auto load_line = [&](uint32_t l, uint32_t n0, uint32_t jj, T(&v)[N1]) {
    const uint32_t n = n0 + (l / N1) * NN + l % N1;
    const TV* Xp = X + (size_t)n * ldx + jj;
    const SN* Sp = KIN ? S + n : nullptr;
    SN sv[N1];
    TV xv[N1];
#pragma unroll
    for (int c = 0; c < N1; ++c) {
      xv[c] = Xp[c * zx];
      if constexpr (KIN) sv[c] = Sp[(size_t)c * NNN];
    }
#pragma unroll
    for (int c = 0; c < N1; ++c) {
      if constexpr (!KIN) v[c] = (T)xv[c];
      else if constexpr (std::is_same<T, TV>::value) v[c] = sv[c] * xv[c] * (T)xc;
      else v[c] = (T)((double)sv[c] * (double)xv[c] * xc);  // scaled in FP64, rounded once
    }
  };
  // line index of round k (rounds past the last line repeat it)
  const auto line_of = [&](uint32_t rr, int k) -> uint32_t {
    const uint32_t l = rr + Q * k;
    return l < (uint32_t)N2 ? l : (uint32_t)N2 - 1;
  };
  // z lines: u[q] = Lq x for the Q planes
  T after = T(0);
  const PlCoef<T, TL> fL0(eo, T(0));
#pragma unroll
  for (int k = 0; k < K3; ++k) {
    const uint32_t l = line_of(r, k);
    T v[N1], vp[HE], vm[HO], oe[QE], oo[QO], u[Q];
    load_line(l, n00, j, v);
    pl_split<N1>(v, vp, vm);
    pl_halves<TL, false>(fL0, vp, vm, oe, oo);
    pl_join<Q>(oe, oo, u);
#pragma unroll
    for (int q = 0; q < Q; ++q) lds[q * PS + l * NS + slot] = u[q];
    after = u[0];
  }
  wave_lds_fence();
  // this lane's plane: entries (b, a) at pl[(b N1 + a) NS]
  T* const pl = lds + r * PS + slot;
  T me[N1][HE], mo[N1][HO];  // m = M (x) M u, even and odd in x
  T pe[N1][HE], po[N1][HO];  // the plane operator's result
  const auto u_line = [&](const T* pu, int b, T(&p)[HE], T(&m)[HO]) {
    T v[N1];
#pragma unroll
    for (int a = 0; a < N1; ++a) v[a] = pu[(a * N1 + b) * NS];
    pl_split<N1>(v, p, m);
  };
  if constexpr (KIN) {
    const PlCoef<T, TM> fM(eo, after);
    const PlCoef<T, TD> fD(eo, after);
    const T wk = hq * wg;
#pragma unroll
    for (int b = 0; b < N1; ++b) {
      T p[HE], m[HO];
      u_line(pl, b, p, m);
      pl_halves<TM, false>(fM, p, m, me[b], mo[b]);
      pl_halves<TD, false>(fD, p, m, pe[b], po[b]);
    }
    // y columns of M x (ca) and D x (cb), in place: m = M ca, k2 = D ca + M cb
    const auto kin_column = [&](auto ca, auto cb) {
      T a[N1], d[N1], ap[HE], am[HO], dp[HE], dm[HO], oe[HE], oo[HO], y[N1];
#pragma unroll
      for (int b = 0; b < N1; ++b) { a[b] = ca(b); d[b] = cb(b); }
      pl_split<N1>(a, ap, am);
      pl_split<N1>(d, dp, dm);
      pl_halves<TM, false>(fM, ap, am, oe, oo);
      pl_join<N1>(oe, oo, y);
#pragma unroll
      for (int b = 0; b < N1; ++b) ca(b) = y[b];
      pl_halves<TD, false>(fD, ap, am, oe, oo);
      pl_halves<TM, true>(fM, dp, dm, oe, oo);
      pl_join<N1>(oe, oo, y);
#pragma unroll
      for (int b = 0; b < N1; ++b) cb(b) = wk * y[b];
    };
#pragma unroll
    for (int i = 0; i < HE; ++i)
      kin_column([&](int b) -> T& { return me[b][i]; }, [&](int b) -> T& { return pe[b][i]; });
#pragma unroll
    for (int i = 0; i < HO; ++i)
      kin_column([&](int b) -> T& { return mo[b][i]; }, [&](int b) -> T& { return po[b][i]; });
  } else {
#pragma unroll
    for (int b = 0; b < N1; ++b) {
#pragma unroll
      for (int i = 0; i < HE; ++i) pe[b][i] = T(0);
#pragma unroll
      for (int i = 0; i < HO; ++i) po[b][i] = T(0);
    }
  }
  const PlCoef<T, TL> fL(eo, KIN ? pe[N1 - 1][HE - 1] : after);
  const PlTransposed<PlCoef<T, TL>, Q> fLt{fL};
  // a Gauss line of the plane through its weights, in place: c <- Lq^T (w .* (Lq c))
  const auto gauss_line = [&](T(&c)[N1], const T(&wq)[Q]) {
    T cp[HE], cm[HO], oe[QE], oo[QO], t[Q], tp[QE], tm[QO], re[HE], ro[HO];
    pl_split<N1>(c, cp, cm);
    pl_halves<TL, false>(fL, cp, cm, oe, oo);
    pl_join<Q>(oe, oo, t);
#pragma unroll
    for (int q = 0; q < Q; ++q) t[q] *= wq[q];
    pl_split<Q>(t, tp, tm);
    pl_halves<TLt, false>(fLt, tp, tm, re, ro);
    pl_join<N1>(re, ro, c);
  };
  // the kinetic FP64 kernel at p = 5 reads the plane again for each pair of Gauss
  // lines: its registers do not hold u, m and p at once (keeping u spills, 477
  // against 233 us at 24 cells, B = 12)
  constexpr bool REREAD = KIN && sizeof(T) == 8 && P == 5;
  T up[REREAD ? 1 : N1][HE], um[REREAD ? 1 : N1][HO];
  if constexpr (!REREAD) {
#pragma unroll
    for (int b = 0; b < N1; ++b) u_line(pl, b, up[b], um[b]);
  }
  uint32_t again = 0;  // a 0 the compiler does not see: the plane is read again, not kept
  static_for<0, QE>([&](auto kk) {
    constexpr int k = decltype(kk)::value;
    constexpr bool mid = 2 * k + 1 == Q;
    if constexpr (REREAD) asm("" : "+v"(again));
    T w0[Q], w1[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      w0[q] = we[k * Q + q];
      w1[q] = we[(Q - 1 - k) * Q + q];
    }
    T c0[N1], c1[N1];
#pragma unroll
    for (int b = 0; b < N1; ++b) {
      T tp[HE], tm[HO];
      if constexpr (REREAD) {
        u_line(pl + again, b, tp, tm);
      } else {
#pragma unroll
        for (int i = 0; i < HE; ++i) tp[i] = up[b][i];
#pragma unroll
        for (int i = 0; i < HO; ++i) tm[i] = um[b][i];
      }
      T ev = T(0), ov = T(0);
      static_for<0, HO>([&](auto jj) {
        constexpr int J = decltype(jj)::value;
        ev += fL.template at<k, J, 0>() * tp[J];
        if constexpr (!mid) ov += fL.template at<k, J, 1>() * tm[J];
      });
      if constexpr (N1 % 2 == 1) ev += fL.template at<k, 0, 2>() * tp[HE - 1];
      c0[b] = ev + ov;
      c1[b] = ev - ov;
    }
    gauss_line(c0, w0);
    if constexpr (!mid) gauss_line(c1, w1);
#pragma unroll
    for (int b = 0; b < N1; ++b) {
      const T sp = mid ? c0[b] : c0[b] + c1[b], sm = c0[b] - c1[b];
      static_for<0, HE>([&](auto ii) {
        constexpr int I = decltype(ii)::value;
        pe[b][I] += fLt.template at<I, k, mid ? 2 : 0>() * sp;
        if constexpr (!mid && I < HO) po[b][I] += fLt.template at<I, k, 1>() * sm;
      });
    }
  });
  const auto put_plane = [&](T(&ve)[N1][HE], T(&vo)[N1][HO]) {
#pragma unroll
    for (int b = 0; b < N1; ++b) {
      T y[N1];
      pl_join<N1>(ve[b], vo[b], y);
#pragma unroll
      for (int a = 0; a < N1; ++a) pl[(a * N1 + b) * NS] = y[a];
    }
  };
  put_plane(pe, po);
  wave_lds_fence();
  // the lane's place found again (and with dotp its input read again), from numbers
  // whose origin the compiler does not see: kept through the planes, they would cost
  // registers that the planes need
  uint32_t sid2 = sid, r2 = r;
  if constexpr (XN) asm("" : "+v"(sid2), "+v"(r2));
  // z lines back: y = Lq^T p + E m
  T ze[K3][HE], zo[K3][HO];
#pragma unroll
  for (int k = 0; k < K3; ++k) {
    const uint32_t l = line_of(r2, k);
    T v[Q], vp[QE], vm[QO];
#pragma unroll
    for (int q = 0; q < Q; ++q) v[q] = lds[q * PS + l * NS + slot];
    pl_split<Q>(v, vp, vm);
    pl_halves<TLt, false>(fLt, vp, vm, ze[k], zo[k]);
  }
  if constexpr (KIN) {
    // the sums are complete here, before E's coefficients take Lq's registers
    if constexpr (sizeof(T) == 8) {
#pragma unroll
      for (int k = 0; k < K3; ++k) {
#pragma unroll
        for (int i = 0; i < HE; ++i) asm volatile("" : "+v"(ze[k][i]));
#pragma unroll
        for (int i = 0; i < HO; ++i) asm volatile("" : "+v"(zo[k][i]));
      }
    }
    wave_lds_fence();
    put_plane(me, mo);
    wave_lds_fence();
  }
  const PlCoef<T, TE> fE(eo, ze[K3 - 1][0]);
  double dotv = 0.0;
  const uint32_t e2 = cell_of(sid2), j2 = sid2 - e2 * B, n2 = XN ? first_node(e2) : 0;
  T* const yc = Yc + (size_t)e2 * NE * B + j2;
  const uint32_t zy = N2 * B;
#pragma unroll
  for (int k = 0; k < K3; ++k) {
    const uint32_t l = line_of(r2, k);
    T xl[N1];
    if constexpr (XN) {
      if (dotp) load_line(l, n2, j2, xl);
    }
    if constexpr (KIN) {
      T v[Q], vp[QE], vm[QO];
#pragma unroll
      for (int q = 0; q < Q; ++q) v[q] = lds[q * PS + l * NS + slot];
      pl_split<Q>(v, vp, vm);
      T he[HE], ho[HO];
      pl_halves<TE, false>(fE, vp, vm, he, ho);
#pragma unroll
      for (int i = 0; i < HE; ++i) ze[k][i] += hq * he[i];
#pragma unroll
      for (int i = 0; i < HO; ++i) zo[k][i] += hq * ho[i];
    }
    T y[N1];
    pl_join<N1>(ze[k], zo[k], y);
    if (live && r2 + Q * k < (uint32_t)N2) {
      T* const yl = yc + l * B;
#pragma unroll
      for (int c = 0; c < N1; ++c) yl[(size_t)c * zy] = y[c];
      if constexpr (XN) {
        if (dotp) {
#pragma unroll
          for (int c = 0; c < N1; ++c) dotv += (double)xl[c] * (double)y[c];
        }
      }
    }
  }
  if constexpr (XN) {
    if (dotp) {
      wave_lds_fence();
      double* red = reinterpret_cast<double*>(lds);
      red[lane] = dotv;
      wave_lds_fence();
      if (r == 0 && live) {
        double t = 0.0;
#pragma unroll
        for (int q = 0; q < Q; ++q) t += red[q * NS + slot];
        dotp[(size_t)j2 * (uint32_t)g.ncell + e2] = t;
      }
    }
  }
}

// ---------------------------------------- cell product line by line (MINRES, FP64)
// The FP64 product of the MINRES steps: the same chain as k_cell_plane, but each
// contraction of the tensor along a line of the cell, with the input scaled on the
// fly and the cell's dots x.(H_e x).  An iterate that a step limit stops is not
// determined by its inputs in 64 bits: once a Ritz value has converged the Lanczos
// vectors amplify rounding (two orders of the same sums gave iterates 1e-8 to 3e-2
// apart after 32 to 64 steps on meshes of 25 to 63 nodes per axis, 1e-15 to 1e-10 on
// 91 to 115).  So the steps keep one order of arithmetic, this one, and an iterate
// stopped after k steps stays what it has been; its price is the plane kernel's
// gain in FP64 solves (24 cells p = 5 B = 12: 261 against 233 us, 30 p = 4 B = 64:
// 1383 against 1139).  Do not regroup a sum here.
//
// One work-group handles one cell and CG columns; an item is one line of the cell's
// tensor along one axis for one column.  Intermediates live in LDS as [entry][CG],
// with padded line strides (N1 and Q rounded up to odd: 5, 7 at p = 4; 7, 9 at
// p = 5) so that the 64 lanes of a wave spread over the banks.  The exception is
// region D at p = 5 (Q = 8): unpadded lines, entry x of line (c, y) at slot x ^ y,
// which spreads the lanes as the stride 9 does and puts the lines that one stage-6
// item reads 512 B apart, so that the compiler pairs those accesses.  The kinetic
// chain runs first and the x-line input stays in registers for the potential chain;
// the y and z stages overwrite their input in place.  Region Bk is dead once stage
// 3 has run, so D shares its memory:
//   1  x lines (c,b):  ka = M x -> A,  kb = D x -> Bk      (x gathered from HBM)
//   2  y lines (c,a):  k1 = M ka -> A,  k2 = D ka + M kb -> Bk
//   3  z lines (b,a):  yk = D k1 + M k2 -> A
//   4  x lines (c,b):  t1[c][b][qx] = Lq x -> D             (x from registers)
//   5  y lines (c,qx): t2[c][qy][qx] = Lq t1 -> D
//   6  z lines (qy,qx): s2 = Lq^T (w .* (Lq t2)) -> D
//   7  y lines (c,qx): s1[c][b][qx] = Lq^T s2 -> D
//   8  x lines (c,b):  Yc[e][(c,b,a)][j] = (Lq^T s1)[a] + (h/4) yk[a]
__host__ __device__ constexpr int cmax(int a, int b) { return a > b ? a : b; }

// Coefficient W (0 even, 1 odd, 2 middle) of row I, column J of operator A: a scalar
// load from the table eo (EoTable<P>::v).
template <class A, int I, int J, int W>
__device__ inline double eo_coef(const double* __restrict__ eo) {
  using E = EoTable<A::kP>;
  constexpr int c = E::C(A::kK);
  constexpr int idx = E::base(A::kK) + I * E::stride(A::kK) +
                      (W == 0 ? J : W == 1 ? c / 2 + J : 2 * (c / 2));
  return eo[idx];
}
// Adds row I's even and odd sums of A applied to the split input (xp, xm).
template <class A, int I>
__device__ inline void eo_row(const double (&xp)[(A::C + 1) / 2], const double (&xm)[A::C / 2],
                              double& e, double& o, const double* __restrict__ eo) {
  static_for<0, A::C / 2>([&](auto j) {
    constexpr int J = decltype(j)::value;
    e += eo_coef<A, I, J, 0>(eo) * xp[J];
    if constexpr (2 * I + 1 != A::R) o += eo_coef<A, I, J, 1>(eo) * xm[J];
  });
  if constexpr (A::C % 2 == 1) e += eo_coef<A, I, 0, 2>(eo) * xp[A::C / 2];
}
// The R outputs of one or more even-odd contractions: rows(i, e, o) adds the
// sums of row i, put(i, y) receives output i (i an integral constant).
template <int R, typename Rows, typename Put>
__device__ inline void eo_out(Rows&& rows, Put&& put) {
  static_for<0, (R + 1) / 2>([&](auto i) {
    constexpr int I = decltype(i)::value;
    double e = 0.0, o = 0.0;
    rows(i, e, o);
    if constexpr (2 * I + 1 == R) {
      put(i, e);
    } else {
      put(i, e + o);
      put(ic<R - 1 - I>{}, e - o);
    }
  });
}
#define IDFT_IC(x) decltype(x)::value
// Entry A of a line from its even-odd split (pl_split): the inverse of the
// split, to rounding.
template <int C, int A>
__device__ inline double eo_unsplit(const double (&xp)[(C + 1) / 2], const double (&xm)[C / 2]) {
  if constexpr (2 * A + 1 == C) {
    return xp[A];
  } else if constexpr (A < C / 2) {
    return 0.5 * (xp[A] + xm[A]);
  } else {
    constexpr int J = C - 1 - A;
    return 0.5 * (xp[J] - xm[J]);
  }
}

template <int P, int CG>
__global__ __launch_bounds__(kThreads) void k_cell_line(
    Geo g, double hq, const double* __restrict__ W, const double* __restrict__ S,
    const double* __restrict__ X, const double* __restrict__ xn, const double* __restrict__ xcol,
    double* __restrict__ Yc, int B, double* __restrict__ dotp, const double* __restrict__ eo) {
  constexpr int N1 = P + 1, Q = P + 3, N2 = N1 * N1, NE = N2 * N1, Q2 = Q * Q;
  constexpr int QP = Q | 1, N1P = N1 | 1, NV = CG;
  constexpr int HE = (N1 + 1) / 2, HO = N1 / 2, QE = (Q + 1) / 2, QO = Q / 2;
  // x-line items per thread (lines x columns over the work-group)
  constexpr int KI = (N2 * NV + kThreads - 1) / kThreads;
  typedef SfTab<P, 0> TL;
  typedef SfTab<P, 1> TLt;
  typedef SfTab<P, 2> TM;
  typedef SfTab<P, 3> TD;
  // regions, each [entry][NV]:
  //   A  [(c,b)][N1P]      ka -> k1 -> yk            (kinetic chain, in place)
  //   Bk [(c,b)][N1P]      kb -> k2                  (stages 1-3)
  //   D  [c][Q][QS]        t1 -> t2 -> s2 -> s1      (stages 4-8, over Bk)
  // SWZ: D unpadded (QS = Q = 8), entry (c, y, x) at slot x ^ y of its line
  constexpr bool SWZ = Q == 8;
  constexpr int QS = SWZ ? Q : QP;
  __shared__ __align__(16) double rA[N2 * N1P * NV];
  __shared__ __align__(16) double rBD[cmax(N2 * N1P, N1 * Q * QS) * NV];
  double* const rB = rBD;
  // Byte offsets into D of entry (c, y, x), column jv, from a per-item base and the
  // one index that is a compile-time constant at the access (so that the rest folds
  // into the LDS instruction's offset field):
  //   dy(c, x, jv) then at_y(base, y);  dx(c, y, jv) then at_x(base, x);
  //   dc(y, x, jv) then at_c(base, c).
  // With SWZ the slot x ^ y is an XOR of the offset's slot bits (the slot
  // field, NV sizeof(double) bytes per slot and 8 slots, holds no other bits).
  constexpr uint32_t SB = NV * sizeof(double);
  const auto dy = [](uint32_t c, uint32_t x, uint32_t jv) -> uint32_t {
    return (c * Q * QS + x) * SB + jv * (uint32_t)sizeof(double);
  };
  const auto at_y = [](uint32_t base, uint32_t y) -> uint32_t {
    return SWZ ? (base ^ (y * SB)) + y * QS * SB : base + y * QS * SB;
  };
  const auto dx = [](uint32_t c, uint32_t y, uint32_t jv) -> uint32_t {
    return ((c * Q + y) * QS + (SWZ ? y : 0u)) * SB + jv * (uint32_t)sizeof(double);
  };
  const auto at_x = [](uint32_t base, uint32_t x) -> uint32_t {
    return SWZ ? base ^ (x * SB) : base + x * SB;
  };
  const auto dc = [](uint32_t y, uint32_t x, uint32_t jv) -> uint32_t {
    return (y * QS + (SWZ ? (x ^ y) : x)) * SB + jv * (uint32_t)sizeof(double);
  };
  const auto at_c = [](uint32_t base, uint32_t c) -> uint32_t { return base + c * Q * QS * SB; };
  char* const rDb = reinterpret_cast<char*>(rBD);
  const auto dref = [rDb](uint32_t off) -> double& { return *reinterpret_cast<double*>(rDb + off); };
  // (cell, column group) pairs dealt to the 8 XCDs in contiguous runs, the
  // groups of one cell at consecutive slots of one XCD, so that they share
  // that XCD's L2 for the cell's rows of X and of the cell scratch (each group
  // holds CG of the B columns of a row).  Every index below fits in 32 bits
  // (the host checks N B and cells n_e B against 2^32).
  const uint32_t ncell = (uint32_t)g.ncell, nc = (uint32_t)g.nc, np = (uint32_t)g.p;
  const uint32_t NN = (uint32_t)g.N1, ub = (uint32_t)B;
  const uint32_t ngrp = (ub + CG - 1) / CG, npair = ncell * ngrp;
  const uint32_t per = (npair + 7) / 8;
  const uint32_t k = (blockIdx.x % 8) * per + blockIdx.x / 8;
  if (k >= npair) return;
  const uint32_t e = k / ngrp;
  const int c0 = (int)(k % ngrp) * CG;
  const int bw = min(CG, B - c0);
  const int tid = threadIdx.x;
  const uint32_t cx = e % nc, cy = (e / nc) % nc, cz = e / (nc * nc);
  const double* we = W + e * (uint32_t)(Q2 * Q);
  // this thread's column (every item of a thread has column tid % NV, since kThreads
  // is a multiple of NV) and its scale, loaded first: a later load would make its
  // first use wait for the weights too
  const int jv = tid % NV;
  const double xc = xcol ? xcol[c0 + min(jv, bw - 1)] : 1.0;
  // the quadrature weights of this thread's stage-6 items, loaded now so that
  // their latency hides behind stages 1-5 (item it6 = tid + k6 kThreads takes
  // w_e[qz][ln6] for its line ln6 = it6 / NV)
  constexpr int K6 = (Q2 * NV + kThreads - 1) / kThreads;
  double wpre[K6][Q];
#pragma unroll
  for (int k6 = 0; k6 < K6; ++k6) {
    const int it6 = tid + k6 * kThreads;
    const int ln6 = it6 < Q2 * NV ? it6 / NV : 0;
#pragma unroll
    for (int qz = 0; qz < Q; ++qz) wpre[k6][qz] = we[qz * Q2 + ln6];
  }
  // the input lines stay in registers from stage 1 to stage 8 (even-odd split)
  double keep_p[KI][HE], keep_m[KI][HO];
  // stage 1: x lines ln = c*N1 + b of the gathered input -> ka = M x, kb = D x
#pragma unroll
  for (int ki = 0; ki < KI; ++ki) {
    const int it = tid + ki * kThreads;
    if (it >= N2 * NV) break;
    const int ln = it / NV;
    double v[N1];
    const uint32_t b = ln % N1, c = ln / N1;
    const uint32_t n0 = ((cz * np + c) * NN + (cy * np + b)) * NN + cx * np;
    // the line's N1 nodes are consecutive: one base pointer per array, the nodes at
    // immediate offsets (the X rows B apart), all loads issued before the first product
    const double* Sp = S + n0;
    if (jv < bw) {
      const double* Xp = X + (size_t)n0 * ub + (uint32_t)(c0 + jv);
      double sv[N1], xv[N1], nv[N1];
#pragma unroll
      for (int a = 0; a < N1; ++a) {
        sv[a] = Sp[a];
        xv[a] = Xp[(size_t)a * ub];
        nv[a] = xn[n0 + a];
      }
#pragma unroll
      for (int a = 0; a < N1; ++a) {
        double x = sv[a] * xv[a];
        x *= nv[a];
        if (xcol) x *= xc;
        v[a] = x;
      }
    } else {
#pragma unroll
      for (int a = 0; a < N1; ++a) v[a] = 0.0;
    }
    pl_split<N1>(v, keep_p[ki], keep_m[ki]);
    eo_out<N1>(
        [&](auto i, double& s, double& d) { eo_row<TM, IDFT_IC(i)>(keep_p[ki], keep_m[ki], s, d, eo); },
        [&](auto a2, double r) { rA[(ln * N1P + IDFT_IC(a2)) * NV + jv] = r; });
    eo_out<N1>(
        [&](auto i, double& s, double& d) { eo_row<TD, IDFT_IC(i)>(keep_p[ki], keep_m[ki], s, d, eo); },
        [&](auto a2, double r) { rB[(ln * N1P + IDFT_IC(a2)) * NV + jv] = r; });
  }
  __syncthreads();
  // stage 2: y lines (c, a) of the kinetic chain, in place:
  // k1 = M ka (over ka), k2 = D ka + M kb (over kb)
  for (int it = tid; it < N2 * NV; it += kThreads) {
    const int l2 = it / NV;
    const int a = l2 % N1, c = l2 / N1;
    double va[N1], vb[N1], ap[HE], am[HO], bp[HE], bm[HO];
#pragma unroll
    for (int b = 0; b < N1; ++b) {
      va[b] = rA[((c * N1 + b) * N1P + a) * NV + jv];
      vb[b] = rB[((c * N1 + b) * N1P + a) * NV + jv];
    }
    pl_split<N1>(va, ap, am);
    pl_split<N1>(vb, bp, bm);
    eo_out<N1>([&](auto i, double& s, double& d) { eo_row<TM, IDFT_IC(i)>(ap, am, s, d, eo); },
               [&](auto b2, double r) { rA[((c * N1 + IDFT_IC(b2)) * N1P + a) * NV + jv] = r; });
    eo_out<N1>(
        [&](auto i, double& s, double& d) {
          eo_row<TD, IDFT_IC(i)>(ap, am, s, d, eo);
          eo_row<TM, IDFT_IC(i)>(bp, bm, s, d, eo);
        },
        [&](auto b2, double r) { rB[((c * N1 + IDFT_IC(b2)) * N1P + a) * NV + jv] = r; });
  }
  __syncthreads();
  // stage 3: z lines (b, a) of the kinetic chain: yk = D k1 + M k2 (over k1)
  for (int it = tid; it < N2 * NV; it += kThreads) {
    const int l2 = it / NV;  // l2 = b * N1 + a
    const int a = l2 % N1, b = l2 / N1;
    double v1[N1], v2[N1], p1[HE], m1[HO], p2[HE], m2[HO];
#pragma unroll
    for (int c = 0; c < N1; ++c) {
      v1[c] = rA[((c * N1 + b) * N1P + a) * NV + jv];
      v2[c] = rB[((c * N1 + b) * N1P + a) * NV + jv];
    }
    pl_split<N1>(v1, p1, m1);
    pl_split<N1>(v2, p2, m2);
    eo_out<N1>(
        [&](auto i, double& s, double& d) {
          eo_row<TD, IDFT_IC(i)>(p1, m1, s, d, eo);
          eo_row<TM, IDFT_IC(i)>(p2, m2, s, d, eo);
        },
        [&](auto c2, double r) { rA[((IDFT_IC(c2) * N1 + b) * N1P + a) * NV + jv] = r; });
  }
  __syncthreads();
  // stage 4: x lines of the potential chain from the kept input:
  // t1[c][b][qx] = Lq x (over k2, which stage 3 has consumed)
#pragma unroll
  for (int ki = 0; ki < KI; ++ki) {
    const int it = tid + ki * kThreads;
    if (it >= N2 * NV) break;
    const int ln = it / NV;
    const int b = ln % N1, c = ln / N1;
    const uint32_t base = dx(c, b, jv);
    eo_out<Q>(
        [&](auto i, double& s, double& d) { eo_row<TL, IDFT_IC(i)>(keep_p[ki], keep_m[ki], s, d, eo); },
        [&](auto q, double r) { dref(at_x(base, IDFT_IC(q))) = r; });
  }
  __syncthreads();
  // stage 5: y lines (c, qx): t2[c][qy][qx] = Lq t1, in place (over t1)
  for (int it = tid; it < N1 * Q * NV; it += kThreads) {
    const int ln = it / NV;
    const int qx = ln % Q, c = ln / Q;
    const uint32_t base = dy(c, qx, jv);
    double v[N1], vp[HE], vm[HO];
#pragma unroll
    for (int b = 0; b < N1; ++b) v[b] = dref(at_y(base, b));
    pl_split<N1>(v, vp, vm);
    eo_out<Q>([&](auto i, double& s, double& d) { eo_row<TL, IDFT_IC(i)>(vp, vm, s, d, eo); },
              [&](auto qy, double r) { dref(at_y(base, IDFT_IC(qy))) = r; });
  }
  __syncthreads();
  // stage 6: z lines (qy, qx) through the quadrature weights, in place:
  // s2 = Lq^T (w .* (Lq t2)) (over t2)
#pragma unroll
  for (int k6 = 0; k6 < K6; ++k6) {
    const int it = tid + k6 * kThreads;
    if (it >= Q2 * NV) break;
    const int ln = it / NV;  // ln = qy * Q + qx
    const int qx = ln % Q, qy = ln / Q;
    const uint32_t base = dc(qy, qx, jv);
    double v[N1], vp[HE], vm[HO];
#pragma unroll
    for (int c = 0; c < N1; ++c) v[c] = dref(at_c(base, c));
    pl_split<N1>(v, vp, vm);
    double u[Q], up[QE], um[QO];
    eo_out<Q>([&](auto i, double& s, double& d) { eo_row<TL, IDFT_IC(i)>(vp, vm, s, d, eo); },
              [&](auto qz, double r) { u[IDFT_IC(qz)] = r * wpre[k6][IDFT_IC(qz)]; });
    pl_split<Q>(u, up, um);
    eo_out<N1>([&](auto i, double& s, double& d) { eo_row<TLt, IDFT_IC(i)>(up, um, s, d, eo); },
               [&](auto c, double r) { dref(at_c(base, IDFT_IC(c))) = r; });
  }
  __syncthreads();
  // stage 7: y lines back (c, qx), in place: s1[c][b][qx] = Lq^T s2 (over s2)
  for (int it = tid; it < N1 * Q * NV; it += kThreads) {
    const int ln = it / NV;
    const int qx = ln % Q, c = ln / Q;
    const uint32_t base = dy(c, qx, jv);
    double v[Q], vp[QE], vm[QO];
#pragma unroll
    for (int qy = 0; qy < Q; ++qy) v[qy] = dref(at_y(base, qy));
    pl_split<Q>(v, vp, vm);
    eo_out<N1>([&](auto i, double& s, double& d) { eo_row<TLt, IDFT_IC(i)>(vp, vm, s, d, eo); },
               [&](auto b, double r) { dref(at_y(base, IDFT_IC(b))) = r; });
  }
  __syncthreads();
  // stage 8: x lines back (c, b) plus the kinetic part, into the cell scratch; with
  // dotp also the cell's x.(H_e x) per column, into dotp[column * ncell + cell] (x
  // from the kept input lines: each item holds the same line as in stage 1)
  double dotv = 0.0;
#pragma unroll
  for (int ki = 0; ki < KI; ++ki) {
    const int it = tid + ki * kThreads;
    if (it >= N2 * NV) break;
    const int ln = it / NV;
    if (jv >= bw) continue;
    const int b = ln % N1, c = ln / N1;
    const uint32_t base = dx(c, b, jv);
    double v[Q], vp[QE], vm[QO];
#pragma unroll
    for (int qx = 0; qx < Q; ++qx) v[qx] = dref(at_x(base, qx));
    pl_split<Q>(v, vp, vm);
    double* yp = Yc + (size_t)((e * NE + ln * N1) * ub + c0 + jv);
    eo_out<N1>([&](auto i, double& s, double& d) { eo_row<TLt, IDFT_IC(i)>(vp, vm, s, d, eo); },
               [&](auto a, double r) {
                 constexpr int A = IDFT_IC(a);
                 const double y = hq * rA[(ln * N1P + A) * NV + jv] + r;
                 yp[(size_t)A * ub] = y;
                 if (dotp) dotv += eo_unsplit<N1, A>(keep_p[ki], keep_m[ki]) * y;
               });
  }
  if (dotp) {
    // per column jv: the threads tid = jv (mod NV) (kThreads and 64 are
    // multiples of NV), summed over each wave, then over the 4 waves
    __syncthreads();  // stage 8 has read rA
    const int lane = tid & 63, wave = tid >> 6;
    double t = dotv;
#pragma unroll
    for (int o = 32; o >= NV; o >>= 1) t += __shfl_xor(t, o, 64);
    if (lane < NV) rA[wave * NV + lane] = t;
    __syncthreads();
    if (tid < bw) {
      double d = 0.0;
#pragma unroll
      for (int w = 0; w < kThreads / 64; ++w) d += rA[w * NV + tid];
      dotp[(size_t)(uint32_t)(c0 + tid) * ncell + e] = d;
    }
  }
}
#undef IDFT_IC

// Phase 2: every node sums its contributions from the (at most 8) cells that
// share it -- found arithmetically on the structured mesh, so no atomics and
// no colouring -- and combines them with up to three other blocks:
//   Y = beta Y + alpha S[n] sum + a ca[j] xn[n] X + b cb[j] Z + c cc[j] W
// (xn, the operator input's node scale, optional).  With `partial`, the
// per-column block partials of V.Y (FP64) for the scaled operator input
// V = xcol[j] xn[n] Xin, optionally stored.  Nodes are taken in their
// linear order n = (iz N1 + iy) N1 + ix: block b covers R consecutive chunks
// of per = 256 / (B / VW) nodes, [(b R + r) per, (b R + r + 1) per), so a
// chunk may cross x rows and every lane has work; thread t owns column group
// t % (B / VW) and position t / (B / VW) within each chunk.
// VW consecutive elements of a node-major row (16-byte aligned for VW > 1).
template <typename T, int VW>
__device__ inline void vload(const T* __restrict__ p, T (&o)[VW]) {
  if constexpr (VW == 1) {
    o[0] = p[0];
  } else if constexpr (VW == 2) {
    typedef typename std::conditional<std::is_same<T, float>::value, float2, double2>::type v2;
    const v2 v = *reinterpret_cast<const v2*>(p);
    o[0] = v.x; o[1] = v.y;
  } else {
    const typename Vec4<T>::type v = *reinterpret_cast<const typename Vec4<T>::type*>(p);
    o[0] = v.x; o[1] = v.y; o[2] = v.z; o[3] = v.w;
  }
}
template <typename T, int VW>
__device__ inline void vstore(T* __restrict__ p, const T (&o)[VW]) {
  if constexpr (VW == 1) {
    p[0] = o[0];
  } else if constexpr (VW == 2) {
    typedef typename std::conditional<std::is_same<T, float>::value, float2, double2>::type v2;
    *reinterpret_cast<v2*>(p) = v2{o[0], o[1]};
  } else {
    typedef typename Vec4<T>::type v4;
    *reinterpret_cast<v4*>(p) = v4{o[0], o[1], o[2], o[3]};
  }
}

// Sum of the (at most 8) cell contributions of node nidx for the VW columns
// from j0: the cells sharing the node are found arithmetically on the
// structured mesh (nodes n = (iz N1 + iy) N1 + ix).
// The cells sharing node index i along one axis: (c0, a0) and, when the node
// lies on an interior cell face (n = 2), (c1, a1), cell c and local index a,
// in the order (left cell, right cell).
struct AxisCells {
  uint32_t c0, a0, c1, a1;
  int n;
};
template <int P>
__device__ inline AxisCells axis_cells(uint32_t i, uint32_t nc) {
  const uint32_t q = i / P, r = i - q * P;
  AxisCells A;
  if (r != 0) { A.c0 = A.c1 = q; A.a0 = A.a1 = r; A.n = 1; }
  else if (q == 0) { A.c0 = A.c1 = 0; A.a0 = A.a1 = 0; A.n = 1; }
  else if (q == nc) { A.c0 = A.c1 = nc - 1; A.a0 = A.a1 = P; A.n = 1; }
  else { A.c0 = q - 1; A.a0 = P; A.c1 = q; A.a1 = 0; A.n = 2; }
  return A;
}
template <typename TY, int P, int VW>
__device__ inline void gather_node(const Geo& g, FastDiv divN1, uint32_t B, uint32_t nidx,
                                   const TY* __restrict__ Yc, uint32_t j0, double (&sum)[VW]) {
  constexpr uint32_t n1 = P + 1, ne = n1 * n1 * n1;
  const uint32_t N1 = g.N1, nc = g.nc;
  const uint32_t row = fast_div(nidx, divN1), ix = nidx - row * N1;
  const uint32_t iz = fast_div(row, divN1), iy = row - iz * N1;
  // contributions (cell, local index) along each axis (selects, no arrays:
  // run-time-indexed arrays would live in scratch memory)
  const AxisCells X = axis_cells<P>(ix, nc), Y = axis_cells<P>(iy, nc), Z = axis_cells<P>(iz, nc);
  // all 8 contribution slots are loaded before the first is summed, so
  // the loads are in flight together
  TY c8[8][VW];
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const int kz = k >> 2, ky = (k >> 1) & 1, kx = k & 1;
    // no branch: a contribution the node does not have loads the node's
    // first one (same cache line) and is then zeroed, so that all eight
    // loads are issued before the first wait (behind a per-load branch
    // the compiler waits for each load in turn)
    const bool ok = kz < Z.n && ky < Y.n && kx < X.n;
    const bool sz = ok && kz, sy = ok && ky, sx = ok && kx;
    // the host checks cells n_e B < 2^32
    const uint32_t e = ((sz ? Z.c1 : Z.c0) * nc + (sy ? Y.c1 : Y.c0)) * nc + (sx ? X.c1 : X.c0);
    const uint32_t l = ((sz ? Z.a1 : Z.a0) * n1 + (sy ? Y.a1 : Y.a0)) * n1 + (sx ? X.a1 : X.a0);
    TY t[VW];
    vload<TY, VW>(Yc + ((e * ne + l) * B + j0), t);
#pragma unroll
    for (int v = 0; v < VW; ++v) c8[k][v] = ok ? t[v] : TY(0);
  }
#pragma unroll
  for (int v = 0; v < VW; ++v) sum[v] = 0.0;
#pragma unroll
  for (int k = 0; k < 8; ++k)
#pragma unroll
    for (int v = 0; v < VW; ++v) sum[v] += (double)c8[k][v];
}

template <typename TY, typename T, int P, int VW>
__global__ __launch_bounds__(kThreads) void k_cell_gather(
    Geo g, FastDiv divN1, uint32_t B, uint32_t R, const TY* __restrict__ Yc, const T* __restrict__ S,
    T* __restrict__ Y, double alpha, double beta, const T* __restrict__ X, double a,
    const double* __restrict__ ca, const T* __restrict__ Z, double b,
    const double* __restrict__ cb, const T* __restrict__ W, double c,
    const double* __restrict__ cc, const T* __restrict__ Xin, const double* __restrict__ xn,
    const double* __restrict__ xcol, T* __restrict__ V, double* __restrict__ partial) {
  __shared__ double red[1][kThreads * VW];
  const uint32_t N1 = g.N1;
  const uint32_t nb = B / VW;  // column groups of a node
  const uint32_t tid = threadIdx.x, per = kThreads / nb;
  const uint32_t jg = tid % nb, off = tid / nb, j0 = jg * VW;
  double dot[1][VW];
#pragma unroll
  for (int v = 0; v < VW; ++v) dot[0][v] = 0.0;
  if (off < per) {
    double caj[VW], cbj[VW], ccj[VW], xs[VW];
#pragma unroll
    for (int v = 0; v < VW; ++v) {
      caj[v] = X ? a * (ca ? ca[j0 + v] : 1.0) : 0.0;
      cbj[v] = Z ? b * (cb ? cb[j0 + v] : 1.0) : 0.0;
      ccj[v] = W ? c * (cc ? cc[j0 + v] : 1.0) : 0.0;
      xs[v] = xcol ? xcol[j0 + v] : 1.0;
    }
    const uint32_t nn = N1 * N1 * N1;
    for (uint32_t rr = 0; rr < R; ++rr) {
      const uint32_t nidx = (blockIdx.x * R + rr) * per + off;
      if (nidx >= nn) break;
      double sum[VW];
      gather_node<TY, P, VW>(g, divN1, B, nidx, Yc, j0, sum);
      const uint32_t n = nidx;
      const uint32_t i = n * B + j0;
      const double sn = xn ? xn[n] : 1.0;
      const double sa = alpha * (double)S[n];
      T xv[VW], zv[VW], wv[VW], yv[VW], xin[VW], yo[VW];
      if (X) vload<T, VW>(X + i, xv);
      if (Z) vload<T, VW>(Z + i, zv);
      if (W) vload<T, VW>(W + i, wv);
      if (beta != 0.0) vload<T, VW>(Y + i, yv);
      if (partial) vload<T, VW>(Xin + i, xin);
#pragma unroll
      for (int v = 0; v < VW; ++v) {
        double t = sa * sum[v];
        if (X) t += caj[v] * (sn * (double)xv[v]);
        if (Z) t += cbj[v] * (double)zv[v];
        if (W) t += ccj[v] * (double)wv[v];
        if (beta != 0.0) t += beta * (double)yv[v];
        yo[v] = (T)t;
      }
      if (partial) {
        T vv[VW];
#pragma unroll
        for (int v = 0; v < VW; ++v) {
          vv[v] = (T)(xs[v] * (sn * (double)xin[v]));
          dot[0][v] += (double)vv[v] * (double)yo[v];
        }
        if (V) vstore<T, VW>(V + i, vv);
      }
      vstore<T, VW>(Y + i, yo);
    }
  }
  if (partial) {
    double t;
    if (xn) {  // a MINRES step: its fixed order of sums
      t = ordered_groups<1, VW>(red, dot, per, nb, tid, tid);
    } else {
      tree_groups<1, VW>(red, dot, per, nb, tid, off);
      t = red[0][tid];
    }
    if (tid < B) partial[((int64_t)blockIdx.y * gridDim.x + blockIdx.x) * B + tid] = t;
  }
}

// Node sums of the quadrature operator's cell products (k_cell_plane without the
// kinetic chain) and, while a node's row is at hand, the pair sums
//   partial[k gridDim.x + block] = sum over the block's nodes of
//                                  asc[n] A[n][i_k] T[n][j_k],  k < np <= 256,
// T = sum_e Yc optionally stored (T2, row length ldt).  Where A's node scale
// asc is 0 (the boundary) A counts as 0, whatever it holds.
// Bound by HBM: Yc, A and T2 once.  The rows of A and T of a chunk of
// per = 256 / (wb / VW) nodes go through LDS, because a pair's two columns sit in
// different lanes; thread t sums pair t % np over every (256 / np)-th node of
// the chunk, so 8 to 256 pairs keep most lanes busy.  It replaces an
// interpolation of both blocks to the quadrature points per pair (1.80 ms for 14
// pairs at 121^3 nodes x 12 columns) and 8 launches of coloured cells
// (2.18 ms for the operator).
template <int P, int VW>
__global__ __launch_bounds__(kThreads) void k_quad_gather(
    Geo g, FastDiv divN1, uint32_t wb, uint32_t R, const double* __restrict__ Yc,
    const double* __restrict__ A, uint32_t lda, const double* __restrict__ asc,
    double* __restrict__ T2, uint32_t ldt, const int* __restrict__ pairs, uint32_t np,
    double* __restrict__ partial) {
  __shared__ double ta[kThreads * VW], tb[kThreads * VW], red[kThreads];
  const uint32_t nb = wb / VW, tid = threadIdx.x, per = kThreads / nb;
  const uint32_t jg = tid % nb, off = tid / nb, j0 = jg * VW;
  const uint32_t nn = (uint32_t)g.N;
  const uint32_t nsl = np ? kThreads / np : 1, sl = np ? tid / np : 0;
  uint32_t pi = 0, pj = 0;
  if (np && sl < nsl) {
    pi = pairs[2 * (tid % np)];
    pj = pairs[2 * (tid % np) + 1];
  }
  double acc = 0.0;
  const uint32_t ngroups = (nn + R * per - 1) / (R * per);
  for (uint32_t grp = blockIdx.x; grp < ngroups; grp += gridDim.x)
    for (uint32_t rr = 0; rr < R; ++rr) {
      const uint32_t n0 = (grp * R + rr) * per;  // uniform: every thread reaches the barriers
      if (n0 >= nn) break;
      const uint32_t cnt = min(per, nn - n0), n = n0 + off;
      if (off < cnt) {
        double sum[VW];
        gather_node<double, P, VW>(g, divN1, wb, n, Yc, j0, sum);
        if (T2) vstore<double, VW>(T2 + (size_t)n * ldt + j0, sum);
        if (np) {
          double av[VW];
          vload<double, VW>(A + (size_t)n * lda + j0, av);
          const double sc = asc ? asc[n] : 1.0;
#pragma unroll
          for (int v = 0; v < VW; ++v) {
            ta[off * wb + j0 + v] = sc == 0.0 ? 0.0 : sc * av[v];
            tb[off * wb + j0 + v] = sum[v];
          }
        }
      }
      if (np) {
        __syncthreads();
        if (sl < nsl)
          for (uint32_t m = sl; m < cnt; m += nsl) acc += ta[m * wb + pi] * tb[m * wb + pj];
        __syncthreads();
      }
    }
  if (np) {
    red[tid] = acc;
    tree_cols(red, (int)nsl, (int)np, (int)tid, (int)(sl < nsl ? sl : kThreads));
    if (tid < np) partial[(size_t)tid * gridDim.x + blockIdx.x] = red[tid];
  }
}

// MINRES step, phase 2 with the Lanczos recurrence fused in (sum-factorised
// cell products, whose cell kernel has already produced v.Hv, so that the
// step's alpha is known before this kernel runs):
//   r_new = S sum + (cvn_j D r2 + ca2_j r2) + cr1_j r1
// with cvn = -eps/beta, ca2 = -alpha/beta, cr1 = -beta/beta_old (per column,
// from the state), and block partials of the three node dots the next step
// needs: r_new.D r_new (beta^2), D^2 r_new^2 and D r_new.r2, at
// partial[(k B + j) nblk + block] for k = 0, 1, 2.  r_new may be r1 (each
// thread reads and writes the same entries).
template <typename TY, typename T, int P, int VW>
__global__ __launch_bounds__(kThreads) void k_minres_gather(
    Geo g, FastDiv divN1, uint32_t B, uint32_t R, const TY* __restrict__ Yc,
    const T* __restrict__ S, const double* __restrict__ D, const T* __restrict__ r2,
    const T* r1, T* rnew, const double* __restrict__ st, double* __restrict__ partial) {
  __shared__ double red[3][kThreads * VW];
  const uint32_t N1 = g.N1;
  const uint32_t nb = B / VW;
  const uint32_t tid = threadIdx.x, per = kThreads / nb;
  const uint32_t jg = tid % nb, off = tid / nb, j0 = jg * VW;
  double q[3][VW];
#pragma unroll
  for (int v = 0; v < VW; ++v) q[0][v] = q[1][v] = q[2][v] = 0.0;
  if (off < per) {
    double cvn[VW], ca2[VW], cr1[VW];
#pragma unroll
    for (int v = 0; v < VW; ++v) {
      cvn[v] = st[MS_CVN * B + j0 + v];
      ca2[v] = st[MS_CA2 * B + j0 + v];
      cr1[v] = st[MS_CR1 * B + j0 + v];
    }
    const uint32_t nn = N1 * N1 * N1;
    // groups of R consecutive chunks, strided over a grid of at most
    // kMinresGatherBlocks work-groups (fewer partial rows to reduce)
    const uint32_t ngroups = (nn + R * per - 1) / (R * per);
    for (uint32_t grp = blockIdx.x; grp < ngroups; grp += gridDim.x)
    for (uint32_t rr = 0; rr < R; ++rr) {
      const uint32_t n = (grp * R + rr) * per + off;
      if (n >= nn) break;
      double sum[VW];
      gather_node<TY, P, VW>(g, divN1, B, n, Yc, j0, sum);
      const uint32_t i = n * B + j0;
      const double dn = D[n];
      const double sn = (double)S[n];
      T xv[VW], zv[VW], ro[VW];
      vload<T, VW>(r2 + i, xv);
      vload<T, VW>(r1 + i, zv);
#pragma unroll
      for (int v = 0; v < VW; ++v) {
        const double x = (double)xv[v];
        const double t = sn * sum[v] + (cvn[v] * dn + ca2[v]) * x + cr1[v] * (double)zv[v];
        ro[v] = (T)t;
        const double r = (double)ro[v], dr = dn * r;
        q[0][v] += r * dr;
        q[1][v] += dr * dr;
        q[2][v] += dr * x;
      }
      vstore<T, VW>(rnew + i, ro);
    }
  }
  // partials column-major, [k][column][block], so that each column's
  // reduction reads contiguous memory
  const int64_t nblk = (int64_t)gridDim.x;
  const double t = ordered_groups<3, VW>(red, q, per, nb, tid, tid);
  if (tid < 3 * B) partial[(int64_t)tid * nblk + blockIdx.x] = t;
}

// ------------------------------------------------------ Hamiltonian build
// H_e = K_e/2 + V_e,  V_e = N^T diag(v JxW) N by sum factorisation.
template <int P>
__global__ __launch_bounds__(kThreads) void k_build_h(Geo g, const double* __restrict__ Lq,
                                                      const double* __restrict__ M1,
                                                      const double* __restrict__ D1, double hh,
                                                      const double* __restrict__ veff,
                                                      const double* __restrict__ jxw,
                                                      double* __restrict__ h64,
                                                      float* __restrict__ h32) {
  constexpr int N1 = P + 1, Q = P + 3, NE = ne_of(P), NEP = nep_of(P), RT = NEP / 16;
  constexpr int N2 = N1 * N1;
  __shared__ double W[Q * Q * Q];
  __shared__ double Pq[Q * N2];         // Pq[q][a][a'] = L_a(q) L_a'(q)
  __shared__ double T1[Q * Q * N2];     // [qz][qy][a][a']
  __shared__ double T2[Q * N2 * N2];    // [qz][b][b'][a][a']
  __shared__ double sM[N2], sD[N2];
  const int64_t e = blockIdx.x;
  const int tid = threadIdx.x;
  for (int i = tid; i < Q * Q * Q; i += kThreads) W[i] = veff[e * Q * Q * Q + i] * jxw[i];
  for (int i = tid; i < Q * N2; i += kThreads) {
    const int q = i / N2, a = (i / N1) % N1, a2 = i % N1;
    Pq[i] = Lq[q * N1 + a] * Lq[q * N1 + a2];
  }
  for (int i = tid; i < N2; i += kThreads) { sM[i] = M1[i]; sD[i] = D1[i]; }
  __syncthreads();
  for (int i = tid; i < Q * Q * N2; i += kThreads) {
    const int aa = i % N2, qzy = i / N2;
    double s = 0.0;
#pragma unroll
    for (int qx = 0; qx < Q; ++qx) s += Pq[qx * N2 + aa] * W[qzy * Q + qx];
    T1[i] = s;
  }
  __syncthreads();
  for (int i = tid; i < Q * N2 * N2; i += kThreads) {
    const int aa = i % N2, bb = (i / N2) % N2, qz = i / (N2 * N2);
    double s = 0.0;
#pragma unroll
    for (int qy = 0; qy < Q; ++qy) s += Pq[qy * N2 + bb] * T1[(qz * Q + qy) * N2 + aa];
    T2[i] = s;
  }
  __syncthreads();
  constexpr int NTILE = ntiles_of(P);
  double* o64 = h64 + (size_t)e * NTILE * 256;
  float* o32 = h32 ? h32 + (size_t)e * NTILE * 256 : nullptr;
  for (int idx = tid; idx < NTILE * 256; idx += kThreads) {
    const int s = idx % 4, lane = (idx / 4) % 64, blk = idx / 256;
    int rt = 0;
    while (rt + 1 < RT && tile_index(RT, rt + 1, rt + 1) <= blk) ++rt;
    const int kg = rt + (blk - tile_index(RT, rt, rt));
    const int row = rt * 16 + lane % 16, col = kg * 16 + s * 4 + lane / 16;
    double v = 0.0;
    if (row < NE && col < NE) {
      const int a = row % N1, b = (row / N1) % N1, c = row / N2;
      const int a2 = col % N1, b2 = (col / N1) % N1, c2 = col / N2;
      const int aa = a * N1 + a2, bb = b * N1 + b2, cc = c * N1 + c2;
      double vv = 0.0;
#pragma unroll
      for (int qz = 0; qz < Q; ++qz) vv += Pq[qz * N2 + cc] * T2[(qz * N2 + bb) * N2 + aa];
      const double k = hh * (sD[aa] * sM[bb] * sM[cc] + sM[aa] * sD[bb] * sM[cc] +
                             sM[aa] * sM[bb] * sD[cc]);
      v = 0.5 * k + vv;
    }
    o64[idx] = v;
    if (o32) o32[idx] = (float)v;
  }
}

// ------------------------------------------------------ tensor contraction
// in [N1][N1][N1][NC] -> out [Q][Q][Q][NC] with A [Q][N1] (all in LDS).
template <int N1, int Q, int NC>
__device__ void tp_eval(const double* A, const double* in, double* t1, double* t2, double* out) {
  const int tid = threadIdx.x;
  for (int i = tid; i < N1 * N1 * Q * NC; i += kThreads) {
    const int col = i % NC, qx = (i / NC) % Q, cb = i / (NC * Q);
    const double* src = in + cb * N1 * NC + col;
    double s = 0.0;
#pragma unroll
    for (int a = 0; a < N1; ++a) s += A[qx * N1 + a] * src[a * NC];
    t1[i] = s;
  }
  __syncthreads();
  for (int i = tid; i < N1 * Q * Q * NC; i += kThreads) {
    const int col = i % NC, qx = (i / NC) % Q, qy = (i / (NC * Q)) % Q, c = i / (NC * Q * Q);
    const double* src = t1 + (c * N1 * Q + qx) * NC + col;
    double s = 0.0;
#pragma unroll
    for (int b = 0; b < N1; ++b) s += A[qy * N1 + b] * src[b * Q * NC];
    t2[i] = s;
  }
  __syncthreads();
  for (int i = tid; i < Q * Q * Q * NC; i += kThreads) {
    const int col = i % NC, qxy = (i / NC) % (Q * Q), qz = i / (NC * Q * Q);
    const double* src = t2 + qxy * NC + col;
    double s = 0.0;
#pragma unroll
    for (int c = 0; c < N1; ++c) s += A[qz * N1 + c] * src[c * Q * Q * NC];
    out[i] = s;
  }
  __syncthreads();
}

// Transpose: in [Q][Q][Q][NC] -> out [N1][N1][N1][NC] (integration against N).
template <int N1, int Q, int NC>
__device__ void tp_integrate(const double* A, const double* in, double* t1, double* t2,
                             double* out) {
  const int tid = threadIdx.x;
  for (int i = tid; i < Q * Q * N1 * NC; i += kThreads) {  // t1[qz][qy][a][col]
    const int col = i % NC, a = (i / NC) % N1, qzy = i / (NC * N1);
    const double* src = in + qzy * Q * NC + col;
    double s = 0.0;
#pragma unroll
    for (int qx = 0; qx < Q; ++qx) s += A[qx * N1 + a] * src[qx * NC];
    t1[i] = s;
  }
  __syncthreads();
  for (int i = tid; i < Q * N1 * N1 * NC; i += kThreads) {  // t2[qz][b][a][col]
    const int col = i % NC, a = (i / NC) % N1, b = (i / (NC * N1)) % N1, qz = i / (NC * N1 * N1);
    const double* src = t1 + (qz * Q * N1 + a) * NC + col;
    double s = 0.0;
#pragma unroll
    for (int qy = 0; qy < Q; ++qy) s += A[qy * N1 + b] * src[qy * N1 * NC];
    t2[i] = s;
  }
  __syncthreads();
  for (int i = tid; i < N1 * N1 * N1 * NC; i += kThreads) {  // out[c][b][a][col]
    const int col = i % NC, ba = (i / NC) % (N1 * N1), c = i / (NC * N1 * N1);
    const double* src = t2 + ba * NC + col;
    double s = 0.0;
#pragma unroll
    for (int qz = 0; qz < Q; ++qz) s += A[qz * N1 + c] * src[qz * N1 * N1 * NC];
    out[i] = s;
  }
  __syncthreads();
}

template <int N1, int Q, int NC>
struct TpScratch {
  static constexpr int kIn = (N1 * N1 * N1 > Q * Q * Q ? N1 * N1 * N1 : Q * Q * Q) * NC;
  static constexpr int kT1 = (N1 * N1 * Q > Q * Q * N1 ? N1 * N1 * Q : Q * Q * N1) * NC;
  static constexpr int kT2 = (N1 * Q * Q > Q * N1 * N1 ? N1 * Q * Q : Q * N1 * N1) * NC;
  static constexpr int kOut = kIn;
};

// -------------------------------------------------------------- density
template <int P, int NC>
__global__ __launch_bounds__(kThreads) void k_density(Geo g, const double* __restrict__ Lq,
                                                      const double* __restrict__ X,
                                                      const double* __restrict__ S, int B,
                                                      const double* __restrict__ occ,
                                                      double* __restrict__ rho) {
  constexpr int N1 = P + 1, Q = P + 3, NE = ne_of(P), NQ = Q * Q * Q;
  typedef TpScratch<N1, Q, NC> Sz;
  __shared__ double A[Q * N1];
  __shared__ double sin_[Sz::kIn], t1[Sz::kT1], t2[Sz::kT2], sout[Sz::kOut];
  __shared__ double acc[NQ];
  __shared__ int64_t nodes[NE];
  const int64_t e = blockIdx.x;
  const int64_t cx = e % g.nc, cy = (e / g.nc) % g.nc, cz = e / ((int64_t)g.nc * g.nc);
  const int tid = threadIdx.x;
  for (int i = tid; i < Q * N1; i += kThreads) A[i] = Lq[i];
  for (int l = tid; l < NE; l += kThreads) nodes[l] = cell_node(g, cx, cy, cz, l);
  for (int q = tid; q < NQ; q += kThreads) acc[q] = 0.0;
  __syncthreads();
  for (int j0 = 0; j0 < B; j0 += NC) {
    for (int i = tid; i < NE * NC; i += kThreads) {
      const int l = i / NC, k = i % NC, j = j0 + k;
      sin_[i] = j < B ? S[nodes[l]] * X[nodes[l] * B + j] : 0.0;
    }
    __syncthreads();
    tp_eval<N1, Q, NC>(A, sin_, t1, t2, sout);
    for (int q = tid; q < NQ; q += kThreads) {
      double s = 0.0;
#pragma unroll
      for (int k = 0; k < NC; ++k) {
        const int j = j0 + k;
        if (j < B) { const double v = sout[q * NC + k]; s += 2.0 * occ[j] * v * v; }
      }
      acc[q] += s;
    }
    __syncthreads();
  }
  for (int q = tid; q < NQ; q += kThreads) rho[e * NQ + q] = acc[q];
}

// --------------------------------------------- quadrature cell operator
// Y += N^T diag(wq) N X on the cells of one colour (no write conflicts): the
// quadrature operator of an adjoint solve's right-hand side, whose order of sums is
// fixed as that of the solve's steps is (see k_cell_line).  8 launches, 2.18 ms at
// 121^3 nodes x 12 columns, once per solve; launch_quad_pairs takes 0.3 ms there.
template <int P, int NC>
__global__ __launch_bounds__(kThreads) void k_quad_operator(Geo g, const double* __restrict__ Lq,
                                                            const double* __restrict__ X, int B,
                                                            const double* __restrict__ wq,
                                                            double* __restrict__ Y, int colour,
                                                            int64_t nw) {
  constexpr int N1 = P + 1, Q = P + 3, NE = ne_of(P), NQ = Q * Q * Q;
  typedef TpScratch<N1, Q, NC> Sz;
  __shared__ double A[Q * N1];
  __shared__ double sin_[Sz::kIn], t1[Sz::kT1], t2[Sz::kT2], sout[Sz::kOut];
  __shared__ int64_t nodes[NE];
  const int64_t e = colour_cell(g, colour, blockIdx.x, nw);
  if (e < 0) return;
  const int64_t cx = e % g.nc, cy = (e / g.nc) % g.nc, cz = e / ((int64_t)g.nc * g.nc);
  const int tid = threadIdx.x;
  for (int i = tid; i < Q * N1; i += kThreads) A[i] = Lq[i];
  for (int l = tid; l < NE; l += kThreads) nodes[l] = cell_node(g, cx, cy, cz, l);
  __syncthreads();
  for (int j0 = 0; j0 < B; j0 += NC) {
    for (int i = tid; i < NE * NC; i += kThreads) {
      const int l = i / NC, j = j0 + i % NC;
      sin_[i] = j < B ? X[nodes[l] * B + j] : 0.0;
    }
    __syncthreads();
    tp_eval<N1, Q, NC>(A, sin_, t1, t2, sout);
    for (int i = tid; i < NQ * NC; i += kThreads) sout[i] *= wq[e * NQ + i / NC];
    __syncthreads();
    tp_integrate<N1, Q, NC>(A, sout, t1, t2, sin_);
    for (int i = tid; i < NE * NC; i += kThreads) {
      const int l = i / NC, j = j0 + i % NC;
      if (j < B) Y[nodes[l] * B + j] += sin_[i];
    }
    __syncthreads();
  }
}

// ------------------------------------------------------------ v_xc -> quad
// Child Q1 field (3 child nodes per parent axis) to the parent Gauss points.
template <int P>
__global__ __launch_bounds__(kThreads) void k_vxc_to_quad(Geo g, const double* __restrict__ Wq,
                                                          const double* __restrict__ pot,
                                                          const double* __restrict__ potBase,
                                                          double* __restrict__ veff) {
  constexpr int Q = P + 3, NQ = Q * Q * Q;
  typedef TpScratch<3, Q, 1> Sz;
  __shared__ double A[Q * 3];
  __shared__ double sin_[Sz::kIn], t1[Sz::kT1], t2[Sz::kT2], sout[Sz::kOut];
  const int64_t e = blockIdx.x;
  const int64_t cx = e % g.nc, cy = (e / g.nc) % g.nc, cz = e / ((int64_t)g.nc * g.nc);
  const int tid = threadIdx.x;
  for (int i = tid; i < Q * 3; i += kThreads) A[i] = Wq[i];
  for (int i = tid; i < 27; i += kThreads) {
    const int a = i % 3, b = (i / 3) % 3, c = i / 9;
    sin_[i] = pot[((2 * cz + c) * g.NV1 + (2 * cy + b)) * (int64_t)g.NV1 + (2 * cx + a)];
  }
  __syncthreads();
  tp_eval<3, Q, 1>(A, sin_, t1, t2, sout);
  for (int q = tid; q < NQ; q += kThreads) veff[e * NQ + q] = potBase[e * NQ + q] + sout[q];
}

// ------------------------------------------------------------------ force
// S(q) = sum_j Psi_j(q) P_j(q) at Q points per axis (child: Q=4 via Ac; parent:
// Q=p+3 via Lq), then force[child node] += sum_q W(q) N^child(q) S(q).
template <int P, int Q, int NC>
__global__ __launch_bounds__(kThreads) void k_force(Geo g, const double* __restrict__ Aeval,
                                                    const double* __restrict__ Wchild,
                                                    const double* __restrict__ Psi,
                                                    const double* __restrict__ Pv, int B,
                                                    double jxwChild,
                                                    const double* __restrict__ jxwParent,
                                                    double* __restrict__ force, int colour,
                                                    int64_t nw) {
  constexpr int N1 = P + 1, NE = ne_of(P), NQ = Q * Q * Q, H = NC / 2;
  typedef TpScratch<N1, Q, NC> Sz;
  __shared__ double A[Q * N1];
  __shared__ double Wc[Q * 3];
  __shared__ double sin_[Sz::kIn], t1[Sz::kT1], t2[Sz::kT2], sout[Sz::kOut];
  __shared__ double Sq[NQ];
  __shared__ double u1[3 * 3 * Q], u2[3 * 3 * 3];
  __shared__ double v1[Q * Q * 3];
  __shared__ int64_t nodes[NE];
  const int64_t e = colour_cell(g, colour, blockIdx.x, nw);
  if (e < 0) return;
  const int64_t cx = e % g.nc, cy = (e / g.nc) % g.nc, cz = e / ((int64_t)g.nc * g.nc);
  const int tid = threadIdx.x;
  for (int i = tid; i < Q * N1; i += kThreads) A[i] = Aeval[i];
  for (int i = tid; i < Q * 3; i += kThreads) Wc[i] = Wchild[i];
  for (int l = tid; l < NE; l += kThreads) nodes[l] = cell_node(g, cx, cy, cz, l);
  for (int q = tid; q < NQ; q += kThreads) Sq[q] = 0.0;
  __syncthreads();
  for (int j0 = 0; j0 < B; j0 += H) {
    for (int i = tid; i < NE * NC; i += kThreads) {
      const int l = i / NC, k = i % NC, j = j0 + (k % H);
      double v = 0.0;
      if (j < B) v = (k < H) ? Psi[nodes[l] * B + j] : Pv[nodes[l] * B + j];
      sin_[i] = v;
    }
    __syncthreads();
    tp_eval<N1, Q, NC>(A, sin_, t1, t2, sout);
    for (int q = tid; q < NQ; q += kThreads) {
      double s = 0.0;
#pragma unroll
      for (int k = 0; k < H; ++k) s += sout[q * NC + k] * sout[q * NC + H + k];
      Sq[q] += s;
    }
    __syncthreads();
  }
  for (int q = tid; q < NQ; q += kThreads) Sq[q] *= jxwParent ? jxwParent[q] : jxwChild;
  __syncthreads();
  // integrate against the child basis: out[c][b][a] (3 child nodes per axis)
  for (int i = tid; i < Q * Q * 3; i += kThreads) {  // v1[qz][qy][a]
    const int a = i % 3, qzy = i / 3;
    double s = 0.0;
    for (int qx = 0; qx < Q; ++qx) s += Wc[qx * 3 + a] * Sq[qzy * Q + qx];
    v1[i] = s;
  }
  __syncthreads();
  for (int i = tid; i < Q * 9; i += kThreads) {  // u1[qz][b][a]
    const int a = i % 3, b = (i / 3) % 3, qz = i / 9;
    double s = 0.0;
    for (int qy = 0; qy < Q; ++qy) s += Wc[qy * 3 + b] * v1[(qz * Q + qy) * 3 + a];
    u1[i] = s;
  }
  __syncthreads();
  for (int i = tid; i < 27; i += kThreads) {
    const int ba = i % 9, c = i / 9;
    double s = 0.0;
    for (int qz = 0; qz < Q; ++qz) s += Wc[qz * 3 + c] * u1[qz * 9 + ba];
    u2[i] = s;
  }
  __syncthreads();
  for (int i = tid; i < 27; i += kThreads) {
    const int a = i % 3, b = (i / 3) % 3, c = i / 9;
    force[((2 * cz + c) * g.NV1 + (2 * cy + b)) * (int64_t)g.NV1 + (2 * cx + a)] += u2[i];
  }
}

// --------------------------------------------------------- vector kernels
// Y = beta Y + ns[n] (a ca[j] X + b cb[j] Z + c cc[j] W); null coefficient
// pointers read as 1, null operands as 0.  N * B < 2^32 (checked by the host).
template <typename T>
__global__ void k_lincomb(uint32_t NB, uint32_t B, T* __restrict__ Y, double beta,
                          const T* __restrict__ X, double a, const double* __restrict__ ca,
                          const T* __restrict__ Z, double b, const double* __restrict__ cb,
                          const T* __restrict__ W, double c, const double* __restrict__ cc,
                          const double* __restrict__ ns) {
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < NB; i += gridDim.x * blockDim.x) {
    const uint32_t n = i / B, j = i - n * B;
    double v = 0.0;
    if (X) v = a * (ca ? ca[j] : 1.0) * (double)X[i];
    if (Z) v += b * (cb ? cb[j] : 1.0) * (double)Z[i];
    if (W) v += c * (cc ? cc[j] : 1.0) * (double)W[i];
    if (ns) v *= ns[n];
    if (beta != 0.0) v += beta * (double)Y[i];
    Y[i] = (T)v;
  }
}

// Y = a ca[j] X + b cb[j] Z with operands and result of different types
// (null coefficient pointers read as 1), in FP64 arithmetic and rounded once:
// the same expression as k_lincomb, so that a conversion pass before or after
// it is not needed.  Y may be X (each entry is read, then written, by one
// thread).  N * B < 2^32 (checked by the host).
template <typename TY, typename TX, typename TZ>
__global__ void k_lincomb_mixed(uint32_t NB, uint32_t B, TY* Y, const TX* X, double a,
                                const double* __restrict__ ca,
                                const TZ* __restrict__ Z, double b, const double* __restrict__ cb) {
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < NB; i += gridDim.x * blockDim.x) {
    const uint32_t n = i / B, j = i - n * B;
    double v = a * (ca ? ca[j] : 1.0) * (double)X[i];
    v += b * (cb ? cb[j] : 1.0) * (double)Z[i];
    Y[i] = (TY)v;
  }
}

__global__ void k_scale_product(int64_t n, double* __restrict__ y, const float* __restrict__ a,
                                const double* __restrict__ b) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = (double)a[i] * b[i];
}
__global__ void k_d2f(int64_t n, float* __restrict__ y, const double* __restrict__ x) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    y[i] = (float)x[i];
}
__global__ void k_f2d(int64_t n, double* __restrict__ y, const float* __restrict__ x) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    y[i] = (double)x[i];
}

// Column-wise partial dot products.  Thread t of a block owns column t % B and
// strides over nodes; FP64 accumulation; block results reduced in LDS.
template <typename T>
__global__ __launch_bounds__(kThreads) void k_coldot(int64_t N, int B, const T* __restrict__ X,
                                                     const T* __restrict__ Y,
                                                     const double* __restrict__ w,
                                                     double* __restrict__ partial) {
  __shared__ double red[kThreads];
  const int tid = threadIdx.x;
  const int per = kThreads / B;  // nodes per block step (B <= 256)
  const int col = tid % B, off = tid / B;
  double s = 0.0;
  if (off < per) {
    for (int64_t n = (int64_t)blockIdx.x * per + off; n < N; n += (int64_t)gridDim.x * per) {
      const double x = (double)X[n * B + col], y = (double)Y[n * B + col];
      s += w ? w[n] * x * y : x * y;
    }
  }
  red[tid] = s;
  __syncthreads();
  if (tid < B) {
    double t = 0.0;
    for (int k = 0; k < per; ++k) t += red[k * B + tid];
    partial[(int64_t)blockIdx.x * B + tid] = t;
  }
}

__global__ __launch_bounds__(kThreads) void k_sum_partials(int nblk, int B,
                                                            const double* __restrict__ partial,
                                                            double* __restrict__ out) {
  __shared__ double red[kThreads];
  const int j = blockIdx.x;
  const double s = block_sum_col(partial, nblk, B, j, red);
  if (threadIdx.x == 0) out[j] = s;
}

// Sums of contiguous rows: out[j] = sum of partial[j nblk .. (j + 1) nblk).
__global__ __launch_bounds__(kRedThreads) void k_sum_rows(int nblk, const double* __restrict__ partial,
                                                           double* __restrict__ out) {
  __shared__ double red[kRedThreads / 64];
  const int j = blockIdx.x;
  const double s = block_sum_contig<kRedThreads>(partial + (int64_t)j * nblk, nblk, red);
  if (threadIdx.x == 0) out[j] = s;
}

// Gram partials: block (bx, by) accumulates the entries ij in
// [by * 256, by * 256 + 256) of G = X^T Y over the chunks of `rows` nodes
// bx, bx + gridDim.x, ..., whose rows of X and Y are staged in LDS (the loads
// of a chunk issued together).  Partials column-major, partial[ij nblk + bx],
// so that each entry's reduction reads contiguous memory.
__global__ __launch_bounds__(kThreads) void k_gram(int64_t N, int B, int rows,
                                                   const double* __restrict__ X,
                                                   const double* __restrict__ Y,
                                                   double* __restrict__ partial) {
  extern __shared__ double lds[];
  double* xs = lds;
  double* ys = lds + rows * B;
  const int tid = threadIdx.x;
  const int BB = B * B, RB = rows * B;
  const int ij = blockIdx.y * kThreads + tid;
  const int i = ij / B, j = ij % B;
  double acc = 0.0;
  for (int64_t n0 = (int64_t)blockIdx.x * rows; n0 < N; n0 += (int64_t)gridDim.x * rows) {
    const int cnt = (int)((N - n0) < rows ? (N - n0) : rows);
    const int ce = cnt * B;  // entries of this chunk (contiguous in X and Y)
    __syncthreads();
    // four entries per thread per round, their loads issued together
    for (int t0 = tid; t0 < RB; t0 += 4 * kThreads) {
      double xv[4], yv[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int t = t0 + u * kThreads;
        const bool ok = t < ce;
        const int64_t g = ok ? n0 * B + t : 0;
        xv[u] = X[g];
        yv[u] = Y[g];
        if (!ok) xv[u] = yv[u] = 0.0;
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int t = t0 + u * kThreads;
        if (t < RB) {
          xs[t] = xv[u];
          ys[t] = yv[u];
        }
      }
    }
    __syncthreads();
    if (ij < BB)
      for (int r = 0; r < cnt; ++r) acc += xs[r * B + i] * ys[r * B + j];
  }
  if (ij < BB) partial[(int64_t)ij * gridDim.x + blockIdx.x] = acc;
}

// Y = beta Y + ns[n] (X Q)[n]  (X != Y) over tiles of `rows` nodes: the
// tile's rows of X (contiguous) are staged in LDS with their loads issued
// together, then each thread forms the outputs t, t + 256, ... of the tile
// (node t / B, column t % B) from LDS, and the tile is written contiguously.
__global__ __launch_bounds__(kThreads) void k_right_mult(uint32_t N, uint32_t B, uint32_t rows,
                                                         const double* __restrict__ X,
                                                         const double* __restrict__ Q,
                                                         double* __restrict__ Y,
                                                         const double* __restrict__ ns,
                                                         double beta) {
  extern __shared__ double lds[];
  double* qs = lds;
  double* xt = lds + B * B;
  const uint32_t tid = threadIdx.x, RB = rows * B;
  for (uint32_t i = tid; i < B * B; i += kThreads) qs[i] = Q[i];
  for (uint32_t n0 = blockIdx.x * rows; n0 < N; n0 += gridDim.x * rows) {
    const uint32_t cnt = min(rows, N - n0), ce = cnt * B;
    const uint32_t base = n0 * B;  // N B < 2^32 (checked by the host)
    __syncthreads();  // the previous tile's outputs have read xt
    for (uint32_t t0 = tid; t0 < ce; t0 += 4 * kThreads) {
      double xv[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const uint32_t t = t0 + u * kThreads;
        xv[u] = X[t < ce ? base + t : base];
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const uint32_t t = t0 + u * kThreads;
        if (t < ce) xt[t] = xv[u];
      }
    }
    __syncthreads();
    for (uint32_t t = tid; t < ce; t += kThreads) {
      const uint32_t r = t / B, j = t - r * B;
      const double* xr = xt + r * B;
      double s = 0.0;
      for (uint32_t i = 0; i < B; ++i) s += xr[i] * qs[i * B + j];
      if (ns) s *= ns[n0 + r];
      Y[base + t] = beta != 0.0 ? beta * Y[base + t] + s : s;
    }
  }
}

template <typename T>
__global__ __launch_bounds__(kThreads) void k_residual(int64_t N, int B, const T* __restrict__ HX,
                                                       const T* __restrict__ X,
                                                       const double* __restrict__ ev,
                                                       double* __restrict__ partial) {
  __shared__ double red[kThreads];
  const int tid = threadIdx.x;
  const int per = kThreads / B;
  const int col = tid % B, off = tid / B;
  double s = 0.0;
  if (off < per) {
    const double lam = ev[col];
    for (int64_t n = (int64_t)blockIdx.x * per + off; n < N; n += (int64_t)gridDim.x * per) {
      const double r = (double)HX[n * B + col] - lam * (double)X[n * B + col];
      s += r * r;
    }
  }
  red[tid] = s;
  __syncthreads();
  if (tid < B) {
    double t = 0.0;
    for (int k = 0; k < per; ++k) t += red[k * B + tid];
    partial[(int64_t)blockIdx.x * B + tid] = t;
  }
}

__global__ void k_loss(int64_t nQ, int nq, const double* __restrict__ rho,
                       const double* __restrict__ rhoT, const double* __restrict__ w,
                       const double* __restrict__ veff, const double* __restrict__ jxw,
                       double* __restrict__ u, double* __restrict__ partial) {
  __shared__ double red[4][kThreads];
  const int tid = threadIdx.x;
  double s0 = 0, s1 = 0, s2 = 0, s3 = 0;
  for (int64_t q = blockIdx.x * (int64_t)kThreads + tid; q < nQ; q += (int64_t)gridDim.x * kThreads) {
    const double jw = jxw[q % nq];
    const double rd = rhoT[q] - 0.5 * rho[q];
    u[q] = rd * w[q];
    s0 += rd * rd * w[q] * jw;
    s1 += rd * rd * jw;
    s2 += fabs(rd * jw);
    s3 += veff[q] * rho[q] * jw;
  }
  red[0][tid] = s0; red[1][tid] = s1; red[2][tid] = s2; red[3][tid] = s3;
  __syncthreads();
  for (int st = kThreads / 2; st > 0; st >>= 1) {
    if (tid < st)
      for (int k = 0; k < 4; ++k) red[k][tid] += red[k][tid + st];
    __syncthreads();
  }
  if (tid < 4) partial[blockIdx.x * 4 + tid] = red[tid][0];
}

__global__ void k_zero_rows(uint32_t NB, uint32_t B, double* __restrict__ X,
                            const unsigned char* __restrict__ mask) {
  for (uint32_t t = blockIdx.x * blockDim.x + threadIdx.x; t < NB; t += gridDim.x * blockDim.x)
    if (mask[t / B]) X[t] = 0.0;
}


// Zeroes the rows of the boundary nodes of the mesh, found by arithmetic: a
// thread per entry of a boundary row, so only those rows are touched (a pass
// with a node mask looks at every node: 23.7 us at 121^3 nodes x 12 columns
// and 284 us at 161^3 x 80; with this kernel vmult went from 376 to 359 us
// and from 6492 to 6210 us there).
// Boundary nodes in order: the planes iz = 0 and iz = N1 - 1, then for each
// iz between them the ring of 4 (N1 - 1) nodes (rows iy = 0 and iy = N1 - 1,
// then the end nodes of the rows between).
__global__ __launch_bounds__(kThreads) void k_zero_boundary(uint32_t N1, uint32_t B, uint32_t nbn,
                                                            double* __restrict__ X) {
  const uint64_t tot = (uint64_t)nbn * B;
  for (uint64_t t = (uint64_t)blockIdx.x * kThreads + threadIdx.x; t < tot;
       t += (uint64_t)gridDim.x * kThreads) {
    uint32_t i = (uint32_t)(t / B);
    const uint32_t j = (uint32_t)(t - (uint64_t)i * B), pl = N1 * N1, ring = 4 * (N1 - 1);
    uint32_t ix, iy, iz;
    if (i < 2 * pl) {
      iz = i < pl ? 0 : N1 - 1;
      i = i < pl ? i : i - pl;
      iy = i / N1;
      ix = i - iy * N1;
    } else {
      i -= 2 * pl;
      iz = 1 + i / ring;
      i -= (iz - 1) * ring;
      if (i < 2 * N1) {
        iy = i < N1 ? 0 : N1 - 1;
        ix = i < N1 ? i : i - N1;
      } else {
        i -= 2 * N1;
        iy = 1 + i / 2;
        ix = (i & 1) ? N1 - 1 : 0;
      }
    }
    X[(((uint64_t)iz * N1 + iy) * N1 + ix) * B + j] = 0.0;
  }
}

// ------------------------------------------------------------- MINRES
// Per-column state st[k * B + j] (see MinresSlot); one thread per column.
__global__ __launch_bounds__(kThreads) void k_minres_start(int B, int nblk,
                                                            const double* __restrict__ partial,
                                                            const double* __restrict__ negEig,
                                                            double* __restrict__ st, int nq) {
  __shared__ double red[kThreads];
  const int j = blockIdx.x;
  const double s = block_sum_col(partial, nblk, B, j, red);
  __syncthreads();
  const double q2 = nq >= 2 ? block_sum_col(partial + (int64_t)nblk * B, nblk, B, j, red) : 0.0;
  if (threadIdx.x != 0) return;
  st[MS_Q2 * B + j] = q2;
  st[MS_Q3 * B + j] = 0.0;
  const double beta = sqrt(fmax(s, 0.0));
  st[MS_BETA * B + j] = beta;
  st[MS_OLDB * B + j] = 0.0;
  st[MS_DBAR * B + j] = 0.0;
  st[MS_EPSLN * B + j] = 0.0;
  st[MS_PHIBAR * B + j] = beta;
  st[MS_CS * B + j] = -1.0;
  st[MS_SN * B + j] = 0.0;
  st[MS_IT * B + j] = 0.0;
  st[MS_BETA1 * B + j] = beta;
  const bool done = !(beta > st[MS_TOL * B + j]);
  st[MS_DONE * B + j] = done ? 1.0 : 0.0;
  st[MS_CV * B + j] = done ? 0.0 : 1.0 / beta;
  st[MS_CVN * B + j] = st[MS_CV * B + j] * negEig[j];
  st[MS_CR1 * B + j] = 0.0;
}

__global__ __launch_bounds__(kThreads) void k_minres_alpha(int B, int nblk,
                                                            const double* __restrict__ partial,
                                                            double* __restrict__ st) {
  __shared__ double red[kThreads];
  const int j = blockIdx.x;
  const double s = block_sum_col(partial, nblk, B, j, red);
  if (threadIdx.x != 0) return;
  st[MS_ALFA * B + j] = s;
  const bool done = st[MS_DONE * B + j] != 0.0;
  st[MS_CA2 * B + j] = done ? 0.0 : -s / st[MS_BETA * B + j];
}

// alpha of a fused step: v.(H~ v) from the per-cell dots x_e.(H_e x_e)
// (x = S v the cell product's input) plus the node terms of the step's
// output, v.(cvn D r2 + cr1 r1) = cv (cvn Q2 + cr1 Q3) with v = cv D r2.
__global__ __launch_bounds__(kRedThreads) void k_minres_alpha_cell(int B, int ncell,
                                                                    const double* __restrict__ cd,
                                                                    double* __restrict__ st) {
  __shared__ double red[kRedThreads / 64];
  const int j = blockIdx.x;
  const double s = block_sum_contig<kRedThreads>(cd + (int64_t)j * ncell, ncell, red);
  if (threadIdx.x != 0) return;
  const double cv = st[MS_CV * B + j];
  const double a = s + cv * (st[MS_CVN * B + j] * st[MS_Q2 * B + j] +
                             st[MS_CR1 * B + j] * st[MS_Q3 * B + j]);
  st[MS_ALFA * B + j] = a;
  const bool done = st[MS_DONE * B + j] != 0.0;
  st[MS_CA2 * B + j] = done ? 0.0 : -a / st[MS_BETA * B + j];
}

// Lanczos bound of the spectrum with its scalars on the device (one host round trip
// for the k steps where dots read by the host took two per step: about 25 us each, a
// tenth of a small problem's evaluation).  r_j are the unscaled vectors, v_j = r_j inv_j;
// lan holds [k] alphas, [k] betas, then inv_j, inv_{j-1}, ca = -alpha inv_j and
// cb = -beta_{j-1} inv_{j-1}.
// r_0: the n-th number in (-1, 1) of the splitmix64 sequence from `seed`, 0 on the
// boundary, with the block partials of r_0 . r_0.
template <typename T>
__global__ __launch_bounds__(kThreads) void k_lan_start(uint32_t N, uint64_t seed,
                                                        const unsigned char* __restrict__ mask,
                                                        T* __restrict__ r,
                                                        double* __restrict__ partial) {
  __shared__ double red[kThreads / 64];
  double t = 0.0;
  for (uint32_t n = blockIdx.x * kThreads + threadIdx.x; n < N; n += gridDim.x * kThreads) {
    uint64_t z = seed + 0x9e3779b97f4a7c15ULL * ((uint64_t)n + 1);
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ULL;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebULL;
    z ^= z >> 31;
    const T v = (T)(mask[n] ? 0.0 : 2.0 * ((double)(z >> 11) * 0x1.0p-53) - 1.0);
    r[n] = v;
    t += (double)v * (double)v;
  }
  t = block_total<kThreads>(t, red);
  if (threadIdx.x == 0) partial[blockIdx.x] = t;
}
// j < 0: the norm of r_0; else beta_j = |r_{j+1}|.  A vanishing vector gets inv = 0: the
// steps after it are zero and the host cuts them off.
__global__ __launch_bounds__(kRedThreads) void k_lan_beta(int nblk, const double* __restrict__ partial,
                                                          int k, int j, double* __restrict__ lan) {
  __shared__ double red[kRedThreads / 64];
  const double b = sqrt(fmax(block_sum_contig<kRedThreads>(partial, nblk, red), 0.0));
  if (threadIdx.x != 0) return;
  double* c = lan + 2 * k;
  const double inv = c[0];
  if (j >= 0) lan[k + j] = b;
  c[0] = b > 0.0 ? 1.0 / b : 0.0;
  c[1] = inv;
  c[3] = j >= 0 ? -b * inv : 0.0;
}
__global__ __launch_bounds__(kRedThreads) void k_lan_alpha(int nblk, const double* __restrict__ partial,
                                                           int k, int j, double* __restrict__ lan) {
  __shared__ double red[kRedThreads / 64];
  const double a = block_sum_contig<kRedThreads>(partial, nblk, red);
  if (threadIdx.x != 0) return;
  lan[j] = a;
  lan[2 * k + 2] = -a * lan[2 * k];
}
// y <- y + ca r + cb rp, with the block partials of y . y
template <typename T>
__global__ __launch_bounds__(kThreads) void k_lan_update(uint32_t N, T* __restrict__ y,
                                                         const T* __restrict__ r,
                                                         const T* __restrict__ rp,
                                                         const double* __restrict__ c,
                                                         double* __restrict__ partial) {
  __shared__ double red[kThreads / 64];
  const double ca = c[2], cb = c[3];
  double t = 0.0;
  for (uint32_t n = blockIdx.x * kThreads + threadIdx.x; n < N; n += gridDim.x * kThreads) {
    double v = (double)y[n] + ca * (double)r[n];
    if (rp) v += cb * (double)rp[n];
    const T o = (T)v;
    y[n] = o;
    t += (double)o * (double)o;
  }
  t = block_total<kThreads>(t, red);
  if (threadIdx.x == 0) partial[blockIdx.x] = t;
}

// Partials of r.D r and (D r).(D r) per column (rows [0, nblk) and
// [nblk, 2 nblk) of partial): the start of a fused MINRES solve.
__global__ __launch_bounds__(kThreads) void k_minres_start_dots(int64_t N, int B,
                                                                const double* __restrict__ r,
                                                                const double* __restrict__ D,
                                                                double* __restrict__ partial) {
  __shared__ double red[2][kThreads];
  const int tid = threadIdx.x;
  const int per = kThreads / B;
  const int col = tid % B, off = tid / B;
  double s1 = 0.0, s2 = 0.0;
  if (off < per) {
    for (int64_t n = (int64_t)blockIdx.x * per + off; n < N; n += (int64_t)gridDim.x * per) {
      const double v = r[n * B + col], dv = D[n] * v;
      s1 += v * dv;
      s2 += dv * dv;
    }
  }
  red[0][tid] = s1;
  red[1][tid] = s2;
  __syncthreads();
  if (tid < B) {
    double t1 = 0.0, t2 = 0.0;
    for (int k = 0; k < per; ++k) {
      t1 += red[0][k * B + tid];
      t2 += red[1][k * B + tid];
    }
    partial[(int64_t)blockIdx.x * B + tid] = t1;
    partial[((int64_t)gridDim.x + blockIdx.x) * B + tid] = t2;
  }
}

// r_new = y + ca2 r2 (stored in rnew), partial dot(r_new, D r_new).  The
// preconditioned vector D r_new is not stored: the next operator
// application and update scale r_new by D on the fly.
template <typename T>
__global__ __launch_bounds__(kThreads) void k_minres_lanczos(int64_t N, int B,
                                                             const T* __restrict__ y,
                                                             const T* __restrict__ r2,
                                                             T* __restrict__ rnew,
                                                             const double* __restrict__ D,
                                                             const double* __restrict__ st,
                                                             double* __restrict__ partial) {
  __shared__ double red[kThreads];
  const int tid = threadIdx.x;
  const int per = kThreads / B;
  const int col = tid % B, off = tid / B;
  double s = 0.0;
  if (off < per) {
    const double c = st[MS_CA2 * B + col];
    for (int64_t n = (int64_t)blockIdx.x * per + off; n < N; n += (int64_t)gridDim.x * per) {
      const int64_t i = n * B + col;
      const double rn = (double)y[i] + c * (double)r2[i];
      const T rt = (T)rn;
      rnew[i] = rt;
      s += (double)rt * (D[n] * (double)rt);
    }
  }
  red[tid] = s;
  __syncthreads();
  if (tid < B) {
    double t = 0.0;
    for (int k = 0; k < per; ++k) t += red[k * B + tid];
    partial[(int64_t)blockIdx.x * B + tid] = t;
  }
}

__global__ __launch_bounds__(kRedThreads) void k_minres_givens(int B, int nblk,
                                                                const double* __restrict__ partial,
                                                                const double* __restrict__ negEig,
                                                                double* __restrict__ st, int nq,
                                                                double* __restrict__ hist) {
  __shared__ double red[3 * (kRedThreads / 64)];
  const int j = blockIdx.x;
  double s, q2 = 0.0, q3 = 0.0;
  if (nq >= 3) {  // fused steps: [k][column][block] partials, the three sums in one pass
    const double* p = partial + (int64_t)j * nblk;
    const int64_t row = (int64_t)B * nblk;
    double a[3][4] = {};  // in block_sum_contig's order
    int b = threadIdx.x;
    for (; b + 3 * kRedThreads < nblk; b += 4 * kRedThreads)
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int k = 0; k < 3; ++k) a[k][u] += p[k * row + b + u * kRedThreads];
    for (; b < nblk; b += kRedThreads)
#pragma unroll
      for (int k = 0; k < 3; ++k) a[k][0] += p[k * row + b];
    s = (a[0][0] + a[0][1]) + (a[0][2] + a[0][3]);
    q2 = (a[1][0] + a[1][1]) + (a[1][2] + a[1][3]);
    q3 = (a[2][0] + a[2][1]) + (a[2][2] + a[2][3]);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      s += __shfl_xor(s, o, 64);
      q2 += __shfl_xor(q2, o, 64);
      q3 += __shfl_xor(q3, o, 64);
    }
    constexpr int kW = kRedThreads / 64;
    const int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
      red[wave] = s;
      red[kW + wave] = q2;
      red[2 * kW + wave] = q3;
    }
    __syncthreads();
    s = q2 = q3 = 0.0;
#pragma unroll
    for (int w = 0; w < kW; ++w) {
      s += red[w];
      q2 += red[kW + w];
      q3 += red[2 * kW + w];
    }
  } else {
    s = block_sum_col<kRedThreads>(partial, nblk, B, j, red);
  }
  if (threadIdx.x != 0) return;
  double* S = st;
  S[MS_Q2 * B + j] = q2;
  S[MS_Q3 * B + j] = q3;
  if (S[MS_DONE * B + j] != 0.0) {
    S[MS_CWV * B + j] = 0.0; S[MS_CWW1 * B + j] = 0.0; S[MS_CWW * B + j] = 0.0;
    S[MS_CX * B + j] = 0.0; S[MS_CV * B + j] = 0.0; S[MS_CR1 * B + j] = 0.0;
    S[MS_CVN * B + j] = 0.0;
    if (hist)
      for (int k = 0; k < 4; ++k) hist[k * B + j] = 0.0;
    return;
  }
  const double oldb = S[MS_BETA * B + j];
  const double beta = sqrt(fmax(s, 0.0));
  const double alfa = S[MS_ALFA * B + j];
  const double cs = S[MS_CS * B + j], sn = S[MS_SN * B + j], dbar = S[MS_DBAR * B + j];
  const double oldeps = S[MS_EPSLN * B + j];
  const double delta = cs * dbar + sn * alfa;
  const double gbar = sn * dbar - cs * alfa;
  const double epsln = sn * beta;
  const double ndbar = -cs * beta;
  const double gamma = fmax(sqrt(gbar * gbar + beta * beta), 1e-300);
  const double ncs = gbar / gamma, nsn = beta / gamma;
  const double phibar0 = S[MS_PHIBAR * B + j];
  const double phi = ncs * phibar0, phibar = nsn * phibar0;
  S[MS_OLDB * B + j] = oldb;
  S[MS_BETA * B + j] = beta;
  S[MS_EPSLN * B + j] = epsln;
  S[MS_DBAR * B + j] = ndbar;
  S[MS_CS * B + j] = ncs;
  S[MS_SN * B + j] = nsn;
  S[MS_PHIBAR * B + j] = phibar;
  S[MS_CWV * B + j] = S[MS_CV * B + j] / gamma;  // v = cv D r: cv of this step
  S[MS_CWW1 * B + j] = -oldeps / gamma;
  S[MS_CWW * B + j] = -delta / gamma;
  S[MS_CX * B + j] = phi;
  S[MS_IT * B + j] += 1.0;
  const bool done = !(phibar > S[MS_TOL * B + j]) || beta == 0.0;
  S[MS_DONE * B + j] = done ? 1.0 : 0.0;
  S[MS_CV * B + j] = done ? 0.0 : 1.0 / beta;
  S[MS_CVN * B + j] = S[MS_CV * B + j] * negEig[j];
  S[MS_CR1 * B + j] = done ? 0.0 : -beta / oldb;
  if (hist) {  // this step's row for k_minres_batch
    hist[j] = S[MS_CWV * B + j];
    hist[B + j] = S[MS_CWW1 * B + j];
    hist[2 * B + j] = S[MS_CWW * B + j];
    hist[3 * B + j] = phi;
  }
}

// w_new = cwv D r + cww1 w1 + cww w  (written over w1);  x += cx w_new,
// where cwv D r = v / gamma, v = cv D r the step's Lanczos vector.
template <typename T, int VW>
__global__ void k_minres_update(uint32_t NB, uint32_t B, const T* __restrict__ r,
                                const double* __restrict__ D, T* __restrict__ w1,
                                const T* __restrict__ w, T* __restrict__ x,
                                const double* __restrict__ st) {
  // VW consecutive columns of one node per thread (B % VW == 0), so every
  // access is one VW-wide load or store
  const uint32_t NG = NB / VW;
  for (uint32_t gi = blockIdx.x * blockDim.x + threadIdx.x; gi < NG; gi += gridDim.x * blockDim.x) {
    const uint32_t i = gi * VW, n = i / B, j = i - n * B;
    T rv[VW], w1v[VW], wv[VW], xv[VW];
    double cwv[VW], cw1[VW], cww[VW], cx[VW];
    vload<T, VW>(r + i, rv);
    vload<T, VW>(w1 + i, w1v);
    vload<T, VW>(w + i, wv);
    vload<T, VW>(x + i, xv);
    vload<double, VW>(st + MS_CWV * B + j, cwv);
    vload<double, VW>(st + MS_CWW1 * B + j, cw1);
    vload<double, VW>(st + MS_CWW * B + j, cww);
    vload<double, VW>(st + MS_CX * B + j, cx);
    const double dn = D[n];
    T wo[VW], xo[VW];
#pragma unroll
    for (int v = 0; v < VW; ++v) {
      const double wn = cwv[v] * (dn * (double)rv[v]) + cw1[v] * (double)w1v[v] +
                        cww[v] * (double)wv[v];
      wo[v] = (T)wn;
      xo[v] = (T)((double)xv[v] + cx[v] * wn);
    }
    vstore<T, VW>(w1 + i, wo);
    vstore<T, VW>(x + i, xo);
  }
}

// The direction and solution updates of n <= kMinresBatch fused steps in one pass:
// for each step, with its Lanczos vector r_i and its coefficients hist[(4 i + k) B + j],
//   w_new = cwv D r_i + cww1 w + cww w1;  x += cx w_new;  (w, w1) <- (w1, w_new).
// Bound by HBM: n + 6 streams where n updates of their own move 5 n (r is read by the
// Lanczos recurrence anyway).  With them inside the gather a step moved 8 streams of
// the block, with batches of 8 it moves 4.75, for 5 more vectors of storage.  All of a
// thread's loads are issued before the first use; the coefficients come from LDS.
// place != nullptr: the newest Lanczos vector `last` is copied there (2 more streams),
// also where place is r_0, whose entry the thread has read by then.
template <int VW>
__global__ __launch_bounds__(kThreads) void k_minres_batch(uint32_t N, uint32_t B, int n,
                                                           MinresVectors rs,
                                                           const double* __restrict__ D,
                                                           double* __restrict__ w,
                                                           double* __restrict__ w1,
                                                           double* __restrict__ x,
                                                           const double* __restrict__ hist,
                                                           const double* last, double* place) {
  __shared__ double sh[kMinresBatch * 4 * kMaxCols];
  const uint32_t tid = threadIdx.x, nb = B / VW, per = kThreads / nb;
  for (uint32_t k = tid; k < 4u * n * B; k += kThreads) sh[k] = hist[k];
  __syncthreads();
  const uint32_t off = tid / nb, j0 = (tid % nb) * VW;
  if (off >= per) return;
  for (uint32_t node = blockIdx.x * per + off; node < N; node += gridDim.x * per) {
    const uint32_t i = node * B + j0;
    double a[VW], b[VW], xv[VW], r[kMinresBatch][VW];
    vload<double, VW>(w + i, a);
    vload<double, VW>(w1 + i, b);
    vload<double, VW>(x + i, xv);
#pragma unroll
    for (int k = 0; k < kMinresBatch; ++k)
      if (k < n) vload<double, VW>(rs.r[k] + i, r[k]);
    double lv[VW];
    if (place) vload<double, VW>(last + i, lv);
    const double dn = D[node];
#pragma unroll
    for (int k = 0; k < kMinresBatch; ++k) {
      if (k >= n) break;
      const double* c = sh + 4 * k * B + j0;
#pragma unroll
      for (int v = 0; v < VW; ++v) {
        const double wn = c[v] * (dn * r[k][v]) + c[B + v] * a[v] + c[2 * B + v] * b[v];
        a[v] = b[v];
        b[v] = wn;
        xv[v] += c[3 * B + v] * wn;
      }
    }
    vstore<double, VW>(w + i, a);
    vstore<double, VW>(w1 + i, b);
    vstore<double, VW>(x + i, xv);
    if (place) vstore<double, VW>(place + i, lv);
  }
}

__global__ void k_copy_done(int B, const double* __restrict__ st, int* __restrict__ flags) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j < B) flags[j] = st[MS_DONE * B + j] != 0.0 ? 1 : 0;
}


// dst[n][j] = src[n][off + j]
__global__ void k_copy_cols(int64_t N, int Bs, int off, int Bd, const double* __restrict__ src,
                            double* __restrict__ dst) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < N * Bd;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t n = i / Bd;
    dst[i] = src[n * Bs + off + (int)(i % Bd)];
  }
}

// dst[n][k] = src[n][idx[k]] (gather, Bd columns) or, with scatter,
// dst[n][idx[k]] = src[n][k] (Bs columns of src into Bd-wide dst).
__global__ void k_cols_by_index(int64_t N, int Bs, int Bd, int Bi, const int* __restrict__ idx,
                                const double* __restrict__ src, double* __restrict__ dst,
                                int scatter) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < N * Bi;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t n = i / Bi;
    const int k = (int)(i - n * Bi);
    if (scatter) dst[n * Bd + idx[k]] = src[n * Bs + k];
    else dst[n * Bd + k] = src[n * Bs + idx[k]];
  }
}

__global__ void k_mul_q(int64_t nQ, int nq, const double* __restrict__ u,
                        const double* __restrict__ jxw, double* __restrict__ out) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < nQ;
       i += (int64_t)gridDim.x * blockDim.x)
    out[i] = u[i] * jxw[i % nq];
}

// partial[blk][k] = sum_n w[n] X[n][i_k] Y[n][j_k]   (np <= 256)
__global__ __launch_bounds__(kThreads) void k_pairdot(int64_t N, int B, const double* __restrict__ X,
                                                      const double* __restrict__ Y,
                                                      const double* __restrict__ w,
                                                      const int* __restrict__ pairs, int np,
                                                      double* __restrict__ partial) {
  __shared__ double red[kThreads];
  const int tid = threadIdx.x;
  const int per = kThreads / np;
  const int k = tid % np, off = tid / np;
  double s = 0.0;
  if (off < per) {
    const int i = pairs[2 * k], j = pairs[2 * k + 1];
    for (int64_t n = (int64_t)blockIdx.x * per + off; n < N; n += (int64_t)gridDim.x * per)
      s += (w ? w[n] : 1.0) * X[n * B + i] * Y[n * B + j];
  }
  red[tid] = s;
  __syncthreads();
  if (tid < np) {
    double t = 0.0;
    for (int m = 0; m < per; ++m) t += red[m * np + tid];
    partial[(int64_t)blockIdx.x * np + tid] = t;
  }
}

// Sparse column combination of the adjoint's two ends, in one pass over T, psi
// and Y (Y may be T):
//   RHS:  Y[n][i] = S[n] (cc[i] T[n][i]) + q[n] sum_e coef[e] psi[n][idx[e]]
//   else: Y[n][i] = S[n] T[n][i]         +      sum_e coef[e] psi[n][idx[e]]
// over the entries e in [start[i], start[i + 1]) of column i; where S[n] = 0
// (the boundary) the T term is 0 whatever T holds and, with RHS, so is Y.  The
// matrix couples degenerate pairs only, a few entries per column, so this is
// bound by HBM (3 streams) where a dense product also spends N B^2 multiply-adds.
// The lists sit in LDS; a lane's psi entries lie in the node's row, which the
// neighbouring lanes read anyway.
template <int VW, bool RHS>
__global__ __launch_bounds__(kThreads) void k_pair_combine(
    uint32_t NG, uint32_t B, const double* T, const double* __restrict__ S,
    const double* __restrict__ q, const double* __restrict__ psi, const double* __restrict__ cc,
    const double* __restrict__ coef_g, const int* __restrict__ list, uint32_t nnz, double* Y) {
  extern __shared__ double lds[];
  double* coef = lds;
  int* start = reinterpret_cast<int*>(lds + nnz);
  const int* idx = start + B + 1;
  for (uint32_t i = threadIdx.x; i < nnz; i += kThreads) coef[i] = coef_g[i];
  for (uint32_t i = threadIdx.x; i < B + 1 + nnz; i += kThreads) start[i] = list[i];
  __syncthreads();
  const uint32_t nb = B / VW;
  for (uint32_t gi = blockIdx.x * kThreads + threadIdx.x; gi < NG; gi += gridDim.x * kThreads) {
    const uint32_t n = gi / nb, j0 = (gi - n * nb) * VW, i = gi * VW;
    const double s = S[n];
    double t[VW], y[VW];
    vload<double, VW>(T + i, t);
    const double* pr = psi + (size_t)n * B;
#pragma unroll
    for (int v = 0; v < VW; ++v) {
      double a = 0.0;
      for (int e = start[j0 + v]; e < start[j0 + v + 1]; ++e) a += coef[e] * pr[idx[e]];
      if constexpr (RHS) y[v] = s == 0.0 ? 0.0 : q[n] * a + s * (cc[j0 + v] * t[v]);
      else y[v] = (s == 0.0 ? 0.0 : s * t[v]) + a;
    }
    vstore<double, VW>(Y + i, y);
  }
}

// Attainable FMA rate: `CH` independent multiply-add chains per thread,
// `iters` rounds, one store per thread (out holds one value per thread).
template <typename T, int CH>
__global__ __launch_bounds__(kThreads) void k_fma_probe(T* __restrict__ out, T a, T b, int iters) {
  T acc[CH];
#pragma unroll
  for (int c = 0; c < CH; ++c) acc[c] = (T)(threadIdx.x + c);
  for (int i = 0; i < iters; ++i) {
#pragma unroll
    for (int c = 0; c < CH; ++c) acc[c] = acc[c] * a + b;
  }
  T s = 0;
#pragma unroll
  for (int c = 0; c < CH; ++c) s += acc[c];
  out[(size_t)blockIdx.x * kThreads + threadIdx.x] = s;
}

inline int grid_for(int64_t n) {
  int64_t g = (n + kThreads - 1) / kThreads;
  if (g > 8192) g = 8192;
  if (g < 1) g = 1;
  return (int)g;
}

}  // namespace

// ============================================================== launchers
int64_t hamiltonian_tile_elems(int p) { return (int64_t)ntiles_of(p) * 256; }

void launch_build_hamiltonian(const Geo& g, const DevTables& t, double hh, const double* veff,
                              const double* jxw, double* h64, float* h32, hipStream_t s) {
  dim3 grid((unsigned)g.ncell), block(kThreads);
  switch (g.p) {
    case 2: k_build_h<2><<<grid, block, 0, s>>>(g, t.Lq.p, t.M1.p, t.D1.p, hh, veff, jxw, h64, h32); break;
    case 3: k_build_h<3><<<grid, block, 0, s>>>(g, t.Lq.p, t.M1.p, t.D1.p, hh, veff, jxw, h64, h32); break;
    case 4: k_build_h<4><<<grid, block, 0, s>>>(g, t.Lq.p, t.M1.p, t.D1.p, hh, veff, jxw, h64, h32); break;
    case 5: k_build_h<5><<<grid, block, 0, s>>>(g, t.Lq.p, t.M1.p, t.D1.p, hh, veff, jxw, h64, h32); break;
    default: throw Error(IDFT_EINVAL, "degree not supported by the HIP kernels (2..5)");
  }
  IDFT_HIP(hipGetLastError());
}

// Columns per work-group (2, 4 or 8: 40.7 KB of LDS at 8, p = 5) of the line-by-line
// kernel of the FP64 MINRES steps, one column per item; the plane kernel takes any
// block width in one way.
bool sf_cols_supported(int cols, bool) { return cols == 2 || cols == 4 || cols == 8; }
bool sf_vc_supported(int cols, int vc, bool fp64) {
  return sf_cols_supported(cols, fp64) && vc == 1;
}

static const double* sf_eo_table(int p);

template <typename T, typename TV, int P, bool XN, bool KIN>
static void cell_plane(const Geo& g, T hq, const T* W, uint32_t wstride,
                       const typename PlaneScale<T, XN>::type* S, const TV* X, int ldx,
                       const double* xcol, T* Yc, int B, double* dotp, hipStream_t s) {
  constexpr int NS = PlaneLanes<P>::NS;
  check_u32(cell_scratch_elems(g, B));
  const uint32_t nslot = (uint32_t)(g.ncell * B);
  const uint32_t nwave = (nslot + NS - 1) / NS;
  const FastDiv divB = make_fastdiv((uint32_t)std::max(B, 2));
  k_cell_plane<T, TV, P, XN, KIN><<<8 * ((nwave + 7) / 8), 64, 0, s>>>(
      g, hq, W, wstride, S, X, (uint32_t)ldx, xcol, Yc, (uint32_t)B, divB, nslot, dotp,
      sf_eo_table(P));
}

template <int P, int CG>
static void cell_line(const Geo& g, const CellOp<double>& op, const double* S, const double* X,
                      const double* xn, const double* xcol, double* Yc, int B, double* dotp,
                      hipStream_t s) {
  check_u32(cell_scratch_elems(g, B));
  const int64_t npair = g.ncell * ((B + CG - 1) / CG);
  check_u32(8 * ((npair + 7) / 8));
  k_cell_line<P, CG><<<(unsigned)(8 * ((npair + 7) / 8)), kThreads, 0, s>>>(
      g, op.kin_scale, op.W, S, X, xn, xcol, Yc, B, dotp, sf_eo_table(P));
}

template <typename T, typename TV, int P>
static void cell_sf_p(const Geo& g, const CellOp<T>& op, const T* S, const TV* X,
                      const double* xn, const double* sxn, const double* xcol, T* Yc, int B,
                      int cg, int vc, double* dotp, hipStream_t s) {
  if (!op.W) throw Error(IDFT_ESTATE, "quadrature weights of the cell operator not set");
  if (!sf_vc_supported(cg, vc, std::is_same<T, double>::value))
    throw Error(IDFT_EINVAL, "shape not supported by the sum-factorised kernel");
  check_u32(g.N * B);
  const T hq = (T)op.kin_scale;
  constexpr uint32_t nq = (P + 3) * (P + 3) * (P + 3);
  // per-cell dots only with node-scaled inputs (the MINRES steps)
  if (dotp && !xn) throw Error(IDFT_EINVAL, "per-cell dots need a node-scaled input");
  // node-scaled inputs (MINRES) come as FP64 vectors; FP32 vectors never
  // carry a node scale.  In FP64 they take the line-by-line kernel, whose order of
  // sums a solve keeps; FP32 products decide no iterate to 64-bit rounding (the
  // sweeps that refine it do), and the plane kernel is 1.1 to 4 times faster there.
  if constexpr (std::is_same<T, double>::value) {
    if (xn) {
      switch (cg) {
        case 2: cell_line<P, 2>(g, op, S, X, xn, xcol, Yc, B, dotp, s); break;
        case 4: cell_line<P, 4>(g, op, S, X, xn, xcol, Yc, B, dotp, s); break;
        default: cell_line<P, 8>(g, op, S, X, xn, xcol, Yc, B, dotp, s); break;
      }
      return;
    }
  } else if constexpr (std::is_same<TV, double>::value) {
    if (xn) {
      if (!sxn) throw Error(IDFT_EINVAL, "node-scaled input without the product of its scales");
      cell_plane<T, TV, P, true, true>(g, hq, op.W, nq, sxn, X, B, xcol, Yc, B, dotp, s);
      return;
    }
  } else {
    if (xn) throw Error(IDFT_EINVAL, "node-scaled input needs FP64 vectors");
  }
  cell_plane<T, TV, P, false, true>(g, hq, op.W, nq, S, X, B, xcol, Yc, B, nullptr, s);
}

template <typename T, typename TV, int P>
static void cell_gemm_p(const Geo& g, const CellOp<T>& op, const T* S, const TV* X,
                        const double* xn, const double* sxn, const double* xcol, T* Yc, int B,
                        const GemmShape& shape, hipStream_t s, double* dotp = nullptr) {
  if (shape.kernel == CK_SUM_FACTOR) {
    cell_sf_p<T, TV, P>(g, op, S, X, xn, sxn, xcol, Yc, B, shape.vectors_per_tile,
                        shape.cells_per_wg, dotp, s);
    return;
  }
  if (dotp) throw Error(IDFT_EINVAL, "per-cell dots need the sum-factorised cell product");
  const T* H = op.H;
  if (!H) throw Error(IDFT_ESTATE, "stored cell matrices not built");
  const int vt = std::min(shape.vectors_per_tile, ((B + 15) / 16) * 16);
  const int nct = std::max(1, std::min(5, vt / 16));
  const int cpw = std::max(1, shape.cells_per_wg);
  const int64_t nwg = (g.ncell + cpw - 1) / cpw;
  dim3 grid((unsigned)(8 * ((nwg + 7) / 8)), (unsigned)((B + 16 * nct - 1) / (16 * nct))),
      block(kThreads);
  if (shape.kernel == CK_TILE_PASS && nct <= (std::is_same<T, float>::value ? 2 : 1)) {
    const dim3 block2(kSymmThreads);
    if (nct == 1) k_cell_symm<T, TV, P, 1><<<grid, block2, 0, s>>>(g, H, S, X, xn, xcol, Yc, B, cpw);
    if constexpr (std::is_same<T, float>::value) {
      if (nct == 2)
        k_cell_symm<T, TV, P, 2><<<grid, block2, 0, s>>>(g, H, S, X, xn, xcol, Yc, B, cpw);
    }
    return;
  }
  switch (nct) {
    case 1: k_cell_gemm<T, TV, P, 1><<<grid, block, 0, s>>>(g, H, S, X, xn, xcol, Yc, B, cpw); break;
    case 2: k_cell_gemm<T, TV, P, 2><<<grid, block, 0, s>>>(g, H, S, X, xn, xcol, Yc, B, cpw); break;
    case 3: k_cell_gemm<T, TV, P, 3><<<grid, block, 0, s>>>(g, H, S, X, xn, xcol, Yc, B, cpw); break;
    case 4: k_cell_gemm<T, TV, P, 4><<<grid, block, 0, s>>>(g, H, S, X, xn, xcol, Yc, B, cpw); break;
    case 5: k_cell_gemm<T, TV, P, 5><<<grid, block, 0, s>>>(g, H, S, X, xn, xcol, Yc, B, cpw); break;
  }
}

// Device addresses of the even-odd tables kEo2..kEo5, per device, set by
// upload_sf_constants (once per device, before any cell product there).
static std::atomic<const double*> g_eo_table[64][4];

void upload_sf_constants() {
  static std::mutex mu;
  static bool done[64] = {};
  int dev = 0;
  IDFT_HIP(hipGetDevice(&dev));
  if (dev < 0 || dev >= 64) throw Error(IDFT_EHIP, "device index out of range");
  std::lock_guard<std::mutex> lk(mu);
  if (done[dev]) return;
  static constexpr EoTable<2> t2 = make_eo_table<2>();
  static constexpr EoTable<3> t3 = make_eo_table<3>();
  static constexpr EoTable<4> t4 = make_eo_table<4>();
  static constexpr EoTable<5> t5 = make_eo_table<5>();
  IDFT_HIP(hipMemcpyToSymbol(HIP_SYMBOL(kEo2), &t2, sizeof(t2), 0, hipMemcpyHostToDevice));
  IDFT_HIP(hipMemcpyToSymbol(HIP_SYMBOL(kEo3), &t3, sizeof(t3), 0, hipMemcpyHostToDevice));
  IDFT_HIP(hipMemcpyToSymbol(HIP_SYMBOL(kEo4), &t4, sizeof(t4), 0, hipMemcpyHostToDevice));
  IDFT_HIP(hipMemcpyToSymbol(HIP_SYMBOL(kEo5), &t5, sizeof(t5), 0, hipMemcpyHostToDevice));
  void* a[4] = {};
  IDFT_HIP(hipGetSymbolAddress(&a[0], HIP_SYMBOL(kEo2)));
  IDFT_HIP(hipGetSymbolAddress(&a[1], HIP_SYMBOL(kEo3)));
  IDFT_HIP(hipGetSymbolAddress(&a[2], HIP_SYMBOL(kEo4)));
  IDFT_HIP(hipGetSymbolAddress(&a[3], HIP_SYMBOL(kEo5)));
  for (int k = 0; k < 4; ++k) g_eo_table[dev][k].store(static_cast<const double*>(a[k]));
  done[dev] = true;
}

// The even-odd table of degree p on the current device.
static const double* sf_eo_table(int p) {
  int dev = 0;
  IDFT_HIP(hipGetDevice(&dev));
  const double* t = (dev >= 0 && dev < 64 && p >= 2 && p <= 5) ? g_eo_table[dev][p - 2].load()
                                                                : nullptr;
  if (!t) throw Error(IDFT_ESTATE, "sum-factorised tables not uploaded on this device");
  return t;
}

int64_t cell_scratch_elems(const Geo& g, int B) { return g.ncell * (int64_t)ne_of(g.p) * B; }

// Columns per gather thread: 16-byte vectors of the node-major rows where B
// allows it.
static int gather_vw(int B, int vbytes) {
  const int w = 16 / vbytes;
  if (B % w == 0) return w;
  return B % 2 == 0 ? 2 : 1;
}

// Gather grid: blocks of R chunks of kThreads / (B / VW) nodes each, with
// R = `rows_req` if positive, else chosen so that the grid has at most about
// kGatherBlocks blocks.
static void gather_grid(const Geo& g, int B, int vw, int rows_req, unsigned& gx, unsigned& gy,
                        uint32_t& R) {
  const int per = kThreads / (B / vw);
  const int64_t chunks = (g.N + per - 1) / per;
  int64_t r = rows_req > 0 ? rows_req : (chunks + kGatherBlocks - 1) / kGatherBlocks;
  if (r < 1) r = 1;
  R = (uint32_t)r;
  gx = (unsigned)((chunks + r - 1) / r);
  gy = 1;
}

int gather_blocks(const Geo& g, int B, int rows, int vbytes) {
  unsigned gx, gy;
  uint32_t R;
  gather_grid(g, B, gather_vw(B, vbytes), rows, gx, gy, R);
  return (int)(gx * gy);
}

template <typename T>
void launch_cell_gemm(const Geo& g, const CellOp<T>& op, const T* S, const T* X,
                      const double* xcol, T* Yc, int B, const GemmShape& shape, hipStream_t s) {
  if (B < 1 || B > kMaxCols) throw Error(IDFT_EINVAL, "block width out of range");
  switch (g.p) {
    case 2: cell_gemm_p<T, T, 2>(g, op, S, X, nullptr, nullptr, xcol, Yc, B, shape, s); break;
    case 3: cell_gemm_p<T, T, 3>(g, op, S, X, nullptr, nullptr, xcol, Yc, B, shape, s); break;
    case 4: cell_gemm_p<T, T, 4>(g, op, S, X, nullptr, nullptr, xcol, Yc, B, shape, s); break;
    case 5: cell_gemm_p<T, T, 5>(g, op, S, X, nullptr, nullptr, xcol, Yc, B, shape, s); break;
    default: throw Error(IDFT_EINVAL, "degree not supported by the HIP kernels (2..5)");
  }
  IDFT_HIP(hipGetLastError());
}
template void launch_cell_gemm<float>(const Geo&, const CellOp<float>&, const float*,
                                      const float*, const double*, float*, int,
                                      const GemmShape&, hipStream_t);
template void launch_cell_gemm<double>(const Geo&, const CellOp<double>&, const double*,
                                       const double*, const double*, double*, int,
                                       const GemmShape&, hipStream_t);

template <typename T, typename TV>
int launch_cell_apply(const Geo& g, const CellOp<T>& op, const T* Sg, const TV* S, const TV* X,
                      T* Yc, int B, const ApplyEpilogue<TV>& ep, const GemmShape& shape,
                      hipStream_t s) {
  if (B < 1 || B > kMaxCols) throw Error(IDFT_EINVAL, "block width out of range");
  switch (g.p) {
    case 2: cell_gemm_p<T, TV, 2>(g, op, Sg, X, ep.xn, ep.sxn, ep.xcol, Yc, B, shape, s); break;
    case 3: cell_gemm_p<T, TV, 3>(g, op, Sg, X, ep.xn, ep.sxn, ep.xcol, Yc, B, shape, s); break;
    case 4: cell_gemm_p<T, TV, 4>(g, op, Sg, X, ep.xn, ep.sxn, ep.xcol, Yc, B, shape, s); break;
    case 5: cell_gemm_p<T, TV, 5>(g, op, Sg, X, ep.xn, ep.sxn, ep.xcol, Yc, B, shape, s); break;
    default: throw Error(IDFT_EINVAL, "degree not supported by the HIP kernels (2..5)");
  }
  IDFT_HIP(hipGetLastError());
  check_u32(g.N * B);
  check_u32(cell_scratch_elems(g, B));
  const FastDiv divN1 = make_fastdiv((uint32_t)g.N1);
  unsigned gx, gy;
  uint32_t R;
  const int vw = gather_vw(B, (int)sizeof(TV));
  gather_grid(g, B, vw, shape.gather_rows, gx, gy, R);
  dim3 grid(gx, gy);
#define IDFT_GATHER(PP, VW)                                                                  \
  k_cell_gather<T, TV, PP, VW><<<grid, kThreads, 0, s>>>(                                    \
      g, divN1, (uint32_t)B, R, Yc, S, ep.Y, ep.alpha, ep.beta, ep.X, ep.a, ep.ca, ep.Z, ep.b,  \
      ep.cb,                                                                                  \
      ep.W, ep.c, ep.cc, X, ep.xn, ep.xcol, ep.V, ep.dot_partial)
#define IDFT_GATHER_P(PP)                                         \
  if (vw == 4) { if constexpr (sizeof(TV) == 4) IDFT_GATHER(PP, 4); } \
  else if (vw == 2) IDFT_GATHER(PP, 2);                           \
  else IDFT_GATHER(PP, 1);
  switch (g.p) {
    case 2: IDFT_GATHER_P(2); break;
    case 3: IDFT_GATHER_P(3); break;
    case 4: IDFT_GATHER_P(4); break;
    case 5: IDFT_GATHER_P(5); break;
  }
#undef IDFT_GATHER_P
#undef IDFT_GATHER
  IDFT_HIP(hipGetLastError());
  return (int)(gx * gy);
}
template int launch_cell_apply<float, float>(const Geo&, const CellOp<float>&, const float*,
                                             const float*, const float*, float*, int,
                                             const ApplyEpilogue<float>&, const GemmShape&,
                                             hipStream_t);
template int launch_cell_apply<double, double>(const Geo&, const CellOp<double>&,
                                               const double*, const double*, const double*,
                                               double*, int,
                                               const ApplyEpilogue<double>&, const GemmShape&,
                                               hipStream_t);
template int launch_cell_apply<float, double>(const Geo&, const CellOp<float>&, const float*,
                                              const double*, const double*, float*, int,
                                              const ApplyEpilogue<double>&, const GemmShape&,
                                              hipStream_t);

int quad_gather_blocks(const Geo& g, int wb, int vw) {
  unsigned gx, gy;
  uint32_t R;
  gather_grid(g, wb, vw, 0, gx, gy, R);
  return (int)std::min<unsigned>(gx, (unsigned)kMinresGatherBlocks);
}

void launch_quad_pairs(const Geo& g, const double* W, int64_t wstride, const double* Bv, int ldb,
                       int wb, double* Yc, const double* A, int lda, const double* asc, double* T2,
                       int ldt, const int* pairs, int np, DevBuf<double>& partial, double* out,
                       hipStream_t s) {
  if (wb < 1 || wb > kMaxCols || np < 0 || np > kThreads)
    throw Error(IDFT_EINVAL, "block or pair count out of range");
  check_u32(g.N);
  check_u32(cell_scratch_elems(g, wb));
  // two columns per 16-byte access where every row starts at an even column
  const int vw = wb % 2 == 0 && (np == 0 || lda % 2 == 0) && (!T2 || ldt % 2 == 0) ? 2 : 1;
  const int nblk = quad_gather_blocks(g, wb, vw);
  if (np) partial.resize((size_t)nblk * np);
  unsigned gx, gy;
  uint32_t R;
  gather_grid(g, wb, vw, 0, gx, gy, R);
  const FastDiv divN1 = make_fastdiv((uint32_t)g.N1);
#define IDFT_QG(PP, VW)                                                                         \
  k_quad_gather<PP, VW><<<nblk, kThreads, 0, s>>>(g, divN1, (uint32_t)wb, R, Yc, A, (uint32_t)lda, \
                                                  asc, T2, (uint32_t)ldt, pairs, (uint32_t)np,  \
                                                  partial.p)
#define IDFT_QP(PP)                                                \
  cell_plane<double, double, PP, false, false>(g, 0.0, W, (uint32_t)wstride, nullptr, Bv, ldb,  \
                                               nullptr, Yc, wb, nullptr, s);                    \
  IDFT_HIP(hipGetLastError());                                     \
  if (vw == 2) IDFT_QG(PP, 2);                                     \
  else IDFT_QG(PP, 1);
  switch (g.p) {
    case 2: IDFT_QP(2); break;
    case 3: IDFT_QP(3); break;
    case 4: IDFT_QP(4); break;
    case 5: IDFT_QP(5); break;
    default: throw Error(IDFT_EINVAL, "degree not supported by the HIP kernels (2..5)");
  }
#undef IDFT_QP
#undef IDFT_QG
  IDFT_HIP(hipGetLastError());
  if (np) {
    k_sum_rows<<<np, kRedThreads, 0, s>>>(nblk, partial.p, out);
    IDFT_HIP(hipGetLastError());
  }
}

void launch_pair_combine(int64_t N, int B, bool rhs, const double* T, const double* S,
                         const double* q, const double* psi, const double* cc, const double* coef,
                         const int* list, int nnz, double* Y, hipStream_t s) {
  check_u32(N * B);
  const size_t lds = (size_t)nnz * sizeof(double) + ((size_t)B + 1 + nnz) * sizeof(int);
  if (lds > 65536) throw Error(IDFT_EINVAL, "too many column pairs");
  const int vw = B % 2 == 0 ? 2 : 1;
  const uint32_t NG = (uint32_t)(N * B / vw);
  const int grid = grid_for(NG);
#define IDFT_PC(VW, RHS)                                                                      \
  k_pair_combine<VW, RHS><<<grid, kThreads, lds, s>>>(NG, (uint32_t)B, T, S, q, psi, cc, coef, \
                                                      list, (uint32_t)nnz, Y)
  if (rhs) { if (vw == 2) IDFT_PC(2, true); else IDFT_PC(1, true); }
  else { if (vw == 2) IDFT_PC(2, false); else IDFT_PC(1, false); }
#undef IDFT_PC
  IDFT_HIP(hipGetLastError());
}

template <typename T, typename TV>
void launch_cell_dot(const Geo& g, const CellOp<T>& op, const T* Sg, const TV* X, int B,
                     const double* xn, const double* sxn, const double* xcol, T* Yc,
                     double* cell_dots, const GemmShape& shape, hipStream_t s) {
  if (B < 1 || B > kMaxCols) throw Error(IDFT_EINVAL, "block width out of range");
  if (shape.kernel != CK_SUM_FACTOR || !cell_dots)
    throw Error(IDFT_EINVAL, "per-cell dots need the sum-factorised cell product");
  switch (g.p) {
    case 2: cell_gemm_p<T, TV, 2>(g, op, Sg, X, xn, sxn, xcol, Yc, B, shape, s, cell_dots); break;
    case 3: cell_gemm_p<T, TV, 3>(g, op, Sg, X, xn, sxn, xcol, Yc, B, shape, s, cell_dots); break;
    case 4: cell_gemm_p<T, TV, 4>(g, op, Sg, X, xn, sxn, xcol, Yc, B, shape, s, cell_dots); break;
    case 5: cell_gemm_p<T, TV, 5>(g, op, Sg, X, xn, sxn, xcol, Yc, B, shape, s, cell_dots); break;
    default: throw Error(IDFT_EINVAL, "degree not supported by the HIP kernels (2..5)");
  }
  IDFT_HIP(hipGetLastError());
}
template void launch_cell_dot<double, double>(const Geo&, const CellOp<double>&, const double*,
                                              const double*, int, const double*, const double*,
                                              const double*, double*, double*, const GemmShape&,
                                              hipStream_t);
template void launch_cell_dot<float, double>(const Geo&, const CellOp<float>&, const float*,
                                             const double*, int, const double*, const double*,
                                             const double*, float*, double*, const GemmShape&,
                                             hipStream_t);

template <typename TY>
int launch_minres_gather(const Geo& g, const TY* Yc, const double* S, const double* D,
                         const double* r2, const double* r1, double* rnew, int B,
                         const double* st, double* partial, int gather_rows, hipStream_t s) {
  if (B < 1 || B > kMaxCols) throw Error(IDFT_EINVAL, "block width out of range");
  check_u32(g.N * B);
  check_u32(cell_scratch_elems(g, B));
  const FastDiv divN1 = make_fastdiv((uint32_t)g.N1);
  unsigned gx, gy;
  uint32_t R;
  const int vw = gather_vw(B, (int)sizeof(double));
  gather_grid(g, B, vw, gather_rows, gx, gy, R);
  gx = std::min<unsigned>(gx, (unsigned)kMinresGatherBlocks);
#define IDFT_MG(PP, VW)                                                            \
  k_minres_gather<TY, double, PP, VW><<<dim3(gx), kThreads, 0, s>>>(               \
      g, divN1, (uint32_t)B, R, Yc, S, D, r2, r1, rnew, st, partial)
#define IDFT_MG_P(PP)   \
  if (vw == 2) IDFT_MG(PP, 2); \
  else IDFT_MG(PP, 1);
  switch (g.p) {
    case 2: IDFT_MG_P(2); break;
    case 3: IDFT_MG_P(3); break;
    case 4: IDFT_MG_P(4); break;
    case 5: IDFT_MG_P(5); break;
    default: throw Error(IDFT_EINVAL, "degree not supported by the HIP kernels (2..5)");
  }
#undef IDFT_MG_P
#undef IDFT_MG
  IDFT_HIP(hipGetLastError());
  return (int)gx;
}
template int launch_minres_gather<double>(const Geo&, const double*, const double*, const double*,
                                          const double*, const double*, double*, int,
                                          const double*, double*, int, hipStream_t);
template int launch_minres_gather<float>(const Geo&, const float*, const double*, const double*,
                                         const double*, const double*, double*, int,
                                         const double*, double*, int, hipStream_t);

template <typename T>
void launch_lincomb(int64_t N, int B, T* Y, double beta, const T* X, double a, const double* ca,
                    const T* Z, double b, const double* cb, const double* ns, hipStream_t s) {
  check_u32(N * B);
  k_lincomb<T><<<grid_for(N * B), kThreads, 0, s>>>((uint32_t)(N * B), (uint32_t)B, Y, beta, X, a,
                                                    ca, Z, b, cb, nullptr, 0.0, nullptr, ns);
  IDFT_HIP(hipGetLastError());
}
template <typename T>
void launch_lincomb3(int64_t N, int B, T* Y, double beta, const T* X, double a, const double* ca,
                     const T* Z, double b, const double* cb, const T* W, double c,
                     const double* cc, const double* ns, hipStream_t s) {
  check_u32(N * B);
  k_lincomb<T><<<grid_for(N * B), kThreads, 0, s>>>((uint32_t)(N * B), (uint32_t)B, Y, beta, X, a,
                                                    ca, Z, b, cb, W, c, cc, ns);
  IDFT_HIP(hipGetLastError());
}
template void launch_lincomb<float>(int64_t, int, float*, double, const float*, double,
                                    const double*, const float*, double, const double*,
                                    const double*, hipStream_t);
template void launch_lincomb<double>(int64_t, int, double*, double, const double*, double,
                                     const double*, const double*, double, const double*,
                                     const double*, hipStream_t);
template void launch_lincomb3<float>(int64_t, int, float*, double, const float*, double,
                                     const double*, const float*, double, const double*,
                                     const float*, double, const double*, const double*,
                                     hipStream_t);
template void launch_lincomb3<double>(int64_t, int, double*, double, const double*, double,
                                      const double*, const double*, double, const double*,
                                      const double*, double, const double*, const double*,
                                      hipStream_t);

void launch_lincomb_d2f(int64_t N, int B, float* Y, const double* X, double a, const double* ca,
                        const double* Z, double b, const double* cb, hipStream_t s) {
  check_u32(N * B);
  k_lincomb_mixed<float, double, double><<<grid_for(N * B), kThreads, 0, s>>>(
      (uint32_t)(N * B), (uint32_t)B, Y, X, a, ca, Z, b, cb);
  IDFT_HIP(hipGetLastError());
}
void launch_lincomb_df2d(int64_t N, int B, double* Y, const double* X, double a,
                         const double* ca, const float* Z, double b, const double* cb,
                         hipStream_t s) {
  check_u32(N * B);
  k_lincomb_mixed<double, double, float><<<grid_for(N * B), kThreads, 0, s>>>(
      (uint32_t)(N * B), (uint32_t)B, Y, X, a, ca, Z, b, cb);
  IDFT_HIP(hipGetLastError());
}
void launch_scale_product(int64_t n, double* y, const float* a, const double* b, hipStream_t s) {
  k_scale_product<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(n, y, a, b);
  IDFT_HIP(hipGetLastError());
}
void launch_convert_d2f(int64_t n, float* y, const double* x, hipStream_t s) {
  k_d2f<<<grid_for(n), kThreads, 0, s>>>(n, y, x);
  IDFT_HIP(hipGetLastError());
}
void launch_convert_f2d(int64_t n, double* y, const float* x, hipStream_t s) {
  k_f2d<<<grid_for(n), kThreads, 0, s>>>(n, y, x);
  IDFT_HIP(hipGetLastError());
}

int coldot_blocks(int64_t N, int B) {
  const int per = kThreads / B;
  int64_t g = (N + per - 1) / per;
  if (g > 1024) g = 1024;
  return (int)(g < 1 ? 1 : g);
}

template <typename T>
int launch_coldot_partial(int64_t N, int B, const T* X, const T* Y, const double* w,
                          double* partial, hipStream_t s) {
  if (B > kThreads) throw Error(IDFT_EINVAL, "block too wide for column reductions");
  const int nb = coldot_blocks(N, B);
  k_coldot<T><<<nb, kThreads, 0, s>>>(N, B, X, Y, w, partial);
  IDFT_HIP(hipGetLastError());
  return nb;
}
template int launch_coldot_partial<double>(int64_t, int, const double*, const double*,
                                           const double*, double*, hipStream_t);

void launch_sum_partials(int nblk, int B, const double* partial, double* out, hipStream_t s) {
  k_sum_partials<<<B, kThreads, 0, s>>>(nblk, B, partial, out);
  IDFT_HIP(hipGetLastError());
}

// Nodes per LDS tile of the Gram kernel: 64 for narrow blocks, about 2048
// entries per tile for wide ones.
static int tall_tile_rows(int B) { return std::max(8, std::min(64, 2048 / std::max(B, 1))); }

// Gram partial rows: enough work-groups to fill the CUs (up to 2048, 8 per
// CU), at most 2^21 partial values.
int gram_partial_blocks(int64_t N, int B) {
  const int rows = tall_tile_rows(B);
  const int64_t cap = std::max<int64_t>(64, std::min<int64_t>(2048, (int64_t(1) << 21) / ((int64_t)B * B)));
  const int64_t g = std::min<int64_t>((N + rows - 1) / rows, cap);
  return (int)(g < 1 ? 1 : g);
}

void launch_gram(int64_t N, int B, const double* X, const double* Y, double* partial, double* G,
                 hipStream_t s) {
  if (B < 1 || B > kMaxCols) throw Error(IDFT_EINVAL, "block width out of range for the Gram kernel");
  const int nb = gram_partial_blocks(N, B), rows = tall_tile_rows(B);
  dim3 grid(nb, (B * B + kThreads - 1) / kThreads);
  k_gram<<<grid, kThreads, 2 * rows * B * sizeof(double), s>>>(N, B, rows, X, Y, partial);
  IDFT_HIP(hipGetLastError());
  k_sum_rows<<<B * B, kRedThreads, 0, s>>>(nb, partial, G);
  IDFT_HIP(hipGetLastError());
}

void launch_right_mult(int64_t N, int B, const double* X, const double* Q, double* Y,
                       const double* ns, double beta, hipStream_t s) {
  if (B < 1 || B > kMaxCols) throw Error(IDFT_EINVAL, "block width out of range");
  check_u32(N * B);
  // Q and the tile within 64 KB of LDS (8 nodes per tile at the widest block)
  const int rows = std::max(8, std::min(64, (8192 - B * B) / B));
  const int64_t tiles = (N + rows - 1) / rows;
  const int grid = (int)std::max<int64_t>(1, std::min<int64_t>(tiles, 4096));
  k_right_mult<<<grid, kThreads, ((size_t)B * B + (size_t)rows * B) * sizeof(double), s>>>(
      (uint32_t)N, (uint32_t)B, (uint32_t)rows, X, Q, Y, ns, beta);
  IDFT_HIP(hipGetLastError());
}

int launch_residual_partial(int64_t N, int B, const double* HX, const double* X,
                            const double* ev, double* partial, hipStream_t s) {
  const int nb = coldot_blocks(N, B);
  k_residual<double><<<nb, kThreads, 0, s>>>(N, B, HX, X, ev, partial);
  IDFT_HIP(hipGetLastError());
  return nb;
}

void launch_vxc_to_quad(const Geo& g, const DevTables& t, const double* pot,
                        const double* potBase, double* veff, hipStream_t s) {
  dim3 grid((unsigned)g.ncell), block(kThreads);
  switch (g.p) {
    case 2: k_vxc_to_quad<2><<<grid, block, 0, s>>>(g, t.Wq.p, pot, potBase, veff); break;
    case 3: k_vxc_to_quad<3><<<grid, block, 0, s>>>(g, t.Wq.p, pot, potBase, veff); break;
    case 4: k_vxc_to_quad<4><<<grid, block, 0, s>>>(g, t.Wq.p, pot, potBase, veff); break;
    case 5: k_vxc_to_quad<5><<<grid, block, 0, s>>>(g, t.Wq.p, pot, potBase, veff); break;
    default: throw Error(IDFT_EINVAL, "degree not supported");
  }
  IDFT_HIP(hipGetLastError());
}

void launch_density(const Geo& g, const DevTables& t, const double* X, const double* S, int B,
                    const double* occ, double* rho, hipStream_t s) {
  dim3 grid((unsigned)g.ncell), block(kThreads);
  switch (g.p) {
    case 2: k_density<2, 8><<<grid, block, 0, s>>>(g, t.Lq.p, X, S, B, occ, rho); break;
    case 3: k_density<3, 8><<<grid, block, 0, s>>>(g, t.Lq.p, X, S, B, occ, rho); break;
    case 4: k_density<4, 8><<<grid, block, 0, s>>>(g, t.Lq.p, X, S, B, occ, rho); break;
    case 5: k_density<5, 8><<<grid, block, 0, s>>>(g, t.Lq.p, X, S, B, occ, rho); break;
    default: throw Error(IDFT_EINVAL, "degree not supported");
  }
  IDFT_HIP(hipGetLastError());
}

void launch_loss(int64_t nQ, int nq, const double* rho, const double* rhoT, const double* w,
                 const double* veff, const double* jxw, double* u, double* partial,
                 hipStream_t s) {
  k_loss<<<256, kThreads, 0, s>>>(nQ, nq, rho, rhoT, w, veff, jxw, u, partial);
  IDFT_HIP(hipGetLastError());
}

void launch_quad_operator(const Geo& g, const DevTables& t, const double* X, int B,
                          const double* wq, double* Y, int colour, hipStream_t s) {
  const int64_t nw = colour_count(g, colour);
  if (nw == 0) return;
  dim3 grid(colour_grid(nw)), block(kThreads);
  switch (g.p) {
    case 2: k_quad_operator<2, 8><<<grid, block, 0, s>>>(g, t.Lq.p, X, B, wq, Y, colour, nw); break;
    case 3: k_quad_operator<3, 8><<<grid, block, 0, s>>>(g, t.Lq.p, X, B, wq, Y, colour, nw); break;
    case 4: k_quad_operator<4, 8><<<grid, block, 0, s>>>(g, t.Lq.p, X, B, wq, Y, colour, nw); break;
    case 5: k_quad_operator<5, 8><<<grid, block, 0, s>>>(g, t.Lq.p, X, B, wq, Y, colour, nw); break;
    default: throw Error(IDFT_EINVAL, "degree not supported");
  }
  IDFT_HIP(hipGetLastError());
}

template <int P>
static void force_p(const Geo& g, const DevTables& t, const double* Psi, const double* Pv, int B,
                    int mode, double jxwChild, const double* jxwParent, double* force,
                    int colour, int64_t nw, hipStream_t s) {
  dim3 grid(colour_grid(nw)), block(kThreads);
  if (mode == 0)
    k_force<P, 4, 8><<<grid, block, 0, s>>>(g, t.Lc.p, t.Wc.p, Psi, Pv, B, jxwChild, nullptr,
                                            force, colour, nw);
  else
    k_force<P, P + 3, 8><<<grid, block, 0, s>>>(g, t.Lq.p, t.Wq.p, Psi, Pv, B, 0.0, jxwParent,
                                                force, colour, nw);
}

void launch_force(const Geo& g, const DevTables& t, const double* Psi, const double* P, int B,
                  int mode, double jxwChild, const double* jxwParent, double* force, int colour,
                  hipStream_t s) {
  const int64_t nw = colour_count(g, colour);
  if (nw == 0) return;
  switch (g.p) {
    case 2: force_p<2>(g, t, Psi, P, B, mode, jxwChild, jxwParent, force, colour, nw, s); break;
    case 3: force_p<3>(g, t, Psi, P, B, mode, jxwChild, jxwParent, force, colour, nw, s); break;
    case 4: force_p<4>(g, t, Psi, P, B, mode, jxwChild, jxwParent, force, colour, nw, s); break;
    case 5: force_p<5>(g, t, Psi, P, B, mode, jxwChild, jxwParent, force, colour, nw, s); break;
    default: throw Error(IDFT_EINVAL, "degree not supported");
  }
  IDFT_HIP(hipGetLastError());
}

void launch_zero_rows(int64_t N, int B, double* X, const unsigned char* mask, hipStream_t s) {
  check_u32(N * B);
  k_zero_rows<<<grid_for(N * B), kThreads, 0, s>>>((uint32_t)(N * B), (uint32_t)B, X, mask);
  IDFT_HIP(hipGetLastError());
}
void launch_zero_boundary(const Geo& g, int B, double* X, hipStream_t s) {
  check_u32(g.N * B);
  const int64_t n1 = g.N1, nbn = 2 * n1 * n1 + (n1 - 2) * 4 * (n1 - 1);
  k_zero_boundary<<<grid_for(nbn * B), kThreads, 0, s>>>((uint32_t)n1, (uint32_t)B, (uint32_t)nbn, X);
  IDFT_HIP(hipGetLastError());
}

void launch_minres_start(int B, int nblk, const double* partial, const double* negEig, double* st,
                         hipStream_t s, int nq) {
  k_minres_start<<<B, kThreads, 0, s>>>(B, nblk, partial, negEig, st, nq);
  IDFT_HIP(hipGetLastError());
}
int launch_minres_start_dots(int64_t N, int B, const double* r, const double* D, double* partial,
                             hipStream_t s) {
  if (B > kThreads) throw Error(IDFT_EINVAL, "block too wide for column reductions");
  const int nb = coldot_blocks(N, B);
  k_minres_start_dots<<<nb, kThreads, 0, s>>>(N, B, r, D, partial);
  IDFT_HIP(hipGetLastError());
  return nb;
}
void launch_minres_alpha_cell(int B, int ncell, const double* cell_dots, double* st, hipStream_t s) {
  k_minres_alpha_cell<<<B, kRedThreads, 0, s>>>(B, ncell, cell_dots, st);
  IDFT_HIP(hipGetLastError());
}
void launch_minres_alpha(int B, int nblk, const double* partial, double* st, hipStream_t s) {
  k_minres_alpha<<<B, kThreads, 0, s>>>(B, nblk, partial, st);
  IDFT_HIP(hipGetLastError());
}
template <typename T>
int launch_minres_lanczos(int64_t N, int B, const T* y, const T* r2, T* rnew, const double* D,
                          const double* st, double* partial, hipStream_t s) {
  const int nb = coldot_blocks(N, B);
  k_minres_lanczos<T><<<nb, kThreads, 0, s>>>(N, B, y, r2, rnew, D, st, partial);
  IDFT_HIP(hipGetLastError());
  return nb;
}
template int launch_minres_lanczos<float>(int64_t, int, const float*, const float*, float*,
                                          const double*, const double*, double*, hipStream_t);
template int launch_minres_lanczos<double>(int64_t, int, const double*, const double*, double*,
                                           const double*, const double*, double*, hipStream_t);
void launch_minres_givens(int B, int nblk, const double* partial, const double* negEig, double* st,
                          hipStream_t s, int nq, double* hist) {
  k_minres_givens<<<B, kRedThreads, 0, s>>>(B, nblk, partial, negEig, st, nq, hist);
  IDFT_HIP(hipGetLastError());
}
void launch_minres_batch(int64_t N, int B, int n, const MinresVectors& rs, const double* D,
                         double* w, double* w1, double* x, const double* hist,
                         const double* last, double* place, hipStream_t s) {
  if (B < 1 || B > kMaxCols || n < 1 || n > kMinresBatch)
    throw Error(IDFT_EINVAL, "block width or batch out of range");
  check_u32(N * B);
  const int vw = B % 2 == 0 ? 2 : 1, per = kThreads / (B / vw);
  // a few work-groups per CU in flight, each over several chunks (its 20 KB of
  // coefficients are loaded once)
  const unsigned grid = (unsigned)std::min<int64_t>((N + per - 1) / per, 8192);
  if (vw == 2)
    k_minres_batch<2><<<grid, kThreads, 0, s>>>((uint32_t)N, (uint32_t)B, n, rs, D, w, w1, x, hist,
                                            last, place);
  else
    k_minres_batch<1><<<grid, kThreads, 0, s>>>((uint32_t)N, (uint32_t)B, n, rs, D, w, w1, x, hist,
                                            last, place);
  IDFT_HIP(hipGetLastError());
}
template <typename T>
void launch_minres_update(int64_t N, int B, const T* r, const double* D, T* w1, const T* w, T* x,
                          const double* st, hipStream_t s) {
  check_u32(N * B);
  if (B % 2 == 0)
    k_minres_update<T, 2><<<grid_for(N * B / 2), kThreads, 0, s>>>((uint32_t)(N * B), (uint32_t)B,
                                                                  r, D, w1, w, x, st);
  else
    k_minres_update<T, 1><<<grid_for(N * B), kThreads, 0, s>>>((uint32_t)(N * B), (uint32_t)B, r,
                                                               D, w1, w, x, st);
  IDFT_HIP(hipGetLastError());
}
template void launch_minres_update<float>(int64_t, int, const float*, const double*, float*,
                                          const float*, float*, const double*, hipStream_t);
template void launch_minres_update<double>(int64_t, int, const double*, const double*, double*,
                                           const double*, double*, const double*, hipStream_t);
static int lan_blocks(int64_t N) { return (int)std::min<int64_t>((N + kThreads - 1) / kThreads, 1024); }
template <typename T>
void launch_lan_start(int64_t N, uint64_t seed, const unsigned char* mask, T* r, double* partial,
                      int k, double* lan, hipStream_t s) {
  check_u32(N);
  const int nb = lan_blocks(N);
  k_lan_start<T><<<nb, kThreads, 0, s>>>((uint32_t)N, seed, mask, r, partial);
  k_lan_beta<<<1, kRedThreads, 0, s>>>(nb, partial, k, -1, lan);
  IDFT_HIP(hipGetLastError());
}
template <typename T>
void launch_lan_step(int64_t N, T* y, const T* r, const T* rp, int nalpha, double* partial, int k,
                     int j, double* lan, hipStream_t s) {
  const int nb = lan_blocks(N);
  k_lan_alpha<<<1, kRedThreads, 0, s>>>(nalpha, partial, k, j, lan);
  k_lan_update<T><<<nb, kThreads, 0, s>>>((uint32_t)N, y, r, rp, lan + 2 * k, partial);
  k_lan_beta<<<1, kRedThreads, 0, s>>>(nb, partial, k, j, lan);
  IDFT_HIP(hipGetLastError());
}
#define IDFT_LAN(T)                                                                            \
  template void launch_lan_start<T>(int64_t, uint64_t, const unsigned char*, T*, double*, int, \
                                    double*, hipStream_t);                                     \
  template void launch_lan_step<T>(int64_t, T*, const T*, const T*, int, double*, int, int,    \
                                   double*, hipStream_t);
IDFT_LAN(float)
IDFT_LAN(double)
#undef IDFT_LAN
void launch_copy_done(int B, const double* st, int* flags, hipStream_t s) {
  k_copy_done<<<(B + 63) / 64, 64, 0, s>>>(B, st, flags);
  IDFT_HIP(hipGetLastError());
}


void launch_copy_cols(int64_t N, int Bs, int off, int Bd, const double* src, double* dst,
                      hipStream_t s) {
  k_copy_cols<<<grid_for(N * Bd), kThreads, 0, s>>>(N, Bs, off, Bd, src, dst);
  IDFT_HIP(hipGetLastError());
}
void launch_gather_cols(int64_t N, int Bs, const double* src, int Bd, const int* idx, double* dst,
                        hipStream_t s) {
  k_cols_by_index<<<grid_for(N * Bd), kThreads, 0, s>>>(N, Bs, Bd, Bd, idx, src, dst, 0);
  IDFT_HIP(hipGetLastError());
}
void launch_scatter_cols(int64_t N, int Bs, const double* src, int Bd, const int* idx, double* dst,
                         hipStream_t s) {
  k_cols_by_index<<<grid_for(N * Bs), kThreads, 0, s>>>(N, Bs, Bd, Bs, idx, src, dst, 1);
  IDFT_HIP(hipGetLastError());
}
void launch_mul_q(int64_t nQ, int nq, const double* u, const double* jxw, double* out,
                  hipStream_t s) {
  k_mul_q<<<grid_for(nQ), kThreads, 0, s>>>(nQ, nq, u, jxw, out);
  IDFT_HIP(hipGetLastError());
}
int launch_pairdot_partial(int64_t N, int B, const double* X, const double* Y, const double* w,
                           const int* pairs, int np, double* partial, hipStream_t s) {
  if (np > kThreads) throw Error(IDFT_EINVAL, "too many degenerate pairs");
  const int nb = coldot_blocks(N, np);
  k_pairdot<<<nb, kThreads, 0, s>>>(N, B, X, Y, w, pairs, np, partial);
  IDFT_HIP(hipGetLastError());
  return nb;
}


// ------------------------------------------------------ FMA rate probe
template <typename T, int CH>
static double fma_probe_t(hipStream_t s) {
  int dev = 0, ncu = 0;
  IDFT_HIP(hipGetDevice(&dev));
  IDFT_HIP(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
  const int blocks = std::max(1, ncu) * 32, iters = 2048;
  T* out = nullptr;
  IDFT_HIP(hipMalloc(&out, sizeof(T) * (size_t)blocks * kThreads));
  hipEvent_t e0 = nullptr, e1 = nullptr;
  float ms = 0.0f;
  hipError_t err = hipEventCreate(&e0);
  if (err == hipSuccess) err = hipEventCreate(&e1);
  if (err == hipSuccess) {
    k_fma_probe<T, CH><<<blocks, kThreads, 0, s>>>(out, (T)0.999, (T)0.001, iters);
    err = hipGetLastError();
  }
  if (err == hipSuccess) err = hipEventRecord(e0, s);
  if (err == hipSuccess) {
    k_fma_probe<T, CH><<<blocks, kThreads, 0, s>>>(out, (T)0.999, (T)0.001, iters);
    err = hipGetLastError();
  }
  if (err == hipSuccess) err = hipEventRecord(e1, s);
  if (err == hipSuccess) err = hipEventSynchronize(e1);
  if (err == hipSuccess) err = hipEventElapsedTime(&ms, e0, e1);
  if (e0) (void)hipEventDestroy(e0);
  if (e1) (void)hipEventDestroy(e1);
  (void)hipFree(out);
  IDFT_HIP(err);
  const double flops = 2.0 * CH * (double)iters * blocks * kThreads;
  return flops / ((double)ms * 1e-3) / 1e12;
}
double launch_fma_probe(bool fp64, int chains, hipStream_t s) {
  switch (chains) {
    case 4: return fp64 ? fma_probe_t<double, 4>(s) : fma_probe_t<float, 4>(s);
    case 8: return fp64 ? fma_probe_t<double, 8>(s) : fma_probe_t<float, 8>(s);
    case 16: return fp64 ? fma_probe_t<double, 16>(s) : fma_probe_t<float, 16>(s);
    default: throw Error(IDFT_EINVAL, "chains must be 4, 8 or 16");
  }
}

}  // namespace idft
