// Dense block kernels of the block-cyclic-reduction factorisation (gfx950).
//
//   gemm_batched   C = beta*C + alpha*(A1*B1 + A2*B2) for a list of complex
//                  blocks, on MFMA (f64 16x16x4 or f32 16x16x4).
//   gj_inverse     inverse of a list of complex blocks by blocked
//                  Gauss-Jordan elimination with partial (row) pivoting.
//
// All blocks are column-major with interleaved complex storage.
#include <climits>
#include <type_traits>
#include "kore_device.hpp"
#include "kore_kernels.hpp"

namespace kore {

// ---------------------------------------------------------------------------
// batched complex GEMM
// ---------------------------------------------------------------------------
// Workgroup = 4 waves, output tile 32 S x 32 S, each wave a quadrant of S x S
// MFMA 16x16 tiles; K staged through LDS in slabs of GT_K = 16 (32 measured
// slower: the larger LDS and register footprint halves the workgroups per CU).
// S = 1 or 2 by gemm_small_tiles below.
constexpr int GT_K = 16;
// complex64 double-buffers its slabs in LDS (one barrier per slab); two slabs
// of complex128 would leave room for two workgroups per CU where three fit
template <class T> constexpr int GT_NBUF = sizeof(T) == 4 ? 2 : 1;
template <class T, int S> struct GemmLds {
  cx<T> A[GT_NBUF<T>][GT_K][32 * S];
  cx<T> B[GT_NBUF<T>][32 * S][GT_K + 1];
};

// Global load of base[off] with a uniform base: one 32-bit offset register
// and no address arithmetic per load.
template <class T> __device__ __forceinline__ cx<T> gld_at(const cx<T>* base, unsigned off) {
  typedef typename cx_vec<T>::type V;
  const V v = *(const __attribute__((address_space(1))) V*)((const __attribute__((address_space(1))) char*)base +
                                                            (size_t)off * sizeof(cx<T>));
  return cx<T>{v.x, v.y};
}

// One tile of C = alpha sum_p A_p B_p + beta C for the workgroup (256
// threads).  A and B tiles wholly or partly outside the matrices read their
// last row or column instead (rows and columns of C that are not stored), so
// that only the last slab of a product has anything to check: its missing k
// count as zero.  With roles given, rows of C whose role is rmin or more are
// replaced (their old values count as zero).
// M3: three real products per complex step in complex64 (below).
template <class T, int S, bool M3 = true>
__device__ __forceinline__ void gemm_tile_body(const GemmDesc<T>& d, const int tile, GemmLds<T, S>& sm,
                                               const int* roles = nullptr, int rmin = 0) {
  using A4 = typename acc4<T>::type;
  constexpr int TS = 32 * S, NQ = 2 * S;      // tile edge, slab elements of A (and of B) per thread
  constexpr int NBUF = GT_NBUF<T>;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr = (wave >> 1) * 16 * S, wc = (wave & 1) * 16 * S;
  const int l16 = lane & 15, lq = lane >> 4;
  const int tiles_m = (d.m + TS - 1) / TS;
  const int i0 = (tile % tiles_m) * TS;
  const int j0 = (tile / tiles_m) * TS;
  // 16 x 16 sub-tiles wholly outside C (edge tiles of sizes that are not
  // multiples of the tile, e.g. 200 = 3*64 + 8) are skipped, wave-uniformly
  bool rv[S], cv[S];
#pragma unroll
  for (int s = 0; s < S; ++s) {
    rv[s] = i0 + wr + 16 * s < d.m;
    cv[s] = j0 + wc + 16 * s < d.n;
  }
  // complex64: three real products per complex step (Karatsuba's 3M
  // form): cre = sum ar br, cim = sum ai bi, csum = sum (ar + ai)(br + bi),
  // and at the end re = cre - cim, im = csum - cre - cim: 3/4 of the
  // matrix-core work of the four-product form, with a normwise error bound
  // of the same order (Higham, Accuracy and Stability of Numerical
  // Algorithms, section 23.2.4); the complex64 factor is a preconditioner
  // whose answers FP64 refinement or GMRES corrects.  complex128 keeps the
  // four products (cre, cim = real and imaginary parts): measured, the 3M
  // form makes the FP64 factor 10 % faster at N = 500 but moves the most
  // ill-conditioned MAC eigenvalues (relative condition 1e16) further from
  // the oracle's than the four-product form does.
  constexpr bool k3m = M3 && sizeof(T) == 4;
  A4 cre[S][S], cim[S][S], csum[S][S];
#pragma unroll
  for (int a = 0; a < S; ++a)
#pragma unroll
    for (int b = 0; b < S; ++b) {
      cre[a][b] = A4{0, 0, 0, 0};
      cim[a][b] = A4{0, 0, 0, 0};
      csum[a][b] = A4{0, 0, 0, 0};
    }

  // Slabs of GT_K k-columns over the (up to two) products, register
  // double-buffered: slab s+1 is requested from memory before slab s is
  // multiplied, so the load latency hides behind the matrix-core work.
  // Thread (kt = tid / 16, l16) loads A[i0 + l16 + 16 q][k0 + kt] and
  // B[k0 + l16][j0 + kt + 16 q]: 16 lanes read consecutive addresses of
  // both, and write consecutive LDS words.
  const int kt = tid >> 4;
  cx<T> ra[NQ], rb[NQ];
  unsigned oa[NQ], ob[NQ];                    // element offsets of the thread from the product's base
  const cx<T>* __restrict__ A = nullptr;      // base of the next slab (uniform)
  const cx<T>* __restrict__ B = nullptr;
  int K = 0;
  int64_t lda = 0;
  auto start = [&](int p) {                   // product p (selects, not indexing: d stays in registers)
    K = p ? d.k[1] : d.k[0];
    lda = p ? d.lda[1] : d.lda[0];
    const int64_t ldb = p ? d.ldb[1] : d.ldb[0];
    A = (p ? d.A[1] : d.A[0]) + i0;
    B = (p ? d.B[1] : d.B[0]) + (int64_t)j0 * ldb;
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      oa[q] = (unsigned)min(l16 + 16 * q, d.m - 1 - i0) + (unsigned)kt * (unsigned)lda;
      ob[q] = (unsigned)min(kt + 16 * q, d.n - 1 - j0) * (unsigned)ldb + (unsigned)l16;
    }
  };
  auto load = [&](int k0) {                   // the slab at k0; A, B move to the next one
    const int rem = K - k0;
    if (rem >= GT_K) {
#pragma unroll
      for (int q = 0; q < NQ; ++q) ra[q] = gld_at<T>(A, oa[q]);
#pragma unroll
      for (int q = 0; q < NQ; ++q) rb[q] = gld_at<T>(B, ob[q]);
    } else {                                  // the product's last slab, rem of 16 columns
      const bool ka = kt < rem, kb = l16 < rem;
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        ra[q] = gld_at<T>(A, ka ? oa[q] : oa[q] - (unsigned)(kt - rem + 1) * (unsigned)lda);
        rb[q] = gld_at<T>(B, kb ? ob[q] : ob[q] - (unsigned)(l16 - rem + 1));
        if (!ka) ra[q] = czero<T>();
        if (!kb) rb[q] = czero<T>();
      }
    }
    A += (int64_t)GT_K * lda;
    B += GT_K;
  };
  auto valid = [&](int p) { return d.A[p] != nullptr && d.k[p] > 0; };
  int p = valid(0) ? 0 : (valid(1) ? 1 : 2), k0 = 0, buf = 0;
  if (p < 2) {
    start(p);
    load(0);
  }
  while (p < 2) {
    const int rem = K - k0;
    if (NBUF == 1) __syncthreads();           // the previous slab has been consumed
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      sm.A[buf][kt][l16 + 16 * q] = ra[q];
      sm.B[buf][kt + 16 * q][l16] = rb[q];
    }
    __syncthreads();
    int pn = p;
    k0 += GT_K;                               // next slab
    if (k0 >= K) {
      pn = (p == 0 && valid(1)) ? 1 : 2;
      k0 = 0;
      if (pn < 2) start(pn);
    }
    if (pn < 2) load(k0);
#pragma unroll
    for (int kk = 0; kk < GT_K; kk += 4) {
      if (kk >= rem) break;                   // uniform
      cx<T> a[S], b[S];
#pragma unroll
      for (int s = 0; s < S; ++s) {
        a[s] = sm.A[buf][kk + lq][wr + 16 * s + l16];
        b[s] = sm.B[buf][wc + 16 * s + l16][kk + lq];
      }
      if constexpr (k3m) {
        T as[S], bs[S];
#pragma unroll
        for (int q = 0; q < S; ++q) {
          as[q] = a[q].re + a[q].im;
          bs[q] = b[q].re + b[q].im;
        }
#pragma unroll
        for (int rs = 0; rs < S; ++rs)
#pragma unroll
          for (int cs = 0; cs < S; ++cs)
            if (rv[rs] && cv[cs]) {
              cre[rs][cs] = mfma16(b[cs].re, a[rs].re, cre[rs][cs]);
              cim[rs][cs] = mfma16(b[cs].im, a[rs].im, cim[rs][cs]);
              csum[rs][cs] = mfma16(bs[cs], as[rs], csum[rs][cs]);
            }
      } else {
#pragma unroll
        for (int rs = 0; rs < S; ++rs)
#pragma unroll
          for (int cs = 0; cs < S; ++cs)
            if (rv[rs] && cv[cs]) cmma<T>(cre[rs][cs], cim[rs][cs], a[rs], b[cs]);
      }
    }
    p = pn;
    if (NBUF == 2) buf ^= 1;
  }
  __syncthreads();                            // LDS is reused by the next tile
  // epilogue: lane holds C[i0+wr+16rs+l16][j0+wc+16cs+mfma_mrow(lq,r)].
  // Per row sub-tile, the old values of C are loaded together before
  // any store, so that their latencies overlap (a load after a store to a
  // possibly aliasing address would wait for the previous one).
  const bool acc = d.beta != T(0);
#pragma unroll
  for (int rs = 0; rs < S; ++rs) {
    const int gi = i0 + wr + 16 * rs + l16;
    cx<T> o[S][4];
    const bool old = acc && gi < d.m && !(roles && roles[gi] >= rmin);
#pragma unroll
    for (int cs = 0; cs < S; ++cs)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int gj = j0 + wc + 16 * cs + mfma_mrow<T>(lq, r);
        o[cs][r] = czero<T>();
        if (old && gj < d.n) o[cs][r] = gld(d.C + (int64_t)gj * d.ldc + gi);
      }
#pragma unroll
    for (int cs = 0; cs < S; ++cs)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int gj = j0 + wc + 16 * cs + mfma_mrow<T>(lq, r);
        if (gi < d.m && gj < d.n) {
          T vre = cre[rs][cs][r], vim = cim[rs][cs][r];
          if constexpr (k3m) {
            vre = cre[rs][cs][r] - cim[rs][cs][r];
            vim = csum[rs][cs][r] - cre[rs][cs][r] - cim[rs][cs][r];
          }
          cx<T> v{d.alpha * vre, d.alpha * vim};
          if (acc) {
            v.re += d.beta * o[cs][r].re;
            v.im += d.beta * o[cs][r].im;
          }
          gst(d.C + (int64_t)gj * d.ldc + gi, v);
        }
      }
  }
}

// Tile edge 32 instead of 64: where it covers much less padding (n = 200: 224
// rows instead of 256; n = 150: 160 instead of 192), and where the launch holds
// few tiles, so that four times the workgroups fill the chip.  Measured, us per
// launch of one n x n x n product per item, edge 64 / 32:
//   complex128  n = 500: 1 item 85 / 33, 8 items 155 / 155, 32 items 618 / 649
//               n = 200: 1 item 36 / 14, 32 items 68 / 65, 150 items 257 / 226
//               n = 374: 16 items 165 / 133, 32 items 273 / 255, 64 items 512 / 529
//               n = 450 (480 rows instead of 512): 64 items 1019 / 1032
//   complex64   n = 500: 1 item 49 / 22, 4 items 54 / 45, 8 items 74 / 83
//               n = 150: 32 items 26 / 21, 150 items 68 / 55
//               n = 450: 64 items 434 / 485
template <class T> static bool gemm_small_tiles(int nitems, int t64, int t32) {
  return t32 < 3.2 * t64 || (int64_t)nitems * t64 < (sizeof(T) == 8 ? 1536 : 384);
}

template <class T, int S>
__global__ __launch_bounds__(256, 3) void gemm_batched_kernel(const GemmDesc<T>* __restrict__ descs, int ndesc,
                                                              int per) {
  __shared__ GemmLds<T, S> sm;
  int di, tile;
  xcd_item(blockIdx.x, per, ndesc, di, tile);
  if (di >= ndesc) return;
  const GemmDesc<T> d = descs[di];
  const int ntiles = ((d.m + 32 * S - 1) / (32 * S)) * ((d.n + 32 * S - 1) / (32 * S));
  for (; tile < ntiles; tile += per) gemm_tile_body<T, S>(d, tile, sm);
}

template <class T> __device__ __forceinline__ T tiny_pivot() { return sizeof(T) == 8 ? T(1e-150) : T(1e-18); }

// ---------------------------------------------------------------------------
// batched Gauss-Jordan inverse with partial pivoting
// ---------------------------------------------------------------------------
// Rows are never moved: column j is eliminated with pivot row r_j (within a
// factor 1 - 2^-11 of the largest |re|+|im| among the rows not used yet, first
// index on ties), so that at the end
//     A^{-1}[k, l] = M[r_k, r^{-1}(l)].
// The update of a block spreads over many workgroups: per panel J = [p0, p0+w)
//   gj_panel_kernel   one workgroup per block: Gauss-Jordan on the panel
//                     columns (pivot rows P), C -> M[:, J], the final columns
//                     J of M; R = M[P, :] (rows before the update) -> scratch;
//   gj_update_kernel  M[i, j] <- [i not in P] M[i, j] + sum_k C[i, k] R[k, j]
//                     for j outside J, on matrix cores;
// then gj_perm_kernel: A^{-1}[k, l] = M[r_k, r^{-1}(l)] into the scratch block,
// which is where the inverse is wanted.  Blocks of up to 112 rows take
// gj_panel_rows_kernel for the panel; those of one panel (up to 32 rows) are complete
// after it, which stores them in their final order: one launch
// (24 rows, complex128: 55 -> 19 us; a kernel that ran the whole elimination of
// a block in one workgroup, used below 96 rows, is gone: 74 rows 193 -> 86 us).
// Scratch layout (per block of more than 32 rows, n x n complex): R
// (32 x n, R[k, j] at R[j 32 + k]), then n ints of row roles (-1 unused,
// c >= 0: the pivot row of column c).  The multi-panel composition: with T
// the product of the panel's elementary transforms, T differs from the identity
// only in the pivot columns P, so for a column j outside J,
// T M[:, j] = [i not in P] M[i, j] + T[:, P] M[P, j], and T[:, P] is exactly what
// in-place elimination leaves in M[:, J].
// Cross-lane moves within rows of 16 lanes (DPP).
template <int CTRL> __device__ __forceinline__ unsigned dpp_u32(unsigned x) {
  return (unsigned)__builtin_amdgcn_update_dpp(0, (int)x, CTRL, 0xF, 0xF, false);
}
template <int CTRL> __device__ __forceinline__ double dpp_t(double x) {
  return __hiloint2double((int)dpp_u32<CTRL>((unsigned)__double2hiint(x)), (int)dpp_u32<CTRL>((unsigned)__double2loint(x)));
}
template <int CTRL> __device__ __forceinline__ float dpp_t(float x) {
  return __uint_as_float(dpp_u32<CTRL>(__float_as_uint(x)));
}

constexpr int GJM_WP = 32;
// Two-level panels for blocks of at least GJ_OUTER_MIN rows: the panels of
// 32 columns are grouped into outer panels O of GJ_WO columns.  A panel's
// rank-32 update is applied to the columns of its outer panel only; once the
// outer panel is complete, the columns outside it receive the composite
// transform of its GJ_WO eliminations in one rank-GJ_WO product (the same
// composition argument as for a single panel, with P = the outer panel's
// pivot rows).  That halves the passes over the block and turns most of the
// update into a product with K = GJ_WO on the matrix cores.  Scratch layout
// then: R (32 x n), n ints of row roles, R_O (GJ_WO x n): 161 n entries, so
// the block needs n >= 161.  Below 256 rows the two extra launches per outer
// panel cost more than the passes they save (measured at 200 rows).
constexpr int GJ_WO = 128;
constexpr int GJ_OUTER_MIN = 256;

// Outer panel [q0, q0 + wo) holding column p0 of an n x n block.
__device__ __forceinline__ void gj_outer_range(int n, int p0, int& q0, int& wo) {
  if (n >= GJ_OUTER_MIN) {
    q0 = (p0 / GJ_WO) * GJ_WO;
    wo = min(GJ_WO, n - q0);
  } else {
    q0 = 0;
    wo = n;
  }
}

// MFMA row index -> column of a 16-column tile, so that register i of lane
// group lq holds column 4 i + lq for both element types (the two instructions
// number their result rows differently, see mfma_mrow).
template <class T> __device__ __forceinline__ int gj_tile_col(int m);
template <> __device__ __forceinline__ int gj_tile_col<double>(int m) { return m; }
template <> __device__ __forceinline__ int gj_tile_col<float>(int m) { return 4 * (m & 3) + (m >> 2); }

// Magnitude bits of a pivot candidate; NaN and infinity count as zero.  A pivot
// key is a valid flag (bit 31), the magnitude's next 22 bits (a double's exponent
// and 11 mantissa bits, a float's and 14) and 511 - row: threshold partial
// pivoting, ties go to the lower row, and one 32-bit maximum per reduction stage.
__device__ __forceinline__ unsigned pivot_bits(double mag) {
  const unsigned b = (unsigned)__double2hiint(mag);
  return b < 0x7FF00000u ? b : 0u;
}
__device__ __forceinline__ unsigned pivot_bits(float mag) {
  const unsigned b = __float_as_uint(mag);
  return b < 0x7F800000u ? b : 0u;
}

// Gauss-Jordan on the panel's columns, TPR threads per row.  The panel's 32
// columns stay in MFMA accumulators; SW = 8 of them at a time are handed to the
// rows' threads through LDS and eliminated there, a step updating only those 8
// columns, and the other columns receive the 8 transforms at once as a product
// on the matrix cores (the composition used for panels and outer panels, one
// level down).
//
// What bounds it is the chain of a column step: key, two barriers with an LDS
// exchange each, multiplier, next key.  Its length is instructions issued
// between those points (about 150 and 1300 clocks a step before, about 100 and
// 920 (complex64) to 1150 clocks now, 200 rows), so the chain holds only what it
// must: the pivot row is stored and read with 8 columns instead of 32, each
// thread forms the reciprocal of its own candidate and updates its other columns
// behind the key's exchange, the waves' keys meet in one LDS maximum, and a
// row's use and identity are masks in its key.  The pivot rows of the other
// columns of the outer panel are gathered while later columns are eliminated
// (fetched after the last step they took 8 of a panel's 44 us, being scattered).
// Measured, one panel of one block, us before / now: complex128 200 rows 47 / 32,
// 500 rows 62 / 48; complex64 200 rows 41 / 27, 500 rows 44 / 36; 256 blocks of 500
// rows: complex128 101 / 65 per launch.  Two threads a row (a thread then stores
// and reads four columns) are faster except for complex128 above 256 rows, whose
// accumulators do not leave room for the second wave (one block of 500 rows: 1100
// against 1000 us for an inversion).
constexpr int GJ_SW = 8;
template <class T, int NMAX> constexpr int GJ_TPR = sizeof(T) == 8 && NMAX > 256 ? 1 : 2;
// columns of a pivot row that a panel keeps in flight: all of an outer panel's
constexpr int gj_gather_cols(int nmax) { return nmax <= 256 ? nmax : nmax <= 384 ? 192 : 128; }

template <class T> __device__ __forceinline__ cx<T> cmul_fma(cx<T> a, cx<T> b) {
  return cx<T>{fma(a.re, b.re, -(a.im * b.im)), fma(a.re, b.im, a.im * b.re)};
}

// What the column steps of a workgroup share.
template <class T, int SW> struct GjLds {
  cx<T> row[2][SW];                       // the pivot row
  cx<T> inv[SW];                          // minus the inverse pivots
  unsigned key[4];                        // best key of a step; steps take the four in turn
  int piv[GJM_WP];                        // pivot row of each of the panel's columns
  int sing;
};

template <int CTRL, class T> __device__ __forceinline__ cx<T> dpp_cx(cx<T> x) {
  return cx<T>{dpp_t<CTRL>(x.re), dpp_t<CTRL>(x.im)};
}

// Gauss-Jordan on kw <= SW columns, TPR threads per row: this thread's v holds
// columns [CPT h, CPT h + CPT) of row r.  The columns are j0 .. of the block and
// s0 .. of the panel.  Returns which of them the row pivots, or -1; v then holds the
// final columns.  ONCE: a step's product is formed first and rounds each entry once
// (two fused multiply-adds round it twice), for a third more operations.
template <class T, int SW, int TPR, bool ONCE>
__device__ __forceinline__ int gj_eliminate(GjLds<T, SW>& sm, cx<T> (&v)[SW / TPR], int& role, int& sing, int j0,
                                            int s0, int kw, int zero_off) {
  constexpr int CPT = SW / TPR;
  const int r = threadIdx.x / TPR, h = threadIdx.x % TPR;
  // A step's key is one mask and one or: rows in use have both zero.  Every
  // column has an unused row left, so the best key is never zero.
  const unsigned rowkey = 0x80000000u | (unsigned)(511 - r);
  unsigned rk = role == -1 && h == 0 ? rowkey : 0u, mk = role == -1 && h == 0 ? 0x7FFFFE00u : 0u;
  unsigned mykey = 0;                   // of the row (of all its lanes)
  // the row's entry x of column s0 + c enters the search for its pivot
  auto compete = [&](cx<T> x, int c) __attribute__((always_inline)) {
    mykey = (pivot_bits(cabs1(x)) & mk) | rk;
    unsigned key = mykey;
    key = max(key, dpp_u32<0xB1>(key));  // quad_perm [1,0,3,2]
    if constexpr (TPR == 2) mykey = key;
    key = max(key, dpp_u32<0x4E>(key));  // quad_perm [2,3,0,1]
    if constexpr (TPR == 4) mykey = key;
    key = max(key, dpp_u32<0x141>(key)); // row_half_mirror
    key = max(key, dpp_u32<0x140>(key)); // row_mirror
    if ((threadIdx.x & 15) == 15)           // one lane per 16
      __hip_atomic_fetch_max(&sm.key[zero_off + (c & 3)], key, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  };
  // minus its reciprocal, should it win
  bool zero = false;
  auto invert = [&](cx<T> x) __attribute__((always_inline)) {
    T den = x.re * x.re + x.im * x.im;
    zero = !(den > T(0));
    if (zero) {
      x = cx<T>{tiny_pivot<T>(), T(0)};
      den = x.re * x.re;
    }
    const T iden = T(1) / den;
    return cx<T>{-(x.re * iden), x.im * iden};
  };
  compete(v[0], s0);
  cx<T> ninv = invert(v[0]);
#pragma unroll
  for (int c = 0; c < SW; ++c) {
    if (c < kw) {                       // uniform
      const int hc = c / CPT, vc = c % CPT;   // where column c is
      __syncthreads();
      const bool isp = sm.key[(s0 + c) & 3] == mykey;
      // only the pivot row's threads store it, behind a second barrier (every
      // wave storing its best candidate beside its key costs more)
      if (isp) {
#pragma unroll
        for (int k = 0; k < CPT; ++k) sm.row[c & 1][CPT * h + k] = v[k];
        if (h == hc) {
          sm.inv[c] = ninv;
          if (zero) sing = min(sing, j0 + c + 1);
        }
        role = j0 + c;
        rk = mk = 0;
      }
      __syncthreads();
      const cx<T> pinv = sm.inv[c];
      cx<T> u[CPT];
#pragma unroll
      for (int k = 0; k < CPT; ++k) u[k] = sm.row[c & 1][CPT * h + k];
      cx<T> x = v[vc];
      // the row's entry in column c, from the lane that holds it
      if constexpr (TPR == 2) x = hc == 0 ? dpp_cx<0xA0>(x) : dpp_cx<0xF5>(x);   // quad_perm [0,0,2,2], [1,1,3,3]
      if constexpr (TPR == 4)
        x = hc == 0 ? dpp_cx<0x00>(x) : hc == 1 ? dpp_cx<0x55>(x) : hc == 2 ? dpp_cx<0xAA>(x) : dpp_cx<0xFF>(x);
      // Rows past n and columns past w hold zeros (and the pivot row's copy
      // too), so the update needs no row or column guard: zeros stay zeros.
      // The pivot row is not scaled here: its column c becomes 1 and the row
      // is multiplied by its inverse pivot once, after the last step (a later
      // step updates it like any other row, which commutes with that scale).
      // So every lane runs the same code, the pivot row with multiplier zero.
      cx<T> nl = cmul(x, pinv);
      if (isp) nl = czero<T>();
      const cx<T> fin{isp ? T(1) : nl.re, nl.im};
      // the next pivot column first: its key is the next link of the chain,
      // and the other columns' updates and the reciprocal run behind it
      const int hn = (c + 1) / CPT, vn = (c + 1) % CPT;
      if (c + 1 < SW) {
        const cx<T> t = ONCE ? cadd(v[vn], cmul_fma(nl, u[vn])) : cfma(v[vn], nl, u[vn]);
        v[vn] = vn == vc && h == hc ? fin : t;
        if (TPR > 1 && vn == 0) {       // the columns of the next lane slice begin
          rk = role == -1 && h == hn ? rowkey : 0u;
          mk = role == -1 && h == hn ? 0x7FFFFE00u : 0u;
        }
        if (c + 1 < kw) compete(v[vn], s0 + c + 1);
      }
      if (threadIdx.x == 0) sm.key[(s0 + c + 2) & 3] = 0;      // last read two steps ago, next written in the next step
#pragma unroll
      for (int k = 0; k < CPT; ++k)
        if (k != vn || c + 1 == SW) {
          const cx<T> t = ONCE ? cadd(v[k], cmul_fma(nl, u[k])) : cfma(v[k], nl, u[k]);
          v[k] = k == vc && h == hc ? fin : t;
        }
      if (c + 1 < SW) ninv = invert(v[vn]);
    }
  }
  const int kp = role >= j0 ? role - (j0) : -1;   // pivot row of these columns: which one
  if (kp >= 0) {                        // the deferred scale
    const cx<T> ip{-sm.inv[kp].re, -sm.inv[kp].im};
    if (h == 0) sm.piv[s0 + kp] = r;
#pragma unroll
    for (int k = 0; k < CPT; ++k) v[k] = cmul(v[k], ip);
  }
  return kp;
}

template <class T, int NMAX>
__global__ __launch_bounds__((NMAX * GJ_TPR<T, NMAX>), (sizeof(T) == 4 ? 4 : 2)) void gj_panel_kernel(
    const InvDesc<T>* __restrict__ descs, int p0) {
  using A4 = typename acc4<T>::type;
  constexpr int SW = GJ_SW, TPR = GJ_TPR<T, NMAX>;
  constexpr int NT = NMAX * TPR, NW = NT / 64, WP = GJM_WP, NK = SW / 4;
  constexpr int RW = 64 / TPR, NRT = RW / 16, CPT = SW / TPR;   // rows and row tiles of a wave, columns per thread
  constexpr int LX = NMAX + (TPR > 1 ? 8 : 0);                  // the two columns of a wave's access in different banks
  static_assert(WP == 32 && SW == 8, "panel split");
  __shared__ cx<T> sX[SW * LX];           // eliminated columns, row by row: column k of row r at k LX + r
  __shared__ cx<T> sR[SW * WP];           // pivot rows before the update
  __shared__ GjLds<T, SW> sm;
  const InvDesc<T> d = descs[blockIdx.x];
  const int n = d.n;
  __builtin_assume(p0 < n);               // no check for an empty panel (complex64, 200 rows: 222 -> 211 us)
  const int64_t ld = d.ld;
  cx<T>* __restrict__ M = d.M;
  cx<T>* __restrict__ R = d.scratch;
  int* __restrict__ roles = reinterpret_cast<int*>(d.scratch + (size_t)WP * n);
  const int w = min(WP, n - p0);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, lq = lane >> 4;
  const int r = tid / TPR, h = tid % TPR;   // owned row, columns [CPT h, CPT h + CPT) of the SW at hand
  const bool live = r < n;
  cx<T>* J = M + (int64_t)p0 * ld;        // the panel's columns
  // row tile rt of the wave, column 16 ct + 4 i + lq
  A4 cre[NRT][2], cim[NRT][2];
#pragma unroll
  for (int rt = 0; rt < NRT; ++rt)
#pragma unroll
    for (int ct = 0; ct < 2; ++ct)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = RW * wave + 16 * rt + l16, j = 16 * ct + 4 * i + lq;
        cx<T> x = gld_at<T>(J, (unsigned)min(j, w - 1) * (unsigned)ld + (unsigned)min(row, n - 1));
        if (row >= n || j >= w) x = czero<T>();
        cre[rt][ct][i] = x.re;
        cim[rt][ct][i] = x.im;
      }
  // every row is unused at the first panel (the scratch holds an earlier call's
  // roles); afterwards a row's role is the column it pivots, or -1
  int role = -2;
  if (live) role = p0 == 0 ? -1 : roles[r];
  // zero in a vector register that the compiler cannot see through: for an LDS
  // address that it knows to be the same in all lanes it would reduce over the
  // lanes once more before an atomic
  int zero_off = 0;
  asm("" : "+v"(zero_off));
  int sing = INT_MAX;                     // smallest singular column (1-based) that this thread has met
  if (tid == 0) sm.sing = INT_MAX;
  if (tid < 4) sm.key[tid] = 0;
  if (tid < WP) sm.piv[tid] = 0;
  __syncthreads();
  int q0, wo;
  gj_outer_range(n, p0, q0, wo);
  // R[k, j] = M[P[k], j] for the columns j of the outer panel (those of the panel
  // itself are not used): the rows of SW columns are requested as soon as they
  // are known and stored after the next SW columns, behind whose steps the
  // scattered reads finish.  GP passes of GC columns, all of an outer panel's, are
  // kept in flight.
  constexpr int GC = NT / SW, GP = gj_gather_cols(NMAX) / GC;
  static_assert(GP * GC >= (NMAX < GJ_OUTER_MIN ? NMAX : GJ_WO), "columns of an outer panel");
  cx<T> gx[GP];
  const int gk = tid % SW, gj = tid / SW;
  auto gather = [&](int s0) __attribute__((always_inline)) {
    const cx<T>* row = M + sm.piv[s0 + gk] + (int64_t)q0 * ld;
#pragma unroll
    for (int t = 0; t < GP; ++t) gx[t] = gld(row + (int64_t)min(gj + t * GC, wo - 1) * ld);
  };
  auto put = [&](int s0) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < GP; ++t) {
      const int j = gj + t * GC;
      if (j < wo) gst(R + (int64_t)(q0 + j) * WP + s0 + gk, gx[t]);
    }
  };
  auto wave_sync = []() __attribute__((always_inline)) {   // LDS written by this wave's other lanes
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };
  // columns [SW s, SW s + SW) between the accumulators and the rows' threads; s
  // is a compile-time constant here, so that the accumulators are never indexed
  auto extract = [&](auto sc) __attribute__((always_inline)) {
    constexpr int S = decltype(sc)::value, CT = S * SW / 16, I0 = (S * SW % 16) / 4;
#pragma unroll
    for (int rt = 0; rt < NRT; ++rt)
#pragma unroll
      for (int k = 0; k < NK; ++k)
        sX[(4 * k + lq) * LX + RW * wave + 16 * rt + l16] = cx<T>{cre[rt][CT][I0 + k], cim[rt][CT][I0 + k]};
  };
  auto update = [&](auto sc, int kw) __attribute__((always_inline)) {
    constexpr int S = decltype(sc)::value, CT = S * SW / 16, I0 = (S * SW % 16) / 4;
    cx<T> b[2][NK];
#pragma unroll
    for (int ct = 0; ct < 2; ++ct)
#pragma unroll
      for (int k = 0; k < NK; ++k) {
        b[ct][k] = sR[(4 * k + lq) * WP + 16 * ct + gj_tile_col<T>(l16)];
        if (4 * k + lq >= kw) b[ct][k] = czero<T>();
      }
#pragma unroll
    for (int rt = 0; rt < NRT; ++rt) {
      cx<T> a[NK];
#pragma unroll
      for (int k = 0; k < NK; ++k) a[k] = sX[(4 * k + lq) * LX + RW * wave + 16 * rt + l16];
#pragma unroll
      for (int ct = 0; ct < 2; ++ct) {        // the product on its own, added once: each entry rounds once
        A4 pre = {0, 0, 0, 0}, pim = {0, 0, 0, 0};
#pragma unroll
        for (int k = 0; k < NK; ++k) cmma<T>(pre, pim, a[k], b[ct][k]);
        cre[rt][ct] += pre;
        cim[rt][ct] += pim;
      }
#pragma unroll
      for (int k = 0; k < NK; ++k) {
        cre[rt][CT][I0 + k] = a[k].re;
        cim[rt][CT][I0 + k] = a[k].im;
      }
      // the row tiles one after the other: overlapped they take more registers than there
      // are (complex128, 24 of them spilled, an inversion of one block of 500 rows 961
      // us instead of 904)
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  auto eliminate = [&](auto sc) __attribute__((always_inline)) {
    constexpr int s0 = decltype(sc)::value * SW;
    const int kw = min(SW, w - s0);
    if (kw <= 0) return;                  // uniform
    extract(sc);
    wave_sync();
    cx<T> v[CPT];
#pragma unroll
    for (int k = 0; k < CPT; ++k) v[k] = sX[(CPT * h + k) * LX + r];
    const int kp = gj_eliminate<T, SW, TPR, NMAX <= 128>(sm, v, role, sing, p0 + s0, s0, kw, zero_off);
#pragma unroll
    for (int k = 0; k < CPT; ++k) sX[(CPT * h + k) * LX + r] = v[k];
    // the pivot rows' other columns go to sR and are cleared: the product then
    // replaces the pivot rows and accumulates into the others (what it leaves in
    // these SW columns is overwritten by their final values)
#pragma unroll
    for (int rt = 0; rt < NRT; ++rt) {
      const int kr = __shfl(kp, (16 * rt + l16) * TPR, 64);
      if (kr >= 0) {
#pragma unroll
        for (int ct = 0; ct < 2; ++ct)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            sR[kr * WP + 16 * ct + 4 * i + lq] = cx<T>{cre[rt][ct][i], cim[rt][ct][i]};
            cre[rt][ct][i] = T(0);
            cim[rt][ct][i] = T(0);
          }
      }
    }
    __syncthreads();
    if (wo > w) {                         // the outer panel has other columns
      if (s0) put(s0 - SW);
      gather(s0);
    }
    update(sc, kw);
  };
  eliminate(std::integral_constant<int, 0>{});
  eliminate(std::integral_constant<int, 1>{});
  eliminate(std::integral_constant<int, 2>{});
  eliminate(std::integral_constant<int, 3>{});
  if (wo > w) put((w - 1) / SW * SW);
#pragma unroll
  for (int rt = 0; rt < NRT; ++rt) {      // C -> M[:, J]
    const int row = RW * wave + 16 * rt + l16;
    if (row < n) {
#pragma unroll
      for (int ct = 0; ct < 2; ++ct)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int j = 16 * ct + 4 * i + lq;
          if (j < w) gst(J + j * ld + row, cx<T>{cre[rt][ct][i], cim[rt][ct][i]});
        }
    }
  }
  if (live && h == 0) roles[r] = role;
  if (tid < w) d.ipiv[p0 + tid] = sm.piv[tid];
  // info: reset by the first panel, then the first singular column wins
  if (sing != INT_MAX) atomicMin(&sm.sing, sing);
  __syncthreads();
  if (tid == 0 && d.info) {
    const int col = sm.sing == INT_MAX ? 0 : sm.sing;
    if (p0 == 0 || (col && *d.info == 0)) *d.info = col;
  }
}

// The same for blocks of up to GJ_ROWS_MAX rows: four threads per row hold all 32 columns of
// the panel, so that every column is eliminated one by one.  Eight at a time, as
// above, cost these blocks accuracy.  Residual of A A^{-1} (geometric mean over 400
// random blocks and more), over that of one column at a time with every step rounded once:
// complex128 65 rows 1.15, 74 rows 1.11, 95 rows 1.11; with the product of eight added once
// and its steps rounded once (the 128-row instance above) still 1.11, 1.06 and 1.06, and 1.01
// at 97 rows over the earlier panel kernel, which updated all 32 columns by fused
// multiply-adds; from 104 rows on 0.99.  This form: 0.99 to 1.00, and 0.95 at 96 to 112 rows.
// Up to 64 rows it is the faster one too (64 rows 59 against 63 us, complex64 51 against 57);
// above it costs up to a seventh: 74 rows 84 -> 90 us, 95 rows 100 -> 112, 112 rows 119 -> 138 in
// complex128, 74 -> 78, 86 -> 93 and 106 -> 118 in complex64.
constexpr int GJ_ROWS_MAX = 112;
template <class T, int NMAX>
__global__ __launch_bounds__(4 * NMAX) void gj_panel_rows_kernel(const InvDesc<T>* __restrict__ descs, int p0) {
  constexpr int WP = GJM_WP, TPR = 4, CPT = WP / TPR, NT = 4 * NMAX;
  __shared__ GjLds<T, WP> sm;
  const InvDesc<T> d = descs[blockIdx.x];
  const int n = d.n;
  const int64_t ld = d.ld;
  cx<T>* __restrict__ M = d.M;
  cx<T>* __restrict__ R = d.scratch;
  int* __restrict__ roles = reinterpret_cast<int*>(d.scratch + (size_t)WP * n);
  const int w = min(WP, n - p0);
  const int tid = threadIdx.x, r = tid / TPR, h = tid % TPR;
  const bool live = r < n;
  cx<T>* J = M + (int64_t)p0 * ld;
  cx<T> v[CPT];
#pragma unroll
  for (int k = 0; k < CPT; ++k) {
    const int j = CPT * h + k;
    v[k] = gld_at<T>(J, (unsigned)min(j, w - 1) * (unsigned)ld + (unsigned)min(r, n - 1));
    if (!live || j >= w) v[k] = czero<T>();
  }
  int role = -2;
  if (live) role = p0 == 0 ? -1 : roles[r];
  int zero_off = 0;                       // see gj_panel_kernel
  asm("" : "+v"(zero_off));
  int sing = INT_MAX;
  if (tid == 0) sm.sing = INT_MAX;
  if (tid < 4) sm.key[tid] = 0;
  if (tid < WP) sm.piv[tid] = 0;
  __syncthreads();
  gj_eliminate<T, WP, TPR, true>(sm, v, role, sing, p0, 0, w, zero_off);
  __syncthreads();                        // all pivot rows are in sm.piv
  // C -> M[:, J]; a block of one panel goes to its place in its final order,
  // A^{-1}[k, l] = C[r_k, r^{-1}(l)]
  const bool whole = NMAX <= 64 && n <= WP;
  if (live) {
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      const int j = CPT * h + k;
      if (j < w) gst(whole ? d.scratch + sm.piv[j] * n + role : J + j * ld + r, v[k]);
    }
    if (h == 0 && !whole) roles[r] = role;
  }
  if (tid < w) d.ipiv[p0 + tid] = sm.piv[tid];
  // R[k, j] = M[P[k], j] for the columns j outside the panel (rows k from w on repeat
  // row 0's place and are not used)
  if (!whole) {
    const int k = tid % WP;
    const cx<T>* row = M + sm.piv[k];
    constexpr int CS = NT / WP, RB = NMAX / CS;
    cx<T> x[RB];
#pragma unroll
    for (int t = 0; t < RB; ++t) x[t] = gld(row + (int64_t)min(tid / WP + t * CS, n - 1) * ld);
#pragma unroll
    for (int t = 0; t < RB; ++t) {
      const int j = tid / WP + t * CS;
      if (j < n && (j < p0 || j >= p0 + w)) gst(R + (int64_t)j * WP + k, x[t]);
    }
  }
  // info: reset by the first panel, then the first singular column wins
  if (sing != INT_MAX) atomicMin(&sm.sing, sing);
  __syncthreads();
  if (tid == 0 && d.info) {
    const int col = sm.sing == INT_MAX ? 0 : sm.sing;
    if (p0 == 0 || (col && *d.info == 0)) *d.info = col;
  }
}

// The panel's update: M[:, j] += M[:, J] R[:, j] for the columns j of its
// outer panel outside J, the pivot rows' old values counting as zero, on the
// batched GEMM's tile with descriptors made here (columns [q0, p0), then
// [p0 + w, q0 + wo)); K = w <= 32.
// M3 = false up to GJ_ROWS_MAX rows: the 3M product's error (relative to the product of
// the norms and not entry by entry) shows there, residual of complex64 inverses over that of four
// products 1.04 at 48 and 64 rows, 1.09 at 74 and 95, 1.12 at 112.
template <class T, bool M3>
__global__ __launch_bounds__(256, 3) void gj_update_kernel(const InvDesc<T>* __restrict__ descs, int ndesc, int per,
                                                           int p0) {
  constexpr int TS = 32;
  __shared__ GemmLds<T, 1> sm;
  int di, t;
  xcd_item(blockIdx.x, per, ndesc, di, t);
  if (di >= ndesc) return;
  const InvDesc<T> v = descs[di];
  const int n = v.n;
  int q0, wo;
  gj_outer_range(n, p0, q0, wo);
  const int w = min(GJM_WP, n - p0);
  const int n0 = p0 - q0, n1 = q0 + wo - (p0 + w);
  const int tm = (n + TS - 1) / TS, tn0 = n0 / TS;
  int jstart = q0, ncols = n0;
  if (t >= tm * tn0) {
    t -= tm * tn0;
    jstart = p0 + w;
    ncols = n1;
  }
  GemmDesc<T> d{};
  d.A[0] = v.M + (int64_t)p0 * v.ld;
  d.lda[0] = v.ld;
  d.k[0] = w;
  d.B[0] = v.scratch + (size_t)jstart * GJM_WP;
  d.ldb[0] = GJM_WP;
  d.A[1] = nullptr;
  d.B[1] = nullptr;
  d.k[1] = 0;
  d.C = v.M + (int64_t)jstart * v.ld;
  d.ldc = v.ld;
  d.m = n;
  d.n = ncols;
  d.alpha = T(1);
  d.beta = T(1);
  gemm_tile_body<T, 1, M3>(d, t, sm, reinterpret_cast<const int*>(v.scratch + (size_t)GJM_WP * n), p0);
}

// S[l n + k] = M[r_k, r^{-1}(l)], the inverse in its final order and place.  Grid:
// (chunks of cc columns, blocks); a wave takes a column at a time, read whole into
// its part of LDS and gathered from there.  Copying M's columns through LDS
// and the result back over M took, for one block of 500 rows, complex128, 17 + 11 us
// (256 blocks 397 + 413); now 4.6 (383).
template <class T>
__global__ __launch_bounds__(256) void gj_perm_kernel(const InvDesc<T>* __restrict__ descs, int cc) {
  __shared__ int sRinv[512];
  __shared__ int sRow[512];
  __shared__ cx<T> sCol[4][512];
  const InvDesc<T> d = descs[blockIdx.y];
  const int n = d.n, l0 = blockIdx.x * cc;
  for (int j = threadIdx.x; j < n; j += 256) {
    const int rj = d.ipiv[j];
    sRow[j] = rj;
    sRinv[rj] = j;
  }
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int l = l0 + wave; l < min(n, l0 + cc); l += 4) {
    const cx<T>* src = d.M + (int64_t)sRinv[l] * d.ld;
    cx<T>* dst = d.scratch + (int64_t)l * n;
    cx<T> v[8];
#pragma unroll
    for (int t = 0; t < 8; ++t)
      if (64 * t < n) v[t] = gld(src + min(lane + 64 * t, n - 1));
#pragma unroll
    for (int t = 0; t < 8; ++t)
      if (64 * t < n) sCol[wave][lane + 64 * t] = v[t];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    for (int k = lane; k < n; k += 64) gst(dst + k, sCol[wave][sRow[k]]);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
}

// End of outer panel O = [q0, q0 + wo): R_O[k, j] = M[P_O[k], j] for the
// columns j outside O (at R_O[j GJ_WO + k]).
template <class T>
__global__ __launch_bounds__(256) void gj_outer_gather_kernel(const InvDesc<T>* __restrict__ descs, int q0) {
  const InvDesc<T> d = descs[blockIdx.y];
  const int n = d.n;
  const int wo = min(GJ_WO, n - q0);
  const int64_t ld = d.ld;
  cx<T>* __restrict__ M = d.M;
  cx<T>* __restrict__ RO = d.scratch + (size_t)(GJM_WP + 1) * n;
  const int* __restrict__ piv = d.ipiv + q0;
  const int total = (n - wo) * GJ_WO;
  for (int idx = blockIdx.x * 256 + threadIdx.x; idx < total; idx += gridDim.x * 256) {
    const int k = idx % GJ_WO, jc = idx / GJ_WO;
    const int j = jc < q0 ? jc : jc + wo;
    cx<T> x = czero<T>();
    if (k < wo) x = gld(M + (int64_t)j * ld + piv[k]);
    RO[(int64_t)j * GJ_WO + k] = x;
  }
}

// M[:, j] += M[:, O] R_O[:, j] for the columns outside O, the rows P_O replaced:
// the batched GEMM's tile on descriptors made here (columns [0, q0), then [q0 + wo, n)).
template <class T, int S>
__global__ __launch_bounds__(256, 3) void gj_outer_update_kernel(const InvDesc<T>* __restrict__ descs, int ndesc,
                                                                 int per, int q0) {
  constexpr int TS = 32 * S;
  __shared__ GemmLds<T, S> sm;
  int di, t;
  xcd_item(blockIdx.x, per, ndesc, di, t);
  if (di >= ndesc) return;
  const InvDesc<T> v = descs[di];
  const int n = v.n;
  const int wo = min(GJ_WO, n - q0);
  const int n1 = n - q0 - wo;
  const int tm = (n + TS - 1) / TS, tn0 = q0 / TS;
  int jstart = 0, ncols = q0;
  if (t >= tm * tn0) {
    t -= tm * tn0;
    jstart = q0 + wo;
    ncols = n1;
  }
  GemmDesc<T> d{};
  d.A[0] = v.M + (int64_t)q0 * v.ld;
  d.lda[0] = v.ld;
  d.k[0] = wo;
  d.B[0] = v.scratch + (size_t)(GJM_WP + 1) * n + (size_t)jstart * GJ_WO;
  d.ldb[0] = GJ_WO;
  d.A[1] = nullptr;
  d.B[1] = nullptr;
  d.k[1] = 0;
  d.C = v.M + (int64_t)jstart * v.ld;
  d.ldc = v.ld;
  d.m = n;
  d.n = ncols;
  d.alpha = T(1);
  d.beta = T(1);
  gemm_tile_body<T, S>(d, t, sm, reinterpret_cast<const int*>(v.scratch + (size_t)GJM_WP * n), q0);
}

// One workgroup per tile of the columns [q0, p0) and [p0 + w, q0 + wo) of an outer panel:
// p0 - q0 is a multiple of the tile's 32, so that is one column of tiles less than the outer
// panel has.
template <class T>
static void launch_gj_updates(const InvDesc<T>* d_descs, int ndesc, int n, int p0, hipStream_t s) {
  const int q0 = n >= GJ_OUTER_MIN ? p0 / GJ_WO * GJ_WO : 0;
  const int wo = n >= GJ_OUTER_MIN && n - q0 > GJ_WO ? GJ_WO : n - q0;
  const int per = ((n + 31) / 32) * ((wo + 31) / 32 - 1);
  if (per == 0) return;
  const dim3 grid(xcd_grid(ndesc, per));
  if constexpr (sizeof(T) == 4) {
    if (n <= GJ_ROWS_MAX) {
      hipLaunchKernelGGL((gj_update_kernel<T, false>), grid, dim3(256), 0, s, d_descs, ndesc, per, p0);
      return;
    }
  }
  hipLaunchKernelGGL((gj_update_kernel<T, true>), grid, dim3(256), 0, s, d_descs, ndesc, per, p0);
}

// The same for the columns [0, q0) and [q0 + wo, n); q0 is a multiple of 128.
template <class T, int S>
static void launch_gj_outer_updates(const InvDesc<T>* d_descs, int ndesc, int n, int q0, hipStream_t s) {
  constexpr int TS = 32 * S;
  const int n1 = n - q0 > GJ_WO ? n - q0 - GJ_WO : 0;
  const int per = ((n + TS - 1) / TS) * (q0 / TS + (n1 + TS - 1) / TS);
  hipLaunchKernelGGL((gj_outer_update_kernel<T, S>), dim3(xcd_grid(ndesc, per)), dim3(256), 0, s, d_descs, ndesc, per,
                     q0);
}

template <class T>
static hipError_t gj_inverse_launches(const InvDesc<T>* d_descs, int ndesc, int n, hipStream_t s) {
  const int nt = (n + 63) / 64;
  for (int p0 = 0; p0 < n; p0 += GJM_WP) {
    // the smallest workgroup that has the rows: fewer waves meet at a step's barriers
    // (an inversion of one block: complex64 300 rows, 384 instead of 512, 424 -> 388 us,
    // 374 rows 520 -> 477; complex128 150 rows, 192 instead of 256, 194 -> 189)
    auto rows = [&](auto nm) {
      constexpr int NMAX = decltype(nm)::value;
      hipLaunchKernelGGL((gj_panel_rows_kernel<T, NMAX>), dim3(ndesc), dim3(4 * NMAX), 0, s, d_descs, p0);
    };
    auto panel = [&](auto nm) {
      constexpr int NMAX = decltype(nm)::value;
      hipLaunchKernelGGL((gj_panel_kernel<T, NMAX>), dim3(ndesc), dim3(NMAX * GJ_TPR<T, NMAX>), 0, s, d_descs, p0);
    };
    constexpr int MID = sizeof(T) == 4 ? 384 : 512;
    if (n <= 64) rows(std::integral_constant<int, 64>{});
    else if (n <= 96) rows(std::integral_constant<int, 96>{});
    else if (n <= GJ_ROWS_MAX) rows(std::integral_constant<int, GJ_ROWS_MAX>{});
    else if (n <= 128) panel(std::integral_constant<int, 128>{});
    else if (n <= 192) panel(std::integral_constant<int, 192>{});
    else if (n <= 256) panel(std::integral_constant<int, 256>{});
    else if (n <= MID) panel(std::integral_constant<int, MID>{});
    else panel(std::integral_constant<int, 512>{});
    if (n <= GJM_WP) return hipGetLastError();             // one panel, stored in its final order
    launch_gj_updates<T>(d_descs, ndesc, n, p0, s);
    const int pe = p0 + GJM_WP;
    if (n >= GJ_OUTER_MIN && (pe % GJ_WO == 0 || pe >= n)) {         // the end of an outer panel
      const int q0 = (p0 / GJ_WO) * GJ_WO;
      const int chunks = (n * GJ_WO + 255) / 256 < 256 ? (n * GJ_WO + 255) / 256 : 256;
      hipLaunchKernelGGL((gj_outer_gather_kernel<T>), dim3(chunks, ndesc), dim3(256), 0, s, d_descs, q0);
      if (gemm_small_tiles<T>(ndesc, nt * nt, 4 * nt * nt))
        launch_gj_outer_updates<T, 1>(d_descs, ndesc, n, q0, s);
      else
        launch_gj_outer_updates<T, 2>(d_descs, ndesc, n, q0, s);
    }
  }
  // four columns a workgroup (one a wave) on few blocks, 16 where that many
  // workgroups would mostly read the pivots
  const int cc = ndesc <= 32 ? 4 : 16;
  hipLaunchKernelGGL((gj_perm_kernel<T>), dim3((n + cc - 1) / cc, ndesc), dim3(256), 0, s, d_descs, cc);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
template <class T>
hipError_t launch_gemm_batched(const GemmDesc<T>* d_descs, int ndesc, GemmTiles t, hipStream_t s) {
  if (ndesc <= 0 || t.t64 <= 0) return hipSuccess;
  if (gemm_small_tiles<T>(ndesc, t.t64, t.t32))
    hipLaunchKernelGGL((gemm_batched_kernel<T, 1>), dim3(xcd_grid(ndesc, t.t32)), dim3(256), 0, s, d_descs, ndesc,
                       t.t32);
  else
    hipLaunchKernelGGL((gemm_batched_kernel<T, 2>), dim3(xcd_grid(ndesc, t.t64)), dim3(256), 0, s, d_descs, ndesc,
                       t.t64);
  return hipGetLastError();
}

template <class T>
hipError_t launch_gj_inverse(const InvDesc<T>* d_descs, int ndesc, int n, hipStream_t s) {
  if (ndesc <= 0) return hipSuccess;
  if (n < 1 || n > 512) return hipErrorInvalidValue;
  return gj_inverse_launches<T>(d_descs, ndesc, n, s);
}

template hipError_t launch_gemm_batched<double>(const GemmDesc<double>*, int, GemmTiles, hipStream_t);
template hipError_t launch_gemm_batched<float>(const GemmDesc<float>*, int, GemmTiles, hipStream_t);
template hipError_t launch_gj_inverse<double>(const InvDesc<double>*, int, int, hipStream_t);
template hipError_t launch_gj_inverse<float>(const InvDesc<float>*, int, int, hipStream_t);

}  // namespace kore
