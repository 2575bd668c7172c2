// memLS on gfx950: PRECOND, NSSOLVER (GMRES + CG on the Schur complement +
// least-squares combination), GMRESV and CGRADV/CGRADS (memLS.f90).
//
// Design:
//  * The matrix lives as vdof*vdof planes of nnz doubles (plane m = entry
//    (m / vdof, m % vdof) of every row-major block).  Each plane is read with
//    16 lanes per CSR row, so every load instruction covers 128 contiguous
//    bytes.
//  * PRECOND's symmetric diagonal scaling is not written back into Val: every
//    SpMV applies y_r(i) = W_r(i) sum_j A_rc(i,j) W_c(j) x_c(j) + fix_r(i) x_r(i)
//    where fix marks the diagonal entries memLS forces to 1 (zero diagonal,
//    Dirichlet-masked DOF; memLS.f90:1815-1820,1923-1929).  This saves the two
//    read+write sweeps over Val per solve.
//  * Dots and norms are two-stage deterministic reductions: parts per
//    workgroup in a fixed order, summed by whichever kernel needs the result.
//  * GMRES orthogonalises with classical Gram-Schmidt and a DGKS second pass
//    (taken when ||w'|| < ||w||/sqrt 2), computing all i projections of a
//    step in one sweep.  memLS uses modified Gram-Schmidt (memLS.f90:743-746);
//    both produce the same Krylov space, and solutions agree to the solver
//    tolerance.
//  * Every decision of a solve (Givens rotations, convergence tests, CGRAD's
//    iteration count, NSSOLVER's least squares) is taken on the device.  A
//    captured solve enqueues every possible iteration; a plain one runs the
//    same launches, polls the flags from pinned memory and stops enqueueing.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>
#include <chrono>
#include <cmath>
#include <cstring>
#include <functional>
#include <memory>
#include <mutex>
#include <vector>

#include "common.hpp"

using crimson::wave_lds_sync;

namespace {

constexpr int kRowLanes = 16;  // lanes per CSR row in the SpMV kernels
// Row kernels deal their workgroups to the XCDs in turns of this many
// (crimson::xcd_block(chunk)): rows gather the vector at neighbours a mesh
// layer away, which the shared MALL then holds for all XCDs.  One FP64
// timestep of the 64x64x320 cylinder: 2036 ms with one contiguous range per
// XCD, 1966 / 1918 / 1916 / 1915 / 1929 ms with turns of 4 / 8 / 16 / 32 /
// 64 for the Schur CG's two row kernels, 1912 ms with the SpMV too.
constexpr unsigned kRowXcdChunk = 16;

struct SubLs {
  double absTol = 0, relTol = 0, iNorm = 0, fNorm = 0, dB = 0, callD = 0;
  int suc = 0, mItr = 0, sD = 0, itr = 0;
};

// A scaled view of a sub-block (rows r0.., cols c0..) of the stored matrix.
// T is the arithmetic type of the solve: the matrix planes, W, the Krylov
// vectors and every accumulation (FP64, or FP32 in the mixed form).
template <class T>
struct MatView {
  const T *base;  // plane 0
  size_t nnz;
  int plane[16];  // plane index of (r, c), r < NR, c < NC: plane[r * 4 + c]
  const T *W;     // W(wdof, nNo)
  const T *fix;   // fix(wdof, nNo) or null
  int wdof, r0, c0;
};

// The column of block k of `row`: stored as is (int) or as its offset from
// the row (short, lhs->d_col16).
__device__ inline int col_at(const int *__restrict__ col, int k, int row) { return col[k]; }
__device__ inline int col_at(const short *__restrict__ col, int k, int row) { return row + (int)col[k]; }
// One 4-wide node entry (32 bytes in FP64, 16 in FP32; aligned) in 16-byte
// pieces.
__device__ inline void load4(const double *__restrict__ p, double (&z)[4]) {
  const double2 a = reinterpret_cast<const double2 *>(p)[0], b = reinterpret_cast<const double2 *>(p)[1];
  z[0] = a.x;
  z[1] = a.y;
  z[2] = b.x;
  z[3] = b.y;
}
__device__ inline void load4(const float *__restrict__ p, float (&z)[4]) {
  const float4 a = *reinterpret_cast<const float4 *>(p);
  z[0] = a.x;
  z[1] = a.y;
  z[2] = a.z;
  z[3] = a.w;
}
__device__ inline void store4(double *__restrict__ p, const double (&z)[4]) {
  reinterpret_cast<double2 *>(p)[0] = make_double2(z[0], z[1]);
  reinterpret_cast<double2 *>(p)[1] = make_double2(z[2], z[3]);
}
__device__ inline void store4(float *__restrict__ p, const float (&z)[4]) {
  *reinterpret_cast<float4 *>(p) = make_float4(z[0], z[1], z[2], z[3]);
}

// LANES lanes per CSR row: 16 for the 3x3 and 4x4 products, 4 for the
// narrow ones (G, D, L) whose per-entry work is too small to feed 16 lanes.
template <int NR, int NC, class T, int LANES, class IX>
__global__ void __launch_bounds__(256) spmv_kernel(int nNo, const int *__restrict__ rowptr,
                                                   const IX *__restrict__ col, MatView<T> A,
                                                   const T *__restrict__ x, T *__restrict__ y, T ya,
                                                   const T *__restrict__ z, T za,
                                                   const double *__restrict__ skip) {
  if (skip && *skip != 0.0) return;
  const int gid = crimson::xcd_block(kRowXcdChunk) * blockDim.x + threadIdx.x;
  const int row = gid / LANES;
  const int lane = threadIdx.x % LANES;
  T acc[NR];
#pragma unroll
  for (int r = 0; r < NR; ++r) acc[r] = T(0);
  if (row < nNo) {
    const int ke = rowptr[row + 1];
    for (int k = rowptr[row] + lane; k < ke; k += LANES) {
      const int j = col_at(col, k, row);
      T xv[NC];
#pragma unroll
      for (int c = 0; c < NC; ++c) xv[c] = A.W[A.c0 + c + (size_t)A.wdof * j] * x[c + (size_t)NC * j];
#pragma unroll
      for (int r = 0; r < NR; ++r)
#pragma unroll
        for (int c = 0; c < NC; ++c) acc[r] += A.base[(size_t)A.plane[r * 4 + c] * A.nnz + k] * xv[c];
    }
  }
#pragma unroll
  for (int off = LANES / 2; off > 0; off >>= 1)
#pragma unroll
    for (int r = 0; r < NR; ++r) acc[r] += __shfl_xor(acc[r], off, LANES);
  if (row < nNo && lane == 0) {
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      T v = A.W[A.r0 + r + (size_t)A.wdof * row] * acc[r];
      if (A.fix && NR == NC && A.r0 == A.c0) v += A.fix[A.r0 + r + (size_t)A.wdof * row] * x[r + (size_t)NC * row];
      v *= ya;
      if (z) v += za * z[r + (size_t)NR * row];
      y[r + (size_t)NR * row] = v;
    }
  }
}

// The Schur product of NSSOLVER's CG (memLS.f90:1719-1735) after G P:
// SP = L P - Gt t1 with t1 = G P, both scaled views of the same CSR rows, in
// one pass: SP_i = W_i sum_j L_ij (W_j P_j) + fix_i P_i - W_i sum_j Gt_ij (W_j t1_j)
// with Ps = W o P and W o t1 precomputed, gathered per column as one entry
// Z(0:3, j) = (Ps_j, W o t1_j) (the same operations, in the same order, as
// the two separate products).
constexpr int kNarrowLanes = 4;
// Workgroups of a CG sweep at most (8 per CU): each writes one part of a dot,
// and every workgroup of the next sweep sums all of them.
constexpr int kCgGrid = 2048;

// What a deciding kernel tells the host of a solve that is not captured: its
// place in the solve's sequence and whether the loop it belongs to is over,
// as one word of pinned memory that the host polls, so that no copy or event
// stands between two steps.  p is null in a captured solve.
struct HostFlag {
  unsigned long long *p;
  unsigned long long seq;
  __device__ void tell(bool stop) const {
    if (p) __hip_atomic_store(p, seq << 1 | (stop ? 1u : 0u), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
};

// A coupled face of the Schur CG (ADDBCMUL's PRE, memLS.f90:1719-1735).  PRE
// adds coef_f S_f valM_f to t1 = G P with S_f = valM_f . t1; with Gt = -G^T
// (DEPART) that is the symmetric rank-one term c_f q_f q_f^T on the
// Schur operator, q_f = W_p o (G^T (W_u o valM_f)) on the columns of the
// face nodes' rows (sup): q_j = W_p(j) sum over the pairs (a, k) of column j
// of valM(i, a) W_u(i, glob(a)) G_i(k), i < min(dof, 3).  So S_f = q_f . P is
// formed from the direction, the denominator P . SP gains c_f S_f^2 and the
// residual update alpha c_f S_f q_f: the operator's kernels see no face.
struct FaceDev {
  const int *glob;
  const double *valM;
  const double *coefp;  // c_f = -res / (1 + res nS) (BCPRE)
  double res;           // the face's coupling coefficient (ADDBCMUL without PRE)
  int nNo, dof;
  const int *sup;
  const double *q;
  int nsup;
};
// Workgroups per face computing S_f's partial sums beside the direction update or the
// product: kFaceDotBlocks for supports of up to kFaceDotShare entries each, twice as
// many (2^kFaceDotMost at most) until a larger one's shares are so small, so that no
// face's few workgroups outlast the sweep they stand beside.
// An outlet of 37,585 nodes (support 77,000), 654,000 rows, FP32: 500 CG iterations took
// 70.0 ms with four, 62.8 with 32.
constexpr int kFaceDotLog = 2, kFaceDotBlocks = 1 << kFaceDotLog, kFaceDotMost = 6, kFaceDotShare = 4096;
// The faces' supports merged for the residual update: the nodes of any of them,
// ascending, each with its first entry (face, place in the face's support) and where
// the others lie in ent, in face order; tptr[t] is the first of the nodes 256 t and
// above.
struct FaceEnt {
  int f, s;
};
struct FaceNode {
  int node, more, end;
  FaceEnt first;
};
struct FaceList {
  int nfc;               // coupled faces
  int nb, lb;            // workgroups, and partial sums of S_f, per face; nb = 1 << lb
  const FaceDev *fd;
  const FaceNode *node;
  const FaceEnt *ent;
  const int *tptr;       // (N / 256 rounded up) + 1 entries
  double *part;          // nb partial sums of S_f per face
  const double *coef;    // c_f
};
// Faces whose terms c_f S_f a workgroup of the residual update keeps in LDS; a node's
// entries then cost it two loads each.  (329,000 rows, 24 faces on the same 12,637
// nodes: an NS solve took 604 ms with every entry summing its face's parts again
// and one thread walking a node's entries among its idle neighbours, 69 so; one
// face 32.)
constexpr int kFaceLds = 256;  // one per thread

// Wave-level sum (64 lanes) then across the 4 waves of a 256-thread group.
template <class T>
__device__ inline T block_sum(T v, T *sh) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  const int w = threadIdx.x / 64;
  if ((threadIdx.x & 63) == 0) sh[w] = v;
  __syncthreads();
  T t = T(0);
  if (threadIdx.x == 0) t = (sh[0] + sh[1]) + (sh[2] + sh[3]);
  __syncthreads();
  return t;
}

// block_sum's value in every thread of the workgroup.
template <class T>
__device__ inline T block_sum_all(T v, T *sh) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  const int w = threadIdx.x / 64;
  if ((threadIdx.x & 63) == 0) sh[w] = v;
  __syncthreads();
  const T t = (sh[0] + sh[1]) + (sh[2] + sh[3]);
  __syncthreads();
  return t;
}

// Entries per lane loaded ahead in the narrow row kernels: the column
// indices of kNarrowUnroll entries (k, k + 4, ...) are loaded together, then
// the gathered vector entries and matrix values, so a lane waits for one
// index load and one gather per kNarrowUnroll entries instead of per entry.
// Indices past the row end are clamped to its last entry (in bounds; the
// product is not added), so the accumulation order is the plain loop's.
constexpr int kNarrowUnroll = 4;

// The Schur operator as two passes, for a matrix whose complement is not
// formed (schur_pattern): on Ps = W_p o P the G product writes
// Z(0:3, i) = (Ps_i, W_u o (W_u o G Ps)_i), and the second pass
// gathers both of its operands of a column as one 4-wide entry (two 16-byte
// loads in FP64, one in FP32): SP_i = W_i (sum_j L_ij Ps_j - Gt_ij . Z(1:3, j)) + fix_i P_i.
// `done`: the CG's converged flag; launches after it return at once.
template <class T, class IX, int U = kNarrowUnroll>
__global__ void __launch_bounds__(256) g_product_kernel(int nNo, const int *__restrict__ rowptr,
                                                        const IX *__restrict__ col, MatView<T> G,
                                                        const T *__restrict__ Ps, T *__restrict__ Z,
                                                        const double *__restrict__ done) {
  if (done && *done != 0.0) return;
  const int gid = crimson::xcd_block(kRowXcdChunk) * blockDim.x + threadIdx.x;
  const int row = gid / kNarrowLanes;
  const int lane = threadIdx.x % kNarrowLanes;
  T acc[3] = {T(0), T(0), T(0)};
  if (row < nNo) {
    const int ke = rowptr[row + 1];
    const T *g0 = G.base + (size_t)G.plane[0] * G.nnz, *g1 = G.base + (size_t)G.plane[4] * G.nnz,
            *g2 = G.base + (size_t)G.plane[8] * G.nnz;
    for (int k = rowptr[row] + lane; k < ke; k += kNarrowLanes * U) {
      int j[U], kc[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        kc[u] = min(k + kNarrowLanes * u, ke - 1);
        j[u] = col_at(col, kc[u], row);
      }
      T xv[U], a0[U], a1[U], a2[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        xv[u] = Ps[j[u]];
        a0[u] = g0[kc[u]];
        a1[u] = g1[kc[u]];
        a2[u] = g2[kc[u]];
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (k + kNarrowLanes * u < ke) {
          acc[0] += a0[u] * xv[u];
          acc[1] += a1[u] * xv[u];
          acc[2] += a2[u] * xv[u];
        }
    }
  }
#pragma unroll
  for (int off = kNarrowLanes / 2; off > 0; off >>= 1)
#pragma unroll
    for (int r = 0; r < 3; ++r) acc[r] += __shfl_xor(acc[r], off, kNarrowLanes);
  if (row < nNo && lane == 0) {
    T z[4];
    z[0] = Ps[row];
#pragma unroll
    for (int r = 0; r < 3; ++r) {
      const T w = G.W[G.r0 + r + (size_t)G.wdof * row];
      z[1 + r] = w * (w * acc[r]);
    }
    store4(Z + (size_t)4 * row, z);
  }
}
template <class T, class IX, int U = kNarrowUnroll>
__global__ void __launch_bounds__(256) schur_kernel(int nNo, const int *__restrict__ rowptr,
                                                    const IX *__restrict__ col, MatView<T> Lv, MatView<T> Gv,
                                                    const T *__restrict__ P, const T *__restrict__ Z,
                                                    T *__restrict__ SP, const double *__restrict__ done) {
  if (done && *done != 0.0) return;
  const int gid = crimson::xcd_block(kRowXcdChunk) * blockDim.x + threadIdx.x;
  const int row = gid / kNarrowLanes;
  const int lane = threadIdx.x % kNarrowLanes;
  T aL = T(0), aG = T(0);
  if (row < nNo) {
    const int ke = rowptr[row + 1];
    const T *lp = Lv.base + (size_t)Lv.plane[0] * Lv.nnz;
    const T *d0 = Gv.base + (size_t)Gv.plane[0] * Gv.nnz, *d1 = Gv.base + (size_t)Gv.plane[1] * Gv.nnz,
            *d2 = Gv.base + (size_t)Gv.plane[2] * Gv.nnz;
    for (int k = rowptr[row] + lane; k < ke; k += kNarrowLanes * U) {
      int j[U], kc[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        kc[u] = min(k + kNarrowLanes * u, ke - 1);
        j[u] = col_at(col, kc[u], row);
      }
      T l[U], ps[U], b0[U], b1[U], b2[U], x0[U], x1[U], x2[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        l[u] = lp[kc[u]];
        b0[u] = d0[kc[u]];
        b1[u] = d1[kc[u]];
        b2[u] = d2[kc[u]];
        T z[4];
        load4(Z + (size_t)4 * j[u], z);
        ps[u] = z[0];
        x0[u] = z[1];
        x1[u] = z[2];
        x2[u] = z[3];
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (k + kNarrowLanes * u < ke) {
          aL += l[u] * ps[u];
          aG += b0[u] * x0[u];
          aG += b1[u] * x1[u];
          aG += b2[u] * x2[u];
        }
    }
  }
#pragma unroll
  for (int off = kNarrowLanes / 2; off > 0; off >>= 1) {
    aL += __shfl_xor(aL, off, kNarrowLanes);
    aG += __shfl_xor(aG, off, kNarrowLanes);
  }
  if (row < nNo && lane == 0) {
    T v = Lv.W[Lv.r0 + (size_t)Lv.wdof * row] * aL;
    if (Lv.fix) v += Lv.fix[Lv.r0 + (size_t)Lv.wdof * row] * P[row];
    const T t2 = Gv.W[Gv.r0 + (size_t)Gv.wdof * row] * aG;
    SP[row] = v - t2;
  }
}

// ----- the Schur complement formed explicitly -----
// S = W_p (L - Gt W_u^2 G) W_p + fix on the graph's two-ring (a node's
// neighbours' neighbours), one row kernel per CG iteration instead of the
// two passes above.
// What it saves: on the Kuhn meshes a row has 65 entries of S (10 bytes each
// with the 2-byte column) against 14.7 blocks of seven planes read in two
// passes (60 bytes each), and one launch less; the vector P is gathered
// directly (the scaling is in S).
// The pattern is a property of the graph: built once per handle on the
// device, one wave per row, the union of the neighbours' rows in an LDS hash
// set.  Where S is not formed (schur_pays, schur_pattern) the two passes stay.
constexpr int kSchurRow = 320;   // entries of a row of S at most: 16 rows' staging fits 64 KB of LDS
constexpr int kSchurHash = 512;  // LDS hash slots per row, a power of two above kSchurRow
// FILL false: cnt[row] = the row's entries (kSchurRow + 1 when it has more);
// FILL true: the row's columns, ascending, at scol[sptr[row]] (as offsets
// from the row when OX is short).
template <class IX, class OX, bool FILL>
__global__ void __launch_bounds__(256) schur_pattern_kernel(int nNo, const int *__restrict__ rowptr,
                                                            const IX *__restrict__ col, int *__restrict__ cnt,
                                                            const int *__restrict__ sptr, OX *__restrict__ scol) {
  __shared__ int key_all[4][kSchurHash];
  __shared__ int list_all[FILL ? 4 : 1][kSchurRow];
  __shared__ int num_all[4];
  const int w = threadIdx.x / 64, lane = threadIdx.x % 64;
  const int row = blockIdx.x * 4 + w;
  if (row >= nNo) return;  // whole waves: nothing below synchronises the workgroup
  int *key = key_all[w];
  int *num = num_all + w;
  for (int t = lane; t < kSchurHash; t += 64) key[t] = -1;
  if (lane == 0) *num = 0;
  wave_lds_sync();
  bool over = false;
  for (int k = rowptr[row]; k < rowptr[row + 1]; ++k) {
    const int j = col_at(col, k, row);
    const int m1 = rowptr[j + 1];
    for (int m = rowptr[j] + lane; m < m1; m += 64) {
      const int c = col_at(col, m, j);
      unsigned h = ((unsigned)c * 2654435761u) >> 23;
      for (int t = 0; t < kSchurHash; ++t, h = (h + 1) & (kSchurHash - 1)) {  // ends when the table is full
        const int old = atomicCAS(&key[h], -1, c);
        if (old == -1) atomicAdd(num, 1);
        if (old == -1 || old == c) break;
      }
    }
    wave_lds_sync();
    if (*(volatile int *)num > kSchurRow) {
      over = true;
      break;
    }
  }
  if (!FILL) {
    if (lane == 0) cnt[row] = over ? kSchurRow + 1 : *num;
    return;
  }
  // the keys compacted, then each written at its rank
  int *list = list_all[FILL ? w : 0];
  int n = 0;
  for (int t = lane; t < kSchurHash; t += 64) {
    const bool has = key[t] >= 0;
    const unsigned long long mask = __ballot(has);
    const int at = n + __popcll(mask & ((1ull << lane) - 1ull));
    if (has && at < kSchurRow) list[at] = key[t];
    n += __popcll(mask);
  }
  wave_lds_sync();
  const int s0 = sptr[row];
  n = min(n, sptr[row + 1] - s0);
  for (int t = lane; t < n; t += 64) {
    const int c = list[t];
    int rank = 0;
    for (int u = 0; u < n; ++u) rank += list[u] < c;
    scol[s0 + rank] = (OX)(sizeof(OX) == 2 ? c - row : c);
  }
}
// The values of S, 16 lanes per row: the row's accumulators and columns in
// LDS; for each neighbour j the lanes take the entries of row j of G (all of
// different columns, so no two lanes add to one accumulator), in row order;
// sums in FP64.
// Dynamic LDS: 16 rows x maxn (double, int).
template <class T, class IX, class OX>
__global__ void __launch_bounds__(256) schur_values_kernel(int nNo, const int *__restrict__ rowptr,
                                                           const IX *__restrict__ col, MatView<T> Lv, MatView<T> Gtv,
                                                           MatView<T> Gv, const int *__restrict__ sptr,
                                                           const OX *__restrict__ scol, T *__restrict__ S, int maxn) {
  extern __shared__ double dyn[];
  const int g = threadIdx.x / 16, lane = threadIdx.x % 16;
  double *acc = dyn + (size_t)g * maxn;
  int *sc = reinterpret_cast<int *>(dyn + (size_t)16 * maxn) + (size_t)g * maxn;
  const int row = crimson::xcd_block(kRowXcdChunk) * 16 + g;
  const bool live = row < nNo;
  const int s0 = live ? sptr[row] : 0, n = live ? sptr[row + 1] - s0 : 0;
  for (int t = lane; t < n; t += 16) {
    sc[t] = col_at(scol, s0 + t, row);
    acc[t] = 0.0;
  }
  wave_lds_sync();
  auto find = [&](int c) {  // c is in the row
    int lo = 0, hi = n - 1;
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (sc[mid] < c)
        lo = mid + 1;
      else
        hi = mid;
    }
    return lo;
  };
  const T *lp = Lv.base + (size_t)Lv.plane[0] * Lv.nnz;
  const T *b0 = Gtv.base + (size_t)Gtv.plane[0] * Gtv.nnz, *b1 = Gtv.base + (size_t)Gtv.plane[1] * Gtv.nnz,
          *b2 = Gtv.base + (size_t)Gtv.plane[2] * Gtv.nnz;
  const T *g0 = Gv.base + (size_t)Gv.plane[0] * Gv.nnz, *g1 = Gv.base + (size_t)Gv.plane[4] * Gv.nnz,
          *g2 = Gv.base + (size_t)Gv.plane[8] * Gv.nnz;
  const int k0 = live ? rowptr[row] : 0, k1 = live ? rowptr[row + 1] : 0;
  for (int kb = k0; kb < k1; kb += 16) {
    const int k = kb + lane;
    int m0 = 0, m1 = 0, j = 0;
    double d0 = 0.0, d1 = 0.0, d2 = 0.0;
    if (k < k1) {
      j = col_at(col, k, row);
      m0 = rowptr[j];
      m1 = rowptr[j + 1];
      const T *w = Gv.W + Gv.r0 + (size_t)Gv.wdof * j;
      d0 = (double)b0[k] * ((double)w[0] * (double)w[0]);
      d1 = (double)b1[k] * ((double)w[1] * (double)w[1]);
      d2 = (double)b2[k] * ((double)w[2] * (double)w[2]);
      acc[find(j)] += (double)lp[k];
    }
    wave_lds_sync();
    const int cnt = min(16, k1 - kb);
    for (int t = 0; t < cnt; ++t) {
      const int a0 = __shfl(m0, t, 16), a1 = __shfl(m1, t, 16), jj = __shfl(j, t, 16);
      const double e0 = __shfl(d0, t, 16), e1 = __shfl(d1, t, 16), e2 = __shfl(d2, t, 16);
      for (int m = a0 + lane; m < a1; m += 16) {
        const double v = e0 * (double)g0[m] + e1 * (double)g1[m] + e2 * (double)g2[m];
        acc[find(col_at(col, m, jj))] -= v;
      }
      wave_lds_sync();
    }
  }
  if (!live) return;
  const double wr = (double)Lv.W[Lv.r0 + (size_t)Lv.wdof * row];
  const double fx = Lv.fix ? (double)Lv.fix[Lv.r0 + (size_t)Lv.wdof * row] : 0.0;
  for (int t = lane; t < n; t += 16) {
    const int c = sc[t];
    double v = wr * acc[t] * (double)Lv.W[Lv.c0 + (size_t)Lv.wdof * c];
    if (c == row) v += fx;
    S[s0 + t] = (T)v;
  }
}
// SP = S P and the workgroup's part of P . SP, 16 lanes per row.  At most
// kCgGrid workgroups walk the row tiles, so that the residual update sums at
// most that many parts; the next tile's row pointers are loaded during a tile.
// Bound by the read of S: 65 entries per row and 458,000 rows (297 MB) take 74 us,
// 4.0 TB/s of a copy's 4.65; the two passes it replaces took 92 us.  A lane loads kSUnroll
// entries at once, so that the Kuhn meshes' rows (65 at most) are one turn (30 to 45 % of
// a Delaunay mesh's rows have more than 80 entries and take a second): 98 us
// with four, 90 with 8 lanes of eight, 99 with 32 lanes of two, 95 with a wave
// per run of four rows summed through LDS; unbounded grid 67 us, but then a dot
// kernel of its own follows.
constexpr int kSLanes = 16, kSUnroll = 5;
template <class T, class OX>
__global__ void __launch_bounds__(256) s_product_kernel(int nNo, int ntile, const int *__restrict__ sptr,
                                                        const OX *__restrict__ scol, const T *__restrict__ S,
                                                        const T *__restrict__ P, T *__restrict__ SP,
                                                        double *__restrict__ dpart, const double *__restrict__ done) {
  __shared__ double sh[4];
  const double stop = *done;
  const int lane = threadIdx.x % kSLanes;
  auto row_of = [&](int vb) {
    return (int)crimson::xcd_block(kRowXcdChunk, vb, ntile) * (256 / kSLanes) + (int)threadIdx.x / kSLanes;
  };
  int rown = row_of(blockIdx.x), kbn = sptr[min(rown, nNo)], ken = sptr[min(rown + 1, nNo)];
  if (stop != 0.0) return;
  double den = 0.0;
  for (int vb = blockIdx.x; vb < ntile; vb += gridDim.x) {
    const int row = rown, kb = kbn, ke = ken;  // rows past the last one: kb = ke
    const int vn = vb + gridDim.x;
    if (vn < ntile) {
      rown = row_of(vn);
      kbn = sptr[min(rown, nNo)];
      ken = sptr[min(rown + 1, nNo)];
    }
    T acc = T(0);
    for (int k = kb + lane; k < ke; k += kSLanes * kSUnroll) {
      T v[kSUnroll], x[kSUnroll];
      int j[kSUnroll];
#pragma unroll
      for (int u = 0; u < kSUnroll; ++u) {
        const int kc = min(k + kSLanes * u, ke - 1);
        j[u] = col_at(scol, kc, row);
        v[u] = S[kc];
      }
#pragma unroll
      for (int u = 0; u < kSUnroll; ++u) x[u] = P[j[u]];
#pragma unroll
      for (int u = 0; u < kSUnroll; ++u)
        if (k + kSLanes * u < ke) acc += v[u] * x[u];
    }
#pragma unroll
    for (int off = kSLanes / 2; off > 0; off >>= 1) acc += __shfl_xor(acc, off, kSLanes);
    if (row < nNo && lane == 0) {
      SP[row] = acc;
      den += (double)P[row] * (double)acc;
    }
  }
  den = block_sum(den, sh);
  if (threadIdx.x == 0) dpart[blockIdx.x] = den;
}
// The sum of n <= kCgGrid parts, in every thread, always in the same order: every
// thread's parts are loaded together (one wait instead of eight).
__device__ inline double sum_parts(const double *__restrict__ part, int n, double more, double *sh) {
  double v[kCgGrid / 256];
#pragma unroll
  for (int u = 0; u < kCgGrid / 256; ++u) {
    const int b = threadIdx.x + 256 * u;
    v[u] = b < n ? part[b] : 0.0;
  }
#pragma unroll
  for (int u = 0; u < kCgGrid / 256; ++u) more += v[u];
  return block_sum_all(more, sh);
}

// gst (double, device): the state of the solve and of its last GMRES and
// CG calls, then the GMRES Hessenberg system, the Gram system and the
// solution coefficients.
enum GstIdx : int {
  G_RI_SKIP = 0,  // the outer loop has stopped (converged or failed)
  G_RI_ITR,
  G_RI_SUC,
  G_RI_INORM,
  G_RI_FNORM,
  G_RI_EPS,
  G_RI_DBPRE,
  G_ERR,  // 1: singular GE
  G_GM_CYC = 8,  // this GMRES call does nothing more (done, or not running)
  G_GM_ARN,      // no further Arnoldi step in this cycle
  G_GM_EPS,
  G_GM_I,
  G_GM_ITR,
  G_GM_SUC,
  G_GM_INORM,
  G_GM_FNORM,
  G_GM_DBPRE,
  G_GM_SCALE,
  G_GM_APPLY,
  G_GM_EARLY,
  G_GM_LASTF,  // fNorm and dB of the last GMRES call that ran to the end
  G_GM_LASTD,
  G_CG_ITR = 24,
  G_CG_SUC,
  G_CG_INORM,
  G_CG_ERR,
  G_CG_ERRO,
  G_RC_N2 = 30,
  G_NS_CNT,
  G_GM_E0,  // the first residual norm of the GMRES call
  G_GM_N1,  // ||y'||^2 after an Arnoldi step's first pass, and whether it took the second
  G_GM_TWICE,
  G_ARR = 64
};

// ----- dots and the Arnoldi step -----
// v (1024 threads) summed over the workgroup, in every thread, always in the
// same order.
constexpr int kDotThreads = 1024, kDotGrid = 256, kDotGroup = 8;
__device__ inline double wave_sum(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}
__device__ inline double block_sum_1024(double v, double *sh) {
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x / 64] = v;
  __syncthreads();
  double t = threadIdx.x % 64 < 16 ? sh[threadIdx.x % 64] : 0.0;
#pragma unroll
  for (int off = 8; off > 0; off >>= 1) t += __shfl_xor(t, off, 16);
  t = __shfl(t, 0, 64);
  __syncthreads();
  return t;
}
// Parts of the dots of v with U_j = U0 + j ustride, j < m, and of v with itself
// as the m-th when self: part[j * gridDim.x + blockIdx.x], summed by the kernel
// that needs them.  At most kDotGrid workgroups of 16 waves walk the entries;
// a grid row takes kDotGroup vectors.  (All vectors in one grid row, one after the
// other with two barriers each, took 43 us for 50 vectors of 20,000 entries.)
template <class T>
__device__ inline void dots_body(size_t L, const T *__restrict__ v, const T *__restrict__ U0, size_t ustride, int m,
                                 int self, double *__restrict__ part, double (*sh)[kDotGroup]) {
  const int j0 = blockIdx.y * kDotGroup, nb = gridDim.x;
  const int n = min(kDotGroup, m + self - j0);
  double acc[kDotGroup];
#pragma unroll
  for (int q = 0; q < kDotGroup; ++q) acc[q] = 0.0;
  for (size_t e = (size_t)blockIdx.x * kDotThreads + threadIdx.x; e < L; e += (size_t)nb * kDotThreads) {
    const double x = (double)v[e];
    T u[kDotGroup];
#pragma unroll
    for (int q = 0; q < kDotGroup; ++q) u[q] = j0 + q < m ? U0[ustride * (j0 + q) + e] : v[e];
#pragma unroll
    for (int q = 0; q < kDotGroup; ++q) acc[q] += (double)u[q] * x;
  }
#pragma unroll
  for (int q = 0; q < kDotGroup; ++q)
    if (q < n) acc[q] = wave_sum(acc[q]);  // n is the workgroup's
  if ((threadIdx.x & 63) == 0)
#pragma unroll
    for (int q = 0; q < kDotGroup; ++q) sh[threadIdx.x / 64][q] = acc[q];
  __syncthreads();
  if ((int)threadIdx.x < n) {
    double t = 0.0;
    for (int w = 0; w < kDotThreads / 64; ++w) t += sh[w][threadIdx.x];
    part[(size_t)(j0 + threadIdx.x) * nb + blockIdx.x] = t;
  }
}
template <class T>
__global__ void __launch_bounds__(kDotThreads) dots_kernel(size_t L, const T *__restrict__ v,
                                                           const T *__restrict__ U0, size_t ustride, int m, int self,
                                                           double *__restrict__ part,
                                                           const double *__restrict__ skip) {
  if (skip && *skip != 0.0) return;
  __shared__ double sh[kDotThreads / 64][kDotGroup];
  dots_body(L, v, U0, ustride, m, self, part, sh);
}
// The sum of n <= kDotGrid parts by one wave, in every lane.
__device__ inline double wave_parts(const double *__restrict__ part, int n) {
  const int lane = threadIdx.x % 64;
  double v[kDotGrid / 64];
#pragma unroll
  for (int u = 0; u < kDotGrid / 64; ++u) v[u] = lane + 64 * u < n ? part[lane + 64 * u] : 0.0;
  double t = 0.0;
#pragma unroll
  for (int u = 0; u < kDotGrid / 64; ++u) t += v[u];
  return wave_sum(t);
}

// One Arnoldi step (classical Gram-Schmidt with one DGKS pass) without a host
// decision:
//   arnoldi_spmv   u = w / ||w|| (the new basis vector) and y = A u; a workgroup of
//                  its own does gm_givens of the step before (small systems)
//   face_apply     the coupled faces' terms on y (when there are any)
//   dots           y against the basis, and y . y
//   then, up to kOrthMost entries, where a launch costs more than its work:
//   arnoldi_orth   y -= U h, parts of y . y, and y against the basis again
//   arnoldi_orth   the second pass, where ||y'||^2 < ||y||^2 / 2 (every workgroup
//                  takes that decision itself from the same parts), and W o y
// or, for longer vectors, whose second pass over the basis should not be made before
// it is known to be needed:
//   arnoldi_sub    y -= U h, W o y for the next product, parts of y . y
//   dots, sub      the second pass
//   gm_givens      the Hessenberg column, rotations, test and 1 / ||y||
// Every U_j is stored normalised.  The product gathers W o w, one aligned entry of 2
// or 4 components per column, in place of W and w.
// Arnoldi step i's Hessenberg column, rotations and test; H (sD+1, sD)
// column-major; s2: ||y||^2 after the second pass, where it was taken.  One
// workgroup.  The column and the rotations pass through LDS, where the
// chain of rotations takes an LDS read a step instead of a memory round trip.
struct Givens {
  double *g;
  int i, sD;
  const double *h1, *h2, *n2;
  int nb;
  double *H, *cs, *sn, *err;
  HostFlag hf;
};
__device__ inline void gm_givens(const Givens &G, double s2, double (&w3)[3][256]) {
#pragma clang fp contract(off)
  double *g = G.g;
  if (g[G_GM_ARN] != 0.0) {
    if (threadIdx.x == 0) G.hf.tell(true);
    return;
  }
  __syncthreads();  // (w3 may have been read)
  double(&hc)[256] = w3[0], (&c)[256] = w3[1], (&s)[256] = w3[2];
  const int t = threadIdx.x, i = G.i, ld = G.sD + 1;
  const bool gt = g[G_GM_TWICE] != 0.0;
  if (t < i) {
    hc[t] = G.h1[t] + (gt ? G.h2[t] : 0.0);
    if (t < i - 1) {
      c[t] = G.cs[t];
      s[t] = G.sn[t];
    }
  }
  __syncthreads();
  if (t == 0) {
    const double hl = sqrt(gt ? s2 : g[G_GM_N1]);
    g[G_GM_ITR] = g[G_GM_ITR] + 1.0;
    g[G_GM_SCALE] = 1.0 / hl;
    double a = hc[0];
    for (int j = 1; j <= i - 1; ++j) {
      const double b = hc[j];
      hc[j - 1] = c[j - 1] * a + s[j - 1] * b;
      a = -s[j - 1] * a + c[j - 1] * b;
    }
    const double tmp = sqrt(a * a + hl * hl);
    const double ci = a / tmp, si = hl / tmp;
    G.cs[i - 1] = ci;
    G.sn[i - 1] = si;
    hc[i - 1] = tmp;
    const double e = G.err[i - 1];
    G.err[i] = -si * e;
    G.err[i - 1] = ci * e;
    g[G_GM_I] = (double)i;
    const bool done = fabs(-si * e) < g[G_GM_EPS];
    if (done) {
      g[G_GM_SUC] = 1.0;
      g[G_GM_ARN] = 1.0;
    }
    G.hf.tell(done);
  }
  __syncthreads();
  if (t < i) G.H[t + (size_t)ld * (i - 1)] = hc[t];
}
template <int NC>
struct ArnoldiPad {
  static constexpr int n = NC == 3 ? 4 : NC;  // components of a gathered entry
};
template <int NC, class T>
__device__ inline void load_entry(const T *__restrict__ p, T (&x)[NC]) {
  if constexpr (NC >= 3) {
    T z[4];
    load4(p, z);
#pragma unroll
    for (int c = 0; c < NC; ++c) x[c] = z[c];
  } else {
#pragma unroll
    for (int c = 0; c < NC; ++c) x[c] = p[c];
  }
}
template <int NC, class T, class IX>
__global__ void __launch_bounds__(256) arnoldi_spmv_kernel(int nNo, const int *__restrict__ rowptr,
                                                           const IX *__restrict__ col, MatView<T> A,
                                                           const T *__restrict__ w, const T *__restrict__ ws,
                                                           T *__restrict__ u, T *__restrict__ y, Givens G) {
  constexpr int LANES = NC >= 3 ? kRowLanes : kNarrowLanes, PAD = ArnoldiPad<NC>::n;
  __shared__ double sh[4], w3[3][256];
  // G.i > 0: the step before ends here, workgroup 0 with its gm_givens, the others
  // with 1 / ||w||.  (A step launched past the last one, while workgroup 0 tells so,
  // writes vectors that nothing reads.)
  double stop = G.g[G_GM_ARN], scale = G.g[G_GM_SCALE];
  if (G.i > 0) {
    // workgroup 0 may set the flag during this launch: one thread's read counts
    if (threadIdx.x == 0) w3[0][0] = stop;
    const double n1 = G.g[G_GM_N1], twice = G.g[G_GM_TWICE];
    const double s2 = block_sum_all((int)threadIdx.x < G.nb ? G.n2[threadIdx.x] : 0.0, sh);
    if (blockIdx.x == 0) {
      gm_givens(G, s2, w3);
      return;
    }
    stop = w3[0][0];
    scale = 1.0 / sqrt(twice != 0.0 ? s2 : n1);
  }
  const int own = G.i > 0 ? 1 : 0;
  const int gid = crimson::xcd_block(kRowXcdChunk, blockIdx.x - own, gridDim.x - own) * blockDim.x + threadIdx.x;
  const int row = gid / LANES, lane = threadIdx.x % LANES;
  const int kb = rowptr[min(row, nNo)], ke = rowptr[min(row + 1, nNo)];
  if (stop != 0.0) return;
  T acc[NC];
#pragma unroll
  for (int r = 0; r < NC; ++r) acc[r] = T(0);
  for (int k = kb + lane; k < ke; k += LANES) {
    T a[NC * NC], x[NC];
    const int j = col_at(col, k, row);
#pragma unroll
    for (int r = 0; r < NC; ++r)
#pragma unroll
      for (int c = 0; c < NC; ++c) a[r * NC + c] = A.base[(size_t)A.plane[r * 4 + c] * A.nnz + k];
    load_entry<NC>(ws + (size_t)PAD * j, x);
#pragma unroll
    for (int r = 0; r < NC; ++r)
#pragma unroll
      for (int c = 0; c < NC; ++c) acc[r] += a[r * NC + c] * x[c];
  }
#pragma unroll
  for (int off = LANES / 2; off > 0; off >>= 1)
#pragma unroll
    for (int r = 0; r < NC; ++r) acc[r] += __shfl_xor(acc[r], off, LANES);
  if (row < nNo && lane == 0) {
    const T s = (T)scale;
#pragma unroll
    for (int r = 0; r < NC; ++r) {
      const size_t e = r + (size_t)NC * row, f = A.r0 + r + (size_t)A.wdof * row;
      const T ur = s * w[e];
      u[e] = ur;
      y[e] = A.W[f] * (s * acc[r]) + A.fix[f] * ur;
    }
  }
}
// whether the second pass is taken: parts n1[0, nb) of ||y'||^2 against n0 =
// ||y||^2; the same answer in every thread of every workgroup
__device__ inline bool dgks_pass(const double *__restrict__ n0, const double *__restrict__ n1, int nb, double *sh) {
  const double s = block_sum_1024((int)threadIdx.x < nb ? n1[threadIdx.x] : 0.0, sh);
  return s < 0.5 * *n0;
}
template <class T>
__global__ void __launch_bounds__(kDotThreads) dots2_kernel(size_t L, const T *__restrict__ v,
                                                            const T *__restrict__ U0, size_t ustride, int m,
                                                            double *__restrict__ part,
                                                            const double *__restrict__ n0,
                                                            const double *__restrict__ n1, int nb,
                                                            const double *__restrict__ skip) {
  if (*skip != 0.0) return;
  __shared__ double sh[kDotThreads / 64][kDotGroup];
  if (!dgks_pass(n0, n1, nb, &sh[0][0])) return;
  dots_body(L, v, U0, ustride, m, 0, part, sh);
}
// h = the dots' sums (np parts each; self: the m-th is ||y||^2), y -= U h and
// its scaled copy, parts of y . y.  n1 (the second pass): taken or left
// as dgks_pass says, which is noted in g.
constexpr int kSubGrid = 1024;
template <class T>
__device__ inline void sub_coefs(int m, int self, const double *__restrict__ part, int np, double *__restrict__ h,
                                 T (&cs)[256]) {
  for (int j = threadIdx.x / 64; j < m + self; j += kDotThreads / 64) {
    const double t = wave_parts(part + (size_t)j * np, np);
    if (threadIdx.x % 64 == 0) {
      if (j < m) cs[j] = (T)t;
      if (blockIdx.x == 0) h[j] = t;
    }
  }
}
// sum over j = js, js + JS, ... of cs_j U_j(e)
template <class T, int JS>
__device__ inline T sub_sum(const T (&cs)[256], const T *__restrict__ U0, size_t ustride, int m, int js, size_t e) {
  T t = T(0);
  int j = js;
  for (; j + 7 * JS < m; j += 8 * JS) {
    T u[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) u[q] = U0[ustride * (j + q * JS) + e];
#pragma unroll
    for (int q = 0; q < 8; ++q) t += cs[j + q * JS] * u[q];
  }
  for (; j < m; j += JS) t += cs[j] * U0[ustride * j + e];
  return t;
}
template <class T>
__global__ void __launch_bounds__(kDotThreads) arnoldi_sub_kernel(
    size_t L, int nc, int pad, const T *__restrict__ W, int wdof, int w0, T *__restrict__ y, T *__restrict__ ys,
    const T *__restrict__ U0, size_t ustride, int m, int self, const double *__restrict__ part, int np,
    double *__restrict__ h, double *__restrict__ npart, const double *__restrict__ n0, const double *__restrict__ n1,
    double *__restrict__ g) {
  if (g[G_GM_ARN] != 0.0) return;
  __shared__ double sh[16];
  __shared__ T cs[256];
  if (n1) {
    const double s1 = block_sum_1024((int)threadIdx.x < (int)gridDim.x ? n1[threadIdx.x] : 0.0, sh);
    const bool take = s1 < 0.5 * *n0;  // dgks_pass
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      g[G_GM_N1] = s1;
      g[G_GM_TWICE] = take ? 1.0 : 0.0;
    }
    if (!take) return;
  }
  sub_coefs(m, self, part, np, h, cs);
  __syncthreads();
  double s = 0.0;
  for (size_t e = (size_t)blockIdx.x * kDotThreads + threadIdx.x; e < L; e += (size_t)gridDim.x * kDotThreads) {
    const T v = y[e] - sub_sum<T, 1>(cs, U0, ustride, m, 0, e);
    y[e] = v;
    const size_t i = e / nc, c = e % nc;
    ys[pad * i + c] = W[w0 + c + wdof * i] * v;
    s += (double)v * (double)v;
  }
  s = block_sum_1024(s, sh);
  if (threadIdx.x == 0) npart[blockIdx.x] = s;
}
// The same for at most kOrthMost entries, 1024 / JS of them in a workgroup (JS
// threads share an entry's sum over the basis, so that a short vector does not leave a
// thread alone with a chain of m loads).  FIRST: also the workgroup's parts of the
// dots of the new y with the basis, whose entries it has just read; otherwise the
// second pass and the scaled copy.  22,500 entries, up to 100 vectors: a step of
// seven launches took 51 us, one of five takes 40.
constexpr size_t kOrthMost = (size_t)kDotGrid * kDotThreads;
template <class T, int JS, bool FIRST>
__global__ void __launch_bounds__(kDotThreads) arnoldi_orth_kernel(
    size_t L, int nc, int pad, const T *__restrict__ W, int wdof, int w0, T *__restrict__ y, T *__restrict__ ys,
    const T *__restrict__ U0, size_t ustride, int m, const double *__restrict__ part, int np, double *__restrict__ h,
    double *__restrict__ npart, double *__restrict__ part2, const double *__restrict__ n0,
    const double *__restrict__ n1, double *__restrict__ g) {
  constexpr int kE = kDotThreads / JS;
  __shared__ double sh[16];
  __shared__ T cs[256];
  __shared__ T comb[kDotThreads];
  const int js = threadIdx.x / kE, te = threadIdx.x % kE;
  const size_t base = (size_t)blockIdx.x * kE, e = base + te;
  const bool own = js == 0 && e < L;
  const T yo = own ? y[e] : T(0);
  if (g[G_GM_ARN] != 0.0) return;
  bool take = true;
  if (!FIRST) {
    const double s1 = block_sum_1024((int)threadIdx.x < (int)gridDim.x ? n1[threadIdx.x] : 0.0, sh);
    take = s1 < 0.5 * *n0;  // dgks_pass
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      g[G_GM_N1] = s1;
      g[G_GM_TWICE] = take ? 1.0 : 0.0;
    }
  }
  T t = T(0);
  if (take) {  // the workgroup's
    sub_coefs(m, FIRST ? 1 : 0, part, np, h, cs);
    __syncthreads();
    if (e < L) t = sub_sum<T, JS>(cs, U0, ustride, m, js, e);
  }
  if (JS > 1) {
    comb[threadIdx.x] = t;
    __syncthreads();
    if (js == 0)
#pragma unroll
      for (int q = 1; q < JS; ++q) t += comb[te + q * kE];
  }
  const T v = yo - t;
  if (own) {
    if (take) y[e] = v;
    if (!FIRST) {
      const size_t i = e / nc, c = e % nc;
      ys[pad * i + c] = W[w0 + c + wdof * i] * v;
    }
  }
  if (!take) return;
  const double s = block_sum_1024(own ? (double)v * (double)v : 0.0, sh);  // (its barriers: comb is read)
  if (threadIdx.x == 0) npart[blockIdx.x] = s;
  if (!FIRST) return;
  if (js == 0) comb[te] = own ? v : T(0);
  __syncthreads();
  constexpr int kQ = 4;  // vectors of a wave in flight
  for (int j0 = threadIdx.x / 64; j0 < m; j0 += kQ * (kDotThreads / 64)) {
    double acc[kQ];
#pragma unroll
    for (int q = 0; q < kQ; ++q) acc[q] = 0.0;
#pragma unroll 4
    for (int k = 0; k < kE; k += 64) {
      const int x = k + threadIdx.x % 64;
      const size_t ec = base + x < L ? base + x : L - 1;  // (its y is zero)
      const double yv = (double)comb[x];
#pragma unroll
      for (int q = 0; q < kQ; ++q) {
        const int j = j0 + q * (kDotThreads / 64);
        acc[q] += (double)U0[ustride * (j < m ? j : m - 1) + ec] * yv;
      }
    }
#pragma unroll
    for (int q = 0; q < kQ; ++q) {
      const int j = j0 + q * (kDotThreads / 64);
      acc[q] = wave_sum(acc[q]);
      if (j < m && threadIdx.x % 64 == 0) part2[(size_t)j * gridDim.x + blockIdx.x] = acc[q];
    }
  }
}
// The cycle's first vector: w (already R or R - A X with the faces' PRE), its
// scaled copy and parts of w . w.
template <class T>
__global__ void __launch_bounds__(kDotThreads) arnoldi_first_kernel(size_t L, int nc, int pad,
                                                                    const T *__restrict__ W, int wdof, int w0,
                                                                    const T *__restrict__ w, T *__restrict__ ws,
                                                                    double *__restrict__ npart,
                                                                    const double *__restrict__ skip) {
  if (*skip != 0.0) return;
  __shared__ double sh[16];
  double s = 0.0;
  for (size_t e = (size_t)blockIdx.x * kDotThreads + threadIdx.x; e < L; e += (size_t)gridDim.x * kDotThreads) {
    const T v = w[e];
    const size_t i = e / nc, c = e % nc;
    ws[pad * i + c] = W[w0 + c + wdof * i] * v;
    s += (double)v * (double)v;
  }
  s = block_sum_1024(s, sh);
  if (threadIdx.x == 0) npart[blockIdx.x] = s;
}

// ----- plain vector sweeps (skip: return at once when *skip is set; may be null) -----
template <class T>
__global__ void fill_kernel(size_t L, T *__restrict__ x, const double *__restrict__ skip) {
  if (skip && *skip != 0.0) return;
  const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e < L) x[e] = T(0);
}
template <class T>
__global__ void copy_kernel(size_t L, const T *__restrict__ src, T *__restrict__ dst,
                            const double *__restrict__ skip) {
  if (skip && *skip != 0.0) return;
  const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e < L) dst[e] = src[e];
}
// z = x - y
template <class T>
__global__ void diff_kernel(size_t L, const T *__restrict__ x, const T *__restrict__ y, T *__restrict__ z,
                            const double *__restrict__ skip) {
  if (skip && *skip != 0.0) return;
  const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e < L) z[e] = x[e] - y[e];
}
// y = x + sign sum_j coef[j] U_j, j < m (*m_dev when given); x may be y
template <class T>
__global__ void combine_kernel(size_t L, const T *__restrict__ x, T *__restrict__ y, const T *__restrict__ U0,
                               size_t ustride, int m, const double *__restrict__ m_dev,
                               const double *__restrict__ coef, double sign, const double *__restrict__ skip) {
  if (skip && *skip != 0.0) return;
  const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= L) return;
  if (m_dev) m = (int)*m_dev;
  T w = x[e];
  int j = 0;
  for (; j + 8 <= m; j += 8) {
    T u[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) u[q] = U0[ustride * (j + q) + e];
#pragma unroll
    for (int q = 0; q < 8; ++q) w += (T)(sign * coef[j + q]) * u[q];
  }
  for (; j < m; ++j) w += (T)(sign * coef[j]) * U0[ustride * j + e];
  y[e] = w;
}
// y = x * w elementwise (types may differ: the FP64 right-hand side in and
// the solution out of an FP32 solve)
template <class TX, class TW, class TY>
__global__ void mul_kernel(size_t L, const TX *__restrict__ x, const TW *__restrict__ w, TY *__restrict__ y) {
  const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= L) return;
  y[e] = (TY)(x[e] * w[e]);
}
// The NS solver's vectors hold the velocity (3, N) and behind it the
// pressure (N).  W o Ri (4, N) in that layout, into both r0 and r.
template <class T>
__global__ void ns_split_kernel(int N, const double *__restrict__ Ri, const T *__restrict__ W, T *__restrict__ r0,
                                T *__restrict__ r) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= N) return;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const size_t s = c + (size_t)4 * i, d = c < 3 ? c + (size_t)3 * i : (size_t)3 * N + i;
    const T v = (T)(Ri[s] * W[s]);
    r0[d] = v;
    r[d] = v;
  }
}
// The solution: velocity sum_k cu[k] U_k, pressure sum_k cp[k] P_k (U_k and P_k
// behind each other in X_k), times W, into Ri (4, N).
template <class T>
__global__ void ns_join_kernel(int N, const T *__restrict__ X0, const double *__restrict__ cnt,
                               const double *__restrict__ cu, const double *__restrict__ cp, const T *__restrict__ W,
                               double *__restrict__ Ri, const double *__restrict__ skip) {
  if (*skip != 0.0) return;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= N) return;
  const int n = (int)*cnt;
  const size_t st = (size_t)4 * N;
  T v[4] = {T(0), T(0), T(0), T(0)};
  for (int k = 0; k < n; ++k) {
    const T a = (T)cu[k], b = (T)cp[k];
#pragma unroll
    for (int c = 0; c < 3; ++c) v[c] += a * X0[st * k + 3 * (size_t)i + c];
    v[3] += b * X0[st * k + (size_t)3 * N + i];
  }
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const size_t s = c + (size_t)4 * i;
    Ri[s] = (double)(v[c] * W[s]);
  }
}

// PRECOND part 1: W from the diagonal, fix for zero diagonals.
template <class T>
__global__ void precond_diag_kernel(int N, int dof, int vdof, const T *__restrict__ V, size_t nnz,
                                    const int *__restrict__ diag, T *__restrict__ W, T *__restrict__ fix) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= N) return;
  const int d = diag[i];
  for (int r = 0; r < dof; ++r) {
    const T a = V[(size_t)(r * vdof + r) * nnz + d];
    W[r + (size_t)dof * i] = (a == T(0)) ? T(1) : T(1) / sqrt(fabs(a));
    fix[r + (size_t)dof * i] = (a == T(0)) ? T(1) : T(0);
  }
}
// Dirichlet masking of W by a face's val (memLS.f90:1831-1841)
template <class T>
__global__ void precond_face_kernel(int n, int dof, int fdof, const int *__restrict__ glob,
                                    const double *__restrict__ val, T *__restrict__ W) {
  const int a = blockIdx.x * blockDim.x + threadIdx.x;
  if (a >= n) return;
  const int nc = fdof < dof ? fdof : dof;
  const int Ac = glob[a];
  for (int i = 0; i < nc; ++i) W[i + (size_t)dof * Ac] *= (T)val[i + (size_t)fdof * a];
}
// After masking: diagonal entries that scale to zero are forced to one.
template <class T>
__global__ void precond_fix_kernel(int N, int dof, int vdof, const T *__restrict__ V, size_t nnz,
                                   const int *__restrict__ diag, const T *__restrict__ W, T *__restrict__ fix) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= N) return;
  const int d = diag[i];
  for (int r = 0; r < dof; ++r) {
    const T a = V[(size_t)(r * vdof + r) * nnz + d];
    const T w = W[r + (size_t)dof * i];
    if (a == T(0) || (a * w) * w == T(0)) fix[r + (size_t)dof * i] = T(1);
  }
}
// valM = val * W for a coupled face (kept in FP64: faces are small)
template <class T>
__global__ void face_valm_kernel(int n, int dof, int fdof, const int *__restrict__ glob,
                                 const double *__restrict__ val, const T *__restrict__ W,
                                 double *__restrict__ valM) {
  const int a = blockIdx.x * blockDim.x + threadIdx.x;
  if (a >= n) return;
  const int nc = fdof < dof ? fdof : dof;
  for (int i = 0; i < nc; ++i)
    valM[i + (size_t)fdof * a] = val[i + (size_t)fdof * a] * (double)W[i + (size_t)dof * glob[a]];
}
// ADDBCMUL (memLS.f90:206-268) on the coupled faces: with ADD, Y += res_f (v_f .
// X) v_f; with PRE, then Y += coef_f (v_f . Y) v_f, every dot taken before any
// update of its kind (memLS's copy unCondU).  One 1024-thread workgroup per
// face when no two share a node (then they do not see each other's
// updates), one for all of them otherwise (each face in turn between
// barriers).  Replaces a dot and an update launch per face and kind.  Faces that
// share nodes and have more than kFaceSerial of them together take those launches
// (face_dot, face_add): one workgroup walks them all too slowly.  30 Arnoldi steps of
// GMRESV in one workgroup and in launches, ms: 8 faces with 1,100 nodes together 2.10
// and 2.16, 24 with 3,300 3.40 and 3.45, 8 with 6,800 5.14 and 4.69, 24 with 13,700
// 7.43 and 6.17, 56,000 20.1 and 10.8, 301,000 88 and 22.5.
constexpr int kFaceAdd = 1, kFacePre = 2;
constexpr size_t kFaceSerial = 4096;
// F's valM . x, by 1024 threads
template <class T>
__device__ inline double face_dot(const FaceDev &F, int xdof, const T *__restrict__ x, double *sh) {
  const int nc = F.dof < xdof ? F.dof : xdof;
  double s = 0.0;
  for (int a = threadIdx.x; a < F.nNo; a += 1024)
    for (int i = 0; i < nc; ++i) s += F.valM[i + (size_t)F.dof * a] * (double)x[i + (size_t)xdof * F.glob[a]];
  return block_sum_1024(s, sh);
}
template <class T>
__global__ void __launch_bounds__(1024) face_dot_kernel(const FaceDev *__restrict__ fd, int xdof,
                                                        const T *__restrict__ x, double *__restrict__ sum,
                                                        const double *__restrict__ skip) {
  if (skip && *skip != 0.0) return;
  __shared__ double sh[16];
  const double d = face_dot(fd[blockIdx.x], xdof, x, sh);
  if (threadIdx.x == 0) sum[blockIdx.x] = d;
}
template <class T>
__global__ void __launch_bounds__(256) face_add_kernel(const FaceDev *__restrict__ fd, int f, int kind, int xdof,
                                                       const double *__restrict__ sum, T *__restrict__ Y,
                                                       const double *__restrict__ skip) {
  if (skip && *skip != 0.0) return;
  const int a = blockIdx.x * 256 + threadIdx.x;
  const FaceDev F = fd[f];
  if (a >= F.nNo) return;
  const double c = (kind == kFaceAdd ? F.res : *F.coefp) * sum[f];
  const int nc = F.dof < xdof ? F.dof : xdof;
  for (int i = 0; i < nc; ++i) Y[i + (size_t)xdof * F.glob[a]] += (T)(F.valM[i + (size_t)F.dof * a] * c);
}
template <class T>
__global__ void __launch_bounds__(1024) face_apply_kernel(const FaceDev *__restrict__ fd, int nfc, int what, int xdof,
                                                          const T *__restrict__ X, T *__restrict__ Y,
                                                          double *__restrict__ sum, const double *__restrict__ skip) {
  if (skip && *skip != 0.0) return;
  __shared__ double sh[16];
  const int f0 = gridDim.x > 1 ? blockIdx.x : 0, f1 = gridDim.x > 1 ? f0 + 1 : nfc;
  auto dot = [&](const FaceDev &F, const T *x) { return face_dot(F, xdof, x, sh); };
  auto add = [&](const FaceDev &F, double c) {
    const int nc = F.dof < xdof ? F.dof : xdof;
    for (int a = threadIdx.x; a < F.nNo; a += 1024)
      for (int i = 0; i < nc; ++i) Y[i + (size_t)xdof * F.glob[a]] += (T)(F.valM[i + (size_t)F.dof * a] * c);
  };
  for (int kind = kFaceAdd; kind <= kFacePre; kind <<= 1) {
    if (!(what & kind)) continue;
    for (int f = f0; f < f1; ++f) {
      const double d = dot(fd[f], kind == kFaceAdd ? X : Y);
      if (threadIdx.x == 0) sum[f] = d;
    }
    __syncthreads();
    for (int f = f0; f < f1; ++f) {
      add(fd[f], (kind == kFaceAdd ? fd[f].res : *fd[f].coefp) * sum[f]);
      __syncthreads();
    }
  }
}
// BCPRE's nS of the coupled faces (memLS.f90:1683-1716: ||valM||^2 over nsd
// components) and their PRE coefficients -res / (1 + res nS), a workgroup each
__global__ void __launch_bounds__(1024) face_coef_kernel(const FaceDev *__restrict__ fd, int nsd,
                                                         double *__restrict__ coef) {
  __shared__ double sh[16];
  const FaceDev F = fd[blockIdx.x];
  const int nc = F.dof < nsd ? F.dof : nsd;
  double s = 0.0;
  for (int a = threadIdx.x; a < F.nNo; a += 1024)
    for (int i = 0; i < nc; ++i) s += F.valM[i + (size_t)F.dof * a] * F.valM[i + (size_t)F.dof * a];
  s = block_sum_1024(s, sh);
  if (threadIdx.x == 0) coef[blockIdx.x] = -F.res / (1.0 + F.res * s);
}
// The face functional's coefficients q (FaceDev), one thread per support
// column, its pairs in their stored order, in FP64.
template <class T>
__global__ void face_q_kernel(int nsup, const int *__restrict__ sup, const int *__restrict__ qptr,
                              const int *__restrict__ qa, const int *__restrict__ qk, const int *__restrict__ glob,
                              const double *__restrict__ valM, int dof, MatView<T> G, double *__restrict__ q) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= nsup) return;
  const int nc = dof < 3 ? dof : 3;
  double v = 0.0;
  for (int p = qptr[s]; p < qptr[s + 1]; ++p) {
    const int a = qa[p], k = qk[p];
    const size_t g = glob[a];
    for (int i = 0; i < nc; ++i)
      v += valM[i + (size_t)dof * a] * (double)G.W[G.r0 + i + (size_t)G.wdof * g] *
           (double)G.base[(size_t)G.plane[4 * i] * G.nnz + k];
  }
  q[s] = v * (double)G.W[G.c0 + (size_t)G.wdof * sup[s]];
}
// AoS (vdof*vdof, nnz) -> planes, and Gt = -mG^T via the transpose map
template <class TS, class TD>
__global__ void aos_to_planes_kernel(size_t nnz, int m, const TS *__restrict__ aos, TD *__restrict__ V) {
  const size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nnz) return;
  for (int p = 0; p < m; ++p) V[(size_t)p * nnz + k] = (TD)aos[(size_t)m * k + p];
}
template <class TS, class TD>
__global__ void convert_kernel(size_t n, const TS *__restrict__ a, TD *__restrict__ b) {
  const size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  b[k] = (TD)a[k];
}
template <class T>
__global__ void gt_kernel(size_t nnz, const T *__restrict__ V, const int *__restrict__ tr, T *__restrict__ Gt) {
  const size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nnz) return;
  const int l = tr[k];
  Gt[0 * nnz + l] = -V[3 * nnz + k];
  Gt[1 * nnz + l] = -V[7 * nnz + k];
  Gt[2 * nnz + l] = -V[11 * nnz + k];
}

// ----- CG (device-resident iterations with a convergence flag) -----
// Three launches per iteration (two on a formed Schur complement of up to kCgPaired
// rows, below): SP = S P with the
// parts of P . SP (s_product_kernel), the residual update with the parts of
// R . R, and the direction update, which also advances the state.  Every
// workgroup sums the parts it needs itself, in one fixed order, so that no
// one-workgroup launch stands between two sweeps; before, the product, the
// face term, the dot, the update, the error and the direction took seven
// launches (28.3 us of kernels per iteration at 36,000 nodes, 120 us at
// 458,000).
// The state is kept twice (kCgState doubles each): iteration k reads copy k & 1 and
// the direction update (paired: the product) writes the other, so that no workgroup reads what
// another is writing.
// State: 0 err, 1 errO, 2 eps2, 3 alpha, 5 done, 6 itr, 7 mItr, 8 suc.
constexpr int kCgState = 16;
// Top-of-iteration test of CGRAD (memLS.f90:413-427): stop at mItr or when
// err < eps^2; otherwise errO = err and count the iteration.
__device__ inline void check_next(double *scal) {
  if (scal[5] != 0.0) return;
  if (scal[6] >= scal[7]) {
    scal[5] = 1.0;
    return;
  }
  if (scal[0] < scal[2]) {
    scal[8] = 1.0;
    scal[5] = 1.0;
    return;
  }
  scal[1] = scal[0];  // errO = err
  scal[6] += 1.0;
}
__device__ inline double face_sum(const FaceList &fl, int f) {
  const double *p = fl.part + (f << fl.lb);
  double S = 0.0;
#pragma unroll
  for (int b = 0; b < kFaceDotBlocks; ++b) S += p[b];
  for (int b = kFaceDotBlocks; b < fl.nb; ++b) S += p[b];
  return S;
}
// Workgroup b of a face's nb: its share of q_f . P, entries b * 256 + t +
// 256 nb u; p_at(j) gives the direction at column j.
template <class P>
__device__ inline void face_part(const FaceList &fl, int wg, double *sh, P p_at) {
  const int f = wg >> fl.lb, b = wg & (fl.nb - 1);
  const int *sup = fl.fd[f].sup;
  const double *q = fl.fd[f].q;
  const int ns = fl.fd[f].nsup;
  double s = 0.0;
  const int step = 256 << fl.lb;
  for (int e0 = b * 256 + threadIdx.x; e0 < ns; e0 += 4 * step) {  // four entries' loads together
    int j[4];
    double qv[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int e = min(e0 + step * u, ns - 1);
      j[u] = sup[e];
      qv[u] = e0 + step * u < ns ? q[e] : 0.0;
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) s += qv[u] * (double)p_at(j[u]);
  }
  s = block_sum(s, sh);
  if (threadIdx.x == 0) fl.part[wg] = s;
}
// The first direction P = R (and Ps = W_p o P for the two-pass operator), X = 0 in
// place of the right-hand side, which moves to Rv.
template <class T>
__global__ void __launch_bounds__(256) cg_begin_vec_kernel(size_t L, T *__restrict__ X, T *__restrict__ Rv,
                                                           T *__restrict__ P, const T *__restrict__ W, int wdof,
                                                           int off, T *__restrict__ Ps,
                                                           const double *__restrict__ skip) {
  if (skip && *skip != 0.0) return;
  const size_t e = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= L) return;
  const T r = X[e];
  Rv[e] = r;
  P[e] = r;
  if (Ps) Ps[e] = W[off + (size_t)wdof * e] * r;
  X[e] = T(0);
}
// the faces' dots with the first direction
template <class T>
__global__ void __launch_bounds__(256) cg_begin_face_kernel(FaceList fl, const T *__restrict__ P,
                                                            const double *__restrict__ skip) {
  if (skip && *skip != 0.0) return;
  __shared__ double sh[4];
  face_part(fl, blockIdx.x, sh, [&](int j) { return P[j]; });
}
// parts of P . SP for an operator that does not form them
template <class T>
__global__ void __launch_bounds__(256) cg_den_kernel(size_t L, const T *__restrict__ P, const T *__restrict__ SP,
                                                     double *__restrict__ dpart, const double *__restrict__ done) {
  if (*done != 0.0) return;
  __shared__ double sh[4];
  double s = 0.0;
  for (size_t e = (size_t)blockIdx.x * 256 + threadIdx.x; e < L; e += (size_t)gridDim.x * 256)
    s += (double)P[e] * (double)SP[e];
  s = block_sum(s, sh);
  if (threadIdx.x == 0) dpart[blockIdx.x] = s;
}
// R -= alpha SP (with the faces' rank-one terms), alpha = errO / (P . SP);
// the workgroup's part of R . R.  E entries per thread and turn (cg_grid).
// PAIR (the formed Schur complement): R sits in Q, which takes P too, and X +=
// alpha P is done here.
template <class T>
struct Pair;
template <>
struct Pair<double> {
  using type = double2;
};
template <>
struct Pair<float> {
  using type = float2;
};
template <class T>
using PairT = typename Pair<T>::type;
template <class T, int E, bool PAIR>
__global__ void __launch_bounds__(256) cg_r_kernel(size_t L, double *__restrict__ scal,
                                                   const double *__restrict__ dpart, int nd, FaceList fl,
                                                   T *__restrict__ R, const T *__restrict__ SP,
                                                   double *__restrict__ rpart, PairT<T> *__restrict__ Q,
                                                   T *__restrict__ X, const T *__restrict__ P) {
  __shared__ double sh[4], fc[kFaceLds];
  __shared__ T corr[E * 256];
  const double stop = scal[5], errO = scal[1];
  T r[E], sp[E], x[E], p[E];
  auto load = [&](size_t base) {
#pragma unroll
    for (int t = 0; t < E; ++t) {
      const size_t e = base + threadIdx.x + 256 * t;
      if constexpr (PAIR) {
        r[t] = e < L ? Q[e].x : T(0);
        x[t] = e < L ? X[e] : T(0);
        p[t] = e < L ? P[e] : T(0);
      } else {
        r[t] = e < L ? R[e] : T(0);
      }
      sp[t] = e < L ? SP[e] : T(0);
    }
  };
  const int nt = (int)((L + 255) / 256);
  int e0 = 0, e1 = 0;  // the faces' nodes of the turn
  auto range = [&](size_t base) {
    if (fl.nfc == 0) return;
    const int t0 = (int)(base / 256);
    e0 = fl.tptr[t0];
    e1 = fl.tptr[min(t0 + E, nt)];
  };
  size_t base = (size_t)blockIdx.x * (E * 256);
  load(base);  // all in flight while the parts are summed
  range(base);
  // a face's first parts and coefficient are in flight with them; what follows from
  // these is LDS work that a launch past the end of the solve need not do
  double d = 0.0, fp[kFaceDotBlocks] = {}, cf = 0.0;
  if ((int)threadIdx.x < fl.nfc) {
#pragma unroll
    for (int b = 0; b < kFaceDotBlocks; ++b) fp[b] = fl.part[(threadIdx.x << fl.lb) + b];
    cf = fl.coef[threadIdx.x];
  }
  if (stop != 0.0) return;
  if ((int)threadIdx.x < fl.nfc) {
    double S = 0.0;
#pragma unroll
    for (int b = 0; b < kFaceDotBlocks; ++b) S += fp[b];
    for (int b = kFaceDotBlocks; b < fl.nb; ++b) S += fl.part[(threadIdx.x << fl.lb) + b];
    d = (fc[threadIdx.x] = cf * S) * S;
  }
  for (int f = threadIdx.x + kFaceLds; f < fl.nfc; f += kFaceLds) {
    const double S = face_sum(fl, f);
    d += fl.coef[f] * S * S;
  }
  const double den = sum_parts(dpart, nd, d, sh);
  const double a = errO / den;  // CGRAD's alpha
  if (blockIdx.x == 0 && threadIdx.x == 0) scal[3] = a;
  const T alpha = (T)a;
  double s = 0.0;
  while (base < L) {
    if (e1 > e0) {  // the same for the whole workgroup
#pragma unroll
      for (int t = 0; t < E; ++t) corr[threadIdx.x + 256 * t] = T(0);
      __syncthreads();
      auto term = [&](FaceEnt en) {
        const FaceDev &F = fl.fd[en.f];
        return (en.f < kFaceLds ? fc[en.f] : fl.coef[en.f] * face_sum(fl, en.f)) * F.q[en.s];
      };
      for (int e = e0 + threadIdx.x; e < e1; e += 256) {
        const FaceNode fn = fl.node[e];
        double v = term(fn.first);
        for (int x = fn.more; x < fn.end; ++x) v += term(fl.ent[x]);
        corr[fn.node - (int)base] = (T)v;
      }
      __syncthreads();
#pragma unroll
      for (int t = 0; t < E; ++t) sp[t] += corr[threadIdx.x + 256 * t];
      __syncthreads();
    }
#pragma unroll
    for (int t = 0; t < E; ++t) {
      const size_t e = base + threadIdx.x + 256 * t;
      if (e < L) {
        const T v = r[t] - alpha * sp[t];
        if constexpr (PAIR) {
          Q[e] = PairT<T>{v, p[t]};
          X[e] = x[t] + alpha * p[t];
        } else {
          R[e] = v;
        }
        s += (double)v * (double)v;
      }
    }
    base += (size_t)gridDim.x * (E * 256);
    if (base < L) {
      load(base);
      range(base);
    }
  }
  s = block_sum(s, sh);
  if (threadIdx.x == 0) rpart[blockIdx.x] = s;
}
// err = R . R from the parts, beta = err / errO; X += alpha P, the next
// direction Pn = R + beta P (with its scaled copy Ps, and in the first
// workgroups the faces' dots with it), and the next iteration's state.
template <class T, int E>
__global__ void __launch_bounds__(256) cg_p_kernel(size_t L, const double *__restrict__ scal,
                                                   double *__restrict__ next, const double *__restrict__ rpart, int nr,
                                                   FaceList fl, T *__restrict__ X, const T *__restrict__ R,
                                                   const T *__restrict__ P, T *__restrict__ Pn,
                                                   const T *__restrict__ W, int wdof, int off, T *__restrict__ Ps,
                                                   HostFlag hf) {
  const int nf = fl.nfc * fl.nb, blk = (int)blockIdx.x - nf;
  __shared__ double sh[4];
  const double stop = scal[5], errO = scal[1], al = scal[3];
  T r[E], p[E], x[E];
  auto load = [&](size_t base) {
#pragma unroll
    for (int t = 0; t < E; ++t) {
      const size_t e = base + threadIdx.x + 256 * t;
      r[t] = e < L ? R[e] : T(0);
      p[t] = e < L ? P[e] : T(0);
      x[t] = e < L ? X[e] : T(0);
    }
  };
  size_t base = (size_t)max(blk, 0) * (E * 256);
  if (blk >= 0) load(base);  // in flight while the parts are summed
  if (stop != 0.0) {
    if (blockIdx.x == 0 && threadIdx.x < kCgState) next[threadIdx.x] = scal[threadIdx.x];
    if (blockIdx.x == 0 && threadIdx.x == 0) hf.tell(true);
    return;
  }
  const double n = sqrt(sum_parts(rpart, nr, 0.0, sh));  // NORMS(R)
  const double err = n * n;
  const T alpha = (T)al, beta = (T)(err / errO);
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    double st[kCgState];
    for (int k = 0; k < kCgState; ++k) st[k] = scal[k];
    st[0] = err;
    check_next(st);
    for (int k = 0; k < kCgState; ++k) next[k] = st[k];
    hf.tell(st[5] != 0.0);
  }
  if (blk < 0) {
    face_part(fl, blockIdx.x, sh, [&](int j) { return R[j] + beta * P[j]; });
    return;
  }
  while (base < L) {
#pragma unroll
    for (int t = 0; t < E; ++t) {
      const size_t e = base + threadIdx.x + 256 * t;
      if (e >= L) continue;
      X[e] = x[t] + alpha * p[t];
      const T v = r[t] + beta * p[t];
      Pn[e] = v;
      if (Ps) Ps[e] = W[off + (size_t)wdof * e] * v;
    }
    base += (size_t)(gridDim.x - nf) * (E * 256);
    if (base < L) load(base);
  }
}

// ----- the CG on the formed Schur complement: two launches per iteration -----
// The residual and the direction sit together, Q(j) = (R, P), one 16-byte entry
// (8 in FP32): the product gathers Q and takes the new direction R + beta P of
// every column as it goes, so that no sweep stands between the residual update
// and the product.  Taken up to kCgPaired rows, where a launch costs more than the
// wider gather.  Whole NS solves of the workloads' iteration counts, three launches
// and two: 21,800 rows 9.6 and 8.6 ms, 36,000 15.9 and 15.1, 50,000 15.6 and 14.9,
// 68,000 17.1 and 17.2, 141,000 28.0 and 28.9 (FP32: 4.2 and 3.7, 4.7 and 4.5, 4.9
// and 4.7, 6.5 and 6.4, 10.2 and 10.4).
constexpr int kCgPaired = 1 << 16;
// Q = (X, 0), X = 0
template <class T>
__global__ void __launch_bounds__(256) cg_pair_kernel(size_t L, T *__restrict__ X, PairT<T> *__restrict__ Q,
                                                      const double *__restrict__ skip) {
  if (skip && *skip != 0.0) return;
  const size_t e = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= L) return;
  Q[e] = PairT<T>{X[e], T(0)};
  X[e] = T(0);
}
// The state after the iteration whose residual's parts are rpart[0, nr): err = R .
// R and the next test; returns beta = err / errO.
__device__ inline double cg_advance(const double *__restrict__ scal, const double *__restrict__ rpart, int nr,
                                    double (&st)[kCgState], double *sh) {
  const double n = sqrt(sum_parts(rpart, nr, 0.0, sh));  // NORMS(R)
  const double err = n * n, beta = err / scal[1];
#pragma unroll
  for (int k = 0; k < kCgState; ++k) st[k] = scal[k];
  st[0] = err;
  check_next(st);
  return beta;
}
// The state after the last iteration (a captured loop's end).
__global__ void __launch_bounds__(256) cg_close_kernel(const double *__restrict__ scal, double *__restrict__ next,
                                                       const double *__restrict__ rpart, int nr) {
  __shared__ double sh[4];
  double st[kCgState];
  if (scal[5] != 0.0) {
    if (threadIdx.x < kCgState) next[threadIdx.x] = scal[threadIdx.x];
    return;
  }
  (void)cg_advance(scal, rpart, nr, st, sh);
  if (threadIdx.x == 0)
    for (int k = 0; k < kCgState; ++k) next[k] = st[k];
}
// The new direction P = R + beta P of every row, SP = S P and the workgroup's part
// of P . SP, 16 lanes per row; the first workgroups take the faces' dots with P.
// next null: the first iteration (beta 0, no state to advance).  The first rows'
// entries are in flight while the residual's parts are summed.
template <class T, class OX>
__global__ void __launch_bounds__(256) s_dir_product_kernel(int nNo, int ntile, const int *__restrict__ sptr,
                                                        const OX *__restrict__ scol, const T *__restrict__ S,
                                                        const PairT<T> *__restrict__ Q, T *__restrict__ P,
                                                        T *__restrict__ SP, double *__restrict__ dpart,
                                                        const double *__restrict__ scal, double *__restrict__ next,
                                                        const double *__restrict__ rpart, int nr, FaceList fl,
                                                        HostFlag hf) {
  __shared__ double sh[4];
  const double stop = scal[5];
  const int nf = fl.nfc * fl.nb, blk = (int)blockIdx.x - nf, nwg = (int)gridDim.x - nf;
  const int lane = threadIdx.x % kSLanes;
  auto row_of = [&](int vb) {
    return (int)crimson::xcd_block(kRowXcdChunk, vb, ntile) * (256 / kSLanes) + (int)threadIdx.x / kSLanes;
  };
  int row = 0, kb = 0, ke = 0;
  T v[kSUnroll];
  PairT<T> x[kSUnroll], own;
  auto load = [&](int k) {
    int j[kSUnroll];
#pragma unroll
    for (int u = 0; u < kSUnroll; ++u) {
      const int kc = max(min(k + kSLanes * u, ke - 1), 0);
      j[u] = col_at(scol, kc, row);
      v[u] = S[kc];
    }
#pragma unroll
    for (int u = 0; u < kSUnroll; ++u) x[u] = Q[min((unsigned)j[u], (unsigned)nNo - 1u)];  // (a row past the end or empty)
  };
  if (blk >= 0) {
    row = row_of(blk);
    kb = sptr[min(row, nNo)];
    ke = sptr[min(row + 1, nNo)];  // rows past the last one: kb = ke
    own = Q[min(row, nNo - 1)];
    load(kb + lane);
  }
  double beta = 0.0;
  if (next) {
    if (stop != 0.0) {
      if (blockIdx.x == 0 && threadIdx.x < kCgState) next[threadIdx.x] = scal[threadIdx.x];
      if (blockIdx.x == 0 && threadIdx.x == 0) hf.tell(true);
      return;
    }
    double st[kCgState];
    beta = cg_advance(scal, rpart, nr, st, sh);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      for (int k = 0; k < kCgState; ++k) next[k] = st[k];
      hf.tell(st[5] != 0.0);
    }
    if (st[5] != 0.0) return;
  } else if (stop != 0.0) {
    return;
  }
  const T bt = (T)beta;
  if (blk < 0) {
    face_part(fl, blockIdx.x, sh, [&](int j) {
      const PairT<T> q = Q[j];
      return q.x + bt * q.y;
    });
    return;
  }
  double den = 0.0;
  for (int vb = blk;;) {
    const int vn = vb + nwg;
    int rown = 0, kbn = 0, ken = 0;
    if (vn < ntile) {
      rown = row_of(vn);
      kbn = sptr[min(rown, nNo)];
      ken = sptr[min(rown + 1, nNo)];
    }
    T acc = T(0);
    for (int k = kb + lane; k < ke; k += kSLanes * kSUnroll) {
      if (k != kb + lane) load(k);
#pragma unroll
      for (int u = 0; u < kSUnroll; ++u)
        if (k + kSLanes * u < ke) acc += v[u] * (x[u].x + bt * x[u].y);
    }
#pragma unroll
    for (int off = kSLanes / 2; off > 0; off >>= 1) acc += __shfl_xor(acc, off, kSLanes);
    if (row < nNo && lane == 0) {
      const T pr = own.x + bt * own.y;
      P[row] = pr;
      SP[row] = acc;
      den += (double)pr * (double)acc;
    }
    if (vn >= ntile) break;
    vb = vn;
    row = rown;
    kb = kbn;
    ke = ken;
    own = Q[min(row, nNo - 1)];
    load(kb + lane);
  }
  den = block_sum(den, sh);
  if (threadIdx.x == 0) dpart[blk] = den;
}
}  // namespace

// What handles keep between solves, process-wide: every handle that holds a workspace
// or a complement's pattern, under one lock.  Never destroyed: handles may be freed
// after this library's static objects.
namespace crimson {
namespace {
std::mutex &g_work_lock = *new std::mutex;
std::vector<crimson_lhs *> &g_work_lhs = *new std::vector<crimson_lhs *>;
size_t g_work_bytes = 0;
// under the lock: l among the holders or not
void work_note(crimson_lhs *l) {
  auto at = std::find(g_work_lhs.begin(), g_work_lhs.end(), l);
  const bool holds = l->work[0] || l->work[1] || l->spat;
  if (holds && at == g_work_lhs.end()) g_work_lhs.push_back(l);
  if (!holds && at != g_work_lhs.end()) g_work_lhs.erase(at);
}
std::unique_ptr<SolveWorkBase> work_drop(crimson_lhs *l, int k) {  // under the lock
  std::unique_ptr<SolveWorkBase> w = std::move(l->work[k]);
  if (w) g_work_bytes -= w->bytes();
  work_note(l);
  return w;
}
std::unique_ptr<SolveWorkBase> work_take(crimson_lhs *l, bool fp32) {
  std::lock_guard<std::mutex> hold(g_work_lock);
  return work_drop(l, fp32 ? 1 : 0);
}
void work_keep(crimson_lhs *l, bool fp32, std::unique_ptr<SolveWorkBase> w, size_t most) {
  std::lock_guard<std::mutex> hold(g_work_lock);
  std::unique_ptr<SolveWorkBase> old = work_drop(l, fp32 ? 1 : 0);
  if (g_work_bytes + w->bytes() > most) return;
  g_work_bytes += w->bytes();
  l->work[fp32 ? 1 : 0] = std::move(w);
  work_note(l);
}
std::shared_ptr<const SchurPattern> pattern_of(crimson_lhs *l) {
  std::lock_guard<std::mutex> hold(g_work_lock);
  return l->spat;
}
void pattern_keep(crimson_lhs *l, std::shared_ptr<const SchurPattern> p) {
  std::lock_guard<std::mutex> hold(g_work_lock);
  l->spat = std::move(p);
  work_note(l);
}
void work_forget(crimson_lhs *l) {  // under the lock
  (void)work_drop(l, 0);
  (void)work_drop(l, 1);
  l->spat.reset();
  work_note(l);
}
}  // namespace
bool release_idle_work() {
  std::lock_guard<std::mutex> hold(g_work_lock);
  const bool any = !g_work_lhs.empty();
  while (!g_work_lhs.empty()) work_forget(g_work_lhs.back());
  return any;
}
}  // namespace crimson

extern "C" int crimson_release_workspaces(void) {
  (void)crimson::release_idle_work();
  return CRIMSON_OK;
}

struct crimson_ls {
  SubLs GM, CG, RI;
  int LS_type = 0, Resm = 0, Resc = 0;
};

namespace {

double now_s() {
  return std::chrono::duration<double>(std::chrono::steady_clock::now().time_since_epoch()).count();
}

// The stored matrix planes and the -mG^T buffer in the solve's type.
inline const double *planes(const crimson_lhs *l, double) { return l->d_V.p; }
inline const float *planes(const crimson_lhs *l, float) { return l->d_V32.p; }
inline crimson::DBuf<double> &gt_buf(crimson_lhs *l, double) { return l->d_Gt; }
inline crimson::DBuf<float> &gt_buf(crimson_lhs *l, float) { return l->d_Gt32; }

// What every kernel of a solve shares: the handle, the stream, PRECOND's
// scaling, the reduction scratch and the coupled faces.
template <class T>
struct Ctx {
  crimson_lhs *lhs = nullptr;
  hipStream_t s = nullptr;
  int N = 0, dof = 0;
  crimson::DBuf<T> W, fix;
  crimson::DBuf<double> part;    // dot parts: kDotGrid per dot, 2 * kCgGrid in the CG
  crimson::DBuf<double> cgst;    // the CG's state, twice
  crimson::DBuf<FaceDev> fdev;   // the coupled faces, in face order
  crimson::DBuf<double> fcoef;   // their PRE coefficients
  crimson::DBuf<double> fsum;    // one dot per coupled face (face_apply_kernel)
  crimson::DBuf<double> fpart;   // the Schur CG's face dot parts (1 << flb per face)
  int flb = 0;
  std::vector<FaceDev> hfdev;    // fdev on the host
  bool disjoint = true;          // no two coupled faces share a node
  size_t fnodes = 0;             // the coupled faces' nodes together
  int nfc() const { return (int)hfdev.size(); }
  // their merged supports (FaceList), for the faces whose supports fent_sig lists
  std::vector<unsigned long long> fent_sig;
  crimson::DBuf<FaceNode> fnode;
  crimson::DBuf<FaceEnt> fent;
  crimson::DBuf<int> ftptr;
  FaceList face_list() const {
    return FaceList{nfc(), 1 << flb, flb, fdev.p, fnode.p, fent.p, ftptr.p, fpart.p, fcoef.p};
  }

  int init(crimson_lhs *l, int d, hipStream_t st) {
    lhs = l;
    s = st;
    N = l->nNo;
    dof = d;
    const size_t L = (size_t)dof * N;
    CR_TRY(W.alloc(L));
    CR_TRY(fix.alloc(L));
    CR_TRY(part.alloc((size_t)kDotGrid * 3 * 264));
    CR_TRY(cgst.alloc(2 * kCgState));
    return CRIMSON_OK;
  }
};
static_assert(kDotGrid * 3 * 264 >= 2 * kCgGrid, "the CG's parts fit the dots'");

template <class T>
MatView<T> view(const Ctx<T> &c, const T *base, int vdof, int r0, int c0, int nr, int nc, const T *W, const T *fix,
                int wdof) {
  MatView<T> A;
  A.base = base;
  A.nnz = (size_t)c.lhs->nnz;
  for (int k = 0; k < 16; ++k) A.plane[k] = 0;
  for (int r = 0; r < nr; ++r)
    for (int cc = 0; cc < nc; ++cc) A.plane[r * 4 + cc] = (r0 + r) * vdof + (c0 + cc);
  A.W = W;
  A.fix = fix;
  A.wdof = wdof;
  A.r0 = r0;
  A.c0 = c0;
  return A;
}

// y = ya * (A x) + za * z
template <class T>
int spmv(Ctx<T> &c, const MatView<T> &A, int nr, int nc, const T *x, T *y, double ya = 1.0, const T *z = nullptr,
         double za = 0.0, const double *skip = nullptr) {
  const unsigned TB = 256;
  const unsigned G = crimson::grid_for((size_t)c.N * kRowLanes, TB);
  const unsigned Gn = crimson::grid_for((size_t)c.N * kNarrowLanes, TB);
  const int *rp = c.lhs->d_rowptr.p, *cl = c.lhs->d_col.p;
  const short *c16 = c.lhs->d_col16.p;
#define CR_SPMV_IX(R_, C_, CL_)                                                                           \
  do {                                                                                                     \
    if (R_ * C_ >= 9)                                                                                      \
      spmv_kernel<R_, C_, T, kRowLanes><<<G, TB, 0, c.s>>>(c.N, rp, CL_, A, x, y, (T)ya, z, (T)za, skip);   \
    else                                                                                                   \
      spmv_kernel<R_, C_, T, kNarrowLanes><<<Gn, TB, 0, c.s>>>(c.N, rp, CL_, A, x, y, (T)ya, z, (T)za, skip); \
  } while (0)
#define CR_SPMV(R_, C_)                  \
  do {                                   \
    if (c16)                             \
      CR_SPMV_IX(R_, C_, c16);           \
    else                                 \
      CR_SPMV_IX(R_, C_, cl);            \
  } while (0)
  if (nr == 3 && nc == 3) CR_SPMV(3, 3);
  else if (nr == 4 && nc == 4) CR_SPMV(4, 4);
  else if (nr == 3 && nc == 1) CR_SPMV(3, 1);
  else if (nr == 1 && nc == 3) CR_SPMV(1, 3);
  else if (nr == 1 && nc == 1) CR_SPMV(1, 1);
  else if (nr == 2 && nc == 2) CR_SPMV(2, 2);
  else if (nr == 2 && nc == 1) CR_SPMV(2, 1);
  else if (nr == 1 && nc == 2) CR_SPMV(1, 2);
  else {
    crimson::set_error("spmv block %dx%d not instantiated", nr, nc);
    return CRIMSON_EUNSUPPORTED;
  }
#undef CR_SPMV
#undef CR_SPMV_IX
  CR_HIP(hipGetLastError());
  return CRIMSON_OK;
}

// What a CG's operator needs beside its direction: the coupled faces' rank-one
// terms, and the scaled copy Ps(i) = W(off + wdof i) P(i) kept by the
// direction update (Ps null: none).
template <class T>
struct CgAux {
  FaceList fl{};
  const T *W = nullptr;
  int wdof = 0, off = 0;
  T *Ps = nullptr;
};
// Entries per thread and workgroups of the CG's vector sweeps.
struct CgGrid {
  int entries, blocks;
};
constexpr size_t kCgWide = (size_t)256 * kCgGrid / 2;  // entries past which a thread takes four
inline CgGrid cg_grid(size_t L) {
  const int E = L > kCgWide ? 4 : 1;
  return CgGrid{E, (int)std::min<size_t>((L + (size_t)256 * E - 1) / ((size_t)256 * E), kCgGrid)};
}
// The iterations' vector work: iteration `it` after its operator left SP and nd
// parts of P . SP.  P and Pn swap roles every iteration.
template <class T>
int cg_sweeps(Ctx<T> &c, size_t L, int it, int nd, const CgAux<T> &ax, T *X, T *R, const T *P, T *Pn, const T *SP,
              HostFlag hf) {
  double *scal = c.cgst.p + (it & 1) * kCgState, *next = c.cgst.p + ((it + 1) & 1) * kCgState;
  double *dpart = c.part.p, *rpart = c.part.p + kCgGrid;
  const CgGrid g = cg_grid(L);
  const int gp = g.blocks + ax.fl.nfc * ax.fl.nb;
  if (g.entries == 1) {
    cg_r_kernel<T, 1, false><<<g.blocks, 256, 0, c.s>>>(L, scal, dpart, nd, ax.fl, R, SP, rpart, nullptr, nullptr,
                                                        nullptr);
    cg_p_kernel<T, 1><<<gp, 256, 0, c.s>>>(L, scal, next, rpart, g.blocks, ax.fl, X, R, P, Pn, ax.W, ax.wdof, ax.off,
                                           ax.Ps, hf);
  } else {
    cg_r_kernel<T, 4, false><<<g.blocks, 256, 0, c.s>>>(L, scal, dpart, nd, ax.fl, R, SP, rpart, nullptr, nullptr,
                                                        nullptr);
    cg_p_kernel<T, 4><<<gp, 256, 0, c.s>>>(L, scal, next, rpart, g.blocks, ax.fl, X, R, P, Pn, ax.W, ax.wdof, ax.off,
                                           ax.Ps, hf);
  }
  CR_HIP(hipGetLastError());
  return CRIMSON_OK;
}
// R = P = X, X = 0, and the faces' dots with the first direction.
template <class T>
int cg_begin_vec(Ctx<T> &c, size_t L, const CgAux<T> &ax, T *X, T *R, T *P, const double *skip) {
  cg_begin_vec_kernel<T><<<crimson::grid_for(L, 256), 256, 0, c.s>>>(L, X, R, P, ax.W, ax.wdof, ax.off, ax.Ps, skip);
  if (ax.fl.nfc > 0) cg_begin_face_kernel<T><<<ax.fl.nfc * ax.fl.nb, 256, 0, c.s>>>(ax.fl, P, skip);
  CR_HIP(hipGetLastError());
  return CRIMSON_OK;
}

// Parts of P . SP of an operator that leaves none.
template <class T>
int cg_den(Ctx<T> &c, size_t L, const T *P, const T *SP, const double *done, int &nd) {
  nd = (int)std::min<size_t>((L + 255) / 256, kCgGrid);
  cg_den_kernel<T><<<nd, 256, 0, c.s>>>(L, P, SP, c.part.p, done);
  CR_HIP(hipGetLastError());
  return CRIMSON_OK;
}

// ----- the Schur operator: formed (schur_pattern) or in two passes -----
// An allocation that may fail without failing the solve: the error state is
// cleared and the caller takes the path that needs no such buffer.
template <class B>
bool try_alloc(B &b, size_t n) {
  if (b.alloc(n) == CRIMSON_OK) return true;
  (void)hipGetLastError();
  return false;
}

// Whether S's columns fit 2-byte offsets (twice the graph's band).
bool schur_narrow(const crimson_lhs *l) { return l->d_col16.p && 2 * l->band <= 32767; }
// How scattered the numbering is: the distinct 16-entry lines that the columns of 16
// consecutive rows name, per row, over a sample of the rows.  1 on a structured
// numbering, 14 on the same mesh numbered at random.
double lines_per_row(crimson_lhs *l) {
  if (l->lines >= 0.0) return l->lines;
  const int nt = std::max(1, l->nNo / 16), take = std::min(nt, 128);
  size_t lines = 0, rows = 0;
  std::vector<int> c;
  for (int k = 0; k < take; ++k) {
    const int r0 = 16 * (int)((long long)k * nt / take), r1 = std::min(r0 + 16, l->nNo);
    c.assign(l->h_col.begin() + l->h_rowptr[r0], l->h_col.begin() + l->h_rowptr[r1]);
    for (int &v : c) v /= 16;
    std::sort(c.begin(), c.end());
    lines += std::unique(c.begin(), c.end()) - c.begin();
    rows += r1 - r0;
  }
  return l->lines = (double)lines / (double)rows;
}
// Whether S is formed, as far as the graph's size and numbering tell.  Up to
// kCgPaired rows always: its two launches an iteration are what counts there.
// Beyond, S saves bytes (a Kuhn mesh's 65 entries of 10 bytes a row against 14.7
// blocks of 60; FP32 6 against 32; 2 more with 4-byte columns, of S, and 4 a block, of
// the matrix) and pays in gathers, 65 a row instead of 29, which leave the L2 once
// the vector has outgrown it and the numbering is scattered; in FP32, where it saves
// least, once the mesh is large.  Ms of a loose NS solve, formed and two passes
// (lines_per_row in brackets):
//   FP64, 2-byte columns  141 k 6.9, 9.2; 458 k 27.3, 34.6; 1,078 k 75.6, 94.1
//     4-byte [14]         141 k 12.5, 13.5; 327 k 34.6, 40.1; 390 k 51.3, 50.2;
//                         458 k 65.8, 62.0; 1,078 k 265, 201
//     [7.5]               270 k 19.3, 25.8; 458 k 45.2, 48.6; 1,078 k 160, 147
//     [5.2]               458 k 39.4, 43.7; 1,078 k 124, 126
//     [1]                 511 k 66.3, 73.7; 1,078 k 75.9, 94.1
//   FP32, 2-byte columns  141 k 6.0, 6.8; 458 k 17.7, 18.4; 675 k 29.5, 31.5;
//                         1,078 k 52.9, 50.9
//     4-byte [14]         72 k 5.8, 5.8; 141 k 11.0, 9.9; 458 k 41.5, 40.5
//     [7.5]               81 k 5.2, 5.6; 270 k 15.5, 16.3; 458 k 26.7, 31.1;
//                         1,078 k 109, 100
//     [1]                 300 k 27.7, 28.9; 378 k 31.1, 31.9; 486 k 38.1, 37.4;
//                         511 k 42.1, 40.0; 1,078 k 52.9, 50.3
bool schur_pays(crimson_lhs *l, bool fp32) {
  const int N = l->nNo;
  if (N <= kCgPaired) return true;
  if (fp32) return schur_narrow(l) ? N <= 3 << 18 : N <= 15 << 15 && (l->d_col16.p || lines_per_row(l) <= 10.0);
  if (N <= 5 << 16 || l->d_col16.p) return true;  // (2-byte columns: a window of 65,536 entries)
  return lines_per_row(l) <= (N <= 1 << 19 ? 10.0 : 6.0);
}

// The pattern of S, built once per handle and kept with it until it is released
// (release_idle_work); out stays empty where the graph keeps the two passes (two_pass)
// or an allocation failed (the next solve tries again).  A row of more than kSchurRow
// entries, anywhere, keeps the whole graph on the two passes: so do the Delaunay
// meshes of point clouds from about 6,500 nodes on, whose convex hull has a few nodes of
// many neighbours (1 row of 6,480, 10 of 14,007); meshes of bounded degree have none
// (a Delaunay mesh without its hull's slivers: 110 at most).  At most kSchurFill entries
// per block, kSchurFillLong past kCgPaired rows (a block and an entry of FP64 and 4-byte
// columns take as many bytes at 5.3).  At a fill of 4.8, ms formed and in two passes: 39 k
// rows FP64 2.2, 2.8, FP32 1.8, 2.2; 238 k rows FP64 9.6, 11.5, FP32 7.5, 7.2.
constexpr int kSchurFill = 6, kSchurFillLong = 5;
template <class IX, class OX>
int schur_pattern_fill(crimson_lhs *l, const IX *col, const crimson::SchurPattern &p, const OX *scol) {
  schur_pattern_kernel<IX, OX, true><<<crimson::grid_for(l->nNo, 4), 256, 0, l->stream>>>(
      l->nNo, l->d_rowptr.p, col, nullptr, p.ptr.p, const_cast<OX *>(scol));
  CR_HIP(hipGetLastError());
  CR_HIP(hipStreamSynchronize(l->stream));
  return CRIMSON_OK;
}
int schur_pattern(crimson_lhs *l, std::shared_ptr<const crimson::SchurPattern> &out) {
  out = crimson::pattern_of(l);
  if (out || l->two_pass) return CRIMSON_OK;
  const int N = l->nNo;
  auto p = std::make_shared<crimson::SchurPattern>();
  crimson::DBuf<int> cnt;
  if (!try_alloc(cnt, (size_t)N) || !try_alloc(p->ptr, (size_t)N + 1)) return CRIMSON_OK;
  const unsigned G = crimson::grid_for(N, 4);
  if (l->d_col16.p)
    schur_pattern_kernel<short, int, false><<<G, 256, 0, l->stream>>>(N, l->d_rowptr.p, l->d_col16.p, cnt.p, nullptr,
                                                                      nullptr);
  else
    schur_pattern_kernel<int, int, false><<<G, 256, 0, l->stream>>>(N, l->d_rowptr.p, l->d_col.p, cnt.p, nullptr,
                                                                    nullptr);
  CR_HIP(hipGetLastError());
  std::vector<int> ptr((size_t)N + 1);
  CR_HIP(hipMemcpyAsync(ptr.data() + 1, cnt.p, (size_t)N * sizeof(int), hipMemcpyDeviceToHost, l->stream));
  CR_HIP(hipStreamSynchronize(l->stream));
  ptr[0] = 0;
  const long long fill = N <= kCgPaired ? kSchurFill : kSchurFillLong;
  for (int i = 1; i <= N; ++i) {
    p->row = std::max(p->row, ptr[i]);
    p->nnz += ptr[i];
    ptr[i] = (int)p->nnz;
    if (p->row > kSchurRow || p->nnz > fill * l->nnz || p->nnz > 0x7fffff00LL) {
      l->two_pass = true;
      return CRIMSON_OK;
    }
  }
  CR_TRY(p->ptr.upload(ptr.data(), ptr.size(), l->stream));
  CR_HIP(hipStreamSynchronize(l->stream));
  const bool narrow = schur_narrow(l);
  if (!(narrow ? try_alloc(p->col16, (size_t)p->nnz) : try_alloc(p->col, (size_t)p->nnz))) return CRIMSON_OK;
  if (narrow)
    CR_TRY(schur_pattern_fill(l, l->d_col16.p, *p, p->col16.p));
  else if (l->d_col16.p)
    CR_TRY(schur_pattern_fill(l, l->d_col16.p, *p, p->col.p));
  else
    CR_TRY(schur_pattern_fill(l, l->d_col.p, *p, p->col.p));
  out = p;
  crimson::pattern_keep(l, out);
  return CRIMSON_OK;
}

template <class T>
struct SchurOp {
  const crimson::SchurPattern *pat = nullptr;  // formed: S's pattern and values
  T *S = nullptr;
  MatView<T> L, Gt, G;
  T *Z = nullptr, *Ps = nullptr;  // two passes: Z(4, N) and the scaled direction
};
// S's values from the matrix and the scaling of this solve.
template <class T>
int schur_form(Ctx<T> &c, const SchurOp<T> &o) {
  if (!o.pat) return CRIMSON_OK;
  crimson_lhs *l = c.lhs;
  const crimson::SchurPattern &p = *o.pat;
  const unsigned G = crimson::grid_for(l->nNo, 16);
  const size_t sh = (size_t)16 * p.row * (sizeof(double) + sizeof(int));
#define CR_SV(IX_, CP_, OX_, SP_)                                                                               \
  schur_values_kernel<T, IX_, OX_><<<G, 256, sh, c.s>>>(l->nNo, l->d_rowptr.p, CP_, o.L, o.Gt, o.G, p.ptr.p, SP_, \
                                                        o.S, p.row)
  if (p.col16.p)
    CR_SV(short, l->d_col16.p, short, p.col16.p);
  else if (l->d_col16.p)
    CR_SV(short, l->d_col16.p, int, p.col.p);
  else
    CR_SV(int, l->d_col.p, int, p.col.p);
#undef CR_SV
  CR_HIP(hipGetLastError());
  return CRIMSON_OK;
}
// SP = S P of the formed complement with the new direction and the parts of P . SP.
template <class T>
int schur_dir_product(Ctx<T> &c, const SchurOp<T> &o, const PairT<T> *Q, T *P, T *SP, const double *scal, double *next,
                      int nr, const FaceList &fl, HostFlag hf, int &nd) {
  const int N = c.N, ntile = (int)crimson::grid_for((size_t)N, 256 / kSLanes);
  nd = std::min(ntile, kCgGrid);
  const int G = nd + fl.nfc * fl.nb;
  const crimson::SchurPattern &p = *o.pat;
  double *dpart = c.part.p, *rpart = c.part.p + kCgGrid;
  if (p.col16.p)
    s_dir_product_kernel<T, short><<<G, 256, 0, c.s>>>(N, ntile, p.ptr.p, p.col16.p, o.S, Q, P, SP, dpart, scal, next,
                                                       rpart, nr, fl, hf);
  else
    s_dir_product_kernel<T, int><<<G, 256, 0, c.s>>>(N, ntile, p.ptr.p, p.col.p, o.S, Q, P, SP, dpart, scal, next,
                                                     rpart, nr, fl, hf);
  CR_HIP(hipGetLastError());
  return CRIMSON_OK;
}
// SP = S P and the parts of P . SP; the faces' terms join in the CG's sweeps.
template <class T>
int schur_apply(Ctx<T> &c, const SchurOp<T> &o, const T *P, T *SP, const double *done, int &nd) {
  crimson_lhs *l = c.lhs;
  const int N = l->nNo;
  double *dpart = c.part.p;
  if (o.pat) {
    const int ntile = (int)crimson::grid_for((size_t)N, 256 / kSLanes);
    nd = std::min(ntile, kCgGrid);
    const crimson::SchurPattern &p = *o.pat;
    if (p.col16.p)
      s_product_kernel<T, short><<<nd, 256, 0, c.s>>>(N, ntile, p.ptr.p, p.col16.p, o.S, P, SP, dpart, done);
    else
      s_product_kernel<T, int><<<nd, 256, 0, c.s>>>(N, ntile, p.ptr.p, p.col.p, o.S, P, SP, dpart, done);
    CR_HIP(hipGetLastError());
    return CRIMSON_OK;
  }
  const unsigned gr = crimson::grid_for((size_t)N * kNarrowLanes, 256);
  if (l->d_col16.p) {
    g_product_kernel<T, short><<<gr, 256, 0, c.s>>>(N, l->d_rowptr.p, l->d_col16.p, o.G, o.Ps, o.Z, done);
    schur_kernel<T, short><<<gr, 256, 0, c.s>>>(N, l->d_rowptr.p, l->d_col16.p, o.L, o.Gt, P, o.Z, SP, done);
  } else {
    g_product_kernel<T, int><<<gr, 256, 0, c.s>>>(N, l->d_rowptr.p, l->d_col.p, o.G, o.Ps, o.Z, done);
    schur_kernel<T, int><<<gr, 256, 0, c.s>>>(N, l->d_rowptr.p, l->d_col.p, o.L, o.Gt, P, o.Z, SP, done);
  }
  return cg_den(c, (size_t)N, P, SP, done, nd);
}

// The support of a coupled face's dot functional (FaceDev): the columns of
// the face nodes' rows, each with its (face node, CSR entry) pairs, from the
// host copy of the pattern; built once per face (the pattern is fixed).
int face_support(crimson_lhs *l, CrFace &fa) {
  if (fa.qpat) return CRIMSON_OK;
  std::vector<std::array<int, 3>> t;  // (column j, face node a, entry k)
  for (int a = 0; a < fa.nNo; ++a) {
    const int g = fa.glob[a];
    for (int k = l->h_rowptr[g]; k < l->h_rowptr[g + 1]; ++k) t.push_back({l->h_col[k], a, k});
  }
  std::sort(t.begin(), t.end());
  std::vector<int> sup, ptr, qa, qk;
  for (size_t p = 0; p < t.size(); ++p) {
    if (p == 0 || t[p][0] != t[p - 1][0]) {
      sup.push_back(t[p][0]);
      ptr.push_back((int)p);
    }
    qa.push_back(t[p][1]);
    qk.push_back(t[p][2]);
  }
  ptr.push_back((int)t.size());
  fa.nsup = (int)sup.size();
  fa.h_sup = sup;
  fa.support = crimson::next_alloc_serial();
  if (fa.nsup > 0) {
    CR_TRY(fa.d_sup.upload(sup.data(), sup.size(), l->stream));
    CR_TRY(fa.d_qptr.upload(ptr.data(), ptr.size(), l->stream));
    CR_TRY(fa.d_qa.upload(qa.data(), qa.size(), l->stream));
    CR_TRY(fa.d_qk.upload(qk.data(), qk.size(), l->stream));
    CR_TRY(fa.d_q.alloc(sup.size()));
    CR_HIP(hipStreamSynchronize(l->stream));
  }
  fa.qpat = true;
  return CRIMSON_OK;
}

// The merged supports of the coupled faces (FaceList), kept with the workspace
// while the same faces are coupled.
template <class T>
int face_list(Ctx<T> &c) {
  crimson_lhs *l = c.lhs;
  if (c.nfc() == 0) return CRIMSON_OK;
  std::vector<unsigned long long> sig;
  for (const auto &fa : l->face)
    if (fa.coupled) sig.push_back(fa.support);
  if (sig == c.fent_sig && c.ftptr.p) return CRIMSON_OK;
  const int N = l->nNo;
  std::vector<int> count((size_t)N, 0);
  size_t total = 0;
  for (const auto &fa : l->face)
    if (fa.coupled)
      for (int j : fa.h_sup) {
        ++count[j];
        ++total;
      }
  // sized by the entries, whatever the faces share: a capture's buffers stay in place
  std::vector<FaceNode> node(total, FaceNode{});
  std::vector<FaceEnt> ent(total);
  std::vector<int> ptr((size_t)(N + 255) / 256 + 1, 0);
  int u = 0, e = 0;
  for (int j = 0; j < N; ++j) {
    if (j % 256 == 0) ptr[j / 256] = u;
    if (count[j] == 0) continue;
    node[u++] = FaceNode{j, e + 1, e + count[j], FaceEnt{0, 0}};
    e += count[j];
    count[j] = e - count[j];  // the node's next entry
  }
  ptr.back() = u;
  int f = 0;
  for (const auto &fa : l->face) {
    if (!fa.coupled) continue;
    for (size_t k = 0; k < fa.h_sup.size(); ++k) ent[count[fa.h_sup[k]]++] = FaceEnt{f, (int)k};
    ++f;
  }
  for (int k = 0; k < u; ++k) node[k].first = ent[node[k].more - 1];
  c.fent_sig.clear();
  CR_TRY(c.fent.upload(ent.data(), ent.size(), c.s));
  CR_TRY(c.fnode.upload(node.data(), node.size(), c.s));
  CR_TRY(c.ftptr.upload(ptr.data(), ptr.size(), c.s));
  CR_HIP(hipStreamSynchronize(c.s));
  c.fent_sig = sig;
  return CRIMSON_OK;
}
// The faces' functionals q for this solve's matrix and scaling.
template <class T>
int face_functionals(Ctx<T> &c, const MatView<T> &G) {
  for (auto &fa : c.lhs->face)
    if (fa.coupled && fa.nsup > 0)
      face_q_kernel<T><<<crimson::grid_for(fa.nsup, 256), 256, 0, c.s>>>(
          fa.nsup, fa.d_sup.p, fa.d_qptr.p, fa.d_qa.p, fa.d_qk.p, fa.d_glob.p, fa.d_valM.p, fa.dof, G, fa.d_q.p);
  CR_HIP(hipGetLastError());
  return CRIMSON_OK;
}

__device__ inline double dmax(double a, double b) { return a < b ? b : a; }  // std::max's choice

// The deciding kernels: one workgroup of kDotThreads, which sums the dots'
// parts; thread 0 decides, in the order of operations of the host form of
// memLS (FMA contraction off).
__device__ inline double sum_dots(const double *__restrict__ part, int n, double *sh) {
  double v = 0.0;
  for (int k = threadIdx.x; k < n; k += kDotThreads) v += part[k];
  return block_sum_1024(v, sh);
}
__global__ void __launch_bounds__(kDotThreads) ns_begin_kernel(double *__restrict__ g, const double *__restrict__ part,
                                                               int nb, double absTol, double relTol) {
#pragma clang fp contract(off)
  __shared__ double sh[16];
  const double eps = sqrt(sum_dots(part, nb, sh));
  if (threadIdx.x != 0) return;
  g[G_RI_INORM] = eps;
  g[G_RI_FNORM] = eps;
  g[G_RI_EPS] = dmax(absTol, relTol * eps);
  g[G_RI_SKIP] = 0.0;
  g[G_RI_SUC] = 0.0;
  g[G_RI_ITR] = 0.0;
  g[G_ERR] = 0.0;
  g[G_GM_ITR] = 0.0;
  g[G_CG_ITR] = 0.0;
  g[G_GM_LASTF] = g[G_GM_LASTD] = 0.0;
}
// skip (may be null): the outer loop is over, the call does nothing
__global__ void gm_begin_kernel(double *__restrict__ g, const double *__restrict__ skip) {
  g[G_GM_ARN] = 1.0;
  if (skip && *skip != 0.0) {
    g[G_GM_CYC] = 1.0;
    return;
  }
  g[G_GM_CYC] = 0.0;
  g[G_GM_SUC] = 0.0;
  g[G_GM_EARLY] = 0.0;
}
// the norm of a cycle's first vector (parts npart[0, nb)), the first cycle's
// targets; count: this cycle's residual took a product
__global__ void __launch_bounds__(kDotThreads) gm_cycle_kernel(double *__restrict__ g, int l, int count,
                                                               double absTol, double relTol,
                                                               const double *__restrict__ npart, int nb,
                                                               double *__restrict__ err) {
#pragma clang fp contract(off)
  if (g[G_GM_CYC] != 0.0) return;
  __shared__ double sh[16];
  const double e0 = sqrt(sum_dots(npart, nb, sh));
  if (threadIdx.x != 0) return;
  err[0] = e0;
  if (l == 1) {
    const double eps = e0;
    g[G_GM_E0] = e0;
    if (eps <= absTol) {
      g[G_GM_EARLY] = 1.0;
      g[G_GM_CYC] = 1.0;
      g[G_GM_ARN] = 1.0;
      return;
    }
    g[G_GM_INORM] = eps;
    g[G_GM_FNORM] = eps;
    g[G_GM_EPS] = dmax(absTol, relTol * eps);
  }
  if (count) g[G_GM_ITR] = g[G_GM_ITR] + 1.0;
  g[G_GM_DBPRE] = g[G_GM_FNORM];
  g[G_GM_SCALE] = 1.0 / e0;
  g[G_GM_ARN] = 0.0;
  g[G_GM_I] = 0.0;
}
__global__ void __launch_bounds__(kDotThreads) gm_givens_kernel(Givens G) {
  __shared__ double sh[16], w3[3][256];
  const double *n2 = G.n2;
  const double s2 = block_sum_1024((int)threadIdx.x < G.nb ? n2[threadIdx.x] : 0.0, sh);
  gm_givens(G, s2, w3);
}
// the cycle's back substitution, one thread per unknown, a column at a time
// (its read is in flight during the column before)
__global__ void __launch_bounds__(256) gm_solve_kernel(double *__restrict__ g, int sD, const double *__restrict__ H,
                                                       const double *__restrict__ err, double *__restrict__ y) {
#pragma clang fp contract(off)
  if (g[G_GM_CYC] != 0.0) return;
  __shared__ double yj[2];
  const int ld = sD + 1, t = threadIdx.x;
  const int i = (int)g[G_GM_I];
  double v = t < i ? err[t] : 0.0;
  double h = i > 0 && t < i ? H[t + (size_t)ld * (i - 1)] : 0.0;
  for (int j = i - 1; j >= 0; --j) {
    const double hn = j > 0 && t < j ? H[t + (size_t)ld * (j - 1)] : 0.0;
    if (t == j) {
      v = v / h;
      yj[j & 1] = v;
    }
    __syncthreads();
    if (t < j) v = v - h * yj[j & 1];
    h = hn;
  }
  if (t < i) y[t] = v;
  if (t == 0) {
    g[G_GM_APPLY] = (double)i;
    g[G_GM_FNORM] = fabs(err[i]);
  }
}
__global__ void gm_endcycle_kernel(double *__restrict__ g) {
  if (g[G_GM_CYC] != 0.0) return;
  if (g[G_GM_SUC] != 0.0) g[G_GM_CYC] = 1.0;
  g[G_GM_ARN] = 1.0;
  g[G_GM_LASTF] = g[G_GM_FNORM];
  g[G_GM_LASTD] = g[G_GM_DBPRE];
}
// skip and g may be null (a plain CG solve)
__global__ void __launch_bounds__(kDotThreads) cg_begin_kernel(double *__restrict__ scal, double *__restrict__ g,
                                                               const double *__restrict__ skip,
                                                               const double *__restrict__ part, int nb, double absTol,
                                                               double relTol, int mItr) {
#pragma clang fp contract(off)
  if (skip && *skip != 0.0) {
    if (threadIdx.x == 0) scal[5] = 1.0;
    return;
  }
  __shared__ double sh[16];
  const double e = sqrt(sum_dots(part, nb, sh));
  if (threadIdx.x != 0) return;
  if (g) g[G_CG_INORM] = e;
  double eps = dmax(absTol, relTol * e);
  eps = eps * eps;
  scal[0] = e * e;
  scal[1] = e * e;
  scal[2] = eps;
  scal[3] = scal[4] = scal[5] = scal[6] = 0.0;
  scal[7] = (double)mItr;
  scal[8] = 0.0;
  scal[9] = e;
  check_next(scal);  // the first iteration's test
}
__global__ void cg_end_kernel(const double *__restrict__ scal, double *__restrict__ g,
                              const double *__restrict__ skip) {
  if (*skip != 0.0) return;
  g[G_CG_ITR] = g[G_CG_ITR] + (double)(int)scal[6];
  g[G_CG_SUC] = scal[8];
  g[G_CG_ERR] = scal[0];
  g[G_CG_ERRO] = scal[1];
}
// NSSOLVER iteration i's dots in one launch, grid z: MX(iB) against MX(1..iB),
// MX(iBB) against MX(1..iBB), and the right-hand side against the two
// (L = 4 N: velocity and pressure parts together).
template <class T>
__global__ void __launch_bounds__(kDotThreads) ns_dots_kernel(size_t L, const T *__restrict__ MX,
                                                              const T *__restrict__ r0, int iB,
                                                              double *__restrict__ part, size_t pz,
                                                              const double *__restrict__ skip) {
  if (*skip != 0.0) return;
  __shared__ double sh[kDotThreads / 64][kDotGroup];
  const int z = blockIdx.z;
  const T *b = MX + L * (size_t)(iB - 1);
  const int m = z == 0 ? iB : z == 1 ? iB + 1 : 2;
  if ((int)blockIdx.y * kDotGroup >= m) return;
  dots_body(L, z == 0 ? b : z == 1 ? b + L : r0, z == 2 ? b : MX, L, m, 0, part + pz * z, sh);
}
// NSSOLVER iteration i's Gram rows iB = 2i-1, iBB = 2i from their dots
// (ns_dots_kernel's parts), then GE (memLS.f90:607-677) and the stopping test;
// A (nB, nB), C the GE scratch (Nn, Nn+1) when it does not fit the workgroup's.
// Pivot search and back substitution by thread 0, the eliminations by all.
constexpr int kGeLds = 48;
__global__ void __launch_bounds__(kDotThreads) ns_gram_kernel(double *__restrict__ g, int i, int nB,
                                                              const double *__restrict__ part, size_t pz, int nb,
                                                              double *__restrict__ A, double *__restrict__ Bv,
                                                              double *__restrict__ xB, double *__restrict__ Cg,
                                                              HostFlag hf) {
#pragma clang fp contract(off)
  if (g[G_RI_SKIP] != 0.0) {
    if (threadIdx.x == 0) hf.tell(true);
    return;
  }
  __shared__ double Cl[kGeLds * (kGeLds + 1)];
  __shared__ int piv, bad;
  const int iB = 2 * i - 1, iBB = 2 * i, Nn = iBB, t = threadIdx.x;
  for (int d = t / 64; d < iB + iBB + 2; d += kDotThreads / 64) {
    const int z = d < iB ? 0 : d < iB + iBB ? 1 : 2;
    const int j = z == 0 ? d : z == 1 ? d - iB : d - iB - iBB;
    const double v = wave_parts(part + pz * z + (size_t)j * nb, nb);
    if (t % 64 == 0) {
      if (z == 2) {
        Bv[iB - 1 + j] = v;
      } else {
        const int k = z == 0 ? iB - 1 : iBB - 1;
        A[j + (size_t)nB * k] = v;
        A[k + (size_t)nB * j] = v;
      }
    }
  }
  if (t == 0) {
    g[G_RI_DBPRE] = g[G_RI_FNORM];
    bad = 0;
  }
  __syncthreads();
  if (Nn == 2) {
    if (t == 0) {
      const double a11 = A[0], a21 = A[1], a12 = A[nB], a22 = A[nB + 1], b0 = Bv[0], b1 = Bv[1];
      const double pivot = a11 * a22 - a21 * a12;
      xB[0] = (b0 * a22 - b1 * a12) / pivot;
      xB[1] = (b1 * a11 - b0 * a21) / pivot;
    }
  } else {
    double *C = Nn <= kGeLds ? Cl : Cg;
#define CC(r, cc) C[(r) + (size_t)Nn * (cc)]
    for (int e = t; e < Nn * (Nn + 1); e += kDotThreads) {
      const int r = e % Nn, cc = e / Nn;
      C[e] = cc < Nn ? A[r + (size_t)nB * cc] : Bv[r];
    }
    __syncthreads();
    for (int m = 0; m < Nn - 1; ++m) {
      if (t == 0) {
        int ipv = m;
        double pivot = fabs(CC(m, m));
        for (int r = m + 1; r < Nn; ++r)
          if (fabs(CC(r, m)) > pivot) {
            ipv = r;
            pivot = fabs(CC(r, m));
          }
        piv = ipv;
        if (pivot < 2.0 * 2.220446049250313e-16) bad = 1;
      }
      __syncthreads();
      if (bad) break;
      const int ipv = piv;
      if (ipv != m)
        for (int cc = m + t; cc <= Nn; cc += kDotThreads) {
          const double v = CC(m, cc);
          CC(m, cc) = CC(ipv, cc);
          CC(ipv, cc) = v;
        }
      __syncthreads();
      const int nr = Nn - 1 - m, ncol = Nn - m;  // rows below m, columns past m
      for (int e = t; e < nr * ncol; e += kDotThreads) {
        const int r = m + 1 + e % nr, cc = m + 1 + e / nr;
        const double sv = CC(r, m) / CC(m, m);
        CC(r, cc) = CC(r, cc) - sv * CC(m, cc);
      }
      __syncthreads();
    }
    if (t == 0 && !bad) {
      for (int j = Nn - 1; j >= 0; --j) {
        double v = CC(j, Nn);
        for (int r = j + 1; r < Nn; ++r) v = v - CC(j, r) * CC(r, Nn);
        v = v / CC(j, j);
        CC(j, Nn) = v;
        xB[j] = v;
      }
    }
#undef CC
  }
  if (t != 0) return;
  if (bad) {
    g[G_ERR] = 1.0;
    g[G_RI_SKIP] = 1.0;
    hf.tell(true);
    return;
  }
  double sxb = 0.0;
  for (int k = 0; k < iBB; ++k) sxb = sxb + xB[k] * Bv[k];
  const double iN = g[G_RI_INORM];
  const double fN = sqrt(iN * iN - sxb);
  g[G_RI_FNORM] = fN;
  const bool done = fN < g[G_RI_EPS];
  if (done) {
    g[G_RI_SUC] = 1.0;
    g[G_RI_ITR] = (double)i;
    g[G_RI_SKIP] = 1.0;
  }
  hf.tell(done);
}
// after the outer loop: the iteration count, and the solution's
// coefficients cu(k) = xB(2k), cp(k) = xB(2k-1) (1-based)
__global__ void ns_final_kernel(double *__restrict__ g, int mItr, const double *__restrict__ xB,
                                double *__restrict__ cu, double *__restrict__ cp) {
  if (g[G_ERR] != 0.0) return;
  if (g[G_RI_SUC] == 0.0) g[G_RI_ITR] = (double)mItr;
  const int nit = (int)g[G_RI_ITR];
  g[G_NS_CNT] = 2.0 * nit;
  for (int k = 1; k <= nit; ++k) {
    cu[k - 1] = xB[2 * k - 1];
    cp[k - 1] = xB[2 * k - 2];
  }
}
__global__ void __launch_bounds__(kDotThreads) ns_rc_kernel(double *__restrict__ g, const double *__restrict__ part,
                                                            int nb) {
  if (g[G_ERR] != 0.0) return;
  __shared__ double sh[16];
  const double s = sum_dots(part, nb, sh);
  if (threadIdx.x == 0) g[G_RC_N2] = s;
}

struct SegCapture;
int seg_cut(SegCapture *cap);
// The workspaces of a solve and its progress.  A captured solve owns one and enqueues
// every possible iteration (GMRES: mItr cycles of sD Arnoldi steps; CGRAD: mItr
// iterations; NSSOLVER: mItr outer iterations), whose launches past
// convergence see their flag and return at once.  A plain solve runs the same launch sequence,
// polls the flags a step behind (HostFlag) and stops enqueueing; its workspace
// stays with the matrix handle for the next solve (take_work).
template <class T>
struct SolveWork : crimson::SolveWorkBase {
  Ctx<T> c;
  crimson::DBuf<T> r0, r, X, MX;          // NS: (3,N)|(N) vectors; X: U_i|P_i, MX: their images
  crimson::DBuf<T> t3, t4, t5, ps, z;     // CG: R (paired: Q), the directions; two-pass operator: Ps, Z
  crimson::DBuf<T> wa, wb, ws, gmU;       // GMRES: the two working vectors, W o w, the basis
  crimson::DBuf<double> gst, npart, h;    // state and small systems; norm parts (2 kSubGrid); h1, h2
  int sD = 0, nB = 0, mRI = 0, mGM = 0, mCG = 0;
  double riAbs = 0, riRel = 0, gmAbs = 0, gmRel = 0, cgAbs = 0, cgRel = 0;
  // the Schur complement where it is formed (schur_ready): its pattern and values
  std::shared_ptr<const crimson::SchurPattern> spat;
  crimson::DBuf<T> S;
  bool paired = false;    // its CG keeps R and P together (kCgPaired)
  SegCapture *cap = nullptr;  // the capture in progress, cut between the solve's phases
  size_t oH = 0, ocs = 0, osn = 0, oerr = 0, oy = 0, oA = 0, oBv = 0, oxB = 0, oC = 0, ocu = 0, ocp = 0;
  // a plain solve's flag word (pinned) and the number of its last teller
  bool polled = false;
  unsigned long long *word = nullptr, seq = 0;
  double tGM = 0.0, tCG = 0.0;  // its time in the momentum solves and in the CG (callD)

  ~SolveWork() override {
    if (word) (void)hipHostFree(word);
  }
  size_t bytes() const override {
    return sizeof(T) * (c.W.n + c.fix.n + r0.n + r.n + X.n + MX.n + t3.n + t4.n + t5.n + ps.n + z.n + wa.n + wb.n +
                        ws.n + gmU.n + S.n) +
           sizeof(double) * (c.part.n + gst.n + npart.n + h.n);
  }
  double *G(size_t off) { return gst.p + off; }
  int cut();
  int poll_ready() {
    polled = true;
    if (word) return CRIMSON_OK;
    if (hipHostMalloc((void **)&word, 64) != hipSuccess) {
      word = nullptr;
      (void)hipGetLastError();
      crimson::set_error("hipHostMalloc of the solve's flag word failed");
      return CRIMSON_ENOMEM;
    }
    *(volatile unsigned long long *)word = 0;
    return CRIMSON_OK;
  }
  HostFlag flag() { return polled ? HostFlag{word, ++seq} : HostFlag{nullptr, 0}; }
  // Waits for teller `k` (or a later one); *stop: whether its loop is over.  Ends also when the
  // stream has failed, or is idle without the teller having told.
  int wait(unsigned long long k, bool *stop) {
    const volatile unsigned long long *w = word;
    for (unsigned n = 1;; ++n) {
      const unsigned long long v = *w;
      if (v >> 1 >= k) {
        *stop = v & 1;
        return CRIMSON_OK;
      }
      if (n % 4096 == 0) {
        const hipError_t e = hipStreamQuery(c.s);
        if (e == hipErrorNotReady) continue;
        if (e == hipSuccess && *w >> 1 >= k) continue;
        crimson::set_error("memLS: the solve's stream ended before its step reported: %s", hipGetErrorString(e));
        return CRIMSON_EHIP;
      }
    }
  }
};
template <class T>
int SolveWork<T>::cut() {
  return seg_cut(cap);
}

inline int dot_blocks(size_t L) { return (int)std::min<size_t>((L + kDotThreads - 1) / kDotThreads, kDotGrid); }
template <class T>
int dots(Ctx<T> &c, size_t L, const T *v, const T *U0, size_t ustride, int m, bool self, double *part,
         const double *skip) {
  dots_kernel<T><<<dim3(dot_blocks(L), (m + (self ? 1 : 0) + kDotGroup - 1) / kDotGroup), kDotThreads, 0, c.s>>>(
      L, v, U0, ustride, m, self ? 1 : 0, part, skip);
  CR_HIP(hipGetLastError());
  return CRIMSON_OK;
}
template <class T>
int face_apply(Ctx<T> &c, int what, int xdof, const T *X, T *Y, const double *skip) {
  if (c.nfc() == 0) return CRIMSON_OK;
  if (c.disjoint || c.fnodes <= kFaceSerial) {
    face_apply_kernel<T><<<c.disjoint ? c.nfc() : 1, 1024, 0, c.s>>>(c.fdev.p, c.nfc(), what, xdof, X, Y, c.fsum.p,
                                                                    skip);
  } else {
    for (int kind = kFaceAdd; kind <= kFacePre; kind <<= 1) {
      if (!(what & kind)) continue;
      face_dot_kernel<T><<<c.nfc(), 1024, 0, c.s>>>(c.fdev.p, xdof, kind == kFaceAdd ? X : Y, c.fsum.p, skip);
      for (int f = 0; f < c.nfc(); ++f)
        if (c.hfdev[f].nNo > 0)
          face_add_kernel<T><<<crimson::grid_for(c.hfdev[f].nNo, 256), 256, 0, c.s>>>(c.fdev.p, f, kind, xdof,
                                                                                     c.fsum.p, Y, skip);
    }
  }
  CR_HIP(hipGetLastError());
  return CRIMSON_OK;
}

template <class T, class IX>
void arnoldi_spmv_ix(Ctx<T> &c, const MatView<T> &A, int nd, const IX *col, const T *w, const T *ws, T *u, T *y,
                     const Givens &gv) {
  const int *rp = c.lhs->d_rowptr.p;
  const unsigned own = gv.i > 0 ? 1 : 0, G = crimson::grid_for((size_t)c.N * kRowLanes, 256) + own,
                 Gn = crimson::grid_for((size_t)c.N * kNarrowLanes, 256) + own;
  switch (nd) {
    case 1: arnoldi_spmv_kernel<1, T, IX><<<Gn, 256, 0, c.s>>>(c.N, rp, col, A, w, ws, u, y, gv); break;
    case 2: arnoldi_spmv_kernel<2, T, IX><<<Gn, 256, 0, c.s>>>(c.N, rp, col, A, w, ws, u, y, gv); break;
    case 3: arnoldi_spmv_kernel<3, T, IX><<<G, 256, 0, c.s>>>(c.N, rp, col, A, w, ws, u, y, gv); break;
    default: arnoldi_spmv_kernel<4, T, IX><<<G, 256, 0, c.s>>>(c.N, rp, col, A, w, ws, u, y, gv); break;
  }
}
// The two passes over vectors of at most kOrthMost entries: a workgroup's
// entries so few that the vector has as many workgroups as the parts allow.
template <class T, int JS>
void arnoldi_orth(Ctx<T> &c, size_t L, int nd, const MatView<T> &A, T *y, T *ys, const T *U, int m, double *h1,
                  double *h2, double *n1, double *n2, double *g, int &nb) {
  const int pad = nd == 3 ? 4 : nd;
  nb = (int)crimson::grid_for(L, kDotThreads / JS);
  double *part2 = c.part.p + (size_t)kDotGrid * 264;
  arnoldi_orth_kernel<T, JS, true><<<nb, kDotThreads, 0, c.s>>>(L, nd, pad, A.W, A.wdof, A.c0, y, ys, U, L, m, c.part.p,
                                                                dot_blocks(L), h1, n1, part2, nullptr, nullptr, g);
  arnoldi_orth_kernel<T, JS, false><<<nb, kDotThreads, 0, c.s>>>(L, nd, pad, A.W, A.wdof, A.c0, y, ys, U, L, m, part2,
                                                                 nb, h2, n2, nullptr, h1 + m, n1, g);
}

// GMRES (memLS.f90:681-788) for the operator x -> A x + ADD(x), left
// preconditioned by PRE (pre: the NS solver's momentum solves; GMRESV takes
// none, and counts the first residual too, :827-829); R, X are (nd, N).  Classical Gram-Schmidt with
// a DGKS second pass where memLS orthogonalises one vector after the other
// (:743-746): the same Krylov space, solutions equal to the solver tolerance.
struct GmParams {
  int mItr, sD;
  double absTol, relTol;
  bool pre, count_first;
};
template <class T>
int gmres_run(SolveWork<T> &w, const MatView<T> &A, int nd, const T *R, T *X, const GmParams &p, const double *skip) {
  Ctx<T> &c = w.c;
  const size_t L = (size_t)nd * c.N;
  const int pad = nd == 3 ? 4 : nd;
  double *g = w.gst.p, *h1 = w.h.p, *h2 = w.h.p + 256, *n1 = w.npart.p, *n2 = w.npart.p + kSubGrid;
  const double *cyc = g + G_GM_CYC, *arn = g + G_GM_ARN;
  T *U = w.gmU.p, *v = w.wa.p, *y = w.wb.p;
  const unsigned GL = crimson::grid_for(L, 256);
  const bool small = L <= kOrthMost;
  const int nb0 = (int)std::min<size_t>((L + kDotThreads - 1) / kDotThreads, kSubGrid), np = dot_blocks(L);
  int nb = nb0;  // parts of n1 and n2
  auto givens = [&](int i, HostFlag hf) {
    return Givens{g, i, p.sD, h1, h2, n2, nb, w.G(w.oH), w.G(w.ocs), w.G(w.osn), w.G(w.oerr), hf};
  };
  gm_begin_kernel<<<1, 1, 0, c.s>>>(g, skip);
  fill_kernel<T><<<GL, 256, 0, c.s>>>(L, X, skip);
  for (int l = 1; l <= p.mItr; ++l) {
    if (l == 1) {
      copy_kernel<T><<<GL, 256, 0, c.s>>>(L, R, v, cyc);  // X = 0: R - A X is R
    } else {
      CR_TRY(spmv(c, A, nd, nd, X, v, 1.0, static_cast<const T *>(nullptr), 0.0, cyc));
      CR_TRY(face_apply(c, kFaceAdd, nd, X, v, cyc));
      diff_kernel<T><<<GL, 256, 0, c.s>>>(L, R, v, v, cyc);
    }
    if (p.pre) CR_TRY(face_apply(c, kFacePre, nd, v, v, cyc));
    arnoldi_first_kernel<T><<<nb0, kDotThreads, 0, c.s>>>(L, nd, pad, A.W, A.wdof, A.c0, v, w.ws.p, n1, cyc);
    gm_cycle_kernel<<<1, kDotThreads, 0, c.s>>>(g, l, l > 1 || p.count_first, p.absTol, p.relTol, n1, nb0,
                                                w.G(w.oerr));
    bool stop = false;
    for (int i = 1; i <= p.sD; ++i) {
      T *u = U + L * (size_t)(i - 1);
      const bool ends = small && i > 1;  // the step before ends in this one's product
      const Givens gv = givens(ends ? i - 1 : 0, ends ? w.flag() : HostFlag{nullptr, 0});
      if (c.lhs->d_col16.p)
        arnoldi_spmv_ix(c, A, nd, c.lhs->d_col16.p, v, w.ws.p, u, y, gv);
      else
        arnoldi_spmv_ix(c, A, nd, c.lhs->d_col.p, v, w.ws.p, u, y, gv);
      CR_TRY(face_apply(c, kFaceAdd | (p.pre ? kFacePre : 0), nd, u, y, arn));
      CR_TRY(dots(c, L, y, U, L, i, true, c.part.p, arn));
      if (small) {
        if (L <= kOrthMost / 4)
          arnoldi_orth<T, 4>(c, L, nd, A, y, w.ws.p, U, i, h1, h2, n1, n2, g, nb);
        else if (L <= kOrthMost / 2)
          arnoldi_orth<T, 2>(c, L, nd, A, y, w.ws.p, U, i, h1, h2, n1, n2, g, nb);
        else
          arnoldi_orth<T, 1>(c, L, nd, A, y, w.ws.p, U, i, h1, h2, n1, n2, g, nb);
        if (i == p.sD) gm_givens_kernel<<<1, kDotThreads, 0, c.s>>>(givens(i, w.flag()));
      } else {
        auto sub = [&](int self, double *h, double *n, const double *s0, const double *s1) {
          arnoldi_sub_kernel<T><<<nb, kDotThreads, 0, c.s>>>(L, nd, pad, A.W, A.wdof, A.c0, y, w.ws.p, U, L, i, self,
                                                             c.part.p, np, h, n, s0, s1, g);
        };
        sub(1, h1, n1, nullptr, nullptr);
        dots2_kernel<T><<<dim3(np, (i + kDotGroup - 1) / kDotGroup), kDotThreads, 0, c.s>>>(
            L, y, U, L, i, c.part.p, h1 + i, n1, nb, arn);
        sub(0, h2, n2, h1 + i, n1);
        gm_givens_kernel<<<1, kDotThreads, 0, c.s>>>(givens(i, w.flag()));
      }
      CR_HIP(hipGetLastError());
      std::swap(v, y);
      // a plain solve looks at the step before while this one runs
      if (w.polled && i > 1) CR_TRY(w.wait(ends && i < p.sD ? w.seq : w.seq - 1, &stop));
      if (stop) break;
    }
    gm_solve_kernel<<<1, 256, 0, c.s>>>(g, p.sD, w.G(w.oH), w.G(w.oerr), w.G(w.oy));
    combine_kernel<T><<<GL, 256, 0, c.s>>>(L, X, X, U, L, 0, g + G_GM_APPLY, w.G(w.oy), 1.0, cyc);
    gm_endcycle_kernel<<<1, 1, 0, c.s>>>(g);
    CR_HIP(hipGetLastError());
    if (w.polled) {
      if (!stop) CR_TRY(w.wait(w.seq, &stop));
      if (stop) break;
    }
  }
  return CRIMSON_OK;
}

// CGRAD / CGRADV / CGRADS (memLS.f90:367-430): op(P, SP, done, nd) computes SP and
// nd parts of P . SP; X holds the right-hand side in and the solution out.
// *state: the state's copy that holds the end.
constexpr int kCgLag = 4;  // iterations a plain solve runs ahead of the flag it has read
template <class T, class Op>
int cg_run(SolveWork<T> &w, size_t L, T *X, Op op, T *R, T *P, T *P2, T *SP, const CgAux<T> &ax, double absTol,
           double relTol, int mItr, double *g, const double *skip, double **state) {
  Ctx<T> &c = w.c;
  CR_TRY(dots(c, L, X, static_cast<const T *>(nullptr), 0, 0, true, c.part.p, skip));
  cg_begin_kernel<<<1, kDotThreads, 0, c.s>>>(c.cgst.p, g, skip, c.part.p, dot_blocks(L), absTol, relTol, mItr);
  CR_TRY(cg_begin_vec(c, L, ax, X, R, P, skip));
  const unsigned long long s0 = w.seq;
  int it = 0;
  // the flag is raised at the top of the iteration after the last one, so a
  // plain solve runs past mItr by its lag at most
  for (; w.polled || it < mItr; ++it) {
    int nd = 0;
    CR_TRY(op(P, SP, c.cgst.p + (it & 1) * kCgState + 5, nd));
    CR_TRY(cg_sweeps(c, L, it, nd, ax, X, R, P, P2, SP, w.flag()));
    std::swap(P, P2);
    bool stop = false;
    if (w.polled && it >= kCgLag) CR_TRY(w.wait(s0 + 1 + it - kCgLag, &stop));
    if (stop) {
      ++it;
      break;
    }
  }
  *state = c.cgst.p + (it & 1) * kCgState;
  return CRIMSON_OK;
}

// cg_run on the formed Schur complement in two launches (s_dir_product_kernel, cg_r_kernel<PAIR>).
template <class T>
int cg_run_paired(SolveWork<T> &w, const SchurOp<T> &o, size_t L, T *X, PairT<T> *Q, T *P, T *SP, const FaceList &fl,
                  double absTol, double relTol, int mItr, double *g, const double *skip, double **state) {
  Ctx<T> &c = w.c;
  CR_TRY(dots(c, L, X, static_cast<const T *>(nullptr), 0, 0, true, c.part.p, skip));
  cg_begin_kernel<<<1, kDotThreads, 0, c.s>>>(c.cgst.p, g, skip, c.part.p, dot_blocks(L), absTol, relTol, mItr);
  cg_pair_kernel<T><<<crimson::grid_for(L, 256), 256, 0, c.s>>>(L, X, Q, skip);
  static_assert(kCgPaired <= kCgWide, "one entry a thread");
  const CgGrid cg = cg_grid(L);
  double *dpart = c.part.p, *rpart = c.part.p + kCgGrid;
  auto st = [&](int it) { return c.cgst.p + (it & 1) * kCgState; };
  const unsigned long long s0 = w.seq;
  int it = 0;
  // the product of iteration it tells whether the solve ended with iteration it - 1,
  // so a plain solve runs past mItr by its lag at most
  for (; w.polled || it < mItr; ++it) {
    int nd = 0;
    CR_TRY(schur_dir_product(c, o, Q, P, SP, it ? st(it - 1) : st(0), it ? st(it) : nullptr, cg.blocks, fl,
                         it ? w.flag() : HostFlag{nullptr, 0}, nd));
    cg_r_kernel<T, 1, true><<<cg.blocks, 256, 0, c.s>>>(L, st(it), dpart, nd, fl, nullptr, SP, rpart, Q, X, P);
    CR_HIP(hipGetLastError());
    bool stop = false;
    if (w.polled && it > kCgLag) CR_TRY(w.wait(s0 + it - kCgLag, &stop));
    if (stop) {
      *state = st(it);
      return CRIMSON_OK;
    }
  }
  if (it > 0) cg_close_kernel<<<1, 256, 0, c.s>>>(st(it - 1), st(it), rpart, cg.blocks);
  CR_HIP(hipGetLastError());
  *state = st(it);
  return CRIMSON_OK;
}

// NSSOLVER (memLS.f90:1460-1759) on d_Ri (4, N), PRECOND's W applied on the
// way in and out.
template <class T>
int ns_run(SolveWork<T> &w, double *d_Ri) {
  Ctx<T> &c = w.c;
  crimson_lhs *l = c.lhs;
  const int N = c.N;
  const size_t mn = (size_t)3 * N, st = (size_t)4 * N;
  double *g = w.gst.p;
  const double *ri = g + G_RI_SKIP;
  const unsigned gN = crimson::grid_for(N, 256), Gmn = crimson::grid_for(mn, 256), Gst = crimson::grid_for(st, 256);
  ns_split_kernel<T><<<gN, 256, 0, c.s>>>(N, d_Ri, c.W.p, w.r0.p, w.r.p);
  CR_TRY(dots(c, st, w.r0.p, static_cast<const T *>(nullptr), 0, 0, true, c.part.p, nullptr));
  ns_begin_kernel<<<1, kDotThreads, 0, c.s>>>(g, c.part.p, dot_blocks(st), w.riAbs, w.riRel);
  // DEPART: views on the 4x4 planes (memLS.f90:1612-1679); Gt = -mG^T
  const T *V = planes(l, T(0));
  const MatView<T> mK = view<T>(c, V, 4, 0, 0, 3, 3, c.W.p, c.fix.p, 4);
  const MatView<T> mG = view<T>(c, V, 4, 0, 3, 3, 1, c.W.p, nullptr, 4);
  const MatView<T> mD = view<T>(c, V, 4, 3, 0, 1, 3, c.W.p, nullptr, 4);
  const MatView<T> mL = view<T>(c, V, 4, 3, 3, 1, 1, c.W.p, c.fix.p, 4);
  MatView<T> Gt = mD;
  if (!l->gt_is_d) {
    crimson::DBuf<T> &gtb = gt_buf(l, T(0));
    gt_kernel<T><<<crimson::grid_for(l->nnz, 256), 256, 0, c.s>>>(l->nnz, V, l->d_tr.p, gtb.p);
    Gt = view<T>(c, gtb.p, 1, 0, 0, 1, 3, c.W.p, nullptr, 4);
    Gt.plane[0] = 0;
    Gt.plane[1] = 1;
    Gt.plane[2] = 2;
    Gt.r0 = 3;
    Gt.c0 = 0;
  }
  // BCPRE (memLS.f90:1683-1716) and the faces' functionals
  if (c.nfc() > 0) face_coef_kernel<<<c.nfc(), 1024, 0, c.s>>>(c.fdev.p, 3, c.fcoef.p);
  CR_TRY(face_functionals(c, mG));
  SchurOp<T> so;
  so.pat = w.spat.get();
  so.S = w.S.p;
  so.L = mL;
  so.Gt = Gt;
  so.G = mG;
  so.Z = w.z.p;
  CR_TRY(schur_form(c, so));
  CgAux<T> ax;
  ax.fl = c.face_list();
  if (!so.pat) {
    ax.W = c.W.p;
    ax.wdof = 4;
    ax.off = mG.c0;
    ax.Ps = so.Ps = w.ps.p;
  }
  // Schur operator of CGRAD: SP = L P - Gt (G P + PRE)
  auto schur_op = [&](const T *Pv, T *SPv, const double *done, int &nd) -> int {
    return schur_apply(c, so, Pv, SPv, done, nd);
  };
  const GmParams gm{w.mGM, w.sD, w.gmAbs, w.gmRel, true, false};
  const int nb = dot_blocks(st);
  const size_t pz = (size_t)kDotGrid * 264;
  for (int i = 1; i <= w.mRI; ++i) {
    const int iB = 2 * i - 1, iBB = 2 * i;
    T *Ui = w.X.p + st * (i - 1), *Pi = Ui + mn;
    T *MUb = w.MX.p + st * (iB - 1), *MPb = MUb + mn, *MUbb = MUb + st, *MPbb = MUbb + mn;
    CR_TRY(w.cut());
    double t0 = now_s();
    CR_TRY(gmres_run(w, mK, 3, w.r.p, Ui, gm, ri));
    double t1 = now_s();
    w.tGM += t1 - t0;
    CR_TRY(w.cut());
    CR_TRY(spmv(c, mD, 1, 3, Ui, Pi, -1.0, w.r.p + mn, 1.0, ri));  // P = Rc - D U
    double *state = nullptr;
    if (w.paired)
      CR_TRY(cg_run_paired(w, so, (size_t)N, Pi, reinterpret_cast<PairT<T> *>(w.t3.p), w.t4.p, MPb, ax.fl, w.cgAbs,
                           w.cgRel, w.mCG, g, ri, &state));
    else
      CR_TRY(cg_run(w, (size_t)N, Pi, schur_op, w.t3.p, w.t4.p, w.t5.p, MPb, ax, w.cgAbs, w.cgRel, w.mCG, g, ri,
                    &state));
    cg_end_kernel<<<1, 1, 0, c.s>>>(state, g, ri);
    t0 = now_s();
    w.tCG += t0 - t1;
    CR_TRY(w.cut());
    CR_TRY(spmv(c, mG, 3, 1, Pi, MUb, 1.0, static_cast<const T *>(nullptr), 0.0, ri));
    diff_kernel<T><<<Gmn, 256, 0, c.s>>>(mn, w.r.p, MUb, MUbb, ri);  // MU(iBB) = Rm - MU(iB)
    CR_TRY(gmres_run(w, mK, 3, MUbb, Ui, gm, ri));
    w.tGM += now_s() - t0;
    CR_TRY(w.cut());
    CR_TRY(spmv(c, mK, 3, 3, Ui, MUbb, 1.0, static_cast<const T *>(nullptr), 0.0, ri));
    CR_TRY(face_apply(c, kFaceAdd, 3, Ui, MUbb, ri));
    CR_TRY(spmv(c, mL, 1, 1, Pi, MPb, 1.0, static_cast<const T *>(nullptr), 0.0, ri));
    CR_TRY(spmv(c, mD, 1, 3, Ui, MPbb, 1.0, static_cast<const T *>(nullptr), 0.0, ri));
    ns_dots_kernel<T><<<dim3(nb, (iBB + kDotGroup - 1) / kDotGroup, 3), kDotThreads, 0, c.s>>>(
        st, w.MX.p, w.r0.p, iB, c.part.p, pz, ri);
    ns_gram_kernel<<<1, kDotThreads, 0, c.s>>>(g, i, w.nB, c.part.p, pz, nb, w.G(w.oA), w.G(w.oBv), w.G(w.oxB),
                                               w.G(w.oC), w.flag());
    CR_HIP(hipGetLastError());
    if (w.polled) {
      bool stop = false;
      CR_TRY(w.wait(w.seq, &stop));
      if (stop) break;
    }
    combine_kernel<T><<<Gst, 256, 0, c.s>>>(st, w.r0.p, w.r.p, w.MX.p, st, iBB, nullptr, w.G(w.oxB), -1.0, ri);
  }
  ns_final_kernel<<<1, 1, 0, c.s>>>(g, w.mRI, w.G(w.oxB), w.G(w.ocu), w.G(w.ocp));
  // the remaining pressure residual's share (Resc)
  const double *err = g + G_ERR;
  combine_kernel<T><<<gN, 256, 0, c.s>>>(N, w.r0.p + mn, w.r.p + mn, w.MX.p + mn, st, 0, g + G_NS_CNT, w.G(w.oxB),
                                         -1.0, err);
  CR_TRY(dots(c, N, w.r.p + mn, static_cast<const T *>(nullptr), 0, 0, true, c.part.p, err));
  ns_rc_kernel<<<1, kDotThreads, 0, c.s>>>(g, c.part.p, dot_blocks(N));
  ns_join_kernel<T><<<gN, 256, 0, c.s>>>(N, w.X.p, g + G_RI_ITR, w.G(w.ocu), w.G(w.ocp), c.W.p, d_Ri, err);
  CR_HIP(hipGetLastError());
  return CRIMSON_OK;
}

// Whether no two coupled faces share a node.
bool faces_disjoint(const crimson_lhs *l) {
  std::vector<int> nodes;
  for (const auto &fa : l->face)
    if (fa.coupled) nodes.insert(nodes.end(), fa.glob.begin(), fa.glob.end());
  std::sort(nodes.begin(), nodes.end());
  return std::adjacent_find(nodes.begin(), nodes.end()) == nodes.end();
}

// The coupled faces of this solve (memLS.f90:1965-1986; res[f] != 0 couples Neumann face
// f) on the device.
template <class T>
int face_setup(Ctx<T> &c, const int *incL, const double *res, bool ns) {
  crimson_lhs *l = c.lhs;
  std::vector<FaceDev> fd;
  int n = 0;
  c.fnodes = 0;
  for (int f = 0; f < l->nFaces; ++f) {
    CrFace &fa = l->face[f];
    fa.inc = !(incL && incL[f] == 0);
    fa.coupled = false;
    if (!fa.inc || !fa.created) continue;
    if (fa.bGrp == CRIMSON_BC_NEU && res && res[f] != 0.0) {
      fa.res = res[f];
      fa.coupled = true;
      ++n;
    }
  }
  CR_TRY(c.fcoef.alloc(std::max(1, n)));
  CR_TRY(c.fsum.alloc(std::max(1, n)));
  for (auto &fa : l->face) {
    if (!fa.coupled) continue;
    CR_TRY(fa.d_valM.alloc((size_t)fa.dof * fa.nNo));
    if (ns) CR_TRY(face_support(l, fa));
    FaceDev d{};
    d.glob = fa.d_glob.p;
    d.valM = fa.d_valM.p;
    d.coefp = c.fcoef.p + fd.size();
    d.res = fa.res;
    d.nNo = fa.nNo;
    d.dof = fa.dof;
    d.sup = ns ? fa.d_sup.p : nullptr;
    d.q = ns ? fa.d_q.p : nullptr;
    d.nsup = ns ? fa.nsup : 0;
    fd.push_back(d);
    c.fnodes += fa.nNo;
  }
  int longest = 0;
  for (const FaceDev &d : fd) longest = std::max(longest, d.nsup);
  c.flb = kFaceDotLog;
  while ((kFaceDotShare << c.flb) < longest && c.flb < kFaceDotMost) ++c.flb;
  CR_TRY(c.fpart.alloc((size_t)std::max(1, n) << c.flb));
  c.disjoint = faces_disjoint(l);
  const bool same = fd.size() == c.hfdev.size() && c.fdev.p &&
                    std::equal(fd.begin(), fd.end(), c.hfdev.begin(), [](const FaceDev &a, const FaceDev &b) {
                      return a.glob == b.glob && a.valM == b.valM && a.coefp == b.coefp && a.res == b.res &&
                             a.nNo == b.nNo && a.dof == b.dof && a.sup == b.sup && a.q == b.q && a.nsup == b.nsup;
                    });
  c.hfdev = fd;
  if (!same && !fd.empty()) {
    CR_TRY(c.fdev.upload(c.hfdev.data(), fd.size(), c.s));
    CR_HIP(hipStreamSynchronize(c.s));
  }
  if (ns) CR_TRY(face_list(c));
  return CRIMSON_OK;
}

// The Schur complement's pattern and storage; spat stays empty when the two
// passes are taken.
template <class T>
int schur_ready(SolveWork<T> &w, crimson_lhs *l) {
  w.spat.reset();
  if (!schur_pays(l, sizeof(T) == 4)) return CRIMSON_OK;
  CR_TRY(schur_pattern(l, w.spat));
  if (w.spat && !try_alloc(w.S, (size_t)w.spat->nnz)) w.spat.reset();
  return CRIMSON_OK;
}

// Workspaces and face set-up of one solve (allocations and uploads: all
// before any capture).
template <class T>
int work_setup(SolveWork<T> &w, crimson_lhs *l, crimson_ls *ls, int dof, const int *incL, const double *res,
               hipStream_t s) {
  Ctx<T> &c = w.c;
  CR_TRY(c.init(l, dof, s));
  const bool ns = ls->LS_type == CRIMSON_LS_NS;
  const size_t N = l->nNo, st = (size_t)dof * N;
  w.mRI = ls->RI.mItr;
  w.mGM = ls->GM.mItr;
  w.mCG = ls->CG.mItr;
  w.sD = ns ? ls->GM.sD : ls->RI.sD;
  w.nB = 2 * w.mRI;
  w.riAbs = ls->RI.absTol;
  w.riRel = ls->RI.relTol;
  w.gmAbs = ls->GM.absTol;
  w.gmRel = ls->GM.relTol;
  w.cgAbs = ls->CG.absTol;
  w.cgRel = ls->CG.relTol;
  CR_TRY(w.r0.alloc(st));
  CR_TRY(w.npart.alloc(2 * kSubGrid));
  CR_TRY(w.h.alloc(512));
  size_t o = G_ARR;
  auto place = [&](size_t &at, size_t n) {
    at = o;
    o += n;
  };
  if (ls->LS_type != CRIMSON_LS_CG) {
    place(w.oH, (size_t)(w.sD + 1) * w.sD);
    place(w.ocs, w.sD);
    place(w.osn, w.sD);
    place(w.oerr, w.sD + 1);
    place(w.oy, w.sD);
    const size_t nd = ns ? 3 : dof;
    CR_TRY(w.wa.alloc(nd * N));
    CR_TRY(w.wb.alloc(nd * N));
    CR_TRY(w.ws.alloc((nd == 3 ? 4 : nd) * N));
    CR_TRY(w.gmU.alloc(nd * N * w.sD));
  }
  if (ns) {
    place(w.oA, (size_t)w.nB * w.nB);
    place(w.oBv, w.nB);
    place(w.oxB, w.nB);
    place(w.oC, (size_t)w.nB * (w.nB + 1));
    place(w.ocu, w.mRI);
    place(w.ocp, w.mRI);
    CR_TRY(w.r.alloc(st));
    CR_TRY(w.X.alloc(st * w.mRI));
    CR_TRY(w.MX.alloc(st * w.nB));
    if (!l->gt_is_d) CR_TRY(gt_buf(l, T(0)).alloc((size_t)3 * l->nnz));
    CR_TRY(schur_ready(w, l));
    w.paired = w.spat && N <= kCgPaired;
    if (!w.spat) {
      CR_TRY(w.ps.alloc(N));
      CR_TRY(w.z.alloc((size_t)4 * N));
    }
  } else {
    CR_TRY(w.X.alloc(st));
  }
  if (ls->LS_type != CRIMSON_LS_GMRES) {
    const size_t n = ns ? N : st;
    CR_TRY(w.t3.alloc(ns && w.paired ? 2 * n : n));
    CR_TRY(w.t4.alloc(n));
    if (!(ns && w.paired)) CR_TRY(w.t5.alloc(n));
  }
  const unsigned long long before = w.gst.serial;
  CR_TRY(w.gst.alloc(o));
  if (w.gst.serial != before) CR_HIP(hipMemsetAsync(w.gst.p, 0, o * sizeof(double), s));
  CR_TRY(face_setup(c, incL, res, ns));
  CR_HIP(hipStreamSynchronize(s));
  return CRIMSON_OK;
}

// PRECOND (memLS.f90:1763-1943) as the W/fix vectors.
template <class T>
int precond(Ctx<T> &c) {
  crimson_lhs *l = c.lhs;
  const int N = c.N, dof = c.dof;
  const unsigned gN = crimson::grid_for(N, 256);
  const T *V = planes(l, T(0));
  precond_diag_kernel<T><<<gN, 256, 0, c.s>>>(N, dof, l->vdof, V, l->nnz, l->d_diag.p, c.W.p, c.fix.p);
  for (auto &fa : l->face)
    if (fa.created && fa.inc && fa.bGrp == CRIMSON_BC_DIR && fa.nNo > 0)
      precond_face_kernel<T><<<crimson::grid_for(fa.nNo, 256), 256, 0, c.s>>>(fa.nNo, dof, fa.dof, fa.d_glob.p,
                                                                              fa.d_val.p, c.W.p);
  precond_fix_kernel<T><<<gN, 256, 0, c.s>>>(N, dof, l->vdof, V, l->nnz, l->d_diag.p, c.W.p, c.fix.p);
  for (auto &fa : l->face)
    if (fa.coupled && fa.nNo > 0)
      face_valm_kernel<T><<<crimson::grid_for(fa.nNo, 256), 256, 0, c.s>>>(fa.nNo, dof, fa.dof, fa.d_glob.p,
                                                                            fa.d_val.p, c.W.p, fa.d_valM.p);
  CR_HIP(hipGetLastError());
  return CRIMSON_OK;
}

// The solve's statistics from a copy of the first G_ARR entries of gst
// into ls's fields, as NSSOLVER leaves them; CRIMSON_ESINGULAR when GE met a
// singular pivot (a plain solve's statistics then reach up to GE, a captured one's are
// untouched).  A GMRES call whose residual is below absTol at once leaves iNorm and
// fNorm as they were (GMRES, memLS.f90:681-788): with no other call in the solve ls
// keeps its own.
int ns_stats(const double *h, crimson_ls *ls, bool plain) {
  const bool singular = h[G_ERR] != 0.0;
  if (singular) crimson::set_error("memLS GE: singular matrix");
  if (singular && !plain) return CRIMSON_ESINGULAR;
  ls->RI.iNorm = h[G_RI_INORM];
  ls->RI.fNorm = h[G_RI_FNORM];
  ls->RI.suc = h[G_RI_SUC] != 0.0;
  ls->RI.callD = 0.0;
  const bool ran = h[G_GM_LASTD] != 0.0;
  if (ran) {
    ls->GM.iNorm = h[G_GM_INORM];
    ls->GM.fNorm = h[G_GM_FNORM];
  }
  ls->GM.itr = (int)h[G_GM_ITR];
  ls->GM.suc = h[G_GM_SUC] != 0.0;
  ls->GM.dB = ran && !(plain && h[G_GM_EARLY] != 0.0) ? 10.0 * std::log(h[G_GM_LASTF] / h[G_GM_LASTD]) : 0.0;
  ls->GM.callD = 0.0;
  ls->CG.iNorm = h[G_CG_INORM];
  ls->CG.fNorm = std::sqrt(h[G_CG_ERR]);
  ls->CG.itr = (int)h[G_CG_ITR];
  ls->CG.suc = h[G_CG_SUC] != 0.0;
  ls->CG.dB = 5.0 * std::log(h[G_CG_ERR] / h[G_CG_ERRO]);
  ls->CG.callD = 0.0;
  if (singular) {
    ls->RI.dB = h[G_RI_DBPRE];
    return CRIMSON_ESINGULAR;
  }
  ls->RI.itr = (int)h[G_RI_ITR];
  ls->RI.dB = 10.0 * std::log(h[G_RI_FNORM] / h[G_RI_DBPRE]);
  const double rcn = std::sqrt(h[G_RC_N2]) / ls->RI.fNorm;
  ls->Resc = (int)std::lround(100.0 * rcn * rcn);
  ls->Resm = 100 - ls->Resc;
  return CRIMSON_OK;
}

// GMRESV (memLS.f90:792-883) and CGRADV/CGRADS on the whole system: W R in
// r0, the solution in X, out as W X.
template <class T>
int gmresv(SolveWork<T> &w, crimson_ls *ls) {
  Ctx<T> &c = w.c;
  const int dof = c.dof;
  const MatView<T> A = view<T>(c, planes(c.lhs, T(0)), dof, 0, 0, dof, dof, c.W.p, c.fix.p, dof);
  double *g = w.gst.p;
  CR_HIP(hipMemsetAsync(g + G_GM_ITR, 0, sizeof(double), c.s));
  CR_TRY(gmres_run(w, A, dof, w.r0.p, w.X.p, GmParams{ls->RI.mItr, w.sD, ls->RI.absTol, ls->RI.relTol, false, true},
                   nullptr));
  double h[G_ARR];
  CR_HIP(hipMemcpyAsync(h, g, sizeof(h), hipMemcpyDeviceToHost, c.s));
  CR_HIP(hipStreamSynchronize(c.s));
  SubLs &r = ls->RI;
  r.suc = h[G_GM_EARLY] == 0.0 && h[G_GM_SUC] != 0.0;
  r.itr = h[G_GM_EARLY] != 0.0 ? 0 : (int)h[G_GM_ITR];
  if (h[G_GM_EARLY] != 0.0) {
    r.iNorm = r.fNorm = h[G_GM_E0];
    r.callD = r.dB = 0.0;
    return CRIMSON_OK;
  }
  r.iNorm = h[G_GM_INORM];
  r.fNorm = h[G_GM_FNORM];
  r.dB = 10.0 * std::log(h[G_GM_FNORM] / h[G_GM_DBPRE]);
  return CRIMSON_OK;
}
template <class T>
int cgradv(SolveWork<T> &w, crimson_ls *ls) {
  Ctx<T> &c = w.c;
  const int dof = c.dof;
  const size_t L = (size_t)dof * c.N;
  const MatView<T> A = view<T>(c, planes(c.lhs, T(0)), dof, 0, 0, dof, dof, c.W.p, c.fix.p, dof);
  copy_kernel<T><<<crimson::grid_for(L, 256), 256, 0, c.s>>>(L, w.r0.p, w.X.p, nullptr);
  auto op = [&](const T *Pv, T *SPv, const double *done, int &nd) -> int {
    CR_TRY(spmv<T>(c, A, dof, dof, Pv, SPv, 1.0, static_cast<const T *>(nullptr), 0.0, done));
    return cg_den(c, L, Pv, SPv, done, nd);
  };
  double *state = nullptr;
  SubLs &r = ls->RI;
  CR_TRY(cg_run(w, L, w.X.p, op, w.t3.p, w.t4.p, w.t5.p, w.r0.p, CgAux<T>(), r.absTol, r.relTol, r.mItr,
                static_cast<double *>(nullptr), static_cast<const double *>(nullptr), &state));
  double h[kCgState];
  CR_HIP(hipMemcpyAsync(h, state, sizeof(h), hipMemcpyDeviceToHost, c.s));
  CR_HIP(hipStreamSynchronize(c.s));
  r.iNorm = h[9];
  r.suc = h[8] != 0.0;
  r.fNorm = std::sqrt(h[0]);
  r.dB = 5.0 * std::log(h[0] / h[1]);
  r.itr = (int)h[6];
  return CRIMSON_OK;
}

// The workspace of a plain solve stays with the matrix handle: allocating and
// freeing it took 5 to 7 ms a solve, a third of the reference case's.  Kept
// while the process keeps at most kKeepBytes of them (a larger one is freed after its
// solve, where the solve is long); a solve takes it out, so that no other thread's
// release_idle_work frees it meanwhile; given back with the handle, or when an
// allocation fails (release_idle_work).  Solves of one handle run one at a time
// (crimson_lhs::busy): they share its faces' buffers and the complement's pattern.
constexpr size_t kKeepBytes = (size_t)8 << 30;
template <class T>
std::unique_ptr<SolveWork<T>> take_work(crimson_lhs *l) {
  std::unique_ptr<crimson::SolveWorkBase> w = crimson::work_take(l, sizeof(T) == 4);
  if (w) return std::unique_ptr<SolveWork<T>>(static_cast<SolveWork<T> *>(w.release()));
  return std::make_unique<SolveWork<T>>();
}

// One memLS_SOLVE in arithmetic type T.  d_Ri is the FP64 (dof,N) right-hand
// side in and solution out; for T = float the solve runs on an FP32 copy.
template <class T>
int solve_run(SolveWork<T> &w, crimson_lhs *l, crimson_ls *ls, int dof, double *d_Ri, const int *incL,
              const double *res) {
  Ctx<T> &c = w.c;
  const double t0 = now_s();
  CR_TRY(work_setup(w, l, ls, dof, incL, res, l->stream));
  CR_TRY(w.poll_ready());
  w.tGM = w.tCG = 0.0;
  CR_TRY(precond(c));
  if (ls->LS_type == CRIMSON_LS_NS) {
    CR_TRY(ns_run(w, d_Ri));
    double h[G_ARR];
    CR_HIP(hipMemcpyAsync(h, w.gst.p, sizeof(h), hipMemcpyDeviceToHost, c.s));
    CR_HIP(hipStreamSynchronize(c.s));
    CR_TRY(ns_stats(h, ls, true));
    ls->RI.callD = now_s() - t0;
    ls->GM.callD = w.tGM;
    ls->CG.callD = w.tCG;
    return CRIMSON_OK;
  }
  const size_t L = (size_t)dof * c.N;
  mul_kernel<double, T, T><<<crimson::grid_for(L, 256), 256, 0, c.s>>>(L, d_Ri, c.W.p, w.r0.p);
  CR_HIP(hipGetLastError());
  if (ls->LS_type == CRIMSON_LS_GMRES)
    CR_TRY(gmresv(w, ls));
  else
    CR_TRY(cgradv(w, ls));
  if (ls->LS_type == CRIMSON_LS_CG || ls->RI.itr > 0) ls->RI.callD = now_s() - t0;
  mul_kernel<T, T, double><<<crimson::grid_for(L, 256), 256, 0, c.s>>>(L, w.X.p, c.W.p, d_Ri);
  CR_HIP(hipGetLastError());
  CR_HIP(hipStreamSynchronize(c.s));
  return CRIMSON_OK;
}
template <class T>
int solve_impl(crimson_lhs *l, crimson_ls *ls, int dof, double *d_Ri, const int *incL, const double *res) {
  std::unique_ptr<SolveWork<T>> w = take_work<T>(l);
  const int rc = solve_run(*w, l, ls, dof, d_Ri, incL, res);
  if (rc) {
    (void)hipStreamSynchronize(l->stream);  // nothing of the workspace is in use when it goes
    return rc;
  }
  crimson::work_keep(l, sizeof(T) == 4, std::move(w), kKeepBytes);
  return CRIMSON_OK;
}

int solve_dev(crimson_lhs *l, crimson_ls *ls, int dof, double *d_Ri, const int *incL, const double *res) {
  if (l->vdof != dof || !(l->prec == 32 ? (const void *)l->d_V32.p : (const void *)l->d_V.p)) {
    crimson::set_error("lhs holds no matrix of block size %d (stored: %d)", dof, l->vdof);
    return CRIMSON_ESTATE;
  }
  if (ls->LS_type == CRIMSON_LS_NS && dof != 4) {
    crimson::set_error("LS_TYPE_NS needs dof = 4 (got %d)", dof);
    return CRIMSON_EUNSUPPORTED;
  }
  if (l->prec == 32) return solve_impl<float>(l, ls, dof, d_Ri, incL, res);
  return solve_impl<double>(l, ls, dof, d_Ri, incL, res);
}

// The device-driven solve of a capture: the limits it can enqueue, then its
// set-up (all allocations and uploads) and its launches.
template <class T>
int ns_graph_setup(SolveWork<T> &w, crimson_lhs *l, crimson_ls *ls, const int *incL, const double *res,
                   hipStream_t s) {
  if (ls->LS_type != CRIMSON_LS_NS) {
    crimson::set_error("the device-driven solve is the NS solver's (LS_TYPE_NS)");
    return CRIMSON_EUNSUPPORTED;
  }
  if (ls->RI.mItr < 1 || ls->GM.mItr < 1 || ls->CG.mItr < 1 || ls->GM.sD < 1 || 2 * ls->RI.mItr > 255 ||
      ls->GM.sD > 255) {
    crimson::set_error("device-driven NS solve: iteration limits out of range (RI %d, GM %d x %d, CG %d)",
                       ls->RI.mItr, ls->GM.mItr, ls->GM.sD, ls->CG.mItr);
    return CRIMSON_EARG;
  }
  return work_setup(w, l, ls, 4, incL, res, s);
}
template <class T>
int ns_graph_enqueue(SolveWork<T> &w, double *d_Ri) {
  CR_TRY(precond(w.c));
  return ns_run(w, d_Ri);
}

// The signature of what a device-driven solve baked in: the matrix and
// face buffers it reads and the solver's settings.
std::vector<unsigned long long> ns_signature(const crimson_lhs *l, const crimson_ls *ls) {
  std::vector<unsigned long long> v = {l->d_V.serial, l->d_V32.serial, l->d_Gt.serial, l->d_Gt32.serial,
                                       (unsigned long long)l->vdof, (unsigned long long)l->prec,
                                       (unsigned long long)l->gt_is_d, (unsigned long long)ls->RI.mItr,
                                       (unsigned long long)ls->GM.mItr, (unsigned long long)ls->GM.sD,
                                       (unsigned long long)ls->CG.mItr};
  for (const auto &fa : l->face) {
    v.push_back(fa.d_glob.serial);
    v.push_back(fa.d_val.serial);
    v.push_back(fa.d_valM.serial);
    v.push_back(fa.d_sup.serial);
    v.push_back(fa.d_q.serial);
    v.push_back((unsigned long long)fa.coupled);
  }
  return v;
}

// A graph holding device-driven solves: the workspaces, and after a replay
// each captured solve's statistics (the last one's into ls).
template <class T>
struct NsGraphExtra : crimson::GraphExtra {
  SolveWork<T> w;
  crimson_lhs *lhs = nullptr;
  crimson_ls *ls = nullptr;
  int nsolve = 0;
  crimson::DBuf<double> stat;  // G_ARR doubles per captured solve
  std::vector<double> hstat;
  // Faces that crimson_bc_create gave other nodes since the capture, in buffers of the
  // same sizes: their supports and the merged list follow, in place (buffers of other
  // sizes change the signature, and the replay is refused).
  int before_launch() override {
    Ctx<T> &c = w.c;
    std::vector<unsigned long long> sig;
    for (auto &fa : lhs->face)
      if (fa.coupled) {
        CR_TRY(face_support(lhs, fa));
        sig.push_back(fa.support);
      }
    if (sig == c.fent_sig || (int)sig.size() != c.nfc()) return CRIMSON_OK;
    if (c.disjoint && !faces_disjoint(lhs)) {
      crimson::set_error("crimson_graph_launch: coupled faces share nodes since the capture; capture it again");
      return CRIMSON_ESTATE;
    }
    return face_list(c);
  }
  int after_launch() override {
    hstat.resize((size_t)G_ARR * nsolve);
    CR_HIP(hipMemcpy(hstat.data(), stat.p, hstat.size() * sizeof(double), hipMemcpyDeviceToHost));
    int rc = CRIMSON_OK;
    for (int k = 0; k < nsolve && rc == CRIMSON_OK; ++k) rc = ns_stats(hstat.data() + (size_t)G_ARR * k, ls, false);
    return rc;
  }
  std::vector<unsigned long long> signature() const override { return ns_signature(lhs, ls); }
  int record_stats(int k) {
    CR_HIP(hipMemcpyAsync(stat.p + (size_t)G_ARR * k, w.gst.p, (size_t)G_ARR * sizeof(double),
                          hipMemcpyDeviceToDevice, w.c.s));
    return CRIMSON_OK;
  }
};

}  // namespace

extern "C" int crimson_ls_create(int lsType, int present, double relTol, double absTol, int maxItr, int dimKry,
                                 const double *relTolIn, const double *absTolIn, const int *maxItrIn,
                                 crimson_ls **out) {
  if (!out) {
    crimson::set_error("crimson_ls_create: null output");
    return CRIMSON_EARG;
  }
  crimson_ls *ls = new crimson_ls();
  ls->LS_type = lsType;
  switch (lsType) {  // memLS.f90:1394-1416
    case CRIMSON_LS_NS:
      ls->RI.relTol = 4e-1;
      ls->GM.relTol = 1e-2;
      ls->CG.relTol = 1e-1;
      ls->RI.mItr = 10;
      ls->GM.mItr = 3;
      ls->CG.mItr = 500;
      ls->GM.sD = 50;
      break;
    case CRIMSON_LS_GMRES:
      ls->RI.relTol = 1e-2;
      ls->RI.mItr = 2;
      ls->RI.sD = 150;
      break;
    case CRIMSON_LS_CG:
      ls->RI.relTol = 1e-4;
      ls->RI.mItr = 1000;
      break;
    default:
      delete ls;
      crimson::set_error("Solver type LS_TYPE %d is not defined", lsType);
      return CRIMSON_EARG;
  }
  ls->RI.absTol = 1e-10;
  ls->GM.absTol = 1e-10;
  ls->CG.absTol = 1e-10;
  if (present & 1) ls->RI.relTol = relTol;
  if (present & 2) ls->RI.absTol = absTol;
  if (present & 4) ls->RI.mItr = maxItr;
  if (present & 8) {
    ls->RI.sD = dimKry;
    ls->GM.sD = dimKry;
  }
  if ((present & 16) && relTolIn) {
    ls->GM.relTol = relTolIn[0];
    ls->CG.relTol = relTolIn[1];
  }
  if ((present & 32) && absTolIn) {
    ls->GM.absTol = absTolIn[0];
    ls->CG.absTol = absTolIn[1];
  }
  if ((present & 64) && maxItrIn) {
    ls->GM.mItr = maxItrIn[0];
    ls->CG.mItr = maxItrIn[1];
  }
  // NS keeps 2*maxItr least-squares columns, each a row of one projection
  // sweep (at most 255 per sweep); GMRES keeps dimKry+1 basis vectors.
  const bool bad_ns = lsType == CRIMSON_LS_NS && (ls->RI.mItr > 127 || ls->GM.sD < 1 || ls->GM.sD > 250);
  const bool bad_gm = lsType == CRIMSON_LS_GMRES && (ls->RI.sD < 1 || ls->RI.sD > 250);
  if (ls->RI.mItr < 1 || bad_ns || bad_gm) {
    crimson::set_error("solver limits out of range (maxItr %d, dimKry %d/%d; supported: maxItr >= 1, "
                       "NS maxItr <= 127, dimKry 1..250)",
                       ls->RI.mItr, ls->RI.sD, ls->GM.sD);
    delete ls;
    return CRIMSON_EUNSUPPORTED;
  }
  *out = ls;
  return CRIMSON_OK;
}

extern "C" int crimson_ls_free(crimson_ls *ls) {
  delete ls;
  return CRIMSON_OK;
}

extern "C" int crimson_lhs_create(int gnNo, int nNo, int nnz, const int *gNodes, const int *rowPtr,
                                  const int *colPtr, int nFaces, crimson_lhs **out) {
  if (!out || !rowPtr || !colPtr || nNo <= 0 || nnz <= 0 || nFaces < 0 || gnNo != nNo) {
    crimson::set_error("crimson_lhs_create: invalid arguments (single task: gnNo must equal nNo)");
    return CRIMSON_EARG;
  }
  if (gNodes)
    for (int a = 0; a < nNo; ++a)
      if (gNodes[a] != a + 1) {
        crimson::set_error("crimson_lhs_create: gNodes must be the identity on one task");
        return CRIMSON_EUNSUPPORTED;
      }
  crimson_lhs *l = new crimson_lhs();
  l->nNo = nNo;
  l->nnz = nnz;
  l->nFaces = nFaces;
  l->face.resize(nFaces);
  l->h_rowptr.resize(nNo + 1);
  l->h_col.resize(nnz);
  l->h_diag.assign(nNo, -1);
  l->h_tr.assign(nnz, -1);
  auto fail = [&](int code) {
    crimson_lhs_free(l);
    return code;
  };
  for (int i = 0; i <= nNo; ++i) l->h_rowptr[i] = rowPtr[i] - 1;
  if (l->h_rowptr[0] != 0 || l->h_rowptr[nNo] != nnz) {
    crimson::set_error("rowPtr must run from 1 to nnz+1");
    return fail(CRIMSON_EARG);
  }
  for (int k = 0; k < nnz; ++k) {
    l->h_col[k] = colPtr[k] - 1;
    if (l->h_col[k] < 0 || l->h_col[k] >= nNo) {
      crimson::set_error("colPtr(%d)=%d out of range", k + 1, colPtr[k]);
      return fail(CRIMSON_EARG);
    }
  }
  for (int i = 0; i < nNo; ++i) {
    if (l->h_rowptr[i + 1] < l->h_rowptr[i]) {
      crimson::set_error("rowPtr not monotone at %d", i + 1);
      return fail(CRIMSON_EARG);
    }
    for (int k = l->h_rowptr[i]; k < l->h_rowptr[i + 1]; ++k) {
      if (l->h_col[k] == i && l->h_diag[i] < 0) l->h_diag[i] = k;
      // transpose position (the DEPART search, memLS.f90:1668-1679, done once)
      const int j = l->h_col[k];
      for (int m = l->h_rowptr[j]; m < l->h_rowptr[j + 1]; ++m)
        if (l->h_col[m] == i) {
          l->h_tr[k] = m;
          break;
        }
    }
    if (l->h_diag[i] < 0) {
      crimson::set_error("row %d has no diagonal block", i + 1);
      return fail(CRIMSON_ENODIAG);
    }
  }
  for (int k = 0; k < nnz; ++k)
    if (l->h_tr[k] < 0) {
      crimson::set_error("CSR graph not symmetric at entry %d", k + 1);
      return fail(CRIMSON_EGRAPH);
    }
  if (hipStreamCreate(&l->stream) != hipSuccess) {
    l->stream = nullptr;
    crimson::set_error("hipStreamCreate failed (is a GPU visible?)");
    return fail(CRIMSON_EHIP);
  }
  if (hipEventCreate(&l->ev0) != hipSuccess || hipEventCreate(&l->ev1) != hipSuccess) {
    crimson::set_error("hipEventCreate failed");
    return fail(CRIMSON_EHIP);
  }
  int rc;
  if ((rc = l->d_rowptr.upload(l->h_rowptr.data(), nNo + 1, l->stream)) ||
      (rc = l->d_col.upload(l->h_col.data(), nnz, l->stream)) ||
      (rc = l->d_diag.upload(l->h_diag.data(), nNo, l->stream)) ||
      (rc = l->d_tr.upload(l->h_tr.data(), nnz, l->stream)))
    return fail(rc);
  {
    std::vector<short> c16(nnz);
    bool fits = true;
    for (int i = 0; i < nNo && fits; ++i)
      for (int k = l->h_rowptr[i]; k < l->h_rowptr[i + 1]; ++k) {
        const int d = l->h_col[k] - i;
        if (d < -32768 || d > 32767) {
          fits = false;
          break;
        }
        l->band = std::max(l->band, std::abs(d));
        c16[k] = (short)d;
      }
    if (fits && (rc = l->d_col16.upload(c16.data(), nnz, l->stream))) return fail(rc);
  }
  if (hipStreamSynchronize(l->stream) != hipSuccess) {
    crimson::set_error("upload of the lhs structure failed");
    return fail(CRIMSON_EHIP);
  }
  *out = l;
  return CRIMSON_OK;
}

extern "C" int crimson_lhs_free(crimson_lhs *l) {
  if (!l) return CRIMSON_OK;
  if (l->stream) (void)hipStreamSynchronize(l->stream);
  if (l->ev0) (void)hipEventDestroy(l->ev0);
  if (l->ev1) (void)hipEventDestroy(l->ev1);
  hipStream_t s = l->stream;
  {
    std::lock_guard<std::mutex> kept(crimson::g_work_lock);
    crimson::work_forget(l);
  }
  delete l;
  if (s) (void)hipStreamDestroy(s);
  return CRIMSON_OK;
}

extern "C" int crimson_bc_create(crimson_lhs *l, int faIn, int nNo, int dof, int bcType, const int *gNodes,
                                 const double *val) {
  if (!l || faIn < 1 || faIn > l->nFaces || nNo < 0 || dof < 1 || (nNo > 0 && !gNodes) ||
      (bcType != CRIMSON_BC_DIR && bcType != CRIMSON_BC_NEU)) {
    crimson::set_error("crimson_bc_create: invalid arguments (faIn=%d of %d)", faIn, l ? l->nFaces : 0);
    return CRIMSON_EARG;
  }
  CrFace &fa = l->face[faIn - 1];
  fa.nNo = nNo;
  fa.dof = dof;
  fa.qpat = false;
  fa.bGrp = bcType;
  fa.res = 0.0;
  fa.created = true;
  fa.glob.resize(nNo);
  for (int a = 0; a < nNo; ++a) {
    fa.glob[a] = gNodes[a] - 1;
    if (fa.glob[a] < 0 || fa.glob[a] >= l->nNo) {
      crimson::set_error("gNodes(%d)=%d out of range", a + 1, gNodes[a]);
      return CRIMSON_EARG;
    }
  }
  fa.val.assign((size_t)dof * nNo, 0.0);
  if (val) std::memcpy(fa.val.data(), val, sizeof(double) * dof * nNo);
  CR_TRY(fa.d_glob.upload(fa.glob.data(), nNo, l->stream));
  CR_TRY(fa.d_val.upload(fa.val.data(), fa.val.size(), l->stream));
  CR_TRY(fa.d_valM.alloc(fa.val.size()));
  CR_HIP(hipStreamSynchronize(l->stream));
  return CRIMSON_OK;
}

extern "C" int crimson_lhs_set_val(crimson_lhs *l, int dof, const double *Val) {
  if (!l || !Val || dof < 1 || dof > 4) {
    crimson::set_error("crimson_lhs_set_val: invalid arguments");
    return CRIMSON_EARG;
  }
  const size_t m = (size_t)dof * dof, nnz = l->nnz;
  crimson::DBuf<double> aos;
  CR_TRY(aos.upload(Val, m * nnz, l->stream));
  CR_TRY(l->d_V.alloc(m * nnz));
  aos_to_planes_kernel<double, double><<<crimson::grid_for(nnz, 256), 256, 0, l->stream>>>(nnz, (int)m, aos.p,
                                                                                            l->d_V.p);
  CR_HIP(hipGetLastError());
  CR_HIP(hipStreamSynchronize(l->stream));
  l->vdof = dof;
  l->prec = 64;
  l->gt_is_d = false;
  return CRIMSON_OK;
}

extern "C" int crimson_lhs_set_precision(crimson_lhs *l, int bits) {
  if (!l || (bits != 32 && bits != 64)) {
    crimson::set_error("crimson_lhs_set_precision: invalid arguments (bits 32 or 64)");
    return CRIMSON_EARG;
  }
  if (bits == l->prec) return CRIMSON_OK;
  const size_t n = (size_t)l->vdof * l->vdof * l->nnz;
  if (l->vdof == 0 || n == 0) {
    crimson::set_error("crimson_lhs_set_precision: no matrix held");
    return CRIMSON_ESTATE;
  }
  const unsigned G = crimson::grid_for(n, 256);
  if (bits == 32) {
    CR_TRY(l->d_V32.alloc(n));
    convert_kernel<double, float><<<G, 256, 0, l->stream>>>(n, l->d_V.p, l->d_V32.p);
  } else {
    CR_TRY(l->d_V.alloc(n));
    convert_kernel<float, double><<<G, 256, 0, l->stream>>>(n, l->d_V32.p, l->d_V.p);
  }
  CR_HIP(hipGetLastError());
  CR_HIP(hipStreamSynchronize(l->stream));
  l->prec = bits;
  return CRIMSON_OK;
}

template <class T>
__global__ void planes_to_aos_kernel(size_t nnz, int m, const T *__restrict__ V, double *__restrict__ aos) {
  const size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nnz) return;
  for (int p = 0; p < m; ++p) aos[(size_t)m * k + p] = (double)V[(size_t)p * nnz + k];
}

extern "C" int crimson_lhs_get_val(crimson_lhs *l, int dof, double *Val) {
  if (!l || !Val || dof != l->vdof || !(l->prec == 32 ? (const void *)l->d_V32.p : (const void *)l->d_V.p)) {
    crimson::set_error("crimson_lhs_get_val: no matrix of block size %d held", dof);
    return CRIMSON_EARG;
  }
  const size_t m = (size_t)dof * dof, nnz = l->nnz;
  crimson::DBuf<double> aos;
  CR_TRY(aos.alloc(m * nnz));
  if (l->prec == 32)
    planes_to_aos_kernel<float><<<crimson::grid_for(nnz, 256), 256, 0, l->stream>>>(nnz, (int)m, l->d_V32.p, aos.p);
  else
    planes_to_aos_kernel<double><<<crimson::grid_for(nnz, 256), 256, 0, l->stream>>>(nnz, (int)m, l->d_V.p, aos.p);
  CR_HIP(hipGetLastError());
  CR_HIP(hipMemcpyAsync(Val, aos.p, m * nnz * sizeof(double), hipMemcpyDeviceToHost, l->stream));
  CR_HIP(hipStreamSynchronize(l->stream));
  return CRIMSON_OK;
}

// Block transpose: block k = (i, j) of dst is block (j, i) of src transposed,
// B'_k(r, c) = B_tr(k)(c, r), every plane of every block.
template <class T>
__global__ void transpose_blocks_kernel(size_t nnz, int m, const int *__restrict__ tr, const T *__restrict__ V,
                                        T *__restrict__ Vt) {
  const size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nnz) return;
  const size_t t = (size_t)tr[k];
  for (int r = 0; r < m; ++r)
    for (int c = 0; c < m; ++c) Vt[(size_t)(r * m + c) * nnz + k] = V[(size_t)(c * m + r) * nnz + t];
}

extern "C" int crimson_lhs_transpose_dev(crimson_lhs *dst, const crimson_lhs *src) {
  if (!dst || !src || dst == src) {
    crimson::set_error("crimson_lhs_transpose_dev: two distinct handles needed");
    return CRIMSON_EARG;
  }
  if (dst->nNo != src->nNo || dst->nnz != src->nnz || dst->h_rowptr != src->h_rowptr || dst->h_col != src->h_col) {
    crimson::set_error("crimson_lhs_transpose_dev: the handles' CSR graphs differ");
    return CRIMSON_EARG;
  }
  const bool f32 = src->prec == 32;
  if (src->vdof < 1 || !(f32 ? (const void *)src->d_V32.p : (const void *)src->d_V.p)) {
    crimson::set_error("crimson_lhs_transpose_dev: src holds no matrix");
    return CRIMSON_ESTATE;
  }
  const int m = src->vdof;
  const size_t nnz = src->nnz, n = (size_t)m * m * nnz;
  CR_HIP(hipStreamSynchronize(src->stream));
  const unsigned G = crimson::grid_for(nnz, 256);
  if (f32) {
    CR_TRY(dst->d_V32.alloc(n));
    transpose_blocks_kernel<float><<<G, 256, 0, dst->stream>>>(nnz, m, dst->d_tr.p, src->d_V32.p, dst->d_V32.p);
  } else {
    CR_TRY(dst->d_V.alloc(n));
    transpose_blocks_kernel<double><<<G, 256, 0, dst->stream>>>(nnz, m, dst->d_tr.p, src->d_V.p, dst->d_V.p);
  }
  CR_HIP(hipGetLastError());
  CR_HIP(hipStreamSynchronize(dst->stream));
  dst->vdof = m;
  dst->prec = src->prec;
  // a formation-produced matrix has D = -G^T blockwise; its transpose keeps
  // that relation (D'_ij = G_ji^T = -D_ij = -G'_ji^T)
  dst->gt_is_d = src->gt_is_d;
  return CRIMSON_OK;
}

extern "C" int crimson_ls_solve_dev(crimson_lhs *l, crimson_ls *ls, int dof, double *d_Ri, const int *incL,
                                    const double *res) {
  if (!l || !ls || !d_Ri) {
    crimson::set_error("crimson_ls_solve_dev: null argument");
    return CRIMSON_EARG;
  }
  std::lock_guard<std::mutex> hold(l->busy);
  return solve_dev(l, ls, dof, d_Ri, incL, res);
}

extern "C" int crimson_ls_solve(crimson_lhs *l, crimson_ls *ls, int dof, double *Ri, const double *Val,
                                const int *incL, const double *res) {
  if (!l || !ls || !Ri || !Val) {
    crimson::set_error("crimson_ls_solve: null argument");
    return CRIMSON_EARG;
  }
  std::lock_guard<std::mutex> hold(l->busy);
  CR_TRY(crimson_lhs_set_val(l, dof, Val));
  crimson::DBuf<double> dR;
  const size_t L = (size_t)dof * l->nNo;
  CR_TRY(dR.upload(Ri, L, l->stream));
  CR_TRY(solve_dev(l, ls, dof, dR.p, incL, res));
  CR_HIP(hipMemcpyAsync(Ri, dR.p, L * sizeof(double), hipMemcpyDeviceToHost, l->stream));
  CR_HIP(hipStreamSynchronize(l->stream));
  return CRIMSON_OK;
}

extern "C" int crimson_ls_stats(const crimson_ls *ls, int sub, double *o) {
  if (!ls || !o || sub < 0 || sub > 2) {
    crimson::set_error("crimson_ls_stats: invalid arguments");
    return CRIMSON_EARG;
  }
  const SubLs &s = sub == 0 ? ls->RI : (sub == 1 ? ls->GM : ls->CG);
  o[0] = s.iNorm;
  o[1] = s.fNorm;
  o[2] = s.itr;
  o[3] = s.suc;
  o[4] = s.dB;
  o[5] = s.callD;
  o[6] = ls->Resm;
  o[7] = ls->Resc;
  return CRIMSON_OK;
}

namespace {
template <class T>
int spmv_timed(crimson_lhs *l, int dof, const T *x, T *y, int reps, double *ms) {
  Ctx<T> c;
  CR_TRY(c.init(l, 4, l->stream));
  const unsigned gN = crimson::grid_for(l->nNo, 256);
  const T *V = planes(l, T(0));
  precond_diag_kernel<T><<<gN, 256, 0, c.s>>>(l->nNo, 4, 4, V, l->nnz, l->d_diag.p, c.W.p, c.fix.p);
  const MatView<T> A = view<T>(c, V, 4, 0, 0, dof, dof, c.W.p, c.fix.p, 4);
  CR_TRY(spmv<T>(c, A, dof, dof, x, y));  // warm-up
  CR_HIP(hipEventRecord(l->ev0, c.s));
  for (int r = 0; r < reps; ++r) CR_TRY(spmv<T>(c, A, dof, dof, x, y));
  CR_HIP(hipEventRecord(l->ev1, c.s));
  CR_HIP(hipEventSynchronize(l->ev1));
  float t = 0.f;
  CR_HIP(hipEventElapsedTime(&t, l->ev0, l->ev1));
  *ms = t / reps;
  return CRIMSON_OK;
}
}  // namespace

extern "C" int crimson_lhs_spmv_dev(crimson_lhs *l, int dof, const double *d_x, double *d_y, int reps, double *ms) {
  if (!l || !d_x || !d_y || reps < 1 || !ms || (dof != 3 && dof != 4) || l->vdof != 4 ||
      !(l->prec == 32 ? (const void *)l->d_V32.p : (const void *)l->d_V.p)) {
    crimson::set_error("crimson_lhs_spmv_dev: invalid arguments (needs a 4x4 matrix, dof 3 or 4)");
    return CRIMSON_EARG;
  }
  if (l->prec == 64) return spmv_timed<double>(l, dof, d_x, d_y, reps, ms);
  // FP32 matrix: the product runs on FP32 copies of x and y
  const size_t L = (size_t)dof * l->nNo;
  crimson::DBuf<float> xf, yf;
  CR_TRY(xf.alloc(L));
  CR_TRY(yf.alloc(L));
  convert_kernel<double, float><<<crimson::grid_for(L, 256), 256, 0, l->stream>>>(L, d_x, xf.p);
  CR_HIP(hipGetLastError());
  CR_TRY(spmv_timed<float>(l, dof, xf.p, yf.p, reps, ms));
  convert_kernel<float, double><<<crimson::grid_for(L, 256), 256, 0, l->stream>>>(L, yf.p, d_y);
  CR_HIP(hipGetLastError());
  CR_HIP(hipStreamSynchronize(l->stream));
  return CRIMSON_OK;
}

namespace {
// Launches per captured segment at most: a device-driven solve enqueues
// every possible iteration, so its launch count grows with its iteration
// limits; the capture is cut into segments (each GMRES call, each CG call,
// the glue between them) and a configuration whose segment would exceed
// this is refused before it is captured.
constexpr size_t kMaxSegmentLaunches = 40000;

// A stream capture cut into segments (crimson_graph::seg), each
// instantiated on its own and launched back to back.
struct SegCapture {
  crimson_graph *g;
  hipStream_t s;
  bool open = false;
  int begin() {
    if (hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal) != hipSuccess) {
      crimson::set_error("hipStreamBeginCapture failed");
      return CRIMSON_EHIP;
    }
    open = true;
    return CRIMSON_OK;
  }
  int close() {
    hipGraph_t gr = nullptr;
    const hipError_t ec = hipStreamEndCapture(s, &gr);
    open = false;
    if (ec != hipSuccess || !gr) {
      crimson::set_error("capture into a HIP graph failed");
      return CRIMSON_EHIP;
    }
    size_t n = 0;
    if (hipGraphGetNodes(gr, nullptr, &n) != hipSuccess) {
      (void)hipGraphDestroy(gr);
      crimson::set_error("hipGraphGetNodes failed");
      return CRIMSON_EHIP;
    }
    if (n == 0) {
      (void)hipGraphDestroy(gr);
      return CRIMSON_OK;
    }
    g->seg.push_back(gr);
    hipGraphExec_t x = nullptr;
    if (hipGraphInstantiate(&x, gr, nullptr, nullptr, 0) != hipSuccess) {
      crimson::set_error("hipGraphInstantiate failed");
      return CRIMSON_EHIP;
    }
    g->segx.push_back(x);
    return CRIMSON_OK;
  }
  int cut() {
    CR_TRY(close());
    return begin();
  }
  void abort() {
    if (!open) return;
    hipGraph_t gr = nullptr;
    (void)hipStreamEndCapture(s, &gr);
    if (gr) (void)hipGraphDestroy(gr);
    open = false;
  }
};

// An upper bound of the launches one segment of a device-driven solve holds, from the
// solver's limits, checked before capturing: 16 launches an Arnoldi step and 4 more per
// coupled face that is not batched, 8 a CG iteration and one per such face.  (Five to
// seven a step, and two to five an iteration, are enqueued, 2 more per face a step where
// the faces share many nodes; the bound keeps what a capture may ask for where it was.)
int check_segment_budget(int mGM, int sD, int mCG, int nfc_launch) {
  const size_t gm = (size_t)mGM * ((size_t)sD * (16 + 4 * nfc_launch) + 16);
  const size_t cg = (size_t)mCG * (8 + nfc_launch) + 8;
  if (gm > kMaxSegmentLaunches || cg > kMaxSegmentLaunches) {
    crimson::set_error("device-driven NS solve: a GMRES call of %d cycles x %d steps (up to %zu launches) or a CG call "
                       "of %d iterations (up to %zu launches) exceeds the %zu launches a captured segment may hold",
                       mGM, sD, gm, mCG, cg, kMaxSegmentLaunches);
    return CRIMSON_EUNSUPPORTED;
  }
  return CRIMSON_OK;
}

int seg_cut(SegCapture *cap) { return cap ? cap->cut() : CRIMSON_OK; }

template <class T>
int capture_into(crimson_graph *g, hipStream_t s, SolveWork<T> &w, const std::function<int()> &body) {
  SegCapture cap{g, s};
  const int nfc = w.c.nfc();
  CR_TRY(check_segment_budget(w.mGM, w.sD, w.mCG, (w.c.disjoint && nfc > 1) ? 1 : nfc));
  CR_TRY(cap.begin());
  w.cap = &cap;
  int rc = body();
  if (!rc) rc = cap.close();
  w.cap = nullptr;
  if (rc) cap.abort();
  g->s = s;
  return rc;
}

void graph_discard(crimson_graph *g) {
  if (g->exec) (void)hipGraphExecDestroy(g->exec);
  if (g->g) (void)hipGraphDestroy(g->g);
  for (hipGraphExec_t x : g->segx) (void)hipGraphExecDestroy(x);
  for (hipGraph_t h : g->seg) (void)hipGraphDestroy(h);
  delete g->extra;
  delete g;
}

template <class T>
int ls_graph_create_t(crimson_lhs *l, crimson_ls *ls, double *d_Ri, const int *incL, const double *res,
                      crimson_graph **out) {
  crimson_graph *g = new crimson_graph();
  auto *ex = new NsGraphExtra<T>();
  g->extra = ex;
  ex->lhs = l;
  ex->ls = ls;
  ex->nsolve = 1;
  int rc = ns_graph_setup<T>(ex->w, l, ls, incL, res, l->stream);
  if (!rc) rc = ex->stat.alloc(G_ARR);
  if (!rc)
    rc = capture_into<T>(g, l->stream, ex->w, [&]() -> int {
      CR_TRY(ns_graph_enqueue<T>(ex->w, d_Ri));
      return ex->record_stats(0);
    });
  if (rc) {
    graph_discard(g);
    return rc;
  }
  g->lhs = l;
  g->sig = ex->signature();
  *out = g;
  return CRIMSON_OK;
}

template <class T>
int step_graph_create_t(crimson_form *f, crimson_lhs *l, crimson_ls *ls, double *d_yold, double *d_acold,
                        double *d_y, double *d_ac, double *d_ya, double *d_aca, const double *d_x, double *d_Res4,
                        const int *d_iBC, const double *d_BC, int ndofBC, int nsurf, const int *surf_ptr,
                        const int *d_glob, const double *d_nabi, const double *c1, const double *c2, double *d_q,
                        const double *faceRes, int nonlinear, crimson_graph **out) {
  crimson_graph *g = new crimson_graph();
  auto *ex = new NsGraphExtra<T>();
  g->extra = ex;
  ex->lhs = l;
  ex->ls = ls;
  ex->nsolve = nonlinear;
  hipStream_t s = crimson::form_stream(f);
  const int N = crimson::form_nshg(f);
  int rc = crimson::form_prepare_to_lhs(f, d_x, l);
  if (!rc) rc = ns_graph_setup<T>(ex->w, l, ls, nullptr, faceRes, s);
  if (!rc) rc = ex->stat.alloc((size_t)G_ARR * nonlinear);
  const crimson_form_params prm = crimson::form_params_of(f);
  if (!rc)
    rc = capture_into<T>(g, s, ex->w, [&]() -> int {
      CR_TRY(crimson_itr_predict_dev(f, d_yold, d_acold, d_y, d_ac, prm.gami));
      CR_TRY(crimson::form_wall_enqueue_predict(f, d_yold, d_acold));
      CR_TRY(crimson_itr_bc_dev(f, d_iBC, d_BC, ndofBC, d_y));
      for (int k = 0; k < nonlinear; ++k) {
        CR_TRY(crimson::form_wall_enqueue_alpha(f));
        CR_TRY(crimson_itr_yalpha_dev(f, d_yold, d_acold, d_y, d_ac, d_ya, d_aca, prm.alfi, prm.almi));
        CR_TRY(crimson::form_enqueue_to_lhs(f, d_ya, d_aca, d_x, d_Res4, l));
        // ElmpvsQ, then bc3Res (elmgmr.f90:528-555)
        for (int q = 0; q < nsurf; ++q)
          CR_TRY(crimson_elmpvsq_coef_dev(f, surf_ptr[q + 1] - surf_ptr[q], d_glob + surf_ptr[q],
                                          d_nabi + (size_t)3 * surf_ptr[q], c1[q], c2[q], d_ya, d_Res4, d_q + q));
        CR_TRY(crimson::form_enqueue_bc3res(f, d_Res4, 1));
        CR_TRY(ns_graph_enqueue<T>(ex->w, d_Res4));
        CR_TRY(ex->record_stats(k));
        CR_TRY(crimson_itr_correct_dev(f, d_y, d_ac, d_Res4, prm.gami, prm.alfi, prm.Delt));
        CR_TRY(crimson::form_wall_enqueue_correct(f, d_Res4));
        CR_TRY(crimson_itr_bc_dev(f, d_iBC, d_BC, ndofBC, d_y));
      }
      CR_HIP(hipMemcpyAsync(d_yold, d_y, (size_t)4 * N * sizeof(double), hipMemcpyDeviceToDevice, s));
      CR_HIP(hipMemcpyAsync(d_acold, d_ac, (size_t)4 * N * sizeof(double), hipMemcpyDeviceToDevice, s));
      CR_TRY(crimson::form_wall_enqueue_update(f));
      return CRIMSON_OK;
    });
  if (rc) {
    graph_discard(g);
    return rc;
  }
  g->f = f;
  g->lhs = l;
  g->sig = crimson::graph_signature(f, l);
  const std::vector<unsigned long long> e = ex->signature();
  g->sig.insert(g->sig.end(), e.begin(), e.end());
  *out = g;
  return CRIMSON_OK;
}
}  // namespace

extern "C" int crimson_ls_graph_create(crimson_lhs *lhs, crimson_ls *ls, int dof, double *d_Ri, const int *incL,
                                       const double *res, crimson_graph **out) {
  if (!lhs || !ls || !d_Ri || !out || dof != 4) {
    crimson::set_error("crimson_ls_graph_create: invalid arguments (the NS solver, dof 4)");
    return CRIMSON_EARG;
  }
  std::lock_guard<std::mutex> hold(lhs->busy);
  if (lhs->vdof != 4 || !(lhs->prec == 32 ? (const void *)lhs->d_V32.p : (const void *)lhs->d_V.p)) {
    crimson::set_error("crimson_ls_graph_create: lhs holds no 4x4 matrix");
    return CRIMSON_ESTATE;
  }
  if (lhs->prec == 32) return ls_graph_create_t<float>(lhs, ls, d_Ri, incL, res, out);
  return ls_graph_create_t<double>(lhs, ls, d_Ri, incL, res, out);
}

extern "C" int crimson_step_graph_create(crimson_form *f, crimson_lhs *lhs, crimson_ls *ls, double *d_yold,
                                         double *d_acold, double *d_y, double *d_ac, double *d_yAlpha,
                                         double *d_acAlpha, const double *d_x, double *d_Res4, const int *d_iBC,
                                         const double *d_BC, int ndofBC, int nsurf, const int *surf_ptr,
                                         const int *d_glob, const double *d_nabi, const double *c1,
                                         const double *c2, double *d_q, const double *faceRes, int nonlinear,
                                         crimson_graph **out) {
  if (!f || !lhs || !ls || !d_yold || !d_acold || !d_y || !d_ac || !d_yAlpha || !d_acAlpha || !d_x || !d_Res4 ||
      !d_iBC || !d_BC || ndofBC < 6 || nsurf < 0 || (nsurf > 0 && (!surf_ptr || !d_glob || !d_nabi || !c1 || !c2 ||
                                                                    !d_q)) ||
      nonlinear < 1 || !out) {
    crimson::set_error("crimson_step_graph_create: invalid arguments");
    return CRIMSON_EARG;
  }
  CR_TRY(crimson::form_wall_step_ready(f));
  for (int q = 0; q < nsurf; ++q)
    if (surf_ptr[q + 1] < surf_ptr[q]) {
      crimson::set_error("crimson_step_graph_create: surf_ptr not monotone");
      return CRIMSON_EARG;
    }
  std::lock_guard<std::mutex> hold(lhs->busy);
  if (crimson::form_params_of(f).precision == 32)
    return step_graph_create_t<float>(f, lhs, ls, d_yold, d_acold, d_y, d_ac, d_yAlpha, d_acAlpha, d_x, d_Res4,
                                      d_iBC, d_BC, ndofBC, nsurf, surf_ptr, d_glob, d_nabi, c1, c2, d_q, faceRes,
                                      nonlinear, out);
  return step_graph_create_t<double>(f, lhs, ls, d_yold, d_acold, d_y, d_ac, d_yAlpha, d_acAlpha, d_x, d_Res4,
                                     d_iBC, d_BC, ndofBC, nsurf, surf_ptr, d_glob, d_nabi, c1, c2, d_q, faceRes,
                                     nonlinear, out);
}
