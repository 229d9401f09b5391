// Device helpers shared by the single-problem and the batched Krylov
// kernels: launch constants, reductions, the solver argument block, SELL-64
// row sums and the Givens rotation (drotg semantics of netlib BLAS, as
// called by lss_mkb_core.c:2539-2560).
#pragma once

#include <hip/hip_runtime.h>

#include "mf_device.h"

namespace mf {

constexpr int SB = 256;         // threads per solver block
constexpr int TILE_NNZ = 4096;  // CRS entries staged per tile (32 KB LDS)
constexpr int MAX_BLOCKS = 4096;
constexpr int MAX_NV = 64;
constexpr int OPB = 512;        // threads per block of the operator + dots kernels

// ---------------------------------------------------------------------
// device helpers
// ---------------------------------------------------------------------
// blocks are dispatched round-robin over the 8 XCDs; give XCD x the x-th
// contiguous range of logical blocks so its L2 sees neighbouring rows
__device__ __forceinline__ int xcd_block(int bid, int nb) {
  int xcd = bid & 7, k = bid >> 3;
  int per = nb >> 3, rem = nb & 7;
  return xcd * per + min(xcd, rem) + k;
}

// the same ranges, taken from their ends backwards
__device__ __forceinline__ int xcd_block_rev(int bid, int nb) {
  const int xcd = bid & 7, k = bid >> 3;
  const int per = nb >> 3, rem = nb & 7;
  return xcd * per + min(xcd, rem) + per + (xcd < rem ? 1 : 0) - 1 - k;
}

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// sum NV per-thread values over the block; results in red[0..nact-1]
template <int NV>
__device__ __forceinline__ void block_sum_multi(const double* acc, int nact, double* red) {
  __shared__ double wsum[SB / 64][NV];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
  for (int i = 0; i < NV; i++) {
    if (i < nact) {
      double v = wave_sum(acc[i]);
      if (lane == 0) wsum[wid][i] = v;
    }
  }
  __syncthreads();
  if ((int)threadIdx.x < nact) {
    double s = 0;
#pragma unroll
    for (int w = 0; w < SB / 64; w++) s += wsum[w][threadIdx.x];
    red[threadIdx.x] = s;
  }
  __syncthreads();
}

// sum of one value per thread over a block of up to OPB threads, the same in
// every thread; the same number of threads gives the same rounding
__device__ __forceinline__ double block_sum_all(double v) {
  __shared__ double wsum[OPB / 64];
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = v;
  __syncthreads();
  double s = 0.0;
  for (int w = 0; w < (int)(blockDim.x >> 6); w++) s += wsum[w];
  return s;
}

struct SolveArgs {
  int n, ntiles, m;
  long long ldv;        // stride of the Krylov vectors
  const int* tile_row;  // CRS-tile path (storage seam)
  const int* row_ptr;
  const int* col;
  const double* val;    // CRS values (tile path) or SELL-64 values
  const float* val32;   // SELL-64 values rounded to FP32 (mixed-precision inner solves)
  int op32;             // 1: the operator kernels read val32
  // 16-bit columns relative to a per-slice base where the slice's columns
  // span less than 65536 rows (null, or sbase[sl] < 0: use scol)
  const uint16_t* scol16;
  const int* sbase;
  const long long* sl_ptr;  // SELL-64 path
  const int* scol;
  const double* dinv;   // null: no preconditioner
  const double* b;
  double* x;
  double* V;            // (m+1) x ldv
  double* H;            // (m+1)^2 | givens 2(m+1) | scale (m+1) | coef (m+1)
  double* partials;     // dot products V_i . w: [i][block]
  double* norms;        // ||w||^2 of an update: [block]
  GmresStat* stat;
  GmresStat* hstat;     // pinned host mirror
  // mixed-precision inner solves: the Krylov basis and the Jacobi inverses
  // are FP32 (Vf is the storage of V read with a stride of ldv floats);
  // sums, dot products, Hessenberg data and the iterate stay FP64
  float* Vf;
  const float* dinv32;
  int v32;
  int ilu;              // batched solves: the member applies ILU(0) factors
};

template <typename VT> __device__ __forceinline__ VT* basis(const SolveArgs& A);
template <> __device__ __forceinline__ double* basis<double>(const SolveArgs& A) { return A.V; }
template <> __device__ __forceinline__ float* basis<float>(const SolveArgs& A) { return A.Vf; }

// v scaled by the Jacobi inverse of row r, when there is one
__device__ __forceinline__ double jacobi(const SolveArgs& A, long long r, double v) {
  if (A.dinv) return v * A.dinv[r];
  if (A.dinv32) return v * (double)A.dinv32[r];
  return v;
}

__device__ __forceinline__ double* Hcol(const SolveArgs& A, int c) { return A.H + (size_t)(A.m + 1) * c; }
__device__ __forceinline__ double* Giv(const SolveArgs& A) { return A.H + (size_t)(A.m + 1) * (A.m + 1); }
__device__ __forceinline__ double* Scale(const SolveArgs& A) { return Giv(A) + 2 * (A.m + 1); }
__device__ __forceinline__ double* Coef(const SolveArgs& A) { return Scale(A) + (A.m + 1); }

// tile range of a logical block
__device__ __forceinline__ void tile_range(const SolveArgs& A, int lb, int& t0, int& t1) {
  t0 = (int)((long long)lb * A.ntiles / gridDim.x);
  t1 = (int)((long long)(lb + 1) * A.ntiles / gridDim.x);
}

// stream one tile's CRS entries into LDS products and return the row sum of
// the calling lane's row (valid when r0 + threadIdx.x < r1)
__device__ __forceinline__ double tile_rows(const SolveArgs& A, const double* x, int r0, int r1,
                                            double* prod) {
  const int k0 = A.row_ptr[r0], k1 = A.row_ptr[r1];
#pragma unroll 4
  for (int k = k0 + threadIdx.x; k < k1; k += SB) prod[k - k0] = A.val[k] * x[A.col[k]];
  __syncthreads();
  double s = 0.0;
  const int r = r0 + threadIdx.x;
  if (r < r1) {
    const int a = A.row_ptr[r] - k0, z = A.row_ptr[r + 1] - k0;
    for (int k = a; k < z; k++) s += prod[k];
  }
  __syncthreads();
  return s;
}

// SELL-64: wavefront = slice of 64 rows, lane = row; entries column-major
// inside the slice, so every load of values and columns is one contiguous
// 512/256-byte access.  Logical block lb owns a contiguous range of slices
// (one contiguous eighth of the matrix per XCD); its 4 wavefronts take the
// range's slices round-robin.
constexpr int SW = SB / 64;  // wavefronts per block

__device__ __forceinline__ void slice_range(int nsl, int lb, int& s0, int& s1) {
  s0 = (int)((long long)lb * nsl / gridDim.x);
  s1 = (int)((long long)(lb + 1) * nsl / gridDim.x);
}

// The slices of one operator block: XCD x owns the x-th contiguous part of
// the slices and its blocks take steps of W consecutive slices (one per
// wavefront) cyclically, so each XCD sweeps one contiguous window of
// the matrix at a time (measured 3% faster than a contiguous range per block,
// which leaves ~2k streams open at scattered addresses).
struct SliceSet {
  int base, step, end;
  // the slices of wavefront w: first(w), first(w) + step, ... < end
  __device__ __forceinline__ int first(int w) const { return base + w; }
};

// block bid of G blocks of W wavefronts
__device__ __forceinline__ SliceSet block_slices(int nsl, int bid, int G, int W) {
  SliceSet S;
  const int nx = G < 8 ? G : 8;
  const int x = bid % nx, q = bid / nx;
  const int nq = G / nx + (x < G % nx ? 1 : 0);
  const int r0 = (int)((long long)x * nsl / nx), r1 = (int)((long long)(x + 1) * nsl / nx);
  S.base = r0 + q * W;
  S.step = nq * W;
  S.end = r1;
  return S;
}

// row sum of the calling lane's row.  The slice is the wavefront's, so its
// offsets and its smallest column are scalars and a lane's addresses are one
// 32-bit offset each; CH entries of the row are in flight while the CH before
// them are gathered and summed (the first chunk costs two dependent trips to
// memory, every further one a single trip).  Loads past the slice's length
// repeat its last entry and their products are dropped by a select, so no
// load waits for a branch.
template <typename VT, int CH, typename CT>
__device__ __forceinline__ void sell_chunk(const VT* val, const CT* col, int k0, int len, int lane,
                                           int (&c)[CH], VT (&v)[CH]) {
#pragma unroll
  for (int k = 0; k < CH; k++) {
    const int q = 64 * min(k0 + k, len - 1);
    c[k] = (int)col[q + lane];
    v[k] = val[q + lane];
  }
}

template <typename VT, typename XT, int CH, typename CT>
__device__ __forceinline__ double sell_row_cols(const VT* val, const CT* col, const XT* x, int len,
                                                int lane) {
  double s = 0.0;
  int c[CH];
  VT v[CH];
  if (len > 0) sell_chunk<VT, CH>(val, col, 0, len, lane, c, v);
  for (int k0 = 0; k0 < len; k0 += CH) {
    XT xv[CH];
#pragma unroll
    for (int k = 0; k < CH; k++) xv[k] = x[(unsigned)c[k]];
    VT w[CH];
#pragma unroll
    for (int k = 0; k < CH; k++) w[k] = v[k];
    if (k0 + CH < len) sell_chunk<VT, CH>(val, col, k0 + CH, len, lane, c, v);
#pragma unroll
    for (int k = 0; k < CH; k++) {
      const double t = (double)w[k] * (double)xv[k];
      s += k0 + k < len ? t : 0.0;
    }
  }
  return s;
}

constexpr int kSellChunk = 8;

template <typename VT, typename XT, int CH = kSellChunk>
__device__ __forceinline__ double sell_row(const SolveArgs& A, const VT* val, const XT* x,
                                           int sl, int lane) {
  sl = __builtin_amdgcn_readfirstlane(sl);
  const long long base = A.sl_ptr[sl];
  const int len = (int)((A.sl_ptr[sl + 1] - base) >> 6);
  // 16-bit columns where the slice has them
  const int cb = A.sbase ? A.sbase[sl] : -1;
  if (cb >= 0)
    return sell_row_cols<VT, XT, CH>(val + base, A.scol16 + base, x + cb, len, lane);
  return sell_row_cols<VT, XT, CH>(val + base, A.scol + base, x, len, lane);
}

// the same row sum for a wavefront that has a single slice: a launch of one
// round is bound by its chain of dependent loads, so up to kSellWide entries
// are requested at once (two trips to memory for a row of a box mesh instead
// of four); groups of four past the slice's length are skipped by a
// wave-uniform test.  before(): loads to issue behind the first columns and
// values (len >= 1: every row of a problem has its diagonal entry)
constexpr int kSellWide = 28;

template <typename VT, typename XT, typename CT, class Before>
__device__ __forceinline__ double sell_row_one_cols(const VT* val, const CT* col, const XT* x,
                                                    int len, int lane, Before before) {
  double s = 0.0;
  for (int k0 = 0; k0 < len; k0 += kSellWide) {
    int c[kSellWide];
    VT v[kSellWide];
    XT xv[kSellWide];
#pragma unroll
    for (int g = 0; g < kSellWide; g += 4)
      if (k0 + g < len)
#pragma unroll
        for (int k = g; k < g + 4; k++) {
          const int q = 64 * min(k0 + k, len - 1);
          c[k] = (int)col[q + lane];
          v[k] = val[q + lane];
        }
    if (k0 == 0) before();
#pragma unroll
    for (int g = 0; g < kSellWide; g += 4)
      if (k0 + g < len)
#pragma unroll
        for (int k = g; k < g + 4; k++) xv[k] = x[(unsigned)c[k]];
#pragma unroll
    for (int g = 0; g < kSellWide; g += 4)
      if (k0 + g < len)
#pragma unroll
        for (int k = g; k < g + 4; k++) {
          const double t = (double)v[k] * (double)xv[k];
          s += k0 + k < len ? t : 0.0;
        }
  }
  return s;
}

template <typename VT, typename XT, class Before>
__device__ __forceinline__ double sell_row_one(const SolveArgs& A, const VT* val, const XT* x,
                                               int sl, int lane, Before before) {
  sl = __builtin_amdgcn_readfirstlane(sl);
  const long long base = A.sl_ptr[sl];
  const int len = (int)((A.sl_ptr[sl + 1] - base) >> 6);
  const int cb = A.sbase ? A.sbase[sl] : -1;
  if (cb >= 0)
    return sell_row_one_cols(val + base, A.scol16 + base, x + cb, len, lane, before);
  return sell_row_one_cols(val + base, A.scol + base, x, len, lane, before);
}

// ---------------------------------------------------------------------
// Gram-Schmidt dot products V_i . w of a 64-row slice on the matrix cores:
// v_mfma_f64_4x4x4 multiplies four 4 x 4 by 4 x 4 blocks; lane l holds row l % 4
// (the vector) and, in block (l / 4) % 4, column l / 16 (the matrix row) of
// the left operand, and the same place of the right one.  With V_{4q + l % 4}
// and w at the rows of slot l / 4 in lane l, one instruction adds 16 rows of
// four dot products to the accumulator, and nothing is exchanged between
// lanes until the block's rows are done (dots_finish).  One wave-wide sum per
// vector (six exchanges) made the dots half of a step on small systems.
// ---------------------------------------------------------------------
// entries of a vector at the rows of the lane's slot: FP64 rows 2s, 2s + 1
// and 32 + 2s, 33 + 2s; FP32 rows 4s .. 4s + 3 (16-byte loads)
__device__ __forceinline__ void slot_rows(const double* v, int slot, double (&r)[4]) {
  const double2 a = *reinterpret_cast<const double2*>(v + 2 * slot);
  const double2 b = *reinterpret_cast<const double2*>(v + 32 + 2 * slot);
  r[0] = a.x; r[1] = a.y; r[2] = b.x; r[3] = b.y;
}
__device__ __forceinline__ void slot_rows(const float* v, int slot, double (&r)[4]) {
  const float4 a = *reinterpret_cast<const float4*>(v + 4 * slot);
  r[0] = a.x; r[1] = a.y; r[2] = a.z; r[3] = a.w;
}
// the same rows of a wave's 64 FP64 values staged in LDS
template <typename VT>
__device__ __forceinline__ void slot_rows_lds(const double* v, int slot, double (&r)[4]) {
  const int a = sizeof(VT) == 8 ? 2 * slot : 4 * slot, b = sizeof(VT) == 8 ? 32 + 2 * slot : a + 2;
  const double2 x = *reinterpret_cast<const double2*>(v + a);
  const double2 y = *reinterpret_cast<const double2*>(v + b);
  r[0] = x.x; r[1] = x.y; r[2] = y.x; r[3] = y.y;
}

// acc[q] += V_{4q + lane % 4} . w over a slice's 64 rows for the vectors i <=
// j; V points at the slice's first row of V_0.  NQ quads cover j + 1 vectors
// (the launch picks the next of kDotQuads); vectors past j repeat the last
// ones and their sums are not used.  A quad's address is a scalar plus the
// lane's offset.
template <int N, typename VT>
__device__ __forceinline__ void dots_load(const VT* V, long long ldv, int j, int lane, int g,
                                          double (&v)[N][4]) {
  const int jq = j >> 2;  // the last quad with a vector <= j
  const long long off = (lane & 3) * ldv, last = min(lane & 3, j & 3) * ldv;
#pragma unroll
  for (int q = 0; q < N; q++)
    slot_rows(V + 4LL * min(g + q, jq) * ldv + (g + q < jq ? off : last), lane >> 2, v[q]);
}
template <int N>
__device__ __forceinline__ void dots_add(const double (&v)[N][4], const double (&w)[4],
                                         double* acc) {
#pragma unroll
  for (int k = 0; k < 4; k++)
#pragma unroll
    for (int q = 0; q < N; q++)
      acc[q] = __builtin_amdgcn_mfma_f64_4x4x4f64(v[q][k], w[k], acc[q], 0, 0, 0);
}
// quads [G, NQ), four in flight together
template <int G, int NQ, typename VT>
__device__ __forceinline__ void dots_slice(const VT* V, long long ldv, int j, int lane,
                                           const double (&w)[4], double (&acc)[NQ]) {
  if constexpr (G < NQ) {
    constexpr int N = NQ - G < 4 ? NQ - G : 4;
    double v[N][4];
    dots_load<N>(V, ldv, j, lane, G, v);
    dots_add<N>(v, w, acc + G);
    dots_slice<G + N, NQ>(V, ldv, j, lane, w, acc);
  }
}

// the block's sums to partials[i * G + pb]: lane 16 i + 4 b holds vector i of
// block b of every quad
template <int NQ>
__device__ __forceinline__ void dots_finish(const double (&acc)[NQ], int j, int G, int pb,
                                            double* partials) {
  __shared__ double red[OPB / 64][MAX_NV];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, nw = blockDim.x >> 6;
#pragma unroll
  for (int q = 0; q < NQ; q++) {
    double d = acc[q];
    d += __shfl_xor(d, 4, 64);
    d += __shfl_xor(d, 8, 64);
    if ((lane & 15) == 0) red[wv][4 * q + (lane >> 4)] = d;
  }
  __syncthreads();
  if ((int)threadIdx.x <= j) {
    double s = 0.0;
    for (int w = 0; w < nw; w++) s += red[w][threadIdx.x];
    partials[(size_t)threadIdx.x * G + pb] = s;
  }
}

template <typename XT, class Before>
__device__ __forceinline__ double sell_row_one_op(const SolveArgs& A, const XT* x, int sl, int lane,
                                                  Before before) {
  return A.op32 ? sell_row_one(A, A.val32, x, sl, lane, before)
                : sell_row_one(A, A.val, x, sl, lane, before);
}

// row sum with the FP64 or the FP32 copy of the values (accumulated in FP64)
template <typename XT>
__device__ __forceinline__ double sell_row_op(const SolveArgs& A, const XT* x, int sl, int lane) {
  return A.op32 ? sell_row(A, A.val32, x, sl, lane) : sell_row(A, A.val, x, sl, lane);
}

// ILU(0) substitution over SELL-64 packed levels: a wavefront owns a slice
// of 64 rows of one level, lane = row, and the factor entries of the slice
// are read column-major (coalesced).  Row ids and columns are device rows;
// the substitutions run in place on the vector.  FT: factor type, VT:
// vector type; the sums are FP64.
template <typename FT>
struct IluSweepArgs {
  const long long* ptr;  // slice start in the packed entries
  const int* col;        // device row of each entry's column
  const FT* val;
  const int* row;        // device row of each packed row (-1: padding)
  const int* len;        // entries of each packed row
  const FT* diag;        // backward sweep: 1/u_ii per packed row
};

// host: the packed factors of a sweep, FP64 or their FP32 copies
IluSweepArgs<double> sweep_args(const IluData::Sweep& W);
IluSweepArgs<float> sweep_args32(const IluData::Sweep& W);

// sum_k val_k v[col_k] over the L entries of one packed row of slice sl (lane
// = row).  A level or colour holds a few hundred slices, so its launch is
// bound by its chain of dependent loads: the slice's offsets are scalars, all
// entries of a row of up to kSellWide are requested at once and the vector
// entries behind them; groups of four past the slice's width are skipped by
// a wave-uniform test.  before(): loads to issue behind the entries
template <typename FT, typename VT, class Before>
__device__ __forceinline__ double packed_row_sum(const long long* ptr, const int* col,
                                                 const FT* val, int sl, int lane, int L,
                                                 const VT* v, Before before) {
  const long long base = ptr[sl];
  const int width = (int)((ptr[sl + 1] - base) >> 6);
  const int* cs = col + base + lane;
  const FT* vs = val + base + lane;
  double s = 0.0;
  if (width == 0) before();
  for (int k0 = 0; k0 < width; k0 += kSellWide) {
    int c[kSellWide];
    FT w[kSellWide];
    VT x[kSellWide];
#pragma unroll
    for (int g = 0; g < kSellWide; g += 4)
      if (k0 + g < width)
#pragma unroll
        for (int k = g; k < g + 4; k++) {
          const int q = 64 * min(k0 + k, width - 1);
          c[k] = cs[q];
          w[k] = vs[q];
        }
    if (k0 == 0) before();
#pragma unroll
    for (int g = 0; g < kSellWide; g += 4)
      if (k0 + g < width)
#pragma unroll
        for (int k = g; k < g + 4; k++) x[k] = v[c[k]];
#pragma unroll
    for (int g = 0; g < kSellWide; g += 4)
      if (k0 + g < width)
#pragma unroll
        for (int k = g; k < g + 4; k++) {
          const double t = s + (double)w[k] * (double)x[k];
          s = k0 + k < L ? t : s;
        }
  }
  return s;
}

// forward: v_i <- v_i - sum_{k before i} l_ik v_k (the v_k are already
// substituted: they belong to earlier levels); backward: v_i <- (v_i -
// sum_{k after i} u_ik v_k) / u_ii.  halt is tested once the row's place is
// known, behind the requests it does not need
template <bool BWD, typename FT, typename VT>
__device__ __forceinline__ void ilu_row(const IluSweepArgs<FT>& W, int sl, int lane, VT* v,
                                        int halt) {
  sl = __builtin_amdgcn_readfirstlane(sl);
  const int pr = sl * 64 + lane;
  const int row = W.row[pr], L = W.len[pr];
  const FT d = BWD ? W.diag[pr] : FT(1);
  if (halt) return;
  const int i = max(row, 0);
  VT own = 0;
  const double s = packed_row_sum(W.ptr, W.col, W.val, sl, lane, L, v, [&]() { own = v[i]; });
  if (row < 0) return;
  const double t = (double)own - s;
  v[i] = (VT)(BWD ? t * (double)d : t);
}

// wavefronts per block of a launch over nsl slices.  Up to one slice per CU a
// block of one wavefront reaches a CU of its own, up to two a block of two;
// beyond that a block of four costs the fewest dispatches.  Measured together
// with packed_row_sum: a colour of 20 slices 3.9 us in blocks of four, 3.5 us
inline int sweep_waves(int nsl, int cus) { return nsl <= cus ? 1 : nsl <= 2 * cus ? 2 : 4; }

// FP64 data of a mixed-precision batch member's refinement steps
struct RefineArgs {
  double* x;            // the solution
  const double* rhs;
  const double* dinv;   // Jacobi inverses of the measure (null: plain norm)
};

// factors of one batch member, FP64 and FP32 copies
struct IluMember {
  IluSweepArgs<double> f, b;
  IluSweepArgs<float> f32, b32;
};

__device__ inline void drotg_dev(double* a, double* b, double* c, double* s) {
  double roe = *b;
  if (fabs(*a) > fabs(*b)) roe = *a;
  double scale = fabs(*a) + fabs(*b);
  double r, z;
  if (scale == 0.0) {
    *c = 1.0; *s = 0.0; r = 0.0; z = 0.0;
  } else {
    double ra = *a / scale, rb = *b / scale;
    r = scale * sqrt(ra * ra + rb * rb);
    r = (roe >= 0 ? 1.0 : -1.0) * r;
    *c = *a / r;
    *s = *b / r;
    z = 1.0;
    if (fabs(*a) > fabs(*b)) z = *s;
    if (fabs(*b) >= fabs(*a) && *c != 0.0) z = 1.0 / *c;
  }
  *a = r;
  *b = z;
}

__device__ __forceinline__ void rot(double* x, double* y, double c, double s) {
  double t = c * (*x) + s * (*y);
  *y = c * (*y) - s * (*x);
  *x = t;
}


}  // namespace mf
