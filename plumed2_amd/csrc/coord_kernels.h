// Device code of the COORDINATION path: neighbour-structure build, the
// cluster-pair kernel, reductions and the FP64 kernels for the inputs the
// cluster path does not cover.  Shared by the single-system context
// (coord.hip) and the multi-system batch (batch.hip); every kernel has
// internal linkage, so each translation unit instantiates what it launches.
//
// What each piece replaces in the reference:
//   k_bin .. k_list   NeighborList::update cells branch + LinkCells
//                     (NeighborList.cpp:168-236, LinkCells.cpp:99-239); the
//                     O(N^2) pair array is never materialised, the list is one
//                     of 8x8-atom cluster pairs
//   k_pack_bbox       ActionAtomistic::retrieveAtoms gather + the image
//                     bookkeeping of Pbc::distance
//   k_pairs           CoordinationBase::calculate pair loop
//                     (CoordinationBase.cpp:178-207) with
//                     fixedRational<N>::calculateSqr (SwitchingFunction.cpp:
//                     203-215) inlined
//   k_gather_reduce,  the OpenMP critical merge + comm.Sum
//   k_finalize,       (CoordinationBase.cpp:209-224)
//   k_gather_systems
//   k_allpairs,       the same loop in FP64 for NOPBC, PAIR, unbounded D_MAX,
//   k_pairmode        cells narrower than 2*cutoff
//
// Several systems (frames, walkers) can share one set of arrays: atoms,
// columns and clusters of system s are contiguous, SysArg[s] holds its cell
// and its column grid, and per-atom / per-cluster system indices select it.
// A single system is the case nsys = 1 with null system-index arrays.
//
// Layout in HBM:
//   slots      8 consecutive slots = one cluster; clusters are runs of atoms
//              in columns of the fractional (a,b) plane sorted along c;
//              float4 {x,y,z local to the cluster origin, requested index}
//   cl_origin  double4 per cluster, FP64 origin fixed at the rebuild
//   cl_bb      2 x float4 per cluster (centre, half extents), every step
//   cl_kr      float2 per cluster: range of fractional c of its atoms
//   list       CSR over i clusters of Entry{code, delta}: code = j cluster |
//              image << 25 | count << 30 | diagonal << 31; delta =
//              o_j + T - o_i (FP32), T the image's lattice translation
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <climits>
#include <cmath>
#include <cstring>
#include <string>

#include "dbuf.h"
#include "fp64_math.h"
#include "p2a_internal.h"
#include "switch_eval.h"

namespace p2a {

#define P2A_HIP(x)                                                                           \
  do {                                                                                       \
    hipError_t e_ = (x);                                                                     \
    if (e_ != hipSuccess) return fail(P2A_ERR_HIP, std::string(#x) + ": " + hipGetErrorString(e_)); \
  } while (0)

constexpr int CL = 8;           // atoms per cluster
constexpr int WAVE = 64;
constexpr int PAIR_BLOCK = 256; // 4 waves per workgroup

struct Entry {
  int code;
  float dx, dy, dz;
};

// lattice vectors of a cell (rows), by value
struct BoxArg {
  double a[9];
};

// cell and column grid of one system
struct SysArg {
  double a[9];    // lattice vectors as rows
  double inv[9];  // inverse of a
  float af[9];    // lattice vectors in FP32 (list search)
  float rb[3];    // list radius as a fraction of the cell along a, b, c (r * |reciprocal row|)
  int ncx, ncy;   // columns along a and b
  int colbase;    // first column of this system in the shared column arrays
  float icx, icy;  // 1/ncx, 1/ncy
  // a cell along the axes (column_window): its squared edges a and b, 1/|c|
  int ortho;
  float aa, bb, invc;
};

struct PbcArg {
  int type;
  double box[9], inv[9], red[9], ired[9];
  int nshift[8];
  double shifts[8][kMaxShift][3];
};

// Entry code bits: j cluster (bits 0-24), image code (bits 25-29:
// (mx+1) + 3(my+1) + 9(mz+1), the lattice translation of the j cluster),
// "count" (bit 30: this entry adds to the value and the virial; each
// unordered pair of atoms is counted by exactly one entry), "diagonal" (bit
// 31: i cluster paired with itself without image, pairs with j == i are
// skipped and counted when j > i).
constexpr int kCjMask = 0x1FFFFFF;
constexpr int kImgShift = 25;
constexpr int kCountBit = 0x40000000;
constexpr int kMaxClusters = kCjMask;

namespace {

// ------------------------------------------------------------------------
// small device helpers
// ------------------------------------------------------------------------
__device__ __forceinline__ double wave_sum(double v) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

template <int CTRL, int ROWS>
__device__ __forceinline__ int dpp_i(int v) {
  return __builtin_amdgcn_update_dpp(0, v, CTRL, ROWS, 0xF, false);
}
constexpr int kShr1 = 0x111, kShr2 = 0x112, kShr4 = 0x114, kShr8 = 0x118;
constexpr int kBcast15 = 0x142, kBcast31 = 0x143;
// exclusive prefix sum over the 64 lanes (all active); total = sum of all lanes
// (uniform)
__device__ __forceinline__ int wave_excl_scan(int x, int& total) {
  int v = x;
  v += dpp_i<kShr1, 0xF>(v);
  v += dpp_i<kShr2, 0xF>(v);
  v += dpp_i<kShr4, 0xF>(v);
  v += dpp_i<kShr8, 0xF>(v);
  v += dpp_i<kBcast15, 0xA>(v);
  v += dpp_i<kBcast31, 0xC>(v);
  total = __builtin_amdgcn_readlane(v, 63);
  return v - x;
}

// exclusive prefix sums of a and c over the workgroup (at most 1024 threads):
// wave scans, then the wave totals from LDS (sw: 32 ints); ta, tc receive
// the workgroup totals
__device__ __forceinline__ void block_excl_scan2(int& a, int& c, int& ta, int& tc, int* sw) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
  int wa, wc;
  const int ea = wave_excl_scan(a, wa);
  const int ec = wave_excl_scan(c, wc);
  if (lane == 0) {
    sw[w] = wa;
    sw[16 + w] = wc;
  }
  __syncthreads();
  int pa = 0, pc = 0;
  ta = 0;
  tc = 0;
  for (int q = 0; q < nw; q++) {
    const int xa = sw[q], xc = sw[16 + q];
    if (q < w) {
      pa += xa;
      pc += xc;
    }
    ta += xa;
    tc += xc;
  }
  a = pa + ea;
  c = pc + ec;
  __syncthreads();
}

// The arguments of one launch over the two groups (or the two directions) of a
// list build; workgroups 0 .. n0-1 are the first one's, the others the second's.
// At the sizes of small groups a build is a row of launches of 2-7 us each, and
// the two halves of one launch run side by side (2,000 atoms in two groups, list built
// in the call: 135 us a call, 73 so and with k_items and the schedule in the fill).
template <class T>
struct Two {
  T s[2];
  int n0;
  __device__ __forceinline__ int side() const { return (int)blockIdx.x >= n0 ? 1 : 0; }
  __device__ __forceinline__ int block(int d) const { return (int)blockIdx.x - (d ? n0 : 0); }
};

__device__ __forceinline__ int nsys_of(const int* idx, int i) { return idx ? idx[i] : 0; }

// Workgroups are dispatched to the 8 XCDs of the chip in turn (workgroup b to
// XCD b mod 8), and each XCD has its own L2.  This index puts the workgroups
// of one XCD on one contiguous run of indices, so that an XCD takes one
// contiguous share of the spatially sorted work items and its L2 holds the
// positions of one region instead of all of them.  A bijection on
// [0, nb) for any grid size.
__device__ __forceinline__ int xcd_block(int b, int nb) {
  const int q = nb >> 3, r = nb & 7, x = b & 7;
  return x * q + min(x, r) + (b >> 3);
}

// ------------------------------------------------------------------------
// rebuild kernels
// ------------------------------------------------------------------------

// Column counting is privatised per workgroup: the workgroup's atoms fall in
// a narrow window of columns (consecutive atoms of one system), counted in
// LDS and added to the global counts once per (workgroup, column).  A window
// wider than kBinLds falls back to one global atomic per atom.
constexpr int kBinLds = 4096;

__device__ __forceinline__ void block_col_range(int col, int* sh, int& lo, int& hi) {
  // col < 0 marks a thread without an atom
  const int t = threadIdx.x;
  sh[t] = col < 0 ? INT_MAX : col;
  sh[256 + t] = col;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if (t < o) {
      sh[t] = min(sh[t], sh[t + o]);
      sh[256 + t] = max(sh[256 + t], sh[256 + t + o]);
    }
    __syncthreads();
  }
  lo = sh[0];
  hi = sh[256];
  __syncthreads();
}

// fractional coordinates, image and column of every atom (atom i of the
// arrays is requested atom off + i); column counts
// mmax (optional): largest |lattice translation| of a wrapped atom, as an
// atomic maximum; mclear is zeroed for the next rebuild (two alternating slots).
// order (optional): the atoms in the slot order of the previous build (norder
// slots, -1 = padding), so that a workgroup's atoms share few columns and its
// counts stay in LDS; otherwise thread i takes atom i.
struct BinSide {
  int n, off;
  int norder;
  const int* order;
  const SysArg* sys;
  int4* info;
  double* key;
  int* col_count;
  const int* col_start;
  int *fill, *tmp;
};
__device__ __forceinline__ void bin_atoms(int blk, int n, const double* __restrict__ pos, int off,
                                          const SysArg* __restrict__ sys, const int* __restrict__ atom_sys,
                                          int4* __restrict__ info, double* __restrict__ key,
                                          int* __restrict__ col_count, int* __restrict__ mmax,
                                          int* __restrict__ mclear, const int* __restrict__ order, int norder) {
  __shared__ int sh[512];
  __shared__ int hist[kBinLds];
  const int s = blk * blockDim.x + threadIdx.x;
  const int i = order ? (s < norder ? order[s] : -1) : (s < n ? s : -1);
  int col = -1;
  int am = 0;
  if (i >= 0) {
    const SysArg& S = sys[nsys_of(atom_sys, i)];
    const double* x = pos + 3 * (size_t)(off + i);
    double sf[3];
    int m[3];
    for (int j = 0; j < 3; j++) {
      sf[j] = x[0] * S.inv[0 * 3 + j] + x[1] * S.inv[1 * 3 + j] + x[2] * S.inv[2 * 3 + j];
      double fl = floor(sf[j]);
      m[j] = (int)fl;
      sf[j] -= fl;
    }
    int cx = min((int)(sf[0] * S.ncx), S.ncx - 1);
    int cy = min((int)(sf[1] * S.ncy), S.ncy - 1);
    cx = max(cx, 0);
    cy = max(cy, 0);
    col = S.colbase + cx + S.ncx * cy;
    info[i] = make_int4(m[0], m[1], m[2], col);
    // a coordinate that is not a number (or infinite) ranks as 0: a NaN key takes no
    // place of its own in k_rank, and the slot left out would hold any index
    key[i] = sf[2] >= 0.0 ? sf[2] : 0.0;
    am = max(abs(m[0]), max(abs(m[1]), abs(m[2])));
  }
  if (mmax) {
    for (int o = 32; o > 0; o >>= 1) am = max(am, __shfl_xor(am, o, 64));
    if ((threadIdx.x & 63) == 0 && am > 0) atomicMax(mmax, am);
    if (s == 0) *mclear = 0;
  }
  int lo, hi;
  block_col_range(col, sh, lo, hi);
  if (hi < 0) return;  // no atom in this workgroup (uniform)
  if (hi - lo >= kBinLds) {
    if (col >= 0) atomicAdd(&col_count[col], 1);
    return;
  }
  const int range = hi - lo + 1;
  for (int j = threadIdx.x; j < range; j += blockDim.x) hist[j] = 0;
  __syncthreads();
  if (col >= 0) atomicAdd(&hist[col - lo], 1);
  __syncthreads();
  for (int j = threadIdx.x; j < range; j += blockDim.x)
    if (hist[j]) atomicAdd(&col_count[lo + j], hist[j]);
}
__global__ __launch_bounds__(256) void k_bin(Two<BinSide> T, const double* pos, const int* atom_sys, int* mmax,
                                             int* mclear) {
  const int d = T.side();
  const BinSide& B = T.s[d];
  bin_atoms(T.block(d), B.n, pos, B.off, B.sys, atom_sys, B.info, B.key, B.col_count, mmax, mclear, B.order, B.norder);
}

// Two exclusive scans of one count array in one pass over it (out0 of in[i],
// out1 of ceil(in[i]/chunk)), across many workgroups: per-block sums, a
// scan of the block sums, then per-block local scans with the block offsets.
// n is read from n_dev when given; out0[n], out1[n] and totals[slot0/1]
// receive the two totals.
constexpr int kScanBlock = 1024;  // elements per workgroup (256 threads x 4)

// the same two scans in one workgroup of 1024 threads (a contiguous run of at
// most 8 counts per thread), for counts that one workgroup scans faster than
// three launches
constexpr int kScanOneMax = 8192;
struct ScanSide {
  int n;
  const int* n_dev;
  const int* in;
  int *out0, *out1;
  int slot0, slot1;
  int* bsum;
};
__global__ __launch_bounds__(1024) void k_scan2_one(Two<ScanSide> A, int chunk, int* __restrict__ totals) {
  __shared__ int sw[32];
  const ScanSide& S = A.s[blockIdx.x];
  const int* __restrict__ in = S.in;
  int* __restrict__ out0 = S.out0;
  int* __restrict__ out1 = S.out1;
  const int n = S.n_dev ? *S.n_dev : S.n;
  const int t = threadIdx.x, T = blockDim.x;
  const int per = (n + T - 1) / T;  // <= 8: n <= kScanOneMax
  const int b = min(n, t * per), e = min(n, b + per);
  int v[8];
  int la = 0, lc = 0;
#pragma unroll
  for (int k = 0; k < 8; k++) v[k] = (b + k < e) ? in[b + k] : 0;
#pragma unroll
  for (int k = 0; k < 8; k++) {
    la += v[k];
    lc += (v[k] + chunk - 1) / chunk;
  }
  int ra = la, rc = lc, ta, tc;
  block_excl_scan2(ra, rc, ta, tc, sw);
#pragma unroll
  for (int k = 0; k < 8; k++) {
    if (b + k < e) {
      out0[b + k] = ra;
      out1[b + k] = rc;
      ra += v[k];
      rc += (v[k] + chunk - 1) / chunk;
    }
  }
  if (t == 0) {
    out0[n] = ta;
    out1[n] = tc;
    totals[S.slot0] = ta;
    totals[S.slot1] = tc;
  }
}

__global__ __launch_bounds__(256) void k_scan2_sums(Two<ScanSide> A, int chunk) {
  __shared__ int sw[32];
  const int d = A.side(), blk = A.block(d);
  const ScanSide& S = A.s[d];
  const int* __restrict__ in = S.in;
  const int n = S.n_dev ? *S.n_dev : S.n;
  const int base = blk * kScanBlock + threadIdx.x * 4;
  int a = 0, c = 0;
  for (int k = 0; k < 4; k++) {
    const int i = base + k;
    if (i < n) {
      a += in[i];
      c += (in[i] + chunk - 1) / chunk;
    }
  }
  int ta, tc;
  block_excl_scan2(a, c, ta, tc, sw);
  if (threadIdx.x == 0) {
    S.bsum[2 * blk] = ta;
    S.bsum[2 * blk + 1] = tc;
  }
}

// every workgroup adds up the block sums before its own (a scan of them in a
// launch between took 5 us)
__global__ __launch_bounds__(256) void k_scan2_apply(Two<ScanSide> A, int chunk, int* __restrict__ totals) {
  __shared__ int sw[32];
  const int d = A.side(), blk = A.block(d);
  const ScanSide& S = A.s[d];
  const int* __restrict__ in = S.in;
  const int* __restrict__ bsum = S.bsum;
  int* __restrict__ out0 = S.out0;
  int* __restrict__ out1 = S.out1;
  const int n = S.n_dev ? *S.n_dev : S.n;
  if (blk > 0 && blk * kScanBlock >= n) return;  // uniform per workgroup
  int pa = 0, pc = 0, ba, bc;
  for (int i = threadIdx.x; i < blk; i += 256) {
    pa += bsum[2 * i];
    pc += bsum[2 * i + 1];
  }
  block_excl_scan2(pa, pc, ba, bc, sw);
  const int base = blk * kScanBlock + threadIdx.x * 4;
  int va[4], vc[4], a = 0, c = 0;
  for (int k = 0; k < 4; k++) {
    const int i = base + k;
    va[k] = (i < n) ? in[i] : 0;
    vc[k] = (i < n) ? (va[k] + chunk - 1) / chunk : 0;
    a += va[k];
    c += vc[k];
  }
  int ta, tc;
  block_excl_scan2(a, c, ta, tc, sw);
  int ra = a + ba, rc = c + bc;
  if (threadIdx.x == 0 && (blk + 1) * kScanBlock >= n) {  // the last one
    out0[n] = ba + ta;
    out1[n] = bc + tc;
    totals[S.slot0] = ba + ta;
    totals[S.slot1] = bc + tc;
  }
  for (int k = 0; k < 4; k++) {
    const int i = base + k;
    if (i < n) {
      out0[i] = ra;
      out1[i] = rc;
    }
    ra += va[k];
    rc += vc[k];
  }
}

__global__ void k_fill_int(int* p, int n, int v) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// three fills in one launch (grid-stride over the longest)
__global__ void k_fill_int3(int* p0, int n0, int v0, int* p1, int n1, int v1, int* p2, int n2, int v2) {
  const int i0 = blockIdx.x * blockDim.x + threadIdx.x, st = gridDim.x * blockDim.x;
  for (int i = i0; i < n0; i += st) p0[i] = v0;
  for (int i = i0; i < n1; i += st) p1[i] = v1;
  for (int i = i0; i < n2; i += st) p2[i] = v2;
}

// flag[0] = 1 when some atom lies farther than sqrt(lim2) from its position
// at the last list build (a NaN coordinate counts as moved); flag[0] must be
// zero before the launch
__global__ __launch_bounds__(256) void k_moved(int n, const double* __restrict__ pos,
                                               const double* __restrict__ ref, double lim2, int* __restrict__ flag) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  bool m = false;
  if (i < n) {
    const double dx = pos[3 * (size_t)i] - ref[3 * (size_t)i];
    const double dy = pos[3 * (size_t)i + 1] - ref[3 * (size_t)i + 1];
    const double dz = pos[3 * (size_t)i + 2] - ref[3 * (size_t)i + 2];
    m = !(dx * dx + dy * dy + dz * dz <= lim2);
  }
  if (__ballot(m) != 0ull && (threadIdx.x & (WAVE - 1)) == 0) atomicOr(flag, 1);
}

__global__ void k_fill_double(double* p, size_t n) {
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  size_t stride = (size_t)gridDim.x * blockDim.x;
  for (; i < n; i += stride) p[i] = 0.0;
}

// atoms listed by column (any order inside a column; k_rank orders them);
// slots within a column are reserved once per (workgroup, column) as in
// k_bin, over the same atom order
__device__ __forceinline__ void scatter_atoms(int blk, int n, const int4* __restrict__ info,
                                              const int* __restrict__ col_start, int* __restrict__ fill,
                                              int* __restrict__ tmp, const int* __restrict__ order, int norder) {
  __shared__ int sh[512];
  __shared__ int hist[kBinLds];
  const int s = blk * blockDim.x + threadIdx.x;
  const int i = order ? (s < norder ? order[s] : -1) : (s < n ? s : -1);
  const int col = (i >= 0) ? info[i].w : -1;
  int lo, hi;
  block_col_range(col, sh, lo, hi);
  if (hi < 0) return;  // uniform
  if (hi - lo >= kBinLds) {
    if (col >= 0) {
      const int k = atomicAdd(&fill[col], 1);
      tmp[col_start[col] + k] = i;
    }
    return;
  }
  const int range = hi - lo + 1;
  for (int j = threadIdx.x; j < range; j += blockDim.x) hist[j] = 0;
  __syncthreads();
  const int local = (col >= 0) ? atomicAdd(&hist[col - lo], 1) : 0;
  __syncthreads();
  // hist[j] becomes this workgroup's first slot in column lo + j
  for (int j = threadIdx.x; j < range; j += blockDim.x)
    if (hist[j]) hist[j] = atomicAdd(&fill[lo + j], hist[j]);
  __syncthreads();
  if (col >= 0) tmp[col_start[col] + hist[col - lo] + local] = i;
}
__global__ __launch_bounds__(256) void k_scatter(Two<BinSide> T) {
  const int d = T.side();
  const BinSide& B = T.s[d];
  scatter_atoms(T.block(d), B.n, B.info, B.col_start, B.fill, B.tmp, B.order, B.norder);
}

// Slots of one column and the bounds of its clusters; one workgroup per column.
// (1) Rank of each atom inside its column by (key, index): a deterministic
//     order.  When the column fits in LDS its atoms are grouped into buckets
//     of key (a counting pass, a scan, a scatter), and each atom is ranked
//     against its own bucket only; larger columns count over the whole
//     column in global memory.
// (2) Per cluster (8 lanes, one per slot): FP64 origin (bounding-box centre
//     of the wrapped positions at the rebuild), FP32 bounding box, range of
//     fractional c (widened outwards so that the FP32 range contains the
//     FP64 keys) and system.  Padding slots come last in a cluster, so its
//     first slot always holds an atom.
// With pk, also what k_pack_bbox would write for these positions.
// Columns hold ~8 atoms per column width of height (a few hundred in cells up
// to ~30 column widths tall); kRankLds bounds the LDS of a workgroup to
// ~21 KB, so that 7 columns share a CU.
constexpr int kRankLds = 1024;
constexpr int kRankBuckets = 256;  // the workgroup size: one scan
__device__ __forceinline__ int rank_bucket(double k) {
  return max(0, min((int)(k * kRankBuckets), kRankBuckets - 1));
}
// clear0, clear1 (optional): the column's atom count and fill position, zeroed
// for the next build.  slot_img (optional): the lattice translations in slot
// order, which k_pack_bbox reads in a row (500,000 atoms: 20 -> 14 us a step,
// this kernel 35 -> 37).
struct RankSide {
  int ncol, off;
  const double* key;
  const int *col_start, *col_cl, *tmp;
  int* slot_loc;
  const int4* info;
  const SysArg* sys;
  double4* origin;
  float4* bb0;
  float2* kr;
  int *cl_sys, *cl_col;
  float4 *pk, *pbb;
  int *clear0, *clear1;
  int4* slot_img;
};
__device__ __forceinline__ void rank_column(int col, int ncol, const double* __restrict__ key,
                                            const int* __restrict__ col_start, const int* __restrict__ col_cl,
                                            const int* __restrict__ tmp, int* __restrict__ slot_loc,
                                            const int4* __restrict__ info, const double* __restrict__ pos, int off,
                                            const SysArg* __restrict__ sys, const int* __restrict__ atom_sys,
                                            double4* __restrict__ origin, float4* __restrict__ bb0,
                                            float2* __restrict__ kr, int* __restrict__ cl_sys,
                                            int* __restrict__ cl_col, float4* __restrict__ pk,
                                            float4* __restrict__ pbb, int4* __restrict__ slot_img, double pscale) {
  __shared__ double sk[kRankLds];
  __shared__ int si[kRankLds];
  __shared__ int ss[kRankLds];
  __shared__ int sbk[kRankLds];  // local indices grouped by key bucket
  __shared__ int bcnt[kRankBuckets], bstart[kRankBuckets + 1];
  __shared__ int sw[32];
  if (col >= ncol) return;
  const int b = col_start[col], n = col_start[col + 1] - b;
  const int c0 = col_cl[col], ncl = col_cl[col + 1] - c0;
  const int base = c0 * CL;
  for (int q = threadIdx.x; q < ncl; q += blockDim.x) cl_col[c0 + q] = col;
  // padding slots at the end of the column's last cluster
  for (int t = n + (int)threadIdx.x; t < ncl * CL; t += blockDim.x) slot_loc[base + t] = -1;
  const bool lds = n <= kRankLds;
  if (lds) {
    // the keys lie in [0, 1): bucket floor(key * kRankBuckets) keeps their
    // order, so an atom's rank is the atoms of the lower buckets plus those of
    // its own bucket below it by (key, index)
    for (int q = threadIdx.x; q < kRankBuckets; q += blockDim.x) bcnt[q] = 0;
    for (int t = threadIdx.x; t < n; t += blockDim.x) {
      const int o = tmp[b + t];
      si[t] = o;
      sk[t] = key[o];
    }
    __syncthreads();
    for (int t = threadIdx.x; t < n; t += blockDim.x)
      atomicAdd(&bcnt[rank_bucket(sk[t])], 1);
    __syncthreads();
    {
      int v = threadIdx.x < kRankBuckets ? bcnt[threadIdx.x] : 0, dummy = 0, tot, tot2;
      block_excl_scan2(v, dummy, tot, tot2, sw);
      if (threadIdx.x < kRankBuckets) {
        bstart[threadIdx.x] = v;
        bcnt[threadIdx.x] = v;  // fill pointer of the bucket
      }
      if (threadIdx.x == 0) bstart[kRankBuckets] = tot;
    }
    __syncthreads();
    for (int t = threadIdx.x; t < n; t += blockDim.x)
      sbk[atomicAdd(&bcnt[rank_bucket(sk[t])], 1)] = t;
    __syncthreads();
    for (int t = threadIdx.x; t < n; t += blockDim.x) {
      const double ka = sk[t];
      const int ia = si[t];
      const int bk = rank_bucket(ka);
      const int p1 = bstart[bk + 1];
      int rank = bstart[bk];
      for (int p = bstart[bk]; p < p1; p++) {
        const int u = sbk[p];
        const double kb = sk[u];
        rank += (kb < ka) || (kb == ka && si[u] < ia);
      }
      slot_loc[base + rank] = ia;
      ss[rank] = ia;
    }
  } else {
    for (int t = threadIdx.x; t < n; t += blockDim.x) {
      const int ia = tmp[b + t];
      const double ka = key[ia];
      int rank = 0;
      for (int u = 0; u < n; u++) {
        const int o = tmp[b + u];
        const double kb = key[o];
        rank += (kb < ka) || (kb == ka && o < ia);
      }
      slot_loc[base + rank] = ia;
    }
  }
  __syncthreads();
  // (2) the column's clusters; the loop bound is uniform over the workgroup.
  // With pk, also what k_pack_bbox would write for these positions: the
  // packed slots (pk) and the boxes of the packed clusters (pbb).
  for (int t0 = 0; t0 < ncl * CL; t0 += blockDim.x) {
    const int t = t0 + (int)threadIdx.x;
    int a = -1;
    if (t < n) a = lds ? ss[t] : slot_loc[base + t];
    double lo[3] = {DBL_MAX, DBL_MAX, DBL_MAX}, hi[3] = {-DBL_MAX, -DBL_MAX, -DBL_MAX};
    double w[3] = {0.0, 0.0, 0.0};
    double klo = DBL_MAX, khi = -DBL_MAX;
    int sy = 0;
    if (a >= 0) {
      sy = nsys_of(atom_sys, a);
      const SysArg& S = sys[sy];
      const int4 m = info[a];
      if (slot_img) slot_img[base + t] = m;
      const double* x = pos + 3 * (size_t)(off + a);
      for (int d = 0; d < 3; d++) {
        w[d] = x[d] - (m.x * S.a[0 * 3 + d] + m.y * S.a[1 * 3 + d] + m.z * S.a[2 * 3 + d]);
        lo[d] = w[d];
        hi[d] = w[d];
      }
      klo = khi = key[a];
    }
    // the 8 lanes of a cluster are aligned in the wave
    for (int o = 1; o < CL; o <<= 1) {
      for (int d = 0; d < 3; d++) {
        lo[d] = fmin(lo[d], __shfl_xor(lo[d], o, 64));
        hi[d] = fmax(hi[d], __shfl_xor(hi[d], o, 64));
      }
      klo = fmin(klo, __shfl_xor(klo, o, 64));
      khi = fmax(khi, __shfl_xor(khi, o, 64));
    }
    const double cx = 0.5 * (lo[0] + hi[0]), cy = 0.5 * (lo[1] + hi[1]), cz = 0.5 * (lo[2] + hi[2]);
    const int c = c0 + t / CL;
    if ((t & (CL - 1)) == 0 && t < ncl * CL) {
      if (cl_sys) cl_sys[c] = sy;
      origin[c] = make_double4(cx, cy, cz, 0.0);
      bb0[2 * c] = make_float4((float)cx, (float)cy, (float)cz, 0.f);
      bb0[2 * c + 1] = make_float4((float)(0.5 * (hi[0] - lo[0])), (float)(0.5 * (hi[1] - lo[1])),
                                   (float)(0.5 * (hi[2] - lo[2])), 0.f);
      kr[c] = make_float2((float)klo - 1.0e-6f, (float)khi + 1.0e-6f);
    }
    if (pk) {
      const int sl = base + t;
      float4 q;
      float ql[3], qh[3];
      if (a < 0) {
        q = make_float4(1.0e5f + 1.0e3f * (float)(sl & 1023), 1.0e5f + 1.0e3f * (float)((sl >> 10) & 1023),
                        1.0e5f + 1.0e3f * (float)(sl >> 20), __int_as_float(-1));
        ql[0] = ql[1] = ql[2] = FLT_MAX;
        qh[0] = qh[1] = qh[2] = -FLT_MAX;
      } else {
        q = make_float4((float)((w[0] - cx) * pscale), (float)((w[1] - cy) * pscale), (float)((w[2] - cz) * pscale),
                        __int_as_float(off + a));
        ql[0] = qh[0] = q.x;
        ql[1] = qh[1] = q.y;
        ql[2] = qh[2] = q.z;
      }
      if (t < ncl * CL) pk[sl] = q;
      for (int o = 1; o < CL; o <<= 1) {
        for (int d = 0; d < 3; d++) {
          ql[d] = fminf(ql[d], __shfl_xor(ql[d], o, 64));
          qh[d] = fmaxf(qh[d], __shfl_xor(qh[d], o, 64));
        }
      }
      if ((t & (CL - 1)) == 0 && t < ncl * CL) {
        pbb[2 * c] = make_float4(0.5f * (ql[0] + qh[0]), 0.5f * (ql[1] + qh[1]), 0.5f * (ql[2] + qh[2]), 0.f);
        pbb[2 * c + 1] = make_float4(0.5f * (qh[0] - ql[0]), 0.5f * (qh[1] - ql[1]), 0.5f * (qh[2] - ql[2]), 0.f);
      }
    }
  }
}

__global__ __launch_bounds__(256) void k_rank(Two<RankSide> T, const double* pos, const int* atom_sys, double pscale) {
  const int d = T.side(), col = T.block(d);
  const RankSide& R = T.s[d];
  if (R.clear0 && threadIdx.x == 0 && col < R.ncol) R.clear0[col] = R.clear1[col] = 0;
  rank_column(col, R.ncol, R.key, R.col_start, R.col_cl, R.tmp, R.slot_loc, R.info, pos, R.off, R.sys, atom_sys,
              R.origin, R.bb0, R.kr, R.cl_sys, R.cl_col, R.pk, R.pbb, R.slot_img, pscale);
}

// Two groups that share atoms: for every slot, the requested index of the same
// atom in the other group (twin, by requested index; negative: not in it), so
// that the pair kernels leave out an atom's pair with itself
__global__ void k_twin_slot(int nslot, const int* __restrict__ slot_loc, int off, const int* __restrict__ twin,
                            int* __restrict__ twin_slot) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= nslot) return;
  const int a = slot_loc[s];
  twin_slot[s] = (a >= 0) ? twin[off + a] : -2;
}

// candidates kept per i cluster between the count and fill passes of the
// list search (j cluster in bits 0-25, image code (mx+1)+3(my+1)+9(mz+1) above)
constexpr int kEll = 384;
static_assert(kEll >= 2 * WAVE, "k_list_stream reads two candidates per lane ahead");
constexpr unsigned kEllCj = 0x3FFFFFFu;

// list entry of i cluster ci for j cluster cj seen through image (mx,my,mz)
__device__ __forceinline__ Entry make_entry(int mode, int ci, int cj, int mx, int my, int mz, const SysArg& SJ,
                                            const double4* __restrict__ orgJ, const double4& oi, double pscale) {
  const double4 oj = orgJ[cj];
  const double Tx = mx * SJ.a[0] + my * SJ.a[3] + mz * SJ.a[6];
  const double Ty = mx * SJ.a[1] + my * SJ.a[4] + mz * SJ.a[7];
  const double Tz = mx * SJ.a[2] + my * SJ.a[5] + mz * SJ.a[8];
  const bool zero = (mx == 0 && my == 0 && mz == 0);
  const bool diag = mode == 0 && cj == ci && zero;
  const bool positive = (mx > 0) || (mx == 0 && (my > 0 || (my == 0 && mz > 0)));
  const bool counted = mode == 1 || (mode == 0 && (cj > ci || (cj == ci && positive)));
  Entry en;
  en.code = cj | (((mx + 1) + 3 * (my + 1) + 9 * (mz + 1)) << kImgShift) | (counted ? kCountBit : 0) |
            (diag ? (int)0x80000000u : 0);
  en.dx = (float)((oj.x + Tx - oi.x) * pscale);
  en.dy = (float)((oj.y + Ty - oi.y) * pscale);
  en.dz = (float)((oj.z + Tz - oi.z) * pscale);
  return en;
}

// entry offsets of a kept list for a new cell: the j cluster's lattice
// translation (mx, my, mz) now uses the lattice vectors a (rows), as the
// packed positions do; one wave per i cluster, lanes over its entries
__global__ __launch_bounds__(256) void k_reimage(int ncl, const int* __restrict__ estart,
                                                 const int* __restrict__ ecount, int ent_cap,
                                                 const double4* __restrict__ orgI, const double4* __restrict__ orgJ,
                                                 BoxArg box, double pscale, Entry* __restrict__ ents) {
  const int lane = threadIdx.x & (WAVE - 1);
  const int ci = blockIdx.x * (blockDim.x / WAVE) + threadIdx.x / WAVE;
  if (ci >= ncl) return;
  const int e0 = estart[ci], n = ecount[ci];
  const double4 oi = orgI[ci];
  for (int k = lane; k < n; k += WAVE) {
    const int e = e0 + k;
    if (e >= ent_cap) break;
    Entry en = ents[e];
    const int cj = en.code & kCjMask;
    const int im = (en.code >> kImgShift) & 31;
    const int mx = im % 3 - 1, my = (im / 3) % 3 - 1, mz = im / 9 - 1;
    const double4 oj = orgJ[cj];
    en.dx = (float)((oj.x + (mx * box.a[0] + my * box.a[3] + mz * box.a[6]) - oi.x) * pscale);
    en.dy = (float)((oj.y + (mx * box.a[1] + my * box.a[4] + mz * box.a[7]) - oi.y) * pscale);
    en.dz = (float)((oj.z + (mx * box.a[2] + my * box.a[5] + mz * box.a[8]) - oi.z) * pscale);
    ents[e] = en;
  }
}

// one value written to device memory in stream order: small descriptors go
// to the device as kernel arguments, so the host never waits for a staging copy
template <class T>
__global__ void k_store(T v, T* __restrict__ dst) {
  if (blockIdx.x == 0 && threadIdx.x == 0) *dst = v;
}

struct ListArgs {
  int nclI;
  const int* nclI_dev;  // device count of i clusters (null: nclI)
  int mode;             // 0 one group, 1 two groups (counting side), 2 two groups (other side)
  int ent_cap;          // capacity of the entry array (fill pass)
  float rlist2;
  double pscale;        // scale of the entry offsets (pack_scale)
};

// Cluster-pair search: one wave per i cluster.  FILL=0 counts and keeps the
// first kEll passing candidates of the cluster (j cluster | image code) in
// `ell`; FILL=1 writes the entries, streaming them from `ell` when the
// cluster's count fits there and searching again otherwise; FILL=2 does only
// the second part, after k_list_stream has done the first.
// Candidates are the clusters of the (column, image) window around the i
// cluster whose range of fractional c overlaps the i cluster's range widened
// by the list radius: a pair closer than r differs by at most r*|c*| in
// fractional c, so the window is exact; in a cell along the axes by what the
// radius leaves after the gap between the two columns (column_window).  (In a
// skewed cell the boxes of clusters reach out of their columns, and an entry
// left out for the columns' sake would move the list's work items, and with
// them the FP32 sums.)  The clusters of a column are sorted along c, so each
// window is one binary-searched run of clusters (both ends searched together).
// Each column lane writes its runs into the wave's candidate list in LDS
// (j cluster | image code, in column order), kCandCap at a time, and the
// lanes then test the listed candidates, two per lane and trip.
// Bound by VALU issue (half of its time at 50,000 atoms) and the search's chain
// of loads.  50,000 atoms, radius 1.3: 14 us; 31 us with whole windows (nine by
// nine columns, 520 candidates for 190 entries) searched end after end.
constexpr int kCandCap = 512;

// t / n and t % n for t >= 0 and a quotient below 2^22 (sys_columns bounds the
// columns), r = 1/n to a few roundings: (float)t r is within three roundings of
// the quotient, which is then off by one at most
__device__ __forceinline__ int div_by(int t, int n, float r, int& rem) {
  int q = (int)((float)t * r);
  rem = t - q * n;
  if (rem < 0) {
    q--;
    rem += n;
  } else if (rem >= n) {
    q++;
    rem -= n;
  }
  return q;
}

// Half width, in fractional c, of the range around the i cluster that can hold a
// cluster within the list radius, for a column whose differences in fractional a
// and b lie in [a0, a1] and [b0, b1] (a cell along the axes: the boxes of
// clusters stay within their columns, so the gap between the columns bounds the
// gap between the boxes); negative where there is none.  The radius is widened
// by more than the rounding of the boxes' coordinates.
__device__ __forceinline__ float column_window(const SysArg& S, float rlist2, float a0, float a1, float b0, float b1) {
  const float fa = fminf(fmaxf(0.f, a0), a1), fb = fminf(fmaxf(0.f, b0), b1);
  const float left = rlist2 * 1.0001f - S.aa * fa * fa - S.bb * fb * fb;
  if (left < 0.f) return -1.f;
  return fminf(__builtin_amdgcn_sqrtf(left) * S.invc + 2.0e-6f, S.rb[2]);
}

// With items, k_list<1> also writes the work items of its cluster ({i cluster,
// first entry, end entry} of `chunk` entries each) and their place in the pair
// kernel's schedule (k_wave_sched): two launches less.
struct ItemArgs {
  int4* items;
  const int* istart;
  int chunk, items_cap;
  int nwaves;       // 0: no schedule
  int nitems;
  long long total;  // cost of all items
  int* wave_start;
};
struct ListSide {
  ListArgs L;
  const int *cl_colI, *cl_sysI;
  const SysArg *sysI, *sysJ;
  const float4 *bbI, *bbJ;
  const float2 *krI, *krJ;
  const int* col_clJ;
  const double4 *orgI, *orgJ;
  int* count;
  const int* start;
  Entry* out;
  unsigned* ell;
  ItemArgs M;
};

// Balanced static schedule of the pair kernel: the items split into nwaves
// contiguous ranges of about equal estimated cost, an item costing its
// entries plus kItemCost (the staging and sums each item pays).  Item i
// (cost prefix P_i, total C) goes to wave floor(P_i * nwaves / C).
constexpr int kItemCost = 32;
__device__ __forceinline__ int sched_wave(long long entry0, int item, long long total, int nwaves) {
  const long long pre = entry0 + (long long)kItemCost * item;
  return (int)min((long long)nwaves - 1, pre * nwaves / total);
}

template <int FILL>
__device__ __forceinline__ void list_clusters(int blk, const ListArgs& L, const int* __restrict__ cl_colI,
                                              const int* __restrict__ cl_sysI, const SysArg* __restrict__ sysI,
                                              const SysArg* __restrict__ sysJ, const float4* __restrict__ bbI,
                                              const float4* __restrict__ bbJ, const float2* __restrict__ krI,
                                              const float2* __restrict__ krJ, const int* __restrict__ col_clJ,
                                              const double4* __restrict__ orgI, const double4* __restrict__ orgJ,
                                              int* __restrict__ count, const int* __restrict__ start,
                                              Entry* __restrict__ out, unsigned* __restrict__ ell,
                                              const ItemArgs& M) {
  __shared__ unsigned s_cand[4][kCandCap];
  __shared__ float4 s_img[4][27];  // FP32 lattice translation of each image code
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x / WAVE);
  const int nclI = L.nclI_dev ? *L.nclI_dev : L.nclI;
  // FILL=0/1: cluster ci = the wave.  FILL=2: the wave's 64 clusters, of which
  // it searches those whose candidates did not all fit in ell (the others are
  // k_list_stream's), in order.  No workgroup barrier below.
  int ci = blk * (blockDim.x / WAVE) + wv;
  unsigned long long pending = 0ull;
  if (FILL == 2) {
    const int c0 = ci * WAVE;
    pending = __ballot(c0 + lane < nclI && count[c0 + lane] > kEll);
    ci = c0;
  } else if (ci >= nclI) {
    return;
  }
  const int cfirst = ci;
  while (FILL != 2 || pending) {
  if (FILL == 2) {
    ci = cfirst + __builtin_ctzll(pending);
    pending &= pending - 1ull;
  }
  const int s = nsys_of(cl_sysI, ci);
  const SysArg& SI = sysI[s];
  const SysArg& SJ = sysJ[s];
  const int colI = cl_colI[ci] - SI.colbase;
  int cxi;
  const int cyi = div_by(colI, SI.ncx, SI.icx, cxi);
  const float4 ic = bbI[2 * ci], ih = bbI[2 * ci + 1];
  const float2 ki = krI[ci];
  // columns that a pair closer than the list radius can lie in; the margin is
  // above the rounding of the fractions
  constexpr float kMargin = 4.0e-6f;
  const bool ortho = SJ.ortho != 0;  // uniform
  const float xi0 = (float)cxi * SI.icx - kMargin, xi1 = (float)(cxi + 1) * SI.icx + kMargin;
  const float yi0 = (float)cyi * SI.icy - kMargin, yi1 = (float)(cyi + 1) * SI.icy + kMargin;
  int x0, x1, y0, y1;
  if (ortho) {
    x0 = (int)floorf((xi0 - SJ.rb[0] * 1.00001f) * SJ.ncx);
    x1 = (int)floorf((xi1 + SJ.rb[0] * 1.00001f) * SJ.ncx);
    y0 = (int)floorf((yi0 - SJ.rb[1] * 1.00001f) * SJ.ncy);
    y1 = (int)floorf((yi1 + SJ.rb[1] * 1.00001f) * SJ.ncy);
  } else {
    x0 = (int)floorf(((float)cxi / SI.ncx - SJ.rb[0]) * SJ.ncx) - 1;
    x1 = (int)floorf(((float)(cxi + 1) / SI.ncx + SJ.rb[0]) * SJ.ncx) + 1;
    y0 = (int)floorf(((float)cyi / SI.ncy - SJ.rb[1]) * SJ.ncy) - 1;
    y1 = (int)floorf(((float)(cyi + 1) / SI.ncy + SJ.rb[1]) * SJ.ncy) + 1;
  }
  // images -1, 0, +1 along a and b cover every candidate when the cell is
  // wider than 2*rlist; each unwrapped column is a distinct (column, image)
  const int xa = max(x0, -SJ.ncx), xb = min(x1, 2 * SJ.ncx - 1);
  const int ya = max(y0, -SJ.ncy), yb = min(y1, 2 * SJ.ncy - 1);
  const int nx = xb - xa + 1, ny = yb - ya + 1;
  const int ncolw = nx * ny;
  const double4 oi = orgI[ci];
  int n = 0;
  const int base = FILL ? start[ci] : 0;
  if (FILL == 1) {
    const int nc = count[ci];
    if (M.items) {
      const int i0 = M.istart[ci], nch = (nc + M.chunk - 1) / M.chunk;
      for (int k = lane; k < nch; k += WAVE) {
        const int it = i0 + k, e = base + k * M.chunk, end = base + min(nc, (k + 1) * M.chunk);
        if (it < M.items_cap) M.items[it] = make_int4(ci, e, end, 0);
        if (M.nwaves) {
          // entries are contiguous: item it + 1 starts where this one ends
          const int w0 = sched_wave(e, it, M.total, M.nwaves);
          const int w1 = it + 1 < M.nitems ? sched_wave(end, it + 1, M.total, M.nwaves) : M.nwaves;
          if (it == 0)
            for (int w = 0; w <= w0; w++) M.wave_start[w] = 0;
          for (int w = w0 + 1; w <= w1; w++) M.wave_start[w] = it + 1;
        }
      }
    }
    if (nc <= kEll) {
      for (int e = lane; e < nc; e += WAVE) {
        const unsigned pk = ell[(size_t)ci * kEll + e];
        const int cj = (int)(pk & kEllCj), im = (int)(pk >> 26);
        if (base + e < L.ent_cap)
          out[base + e] = make_entry(L.mode, ci, cj, im % 3 - 1, (im / 3) % 3 - 1, im / 9 - 1, SJ, orgJ, oi, L.pscale);
      }
      return;
    }
  }
  if (lane < 27) {
    const int mx = lane % 3 - 1, my = (lane / 3) % 3 - 1, mz = lane / 9 - 1;
    s_img[wv][lane] = make_float4(mx * SJ.af[0] + my * SJ.af[3] + mz * SJ.af[6],
                                  mx * SJ.af[1] + my * SJ.af[4] + mz * SJ.af[7],
                                  mx * SJ.af[2] + my * SJ.af[5] + mz * SJ.af[8], 0.f);
  }
  const float sx = SJ.icx, sy = SJ.icy, inx = __builtin_amdgcn_rcpf((float)nx);
  // one lane per window column; it covers the images -1, 0, +1 along c, of
  // which only those whose shifted window meets [0, 1) are searched
  for (int t0 = 0; t0 < ncolw; t0 += WAVE) {
    const int t = t0 + lane;
    int f[3] = {0, 0, 0}, cnt[3] = {0, 0, 0}, img = 0;
    if (t < ncolw) {
      int tx;
      const int ty = div_by(t, nx, inx, tx), cxu = xa + tx, cyu = ya + ty;
      const int mx = cxu < 0 ? -1 : (cxu >= SJ.ncx ? 1 : 0), my = cyu < 0 ? -1 : (cyu >= SJ.ncy ? 1 : 0);
      const int cxw = cxu - mx * SJ.ncx, cyw = cyu - my * SJ.ncy;
      const int col = SJ.colbase + cxw + SJ.ncx * cyw;
      const int c0 = col_clJ[col], c1 = col_clJ[col + 1];
      img = (mx + 1) | ((my + 1) << 2);
      const float zw = ortho ? column_window(SJ, L.rlist2, cxu * sx - xi1, (cxu + 1) * sx - xi0, cyu * sy - yi1,
                                             (cyu + 1) * sy - yi0)
                             : SJ.rb[2];
      const float zlo = ki.x - zw - 1.0e-6f, zhi = ki.y + zw + 1.0e-6f;
      if (zw >= 0.f && c1 > c0) {
#pragma unroll
        for (int m = 0; m < 3; m++) {
          const float lo = zlo - (float)(m - 1), hi = zhi - (float)(m - 1);
          if (hi >= 0.f && lo < 1.f) {
            // [a, .): first cluster whose upper key reaches lo; [., u): first
            // cluster whose lower key exceeds hi
            int a = c0, b = c1, u = c0, v = c1;
            while (a < b || u < v) {
              const int q = min((a + b) >> 1, c1 - 1), r = min((u + v) >> 1, c1 - 1);
              const float ky = krJ[q].y, kx = krJ[r].x;
              if (a < b) {
                if (ky < lo) a = q + 1;
                else b = q;
              }
              if (u < v) {
                if (kx <= hi) u = r + 1;
                else v = r;
              }
            }
            f[m] = a;
            cnt[m] = max(u - a, 0);
          }
        }
      }
    }
    int total;
    const int off = wave_excl_scan(cnt[0] + cnt[1] + cnt[2], total);
    for (int c0 = 0; c0 < total; c0 += kCandCap) {
      const int nc = min(total - c0, kCandCap);
      // this lane's candidates with list index in [c0, c0 + nc)
      int k = off;
#pragma unroll
      for (int m = 0; m < 3; m++) {
        const unsigned code = (unsigned)(((img & 3) + 3 * ((img >> 2) & 3) + 9 * m) << 26);
        const int lo = max(k, c0), hi = min(k + cnt[m], c0 + nc);
        for (int u = lo; u < hi; u++) s_cand[wv][u - c0] = (unsigned)(f[m] + (u - k)) | code;
        k += cnt[m];
      }
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      __builtin_amdgcn_wave_barrier();
      // two candidates per lane and trip: their box loads are in flight together
      for (int u0 = 0; u0 < nc; u0 += 2 * WAVE) {
        unsigned pk[2] = {0u, 0u};
        float4 jc[2], jh[2];
#pragma unroll
        for (int h = 0; h < 2; h++) {
          const int u = u0 + h * WAVE + lane;
          jc[h] = jh[h] = make_float4(0.f, 0.f, 0.f, 0.f);
          if (u < nc) {
            pk[h] = s_cand[wv][u];
            const int cj = (int)(pk[h] & kEllCj);
            jc[h] = bbJ[2 * cj];
            jh[h] = bbJ[2 * cj + 1];
          }
        }
#pragma unroll
        for (int h = 0; h < 2; h++) {
          const int u = u0 + h * WAVE + lane;
          bool pass = false;
          if (u < nc) {
            const float4 T = s_img[wv][pk[h] >> 26];
            const float gx = fmaxf(fabsf(jc[h].x + T.x - ic.x) - ih.x - jh[h].x, 0.f);
            const float gy = fmaxf(fabsf(jc[h].y + T.y - ic.y) - ih.y - jh[h].y, 0.f);
            const float gz = fmaxf(fabsf(jc[h].z + T.z - ic.z) - ih.z - jh[h].z, 0.f);
            pass = fmaf(gz, gz, fmaf(gx, gx, gy * gy)) < L.rlist2;
          }
          const unsigned long long bal = __ballot(pass);
          if (pass) {
            const int k = n + __popcll(bal & ((1ull << lane) - 1));
            if (FILL) {
              const int cj = (int)(pk[h] & kEllCj), im = (int)(pk[h] >> 26);
              if (base + k < L.ent_cap)
                out[base + k] =
                    make_entry(L.mode, ci, cj, im % 3 - 1, (im / 3) % 3 - 1, im / 9 - 1, SJ, orgJ, oi, L.pscale);
            } else if (k < kEll) {
              ell[(size_t)ci * kEll + k] = pk[h];
            }
          }
          n += __popcll(bal);
        }
      }
      // the next chunk overwrites the candidate list read above
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
  }
  if (!FILL && lane == 0) count[ci] = n;
  if (FILL != 2) break;
  }
}

template <int FILL>
__global__ __launch_bounds__(256) void k_list(Two<ListSide> T) {
  const int d = T.side();
  const ListSide& S = T.s[d];
  list_clusters<FILL>(T.block(d), S.L, S.cl_colI, S.cl_sysI, S.sysI, S.sysJ, S.bbI, S.bbJ, S.krI, S.krJ, S.col_clJ,
                      S.orgI, S.orgJ, S.count, S.start, S.out, S.ell, S.M);
}

// Fill pass of the clusters whose candidates all fit in `ell` (count <=
// kEll): their entries in the order the count pass kept them, one wave per
// i cluster, two entries per lane and trip.  The search kernel's registers
// are not held here, so more waves are resident to cover the two dependent
// loads (kept candidate, then the j cluster's origin) of each entry.  Used
// with k_list<2> where the fill covers many clusters (the batch); a single
// system's list is filled by k_list<1> in one launch.
__global__ __launch_bounds__(256) void k_list_stream(ListArgs L, const int* __restrict__ cl_sysI,
                                                     const SysArg* __restrict__ sysJ,
                                                     const double4* __restrict__ orgI,
                                                     const double4* __restrict__ orgJ, const int* __restrict__ count,
                                                     const int* __restrict__ start, Entry* __restrict__ out,
                                                     const unsigned* __restrict__ ell) {
  const int lane = threadIdx.x & 63;
  const int ci = blockIdx.x * (blockDim.x / WAVE) + __builtin_amdgcn_readfirstlane((int)threadIdx.x / WAVE);
  const int nclI = L.nclI_dev ? *L.nclI_dev : L.nclI;
  if (ci >= nclI) return;
  // everything that depends on ci only, and the first two kept candidates of
  // each lane (ell has kEll >= 2 * WAVE slots per cluster, written or not),
  // is loaded before the count decides anything
  const unsigned* kept = ell + (size_t)ci * kEll;
  const unsigned p0 = kept[lane], p1 = kept[WAVE + lane];
  const int nc = count[ci];
  const int base = start[ci];
  const int sy = nsys_of(cl_sysI, ci);
  const double4 oi = orgI[ci];
  if (nc > kEll) return;
  const SysArg& SJ = sysJ[sy];
  for (int e0 = 0; e0 < nc; e0 += 2 * WAVE) {
    const int ea = e0 + lane, eb = e0 + WAVE + lane;
    const unsigned pa = ea < nc ? (e0 == 0 ? p0 : kept[ea]) : 0u, pb = eb < nc ? (e0 == 0 ? p1 : kept[eb]) : 0u;
    const int ja = (int)(pa & kEllCj), ia = (int)(pa >> 26);
    const int jb = (int)(pb & kEllCj), ib = (int)(pb >> 26);
    if (ea < nc && base + ea < L.ent_cap)
      out[base + ea] = make_entry(L.mode, ci, ja, ia % 3 - 1, (ia / 3) % 3 - 1, ia / 9 - 1, SJ, orgJ, oi, L.pscale);
    if (eb < nc && base + eb < L.ent_cap)
      out[base + eb] = make_entry(L.mode, ci, jb, ib % 3 - 1, (ib / 3) % 3 - 1, ib / 9 - 1, SJ, orgJ, oi, L.pscale);
  }
}

// work items {i cluster, first entry, end entry} of `chunk` entries each;
// writes past items_cap are dropped
__global__ void k_items(int ncl, const int* __restrict__ ncl_dev, const int* __restrict__ count,
                        const int* __restrict__ estart, const int* __restrict__ item_start, int4* __restrict__ items,
                        int chunk, int items_cap) {
  int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (ncl_dev) ncl = *ncl_dev;
  if (c >= ncl) return;
  const int n = count[c], e = estart[c];
  int nch = (n + chunk - 1) / chunk;
  for (int k = 0; k < nch; k++) {
    const int it = item_start[c] + k;
    if (it < items_cap) items[it] = make_int4(c, e + k * chunk, e + min(n, (k + 1) * chunk), 0);
  }
}

// the pair kernel's schedule from the items (sched_wave); one thread per item
// writes the first item of each wave it starts.  wave_start has nwaves + 1
// entries; nitems = *nitems_dev when given.
__global__ void k_wave_sched(int nitems, const int* __restrict__ nitems_dev, int items_cap,
                             const int4* __restrict__ items, int nwaves, int* __restrict__ wave_start) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (nitems_dev) nitems = min(*nitems_dev, items_cap);
  if (nitems == 0) {
    for (int w = i; w <= nwaves; w += gridDim.x * blockDim.x) wave_start[w] = 0;
    return;
  }
  if (i >= nitems) return;
  const long long total = (long long)items[nitems - 1].z + (long long)kItemCost * nitems;
  auto wave_of = [&](int q) { return sched_wave(items[q].y, q, total, nwaves); };
  const int wi = wave_of(i);
  const int wp = i == 0 ? -1 : wave_of(i - 1);
  for (int w = wp + 1; w <= wi; w++) wave_start[w] = i;
  if (i == nitems - 1)
    for (int w = wi + 1; w <= nwaves; w++) wave_start[w] = nitems;
}

// ------------------------------------------------------------------------
// per-step kernels
// ------------------------------------------------------------------------

// k_pack and k_bbox in one pass: one thread per slot, the 8 slots of a
// cluster are 8 adjacent lanes, which reduce the cluster's box by shuffles.
// Positions relative to the cluster origin, times pscale (pack_scale).
struct PackSide {
  int nslot;
  const int* slot_loc;
  const int4* slot_img;
  int off;
  const SysArg* sys;
  const double4* origin;
  float4 *out, *bb;
};
__device__ __forceinline__ void pack_bbox(int blk, int nslot, const int* __restrict__ slot_loc,
                                          const int4* __restrict__ slot_img, const double* __restrict__ pos,
                                          int off, const SysArg* __restrict__ sys,
                                          const double4* __restrict__ origin,
                                          float4* __restrict__ out, float4* __restrict__ bb, double pscale) {
  const int s = blk * blockDim.x + threadIdx.x;
  // whole groups of 8 lanes stay together (nslot is a multiple of 8)
  if (s >= nslot) return;
  const int a = slot_loc[s];
  float4 q;
  float lo[3], hi[3];
  if (a < 0) {
    q = make_float4(1.0e5f + 1.0e3f * (float)(s & 1023), 1.0e5f + 1.0e3f * (float)((s >> 10) & 1023),
                    1.0e5f + 1.0e3f * (float)(s >> 20), __int_as_float(-1));
    lo[0] = lo[1] = lo[2] = FLT_MAX;
    hi[0] = hi[1] = hi[2] = -FLT_MAX;
  } else {
    const SysArg& S = *sys;
    const int4 m = slot_img[s];
    const double4 o = origin[s / CL];
    const double* x = pos + 3 * (size_t)(off + a);
    double w[3];
    for (int d = 0; d < 3; d++) w[d] = x[d] - (m.x * S.a[0 * 3 + d] + m.y * S.a[1 * 3 + d] + m.z * S.a[2 * 3 + d]);
    q = make_float4((float)((w[0] - o.x) * pscale), (float)((w[1] - o.y) * pscale), (float)((w[2] - o.z) * pscale),
                    __int_as_float(off + a));
    lo[0] = hi[0] = q.x;
    lo[1] = hi[1] = q.y;
    lo[2] = hi[2] = q.z;
  }
  out[s] = q;
  for (int o = 1; o < CL; o <<= 1) {
    for (int d = 0; d < 3; d++) {
      lo[d] = fminf(lo[d], __shfl_xor(lo[d], o, 64));
      hi[d] = fmaxf(hi[d], __shfl_xor(hi[d], o, 64));
    }
  }
  if ((s & (CL - 1)) == 0) {
    const int c = s / CL;
    bb[2 * c] = make_float4(0.5f * (lo[0] + hi[0]), 0.5f * (lo[1] + hi[1]), 0.5f * (lo[2] + hi[2]), 0.f);
    bb[2 * c + 1] = make_float4(0.5f * (hi[0] - lo[0]), 0.5f * (hi[1] - lo[1]), 0.5f * (hi[2] - lo[2]), 0.f);
  }
}

__global__ __launch_bounds__(256) void k_pack_bbox(Two<PackSide> T, const double* pos, double pscale) {
  const int d = T.side();
  const PackSide& P = T.s[d];
  pack_bbox(T.block(d), P.nslot, P.slot_loc, P.slot_img, pos, P.off, P.sys, P.origin, P.out, P.bb, pscale);
}

// The FP64 helpers below take the reference's rounding: no fused
// multiply-add contraction (the reference's host build has none).  (The sums of
// the FP64 pair loops take fma() where it stands, pair64.)
#pragma clang fp contract(off)

// Tools::pbc (Tools.h:547-570)
__device__ __forceinline__ double pbc1(double x) {
  x += 100.0;
  return (x >= 0) ? x - (double)(int)(x + 0.5) : x - (double)(int)(x - 0.5);
}

// Pbc::distance (Pbc.cpp:362-415)
__device__ void pbc_distance(const PbcArg& P, const double* a, const double* b, double* d) {
  d[0] = b[0] - a[0];
  d[1] = b[1] - a[1];
  d[2] = b[2] - a[2];
  if (P.type == 1) {
    for (int i = 0; i < 3; i++) d[i] = pbc1(d[i] * P.inv[4 * i]) * P.box[4 * i];
  } else if (P.type == 2) {
    double s[3];
    for (int j = 0; j < 3; j++) s[j] = d[0] * P.ired[j] + d[1] * P.ired[3 + j] + d[2] * P.ired[6 + j];
    for (int j = 0; j < 3; j++) s[j] = pbc1(s[j]);
    for (int j = 0; j < 3; j++) d[j] = s[0] * P.red[j] + s[1] * P.red[3 + j] + s[2] * P.red[6 + j];
    if (fabs(s[0]) + fabs(s[1]) + fabs(s[2]) > 0.5) {
      int oct = (s[0] > 0 ? 4 : 0) + (s[1] > 0 ? 2 : 0) + (s[2] > 0 ? 1 : 0);
      double best[3] = {d[0], d[1], d[2]};
      double lbest = best[0] * best[0] + best[1] * best[1] + best[2] * best[2];
      for (int k = 0; k < P.nshift[oct]; k++) {
        double t0 = d[0] + P.shifts[oct][k][0], t1 = d[1] + P.shifts[oct][k][1], t2 = d[2] + P.shifts[oct][k][2];
        double lt = t0 * t0 + t1 * t1 + t2 * t2;
        if (lt < lbest) {
          lbest = lt;
          best[0] = t0;
          best[1] = t1;
          best[2] = t2;
        }
      }
      d[0] = best[0];
      d[1] = best[1];
      d[2] = best[2];
    }
  }
}

#pragma clang fp contract(fast)

// ------------------------------------------------------------------------
// cross-lane sums on the VALU (no LDS): DPP rotations inside 16-lane rows,
// v_permlane16_swap / v_permlane32_swap across rows
// ------------------------------------------------------------------------
template <int CTRL>
__device__ __forceinline__ float dpp_f(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, false));
}
constexpr int kQuadXor1 = 0xB1, kQuadXor2 = 0x4E;  // quad_perm 1,0,3,2 and 2,3,0,1
constexpr int kRor1 = 0x121, kRor2 = 0x122, kRor4 = 0x124, kRor8 = 0x128;

// v[l] + v[l ^ 16]: odd 16-lane rows of one copy swap with even rows of the other
__device__ __forceinline__ float xor16_sum(float v) {
  const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(p[0]) + __uint_as_float(p[1]);
}
// v[l] + v[l ^ 32]
__device__ __forceinline__ float xor32_sum(float v) {
  const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(p[0]) + __uint_as_float(p[1]);
}
// the same moves for a double (both halves take the same path)
template <int CTRL>
__device__ __forceinline__ double dpp_d(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(b & 0xffffffffll), CTRL, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xF, 0xF, false);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
__device__ __forceinline__ double xor16_sum_d(double v) {
  const long long b = __double_as_longlong(v);
  const auto pl = __builtin_amdgcn_permlane16_swap((unsigned)(b & 0xffffffffll), (unsigned)(b & 0xffffffffll), false,
                                                   false);
  const auto ph = __builtin_amdgcn_permlane16_swap((unsigned)(b >> 32), (unsigned)(b >> 32), false, false);
  const double x = __longlong_as_double(((long long)ph[0] << 32) | pl[0]);
  const double y = __longlong_as_double(((long long)ph[1] << 32) | pl[1]);
  return x + y;
}
__device__ __forceinline__ double xor32_sum_d(double v) {
  const long long b = __double_as_longlong(v);
  const auto pl = __builtin_amdgcn_permlane32_swap((unsigned)(b & 0xffffffffll), (unsigned)(b & 0xffffffffll), false,
                                                   false);
  const auto ph = __builtin_amdgcn_permlane32_swap((unsigned)(b >> 32), (unsigned)(b >> 32), false, false);
  const double x = __longlong_as_double(((long long)ph[0] << 32) | pl[0]);
  const double y = __longlong_as_double(((long long)ph[1] << 32) | pl[1]);
  return x + y;
}
// sum over the 64 lanes of a double, without LDS (the value of lane 0 is used)
__device__ __forceinline__ double wave_sum_d(double v) {
  v += dpp_d<kRor8>(v);
  v += dpp_d<kRor4>(v);
  v += dpp_d<kRor2>(v);
  v += dpp_d<kRor1>(v);
  return xor32_sum_d(xor16_sum_d(v));
}

// sum over the 8 lanes l, l^8, l^16, ..., l^56 (lane = ii + 8 jj: the sum over jj)
__device__ __forceinline__ float sum_over_jj(float v) {
  v += dpp_f<kRor8>(v);
  return xor32_sum(xor16_sum(v));
}
// the same sum of three values at once, component jj3_component(lane) in each lane
// (the lanes keep half of the values at the first step and of those left at the
// second: the same additions in half of the instructions, and one store of three
// lanes an atom; 48 systems 730 -> 715 us, 50,000 atoms 38.2 -> 37.3)
__device__ __forceinline__ float sum_over_jj3(float x, float y, float z, int lane) {
  const bool b3 = lane & 8;
  const float u = (b3 ? z : x) + dpp_f<kRor8>(b3 ? x : z);
  const float v = (b3 ? 0.f : y) + dpp_f<kRor8>(b3 ? y : 0.f);
  // even 16-lane rows keep u, odd ones v
  const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(u), __float_as_uint(v), false, false);
  return xor32_sum(__uint_as_float(p[0]) + __uint_as_float(p[1]));
}
// 0, 1, 2 (lanes 0-7, 16-23, 8-15: one of each per atom ii); 3: no component
__device__ __forceinline__ int jj3_component(int lane) {
  return lane >= 32 ? 3 : ((lane & 8) ? ((lane & 16) ? 3 : 2) : (lane >> 4));
}
// sum over the 64 lanes, in every lane
__device__ __forceinline__ float wave_sum_f(float v) {
  v += dpp_f<kRor8>(v);
  v += dpp_f<kRor4>(v);
  v += dpp_f<kRor2>(v);
  v += dpp_f<kRor1>(v);
  return xor32_sum(xor16_sum(v));
}
// value of lane l (uniform)
__device__ __forceinline__ float readlane_f(float v, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
// number of set bits of m in the lanes below this one (v_mbcnt)
__device__ __forceinline__ int bits_below(unsigned long long m) {
  return (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
}

// ------------------------------------------------------------------------
// the pair kernel
// ------------------------------------------------------------------------

// FP32 switch value and derivative factor of fixedRational<2P> on r^2
// without its stretch: sv = 1/(1+x^P) and dfu = x^(P-1) sv^2 with x = r^2/r0^2.
// The stretched value is stretch*sv + shift and dfunc = -2P/r0^2 stretch dfu
// (SwitchingFunction.cpp:203-215); both factors are applied once per work
// item, in FP64 (PairArgs::sv_scale, sv_shift, df_scale, vir_scale).  The
// cluster positions of these switches are stored in units of R_0 (x = r^2).
template <int P>
__device__ __forceinline__ void sw_fixed(float invr0_2, float r2, float& sv, float& dfu) {
  const float x = r2 * invr0_2;
  float xp = 1.0f;
#pragma unroll
  for (int k = 1; k < P; k++) xp *= x;  // x^(P-1)
  const float res = __builtin_amdgcn_rcpf(fmaf(xp, x, 1.0f));
  sv = res;
  dfu = xp * res * res;
}

// x for a pair outside the cut: x^(P-1) stays finite and 1 + x^P overflows,
// so that sv = 1/(1+x^P) and dfu = x^(P-1) sv^2 are exactly 0 (x = 2^ceil(128/P))
template <int P>
__device__ __forceinline__ constexpr float sw_far() {
  return P == 1 ? __builtin_huge_valf()
                : (P == 2 ? 0x1p64f : (P == 3 ? 0x1p43f : (P == 4 ? 0x1p32f : (P == 5 ? 0x1p26f : 0x1p22f))));
}
static_assert(sw_far<6>() == 0x1p22f, "far values cover P <= 6");

template <int P>
__device__ __forceinline__ void sw_fixed_x(float x, float& sv, float& dfu) {
  float xp = 1.0f;
#pragma unroll
  for (int k = 1; k < P; k++) xp *= x;
  const float res = __builtin_amdgcn_rcpf(fmaf(xp, x, 1.0f));
  sv = res;
  dfu = xp * res * res;
}

template <int P>
__device__ __forceinline__ float sw_fixed_value_x(float x) {
  float xp = 1.0f;
#pragma unroll
  for (int k = 1; k < P; k++) xp *= x;
  return __builtin_amdgcn_rcpf(fmaf(xp, x, 1.0f));
}

// band records a wave holds in LDS at once: the band pairs of an item are
// decided in rounds of this many (one per lane)
constexpr int kBandSlots = 64;

struct PairArgs {
  int nitems, items_cap, ent_cap;  // row kernel: items, capacities of the item and entry arrays
  int share;              // the two groups have atoms in common (twinI tells them)
  float dmax2, prune2, band;
  float cut_lo, cut_hi;   // FP32 r^2 at or below cut_lo: inside; in (cut_lo, cut_hi): the band
  float contact2;         // FP32 r^2 of DBL_EPSILON (the contact-matrix rule)
  float invr0_2;          // FP32 constant of fixedRational (1: positions in units of R_0)
  double r2_real;         // FP32 r^2 -> squared distance (generic switches)
  double sv_scale, sv_shift, df_scale, vir_scale;  // per-item FP32 sums -> outputs
  p2a_switch sw;          // FP64 parameters (generic switch and the cut band)
  const PbcArg* pbc;      // device copies of the prepared cells (FP64 cut decisions)
  const int* cl_sys;      // system of each i cluster (null: one system)
  const double* pos64;    // FP64 positions of the requested atoms (band pairs)
  // Value, six virial products and pair count: with item_partials every item
  // writes its own row of ipart; otherwise every workgroup writes one row of
  // `partial` over all of its items.
  int item_partials;
  double* ipart;
  // when set and *skip != 0 (written by an earlier kernel on the stream), the
  // launch does nothing: a pass queued on a list that may be stale
  const int* skip;
};

// FP64 re-evaluation of the squared distance of one pair, used only when the
// FP32 value lies within a narrow band around D_MAX^2: the inclusive cut of
// the reference is then decided on the distance Pbc::distance itself would
// produce from the raw positions (including the rounding of Tools::pbc).
// The pair is oriented as the reference lists it (GROUPA atom first; lower
// index first inside one group) because the rounding of Tools::pbc is not
// symmetric under d -> -d.
__device__ double exact_r2(const PbcArg* __restrict__ P, const double* __restrict__ pos, int reqi, int reqj) {
#pragma clang fp contract(off)
  double d[3];
  const int a = min(reqi, reqj), b = max(reqi, reqj);
  pbc_distance(*P, pos + 3 * (size_t)a, pos + 3 * (size_t)b, d);
  return d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
}

// per-lane FP32 sums of one work item: sv (counted pairs), dfu * d (i
// derivative), dfu * d (x) d (virial, counted pairs)
struct PairAcc {
  float sv, fx, fy, fz, vxx, vxy, vxz, vyy, vyz, vzz;
};

// entries a wave holds in LDS: those of an item, each kind from a multiple of
// 8 and rounds by two, and two rounds of reading ahead
template <int CH>
constexpr int sent_cap() {
  return (CH / CL + 2 + 2) * CL;
}

// The wave's LDS areas for one work item.  A staged j atom is 16 B: its
// position in the i cluster's frame and, in w, its requested index (-1 for
// padding), so that one read serves the pair, the test for an atom's pair with
// itself (TWO) and the band decisions.
struct WaveLds {
  float4* sj;
  Entry* se;    // the item's entries within D_MAX, counting ones first
  // band records of the current round (kBandSlots), once the item is staged
  __device__ __forceinline__ int* sr() const { return (int*)se; }
};

// a band record: staged index (bits 0-9), i slot (10-12), kind (13-14)
__device__ __forceinline__ int band_record(int staged, int ii, int kind) {
  return staged | (ii << 10) | (kind << 13);
}

// A switch other than fixedRational with its type known at compile time
// (P2A_SW_*; kSwFastRational: RATIONAL of even exponents on r^2), FP64, for a
// pair inside D_MAX.  Against switch_calc_sqr, whose type is a variable: one
// reciprocal square root in place of a square root and a division, and no
// code of the other types held in the kernel (together they took 560 spilled
// registers in the pair kernel).
constexpr int kSwFastRational = 100;
template <int K>
__device__ __forceinline__ double switch_known(const p2a_switch& sw, double d2, double& dfunc) {
#pragma clang fp contract(off)
  if constexpr (K == kSwFastRational) {
    double f, df;
    rational_core(sw, d2 * sw.invr0_2, sw.preSecDevF, sw.nnf, sw.mmf, sw.preDfuncF, sw.preRes, f, df);
    df *= 2 * sw.invr0_2;
    dfunc = df * sw.stretch;
    return f * sw.stretch + sw.shift;
  } else if constexpr (K == P2A_SW_FASTGAUSSIAN) {
    // switch_calc_sqr at zero distance: 1, without stretch and shift
    const double e = exp_core(-0.5 * d2);
    dfunc = d2 > 0.0 ? -e * sw.stretch : 0.0;
    return d2 > 0.0 ? e * sw.stretch + sw.shift : 1.0;
  } else {
    const double ir = rsqrt64(d2);
    const double r = d2 > 0.0 ? d2 * ir : 0.0;
    if constexpr (K == P2A_SW_Q) {
      if (!(r > sw.d0)) {
        dfunc = 0.0;
        return sw.stretch + sw.shift;
      }
      const double e = exp(sw.beta * (r - sw.lambda * sw.ref));
      const double s = 1.0 / (1.0 + e);
      dfunc = -sw.beta / (e + 2.0 + 1.0 / e) * ir * sw.stretch;
      return s * sw.stretch + sw.shift;
    } else {
      const double rdist = (r - sw.d0) * sw.invr0;
      if (!(rdist > 0.0)) {
        dfunc = 0.0;
        return sw.stretch + sw.shift;
      }
      double f, df;
      if constexpr (K == P2A_SW_EXP) {
        f = exp_core(-rdist);
        df = -f;
      } else if constexpr (K == P2A_SW_GAUSSIAN) {
        f = exp_core(-0.5 * rdist * rdist);
        df = -rdist * f;
      } else if constexpr (K == P2A_SW_RATIONAL) {
        rational_core(sw, rdist, sw.preSecDev, sw.nn, sw.mm, sw.preDfunc, sw.preRes, f, df);
      } else {
        p2a_switch t = sw;
        t.type = K;
        base_function(t, rdist, f, df);
      }
      dfunc = df * sw.stretch * sw.invr0 * ir;
      return f * sw.stretch + sw.shift;
    }
  }
}

// FP32 switch terms of one pair on its FP32 r^2.  GENERIC: P is the switch's
// type for switch_known, 0 for any switch.
template <int P, bool GENERIC>
__device__ __forceinline__ void pair_switch(const PairArgs& A, float r2, float& sv, float& dfu) {
  if constexpr (GENERIC) {
    double dfd;
    if constexpr (P == 0) sv = (float)switch_calc_sqr(A.sw, (double)r2 * A.r2_real, dfd);
    else sv = (float)switch_known<P>(A.sw, (double)r2 * A.r2_real, dfd);
    dfu = (float)dfd;
  } else {
    sw_fixed<P>(A.invr0_2, r2, sv, dfu);
  }
}

// FP32 separation and r^2 of staged atom pj from i atom pi (the one sequence
// of operations for a pair in the FP32 pass and in its band decisions)
__device__ __forceinline__ float pair_d(const float4& pj, const float4& pi, float& dx, float& dy, float& dz) {
  dx = pj.x - pi.x;
  dy = pj.y - pi.y;
  dz = pj.z - pi.z;
  return fmaf(dx, dx, fmaf(dy, dy, dz * dz));
}

// whether lane (ii, jj) evaluates its pair in a group of kind KIND; TWO: ai is
// the requested index of atom i in the other group
template <bool TWO, bool VO, int KIND>
__device__ __forceinline__ bool pair_keep(const float4& pj, int ii, int jj, int ai) {
  bool keep = true;
  if constexpr (KIND == 0) keep = jj != ii;  // an atom is not paired with itself
  if constexpr (TWO) keep = keep && (__float_as_int(pj.w) != ai);
  if constexpr (VO && KIND == 0) keep = keep && jj > ii;  // value only: each pair once
  return keep;
}

// One group of 8 staged j atoms against the 8 i atoms of the item: lane
// (ii, jj) takes i = ii, j = staged atom g + jj.  KIND is uniform over the
// group: 0 = the i cluster with itself (slot order), 1 = entries that count
// the pair (value, virial, derivative), 2 = derivative only.
// A pair whose FP32 r^2 lies in the band around D_MAX^2 (cut_lo < r2 <
// cut_hi) is left out here and counted in nrec (uniform); band_terms
// decides the item's band pairs on FP64 distances after the pass.
template <int P, bool GENERIC, bool TWO, bool VO, int KIND>
__device__ __forceinline__ void pair_term(const PairArgs& A, const float4& pj, const float4& pi, int ii, int jj,
                                          int ai, int& nrec, int& npair, PairAcc& acc) {
  float dx, dy, dz;
  const float r2 = pair_d(pj, pi, dx, dy, dz);
  const bool keep = pair_keep<TWO, VO, KIND>(pj, ii, jj, ai);
  // inside D_MAX and outside the band: r2 <= cut_lo; in the band: cut_lo < r2 < cut_hi
  const bool cut = keep && r2 <= A.cut_lo;
  const unsigned long long bcut = __ballot(cut);
  nrec += __popcll(__ballot(keep && r2 < A.cut_hi) & ~bcut);
  // a pair outside the cut gets sv = dfu = 0 from x = sw_far (fixed P) or by selection
  float sv, dfu;
  if constexpr (GENERIC) {
    sv = dfu = 0.f;
    if (cut) pair_switch<P, GENERIC>(A, r2, sv, dfu);
  } else {
    // positions are in units of R_0: x = r^2
    const float x = cut ? r2 : sw_far<P>();
    if constexpr (VO) {
      sv = sw_fixed_value_x<P>(x);
      dfu = 0.f;
    } else {
      sw_fixed_x<P>(x, sv, dfu);
    }
  }
  if constexpr (VO) {
    npair += __popcll(bcut);
    acc.sv += sv;
    return;
  }
  const float gx = dfu * dx, gy = dfu * dy, gz = dfu * dz;
  // derivative of atom i over every partner (the full list holds both
  // orientations of each cluster pair)
  acc.fx += gx;
  acc.fy += gy;
  acc.fz += gz;
  if constexpr (KIND == 1) {
    // value and virial once per unordered pair
    npair += __popcll(bcut);
    acc.sv += sv;
    acc.vxx = fmaf(gx, dx, acc.vxx);
    acc.vxy = fmaf(gx, dy, acc.vxy);
    acc.vxz = fmaf(gx, dz, acc.vxz);
    acc.vyy = fmaf(gy, dy, acc.vyy);
    acc.vyz = fmaf(gy, dz, acc.vyz);
    acc.vzz = fmaf(gz, dz, acc.vzz);
  } else if constexpr (KIND == 0) {
    const bool c2 = cut && (jj > ii);
    const float wgt = c2 ? 1.f : 0.f;
    npair += __popcll(__ballot(c2));
    acc.sv = fmaf(wgt, sv, acc.sv);
    const float hx = wgt * gx, hy = wgt * gy, hz = wgt * gz;
    acc.vxx = fmaf(hx, dx, acc.vxx);
    acc.vxy = fmaf(hx, dy, acc.vxy);
    acc.vxz = fmaf(hx, dz, acc.vxz);
    acc.vyy = fmaf(hy, dy, acc.vyy);
    acc.vyz = fmaf(hy, dz, acc.vyz);
    acc.vzz = fmaf(hz, dz, acc.vzz);
  }
}

// Groups [gb, ge) of one kind (uniform bounds, multiples of 8), two groups per
// trip; each lane's next staged atom is read one group ahead (the staging
// area has spare slots past the last group for that read).
template <int P, bool GENERIC, bool TWO, bool VO, int KIND>
__device__ __forceinline__ void pair_groups(const PairArgs& A, int gb, int ge, const float4& pi, int ii, int jj,
                                            int ai, const WaveLds& L, int& nrec, int& npair, PairAcc& acc) {
  int g = gb;
  float4 pa = L.sj[g + jj];
  for (; g + CL < ge; g += 2 * CL) {
    const float4 pb = L.sj[g + CL + jj];
    pair_term<P, GENERIC, TWO, VO, KIND>(A, pa, pi, ii, jj, ai, nrec, npair, acc);
    pa = L.sj[g + 2 * CL + jj];
    pair_term<P, GENERIC, TWO, VO, KIND>(A, pb, pi, ii, jj, ai, nrec, npair, acc);
  }
  if (g < ge) pair_term<P, GENERIC, TWO, VO, KIND>(A, pa, pi, ii, jj, ai, nrec, npair, acc);
}

// The band test of pair_term again for one group, numbering the band pairs in
// program order: those numbered [r0, r0 + kBandSlots) become the wave's band
// records (one round of band_terms).
template <bool TWO, bool VO, int KIND>
__device__ __forceinline__ void band_collect(const PairArgs& A, const float4& pj, const float4& pi, int ii, int jj, int g,
                                             int ai, const WaveLds& L, int r0, int& cnt) {
  float dx, dy, dz;
  const float r2 = pair_d(pj, pi, dx, dy, dz);
  const bool keep = pair_keep<TWO, VO, KIND>(pj, ii, jj, ai);
  const bool cut = keep && r2 <= A.cut_lo;
  const unsigned long long bm = __ballot(keep && r2 < A.cut_hi) & ~__ballot(cut);
  if (bm != 0ull) {
    if ((bm >> (ii + CL * jj)) & 1ull) {
      const int k = cnt + bits_below(bm) - r0;
      if (k >= 0 && k < kBandSlots) L.sr()[k] = band_record(g + jj, ii, KIND);
    }
    cnt += __popcll(bm);
  }
}

// The band pairs of the staged item, in rounds of kBandSlots (record r in
// lane r, collected by band_collect; the first round also counts them): the
// inclusive cut decided on the reference's Pbc::distance
// (exact_r2), and for the pairs inside, their FP32 terms from the FP32
// pass's r^2, added in record order in FP64: the i atom derivatives to
// fadd[3] (lanes jj == 0, atom ii), the row entries to radd (lane q < 8:
// value, six virial products, pair count).
template <int P, bool GENERIC, bool TWO, bool VO>
__device__ __forceinline__ void band_terms(const PairArgs& A, const WaveLds& L, int ci,
                                           const float4* __restrict__ posI, const float4* __restrict__ posJ,
                                           const float4& pi_lane, int ii, int jj, int lane, int ai, int n0, int b1,
                                           int n1, int b2, int n2, double* fadd, double& radd) {
  const PbcArg* pbc = A.pbc + nsys_of(A.cl_sys, ci);
  int nrec = 0;
  for (int r0 = 0; r0 == 0 || r0 < nrec; r0 += kBandSlots) {
    {
      int cnt = 0;
      if (n0) band_collect<TWO, VO, 0>(A, L.sj[jj], pi_lane, ii, jj, 0, ai, L, r0, cnt);
      for (int g = b1; g < b1 + n1; g += CL) band_collect<TWO, VO, 1>(A, L.sj[g + jj], pi_lane, ii, jj, g, ai, L, r0, cnt);
      if constexpr (!VO)
        for (int g = b2; g < b2 + n2; g += CL)
          band_collect<TWO, VO, 2>(A, L.sj[g + jj], pi_lane, ii, jj, g, ai, L, r0, cnt);
      nrec = cnt;
      // the records are read by other lanes of this wave
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
    const int nr = min(kBandSlots, nrec - r0);
    int rii = 0, cnt = 0;
    float sv = 0.f, g[3] = {0.f, 0.f, 0.f}, d[3] = {0.f, 0.f, 0.f};
    if (lane < nr) {
      const int rec = L.sr()[lane];
      const int st = rec & 1023, kind = (rec >> 13) & 3;
      rii = (rec >> 10) & 7;
      const float4 pi = posI[ci * CL + rii];
      const float r2 = pair_d(L.sj[st], pi, d[0], d[1], d[2]);
      const int reqi = __float_as_int(pi.w);
      const int reqj = __float_as_int(L.sj[st].w);
      if (reqi >= 0 && reqj >= 0 && switch_inside(A.sw, exact_r2(pbc, A.pos64, reqi, reqj))) {
        float dfu;
        pair_switch<P, GENERIC>(A, r2, sv, dfu);
        // as the any-switch kernel (P == 0), whose switch ends at D_MAX
        if (GENERIC && P != 0 && !switch_inside(A.sw, (double)r2 * A.r2_real)) sv = dfu = 0.f;
        if constexpr (!VO) {
          g[0] = dfu * d[0];
          g[1] = dfu * d[1];
          g[2] = dfu * d[2];
        }
        // a self pair counts once: the staged index of a self entry is its slot
        cnt = (kind == 1 || (kind == 0 && st > rii)) ? 1 : 0;
      } else {
        sv = 0.f;
      }
    }
    for (int r = 0; r < nr; r++) {
      const int ri = __builtin_amdgcn_readlane(rii, r);
      const int rc = __builtin_amdgcn_readlane(cnt, r);
      const float rs = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(sv), r));
      float rg[3], rd[3];
      for (int c = 0; c < 3; c++) {
        rg[c] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(g[c]), r));
        rd[c] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(d[c]), r));
      }
      if (!VO && jj == 0 && ii == ri)
        for (int c = 0; c < 3; c++) fadd[c] += -A.df_scale * (double)rg[c];
      if (rc && lane < 8) {
        if (lane == 0) radd += A.sv_scale * (double)rs + A.sv_shift;
        else if (lane == 7) radd += 1.0;
        else if (!VO) {
          const int a = lane <= 3 ? 0 : (lane <= 5 ? 1 : 2);
          const int b = lane <= 3 ? lane - 1 : (lane <= 5 ? lane - 3 : 2);
          radd += A.vir_scale * (double)(rg[a] * rd[b]);
        }
      }
    }
    // the next round overwrites the records
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
}

// Row entry `lane` (< 8) of FP32 per-lane sums: value, six virial products,
// pair count (npair uniform); the wave sums are formed in every lane.
template <bool VO>
__device__ __forceinline__ double item_row(const PairArgs& A, const PairAcc& acc, int npair, int lane) {
  float tv[7];
  tv[0] = wave_sum_f(acc.sv);
  if constexpr (!VO) {
    tv[1] = wave_sum_f(acc.vxx);
    tv[2] = wave_sum_f(acc.vxy);
    tv[3] = wave_sum_f(acc.vxz);
    tv[4] = wave_sum_f(acc.vyy);
    tv[5] = wave_sum_f(acc.vyz);
    tv[6] = wave_sum_f(acc.vzz);
  } else {
    tv[1] = tv[2] = tv[3] = tv[4] = tv[5] = tv[6] = 0.f;
  }
  float tq = tv[0];
#pragma unroll
  for (int q = 1; q < 7; q++)
    if (lane == q) tq = tv[q];
  return lane == 0 ? A.sv_scale * (double)tq + A.sv_shift * (double)npair
                   : (lane < 7 ? A.vir_scale * (double)tq : (double)npair);
}

// The same row entries with one entry per pair of lanes: entry `lane` / 2 in the
// even lanes below 16 (bit 3 of the lane: bit 2 of the entry, and so on).  The
// eight sums share their steps: at each of the first three a lane keeps half of
// its values and adds the partner's (xor 8, 4, 2, then 1, 16, 32: the additions
// of wave_sum_f, so the same bits) in about half of the instructions.
__device__ __forceinline__ double item_row_pairs(const PairArgs& A, const PairAcc& acc, int npair, int lane) {
  const bool b3 = lane & 8, b2 = lane & 4, b1 = lane & 2;
  const float lo[4] = {acc.sv, acc.vxx, acc.vxy, acc.vxz}, hi[4] = {acc.vyy, acc.vyz, acc.vzz, 0.f};
  float a[4], b[2];
#pragma unroll
  for (int k = 0; k < 4; k++) a[k] = (b3 ? hi[k] : lo[k]) + dpp_f<kRor8>(b3 ? lo[k] : hi[k]);
#pragma unroll
  for (int k = 0; k < 2; k++) {
    const float give = b2 ? a[k] : a[k + 2];
    b[k] = (b2 ? a[k + 2] : a[k]) +
           __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(give), 0x101F));  // lane ^ 4
  }
  float v = (b1 ? b[1] : b[0]) + dpp_f<kQuadXor2>(b1 ? b[0] : b[1]);
  v += dpp_f<kQuadXor1>(v);
  v = xor32_sum(xor16_sum(v));
  const int e = (lane >> 1) & 7;
  return e == 0 ? A.sv_scale * (double)v + A.sv_shift * (double)npair
                : (e < 7 ? A.vir_scale * (double)v : (double)npair);
}

// Staging of one work item by one wave (i cluster ci, entries [e0, e1)):
//  1. lane-parallel pruning of the chunk's entries against the current
//     bounding boxes (D_MAX); the entries left go to LDS, compacted, counting
//     ones first, each kind from a multiple of 8;
//  2. in rounds of 8 entries, lane (entry, atom) loads one atom of its entry's
//     j cluster (128 B in a row per cluster), adds the image offset and keeps
//     it if it lies within D_MAX of the i cluster's box; the kept atoms are
//     staged in LDS, compacted in (entry, atom) order and grouped by kind
//     (self / counting / derivative-only), each kind padded to a multiple of 8
//     with far-away atoms, so that every group of 8 has one kind.
// A list radius above D_MAX leaves about half of the entries: 5-6 rounds,
// where one lane per listed entry took 8 loads and tests an item, each load 64
// lines.  The slots of se without an entry hold kNoEntry (their lanes load atoms of
// cluster 0 and keep none, whatever these hold); rounds go by two, the next two's
// loads in flight.
// DENSE: an item of which kDenseEntries entries or more are left (a list without
// a margin over D_MAX) takes one lane per entry, eight loads in flight at once:
// the same order; 48 systems, list radius 1.2 = D_MAX: 759 us, in rounds 803.
constexpr int kDenseEntries = 40;
constexpr int kNoEntry = INT_MIN;  // "diagonal" of cluster 0, which is never staged in rounds
// TWIN (rounds only): also the staged slot of each i atom's twin, the same atom in
// the other group, for staged atoms that do not carry their requested index.
// Returns the group bounds (uniform): n0 (0 or 8), [b1, b1+n1), [b2, b2+n2).
struct Twin {
  const float4* idxJ;  // packed positions with requested indices
  int ai;              // requested index of this lane's i atom in the other group, or -2
  float4 pi;           // its position
  int slot;            // out: staged slot of its twin, -1: not in the item
};
template <bool VO, bool DENSE, int CH, bool TWIN = false>
__device__ __forceinline__ void stage_item(const PairArgs& A, const Entry& my, int lane, int e0, int e1, int ci,
                                           const float4& ic, const float4& ih, const float4* __restrict__ posJ,
                                           const float4* __restrict__ bbJ, const WaveLds& L, int& n0, int& b1,
                                           int& n1, int& b2, int& n2, Twin* T = nullptr) {
  static_assert(!(DENSE && TWIN), "twins are found in the rounds");
  bool pass = false;
  const Entry none = {kNoEntry, 0.f, 0.f, 0.f};
  L.se[lane] = none;
  if (lane < sent_cap<CH>() - WAVE) L.se[WAVE + lane] = none;
  if (lane < CH && e0 + lane < e1 && (!VO || (my.code & kCountBit) || my.code < 0)) {
    const int cj = my.code & kCjMask;
    const float4 jc = bbJ[2 * cj], jh = bbJ[2 * cj + 1];
    const float gx = fmaxf(fabsf(jc.x + my.dx - ic.x) - ih.x - jh.x, 0.f);
    const float gy = fmaxf(fabsf(jc.y + my.dy - ic.y) - ih.y - jh.y, 0.f);
    const float gz = fmaxf(fabsf(jc.z + my.dz - ic.z) - ih.z - jh.z, 0.f);
    pass = fmaf(gz, gz, fmaf(gx, gx, gy * gy)) <= A.prune2;
  }
  const unsigned long long mp = __ballot(pass), md = __ballot(my.code < 0), mc = __ballot((my.code & kCountBit) != 0);
  const unsigned long long m1 = mp & mc & ~md, m2 = VO ? 0ull : mp & ~mc & ~md;
  const int p1 = __popcll(m1), p2 = __popcll(m2);
  if (DENSE && p1 + p2 >= kDenseEntries) {  // uniform over the wave
    float4 q[CL];
    int m8 = 0;
    if (pass) {
      const float4* pj = posJ + (size_t)(my.code & kCjMask) * CL;
#pragma unroll
      for (int t = 0; t < CL; t++) q[t] = pj[t];
#pragma unroll
      for (int t = 0; t < CL; t++) {
        q[t].x += my.dx;
        q[t].y += my.dy;
        q[t].z += my.dz;
        const float gx = fmaxf(fabsf(q[t].x - ic.x) - ih.x, 0.f);
        const float gy = fmaxf(fabsf(q[t].y - ic.y) - ih.y, 0.f);
        const float gz = fmaxf(fabsf(q[t].z - ic.z) - ih.z, 0.f);
        if (fmaf(gz, gz, fmaf(gx, gx, gy * gy)) <= A.prune2) m8 |= 1 << t;
      }
    }
    const bool self = pass && my.code < 0, count = (my.code & kCountBit) != 0;
    if (self) m8 = 0xFF;  // keeps slot order
    n0 = (mp & md) ? CL : 0;
    const int cnt = __popc(m8);
    int tot1, tot2 = 0;
    const int o1 = wave_excl_scan(count && !self ? cnt : 0, tot1);
    int o2 = 0;
    if constexpr (!VO) o2 = wave_excl_scan(count || self ? 0 : cnt, tot2);
    n1 = (tot1 + CL - 1) & ~(CL - 1);
    n2 = (tot2 + CL - 1) & ~(CL - 1);
    b1 = n0;
    b2 = n0 + n1;
    int p = self ? 0 : (count ? b1 + o1 : b2 + o2);
#pragma unroll
    for (int t = 0; t < CL; t++)
      if ((m8 >> t) & 1) L.sj[p++] = q[t];
    if (lane < CL) {
      const float4 far = make_float4(1.0e5f, 1.0e5f, 1.0e5f, __int_as_float(-1));
      if (tot1 + lane < n1) L.sj[b1 + tot1 + lane] = far;
      if (tot2 + lane < n2) L.sj[b2 + tot2 + lane] = far;
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
    return;
  }
  const int r1 = (p1 + CL - 1) / CL, rounds = r1 + (p2 + CL - 1) / CL;
  const int at1 = bits_below(m1), at2 = r1 * CL + bits_below(m2);
  if (pass && my.code >= 0) L.se[(my.code & kCountBit) ? at1 : at2] = my;
  // the i cluster with itself keeps slot order (at most one such entry)
  n0 = (mp & md) ? CL : 0;
  if (n0 && lane < CL) L.sj[lane] = posJ[ci * CL + lane];
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  __builtin_amdgcn_wave_barrier();
  b1 = n0;
  int at = n0;       // next staged slot (uniform)
  n1 = 0;
  const unsigned t16 = (unsigned)(lane & 7) * 16u;
  const Entry* se = L.se + (lane >> 3);
  auto pad = [&]() {
    const int end = (at + CL - 1) & ~(CL - 1);
    if (lane < end - at) L.sj[at + lane] = make_float4(1.0e5f, 1.0e5f, 1.0e5f, __int_as_float(-1));
    at = end;
  };
  // atom lane & 7 of the entry: 128 B a cluster, fewer than 2^25 clusters, so
  // the shift drops the code's other bits and the offset has 32
  auto load = [&](const Entry& e) {
    return *(const float4*)((const char*)posJ + (size_t)(((unsigned)e.code << 7) | t16));
  };
  // the same atom's requested index
  auto load_idx = [&](const Entry& e) {
    return *(const int*)((const char*)T->idxJ + (size_t)(((unsigned)e.code << 7) | t16) + 12);
  };
  int tw[CL];
  if constexpr (TWIN) {
    T->slot = -1;
#pragma unroll
    for (int u = 0; u < CL; u++) tw[u] = __builtin_amdgcn_readlane(T->ai, u);
  }
  auto keep_atom = [&](const Entry& e, float4 q, int idx) {
    q.x += e.dx;
    q.y += e.dy;
    q.z += e.dz;
    const float gx = fmaxf(fabsf(q.x - ic.x) - ih.x, 0.f);
    const float gy = fmaxf(fabsf(q.y - ic.y) - ih.y, 0.f);
    const float gz = fmaxf(fabsf(q.z - ic.z) - ih.z, 0.f);
    const bool keep = e.code >= 0 && fmaf(gz, gz, fmaf(gx, gx, gy * gy)) <= A.prune2;
    const unsigned long long m = __ballot(keep);
    if (keep) L.sj[at + bits_below(m)] = q;
    if constexpr (TWIN) {
      bool any = false;
#pragma unroll
      for (int u = 0; u < CL; u++) any = any || idx == tw[u];
      for (unsigned long long f = __ballot(keep && any); f; f &= f - 1) {
        const int l = __builtin_ctzll(f);
        const float4 ql = make_float4(readlane_f(q.x, l), readlane_f(q.y, l), readlane_f(q.z, l), 0.f);
        float dx, dy, dz;
        // (not one of its images, which lie beyond D_MAX)
        if (T->ai == __builtin_amdgcn_readlane(idx, l) && pair_d(ql, T->pi, dx, dy, dz) <= A.dmax2)
          T->slot = at + __popcll(m & ((1ull << l) - 1));
      }
    }
    at += __popcll(m);
  };
  if (rounds > 0) {
    Entry ea = se[0], eb = se[CL];
    float4 va = load(ea), vb = load(eb);
    int xa = 0, xb = 0;
    if constexpr (TWIN) xa = load_idx(ea), xb = load_idx(eb);
    for (int r = 0; r < rounds; r += 2) {
      const Entry qa = ea, qb = eb;
      const float4 wa = va, wb = vb;
      const int ja = xa, jb = xb;
      ea = se[(r + 2) * CL];
      eb = se[(r + 3) * CL];
      va = load(ea);
      vb = load(eb);
      if constexpr (TWIN) xa = load_idx(ea), xb = load_idx(eb);
      if (r == r1) {
        pad();
        n1 = at - b1;
      }
      keep_atom(qa, wa, ja);
      if (r + 1 == r1) {
        pad();
        n1 = at - b1;
      }
      keep_atom(qb, wb, jb);
    }
  }
  if (rounds == r1 && (rounds & 1) == 0) {
    pad();
    n1 = at - b1;
  } else {
    pad();
  }
  b2 = b1 + n1;
  n2 = at - b2;
  // the staging above is read by other lanes of this wave only
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// staged atoms per wave: 64 entries x 8, padding of two kinds, and the
// one-group read-ahead (the largest group end is 520)
template <int CH>
constexpr int stage_cap() {
  return CH * CL + 2 * CL;
}

// FP32 pass: one wave per work item (i cluster, chunk of <= CH list
// entries); a grid smaller than the item count makes the waves loop over
// items.  Staging (stage_item), then a dense loop over the groups of 8
// staged atoms: lane l evaluates the pair (i = l&7 of cluster ci, j = staged
// atom 8g + (l>>3)).  VO (value only): no derivatives and no virial;
// derivative-only entries are skipped, so each unordered pair is visited
// once.  TWO: the groups share atoms.  The pairs in the band around D_MAX^2
// (rare) are decided at the end of their item on FP64 distances, from the
// staged atoms.
// Outputs: fpart[item][8][3], the derivative of each i atom over the item,
// and the value / virial / pair count rows described at PairArgs, all over
// the pairs outside the band plus the FP64 terms of the band pairs inside
// the cut (band_terms).  For the workgroup rows each lane keeps FP32 running
// sums over all of the wave's items; their wave sums are taken once at the
// end, converted to FP64 and added to the wave's band sums, and the waves'
// rows are added in wave order.
// Bound by VALU issue (16.5 M instructions a launch at 50,000 atoms, 18.1 M when
// every listed entry was staged).  Known rational 6-12, 50,000 atoms: 37 us
// (41 before); EXP, 20,000 atoms: 60 us.
template <int P, bool GENERIC, bool TWO, bool VO, int CH>
__device__ __forceinline__ void pairs_body(
    const PairArgs& A, int grid_block, int grid, int nitems, int ent_cap, const int* __restrict__ wave_start,
    const int4* __restrict__ items, const Entry* __restrict__ ents, const float4* __restrict__ posI,
    const float4* __restrict__ posJ, const float4* __restrict__ bbI, const float4* __restrict__ bbJ,
    const int* __restrict__ twinI, double* __restrict__ fpart, double* __restrict__ partial) {
  constexpr int NW = PAIR_BLOCK / WAVE;
  constexpr int CAP = stage_cap<CH>();
  __shared__ float4 sj[NW][CAP];
  __shared__ Entry sent[NW][sent_cap<CH>()];
  __shared__ double stot[NW][8];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int ii = lane & 7, jj = lane >> 3;
  const WaveLds L = {sj[w], sent[w]};
  PairAcc acc = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  int ntot = 0;
  // lanes < 8: the wave's FP64 sums of the band pairs' row entries
  if (lane < 8) stot[w][lane] = 0.0;

  // the next item's descriptor and entries are loaded while the current item
  // computes (a wave handles several items when the grid is persistent)
  // the wave's items: a contiguous range of balanced cost, or every
  // (grid waves)-th item
  const int blk = xcd_block(grid_block, grid);
  const int gw = blk * NW + w;
  int kfirst = gw, kstride = grid * NW, kend = nitems;
  if (wave_start) {
    kfirst = wave_start[gw];
    kend = min(wave_start[gw + 1], nitems);
    kstride = 1;
  }
  int k = kfirst;
  int4 it_n = make_int4(0, 0, 0, 0);
  Entry my_n = {0, 0.f, 0.f, 0.f};
  if (k < kend) {
    it_n = items[k];
    const int e = it_n.y + lane;
    if (lane < CH && e < min(it_n.z, ent_cap)) my_n = ents[e];
  }
  for (; k < kend; k += kstride) {
    const int item = k;
    const int4 it = it_n;
    const Entry my_e = my_n;
    const int kn = k + kstride;
    if (kn < kend) it_n = items[kn];
    const int ci = it.x;
    const int e1 = min(it.z, ent_cap);
    const float4 pi = posI[ci * CL + ii];
    const int ai = TWO ? twinI[ci * CL + ii] : 0;
    const float4 ic = bbI[2 * ci], ih = bbI[2 * ci + 1];
    int n0, b1, n1, b2, n2;
    stage_item<VO, true, CH>(A, my_e, lane, it.y, e1, ci, ic, ih, posJ, bbJ, L, n0, b1, n1, b2, n2);
    if (kn < kend) {
      const int e = it_n.y + lane;
      my_n = (lane < CH && e < min(it_n.z, ent_cap)) ? ents[e] : Entry{0, 0.f, 0.f, 0.f};
    }
    // group bounds are wave-uniform: scalar loops
    n1 = __builtin_amdgcn_readfirstlane(n1);
    n2 = __builtin_amdgcn_readfirstlane(n2);
    b1 = __builtin_amdgcn_readfirstlane(b1);
    b2 = __builtin_amdgcn_readfirstlane(b2);
    int nrec = 0, npair = 0;
    // the pair loops issue ahead of the other waves' staging and item ends
    // (measured: the pass takes ~3% less time than with one priority)
    __builtin_amdgcn_s_setprio(1);
    if (n0) pair_term<P, GENERIC, TWO, VO, 0>(A, L.sj[jj], pi, ii, jj, ai, nrec, npair, acc);
    pair_groups<P, GENERIC, TWO, VO, 1>(A, b1, b1 + n1, pi, ii, jj, ai, L, nrec, npair, acc);
    if constexpr (!VO)
      pair_groups<P, GENERIC, TWO, VO, 2>(A, b2, b2 + n2, pi, ii, jj, ai, L, nrec, npair, acc);
    __builtin_amdgcn_s_setprio(0);
    double fadd[3] = {0.0, 0.0, 0.0}, radd = 0.0;
    if (nrec > 0)
      band_terms<P, GENERIC, TWO, VO>(A, L, ci, posI, posJ, pi, ii, jj, lane, ai, n0, b1, n1, b2, n2, fadd, radd);
    if constexpr (!VO) {
      const float f = sum_over_jj3(acc.fx, acc.fy, acc.fz, lane);
      const int c = jj3_component(lane);
      double add = 0.0;
      if (nrec > 0) {  // uniform, rare
        const double a0 = __shfl(fadd[0], ii, WAVE), a1 = __shfl(fadd[1], ii, WAVE), a2 = __shfl(fadd[2], ii, WAVE);
        add = c == 0 ? a0 : (c == 1 ? a1 : a2);
      }
      if (c < 3) fpart[(size_t)item * (CL * 3) + ii * 3 + c] = -A.df_scale * (double)f + add;
      acc.fx = acc.fy = acc.fz = 0.f;
    }
    if (A.item_partials) {
      if constexpr (VO) {
        const double o = item_row<VO>(A, acc, npair, lane);
        if (lane < 8) A.ipart[(size_t)item * 8 + lane] = o + radd;
      } else {
        double o = item_row_pairs(A, acc, npair, lane);
        if (nrec > 0) o += __shfl(radd, (lane >> 1) & 7, WAVE);
        if (lane < 16 && !(lane & 1)) A.ipart[(size_t)item * 8 + (lane >> 1)] = o;
      }
      acc = PairAcc{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    } else {
      // value and virial stay in the lanes' running sums over the wave's items
      ntot += npair;
      if (nrec > 0 && lane < 8) stot[w][lane] += radd;
    }
    // the next item overwrites the staging read above
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
  if (!A.item_partials) {
    const double o = item_row<VO>(A, acc, ntot, lane);
    if (lane < 8) stot[w][lane] += o;
    __syncthreads();
    if (w == 0 && lane < 8) {
      double s = 0.0;
      for (int v = 0; v < NW; v++) s += stot[v][lane];
      partial[(size_t)blk * 8 + lane] = s;
    }
  }
}

struct PairSide {
  int grid, nitems;
  const int* nitems_dev;   // device item count (null: nitems)
  int items_cap, ent_cap;  // capacities of the item and entry arrays
  // Items of each wave of the grid: [wave_start[g], wave_start[g + 1]) for
  // wave g = xcd_block * 4 + wave (sched_wave); null: items g, g + waves, ...
  const int* wave_start;
  const int4* items;
  const Entry* ents;
  const float4 *posI, *posJ, *bbI, *bbJ;
  const int* twinI;
  double *fpart, *partial;
};
// both directions of two groups in one launch: the second one's workgroups start
// as the first one's end (10,000 x 490,000 atoms: 72 us, one after the other 76;
// 1,000 x 1,000: 10, 19)
template <int P, bool GENERIC, bool TWO, bool VO, int CH>
__global__ __launch_bounds__(PAIR_BLOCK) __attribute__((amdgpu_waves_per_eu(4))) void k_pairs(PairArgs A,
                                                                                             Two<PairSide> T) {
  if (A.skip && *A.skip) return;
  const int d = T.side();
  const PairSide& S = T.s[d];
  const int nitems = S.nitems_dev ? min(*S.nitems_dev, S.items_cap) : S.nitems;
  pairs_body<P, GENERIC, TWO, VO, CH>(A, T.block(d), S.grid, nitems, S.ent_cap, S.wave_start, S.items, S.ents, S.posI,
                                      S.posJ, S.bbI, S.bbJ, S.twinI, S.fpart, S.partial);
}

// virial = -sum dd (x) d (CoordinationBase.cpp:200-206), symmetric
__device__ __forceinline__ void write_virial(double* virial, const double* s6) {
  double xx = -s6[0], xy = -s6[1], xz = -s6[2], yy = -s6[3], yz = -s6[4], zz = -s6[5];
  virial[0] = xx; virial[1] = xy; virial[2] = xz;
  virial[3] = xy; virial[4] = yy; virial[5] = yz;
  virial[6] = xz; virial[7] = yz; virial[8] = zz;
}

// Inputs of the final value / virial / pair-count sum: the workgroup rows of
// the pair kernels.
struct RedArgs {
  int nred;
  const double* partial;
  double* value;
  double* virial;
  double* stats;
  const int* skip;  // as PairArgs::skip
};

// After the pair kernels, in one launch.  With do_red, workgroup 0 forms the
// value, virial and pair count from the rows of R in a fixed order (each
// thread a fixed set of rows, then a fixed tree); the other
// workgroups form the derivatives of the atoms of every i cluster (fixed-order
// sums of the cluster's item partials).  The reduction workgroup comes first
// so that it starts with the first wave of workgroups.
struct GatherSide {
  int ncl;
  const int* ncl_dev;
  const float4* p;
  const int* item_start;
  int items_cap;
  const double* fpart;
};
__device__ __forceinline__ void gather_atoms(int blk, const GatherSide& G, double* __restrict__ deriv) {
  const float4* __restrict__ p = G.p;
  const int* __restrict__ item_start = G.item_start;
  const double* __restrict__ fpart = G.fpart;
  const int items_cap = G.items_cap;
  const int ncl = G.ncl_dev ? *G.ncl_dev : G.ncl;
  const int g = blk * blockDim.x + threadIdx.x;
  if (g >= ncl * CL * 3) return;
  const int c = g / (CL * 3), r = g % (CL * 3);
  // every load that depends only on c goes out before the first wait
  const int i0 = item_start[c];
  const int i1 = min(item_start[c + 1], items_cap);
  const int req = __float_as_int(p[c * CL + r / 3].w);
  if (req < 0) return;
  double sum = 0.0;
  for (int it = i0; it < i1; it += 4) {
    double v[4];
#pragma unroll
    for (int u = 0; u < 4; u++) v[u] = it + u < i1 ? fpart[(size_t)(it + u) * (CL * 3) + r] : 0.0;
#pragma unroll
    for (int u = 0; u < 4; u++) sum += v[u];
  }
  deriv[3 * (size_t)req + r % 3] = sum;
}
__global__ __launch_bounds__(256) void k_gather_reduce(Two<GatherSide> T, double* __restrict__ deriv, int do_red,
                                                       RedArgs R) {
  if (R.skip && *R.skip) return;
  const int t = threadIdx.x;
  const int red = do_red ? 1 : 0;
  if ((int)blockIdx.x >= red) {
    if (!deriv) return;
    const int blk = (int)blockIdx.x - red, d = blk >= T.n0 ? 1 : 0;
    gather_atoms(blk - (d ? T.n0 : 0), T.s[d], deriv);
    return;
  }
  __shared__ double s[8][4];
  double acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  const double4* p4 = reinterpret_cast<const double4*>(R.partial);
  // rows t, t + 256, t + 512, ... of each thread, eight in flight at once
  for (int i0 = t; i0 < R.nred; i0 += 256 * 8) {
    double4 x[8], y[8];
#pragma unroll
    for (int u = 0; u < 8; u++) {
      const int i = i0 + u * 256;
      if (i < R.nred) {
        x[u] = p4[2 * (size_t)i];
        y[u] = p4[2 * (size_t)i + 1];
      } else {
        x[u] = make_double4(0.0, 0.0, 0.0, 0.0);
        y[u] = x[u];
      }
    }
#pragma unroll
    for (int u = 0; u < 8; u++) {
      acc[0] += x[u].x; acc[1] += x[u].y; acc[2] += x[u].z; acc[3] += x[u].w;
      acc[4] += y[u].x; acc[5] += y[u].y; acc[6] += y[u].z; acc[7] += y[u].w;
    }
  }
  // wave sums on the VALU, then the four waves in order
#pragma unroll
  for (int q = 0; q < 8; q++) acc[q] = wave_sum_d(acc[q]);
  if ((t & 63) == 0)
    for (int q = 0; q < 8; q++) s[q][t >> 6] = acc[q];
  __syncthreads();
  if (t == 0) {
    double r[8];
    for (int q = 0; q < 8; q++) r[q] = ((s[q][0] + s[q][1]) + s[q][2]) + s[q][3];
    if (R.value) *R.value = r[0];
    if (R.virial) {
      double v6[6] = {r[1], r[2], r[3], r[4], r[5], r[6]};
      write_virial(R.virial, v6);
    }
    if (R.stats) {
      R.stats[0] = r[7];
      R.stats[1] += r[7];  // running total since the last reset
    }
  }
}

__global__ void k_finalize(int nitems, const double* __restrict__ partial, double* __restrict__ value,
                           double* __restrict__ virial, double* __restrict__ stats_out) {
  __shared__ double s[8][128];
  const int t = threadIdx.x;
  double acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  for (int i = t; i < nitems; i += 128)
    for (int q = 0; q < 8; q++) acc[q] += partial[(size_t)i * 8 + q];
  for (int q = 0; q < 8; q++) s[q][t] = acc[q];
  __syncthreads();
  for (int o = 64; o > 0; o >>= 1) {
    if (t < o)
      for (int q = 0; q < 8; q++) s[q][t] += s[q][t + o];
    __syncthreads();
  }
  if (t == 0) {
    if (value) *value = s[0][0];
    if (virial) {
      double v6[6] = {s[1][0], s[2][0], s[3][0], s[4][0], s[5][0], s[6][0]};
      write_virial(virial, v6);
    }
    if (stats_out) {
      stats_out[0] = s[7][0];
      stats_out[1] += s[7][0];  // running total since the last reset
    }
  }
}

// After the pair kernel of a batch, in one launch: the first nsys workgroups form
// the value, virial and pair count of one system each (the items of a system are
// those of its clusters, contiguous after its columns; lane (row, entry), 16 rows
// in flight, then a fixed tree), the others the derivatives of the atoms.  The
// few workgroups of the sums wait for memory, the many of the derivatives move
// it: one after the other 43 + 55 us (48 systems, 500,000 atoms), together 61 us.
__global__ __launch_bounds__(256) void k_gather_systems(int nsys, const int* __restrict__ sys_colbase,
                                                        const int* __restrict__ col_cl,
                                                        const double* __restrict__ partial,
                                                        double* __restrict__ values, double* __restrict__ virials,
                                                        double* __restrict__ npairs, GatherSide G,
                                                        double* __restrict__ deriv) {
  if ((int)blockIdx.x >= nsys) {
    if (deriv) gather_atoms((int)blockIdx.x - nsys, G, deriv);
    return;
  }
  __shared__ double s[8][4];
  const int sy = blockIdx.x;
  const int t = threadIdx.x, q = t & 7;
  const int c0 = col_cl[sys_colbase[sy]], c1 = col_cl[sys_colbase[sy + 1]];
  const int i0 = min(G.item_start[c0], G.items_cap), i1 = min(G.item_start[c1], G.items_cap);
  double acc = 0.0;
  for (int i = i0 + (t >> 3); i < i1; i += 32 * 16) {
    double v[16];
#pragma unroll
    for (int u = 0; u < 16; u++) v[u] = i + 32 * u < i1 ? partial[(size_t)(i + 32 * u) * 8 + q] : 0.0;
#pragma unroll
    for (int u = 0; u < 16; u++) acc += v[u];
  }
  // the wave's eight rows, then the four waves in order
  for (int o = 8; o < WAVE; o <<= 1) acc += __shfl_xor(acc, o, 64);
  if ((t & 63) < 8) s[q][t >> 6] = acc;
  __syncthreads();
  if (t < 8) s[t][0] = ((s[t][0] + s[t][1]) + s[t][2]) + s[t][3];
  __syncthreads();
  if (t == 0) {
    values[sy] = s[0][0];
    double v6[6] = {s[1][0], s[2][0], s[3][0], s[4][0], s[5][0], s[6][0]};
    write_virial(virials + 9 * (size_t)sy, v6);
    npairs[sy] = s[7][0];
  }
}

// ------------------------------------------------------------------------
// FP64 fallback kernels
// ------------------------------------------------------------------------
// Every requested atom accumulates its own derivative from all its partners
// (no atomics); the value and the virial are taken once per pair.  The
// partners are every atom of the other group (two groups) or of the group,
// or, with a neighbour list (nbr_start non-null), the atoms nbr[nbr_start[i]
// .. nbr_start[i+1]) listed for atom i in both directions.

// minimum image of d = x_q - x_p: PBC 0 none, 1 orthorhombic, 2 any cell
template <int PBC>
__device__ __forceinline__ void wrap64(const PbcArg& P, double* d) {
#pragma clang fp contract(off)
  if constexpr (PBC == 1) {
    for (int i = 0; i < 3; i++) d[i] = pbc1(d[i] * P.inv[4 * i]) * P.box[4 * i];
  } else if constexpr (PBC == 2) {
    const double zero[3] = {0.0, 0.0, 0.0};
    const double v[3] = {d[0], d[1], d[2]};
    pbc_distance(P, zero, v, d);
  }
}

// s and dfunc: SWK = P > 0 for fixedRational<2P> (its exponents unroll), 0 any
template <int SWK>
__device__ __forceinline__ double switch64(const p2a_switch& sw, double d2, double& df) {
#pragma clang fp contract(off)
  if constexpr (SWK > 0) {
    // switch_calc_sqr of RATIONAL_FIXED, for d2 inside D_MAX
    const double rdist = d2 * sw.invr0_2;
    const double rN = ipow(rdist, SWK - 1);
    const double r = 1.0 / (1.0 + rN * rdist);
    double f = -SWK * rN * r * r;
    f *= 2 * sw.invr0_2;
    df = f * sw.stretch;
    return r * sw.stretch + sw.shift;
  } else {
    return switch_calc_sqr(sw, d2, df);
  }
}

struct Sum64 {
  double cv, v[6], np;
};

// the pair (i, j) seen from atom i: f += its derivative; value, virial and
// count when `own` (the pair is listed as i -> j); returns r^2.  The unrolled
// switches leave out every pair that is not inside D_MAX; a distance that is not
// a number or infinite still makes the derivative and the virial no numbers, as 0
// times it: ODD adds that term to f at every pair (no further register: 300 ->
// 305 us a step of 700 x 5,300 atoms on a list), the loop of atoms64 looks at one r^2 a
// partner (49.9 -> 51.0 us at 5,001 atoms; an extra comparison a pair took 55).
template <int PBC, int SWK, bool ODD = false>
__device__ __forceinline__ double pair64(const PbcArg& P, const p2a_switch& sw, const double* xi, const double* xj,
                                       bool own, double* f, Sum64& a) {
#pragma clang fp contract(off)
  // the pair is measured once, as the reference lists it: p -> q with p in
  // GROUPA (two groups) or p < q, d = Pbc::distance(x_p, x_q); atom i is p
  // ("own") or q.  Measured from q, a pair at half a cell could take another
  // of its tied images.  x_j - x_i changes sign exactly.
  double d[3] = {xj[0] - xi[0], xj[1] - xi[1], xj[2] - xi[2]};
  if constexpr (PBC != 0) {
    if (!own)
      for (int k = 0; k < 3; k++) d[k] = -d[k];
    wrap64<PBC>(P, d);
    if (!own)
      for (int k = 0; k < 3; k++) d[k] = -d[k];
  }
  const double r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
  if constexpr (SWK > 0 && ODD)
    for (int k = 0; k < 3; k++) f[k] = fma(0.0, d[k], f[k]);
  if (SWK > 0 && !(r2 <= sw.dmax_2)) return r2;
  double df;
  const double s = switch64<SWK>(sw, r2, df);
  // CoordinationBase: deriv[p] -= df*d, deriv[q] += df*d (one rounding less than
  // the reference's product and sum, as in the virial below)
  for (int k = 0; k < 3; k++) f[k] = fma(-df, d[k], f[k]);
  if (own) {
    const double g[3] = {df * d[0], df * d[1], df * d[2]};
    a.cv += s;
    if (SWK > 0 || switch_inside(sw, r2)) a.np += 1;
    a.v[0] = fma(g[0], d[0], a.v[0]);
    a.v[1] = fma(g[0], d[1], a.v[1]);
    a.v[2] = fma(g[0], d[2], a.v[2]);
    a.v[3] = fma(g[1], d[1], a.v[3]);
    a.v[4] = fma(g[1], d[2], a.v[4]);
    a.v[5] = fma(g[2], d[2], a.v[5]);
  }
  return r2;
}

// the virial of components that are no numbers (q: 0 or NaN each)
__device__ __forceinline__ void odd_virial64(const double* q, Sum64& a) {
  a.v[0] += q[0];
  a.v[1] += q[0] + q[1];
  a.v[2] += q[0] + q[2];
  a.v[3] += q[1];
  a.v[4] += q[1] + q[2];
  a.v[5] += q[2];
}
// NaN in the components that are not finite in x; PBC 2: the image mixes them
template <int PBC>
__device__ __forceinline__ void odd64(const double* x, double* q) {
  for (int k = 0; k < 3; k++) q[k] += 0.0 * x[k];
  if constexpr (PBC == 2) q[0] = q[1] = q[2] = q[0] + q[1] + q[2];
}

// block partials of a 256-thread workgroup, for the final reduction
__device__ __forceinline__ void store_partial64(const Sum64& a, double* __restrict__ partial) {
  __shared__ double red[4][8];
  double r[8] = {a.cv, a.v[0], a.v[1], a.v[2], a.v[3], a.v[4], a.v[5], a.np};
  for (int q = 0; q < 8; q++) r[q] = wave_sum_d(r[q]);
  if ((threadIdx.x & 63) == 0)
    for (int q = 0; q < 8; q++) red[threadIdx.x >> 6][q] = r[q];
  __syncthreads();
  if (threadIdx.x < 8) {
    double t = 0;
    for (int w = 0; w < 4; w++) t += red[w][threadIdx.x];
    partial[(size_t)blockIdx.x * 8 + threadIdx.x] = t;
  }
}

// One side of the all-pairs pass: atoms [i0, i0 + n) against [j0, j0 + m).
struct Side64 {
  int i0, n, j0, m;
  int it;      // atoms a workgroup takes together (1 or kIt64); 0: one per thread
  int blocks;  // workgroups of this side
};
constexpr int kIt64 = 4;
// At most this many workgroups a launch, so that the partials of any launch
// fit the rows of the allocation-free entry point.  With more atom groups
// than that a workgroup takes several in turn.
constexpr int kMaxBlocks64 = 1024;

// `it` atoms against all partners, the lanes of the workgroup over the partners
template <int PBC, int SWK, int IT>
__device__ __forceinline__ void atoms64(const Side64& S, int g, bool two, bool own2, const PbcArg& P,
                                        const p2a_switch& sw, const double* __restrict__ pos,
                                        const long long* __restrict__ absidx, double* __restrict__ deriv, Sum64& a) {
  __shared__ double sf[4][3 * IT];
  const int ib = S.i0 + g * IT;
  const int ni = min(IT, S.i0 + S.n - ib);
  double xi[IT][3], f[IT][3];
#pragma unroll
  for (int u = 0; u < IT; u++) {
    const int i = ib + (u < ni ? u : 0);
    for (int k = 0; k < 3; k++) {
      xi[u][k] = pos[3 * (size_t)i + k];
      f[u][k] = 0.0;
    }
  }
  double z = 0.0;  // NaN once a partner (or the first atom) is not finite
  for (int j = S.j0 + (int)threadIdx.x; j < S.j0 + S.m; j += 256) {
    const double xj[3] = {pos[3 * (size_t)j], pos[3 * (size_t)j + 1], pos[3 * (size_t)j + 2]};
#pragma unroll
    for (int u = 0; u < IT; u++) {
      const int i = ib + u;
      // absidx null: the requested atoms are distinct atoms
      if (u < ni && j != i && !(absidx && absidx[i] == absidx[j])) {
        const double r2 = pair64<PBC, SWK>(P, sw, xi[u], xj, two ? own2 : i < j, f[u], a);
        if (SWK > 0 && u == 0) z = fma(0.0, r2, z);
      }
    }
  }
  if constexpr (SWK > 0) {
#pragma unroll
    for (int u = 1; u < IT; u++)
      for (int k = 0; k < 3; k++) z = fma(0.0, xi[u][k], z);
    if (z != z) {
      double qj[3] = {0.0, 0.0, 0.0};
      for (int j = S.j0 + (int)threadIdx.x; j < S.j0 + S.m; j += 256) odd64<PBC>(pos + 3 * (size_t)j, qj);
#pragma unroll
      for (int u = 0; u < IT; u++) {
        double q[3] = {qj[0], qj[1], qj[2]};
        odd64<PBC>(xi[u], q);
        for (int k = 0; k < 3; k++) f[u][k] += q[k];
        odd_virial64(q, a);
      }
    }
  }
#pragma unroll
  for (int u = 0; u < IT; u++)
    for (int k = 0; k < 3; k++) {
      const double t = wave_sum_d(f[u][k]);
      if ((threadIdx.x & 63) == 0) sf[threadIdx.x >> 6][3 * u + k] = t;
    }
  __syncthreads();
  const int t = threadIdx.x;
  if (t < 3 * ni) deriv[3 * (size_t)ib + t] = ((sf[0][t] + sf[1][t]) + sf[2][t]) + sf[3][t];
  __syncthreads();
}

// All pairs.  Bound by FP64 VALU issue (about 45 instructions a pair without
// a cell): the partners of an atom go over the 256 lanes of a workgroup, so
// that a few hundred atoms already fill the chip, and kIt64 atoms share each
// loaded partner (24 B at a stride of 24 B: with one atom a load the L1 would
// be the bound).  Measured, one thread per atom before -> this: 5,001 atoms
// without a cell 3.24 ms -> 53 us; 100 x 200 atoms in a 3 nm cell 157 -> 4.7 us.
// A side with few partners keeps one thread per atom (its partners are then
// uniform loads), see allpairs_sides.
template <int PBC, int SWK>
__global__ __launch_bounds__(256) void k_allpairs(Side64 S0, Side64 S1, PbcArg P, p2a_switch sw,
                                                  const double* __restrict__ pos,
                                                  const long long* __restrict__ absidx, double* __restrict__ deriv,
                                                  double* __restrict__ partial) {
  const bool two = S1.n > 0;
  const bool first = (int)blockIdx.x < S0.blocks;
  const Side64 S = first ? S0 : S1;
  const int b = first ? (int)blockIdx.x : (int)blockIdx.x - S0.blocks;
  Sum64 a = {0.0, {0.0, 0.0, 0.0, 0.0, 0.0, 0.0}, 0.0};
  if (S.it == 1) {
    for (int g = b; g < S.n; g += S.blocks) atoms64<PBC, SWK, 1>(S, g, two, first, P, sw, pos, absidx, deriv, a);
  } else if (S.it == kIt64) {
    for (int g = b; g * kIt64 < S.n; g += S.blocks)
      atoms64<PBC, SWK, kIt64>(S, g, two, first, P, sw, pos, absidx, deriv, a);
  } else {
    for (int q = b * 256 + (int)threadIdx.x; q < S.n; q += S.blocks * 256) {
      const int i = S.i0 + q;
      const double xi[3] = {pos[3 * (size_t)i], pos[3 * (size_t)i + 1], pos[3 * (size_t)i + 2]};
      double f[3] = {0.0, 0.0, 0.0};
      for (int j = S.j0; j < S.j0 + S.m; j++) {
        if (j == i || (absidx && absidx[i] == absidx[j])) continue;
        const double xj[3] = {pos[3 * (size_t)j], pos[3 * (size_t)j + 1], pos[3 * (size_t)j + 2]};
        pair64<PBC, SWK, true>(P, sw, xi, xj, two ? first : i < j, f, a);
      }
      if (SWK > 0) {
        const double q[3] = {0.0 * f[0], 0.0 * f[1], 0.0 * f[2]};
        odd_virial64(q, a);
      }
      for (int k = 0; k < 3; k++) deriv[3 * (size_t)i + k] = f[k];
    }
  }
  store_partial64(a, partial);
}

// One side of the list pass: atoms [i0, i0 + n), `wide`: a workgroup per
// atom, else a wave per atom.
struct ListSide64 {
  int i0, n, wide, blocks;
};

// atom i against the listed partners p0, p0 + step, ...: each partner's
// index and position are loaded ahead of the pair before it
template <int PBC, int SWK>
__device__ __forceinline__ void listed64(int i, int p0, int step, bool two, bool own2, const PbcArg& P,
                                         const p2a_switch& sw, const double* __restrict__ pos,
                                         const long long* __restrict__ absidx, const int* __restrict__ nbr, int e,
                                         double* f, Sum64& a) {
  const double xi[3] = {pos[3 * (size_t)i], pos[3 * (size_t)i + 1], pos[3 * (size_t)i + 2]};
  int p = p0;
  int j = p < e ? nbr[p] : 0;
  int jn = p + step < e ? nbr[p + step] : 0;
  double x[3] = {pos[3 * (size_t)j], pos[3 * (size_t)j + 1], pos[3 * (size_t)j + 2]};
  for (; p < e; p += step) {
    const int jc = j;
    const double xj[3] = {x[0], x[1], x[2]};
    j = jn;
    for (int k = 0; k < 3; k++) x[k] = pos[3 * (size_t)j + k];
    jn = p + 2 * step < e ? nbr[p + 2 * step] : 0;
    if (jc != i && !(absidx && absidx[i] == absidx[jc]))
      pair64<PBC, SWK, true>(P, sw, xi, xj, two ? own2 : i < jc, f, a);
  }
  if (SWK > 0) {
    const double q[3] = {0.0 * f[0], 0.0 * f[1], 0.0 * f[2]};
    odd_virial64(q, a);
  }
}

// The pairs of a neighbour list.  A list holds tens to thousands of partners:
// long lists (see list_side64) take a workgroup per atom, the others a wave
// per atom.  Bound by the latency of partner index -> position, hence the
// loads ahead.  Measured at 700 x 5,300 atoms with 3,100 / 410 partners
// listed: one thread per atom 3.61 ms, now 22 us.
template <int PBC, int SWK>
__global__ __launch_bounds__(256) void k_listpairs(ListSide64 S0, ListSide64 S1, PbcArg P, p2a_switch sw,
                                                   const double* __restrict__ pos,
                                                   const long long* __restrict__ absidx, double* __restrict__ deriv,
                                                   double* __restrict__ partial, const int* __restrict__ nbr_start,
                                                   const int* __restrict__ nbr) {
  __shared__ double sf[4][3];
  const bool two = S1.n > 0;
  const bool first = (int)blockIdx.x < S0.blocks;
  const ListSide64 S = first ? S0 : S1;
  const int b = first ? (int)blockIdx.x : (int)blockIdx.x - S0.blocks;
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  Sum64 a = {0.0, {0.0, 0.0, 0.0, 0.0, 0.0, 0.0}, 0.0};
  const int per = S.wide ? 1 : 4;
  for (int g = b * per; g < S.n; g += S.blocks * per) {
    const int q = S.wide ? g : g + w;
    double f[3] = {0.0, 0.0, 0.0};
    if (q < S.n) {
      const int i = S.i0 + q;
      const int p0 = nbr_start[i] + (S.wide ? t : lane), e = nbr_start[i + 1];
      listed64<PBC, SWK>(i, p0, S.wide ? 256 : WAVE, two, first, P, sw, pos, absidx, nbr, e, f, a);
    }
    for (int k = 0; k < 3; k++) f[k] = wave_sum_d(f[k]);
    if (!S.wide) {
      if (q < S.n && lane < 3) deriv[3 * (size_t)(S.i0 + q) + lane] = lane == 0 ? f[0] : (lane == 1 ? f[1] : f[2]);
      continue;
    }
    if (lane == 0)
      for (int k = 0; k < 3; k++) sf[w][k] = f[k];
    __syncthreads();
    if (t < 3) deriv[3 * (size_t)(S.i0 + q) + t] = ((sf[0][t] + sf[1][t]) + sf[2][t]) + sf[3][t];
    __syncthreads();
  }
  store_partial64(a, partial);
}

// PAIR: the k-th atom of GROUPA with the k-th of GROUPB
// (with a neighbour list, only the pairs k whose nl_keep[k] is set)
__global__ void k_pairmode(int nA, int use_pbc, PbcArg P, p2a_switch sw, const double* __restrict__ pos,
                           const long long* __restrict__ absidx, double* __restrict__ deriv,
                           double* __restrict__ partial, const int* __restrict__ nl_keep = nullptr) {
#pragma clang fp contract(off)
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  double r[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  if (i < nA) {
    const int j = nA + i;
    double* di = deriv + 3 * (size_t)i;
    double* dj = deriv + 3 * (size_t)j;
    di[0] = di[1] = di[2] = 0.0;
    dj[0] = dj[1] = dj[2] = 0.0;
    if (absidx[i] != absidx[j] && (!nl_keep || nl_keep[i])) {
      const double* xi = pos + 3 * (size_t)i;
      const double* xj = pos + 3 * (size_t)j;
      double d[3];
      if (use_pbc) pbc_distance(P, xi, xj, d);
      else { d[0] = xj[0] - xi[0]; d[1] = xj[1] - xi[1]; d[2] = xj[2] - xi[2]; }
      double r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
      double df;
      double s = switch_calc_sqr(sw, r2, df);
      for (int k = 0; k < 3; k++) {
        di[k] = -df * d[k];
        dj[k] = df * d[k];
      }
      r[0] = s;
      r[1] = df * d[0] * d[0];
      r[2] = df * d[0] * d[1];
      r[3] = df * d[0] * d[2];
      r[4] = df * d[1] * d[1];
      r[5] = df * d[1] * d[2];
      r[6] = df * d[2] * d[2];
      r[7] = switch_inside(sw, r2) ? 1.0 : 0.0;
    }
  }
  const int lane = threadIdx.x & 63;
  for (int q = 0; q < 8; q++) r[q] = wave_sum(r[q]);
  __shared__ double red[4][8];
  if (lane == 0)
    for (int q = 0; q < 8; q++) red[threadIdx.x >> 6][q] = r[q];
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int q = 0; q < 8; q++) {
      double t = 0;
      for (int w = 0; w < (int)(blockDim.x / 64); w++) t += red[w][q];
      partial[(size_t)blockIdx.x * 8 + q] = t;
    }
  }
}

// ------------------------------------------------------------------------
// Neighbour lists of the FP64 path, with the candidate sets of the
// reference (NeighborList::update, NeighborList.cpp:177-308), stored as a
// symmetric CSR: atom i lists every partner j of a listed pair (i,j) or (j,i)
// ------------------------------------------------------------------------

// LinkCells grid of the cells branch: cell of an atom from its scaled
// coordinates (LinkCells::findMyCell, LinkCells.cpp:277-292); `origin` is
// subtracted first when the grid box was built around the atoms (no cell
// given, LinkCells.cpp:49-73)
struct CellGrid {
  double inv[9];  // inverse of the grid box (rows), as Pbc::setBox forms it
  double origin[3];
  int shift_origin;
  int nc[3];
  int use_pbc;  // stencil wraps around (LinkCells::addRequiredCells)
};

#pragma clang fp contract(off)
__device__ __forceinline__ void grid_cell(const CellGrid& G, const double* x, int* c) {
  double m[3] = {x[0], x[1], x[2]};
  if (G.shift_origin)
    for (int k = 0; k < 3; k++) m[k] = m[k] - G.origin[k];
  for (int j = 0; j < 3; j++) {
    // Pbc::realToScaled: matmul(transpose(invBox), d)
    const double f = m[0] * G.inv[j] + m[1] * G.inv[3 + j] + m[2] * G.inv[6 + j];
    int cj = (int)floor((pbc1(f) + 0.5) * G.nc[j]);
    c[j] = min(max(cj, 0), G.nc[j] - 1);
  }
}
#pragma clang fp contract(fast)

// cells a and b are within one stencil (LinkCells::addRequiredCells,
// LinkCells.cpp:183-239: cells c-1..c+1 along each direction, wrapped with
// pbc, every cell when there are fewer than three; without pbc, clipped)
__device__ __forceinline__ bool grid_adjacent(const CellGrid& G, const int* a, const int* b) {
  for (int k = 0; k < 3; k++) {
    const int n = G.nc[k];
    if (G.use_pbc) {
      if (n >= 3) {
        const int d = (b[k] - a[k] + n) % n;
        if (d != 0 && d != 1 && d != n - 1) return false;
      }
    } else if (abs(a[k] - b[k]) > 1) {
      return false;
    }
  }
  return true;
}

__global__ void k_nl_cells(int natoms, CellGrid G, const double* __restrict__ pos, int* __restrict__ cellof) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= natoms) return;
  int c[3];
  grid_cell(G, pos + 3 * (size_t)i, c);
  cellof[3 * i] = c[0];
  cellof[3 * i + 1] = c[1];
  cellof[3 * i + 2] = c[2];
}

// FILL = 0: count[i] = listed partners of atom i; FILL = 1: write them, in
// index order, from start[i].  CELLS: the stencil of link cells, else
// |d|^2 <= cut2.  One wave per atom; four chunks of 64 candidates a trip,
// whose loads go out together (the candidates' latency is the bound), and a
// ballot places the listed ones in index order.  Measured at 700 x 5,300
// atoms: one thread per atom 1.81 ms (count) and 2.21 ms (fill), now 18 and 29 us.
template <int FILL, bool CELLS, int PBC>
__global__ __launch_bounds__(256) void k_nl_atoms(int nA, int nB, PbcArg P, double cut2, CellGrid G,
                                                  const double* __restrict__ pos,
                                                  const int* __restrict__ cellof, int* __restrict__ count,
                                                  const int* __restrict__ start, int* __restrict__ nbr) {
#pragma clang fp contract(off)
  constexpr int U = 4;
  const int natoms = nA + nB;
  const int lane = threadIdx.x & 63;
  const int i = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (i >= natoms) return;
  const bool two = nB > 0;
  const int j0 = two ? (i < nA ? nA : 0) : 0;
  const int j1 = two ? (i < nA ? natoms : nA) : nA;
  double xi[3] = {0.0, 0.0, 0.0};
  int ci[3] = {0, 0, 0};
  for (int k = 0; k < 3; k++) {
    if constexpr (CELLS) ci[k] = cellof[3 * i + k];
    else xi[k] = pos[3 * (size_t)i + k];
  }
  int n = 0;
  const int base = FILL ? start[i] : 0;
  for (int jb = j0; jb < j1; jb += U * WAVE) {
    double x[U][3];
    int c[U][3];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int j = min(jb + u * WAVE + lane, j1 - 1);
      for (int k = 0; k < 3; k++) {
        if constexpr (CELLS) c[u][k] = cellof[3 * j + k];
        else x[u][k] = pos[3 * (size_t)j + k];
      }
    }
    bool in[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int j = jb + u * WAVE + lane;
      // the pair (p, q) as the reference lists it: GROUPA atom first with two
      // groups, the lower index first in one group
      const bool own = two ? i < nA : i < j;
      if constexpr (CELLS) {
        in[u] = own ? grid_adjacent(G, ci, c[u]) : grid_adjacent(G, c[u], ci);
      } else {
        double d[3];
        for (int k = 0; k < 3; k++) d[k] = own ? x[u][k] - xi[k] : xi[k] - x[u][k];
        wrap64<PBC>(P, d);
        in[u] = d[0] * d[0] + d[1] * d[1] + d[2] * d[2] <= cut2;
      }
      in[u] = in[u] && j < j1 && (two || j != i);
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      const unsigned long long m = __ballot(in[u]);
      if (FILL && in[u]) nbr[base + n + bits_below(m)] = jb + u * WAVE + lane;
      n += __popcll(m);
    }
  }
  if (!FILL && lane == 0) count[i] = n;
}

template <int FILL>
inline void launch_nl_atoms(hipStream_t s, int nA, int nB, bool cells, int use_pbc, const PbcArg& P, double cut2,
                            const CellGrid& G, const double* pos, const int* cellof, int* count, const int* start,
                            int* nbr) {
  const dim3 grid((unsigned)((nA + nB + 3) / 4));
#define P2A_NL(C, PBC)                                                                                      \
  hipLaunchKernelGGL((k_nl_atoms<FILL, C, PBC>), grid, dim3(256), 0, s, nA, nB, P, cut2, G, pos, cellof, count, start, nbr)
  const int pbc = use_pbc ? P.type : 0;
  if (cells) P2A_NL(true, 0);
  else if (pbc == 0) P2A_NL(false, 0);
  else if (pbc == 1) P2A_NL(false, 1);
  else P2A_NL(false, 2);
#undef P2A_NL
}

// PAIR with a list: keep[k] = pair k within NL_CUTOFF (classic branch)
__global__ void k_nl_pairs_keep(int nA, int use_pbc, PbcArg P, double cut2, const double* __restrict__ pos,
                                int* __restrict__ keep) {
#pragma clang fp contract(off)
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nA) return;
  const double* xa = pos + 3 * (size_t)i;
  const double* xb = pos + 3 * (size_t)(nA + i);
  double d[3];
  if (use_pbc) pbc_distance(P, xa, xb, d);
  else { d[0] = xb[0] - xa[0]; d[1] = xb[1] - xa[1]; d[2] = xb[2] - xa[2]; }
  keep[i] = d[0] * d[0] + d[1] * d[1] + d[2] * d[2] <= cut2 ? 1 : 0;
}

// exclusive scan of n counts in one workgroup of 1024 threads (contiguous
// chunks per thread); start[n] = total
__global__ __launch_bounds__(1024) void k_scan_small(int n, const int* __restrict__ count, int* __restrict__ start,
                                                     long long* __restrict__ total) {
  __shared__ long long part[1024];
  const int t = threadIdx.x;
  const int per = (n + 1023) / 1024;
  const int a = min(n, t * per), b = min(n, a + per);
  long long sum = 0;
  for (int k = a; k < b; k++) sum += count[k];
  part[t] = sum;
  __syncthreads();
  for (int o = 1; o < 1024; o <<= 1) {
    long long v = t >= o ? part[t - o] : 0;
    __syncthreads();
    part[t] += v;
    __syncthreads();
  }
  long long run = part[t] - sum;
  for (int k = a; k < b; k++) {
    start[k] = (int)run;
    run += count[k];
  }
  if (t == 1023) {
    start[n] = (int)part[1023];
    *total = part[1023];
  }
}

// ------------------------------------------------------------------------
// host helpers shared by the single-system and batch contexts
// ------------------------------------------------------------------------
inline int grid1(size_t n, int b) { return (int)((n + b - 1) / b); }

inline int launch_check(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(P2A_ERR_HIP, std::string(what) + ": " + hipGetErrorString(e));
  return P2A_OK;
}

inline void fill_pbc_arg(const PbcHost& h, PbcArg& P) {
  std::memset(&P, 0, sizeof(P));
  P.type = h.type;
  std::memcpy(P.box, h.box, sizeof(P.box));
  std::memcpy(P.inv, h.inv, sizeof(P.inv));
  std::memcpy(P.red, h.reduced, sizeof(P.red));
  std::memcpy(P.ired, h.invReduced, sizeof(P.ired));
  std::memcpy(P.nshift, h.nshift, sizeof(P.nshift));
  std::memcpy(P.shifts, h.shifts, sizeof(P.shifts));
}

// cell part of a SysArg (column grid and list radius are set by the caller)
inline void sys_cell(const double* box9, double rlist, SysArg& S) {
  PbcHost tmp;
  pbc_setup(box9, tmp);
  std::memcpy(S.a, box9, sizeof(S.a));
  std::memcpy(S.inv, tmp.inv, sizeof(S.inv));
  for (int k = 0; k < 9; k++) S.af[k] = (float)box9[k];
  double w[3];
  pbc_widths(box9, w);
  for (int k = 0; k < 3; k++) S.rb[k] = (float)(rlist / w[k]);
  S.ortho = 1;
  for (int k = 0; k < 9; k++)
    if (k % 4 && box9[k] != 0.0) S.ortho = 0;
  S.aa = (float)(box9[0] * box9[0]);
  S.bb = (float)(box9[4] * box9[4]);
  S.invc = (float)(1.0 / std::fabs(box9[8]));
}

// columns of a group of n atoms in a cell: side ~ cbrt(8/rho), bounded count
inline void sys_columns(const double* box9, int n, SysArg& S) {
  double w[3];
  pbc_widths(box9, w);
  double vol = std::fabs(w[0] * w[1] * w[2]);
  double rho = std::max(n, 1) / vol;
  double side = std::cbrt((double)CL / rho);
  // (div_by: a window holds three times as many)
  S.ncx = std::max(1, (int)std::min(std::floor(w[0] / side), 1048576.0));
  S.ncy = std::max(1, (int)std::min(std::floor(w[1] / side), 1048576.0));
  // keep the column count bounded for very dilute groups
  while ((int64_t)S.ncx * S.ncy > 4 * (int64_t)n + 16) {
    S.ncx = std::max(1, S.ncx / 2);
    S.ncy = std::max(1, S.ncy / 2);
  }
  S.icx = 1.f / S.ncx;
  S.icy = 1.f / S.ncy;
}

// How one side of the all-pairs pass goes over the chip: many atoms with at
// most 64 partners (a solvent against one ion), or more atoms than fill the
// chip as threads: one thread per atom; up to 1,024 atoms: one atom per
// workgroup; above: kIt64 atoms per workgroup share each partner.
inline Side64 side64(int i0, int n, int j0, int m, int max_blocks) {
  Side64 S = {i0, n, j0, m, 0, 0};
  if (n == 0) return S;
  S.it = ((m <= 64 && n > 4096) || n >= (1 << 18)) ? 0 : (n <= 1024 ? 1 : kIt64);
  const int per = S.it == 0 ? 256 : S.it;
  S.blocks = std::max(1, std::min(grid1((size_t)n, per), max_blocks));
  return S;
}

// Side of a list pass over `entries` listed partners: a workgroup per atom
// from 512 partners an atom on (two trips of a workgroup), and for so few
// atoms that waves would leave the chip idle.
constexpr int kMaxListBlocks64 = 4096;
inline ListSide64 list_side64(int i0, int n, int64_t entries) {
  ListSide64 S = {i0, n, 0, 0};
  if (n == 0) return S;
  S.wide = entries >= 512 * (int64_t)n || (n < 1024 && entries >= 128 * (int64_t)n);
  S.blocks = std::min(grid1((size_t)n, S.wide ? 1 : 4), kMaxListBlocks64 / 2);
  return S;
}

// the switch of the FP64 pair kernels that unrolls (0: evaluated generically)
inline int switch64_kind(const p2a_switch& sw) {
  return sw.type == P2A_SW_RATIONAL_FIXED && (sw.nn == 6 || sw.nn == 8) ? sw.nn / 2 : 0;
}

// FP64 pass over every pair (at most kMaxBlocks64 rows of `partial`), or over
// the list nbr_start / nbr of nbr_total partners (at most kMaxListBlocks64
// rows); writes deriv and the rows, whose number is returned.  absidx null:
// the requested atoms are distinct atoms.
inline int launch_pairs64(hipStream_t s, int nA, int nB, int use_pbc, const PbcArg& P, const p2a_switch& sw,
                          const double* pos, const long long* absidx, double* deriv, double* partial,
                          const int* nbr_start = nullptr, const int* nbr = nullptr, int64_t nbr_total = 0) {
  const int pbc = !use_pbc || P.type == 0 ? 0 : P.type;
  const int kind = switch64_kind(sw);
  const bool two = nB > 0;
  Side64 S0, S1;
  ListSide64 L0, L1;
  int grid;
  if (nbr_start) {
    // a symmetric list: with two groups each side holds half of the partners
    L0 = list_side64(0, nA, two ? nbr_total / 2 : nbr_total);
    L1 = list_side64(nA, nB, nbr_total / 2);
    grid = L0.blocks + L1.blocks;
  } else {
    S0 = side64(0, nA, two ? nA : 0, two ? nB : nA, two ? kMaxBlocks64 / 2 : kMaxBlocks64);
    S1 = side64(nA, nB, 0, nA, kMaxBlocks64 - S0.blocks);
    grid = S0.blocks + S1.blocks;
  }
#define P2A_A(PBC, K)                                                                                            \
  do {                                                                                                           \
    if (nbr_start)                                                                                               \
      hipLaunchKernelGGL((k_listpairs<PBC, K>), dim3(grid), dim3(256), 0, s, L0, L1, P, sw, pos, absidx, deriv,  \
                         partial, nbr_start, nbr);                                                               \
    else                                                                                                         \
      hipLaunchKernelGGL((k_allpairs<PBC, K>), dim3(grid), dim3(256), 0, s, S0, S1, P, sw, pos, absidx, deriv,   \
                         partial);                                                                               \
  } while (0)
#define P2A_AK(PBC)                    \
  do {                                 \
    if (kind == 3) P2A_A(PBC, 3);      \
    else if (kind == 4) P2A_A(PBC, 4); \
    else P2A_A(PBC, 0);                \
  } while (0)
  if (pbc == 0) P2A_AK(0);
  else if (pbc == 1) P2A_AK(1);
  else P2A_AK(2);
#undef P2A_AK
#undef P2A_A
  return grid;
}

// the chunk size (entries per work item) and the grid of the pair kernel
struct PairTuning {
  int chunk = 64;        // 32 or 64
  // 0: one wave per item; > 0: persistent grid of that many blocks per CU.
  // The persistent grid also bounds the workgroup rows of the final sum.
  int blocks_per_cu = 4;  // the workgroups of the pair kernel one CU holds at once
};

// ------------------------------------------------------------------------
// COORDINATIONNUMBER rows on the cluster list
// ------------------------------------------------------------------------
// cn_i = sum over the environment atoms j of s(r_ij) (ContactMatrix row times
// ONES, symfunc/CoordinationNumbers.cpp:326-372; ContactMatrix::
// calculateWeight, adjmat/ContactMatrix.h:95-121, skips |r|^2 < DBL_EPSILON).
// In the full cluster list every row atom i meets all its partners as the i
// atom of its own items, so lane (ii, jj) sums the s of its pairs over every
// entry kind.  With weights w (wreq: the weight of each requested atom, 0 for
// atoms that are no row) the kernel also forms the vector-Jacobian product
// sum_k w_k dcn_k/dx: F = sum_k w_k cn_k = sum over pairs (w_i + w_j) s_ij,
// so atom i takes (w_i + w_j)(-dfunc d) from each partner and the box
// derivative takes (w_i + w_j) dfunc d (x) d once per unordered pair.
// Band pairs (r^2 within `band` of D_MAX^2) are decided on the spot on the
// reference's FP64 Pbc::distance, so that they take their place in the lane's
// sums.  With weights the staged atoms carry their weight where the others
// carry their requested index (packed positions pwI / pwJ), which the rare band
// pair then finds by going through the item's rounds again: a third array in
// LDS would cost a quarter of the resident waves.  In groups that share atoms the
// staging notes where each i atom's twin went (Twin): one register a lane, and one
// comparison a pair (3,000 rows in an environment of 30,000 that holds them,
// D_MAX 1.2: a call with weights 131 us, groups apart 121; with the index looked
// for at every pair inside D_MAX 1,855).
// Outputs: rpart[item][8] (row sums of the i atoms), and with WT fpart
// [item][8][3] and per-workgroup rows (0, six box-derivative products, 0).
// 30,000 atoms, WT: 33 us (46 with the weights and indices in LDS arrays of their
// own, three workgroups a CU).
constexpr double kContactEps2 = 2.220446049250313e-16;  // DBL_EPSILON

// requested index of staged atom p of the item in LDS (stage_item's rounds
// again, on the positions that carry the indices); uniform over the wave
template <int CH>
__device__ int staged_index(const PairArgs& A, const WaveLds& L, int p, int n0, int ci, int lane, const float4& ic,
                            const float4& ih, const float4* __restrict__ posJ) {
  if (p < n0) return __float_as_int(posJ[ci * CL + p].w);
  // (self entries come first, then counting and derivative-only ones, each
  // kind padded to a multiple of 8)
  int at = n0;
  bool first = true;
  for (int r = 0; r < sent_cap<CH>() / CL; r++) {
    const Entry e = L.se[r * CL + (lane >> 3)];
    // the first round of the derivative-only entries starts at a multiple of 8
    const bool deriv = __ballot((lane & 7) == 0 && e.code >= 0 && !(e.code & kCountBit)) != 0ull;
    if (deriv && first) {
      at = (at + CL - 1) & ~(CL - 1);
      first = false;
    }
    float4 q = posJ[(e.code & kCjMask) * CL + (lane & 7)];
    const int req = __float_as_int(q.w);
    q.x += e.dx;
    q.y += e.dy;
    q.z += e.dz;
    const float gx = fmaxf(fabsf(q.x - ic.x) - ih.x, 0.f);
    const float gy = fmaxf(fabsf(q.y - ic.y) - ih.y, 0.f);
    const float gz = fmaxf(fabsf(q.z - ic.z) - ih.z, 0.f);
    const bool keep = e.code >= 0 && fmaf(gz, gz, fmaf(gx, gx, gy * gy)) <= A.prune2;
    const unsigned long long m = __ballot(keep);
    const int n = __popcll(m);
    if (p < at + n) {
      const unsigned long long mine = __ballot(keep && at + bits_below(m) == p);
      return p >= at && mine ? __builtin_amdgcn_readlane(req, __builtin_ctzll(mine)) : -1;
    }
    at += n;
  }
  return -1;
}

// per-item constants of the row kernel
struct RowItem {
  int ci, n0, reqi;
  int twin;            // staged slot of this lane's i atom in the other group (TWO, WT)
  float4 ic, ih;
  const float4* idxJ;  // packed positions with requested indices
  const PbcArg* pbc;
};

template <int P, bool GENERIC, bool TWO, bool WT, int KIND, int CH>
__device__ __forceinline__ void row_term(const PairArgs& A, const RowItem& I, const float4& pj, const float4& pi,
                                         int ii, int jj, int g, int lane, int ai, float wi, const WaveLds& L,
                                         PairAcc& acc, int& cnt) {
  float dx, dy, dz;
  const float r2 = pair_d(pj, pi, dx, dy, dz);
  bool keep = r2 >= A.contact2;
  if constexpr (KIND == 0) keep = keep && jj != ii;
  if constexpr (TWO) keep = keep && (WT ? g + jj != I.twin : __float_as_int(pj.w) != ai);
  const float t = r2 - A.dmax2;
  const unsigned long long bm = __ballot(keep && fabsf(t) < A.band);
  bool cut = keep && t <= 0.f;
  if (bm != 0ull) {  // uniform, rare
    for (unsigned long long m = bm; m; m &= m - 1) {
      const int l = __builtin_ctzll(m);
      int reqj;
      if constexpr (WT) reqj = staged_index<CH>(A, L, g + (l >> 3), I.n0, I.ci, lane, I.ic, I.ih, I.idxJ);
      else reqj = __float_as_int(pj.w);
      if (lane == l && keep && I.reqi >= 0 && reqj >= 0)
        cut = switch_inside(A.sw, exact_r2(I.pbc, A.pos64, I.reqi, reqj));
    }
  }
  float sv, dfu;
  if constexpr (GENERIC) {
    sv = dfu = 0.f;
    if (cut) pair_switch<P, GENERIC>(A, r2, sv, dfu);
  } else {
    sw_fixed_x<P>(cut ? r2 : sw_far<P>(), sv, dfu);
  }
  acc.sv += sv;
  cnt += cut ? 1 : 0;
  if constexpr (WT) {
    const float wg = (cut ? wi + pj.w : 0.f) * dfu;
    const float gx = wg * dx, gy = wg * dy, gz = wg * dz;
    acc.fx += gx;
    acc.fy += gy;
    acc.fz += gz;
    bool once = KIND == 1;
    if constexpr (KIND == 0) once = jj > ii;
    if (KIND != 2) {
      const float h = once ? 1.f : 0.f;
      acc.vxx = fmaf(h * gx, dx, acc.vxx);
      acc.vxy = fmaf(h * gx, dy, acc.vxy);
      acc.vxz = fmaf(h * gx, dz, acc.vxz);
      acc.vyy = fmaf(h * gy, dy, acc.vyy);
      acc.vyz = fmaf(h * gy, dz, acc.vyz);
      acc.vzz = fmaf(h * gz, dz, acc.vzz);
    }
  }
}

template <int P, bool GENERIC, bool TWO, bool WT>
__global__ __launch_bounds__(PAIR_BLOCK) __attribute__((amdgpu_waves_per_eu(4))) void k_rows(
    PairArgs A, const int4* __restrict__ items, const Entry* __restrict__ ents, const float4* __restrict__ posI,
    const float4* __restrict__ posJ, const float4* __restrict__ pwI, const float4* __restrict__ pwJ,
    const float4* __restrict__ bbI, const float4* __restrict__ bbJ, const int* __restrict__ twinI,
    double* __restrict__ rpart, double* __restrict__ fpart, double* __restrict__ partial) {
  constexpr int CH = 64;
  constexpr int NW = PAIR_BLOCK / WAVE;
  constexpr int CAP = stage_cap<CH>();
  __shared__ float4 sj[NW][CAP];
  __shared__ Entry sent[NW][sent_cap<CH>()];
  __shared__ double stot[NW][8];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int ii = lane & 7, jj = lane >> 3;
  const int nitems = min(A.nitems, A.items_cap);
  const WaveLds L = {sj[w], sent[w]};
  if (lane < 8) stot[w][lane] = 0.0;
  for (int k = blockIdx.x * NW + w; k < nitems; k += gridDim.x * NW) {
    const int item = k;
    const int4 it = items[item];
    const int ci = it.x;
    const int e1 = min(it.z, A.ent_cap);
    const float4 pi = posI[ci * CL + ii];
    const int ai = TWO ? twinI[ci * CL + ii] : 0;
    RowItem I;
    I.ci = ci;
    I.reqi = __float_as_int(pi.w);
    I.ic = bbI[2 * ci];
    I.ih = bbI[2 * ci + 1];
    I.idxJ = posJ;
    I.pbc = A.pbc + nsys_of(A.cl_sys, ci);
    Entry my_e = {0, 0.f, 0.f, 0.f};
    if (lane < CH && it.y + lane < e1) my_e = ents[it.y + lane];
    int n0, b1, n1, b2, n2;
    Twin T = {posJ, ai, pi, -1};
    stage_item<false, false, CH, TWO && WT>(A, my_e, lane, it.y, e1, ci, I.ic, I.ih, WT ? pwJ : posJ, bbJ, L, n0, b1,
                                            n1, b2, n2, &T);
    I.twin = T.slot;
    n1 = __builtin_amdgcn_readfirstlane(n1);
    n2 = __builtin_amdgcn_readfirstlane(n2);
    b1 = __builtin_amdgcn_readfirstlane(b1);
    b2 = __builtin_amdgcn_readfirstlane(b2);
    I.n0 = n0;
    const float wi = WT ? pwI[ci * CL + ii].w : 0.f;
    PairAcc acc = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    int cnt = 0;
    if (n0) row_term<P, GENERIC, TWO, WT, 0, CH>(A, I, L.sj[jj], pi, ii, jj, 0, lane, ai, wi, L, acc, cnt);
    for (int g = b1; g < b1 + n1; g += CL)
      row_term<P, GENERIC, TWO, WT, 1, CH>(A, I, L.sj[g + jj], pi, ii, jj, g, lane, ai, wi, L, acc, cnt);
    for (int g = b2; g < b2 + n2; g += CL)
      row_term<P, GENERIC, TWO, WT, 2, CH>(A, I, L.sj[g + jj], pi, ii, jj, g, lane, ai, wi, L, acc, cnt);
    // rows of the 8 i atoms: s = stretch * s~ + shift per contributing pair
    const float cs = sum_over_jj(acc.sv), cc = sum_over_jj((float)cnt);
    if (jj == 0) rpart[(size_t)item * CL + ii] = A.sv_scale * (double)cs + A.sv_shift * (double)cc;
    if constexpr (WT) {
      const float f = sum_over_jj3(acc.fx, acc.fy, acc.fz, lane);
      const int c = jj3_component(lane);
      if (c < 3) fpart[(size_t)item * (CL * 3) + ii * 3 + c] = -A.df_scale * (double)f;
      float tv[6];
      tv[0] = wave_sum_f(acc.vxx);
      tv[1] = wave_sum_f(acc.vxy);
      tv[2] = wave_sum_f(acc.vxz);
      tv[3] = wave_sum_f(acc.vyy);
      tv[4] = wave_sum_f(acc.vyz);
      tv[5] = wave_sum_f(acc.vzz);
      if (lane >= 1 && lane < 7) {
        float tq = tv[0];
        for (int q = 1; q < 6; q++)
          if (lane == q + 1) tq = tv[q];
        stot[w][lane] += A.vir_scale * (double)tq;
      }
    }
    // the next item overwrites the staging read above
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
  if constexpr (WT) {
    __syncthreads();
    if (w == 0 && lane < 8) {
      double s = 0.0;
      for (int v = 0; v < NW; v++) s += stot[v][lane];
      partial[(size_t)blockIdx.x * 8 + lane] = s;
    }
  }
}

// rows of the requested atoms 0..nrows-1 (the i group): the fixed-order sum of
// their cluster's item rows; atoms beyond nrows (the environment) are skipped
__global__ __launch_bounds__(256) void k_gather_rows(int nslot, const float4* __restrict__ p,
                                                     const int* __restrict__ item_start, int items_cap,
                                                     const double* __restrict__ rpart, int nrows,
                                                     double* __restrict__ rows) {
  const int sidx = blockIdx.x * blockDim.x + threadIdx.x;
  if (sidx >= nslot) return;
  const int c = sidx / CL, r = sidx % CL;
  const int i0 = item_start[c];
  const int i1 = min(item_start[c + 1], items_cap);
  const int req = __float_as_int(p[sidx].w);
  if (req < 0 || req >= nrows) return;
  double sum = 0.0;
  for (int it = i0; it < i1; it++) sum += rpart[(size_t)it * CL + r];
  rows[req] = sum;
}

// packed positions with the atom's FP32 weight in w: w[k] for the first nrows
// requested atoms, 0 for the others and for padding
__global__ void k_row_weights(int nslot, int nrows, const float4* __restrict__ p, const double* __restrict__ w,
                              float4* __restrict__ pw) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= nslot) return;
  float4 q = p[s];
  const int req = __float_as_int(q.w);
  q.w = req >= 0 && req < nrows ? (float)w[req] : 0.f;
  pw[s] = q;
}

inline void pair_args_generic(PairArgs& A);

inline void launch_rows(const PairArgs& A, bool weighted, int grid, hipStream_t s, const int4* items,
                        const Entry* ents, const float4* posI, const float4* posJ, const float4* pwI,
                        const float4* pwJ, const float4* bbI, const float4* bbJ, const int* twinI, double* rpart,
                        double* fpart, double* partial) {
  const p2a_switch& sw = A.sw;
#define P2A_R(P, GEN, TWO, WT)                                                                                   \
  hipLaunchKernelGGL((k_rows<P, GEN, TWO, WT>), dim3(grid), dim3(PAIR_BLOCK), 0, s, A, items, ents, posI, posJ,   \
                     pwI, pwJ, bbI, bbJ, twinI, rpart, fpart, partial)
#define P2A_RSW(P, GEN)                                        \
  do {                                                         \
    if (A.share) {                                             \
      if (weighted) P2A_R(P, GEN, true, true);                 \
      else P2A_R(P, GEN, true, false);                         \
    } else {                                                   \
      if (weighted) P2A_R(P, GEN, false, true);                \
      else P2A_R(P, GEN, false, false);                        \
    }                                                          \
  } while (0)
  if (sw.type == P2A_SW_RATIONAL_FIXED && sw.nn / 2 == 3) P2A_RSW(3, false);
  else if (sw.type == P2A_SW_RATIONAL_FIXED && sw.nn / 2 == 4) P2A_RSW(4, false);
  else {
    // the other switches run the generic evaluation
    PairArgs G = A;
    pair_args_generic(G);
    const PairArgs& A = G;
    P2A_RSW(0, true);
  }
#undef P2A_RSW
#undef P2A_R
}

// the type a switch is compiled for in switch_known, 0 for none
inline int switch_known_kind(const p2a_switch& sw) {
  if (sw.type == P2A_SW_RATIONAL) return sw.fast ? kSwFastRational : P2A_SW_RATIONAL;
  switch (sw.type) {
    case P2A_SW_EXP: case P2A_SW_GAUSSIAN: case P2A_SW_FASTGAUSSIAN: case P2A_SW_SMAP: case P2A_SW_CUBIC:
    case P2A_SW_TANH: case P2A_SW_COSINUS: case P2A_SW_Q: return sw.type;
    default: return 0;
  }
}

// launch of the pair kernel for a switch, group mode and tuning.  TWOG: the
// caller may have two groups that share atoms, and calls for the value only (else
// those kernels are not compiled); distinct groups run the kernels of one group.
// The other switches have a kernel of their own for the default work items
// (20,000 atoms with EXP: pair pass with derivatives 105 -> 62 us; value only,
// 400,000 atoms, D_MAX 0.8: EXP 275 -> 137 us, TANH 472 -> 338); 32 entries an item
// run the kernel that takes any switch.
template <bool TWOG>
inline void launch_pairs(const PairArgs& A, const Two<PairSide>& T, hipStream_t s, bool value_only, int chunk) {
  const p2a_switch& sw = A.sw;
  const int grid = T.s[0].grid + T.s[1].grid;
#define P2A_K(P, GEN, TWO, VO, CH) \
  hipLaunchKernelGGL((k_pairs<P, GEN, TWO, VO, CH>), dim3(grid), dim3(PAIR_BLOCK), 0, s, A, T)
#define P2A_KCH(P, GEN, TWO, VO)          \
  do {                                    \
    if (chunk == 32) P2A_K(P, GEN, TWO, VO, 32); \
    else P2A_K(P, GEN, TWO, VO, 64);      \
  } while (0)
#define P2A_KSW(P, GEN)                                     \
  do {                                                      \
    if constexpr (TWOG) {                                   \
      if (A.share && value_only) P2A_KCH(P, GEN, true, true);     \
      else if (A.share) P2A_KCH(P, GEN, true, false);       \
      else if (value_only) P2A_KCH(P, GEN, false, true);    \
      else P2A_KCH(P, GEN, false, false);                   \
    } else {                                                \
      P2A_KCH(P, GEN, false, false);                        \
    }                                                       \
  } while (0)
#define P2A_KKN(K)                                              \
  case K:                                                       \
    if constexpr (TWOG) {                                       \
      if (A.share && value_only) P2A_K(K, true, true, true, 64);      \
      else if (A.share) P2A_K(K, true, true, false, 64);        \
      else if (value_only) P2A_K(K, true, false, true, 64);     \
      else P2A_K(K, true, false, false, 64);                    \
    } else {                                                    \
      P2A_K(K, true, false, false, 64);                         \
    }                                                           \
    break
  if (sw.type == P2A_SW_RATIONAL_FIXED) {
    switch (sw.nn / 2) {
      case 1: P2A_KSW(1, false); break;
      case 2: P2A_KSW(2, false); break;
      case 3: P2A_KSW(3, false); break;
      case 4: P2A_KSW(4, false); break;
      case 5: P2A_KSW(5, false); break;
      case 6: P2A_KSW(6, false); break;
      default: P2A_KSW(0, true); break;
    }
    return;
  }
  const int kind = chunk != 64 ? 0 : switch_known_kind(sw);
  switch (kind) {
    P2A_KKN(kSwFastRational);
    P2A_KKN(P2A_SW_RATIONAL);
    P2A_KKN(P2A_SW_EXP);
    P2A_KKN(P2A_SW_GAUSSIAN);
    P2A_KKN(P2A_SW_FASTGAUSSIAN);
    P2A_KKN(P2A_SW_SMAP);
    P2A_KKN(P2A_SW_CUBIC);
    P2A_KKN(P2A_SW_TANH);
    P2A_KKN(P2A_SW_COSINUS);
    P2A_KKN(P2A_SW_Q);
    default: P2A_KSW(0, true); break;
  }
#undef P2A_KKN
#undef P2A_KSW
#undef P2A_KCH
#undef P2A_K
}

// entry starts (out0) and work-item starts (out1, chunks of `chunk`) of the
// n = *n_dev (or n) i clusters of each side; bsum holds 2 * ceil(n / kScanBlock)
// ints
inline void launch_list_scans(hipStream_t s, const ScanSide* sides, int nsides, int chunk, int* totals) {
  Two<ScanSide> T;
  bool one = true;
  int nb[2] = {0, 0};
  for (int d = 0; d < 2; d++) {
    T.s[d] = sides[std::min(d, nsides - 1)];
    if (d >= nsides) continue;
    one = one && sides[d].n <= kScanOneMax;
    nb[d] = std::max(1, grid1(sides[d].n, kScanBlock));
  }
  T.n0 = nb[0];
  if (one) {
    hipLaunchKernelGGL(k_scan2_one, dim3(nsides), dim3(1024), 0, s, T, chunk, totals);
    return;
  }
  hipLaunchKernelGGL(k_scan2_sums, dim3(nb[0] + nb[1]), dim3(256), 0, s, T, chunk);
  hipLaunchKernelGGL(k_scan2_apply, dim3(nb[0] + nb[1]), dim3(256), 0, s, T, chunk, totals);
}

// Scale of the FP32 cluster geometry (packed positions, list offsets,
// boxes): 1/R_0 for the fixedRational switches of the pair kernel (x = r^2
// then needs no multiply), 1 otherwise.
inline bool pair_fixed(const p2a_switch& sw) {
  return sw.type == P2A_SW_RATIONAL_FIXED && sw.nn / 2 >= 1 && sw.nn / 2 <= 6;
}
inline double pack_scale(const p2a_switch& sw) { return pair_fixed(sw) ? std::sqrt(sw.invr0_2) : 1.0; }

// FP32 constants of the pair kernels, the cut band, and the FP64 factors
// that turn the per-item FP32 sums into outputs: for fixedRational<N> the
// kernels sum sv = 1/(1+x^(N/2)) and dfu = x^(N/2-1) sv^2, so that
// value = stretch sum(sv) + shift npair and dfunc = -N/r0^2 stretch dfu
// (SwitchingFunction.cpp:203-215); the generic switches sum s and dfunc.
// The FP32 separations are pack_scale times the real ones, hence the
// 1/pack_scale of the derivative factor and 1/pack_scale^2 of the virial's.
inline void pair_args_switch(const p2a_switch& sw, PairArgs& A) {
  const double k = pack_scale(sw), k2 = k * k;
  A.dmax2 = (float)(sw.dmax_2 * k2);
  const double pr = (sw.dmax + 1e-4) * k;
  A.prune2 = (float)(pr * pr);
  // 1.8x the worst-case FP32 error of r^2 from cluster-local coordinates
  A.band = 4.0e-6f * A.dmax2;
  // the band as two thresholds, each rounded outwards
  A.cut_lo = std::nextafter((float)((double)A.dmax2 - (double)A.band), 0.0f);
  A.cut_hi = std::nextafter((float)((double)A.dmax2 + (double)A.band), HUGE_VALF);
  A.contact2 = (float)(kContactEps2 * k2);
  const bool fixed = pair_fixed(sw);
  A.invr0_2 = fixed ? 1.0f : (float)sw.invr0_2;
  A.r2_real = 1.0 / k2;
  A.sv_scale = fixed ? sw.stretch : 1.0;
  A.sv_shift = fixed ? sw.shift : 0.0;
  const double dfs = fixed ? -(double)sw.nn * sw.invr0_2 * sw.stretch : 1.0;
  A.df_scale = dfs / k;
  A.vir_scale = dfs / k2;
  A.sw = sw;
}

// the factors of pair_args_switch for a kernel that evaluates the switch
// generically (switch_calc_sqr) on the same geometry
inline void pair_args_generic(PairArgs& A) {
  const double k2 = 1.0 / A.r2_real;
  A.sv_scale = 1.0;
  A.sv_shift = 0.0;
  A.df_scale = 1.0 / std::sqrt(k2);
  A.vir_scale = 1.0 / k2;
}

}  // namespace

}  // namespace p2a
