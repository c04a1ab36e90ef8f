// METAD bias grid on gfx950: hill deposition, well-tempered heights, spline
// bias/force, the fused per-step METAD kernel and the force chain rule.
//
// What each piece replaces in the reference:
//   k_hill_chain,   MetaD::update -> getHeight -> addGaussian -> evaluate-
//   k_hill_nodes,   GaussianAndDerivatives -> Grid::addValueAndDerivatives
//   k_deposit_seq   (src/bias/MetaD.cpp:2377-2470, 2280-2305, 1886-1937,
//                   2186-2278; src/tools/Grid.cpp:55-106, 904-910) for many
//                   hills in order (each well-tempered height depends on the
//                   grid left by the previous hill): heights and grid in turn
//                   for many hills, one workgroup for a few
//   k_add_hills     addGaussian for hills of known heights (HILLS restart,
//                   MetaD::readGaussians :1807-1829), all hills in parallel
//   spline()        GridBase::getValueAndDerivatives spline branch
//                   (src/tools/Grid.cpp:442-505) with getSplineNeighbors
//                   (:328-356)
//   k_metad_step    MetaD::calculate (:2315-2375) + MetaD::update on a
//                   device-resident CV
//   k_apply_force   ActionWithValue::checkForForces daxpy
//                   (src/core/ActionWithValue.cpp:337-413)
//
// Layout in HBM: value[node] and gradient[node*ncv + i] in FP64, nodes in the
// column-major order of GridBase::getIndex (first CV fastest).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "fp64_math.h"
#include "p2a_internal.h"

// No fused multiply-add but where fma() stands, so that every evaluation rounds
// the same way wherever it is inlined: deposition in hill order relies on it (a
// corner's value for a height and the node's value on the grid receive
// bit-identical additions).  The spline and the hills of known heights follow the
// reference's FP64 operations one rounding at a time; hills in order do not (a
// product of one exponential per CV, fma() into the nodes, an exponential and a
// reciprocal of their own, HillDim and corner_term): the same formulas in FP64,
// a few roundings apart.
#pragma clang fp contract(off)

namespace p2a {

#define P2A_HIPM(x)                                                                                  \
  do {                                                                                               \
    hipError_t e_ = (x);                                                                             \
    if (e_ != hipSuccess) return fail(P2A_ERR_HIP, std::string(#x) + ": " + hipGetErrorString(e_)); \
  } while (0)

constexpr int kMaxCv = 4;
constexpr int kDepositThreads = 256;
constexpr int WAVE_M = 64;

struct GridArg {
  int ncv;
  int pbc[kMaxCv];
  unsigned nbin[kMaxCv];  // nodes per direction
  int nneigh[kMaxCv];     // support half-width in bins
  double min[kMaxCv], dx[kMaxCv];
  double period[kMaxCv], inv_period[kMaxCv];
  double invsigma[kMaxCv];
  double height0, biasf, kbt, stretchA, stretchB;
  double inv_wt;          // 1 / (kbt (biasf - 1)) for biasf > 1, else 1 / kbt
  double kd[kMaxCv];      // -invsigma * stretchA: scaled distance -> gradient factor
  int welltemp;
  int support;            // prod(2*nneigh+1)
  int may_alias;          // a periodic support wider than the grid visits a node twice
};

// Tools::pbc (Tools.h:547-570)
__device__ __forceinline__ double mpbc1(double x) {
  x += 100.0;
  return (x >= 0) ? x - (double)(int)(x + 0.5) : x - (double)(int)(x - 0.5);
}

// Value::difference (src/core/Value.h:405-416): d2 - d1, wrapped when periodic
__device__ __forceinline__ double vdiff(const GridArg& G, int i, double d1, double d2) {
  if (!G.pbc[i]) return d2 - d1;
  double s = (d2 - d1) * G.inv_period[i];
  s = mpbc1(s);
  return s * G.period[i];
}

// getIndices(x) + getIndex (Grid.cpp:108-132): -1 outside the grid
__device__ long long grid_index_of(const GridArg& G, const double* x, unsigned* ind) {
  for (int i = 0; i < G.ncv; i++) {
    double f = floor((x[i] - G.min[i]) / G.dx[i]);
    if (!(f >= 0.0) || f >= (double)G.nbin[i]) return -1;
    ind[i] = (unsigned)f;
  }
  long long index = ind[G.ncv - 1];
  for (int i = G.ncv - 1; i > 0; --i) index = index * G.nbin[i - 1] + ind[i - 1];
  return index;
}

__device__ __forceinline__ long long flat(const GridArg& G, const unsigned* ind) {
  long long index = ind[G.ncv - 1];
  for (int i = G.ncv - 1; i > 0; --i) index = index * G.nbin[i - 1] + ind[i - 1];
  return index;
}

// spline value and gradient at x; returns false outside the grid
__device__ bool spline(const GridArg& G, const double* __restrict__ val, const double* __restrict__ der,
                       const double* x, double& value, double* dv) {
  unsigned ind[kMaxCv];
  for (int i = 0; i < G.ncv; i++) dv[i] = 0.0;
  value = 0.0;
  if (grid_index_of(G, x, ind) < 0) return false;
  double xfloor[kMaxCv];
  for (int i = 0; i < G.ncv; i++) xfloor[i] = G.min[i] + (double)ind[i] * G.dx[i];
  const unsigned nn = 1u << G.ncv;
  for (unsigned ip = 0; ip < nn; ip++) {
    unsigned ni[kMaxCv];
    unsigned t = ip;
    int cnt = 0;
    for (int j = 0; j < G.ncv; j++) {
      unsigned i0 = t % 2 + ind[j];
      t /= 2;
      if (!G.pbc[j] && i0 == G.nbin[j]) continue;
      if (G.pbc[j] && i0 == G.nbin[j]) i0 = 0;
      ni[cnt++] = i0;
    }
    if (cnt != G.ncv) continue;
    const long long node = flat(G, ni);
    const double grid = val[node];
    double C[kMaxCv], D[kMaxCv], ff = 1.0;
    for (int j = 0; j < G.ncv; j++) {
      // ni[j] equals ind[j] or the next node (possibly wrapped)
      const int x0 = (ni[j] == ind[j]) ? 0 : 1;
      const double dx = G.dx[j];
      const double X = fabs((x[j] - xfloor[j]) / dx - (double)x0);
      const double X2 = X * X, X3 = X2 * X;
      const double yy = fabs(grid) < 0.0000001 ? 0.0 : -der[node * G.ncv + j] / grid;
      const double sg = x0 ? -1.0 : 1.0;
      C[j] = (1.0 - 3.0 * X2 + 2.0 * X3) - sg * yy * (X - 2.0 * X2 + X3) * dx;
      D[j] = (-6.0 * X + 6.0 * X2) - sg * yy * (1.0 - 4.0 * X + 3.0 * X2) * dx;
      D[j] *= sg / dx;
      ff *= C[j];
    }
    for (int j = 0; j < G.ncv; j++) {
      double fd = D[j];
      for (int i = 0; i < G.ncv; i++)
        if (i != j) fd *= C[i];
      dv[j] += grid * fd;
    }
    value += grid * ff;
  }
  return true;
}

// Value and gradient (d) of one hill of height h at the node point xx
// (MetaD.cpp:2244-2275, diagonal); 0 beyond the cutoff
__device__ __forceinline__ double gaussian(const GridArg& G, const double* xx, const double* c, double h,
                                           double* d) {
  double dp[kMaxCv], dp2 = 0.0;
#pragma unroll
  for (int i = 0; i < kMaxCv; i++) {
    if (i >= G.ncv) break;
    d[i] = 0.0;
    dp[i] = vdiff(G, i, c[i], xx[i]) * G.invsigma[i];
    dp2 += dp[i] * dp[i];
  }
  dp2 *= 0.5;
  if (!(dp2 < 6.25)) return 0.0;
  const double bias = h * exp(-dp2);
#pragma unroll
  for (int i = 0; i < kMaxCv; i++) {
    if (i >= G.ncv) break;
    d[i] = -bias * dp[i] * G.invsigma[i] * G.stretchA;
  }
  return G.stretchA * bias + h * G.stretchB;
}

// node of support offset `s` around the bin `ind` (GridBase::getNeighbors,
// Grid.cpp:55-106); false when it falls outside a non-periodic direction
__device__ __forceinline__ bool support_node(const GridArg& G, const unsigned* ind, int s, unsigned* node_ind) {
  for (int i = 0; i < G.ncv; i++) {
    const int w = 2 * G.nneigh[i] + 1;
    const int o = s % w;
    s /= w;
    int i0 = o - G.nneigh[i] + (int)ind[i];
    if (!G.pbc[i] && (i0 < 0 || i0 >= (int)G.nbin[i])) return false;
    if (G.pbc[i] && i0 < 0) i0 = G.nbin[i] - (-i0) % G.nbin[i];
    if (G.pbc[i] && i0 >= (int)G.nbin[i]) i0 %= G.nbin[i];
    node_ind[i] = (unsigned)i0;
  }
  return true;
}

// One hill at a node, as every deposition in hill order forms it.  Per CV:
// s = dp^2/2 of the scaled distance dp, the factor f = exp(-s), and w, dp
// times the gradient's constant; the shape is the product of the factors
// (exp(-dp^2/2) up to rounding, so that the factors of a grid line serve all
// its nodes), and the value and gradient receive fma(height, term, .).  The
// heights' corners and the grid nodes go through the same operations in the
// same order, so a node holds the same bits however the hills were grouped.
struct HillDim {
  double s, f, w;
};
// scaled distance along CV i; PER: some CV is periodic
template <bool PER>
__device__ __forceinline__ double hill_scaled(const GridArg& G, int i, double c, double x) {
  if constexpr (PER) return vdiff(G, i, c, x) * G.invsigma[i];
  return (x - c) * G.invsigma[i];
}
template <bool PER>
__device__ __forceinline__ HillDim hill_dim(const GridArg& G, int i, double c, double x) {
  HillDim H;
  const double dp = hill_scaled<PER>(G, i, c, x);
  H.s = 0.5 * (dp * dp);
  H.f = exp_core(-H.s);
  H.w = dp * G.kd[i];
  return H;
}
// the shape (negative beyond the cutoff: no term)
template <int NCV>
__device__ __forceinline__ double hill_shape(const HillDim* H) {
  double s = H[0].s, e = H[0].f;
#pragma unroll
  for (int i = 1; i < NCV; i++) {
    s += H[i].s;
    e *= H[i].f;
  }
  return s < 6.25 ? e : -1.0;
}

// add one hill of height h centred at c to the grid, all threads of the block
// (distinct nodes per thread unless may_alias, then thread 0 alone)
template <int NCV>
__device__ void add_hill_block(const GridArg& G, double* __restrict__ val, double* __restrict__ der,
                               const unsigned* ind, const double* c, double h) {
  const int t0 = G.may_alias ? 0 : (int)threadIdx.x;
  const int step = G.may_alias ? 1 : (int)blockDim.x;
  if (G.may_alias && threadIdx.x != 0) return;
  for (int s = t0; s < G.support; s += step) {
    unsigned ni[kMaxCv];
    if (!support_node(G, ind, s, ni)) continue;
    const long long node = flat(G, ni);
    double d[NCV];
    // the node's values are on their way while the factors are formed
    const double v = val[node];
#pragma unroll
    for (int i = 0; i < NCV; i++) d[i] = der[node * NCV + i];
    HillDim H[NCV];
#pragma unroll
    for (int i = 0; i < NCV; i++) H[i] = hill_dim<true>(G, i, c[i], G.min[i] + (double)ni[i] * G.dx[i]);
    const double e = hill_shape<NCV>(H);
    if (e < 0.0) continue;
    val[node] = fma(h, fma(G.stretchA, e, G.stretchB), v);
#pragma unroll
    for (int i = 0; i < NCV; i++) der[node * NCV + i] = fma(h, e * H[i].w, d[i]);
  }
}

// MetaD::getHeight (MetaD.cpp:2280-2305): height0 exp(-V / (kbt (biasf - 1)));
// the division is a product with its reciprocal, formed once on the host, so
// that the sequential chain of heights carries no division (the heights move
// by about one rounding of the exponent's argument).  2^n height0 is formed
// beside the polynomial.
__device__ __forceinline__ double wt_fast(double height0, double inv_wt, double inv_wt2, double vbias,
                                          const ExpK& C) {
  const double n = rint(vbias * -inv_wt2);
  const double h = ldexp(height0, (int)n);
  return fma(exp_part(-vbias * inv_wt, n, C), h, h);
}
// where wt_fast holds: finite heights of any run
__device__ __forceinline__ bool wt_in_range(double inv_wt, double vbias) { return fabs(vbias * inv_wt) < 700.0; }
__device__ __forceinline__ double wt_height(const GridArg& G, double vbias) {
  if (!G.welltemp) return G.height0;
  if (wt_in_range(G.inv_wt, vbias)) return wt_fast(G.height0, G.inv_wt, G.inv_wt * ExpK().log2e, vbias, ExpK());
  return G.height0 * exp(-vbias * G.inv_wt);
}

// value and gradient terms of the corner ip of the cell of x: the terms
// `value += grid * ff` and `dv[j] += grid * fd` of GridBase::getValueAndDerivatives
// (Grid.cpp:442-505) for one ip, with the arithmetic of spline() above; a
// corner past the last node of a non-periodic CV gives zeros
__device__ void spline_corner_grad(const GridArg& G, const double* __restrict__ val, const double* __restrict__ der,
                                   const double* x, const unsigned* ind, unsigned ip, double& value, double* dv) {
  value = 0.0;
#pragma unroll
  for (int j = 0; j < kMaxCv; j++) dv[j] = 0.0;
  unsigned ni[kMaxCv];
  unsigned t = ip;
  int cnt = 0;
  for (int j = 0; j < G.ncv; j++) {
    unsigned i0 = t % 2 + ind[j];
    t /= 2;
    if (!G.pbc[j] && i0 == G.nbin[j]) continue;
    if (G.pbc[j] && i0 == G.nbin[j]) i0 = 0;
    ni[cnt++] = i0;
  }
  if (cnt != G.ncv) return;
  const long long node = flat(G, ni);
  const double grid = val[node];
  double C[kMaxCv], D[kMaxCv], ff = 1.0;
#pragma unroll
  for (int j = 0; j < kMaxCv; j++) {
    C[j] = 1.0;
    D[j] = 0.0;
    if (j >= G.ncv) continue;
    const int x0 = (ni[j] == ind[j]) ? 0 : 1;
    const double dx = G.dx[j];
    const double xfloor = G.min[j] + (double)ind[j] * dx;
    const double X = fabs((x[j] - xfloor) / dx - (double)x0);
    const double X2 = X * X, X3 = X2 * X;
    const double yy = fabs(grid) < 0.0000001 ? 0.0 : -der[node * G.ncv + j] / grid;
    const double sg = x0 ? -1.0 : 1.0;
    C[j] = (1.0 - 3.0 * X2 + 2.0 * X3) - sg * yy * (X - 2.0 * X2 + X3) * dx;
    D[j] = (-6.0 * X + 6.0 * X2) - sg * yy * (1.0 - 4.0 * X + 3.0 * X2) * dx;
    D[j] *= sg / dx;
    ff *= C[j];
  }
#pragma unroll
  for (int j = 0; j < kMaxCv; j++) {
    if (j >= G.ncv) continue;
    double fd = D[j];
#pragma unroll
    for (int i = 0; i < kMaxCv; i++)
      if (i != j && i < G.ncv) fd *= C[i];
    dv[j] = grid * fd;
  }
  value = grid * ff;
}

// ------------------------------------------------------------------------
// deposition of hills in order
// ------------------------------------------------------------------------

// 1/x without the scaling steps of a division (|x| is at least 1e-7 where it
// counts): v_rcp_f64, good to 2^-23, and one step of third order
__device__ __forceinline__ double rcp64(double x) {
  const double r = __builtin_amdgcn_rcp(x);
  const double e = fma(-x, r, 1.0);
  return fma(r, fma(e, e, e), r);
}

template <int CTRL>
__device__ __forceinline__ double dpp_m(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_mov_dpp((int)(b & 0xffffffffll), CTRL, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), CTRL, 0xF, 0xF, true);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
// sum over the aligned group of 2^NCV lanes, in every lane of it
template <int NCV>
__device__ __forceinline__ double corner_sum(double v) {
  v += dpp_m<0xB1>(v);                             // quad_perm 1,0,3,2
  if constexpr (NCV >= 2) v += dpp_m<0x4E>(v);     // quad_perm 2,3,0,1
  if constexpr (NCV >= 3) v += dpp_m<0x141>(v);    // row_half_mirror
  if constexpr (NCV >= 4) v += dpp_m<0x140>(v);    // row_mirror
  return v;
}
// value of lane `l` (uniform) of a double, through the scalar unit
__device__ __forceinline__ double readlane_d(double v, int l) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffll), l);
  const int hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// One corner of the spline cell of a hill centre: the node, its coordinates,
// and the parts of the spline term (Grid.cpp:442-505) that depend on the
// position only: the term `grid * prod_j C_j` with C_j = A_j + S_j der_j/grid.
template <int NCV>
struct Corner {
  bool has;           // false past the last node of a non-periodic CV
  int n[NCV];
  double x[NCV], A[NCV], S[NCV];
};
template <int NCV>
__device__ __forceinline__ Corner<NCV> corner_of(const GridArg& G, const double* c, const int* ind, int q) {
  Corner<NCV> K;
  K.has = true;
#pragma unroll
  for (int i = 0; i < NCV; i++) {
    int n = ind[i] + ((q >> i) & 1);
    if (n >= (int)G.nbin[i]) {
      if (G.pbc[i]) n = 0;
      else K.has = false;
    }
    K.n[i] = n;
    const int x0 = n == ind[i] ? 0 : 1;
    const double dx = G.dx[i];
    K.x[i] = G.min[i] + (double)n * dx;
    const double X = fabs((c[i] - (G.min[i] + (double)ind[i] * dx)) / dx - (double)x0);
    const double X2 = X * X, X3 = X2 * X;
    K.A[i] = 1.0 - 3.0 * X2 + 2.0 * X3;
    K.S[i] = (x0 ? -1.0 : 1.0) * (X - 2.0 * X2 + X3) * dx;
  }
  return K;
}
template <int NCV>
__device__ __forceinline__ long long corner_node(const GridArg& G, const Corner<NCV>& K) {
  long long node = K.n[NCV - 1];
#pragma unroll
  for (int i = NCV - 1; i > 0; --i) node = node * G.nbin[i - 1] + K.n[i - 1];
  return node;
}
// the spline term from the node's value g and gradient d: the product of
// A_j g + S_j d_j over a power of g, so that one reciprocal is all the division
// on the way from one height to the next; below 1e-7 the gradient does not
// count (an absent corner has g = 0 and gives 0)
template <int NCV>
__device__ __forceinline__ double corner_term(const Corner<NCV>& K, double g, const double* d) {
  double flat = g, v = fma(K.S[0], d[0], K.A[0] * g);
  double r = 1.0;
  if constexpr (NCV > 1) {
    const double r1 = rcp64(g);
    r = r1;
#pragma unroll
    for (int i = 2; i < NCV; i++) r *= r1;
  }
#pragma unroll
  for (int i = 0; i < NCV; i++) flat *= K.A[i];
#pragma unroll
  for (int i = 1; i < NCV; i++) v *= fma(K.S[i], d[i], K.A[i] * g);
  v *= r;
  return fabs(g) < 0.0000001 ? flat : v;
}

// Hills one after the other in one workgroup: per hill, one wave evaluates
// the 2^NCV spline corners and the height, then the workgroup adds the hill,
// one support node per thread (two L2 round trips a hill).  For the few
// hills of a run in progress, and for periodic supports wider than the
// grid.  Bit for bit the heights and the grid of the kernels below.
constexpr int kSeqThreads = 1024;
template <int NCV>
__global__ __launch_bounds__(kSeqThreads) void k_deposit_seq(GridArg G, double* __restrict__ val,
                                                             double* __restrict__ der, long long nhills,
                                                             const double* __restrict__ centers,
                                                             double* __restrict__ heights, int* __restrict__ err) {
  __shared__ double sh_h;
  const int t = threadIdx.x;
  for (long long k = 0; k < nhills; k++) {
    double c[kMaxCv];
    unsigned ind[kMaxCv];
    for (int i = 0; i < NCV; i++) c[i] = centers[k * NCV + i];
    const bool ok = grid_index_of(G, c, ind) >= 0;  // uniform
    if (t < WAVE_M) {
      double v = 0.0;
      if (ok && G.welltemp && t < (1 << NCV)) {
        int in[NCV];
        for (int i = 0; i < NCV; i++) in[i] = (int)ind[i];
        const Corner<NCV> K = corner_of<NCV>(G, c, in, t);
        if (K.has) {
          const long long node = corner_node<NCV>(G, K);
          double d[NCV];
          for (int i = 0; i < NCV; i++) d[i] = der[node * NCV + i];
          v = corner_term<NCV>(K, val[node], d);
        }
      }
      v = corner_sum<NCV>(v);
      if (t == 0) {
        const double h = (ok && G.welltemp) ? wt_height(G, v) : G.height0;
        if (!ok) atomicCAS(err, 0, (int)(1 + (k < 0x3fffffff ? k : 0x3fffffff)));
        sh_h = h;
        if (heights) heights[k] = ok ? h : 0.0;
      }
    }
    __syncthreads();
    if (!ok) return;
    add_hill_block<NCV>(G, val, der, ind, c, sh_h);
    __syncthreads();
  }
}

// Many hills: epochs of kChainThreads / 2^NCV hills (256 with two CVs), two
// launches each.
//  - k_hill_chain finds the epoch's heights in one workgroup.  Thread t holds
//    corner t mod 2^NCV of hill t / 2^NCV in registers: its value and gradient
//    on the grid before the epoch, to which every earlier hill of the epoch is
//    added as soon as its height is known.  Wave w owns a run of
//    64 / 2^NCV hills: it finds their heights alone, one after the other (the
//    corners of hill k give its height, then all later corners of the wave
//    take hill k), and the later waves follow hill by hill through LDS, so
//    that the next wave is one hill behind when its turn comes.
//    The other workgroups of the launch evaluate the next epoch's shapes,
//    which depend on the centres only: those exponentials are off the chain.
//  - k_hill_nodes adds the epoch to the grid, a thread per node with the
//    hills in order.
// Bound by the latency of the chain height -> corners -> reciprocal ->
// exponential -> height on one wave (0.23 us a hill: some 22 dependent FP64
// operations).  Measured, one workgroup doing everything before -> this: 4,000
// hills on two open CVs (513 x 513 nodes) 4.93 ms -> 0.93 ms (heights) + 0.30 ms
// (grid); 500 hills on two torsions (100 x 100) 3.60 -> 0.21 ms.
constexpr int kChainThreads = 1024;
constexpr int kSeqHills = 4;  // at most this many hills go one after the other

// cells of the hill centres (-1: outside the grid)
template <int NCV>
__global__ __launch_bounds__(256) void k_hill_cells(GridArg G, long long n, const double* __restrict__ centers,
                                                    int* __restrict__ cells) {
  const long long k = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  double c[kMaxCv];
  unsigned ind[kMaxCv];
  for (int i = 0; i < NCV; i++) c[i] = centers[k * NCV + i];
  const bool ok = grid_index_of(G, c, ind) >= 0;
  for (int i = 0; i < NCV; i++) cells[k * NCV + i] = ok ? (int)ind[i] : -1;
}

// node n within the support of a hill in bin `ind`
__device__ __forceinline__ bool in_support(const GridArg& G, int i, int n, int ind) {
  int d = abs(n - ind);
  if (G.pbc[i]) d = min(d, (int)G.nbin[i] - d);
  return d <= G.nneigh[i];
}

// hills of one epoch: their first index in the call and count, centres and cells
struct Epoch {
  long long k0;
  int n;
  const double* centers;
  const int* cells;
};

template <int NCV, bool PER>
__global__ __launch_bounds__(kChainThreads) void k_hill_chain(GridArg G, const double* __restrict__ val,
                                                              const double* __restrict__ der, Epoch E,
                                                              const double* __restrict__ shapes, Epoch N,
                                                              double* __restrict__ shapes_next, int first,
                                                              int* __restrict__ state, double* __restrict__ hbuf,
                                                              double* __restrict__ heights, int* __restrict__ err) {
  constexpr int NN = 1 << NCV;
  constexpr int R = WAVE_M / NN;           // hills of one run
  constexpr int RC = R < 16 ? R : 16;      // hills whose shapes are in registers at once
  constexpr int EH = kChainThreads / NN;   // hills of one epoch
  const int t = threadIdx.x;
  const int r = t / NN, q = t % NN;
  if (blockIdx.x > 0) {
    // row j of the next epoch's shapes: hill j at the corners of the later hills
    const int j = (int)blockIdx.x - 1;
    if (j >= N.n || r / R < j / R) return;
    double e = -1.0;
    if (j < r && r < N.n) {
      HillDim H[NCV];
      bool in = true;
#pragma unroll
      for (int i = 0; i < NCV; i++) {
        int n = N.cells[r * NCV + i] + ((q >> i) & 1);
        if (n >= (int)G.nbin[i]) {
          if (G.pbc[i]) n = 0;
          else in = false;
        }
        in = in && in_support(G, i, n, N.cells[j * NCV + i]);
        H[i] = hill_dim<PER>(G, i, N.centers[j * NCV + i], G.min[i] + (double)n * G.dx[i]);
      }
      if (in) e = hill_shape<NCV>(H);
    }
    shapes_next[(size_t)j * kChainThreads + t] = e;
    return;
  }
  if (E.n == 0) return;
  __shared__ double sh_c[EH][NCV], sh_h[EH];
  __shared__ int sh_bad;
  const int lane = t & (WAVE_M - 1);
  const int w = __builtin_amdgcn_readfirstlane(t / WAVE_M);
  // state[0..1]: hills of the epoch before the first one outside the grid;
  // state[2..3]: that one has been met (this epoch's parity and the last's)
  const int par = (int)((E.k0 / EH) & 1);
  const bool stopped = !first && state[2 + (1 - par)] != 0;
  if (t == 0) sh_bad = stopped ? 0 : E.n;
  // a height not found yet: a NaN with a payload that only an input could
  // carry on, and the inputs' NaNs lose theirs below; so the word itself tells
  // the followers
  constexpr long long kPending = 0x7ff8c0ffee0dd001ll;
  auto plain = [](double x) { return x == x ? x : __builtin_nan(""); };
  if (t < EH) sh_h[t] = __longlong_as_double(kPending);
  __syncthreads();
  if (t < E.n) {
    bool ok = true;
    for (int i = 0; i < NCV; i++) {
      ok = ok && E.cells[t * NCV + i] >= 0;
      sh_c[t][i] = E.centers[t * NCV + i];
    }
    if (!ok) atomicMin(&sh_bad, t);
  }
  __syncthreads();
  const int cnt = __builtin_amdgcn_readfirstlane(sh_bad);
  if (t == 0) {
    state[par] = cnt;
    state[2 + par] = cnt < E.n;
    if (!stopped && cnt < E.n) {
      const long long k = E.k0 + cnt;
      atomicCAS(err, 0, (int)(1 + (k < 0x3fffffff ? k : 0x3fffffff)));
      if (heights) heights[k] = 0.0;
    }
  }
  double* hb = hbuf + (size_t)par * EH;
  if (!G.welltemp) {
    if (t < cnt) {
      hb[t] = G.height0;
      if (heights) heights[E.k0 + t] = G.height0;
    }
    return;
  }
  if (w * R < cnt) {
    // this thread's corner on the grid before the epoch
    const bool mine = r < cnt;
    Corner<NCV> K;
    double g = 0.0, d[NCV];
    {
      double c[NCV];
      int ind[NCV];
#pragma unroll
      for (int i = 0; i < NCV; i++) {
        c[i] = mine ? sh_c[r][i] : G.min[i];
        ind[i] = mine ? E.cells[r * NCV + i] : 0;
        d[i] = 0.0;
      }
      K = corner_of<NCV>(G, c, ind, q);
      if (mine && K.has) {
        const long long node = corner_node<NCV>(G, K);
        g = plain(val[node]);
#pragma unroll
        for (int i = 0; i < NCV; i++) d[i] = plain(der[node * NCV + i]);
      }
    }
    // constants of the chain in registers
    ExpK C;
    double height0 = plain(G.height0), inv_wt = plain(G.inv_wt);
    double inv_wt2 = inv_wt * C.log2e;
    double sA = G.stretchA, sB = G.stretchB;
    asm volatile("" : "+s"(C.hi), "+s"(C.lo), "+s"(sA), "+v"(sB), "+v"(height0), "+v"(inv_wt), "+v"(inv_wt2));
#pragma unroll
    for (int i = 0; i < 6; i++) asm volatile("" : "+s"(C.m[i]));
#pragma unroll
    for (int i = 0; i < 5; i++) asm volatile("" : "+v"(C.a[i]));
    const double* sh = shapes + t;
    auto load = [&](int b, double* e) {
#pragma unroll
      for (int k = 0; k < RC; k++) e[k] = b + k < cnt ? sh[(size_t)(b + k) * kChainThreads] : -1.0;
    };
    // the terms of hill k of shape e at this thread's corner, all but the
    // height (0 outside the support), formed where this stands
    auto terms = [&](int k, double e, double& tv, double* td) {
      const bool in = e >= 0.0;
      tv = in ? fma(sA, e, sB) : 0.0;
      const double ez = in ? e : 0.0;
      double c[NCV];
#pragma unroll
      for (int i = 0; i < NCV; i++) c[i] = sh_c[k][i];
#pragma unroll
      for (int i = 0; i < NCV; i++) td[i] = ez * (hill_scaled<PER>(G, i, c[i], K.x[i]) * G.kd[i]);
      asm volatile("" : "+v"(tv));
#pragma unroll
      for (int i = 0; i < NCV; i++) asm volatile("" : "+v"(td[i]));
    };
    auto apply = [&](double h, double tv, const double* td) {
      g = fma(h, tv, g);
#pragma unroll
      for (int i = 0; i < NCV; i++) d[i] = fma(h, td[i], d[i]);
    };
    // height k of an earlier wave, as soon as it is there (every wave of the
    // workgroup is resident and only waits for earlier ones)
    auto height = [&](int k) {
      while (true) {
        const double h = __hip_atomic_load(&sh_h[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        if (__double_as_longlong(h) != kPending) return h;
        __builtin_amdgcn_s_sleep(1);
      }
    };
    // the hills [b, b + RC) of an earlier wave, each as soon as it is there
    auto follow = [&](int b, const double* e) {
#pragma unroll
      for (int k = 0; k < RC; k++) {
        if (__ballot(e[k] >= 0.0) == 0ull) continue;
        double tv, td[NCV];
        terms(b + k, e[k], tv, td);
        const double h = height(b + k);
        if (e[k] >= 0.0) apply(h, tv, td);
      }
    };
    double ex[RC], eo[RC];
    const int b0 = w * R;
    for (int b = 0; b + RC < b0; b += RC) {
      load(b, ex);
      follow(b, ex);
    }
    if (b0 > 0) load(b0 - RC, ex);
    load(b0, eo);
    if (b0 > 0) {
      follow(b0 - RC, ex);
      (void)height(b0 - 1);
    }
    __builtin_amdgcn_s_setprio(3);
    for (int c = 0; c < R / RC; c++) {
      const int b = b0 + c * RC;
      if (c > 0) load(b, eo);
      // (the hills of this wave's earlier chunks are in: every lane took them)
      double tv, td[NCV];
      terms(b, eo[0], tv, td);
#pragma unroll
      for (int k = 0; k < RC; k++) {
        if (b + k < cnt) {
          const double V = readlane_d(corner_sum<NCV>(corner_term<NCV>(K, g, d)), NN * (c * RC + k));
          // the next hill's terms fill the waits of this hill's exponential
          double tn = 0.0, dn[NCV];
          if (k + 1 < RC) terms(b + k + 1, eo[k + 1], tn, dn);
          double h = wt_fast(height0, inv_wt, inv_wt2, V, C);
          if (__builtin_expect(!wt_in_range(inv_wt, V), 0)) {
            h = height0 * exp(-V * inv_wt);
            if (eo[k] >= 0.0) apply(h, tv, td);
          } else {
            apply(h, tv, td);
          }
          if (lane == 0) __hip_atomic_store(&sh_h[b + k], h, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
          tv = tn;
#pragma unroll
          for (int i = 0; i < NCV; i++) td[i] = k + 1 < RC ? dn[i] : 0.0;
        }
      }
    }
    __builtin_amdgcn_s_setprio(0);
  }
  __syncthreads();
  if (t < cnt) {
    hb[t] = sh_h[t];
    if (heights) heights[E.k0 + t] = sh_h[t];
  }
}

// tiles of 64 nodes (one wave): the smaller the tile, the fewer hills it meets
template <int NCV>
__host__ __device__ constexpr int tile_dim(int i) {
  return NCV == 1 ? 64 : NCV == 2 ? 8 : NCV == 3 ? 4 : (i < 2 ? 4 : 2);
}

// The hills of one epoch onto the grid: a workgroup per tile, which lists the
// hills that reach it (in order) and tabulates HillDim of each along the
// tile's sides; wave 0 then takes its nodes' hills in order, four at a time up
// to the addition, while the other waves tabulate the next hills.  Bound by
// wave 0's walk through the hills of the busiest tiles.  Tiles that no hill
// reaches leave after the list.
// The workgroups are the tiles of the grid or, where that is fewer, `per` tiles
// around each hill, of which the first hill that reaches a tile takes it: the
// launch then follows the supports, not the grid.  A host call with 5 hills on
// 90^4 nodes: 2,760 us over all tiles, their nodes read at once, now 71 (4 hills
// one after the other: 450); on 8,000 x 8,000 nodes 1,100 -> 52, with 512 hills
// 2,320 -> 328.
struct TileMap {
  int per;         // 0: the tiles of the grid
  int early;       // nodes read before it is known whether a hill reaches the tile
  int n[kMaxCv];   // tiles along each CV that a hill's support can reach
};
template <int NCV, bool PER>
__global__ __launch_bounds__(256) void k_hill_nodes(GridArg G, double* __restrict__ val, double* __restrict__ der,
                                                    Epoch E, TileMap M, const int* __restrict__ state,
                                                    const double* __restrict__ hbuf) {
  constexpr int EH = kChainThreads >> NCV;
  constexpr int ST = NCV == 1 ? 64 : NCV == 2 ? 16 : 12;  // sum of the tile's sides
  constexpr int CH = NCV == 1 ? 8 : 32;                   // hills tabulated at once
  constexpr int U = 4;
  // the hills that reach the tile, in order: cell, centre, height
  __shared__ int lcell[EH][NCV];
  __shared__ double lx[EH][NCV], lh[EH];
  constexpr int HP = (EH + 255) / 256;
  __shared__ int2 whit[HP][4];  // a wave's hits and the first of them
  __shared__ double2 tsf[2][CH][ST];
  __shared__ double tw[2][CH][ST];
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  const int par = (int)((E.k0 / EH) & 1);
  const double* hb = hbuf + (size_t)par * EH;
  const int cnt = state[par];
  int o[NCV], owner = 0;
  if (M.per == 0) {
    unsigned b = blockIdx.x;
#pragma unroll
    for (int i = 0; i < NCV; i++) {
      const unsigned nt = (G.nbin[i] + tile_dim<NCV>(i) - 1) / tile_dim<NCV>(i);
      o[i] = (int)(b % nt) * tile_dim<NCV>(i);
      b /= nt;
    }
  } else {
    owner = (int)(blockIdx.x / (unsigned)M.per);
    if (owner >= cnt) return;  // uniform, as the returns below
    unsigned b = blockIdx.x % (unsigned)M.per;
#pragma unroll
    for (int i = 0; i < NCV; i++) {
      const int N = (int)G.nbin[i], nt = (int)((G.nbin[i] + tile_dim<NCV>(i) - 1) / tile_dim<NCV>(i));
      int a = E.cells[owner * NCV + i] - G.nneigh[i];  // the support's first node
      if (a < 0) a = G.pbc[i] ? a + N : 0;
      int q = a / tile_dim<NCV>(i) + (int)(b % (unsigned)M.n[i]);
      if (q >= nt) {
        if (!G.pbc[i]) return;
        q -= nt;
      }
      o[i] = q * tile_dim<NCV>(i);
      b /= (unsigned)M.n[i];
    }
  }
  // the epoch's hills (E.n of them, valid or not)
  int cell[HP][NCV];
  double x[HP][NCV], hh[HP];
#pragma unroll
  for (int p = 0; p < HP; p++) {
    const int h = min(p * 256 + t, E.n - 1);
    hh[p] = hb[h];
#pragma unroll
    for (int i = 0; i < NCV; i++) {
      cell[p][i] = E.cells[h * NCV + i];
      x[p][i] = E.centers[h * NCV + i];
    }
  }
  int l[NCV];
  bool valid = w == 0;
  long long node = 0;
  {
    int q = lane, base = 0, n[NCV];
#pragma unroll
    for (int i = 0; i < NCV; i++) {
      const int a = q % tile_dim<NCV>(i);
      q /= tile_dim<NCV>(i);
      n[i] = o[i] + a;
      l[i] = base + a;
      base += tile_dim<NCV>(i);
      valid = valid && n[i] < (int)G.nbin[i];
    }
    node = n[NCV - 1];
#pragma unroll
    for (int i = NCV - 1; i > 0; --i) node = node * G.nbin[i - 1] + n[i - 1];
  }
  // wave 0's node: on its way while the list is made, or while the tables are formed
  double v = 0.0, d[NCV];
#pragma unroll
  for (int i = 0; i < NCV; i++) d[i] = 0.0;
  auto load = [&]() {
    if (!valid) return;
    v = val[node];
#pragma unroll
    for (int i = 0; i < NCV; i++) d[i] = der[node * NCV + i];
  };
  if (M.early) load();
  bool hit[HP];
  int below[HP];  // hits of this wave before this lane's
#pragma unroll
  for (int p = 0; p < HP; p++) {
    hit[p] = p * 256 + t < cnt;
#pragma unroll
    for (int i = 0; i < NCV; i++) {
      const int T = min(tile_dim<NCV>(i), (int)G.nbin[i] - o[i]);
      int s = o[i] - (cell[p][i] - G.nneigh[i]);  // the tile's first node from the support's first
      if (PER && G.pbc[i]) {
        const int N = (int)G.nbin[i];
        if (s < 0) s += N;  // |o - cell| < N and the support is no wider than the grid
        else if (s >= N) s -= N;
        hit[p] = hit[p] && (s <= 2 * G.nneigh[i] || s + T - 1 >= N);
      } else {
        hit[p] = hit[p] && s <= 2 * G.nneigh[i] && s + T - 1 >= 0;
      }
    }
    const unsigned long long m = __ballot(hit[p]);
    below[p] = __popcll(m & ((1ull << lane) - 1));
    if (lane == 0) whit[p][w] = make_int2(__popcll(m), m ? p * 256 + w * WAVE_M + __ffsll((long long)m) - 1 : INT_MAX);
  }
  __syncthreads();
  int nl = 0, first = INT_MAX;
#pragma unroll
  for (int p = 0; p < HP; p++)
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int2 h = whit[p][q];
      if (q == w) below[p] += nl;
      nl += h.x;
      first = min(first, h.y);
    }
  if (nl == 0 || (M.per && first != owner)) return;
#pragma unroll
  for (int p = 0; p < HP; p++) {
    if (!hit[p]) continue;
    const int at = below[p];
    lh[at] = hh[p];
#pragma unroll
    for (int i = 0; i < NCV; i++) {
      lcell[at][i] = cell[p][i];
      lx[at][i] = x[p][i];
    }
  }
  __syncthreads();
  if (!M.early) load();
  // the tables of the hills [c0, c0 + CH) of the list, by threads q0, q0 + step, ...
  auto tabulate = [&](int c0, int buf, int q0, int step) {
    const int nc = min(CH, nl - c0);
    for (int p = q0; p < nc * ST; p += step) {
      const int c = p / ST;
      int m = p % ST, i = 0;
#pragma unroll
      for (int u = 0; u < NCV - 1; u++)
        if (i == u && m >= tile_dim<NCV>(u)) {
          m -= tile_dim<NCV>(u);
          i = u + 1;
        }
      // a distance beyond the cutoff marks the nodes outside the support
      HillDim H = {1.0e3, 0.0, 0.0};
#pragma unroll
      for (int u = 0; u < NCV; u++) {
        if (i != u) continue;
        const int nd = o[u] + m;
        if (nd < (int)G.nbin[u] && in_support(G, u, nd, lcell[c0 + c][u]))
          H = hill_dim<PER>(G, u, lx[c0 + c][u], G.min[u] + (double)nd * G.dx[u]);
      }
      tsf[buf][c][p % ST] = make_double2(H.s, H.f);
      tw[buf][c][p % ST] = H.w;
    }
  };
  tabulate(0, 0, t, 256);
  __syncthreads();
  for (int c0 = 0, buf = 0; c0 < nl; c0 += CH, buf ^= 1) {
    if (w > 0) {
      tabulate(c0 + CH, buf ^ 1, t - WAVE_M, 256 - WAVE_M);
    } else {
      const int nc = min(CH, nl - c0);
      // the next hills' entries are on their way while these are added
      HillDim H[U][NCV];
      double h[U];
      auto fetch = [&](int cc) {
#pragma unroll
        for (int u = 0; u < U; u++) {
          const int c = min(cc + u, nc - 1);
          h[u] = lh[c0 + c];
#pragma unroll
          for (int i = 0; i < NCV; i++) {
            const double2 y = tsf[buf][c][l[i]];
            H[u][i] = {y.x, y.y, tw[buf][c][l[i]]};
          }
        }
      };
      fetch(0);
      for (int cc = 0; cc < nc; cc += U) {
        double e[U], tv[U], td[U][NCV], hc[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
          e[u] = hill_shape<NCV>(H[u]);
          tv[u] = fma(G.stretchA, e[u], G.stretchB);
#pragma unroll
          for (int i = 0; i < NCV; i++) td[u][i] = e[u] * H[u][i].w;
          if (cc + u >= nc) e[u] = -1.0;
          hc[u] = h[u];
        }
        fetch(cc + U);
#pragma unroll
        for (int u = 0; u < U; u++) {
          if (e[u] >= 0.0) {
            asm volatile("");  // masked lanes, not selects
            v = fma(hc[u], tv[u], v);
#pragma unroll
            for (int i = 0; i < NCV; i++) d[i] = fma(hc[u], td[u][i], d[i]);
          }
        }
      }
    }
    __syncthreads();
  }
  if (!valid) return;
  val[node] = v;
#pragma unroll
  for (int i = 0; i < NCV; i++) der[node * NCV + i] = d[i];
}

// hills of given heights, in parallel (one block per hill)
__global__ __launch_bounds__(kDepositThreads) void k_add_hills(GridArg G, double* __restrict__ val,
                                                                double* __restrict__ der, long long nhills,
                                                                const double* __restrict__ centers,
                                                                const double* __restrict__ heights,
                                                                int* __restrict__ err) {
  const long long k = blockIdx.x;
  if (k >= nhills) return;
  double c[kMaxCv];
  unsigned ind[kMaxCv];
  for (int i = 0; i < G.ncv; i++) c[i] = centers[k * G.ncv + i];
  if (grid_index_of(G, c, ind) < 0) {
    if (threadIdx.x == 0) atomicCAS(err, 0, 1);
    return;
  }
  const double h = heights[k];
  for (int s = threadIdx.x; s < G.support; s += blockDim.x) {
    unsigned ni[kMaxCv];
    if (!support_node(G, ind, s, ni)) continue;
    const long long node = flat(G, ni);
    double xx[kMaxCv], d[kMaxCv];
    for (int i = 0; i < G.ncv; i++) xx[i] = G.min[i] + (double)ni[i] * G.dx[i];
    const double b = gaussian(G, xx, c, h, d);
    unsafeAtomicAdd(&val[node], b);
    for (int i = 0; i < G.ncv; i++) unsafeAtomicAdd(&der[node * G.ncv + i], d[i]);
  }
}

__global__ void k_bias(GridArg G, const double* __restrict__ val, const double* __restrict__ der, long long n,
                       const double* __restrict__ cv, double* __restrict__ bias, double* __restrict__ dout,
                       int* __restrict__ err) {
  const long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  double x[kMaxCv], v, dv[kMaxCv];
  for (int i = 0; i < G.ncv; i++) x[i] = cv[p * G.ncv + i];
  if (!spline(G, val, der, x, v, dv)) {
    atomicCAS(err, 0, 1);
    v = 0.0;
  }
  bias[p] = v;
  if (dout)
    for (int i = 0; i < G.ncv; i++) dout[p * G.ncv + i] = dv[i];
}

// MetaD::calculate + update for one step, one workgroup
__global__ __launch_bounds__(kDepositThreads) void k_metad_step(GridArg G, double* __restrict__ val,
                                                                 double* __restrict__ der,
                                                                 const double* __restrict__ cv, int deposit,
                                                                 double* __restrict__ bias,
                                                                 double* __restrict__ force,
                                                                 double* __restrict__ height,
                                                                 int* __restrict__ err) {
  __shared__ double sh_h;
  __shared__ int sh_ok;
  __shared__ unsigned sh_ind[kMaxCv];
  __shared__ double sh_c[kMaxCv];
  if (threadIdx.x < WAVE_M) {
    // lane t < 2^ncv evaluates corner t; the corners are summed in corner
    // order, as spline() adds them
    const int t = threadIdx.x;
    double c[kMaxCv] = {0.0, 0.0, 0.0, 0.0};
    unsigned ind[kMaxCv] = {0u, 0u, 0u, 0u};
    for (int i = 0; i < G.ncv; i++) c[i] = cv[i];
    int ok = grid_index_of(G, c, ind) >= 0;
    const unsigned nn = 1u << G.ncv;
    double cvv = 0.0, cdv[kMaxCv];
    if (ok && (unsigned)t < nn) {
      spline_corner_grad(G, val, der, c, ind, (unsigned)t, cvv, cdv);
    } else {
#pragma unroll
      for (int j = 0; j < kMaxCv; j++) cdv[j] = 0.0;
    }
    double v = 0.0, dv[kMaxCv] = {0.0, 0.0, 0.0, 0.0};
    for (unsigned q = 0; q < nn; q++) {
      v += __shfl(cvv, (int)q, WAVE_M);
#pragma unroll
      for (int j = 0; j < kMaxCv; j++) dv[j] += __shfl(cdv[j], (int)q, WAVE_M);
    }
    if (t == 0) {
      if (!ok) atomicCAS(err, 0, 1);
      // MetaD.cpp:2348-2350: no bias (and no force) when BIASFACTOR=1
      const bool nobias = (G.biasf == 1.0);
      if (bias) *bias = nobias ? 0.0 : v;
      if (force)
        for (int i = 0; i < G.ncv; i++) force[i] = nobias ? 0.0 : -dv[i];
      // getHeight evaluates the bias of the grid before this hill: the same v
      const double h = wt_height(G, v);
      for (int i = 0; i < G.ncv; i++) {
        sh_ind[i] = ind[i];
        sh_c[i] = c[i];
      }
      sh_h = h;
      sh_ok = ok && deposit;
      if (height) *height = (ok && deposit) ? h : 0.0;
    }
  }
  __syncthreads();
  if (!sh_ok) return;
  unsigned ind[kMaxCv];
  double c[kMaxCv];
  for (int i = 0; i < G.ncv; i++) {
    ind[i] = sh_ind[i];
    c[i] = sh_c[i];
  }
  switch (G.ncv) {
  case 1: add_hill_block<1>(G, val, der, ind, c, sh_h); break;
  case 2: add_hill_block<2>(G, val, der, ind, c, sh_h); break;
  case 3: add_hill_block<3>(G, val, der, ind, c, sh_h); break;
  default: add_hill_block<4>(G, val, der, ind, c, sh_h); break;
  }
}

__global__ void k_apply_force(long long natoms, const double* __restrict__ f, const double* __restrict__ deriv,
                              const double* __restrict__ vcv, double* __restrict__ forces,
                              double* __restrict__ virial) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const double fv = *f;
  if (i < 3 * natoms) forces[i] += fv * deriv[i];
  if (virial && vcv && i < 9) virial[i] += fv * vcv[i];
}

}  // namespace p2a

struct p2a_metad {
  int device = 0;
  hipStream_t own_stream = nullptr, stream = nullptr;
  p2a_metad_spec spec{};
  p2a::GridArg G{};
  size_t size = 0;
  double* val = nullptr;
  double* der = nullptr;
  int* err = nullptr;
  double* scratch = nullptr;  // staging for host-array entry points
  size_t scratch_n = 0;
  // workspace of the deposition in epochs, one block of a fixed size, kept until
  // the context goes (a captured deposition holds its address): shapes of two
  // epochs, heights of two epochs, two epochs' counts, cells of the hills of
  // kCellEpochs epochs and the next
  double* shapes = nullptr;
  double* hbuf = nullptr;
  int* state = nullptr;
  int* cells = nullptr;
  bool first_step = true;
};

namespace p2a {

static int metad_scratch(p2a_metad* m, size_t n) {
  if (n <= m->scratch_n) return P2A_OK;
  if (m->scratch) (void)hipFree(m->scratch);
  m->scratch = nullptr;
  m->scratch_n = 0;
  if (hipMalloc(&m->scratch, n * sizeof(double)) != hipSuccess) return fail(P2A_ERR_NOMEM, "hipMalloc failed");
  m->scratch_n = n;
  return P2A_OK;
}

// The workspace of the deposition in epochs; false when it cannot be had
// (memory, or a stream under capture, where nothing may be allocated): the
// hills then go one after the other.
constexpr int kCellEpochs = 64;
static bool epoch_workspace(p2a_metad* m) {
  if (m->shapes) return true;
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(m->stream, &cap) != hipSuccess || cap != hipStreamCaptureStatusNone) {
    (void)hipGetLastError();
    return false;
  }
  const size_t eh = kChainThreads >> m->G.ncv;
  const size_t nshape = 2 * eh * kChainThreads, nheight = 2 * eh;
  const size_t ncell = (kCellEpochs + 1) * eh * m->G.ncv;
  if (hipMalloc((void**)&m->shapes, (nshape + nheight) * sizeof(double) + (4 + ncell) * sizeof(int)) != hipSuccess) {
    m->shapes = nullptr;
    (void)hipGetLastError();
    return false;
  }
  m->hbuf = m->shapes + nshape;
  m->state = (int*)(m->hbuf + nheight);
  m->cells = m->state + 4;
  return true;
}

template <int NCV>
static void deposit_seq(p2a_metad* m, int64_t nhills, const double* centers, double* heights) {
  hipLaunchKernelGGL(k_deposit_seq<NCV>, dim3(1), dim3(kSeqThreads), 0, m->stream, m->G, m->val, m->der,
                     (long long)nhills, centers, heights, m->err);
}

// Tiles of the grid, and around a hill (M, per): a run of 2 nneigh + 1 nodes
// reaches (2 nneigh + T - 1) / T + 1 tiles of T nodes, and one more where it wraps
// over a last tile that is cut short.
struct TileCount {
  int64_t grid = 1, per = 1;
  TileMap M;
  // workgroups of an epoch of n hills; work-items have a 32-bit count (kMaxTiles)
  int64_t launch(int n) const { return by_hill(n) ? per * n : grid; }
  // a workgroup around a hill costs somewhat more than a tile that no hill
  // reaches (512 hills on 3,000 x 3,000 periodic nodes: 135,424 around the hills
  // 690-713 us, 140,625 tiles 607)
  bool by_hill(int n) const { return per * n * 5 < grid * 4; }
};
constexpr int64_t kMaxTiles = (1 << 24) - 1;
// Up to this many tiles (a few rounds of what the chip holds) the nodes are read
// early: a round's latency counts, not the bytes (4,000 hills on 513 x 513 nodes,
// 4,225 tiles: 1,688 us, read late 1,705).
constexpr int64_t kEarlyTiles = 16384;
template <int NCV>
static TileCount count_tiles(const GridArg& G) {
  TileCount C;
  std::memset(&C.M, 0, sizeof(C.M));
  for (int i = 0; i < NCV; i++) {
    const int64_t T = tile_dim<NCV>(i), nt = (G.nbin[i] + T - 1) / T;
    C.M.n[i] = (int)std::min(nt, (2 * (int64_t)G.nneigh[i] + T - 1) / T + 1 + (G.pbc[i] && G.nbin[i] % T ? 1 : 0));
    C.grid *= nt;
    C.per *= C.M.n[i];
  }
  return C;
}

template <int NCV, bool PER>
static void deposit_epochs(p2a_metad* m, const TileCount& tiles, int64_t nhills, const double* centers,
                           double* heights) {
  constexpr int EH = kChainThreads >> NCV;
  const GridArg& G = m->G;
  hipStream_t s = m->stream;
  const int64_t ne = (nhills + EH - 1) / EH;
  int64_t e0 = 0;  // the epoch whose cells come first in the workspace
  auto epoch = [&](int64_t e) {
    const bool has = e >= 0 && e < ne;
    return Epoch{has ? e * EH : 0, has ? (int)std::min<int64_t>(EH, nhills - e * EH) : 0,
                 has ? centers + e * EH * NCV : centers, has ? m->cells + (e - e0) * EH * NCV : m->cells};
  };
  // launch e finds the heights of epoch e and the shapes of epoch e + 1; e = -1: shapes only
  for (int64_t e = -1; e < ne; e++) {
    if (e < 0 || (e > 0 && e % kCellEpochs == 0)) {
      // the cells of this epoch, the kCellEpochs - 1 after it and the next one
      e0 = std::max<int64_t>(e, 0);
      const int64_t nc = std::min<int64_t>((kCellEpochs + 1) * EH, nhills - e0 * EH);
      hipLaunchKernelGGL(k_hill_cells<NCV>, dim3((unsigned)((nc + 255) / 256)), dim3(256), 0, s, G, (long long)nc,
                         centers + e0 * EH * NCV, m->cells);
    }
    const Epoch E = epoch(e), N = epoch(e + 1);
    const int rows = G.welltemp ? N.n : 0;
    if (E.n == 0 && rows == 0) continue;
    const size_t half = (size_t)EH * kChainThreads;
    hipLaunchKernelGGL((k_hill_chain<NCV, PER>), dim3(1 + rows), dim3(kChainThreads), 0, s, G, m->val, m->der, E,
                       m->shapes + (e & 1) * half, N, m->shapes + ((e + 1) & 1) * half, e == 0 ? 1 : 0, m->state,
                       m->hbuf, heights, m->err);
    if (E.n > 0) {
      TileMap M = tiles.M;
      M.per = tiles.by_hill(E.n) ? (int)tiles.per : 0;
      M.early = !M.per && tiles.grid <= kEarlyTiles;
      hipLaunchKernelGGL((k_hill_nodes<NCV, PER>), dim3((unsigned)tiles.launch(E.n)), dim3(256), 0, s, G, m->val,
                         m->der, E, M, m->state, m->hbuf);
    }
  }
}

static int metad_read_err(p2a_metad* m, const char* what) {
  int e = 0;
  P2A_HIPM(hipMemcpyAsync(&e, m->err, sizeof(int), hipMemcpyDeviceToHost, m->stream));
  P2A_HIPM(hipStreamSynchronize(m->stream));
  if (e) {
    P2A_HIPM(hipMemsetAsync(m->err, 0, sizeof(int), m->stream));
    P2A_HIPM(hipStreamSynchronize(m->stream));
    return fail(P2A_ERR_GRID, std::string(what) + ": Looking for a value outside the grid");
  }
  return P2A_OK;
}

}  // namespace p2a

using namespace p2a;

extern "C" {

int p2a_metad_create(p2a_metad** out, int device, const p2a_metad_spec* spec) {
  if (!out || !spec) return fail(P2A_ERR_ARG, "null argument");
  *out = nullptr;
  const int ncv = spec->ncv;
  if (ncv < 1 || ncv > kMaxCv) return fail(P2A_ERR_UNSUPPORTED, "METAD grid supports 1 to 4 CVs");
  if (spec->pace <= 0) return fail(P2A_ERR_ARG, "PACE should be positive");
  if (spec->biasf < 1.0 && spec->biasf != -1.0) return fail(P2A_ERR_ARG, "well tempered bias factor is nonsensical");
  if (spec->biasf >= 1.0 && spec->kbt <= 0.0)
    return fail(P2A_ERR_ARG,
                "Unless the MD engine passes the temperature to plumed, with well-tempered metad you must specify it using TEMP");
  GridArg G;
  std::memset(&G, 0, sizeof(G));
  G.ncv = ncv;
  size_t size = 1;
  int64_t support = 1;
  for (int i = 0; i < ncv; i++) {
    if (!(spec->gmax[i] > spec->gmin[i])) return fail(P2A_ERR_ARG, "maximum in grid must be larger than minimum");
    if (spec->nbin[i] == 0) return fail(P2A_ERR_ARG, "number of grid points must be greater than zero");
    if (!(spec->sigma[i] > 0.0)) return fail(P2A_ERR_ARG, "SIGMA should be positive");
    G.pbc[i] = spec->periodic[i] != 0;
    G.min[i] = spec->gmin[i];
    G.dx[i] = (spec->gmax[i] - spec->gmin[i]) / (double)spec->nbin[i];
    G.nbin[i] = spec->nbin[i] + (G.pbc[i] ? 0 : 1);
    G.period[i] = spec->gmax[i] - spec->gmin[i];
    G.inv_period[i] = 1.0 / G.period[i];
    G.invsigma[i] = 1.0 / spec->sigma[i];
    // MetaD::getGaussianSupport (MetaD.cpp:1939-1994)
    G.nneigh[i] = (int)std::ceil(std::sqrt(2.0 * 6.25) * spec->sigma[i] / G.dx[i]);
    if (G.pbc[i] && 2 * G.nneigh[i] + 1 > (int)G.nbin[i]) G.may_alias = 1;
    size *= G.nbin[i];
    support *= 2 * G.nneigh[i] + 1;
  }
  if (support > (1 << 30)) return fail(P2A_ERR_UNSUPPORTED, "Gaussian support too large for the grid spacing");
  G.support = (int)support;
  G.height0 = spec->height;
  G.biasf = spec->biasf;
  G.kbt = spec->kbt;
  G.welltemp = spec->biasf >= 1.0;
  G.inv_wt = spec->biasf > 1.0 ? 1.0 / (spec->kbt * (spec->biasf - 1.0)) : (spec->kbt != 0.0 ? 1.0 / spec->kbt : 0.0);
  // dp2cutoff stretch (Tools.h:71-79, MetaD.cpp:762-765)
  G.stretchA = spec->nostretch ? 1.0 : 1.00193418799744762399;
  G.stretchB = spec->nostretch ? 0.0 : -.00193418799744762399;
  for (int i = 0; i < ncv; i++) G.kd[i] = -(G.invsigma[i] * G.stretchA);
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) return fail(P2A_ERR_HIP, "no HIP device available");
  if (device < 0 || device >= ndev) return fail(P2A_ERR_ARG, "device index out of range");
  P2A_HIPM(hipSetDevice(device));
  auto* m = new p2a_metad();
  m->device = device;
  m->spec = *spec;
  m->G = G;
  m->size = size;
  bool ok = hipStreamCreateWithFlags(&m->own_stream, hipStreamNonBlocking) == hipSuccess &&
            hipMalloc(&m->val, size * sizeof(double)) == hipSuccess &&
            hipMalloc(&m->der, size * ncv * sizeof(double)) == hipSuccess &&
            hipMalloc(&m->err, sizeof(int)) == hipSuccess;
  if (!ok) {
    p2a_metad_destroy(m);
    return fail(P2A_ERR_NOMEM, "device allocation of the METAD grid failed");
  }
  m->stream = m->own_stream;
  if (hipMemsetAsync(m->val, 0, size * sizeof(double), m->stream) != hipSuccess ||
      hipMemsetAsync(m->der, 0, size * ncv * sizeof(double), m->stream) != hipSuccess ||
      hipMemsetAsync(m->err, 0, sizeof(int), m->stream) != hipSuccess ||
      hipStreamSynchronize(m->stream) != hipSuccess) {
    p2a_metad_destroy(m);
    return fail(P2A_ERR_HIP, "clearing the METAD grid failed");
  }
  *out = m;
  g_last_error.clear();
  return P2A_OK;
}

int p2a_metad_destroy(p2a_metad* m) {
  if (!m) return P2A_OK;
  (void)hipSetDevice(m->device);
  if (m->stream) (void)hipStreamSynchronize(m->stream);
  if (m->val) (void)hipFree(m->val);
  if (m->der) (void)hipFree(m->der);
  if (m->err) (void)hipFree(m->err);
  if (m->scratch) (void)hipFree(m->scratch);
  if (m->shapes) (void)hipFree(m->shapes);
  if (m->own_stream) (void)hipStreamDestroy(m->own_stream);
  delete m;
  return P2A_OK;
}

int p2a_metad_set_stream(p2a_metad* m, void* stream) {
  if (!m) return fail(P2A_ERR_ARG, "null context");
  // NULL selects the default (null) stream, which orders with every blocking stream
  m->stream = (hipStream_t)stream;
  return P2A_OK;
}

int64_t p2a_metad_grid_size(const p2a_metad* m) { return m ? (int64_t)m->size : 0; }

int p2a_metad_deposit_device(p2a_metad* m, int64_t nhills, const double* centers_dev, double* heights_dev) {
  if (!m || (nhills > 0 && !centers_dev)) return fail(P2A_ERR_ARG, "null argument");
  if (nhills <= 0) return P2A_OK;
  P2A_HIPM(hipSetDevice(m->device));
  const GridArg& G = m->G;
  // A few hills: one workgroup, one launch (a host call with 1 / 2 hills takes
  // 41 / 44 us, in epochs 51 us for 3 and 53 us for 8).  More: in epochs,
  // unless a periodic support is wider than the grid (a node would count
  // twice) or the tiles exceed a launch.
  const bool some = nhills > kSeqHills && !G.may_alias;
  bool per = false;
  for (int i = 0; i < G.ncv; i++) per = per || G.pbc[i];
#define P2A_DEP(N)                                                                         \
  do {                                                                                     \
    const TileCount tiles = count_tiles<N>(G);                                             \
    const int most = (int)std::min<int64_t>(nhills, kChainThreads >> N);                   \
    const bool epochs = some && tiles.launch(most) <= kMaxTiles && epoch_workspace(m);     \
    if (epochs && per) deposit_epochs<N, true>(m, tiles, nhills, centers_dev, heights_dev); \
    else if (epochs) deposit_epochs<N, false>(m, tiles, nhills, centers_dev, heights_dev); \
    else deposit_seq<N>(m, nhills, centers_dev, heights_dev);                              \
  } while (0)
  if (G.ncv == 1) P2A_DEP(1);
  else if (G.ncv == 2) P2A_DEP(2);
  else if (G.ncv == 3) P2A_DEP(3);
  else P2A_DEP(4);
#undef P2A_DEP
  P2A_HIPM(hipGetLastError());
  return P2A_OK;
}

int p2a_metad_deposit(p2a_metad* m, int64_t nhills, const double* centers, double* heights) {
  if (!m || (nhills > 0 && !centers)) return fail(P2A_ERR_ARG, "null argument");
  if (nhills <= 0) return P2A_OK;
  P2A_HIPM(hipSetDevice(m->device));
  const int ncv = m->G.ncv;
  int rc;
  if ((rc = metad_scratch(m, (size_t)nhills * (ncv + 1)))) return rc;
  double* c_dev = m->scratch;
  double* h_dev = m->scratch + (size_t)nhills * ncv;
  P2A_HIPM(hipMemcpyAsync(c_dev, centers, (size_t)nhills * ncv * sizeof(double), hipMemcpyHostToDevice, m->stream));
  if ((rc = p2a_metad_deposit_device(m, nhills, c_dev, h_dev))) return rc;
  if (heights)
    P2A_HIPM(hipMemcpyAsync(heights, h_dev, (size_t)nhills * sizeof(double), hipMemcpyDeviceToHost, m->stream));
  return metad_read_err(m, "METAD deposition");
}

int p2a_metad_add_hills(p2a_metad* m, int64_t nhills, const double* centers, const double* heights) {
  if (!m || (nhills > 0 && (!centers || !heights))) return fail(P2A_ERR_ARG, "null argument");
  if (nhills <= 0) return P2A_OK;
  P2A_HIPM(hipSetDevice(m->device));
  const int ncv = m->G.ncv;
  int rc;
  if ((rc = metad_scratch(m, (size_t)nhills * (ncv + 1)))) return rc;
  double* c_dev = m->scratch;
  double* h_dev = m->scratch + (size_t)nhills * ncv;
  P2A_HIPM(hipMemcpyAsync(c_dev, centers, (size_t)nhills * ncv * sizeof(double), hipMemcpyHostToDevice, m->stream));
  P2A_HIPM(hipMemcpyAsync(h_dev, heights, (size_t)nhills * sizeof(double), hipMemcpyHostToDevice, m->stream));
  hipLaunchKernelGGL(k_add_hills, dim3((unsigned)nhills), dim3(kDepositThreads), 0, m->stream, m->G, m->val, m->der,
                     (long long)nhills, c_dev, h_dev, m->err);
  P2A_HIPM(hipGetLastError());
  return metad_read_err(m, "METAD hills");
}

int p2a_metad_bias_device(p2a_metad* m, int64_t n, const double* cv_dev, double* bias_dev, double* der_dev) {
  if (!m || (n > 0 && (!cv_dev || !bias_dev))) return fail(P2A_ERR_ARG, "null argument");
  if (n <= 0) return P2A_OK;
  P2A_HIPM(hipSetDevice(m->device));
  hipLaunchKernelGGL(k_bias, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, m->stream, m->G, m->val, m->der,
                     (long long)n, cv_dev, bias_dev, der_dev, m->err);
  P2A_HIPM(hipGetLastError());
  return P2A_OK;
}

int p2a_metad_bias(p2a_metad* m, int64_t n, const double* cv, double* bias, double* der) {
  if (!m || (n > 0 && (!cv || !bias))) return fail(P2A_ERR_ARG, "null argument");
  if (n <= 0) return P2A_OK;
  P2A_HIPM(hipSetDevice(m->device));
  const int ncv = m->G.ncv;
  int rc;
  if ((rc = metad_scratch(m, (size_t)n * (2 * ncv + 1)))) return rc;
  double* c_dev = m->scratch;
  double* b_dev = c_dev + (size_t)n * ncv;
  double* d_dev = b_dev + n;
  P2A_HIPM(hipMemcpyAsync(c_dev, cv, (size_t)n * ncv * sizeof(double), hipMemcpyHostToDevice, m->stream));
  if ((rc = p2a_metad_bias_device(m, n, c_dev, b_dev, d_dev))) return rc;
  P2A_HIPM(hipMemcpyAsync(bias, b_dev, (size_t)n * sizeof(double), hipMemcpyDeviceToHost, m->stream));
  if (der) P2A_HIPM(hipMemcpyAsync(der, d_dev, (size_t)n * ncv * sizeof(double), hipMemcpyDeviceToHost, m->stream));
  return metad_read_err(m, "METAD bias");
}

int p2a_metad_step_device(p2a_metad* m, int64_t step, const double* cv_dev, double* bias_dev, double* force_dev,
                          double* height_dev) {
  if (!m || !cv_dev) return fail(P2A_ERR_ARG, "null argument");
  P2A_HIPM(hipSetDevice(m->device));
  // MetaD::update (MetaD.cpp:2379-2385): a hill every PACE steps, never on
  // the first step seen
  int deposit = 0;
  if (step % m->spec.pace == 0 && !m->first_step) deposit = 1;
  else m->first_step = false;
  hipLaunchKernelGGL(k_metad_step, dim3(1), dim3(kDepositThreads), 0, m->stream, m->G, m->val, m->der, cv_dev,
                     deposit, bias_dev, force_dev, height_dev, m->err);
  P2A_HIPM(hipGetLastError());
  return P2A_OK;
}

int p2a_metad_check(p2a_metad* m) {
  if (!m) return fail(P2A_ERR_ARG, "null context");
  P2A_HIPM(hipSetDevice(m->device));
  return metad_read_err(m, "METAD");
}

int p2a_metad_get_grid(p2a_metad* m, double* values, double* derivs) {
  if (!m) return fail(P2A_ERR_ARG, "null context");
  P2A_HIPM(hipSetDevice(m->device));
  if (values) P2A_HIPM(hipMemcpyAsync(values, m->val, m->size * sizeof(double), hipMemcpyDeviceToHost, m->stream));
  if (derivs)
    P2A_HIPM(hipMemcpyAsync(derivs, m->der, m->size * m->G.ncv * sizeof(double), hipMemcpyDeviceToHost, m->stream));
  P2A_HIPM(hipStreamSynchronize(m->stream));
  return P2A_OK;
}

int p2a_metad_set_grid(p2a_metad* m, const double* values, const double* derivs) {
  if (!m) return fail(P2A_ERR_ARG, "null context");
  P2A_HIPM(hipSetDevice(m->device));
  if (values) P2A_HIPM(hipMemcpyAsync(m->val, values, m->size * sizeof(double), hipMemcpyHostToDevice, m->stream));
  if (derivs)
    P2A_HIPM(hipMemcpyAsync(m->der, derivs, m->size * m->G.ncv * sizeof(double), hipMemcpyHostToDevice, m->stream));
  P2A_HIPM(hipStreamSynchronize(m->stream));
  return P2A_OK;
}

int p2a_apply_force_device(void* stream, int64_t natoms, const double* f_dev, const double* deriv_dev,
                           const double* virial_cv_dev, double* forces_dev, double* virial_dev) {
  if (!f_dev || !deriv_dev || !forces_dev) return fail(P2A_ERR_ARG, "null argument");
  long long n = 3 * (long long)natoms;
  long long nt = n > 9 ? n : 9;
  hipLaunchKernelGGL(k_apply_force, dim3((unsigned)((nt + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                     (long long)natoms, f_dev, deriv_dev, virial_cv_dev, forces_dev, virial_dev);
  P2A_HIPM(hipGetLastError());
  return P2A_OK;
}

}  // extern "C"
