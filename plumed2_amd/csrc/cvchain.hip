// DISTANCE between the centres of mass of two atom groups on gfx950, and the
// chain rule that puts a bias force on such a CV back onto the atoms.
//
// What it replaces in the reference (the second CV of a METAD on
// COORDINATION and a distance between two centres):
//   c1: COM ATOMS=...   Center::calculate (src/vatom/Center.cpp:319-445) on
//   c2: COM ATOMS=...   the group made whole by ActionAtomistic::makeWhole
//                       (src/core/ActionAtomistic.cpp:587-607, no MOLINFO)
//   d: DISTANCE ATOMS=c1,c2   Distance::calculate / calculateCV
//                       (src/colvar/Distance.h:141-250): the two centres made
//                       whole, |c2 - c1|, derivatives +-d/|d|, box derivative
//                       by Colvar::setBoxDerivativesNoPbc
//   apply               ActionWithVirtualAtom::apply (src/core/
//                       ActionWithVirtualAtom.cpp:68-124) + ActionWithValue::
//                       checkForForces: F_i += f * w_i * (+-d/|d|); the centres
//                       are linear in the atoms and add no box term
//                       (ActionWithVirtualAtom.h:54-63)
//
// makeWhole is a chain: atom j+1 is placed at x'_j + Pbc::distance(x'_j,
// x_j+1).  Its image differs from the raw position by a lattice vector, and
// Pbc::distance gives the same vector for inputs that differ by a lattice
// vector, so x'_j = x_j + sum_{k<j} t_k with t_k the lattice vector that
// Pbc::distance adds to x_k+1 - x_k.  Each t_k is computed independently (in
// integer lattice coordinates) and the chain becomes an integer prefix sum:
// one workgroup, half of it per group, no sequential walk.  The centre is then
// a fixed-order FP64 sum; it differs from the reference's running sum by
// rounding only.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <cstring>
#include <string>
#include <vector>

#include "coord_kernels.h"

namespace p2a {

constexpr int kCdThreads = 1024;

// integer lattice coordinates of the vector Pbc::distance adds to b - a
__device__ __forceinline__ int3 link_shift(const PbcArg& P, const double* a, const double* b) {
  double d[3];
  pbc_distance(P, a, b, d);
  const double t[3] = {d[0] - (b[0] - a[0]), d[1] - (b[1] - a[1]), d[2] - (b[2] - a[2])};
  // t = n . box (box rows = lattice vectors)  =>  n = t . inv(box)
  int3 n;
  n.x = (int)rint(t[0] * P.inv[0] + t[1] * P.inv[3] + t[2] * P.inv[6]);
  n.y = (int)rint(t[0] * P.inv[1] + t[1] * P.inv[4] + t[2] * P.inv[7]);
  n.z = (int)rint(t[0] * P.inv[2] + t[1] * P.inv[5] + t[2] * P.inv[8]);
  return n;
}

constexpr int kCdHalf = kCdThreads / 2;  // threads of one group
constexpr int kCdWaves = kCdHalf / WAVE;

// One workgroup: threads [0, 512) take group 1, the others group 2, 512 atoms
// of each a trip.  Bound by latency (atom index -> positions -> image -> scan ->
// sums); a trip's images are scanned by wave shuffles and the wave totals from
// LDS (one barrier a trip), the sums of m and m x stay in registers until the
// one reduction at the end.  2 x 500 atoms: 21.3 us with one group after the
// other and a reduction a trip, now 9.6 us.
__global__ __launch_bounds__(kCdThreads) void k_center_distance(PbcArg P, int pbc, const double* __restrict__ pos,
                                                                int n1, int n2, const long long* __restrict__ idx,
                                                                const double* __restrict__ masses,
                                                                double* __restrict__ value,
                                                                double* __restrict__ deriv,
                                                                double* __restrict__ virial) {
  __shared__ int tot[2][2][kCdWaves][3];  // trip parity, group, wave
  __shared__ double red[2][kCdWaves][4];
  __shared__ double g[6], minv[2];
  const int t = threadIdx.x, lane = t & 63;
  const int grp = t / kCdHalf, w = (t % kCdHalf) / WAVE;
  const int n = grp ? n2 : n1, first = grp ? n1 : 0;
  const long long* id = idx + first;
  const double* m = masses ? masses + first : nullptr;
  double acc[4] = {0.0, 0.0, 0.0, 0.0};
  int carry[3] = {0, 0, 0};
  const int trips = (max(n1, n2) + kCdHalf - 1) / kCdHalf;
  for (int trip = 0; trip < trips; trip++) {
    const int k = trip * kCdHalf + t % kCdHalf;
    double x[3] = {0.0, 0.0, 0.0}, mk = 0.0;
    // shift of the link (k-1, k); the first atom of the group has none
    int3 s = make_int3(0, 0, 0);
    if (k < n) {
      const double* xr = pos + 3 * id[k];
      for (int q = 0; q < 3; q++) x[q] = xr[q];
      mk = m ? m[k] : 1.0;
      if (pbc && k > 0) s = link_shift(P, pos + 3 * id[k - 1], xr);
    }
    int v[3] = {s.x, s.y, s.z};
    if (pbc) {
      for (int q = 0; q < 3; q++)
        for (int o = 1; o < 64; o <<= 1) {
          const int y = __shfl_up(v[q], o, 64);
          if (lane >= o) v[q] += y;
        }
      if (lane == 63)
        for (int q = 0; q < 3; q++) tot[trip & 1][grp][w][q] = v[q];
      __syncthreads();
      for (int u = 0; u < kCdWaves; u++)
        for (int q = 0; q < 3; q++) {
          const int y = tot[trip & 1][grp][u][q];
          if (u < w) v[q] += y;
        }
      for (int q = 0; q < 3; q++) v[q] += carry[q];
      for (int u = 0; u < kCdWaves; u++)
        for (int q = 0; q < 3; q++) carry[q] += tot[trip & 1][grp][u][q];
    }
    for (int q = 0; q < 3; q++) {
      if (pbc) x[q] += (double)v[0] * P.box[q] + (double)v[1] * P.box[3 + q] + (double)v[2] * P.box[6 + q];
      acc[q] += mk * x[q];
    }
    acc[3] += mk;
  }
  for (int q = 0; q < 4; q++) acc[q] = wave_sum_d(acc[q]);
  if (lane == 0)
    for (int q = 0; q < 4; q++) red[grp][w][q] = acc[q];
  __syncthreads();
  if (t == 0) {
    double c[2][3];
    for (int h = 0; h < 2; h++) {
      double sum[4] = {0.0, 0.0, 0.0, 0.0};
      for (int u = 0; u < kCdWaves; u++)
        for (int q = 0; q < 4; q++) sum[q] += red[h][u][q];
      minv[h] = 1.0 / sum[3];
      for (int q = 0; q < 3; q++) c[h][q] = sum[q] / sum[3];
    }
    double* c1 = c[0];
    double* c2 = c[1];
    // DISTANCE makes its two atoms whole, then d = c2' - c1 (Distance.h:150-152, 205)
    if (pbc) {
      double d[3];
      pbc_distance(P, c1, c2, d);
      for (int q = 0; q < 3; q++) c2[q] = c1[q] + d[q];
    }
    const double d[3] = {c2[0] - c1[0], c2[1] - c1[1], c2[2] - c1[2]};
    const double v = sqrt(d[0] * d[0] + d[1] * d[1] + d[2] * d[2]);
    const double inv = 1.0 / v;
    for (int q = 0; q < 3; q++) {
      g[q] = -inv * d[q];
      g[3 + q] = inv * d[q];
    }
    *value = v;
    for (int a = 0; a < 3; a++)
      for (int b = 0; b < 3; b++) virial[3 * a + b] = -(c1[a] * g[b]) - c2[a] * g[3 + b];
  }
  __syncthreads();
  for (int k = t; k < n1 + n2; k += blockDim.x) {
    const int h = k < n1 ? 0 : 1;
    const double wk = (masses ? masses[k] : 1.0) * minv[h];
    for (int q = 0; q < 3; q++) deriv[3 * (size_t)k + q] = wk * g[3 * h + q];
  }
}

// Forces of a METAD step on every atom and the cell, written in one pass:
// forces = f[0] * (dCV/dx of the coordination), plus f[1] * (derivative of the
// distance) for the atoms of its groups; virial likewise.  The listed atoms
// (a bitmap tells them) belong to the workgroups after the first nplain.
// Replaces two fills and two additive passes (24 B an atom read and written
// twice more).
struct ListedAtom {
  int atom, k1, k2;  // entry in group 1 / group 2 (-1: not in it)
};
__global__ __launch_bounds__(256) void k_metad_forces(long long natoms, int nplain, const double* __restrict__ f,
                                                      const double* __restrict__ deriv,
                                                      const double* __restrict__ wcv,
                                                      const unsigned* __restrict__ bits, long long nbits, int nlisted,
                                                      const ListedAtom* __restrict__ listed,
                                                      const double* __restrict__ ddist,
                                                      const double* __restrict__ wdist, double* __restrict__ forces,
                                                      double* __restrict__ virial) {
  const double f0 = f[0];
  if ((int)blockIdx.x < nplain) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (blockIdx.x == 0 && threadIdx.x < 9) {
      double v = 0.0 + f0 * wcv[threadIdx.x];
      if (nlisted) v += f[1] * wdist[threadIdx.x];
      virial[threadIdx.x] = v;
    }
    if (i >= 3 * natoms) return;
    const long long a = i / 3;
    if (a < nbits && ((bits[a >> 5] >> (a & 31)) & 1u)) return;
    forces[i] = 0.0 + f0 * deriv[i];
    return;
  }
  const int e = ((int)blockIdx.x - nplain) * 256 + (int)threadIdx.x;
  if (e >= nlisted) return;
  const double f1 = f[1];
  const ListedAtom L = listed[e];
  for (int q = 0; q < 3; q++) {
    double v = 0.0 + f0 * deriv[3 * (size_t)L.atom + q];
    if (L.k1 >= 0) v += f1 * ddist[3 * (size_t)L.k1 + q];
    if (L.k2 >= 0) v += f1 * ddist[3 * (size_t)L.k2 + q];
    forces[3 * (size_t)L.atom + q] = v;
  }
}

// forces[3*idx[k] + q] += f * deriv[3k + q] for the listed atoms, group 1 then
// group 2 (each group's atoms are distinct, so each phase writes distinct
// entries); virial += f * virial_cv
__global__ __launch_bounds__(kCdThreads) void k_apply_force_listed(int n1, const long long* __restrict__ idx1, int n2,
                                                                   const long long* __restrict__ idx2,
                                                                   const double* __restrict__ f,
                                                                   const double* __restrict__ deriv,
                                                                   const double* __restrict__ vcv,
                                                                   double* __restrict__ forces,
                                                                   double* __restrict__ virial) {
  const double fv = *f;
  for (int k = threadIdx.x; k < n1; k += blockDim.x)
    for (int q = 0; q < 3; q++) forces[3 * idx1[k] + q] += fv * deriv[3 * (size_t)k + q];
  __syncthreads();
  for (int k = threadIdx.x; k < n2; k += blockDim.x)
    for (int q = 0; q < 3; q++) forces[3 * idx2[k] + q] += fv * deriv[3 * (size_t)(n1 + k) + q];
  if (virial && vcv && threadIdx.x < 9) virial[threadIdx.x] += fv * vcv[threadIdx.x];
}

}  // namespace p2a

struct p2a_cdist {
  int device = 0;
  int64_t natoms = 0;
  int n1 = 0, n2 = 0;
  int pbc = 1;
  p2a::DBuf<long long> idx;  // group 1 then group 2
  p2a::DBuf<double> masses;
  bool has_masses = false;
  // every atom of the groups once, in index order, and as bits
  p2a::DBuf<p2a::ListedAtom> listed;
  p2a::DBuf<unsigned> bits;
  int nlisted = 0;
  int64_t nbits = 0;
};

using namespace p2a;

extern "C" {

int p2a_cdist_create(p2a_cdist** out, int device, int64_t natoms, int64_t n1, const int64_t* group1, int64_t n2,
                     const int64_t* group2, const double* masses, int use_pbc) {
  if (!out || (n1 > 0 && !group1) || (n2 > 0 && !group2)) return fail(P2A_ERR_ARG, "null argument");
  *out = nullptr;
  if (n1 <= 0 || n2 <= 0) return fail(P2A_ERR_ARG, "at least one atom should be specified");
  if (n1 + n2 > (1 << 26) || natoms > ((int64_t)1 << 40)) return fail(P2A_ERR_UNSUPPORTED, "groups too large");
  for (int g = 0; g < 2; g++) {
    const int64_t* a = g ? group2 : group1;
    const int64_t n = g ? n2 : n1;
    std::vector<int64_t> v(a, a + n);
    for (int64_t x : v)
      if (x < 0 || x >= natoms) return fail(P2A_ERR_ARG, "atom index outside the positions array");
    std::sort(v.begin(), v.end());
    if (std::adjacent_find(v.begin(), v.end()) != v.end())
      return fail(P2A_ERR_ARG, "an atom is listed twice in one group");
  }
  if (masses)
    for (int64_t k = 0; k < n1 + n2; k++)
      if (!(masses[k] > 0.0)) return fail(P2A_ERR_ARG, "masses must be positive");
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) return fail(P2A_ERR_HIP, "no HIP device available");
  if (device < 0 || device >= ndev) return fail(P2A_ERR_ARG, "device index out of range");
  P2A_HIP(hipSetDevice(device));
  auto* c = new p2a_cdist();
  c->device = device;
  c->natoms = natoms;
  c->n1 = (int)n1;
  c->n2 = (int)n2;
  c->pbc = use_pbc ? 1 : 0;
  std::vector<long long> all(group1, group1 + n1);
  all.insert(all.end(), group2, group2 + n2);
  // the listed atoms: (atom, position in the lists), merged per atom
  std::vector<std::pair<long long, int>> by(all.size());
  for (size_t k = 0; k < all.size(); k++) by[k] = {all[k], (int)k};
  std::sort(by.begin(), by.end());
  std::vector<ListedAtom> listed;
  // (indices beyond 32 bits: the additive entry points only)
  if (by.back().first <= INT32_MAX) {
    for (auto& e : by) {
      if (listed.empty() || listed.back().atom != e.first) listed.push_back({(int)e.first, -1, -1});
      if (e.second < (int)n1) listed.back().k1 = e.second;
      else listed.back().k2 = e.second;
    }
    c->nbits = by.back().first + 1;
  }
  std::vector<unsigned> bits((size_t)((c->nbits + 31) / 32), 0u);
  for (auto& e : listed) bits[e.atom >> 5] |= 1u << (e.atom & 31);
  c->nlisted = (int)listed.size();
  int rc;
  if ((rc = c->idx.reserve(all.size())) || (masses && (rc = c->masses.reserve(all.size()))) ||
      (rc = c->listed.reserve(std::max<size_t>(listed.size(), 1))) ||
      (rc = c->bits.reserve(std::max<size_t>(bits.size(), 1)))) {
    delete c;
    return rc;
  }
  if (!listed.empty() &&
      (hipMemcpy(c->listed.p, listed.data(), listed.size() * sizeof(ListedAtom), hipMemcpyHostToDevice) != hipSuccess ||
       hipMemcpy(c->bits.p, bits.data(), bits.size() * sizeof(unsigned), hipMemcpyHostToDevice) != hipSuccess)) {
    delete c;
    return fail(P2A_ERR_HIP, "hipMemcpy of the listed atoms failed");
  }
  if (hipMemcpy(c->idx.p, all.data(), all.size() * sizeof(long long), hipMemcpyHostToDevice) != hipSuccess ||
      (masses && hipMemcpy(c->masses.p, masses, all.size() * sizeof(double), hipMemcpyHostToDevice) != hipSuccess)) {
    delete c;
    return fail(P2A_ERR_HIP, "hipMemcpy of the groups failed");
  }
  c->has_masses = masses != nullptr;
  *out = c;
  g_last_error.clear();
  return P2A_OK;
}

int p2a_cdist_destroy(p2a_cdist* c) {
  if (!c) return P2A_OK;
  (void)hipSetDevice(c->device);
  (void)hipDeviceSynchronize();
  delete c;
  return P2A_OK;
}

int p2a_cdist_calculate_device(p2a_cdist* c, void* stream, const double* box9, const double* pos_dev,
                               double* value_dev, double* deriv_dev, double* virial_dev) {
  if (!c || !pos_dev || !value_dev || !deriv_dev || !virial_dev) return fail(P2A_ERR_ARG, "null argument");
  if (c->pbc && !box9) return fail(P2A_ERR_ARG, "box is required with periodic boundaries");
  P2A_HIP(hipSetDevice(c->device));
  PbcArg P;
  std::memset(&P, 0, sizeof(P));
  if (c->pbc) {
    PbcHost h;
    pbc_setup(box9, h);
    if (h.type == 0) return fail(P2A_ERR_ARG, "the box is singular");
    fill_pbc_arg(h, P);
  }
  hipLaunchKernelGGL(k_center_distance, dim3(1), dim3(kCdThreads), 0, (hipStream_t)stream, P, c->pbc, pos_dev,
                     c->n1, c->n2, (const long long*)c->idx.p,
                     (const double*)(c->has_masses ? c->masses.p : nullptr), value_dev, deriv_dev, virial_dev);
  return launch_check("centre distance");
}

int p2a_cdist_apply_force_device(p2a_cdist* c, void* stream, const double* f_dev, const double* deriv_dev,
                                 const double* virial_cv_dev, double* forces_dev, double* virial_dev) {
  if (!c || !f_dev || !deriv_dev || !forces_dev) return fail(P2A_ERR_ARG, "null argument");
  P2A_HIP(hipSetDevice(c->device));
  hipLaunchKernelGGL(k_apply_force_listed, dim3(1), dim3(kCdThreads), 0, (hipStream_t)stream, c->n1,
                     (const long long*)c->idx.p, c->n2, (const long long*)c->idx.p + c->n1, f_dev, deriv_dev,
                     virial_cv_dev, forces_dev, virial_dev);
  return launch_check("centre distance forces");
}

int p2a_metad_forces_device(void* stream, int64_t natoms, const double* cv_force_dev, const double* deriv_dev,
                            const double* virial_cv_dev, p2a_cdist* c, const double* dist_deriv_dev,
                            const double* dist_virial_dev, double* forces_dev, double* virial_dev) {
  if (!cv_force_dev || !deriv_dev || !virial_cv_dev || !forces_dev || !virial_dev)
    return fail(P2A_ERR_ARG, "null argument");
  if (natoms < 0 || natoms > INT32_MAX) return fail(P2A_ERR_ARG, "the number of atoms must lie in [0, 2^31)");
  if (c) {
    if (!dist_deriv_dev || !dist_virial_dev) return fail(P2A_ERR_ARG, "null argument");
    if (c->nbits == 0 || c->nbits > natoms) return fail(P2A_ERR_ARG, "atom index outside the forces array");
    P2A_HIP(hipSetDevice(c->device));
  }
  const int nplain = std::max(1, grid1(3 * (size_t)natoms, 256));
  const int nlisted = c ? c->nlisted : 0;
  hipLaunchKernelGGL(k_metad_forces, dim3(nplain + grid1((size_t)nlisted, 256)), dim3(256), 0, (hipStream_t)stream,
                     (long long)natoms, nplain, cv_force_dev, deriv_dev, virial_cv_dev,
                     (const unsigned*)(c ? c->bits.p : nullptr), (long long)(c ? c->nbits : 0), nlisted,
                     (const ListedAtom*)(c ? c->listed.p : nullptr), dist_deriv_dev, dist_virial_dev, forces_dev,
                     virial_dev);
  return launch_check("METAD forces");
}

}  // extern "C"
