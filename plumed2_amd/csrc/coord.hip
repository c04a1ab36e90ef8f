// COORDINATION on gfx950: the single-system context and its C ABI.
//
// One context = one COORDINATION action (CoordinationBase.cpp:42-131): its
// groups, switch and neighbour-list settings, the device arrays of the
// cluster-pair structure, and a HIP stream.  The kernels are in
// coord_kernels.h; this file sizes the arrays, decides the rebuild steps
// (NeighborList::prepare, NeighborList.cpp:433-456) and launches.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "coord_kernels.h"

namespace p2a {

struct Dir {  // one cluster-pair list: i clusters of group I against group J
  int I = 0, J = 0;
  DBuf<int> ecount, estart, istart;
  DBuf<Entry> ents;
  DBuf<int4> items;
  DBuf<double> fpart;  // per item: derivative partials of the 8 i atoms
  DBuf<double> rpart;  // per item: per-atom coordination-number rows of the 8 i atoms
  DBuf<int> wave_start;  // the pair kernel's balanced schedule (k_wave_sched)
  int sched_waves = -1;  // the grid it was made for
  int64_t sched_gen = -1;  // and the list build
  DBuf<unsigned> ell;  // candidates the list count pass keeps for the fill pass
  int nitems = 0, item_offset = 0;
  int64_t nentries = 0;
};

struct Group {
  int off = 0, n = 0;
  SysArg S{};   // cell and column grid of this group
  SysArg S_dev{};  // the copy the device holds
  bool S_valid = false;
  int maxcl = 0;   // cluster capacity: n/8 + one partial cluster per column
  int ncol = 1;
  int ncl = 0;  // clusters (device total copied at rebuild)
  // slot_loc of the last build (order_nslot slots, `order`) orders the
  // atoms of the next one; 0 = no such order
  int order_nslot = 0;
  Held order;
  // col_count and fill hold zeros over their whole capacity (k_rank leaves them so)
  Held zero_count, zero_fill;
  DBuf<SysArg> sys;
  DBuf<int4> info, slot_img;
  DBuf<double> key;
  DBuf<int> col_count, col_start, col_cl, fill, tmp, slot_loc, cl_col, twin_slot;
  DBuf<double4> origin;
  DBuf<float4> bb0, bb, p;
  DBuf<float4> pw;  // p with the row weights (k_row_weights)
  DBuf<float2> kr;
};

}  // namespace p2a

struct p2a_coord {
  int device = 0;
  hipStream_t own_stream = nullptr;
  hipStream_t stream = nullptr;
  p2a_coord_spec spec{};
  std::vector<int64_t> abs;  // absolute index of each requested atom
  int natoms = 0;
  bool firsttime = true;
  int path = 0;
  double rlist = 0.0;
  double box_at_build[9] = {0};    // cell the list entries are imaged for
  double box_at_rebuild[9] = {0};  // cell of the last rebuild (wrapping integers, images)
  int max_wrap = 0;                // largest |lattice translation| of a wrapped atom at that rebuild
  bool totals_clear = false;
  bool built = false;
  p2a::Group g[2];
  p2a::DBuf<int> totals;       // [4..7] atoms/clusters per group, [8..11] entries/items per direction
  p2a::Dir dir[2];
  int ndir = 0;
  int nitems = 0;
  int64_t nentries = 0;
  p2a::PairTuning tune;
  int cu_count = 256;
  p2a::DBuf<double> partial, red, stats, pos_buf, deriv_buf, out_buf;
  p2a::DBuf<int> scan_bsum;   // block sums of the list scans
  p2a::DBuf<long long> abs_dev;
  p2a::DBuf<int> twin_dev;  // groups that share atoms: requested index of the atom in the other group, or -2
  int64_t rebuilds = 0;
  bool profiling = false;
  int prof_every = 1;       // events around every prof_every-th pair pass
  int64_t prof_calls = 0;
  double prof_ms = 0.0;
  int64_t prof_launches = 0;
  std::vector<hipEvent_t> ev_pool;
  std::vector<std::pair<hipEvent_t, hipEvent_t>> pending;
  bool has_duplicates = false;  // an absolute index listed twice in one group
  bool distinct = true;         // no absolute index listed twice in the two groups together
  p2a::PbcHost pbc;
  p2a::PbcArg pbc_stage;
  p2a::DBuf<p2a::PbcArg> pbc_dev;
  double pbc_box[9] = {0};
  bool pbc_valid = false;
  double path_box[9] = {0};  // box of the last path decision
  int path_cached = -1;
  // without a neighbour list: list built at D_MAX + skin and kept while no
  // atom has moved more than skin/2 (skin_active: 0 when the cell is too
  // narrow for the larger radius)
  double skin = 0.0, skin_active = 0.0;
  // positions packed ahead by the skin test, for the list of build packed_gen
  const double* packed_pos = nullptr;
  int64_t packed_gen = -1;
  p2a::DBuf<double> pos_ref;  // positions at the last build
  p2a::DBuf<int> moved;
  hipEvent_t moved_ev = nullptr;  // the moved flag has reached host_ro[32]
  int* host_ro = nullptr;  // pinned host words for the few device-to-host reads
  // neighbour list of the FP64 path: partners of every atom (symmetric CSR),
  // or one flag per pair with PAIR; cell of every atom for NLISTCELLS
  p2a::DBuf<int> nl_count, nl_start, nl_nbr, nl_cell;
  p2a::DBuf<long long> nl_total;
  bool nl_valid = false;
  int64_t nl_entries = 0;  // partners listed in nl_nbr
  // per-atom coordination numbers: row and environment indices for the FP64 path
  p2a::DBuf<int> cn_rows, cn_env;
};

namespace p2a {

static int choose_path_uncached(p2a_coord* c, const double* box9);

// decides the evaluation path for this box; 0 = cluster kernel
static int choose_path(p2a_coord* c, const double* box9) {
  if (c->path_cached >= 0 && std::memcmp(c->path_box, box9, sizeof(c->path_box)) == 0) return c->path_cached;
  c->path_cached = choose_path_uncached(c, box9);
  std::memcpy(c->path_box, box9, sizeof(c->path_box));
  return c->path_cached;
}

static int choose_path_uncached(p2a_coord* c, const double* box9) {
  const p2a_switch& sw = c->spec.sw;
  if (c->spec.pair && c->spec.nb > 0) return 2;
  if (!c->spec.pbc || c->has_duplicates) return 1;
  PbcHost p;
  pbc_setup(box9, p);
  if (p.type == 0) return 1;
  if (!(sw.dmax < 1e30)) return 1;
  double rl = c->spec.nl_mode != P2A_NL_NONE ? std::max(c->spec.nl_cutoff, sw.dmax) : sw.dmax;
  double w[3];
  pbc_widths(box9, w);
  double wmin = std::min(w[0], std::min(w[1], w[2]));
  if (wmin <= 2.0 * rl * 1.0001 + 1e-6) return 1;
  c->skin_active = 0.0;
  if (c->spec.nl_mode == P2A_NL_NONE && c->skin > 0.0 && wmin > 2.0 * (sw.dmax + c->skin) * 1.0001 + 1e-6)
    c->skin_active = c->skin;
  return 0;
}

// workgroups of the pair kernel over nitems items
static int pair_grid(const p2a_coord* c, int nitems) {
  const int grid = grid1(nitems, PAIR_BLOCK / WAVE);
  return c->tune.blocks_per_cu > 0 ? std::min(grid, c->tune.blocks_per_cu * c->cu_count) : grid;
}

static int rebuild(p2a_coord* c, const double* box9, const double* pos_dev) {
  const p2a_switch& sw = c->spec.sw;
  // list radius: NL_CUTOFF when a neighbour list is requested (its candidates
  // must cover every pair that can come within D_MAX before the next rebuild),
  // D_MAX + skin otherwise (skin 0: the list is rebuilt every step)
  c->rlist = (c->spec.nl_mode != P2A_NL_NONE ? std::max(c->spec.nl_cutoff, sw.dmax) : sw.dmax + c->skin_active) + 1e-4;
  const int ngroups = c->spec.nb > 0 ? 2 : 1;
  const bool share = ngroups == 2 && !c->distinct;
  hipStream_t s = c->stream;
  int rc;
  for (int gi = 0; gi < ngroups; gi++) {
    Group& G = c->g[gi];
    G.off = gi == 0 ? 0 : (int)c->spec.na;
    G.n = gi == 0 ? (int)c->spec.na : (int)c->spec.nb;
    sys_cell(box9, c->rlist, G.S);
    sys_columns(box9, G.n, G.S);
    G.S.colbase = 0;
    G.ncol = G.S.ncx * G.S.ncy;
    int64_t maxcl64 = (int64_t)G.n / CL + G.ncol + 1;
    if (maxcl64 > kMaxClusters) return fail(P2A_ERR_UNSUPPORTED, "too many atom clusters for the list encoding");
    const int maxcl = (int)maxcl64;
    G.maxcl = maxcl;
    if ((rc = G.sys.reserve(1)) || (rc = G.info.reserve(G.n)) || (rc = G.key.reserve(G.n)) ||
        (rc = G.col_count.reserve(G.ncol + 1)) || (rc = G.col_start.reserve(G.ncol + 1)) ||
        (rc = G.col_cl.reserve(G.ncol + 1)) || (rc = G.fill.reserve(G.ncol + 1)) || (rc = G.tmp.reserve(G.n)) ||
        (rc = G.slot_loc.reserve((size_t)maxcl * CL)) || (rc = G.cl_col.reserve(maxcl)) ||
        (rc = G.origin.reserve(maxcl)) || (rc = G.bb0.reserve(2 * (size_t)maxcl)) ||
        (rc = G.bb.reserve(2 * (size_t)maxcl)) || (rc = G.p.reserve((size_t)maxcl * CL)) ||
        (rc = G.kr.reserve(maxcl)) || (rc = G.slot_img.reserve((size_t)maxcl * CL)) || (share && (rc = G.twin_slot.reserve((size_t)maxcl * CL))))
      return rc;
    // the descriptor goes to the device in stream order when it changed
    if (!G.S_valid || std::memcmp(&G.S, &G.S_dev, sizeof(SysArg)) != 0) {
      hipLaunchKernelGGL(k_store<SysArg>, dim3(1), dim3(64), 0, s, G.S, G.sys.p);
      G.S_dev = G.S;
      G.S_valid = true;
    }
  }
  if ((rc = c->totals.reserve(16))) return rc;
  if (!c->totals_clear) {
    hipLaunchKernelGGL(k_fill_int, dim3(1), dim3(64), 0, s, c->totals.p, 16, 0);
    c->totals_clear = true;
  }
  // two alternating slots for the largest wrap of this rebuild
  const int wslot = 12 + (int)(c->rebuilds & 1);
  Two<BinSide> B;
  Two<RankSide> R;
  ScanSide cols[2];
  std::memset(&B, 0, sizeof(B));
  std::memset(&R, 0, sizeof(R));
  int nbin[2] = {0, 0}, nrank[2] = {0, 0};
  size_t nbsum = 0;  // block sums of the scans: columns first, then the lists
  for (int gi = 0; gi < ngroups; gi++)
    nbsum += 2 * (size_t)grid1(std::max(c->g[gi].ncol, c->g[gi].maxcl), kScanBlock) + 2;
  if ((rc = c->scan_bsum.reserve(nbsum))) return rc;
  int* bsum[2] = {c->scan_bsum.p,
                  c->scan_bsum.p + 2 * (size_t)grid1(std::max(c->g[0].ncol, c->g[0].maxcl), kScanBlock) + 2};
  for (int gi = 0; gi < ngroups; gi++) {
    Group& G = c->g[gi];
    // the atoms are binned in the slot order of the last build when it is
    // still in slot_loc (atoms move little between builds, so a workgroup's
    // column counts stay in LDS); k_rank then writes every slot of the new
    // clusters, padding included
    const bool use_order = G.order_nslot > 0 && G.order.of(G.slot_loc);
    const int norder = use_order ? G.order_nslot : 0;
    G.order_nslot = 0;
    if (!G.zero_count.of(G.col_count) || !G.zero_fill.of(G.fill)) {
      const int nc = (int)G.col_count.n, nf = (int)G.fill.n;
      hipLaunchKernelGGL(k_fill_int3, dim3(std::max(1, std::min(grid1(std::max(nc, nf), 256), 1024))), dim3(256), 0, s,
                         G.col_count.p, nc, 0, G.fill.p, nf, 0, (int*)nullptr, 0, 0);
    }
    G.zero_count.drop();
    G.zero_fill.drop();
    B.s[gi] = BinSide{G.n,     G.off,         norder,          use_order ? G.slot_loc.p : nullptr,
                      G.sys.p, G.info.p,      G.key.p,         G.col_count.p,
                      G.col_start.p, G.fill.p, G.tmp.p};
    nbin[gi] = G.n > 0 ? grid1(use_order ? norder : G.n, 256) : 0;
    // atom and cluster starts of the columns; totals[4 + 2 gi], [5 + 2 gi]
    cols[gi] = ScanSide{G.ncol, nullptr, G.col_count.p, G.col_start.p, G.col_cl.p, 4 + 2 * gi, 5 + 2 * gi, bsum[gi]};
    R.s[gi] = RankSide{G.ncol,   G.off,   G.key.p, G.col_start.p, G.col_cl.p,       G.tmp.p,    G.slot_loc.p,
                       G.info.p, G.sys.p, G.origin.p, G.bb0.p,    G.kr.p,           nullptr,    G.cl_col.p,
                       G.p.p,    G.bb.p,  G.col_count.p, G.fill.p, G.slot_img.p};
    nrank[gi] = G.n > 0 ? G.ncol : 0;
  }
  B.n0 = nbin[0];
  R.n0 = nrank[0];
  if (nbin[0] + nbin[1] > 0)
    hipLaunchKernelGGL(k_bin, dim3(nbin[0] + nbin[1]), dim3(256), 0, s, B, pos_dev, (const int*)nullptr,
                       c->totals.p + wslot, c->totals.p + (25 - wslot));
  launch_list_scans(s, cols, ngroups, CL, c->totals.p);
  if (nbin[0] + nbin[1] > 0) {
    hipLaunchKernelGGL(k_scatter, dim3(nbin[0] + nbin[1]), dim3(256), 0, s, B);
    hipLaunchKernelGGL(k_rank, dim3(nrank[0] + nrank[1]), dim3(256), 0, s, R, pos_dev, (const int*)nullptr,
                       pack_scale(c->spec.sw));
  }
  if ((rc = launch_check("rebuild: binning"))) return rc;
  for (int gi = 0; gi < ngroups; gi++) {
    c->g[gi].zero_count.note(c->g[gi].col_count);
    c->g[gi].zero_fill.note(c->g[gi].fill);
  }
  // cluster counts stay on the device (totals[5 + 2 g]) until the one host
  // read below; the kernels in between are sized by the cluster capacity
  // full cluster-pair lists: one direction for a single group, A->B (the
  // counting side) and B->A for two groups
  c->ndir = ngroups;
  int64_t tot_entries = 0;
  const int wpb = 256 / WAVE;
  const int chunk = c->tune.chunk;
  Two<ListSide> T;
  ScanSide lists[2];
  std::memset(&T, 0, sizeof(T));
  int nlist[2] = {0, 0};
  for (int d = 0; d < c->ndir; d++) {
    Dir& D = c->dir[d];
    D.I = (ngroups == 2) ? d : 0;
    D.J = (ngroups == 2) ? 1 - d : 0;
    Group& GI = c->g[D.I];
    Group& GJ = c->g[D.J];
    ListSide& S = T.s[d];
    const int* ncl_dev = c->totals.p + 5 + 2 * D.I;
    if ((rc = D.ecount.reserve(GI.maxcl + 1)) || (rc = D.estart.reserve(GI.maxcl + 1)) ||
        (rc = D.istart.reserve(GI.maxcl + 1)) || (rc = D.ell.reserve((size_t)GI.maxcl * kEll)))
      return rc;
    S.L.nclI = GI.maxcl;
    S.L.nclI_dev = ncl_dev;
    S.L.mode = (ngroups == 1) ? 0 : (d == 0 ? 1 : 2);
    S.L.ent_cap = 0;
    S.L.rlist2 = (float)(c->rlist * c->rlist);
    S.L.pscale = pack_scale(c->spec.sw);
    S.cl_colI = GI.cl_col.p;
    S.sysI = GI.sys.p;
    S.sysJ = GJ.sys.p;
    S.bbI = GI.bb0.p;
    S.bbJ = GJ.bb0.p;
    S.krI = GI.kr.p;
    S.krJ = GJ.kr.p;
    S.col_clJ = GJ.col_cl.p;
    S.orgI = GI.origin.p;
    S.orgJ = GJ.origin.p;
    S.count = D.ecount.p;
    S.start = D.estart.p;
    S.ell = D.ell.p;
    nlist[d] = grid1(GI.maxcl, wpb);
    lists[d] = ScanSide{GI.maxcl, ncl_dev, D.ecount.p, D.estart.p, D.istart.p, 8 + 2 * d, 9 + 2 * d, bsum[D.I]};
  }
  T.n0 = nlist[0];
  hipLaunchKernelGGL(k_list<0>, dim3(nlist[0] + nlist[1]), dim3(256), 0, s, T);
  launch_list_scans(s, lists, c->ndir, chunk, c->totals.p);
  if ((rc = launch_check("rebuild: list count"))) return rc;
  int* hostT = c->host_ro;
  P2A_HIP(hipMemcpyAsync(hostT, c->totals.p, 16 * sizeof(int), hipMemcpyDeviceToHost, s));
  P2A_HIP(hipStreamSynchronize(s));
  for (int gi = 0; gi < ngroups; gi++) {
    Group& G = c->g[gi];
    G.ncl = hostT[5 + 2 * gi];
    G.order_nslot = G.ncl * CL;
    G.order.note(G.slot_loc);
  }
  c->max_wrap = hostT[wslot];
  c->nitems = 0;
  for (int d = 0; d < c->ndir; d++) {
    Dir& D = c->dir[d];
    Group& GI = c->g[D.I];
    D.nentries = hostT[8 + 2 * d];
    D.nitems = hostT[9 + 2 * d];
    D.item_offset = c->nitems;
    c->nitems += D.nitems;
    tot_entries += D.nentries;
    // the schedule of a persistent grid comes with the items
    const int nw = c->tune.blocks_per_cu > 0 ? pair_grid(c, D.nitems) * (PAIR_BLOCK / WAVE) : 0;
    if ((rc = D.ents.reserve(std::max<int64_t>(D.nentries, 1))) || (rc = D.items.reserve(std::max(D.nitems, 1))) ||
        (rc = D.fpart.reserve((size_t)CL * 3 * std::max(D.nitems, 1))) || (rc = D.wave_start.reserve((size_t)nw + 1)))
      return rc;
    ListSide& S = T.s[d];
    S.L.ent_cap = (int)D.ents.n;
    S.L.nclI = GI.ncl;
    S.L.nclI_dev = nullptr;
    S.out = D.ents.p;
    S.M = ItemArgs{D.items.p, D.istart.p, chunk, (int)D.items.n, nw, D.nitems,
                   (long long)D.nentries + (long long)kItemCost * D.nitems, D.wave_start.p};
    nlist[d] = D.nitems > 0 ? grid1(GI.ncl, wpb) : 0;
    if (nw && D.nitems > 0) {
      D.sched_waves = nw;
      D.sched_gen = c->rebuilds + 1;
    }
  }
  T.n0 = nlist[0];
  if (nlist[0] + nlist[1] > 0) hipLaunchKernelGGL(k_list<1>, dim3(nlist[0] + nlist[1]), dim3(256), 0, s, T);
  c->nentries = tot_entries;
  if (share) {
    for (int gi = 0; gi < 2; gi++) {
      Group& G = c->g[gi];
      if (G.ncl > 0)
        hipLaunchKernelGGL(k_twin_slot, dim3(grid1((size_t)G.ncl * CL, 256)), dim3(256), 0, s, G.ncl * CL,
                           (const int*)G.slot_loc.p, G.off, (const int*)c->twin_dev.p, G.twin_slot.p);
    }
  }
  if ((rc = launch_check("rebuild: list fill"))) return rc;
  if (c->skin_active > 0.0) {
    const size_t n3 = 3 * (size_t)c->natoms;
    if ((rc = c->pos_ref.reserve(n3))) return rc;
    P2A_HIP(hipMemcpyAsync(c->pos_ref.p, pos_dev, n3 * sizeof(double), hipMemcpyDeviceToDevice, s));
  }
  std::memcpy(c->box_at_build, box9, sizeof(c->box_at_build));
  std::memcpy(c->box_at_rebuild, box9, sizeof(c->box_at_rebuild));
  c->built = true;
  c->rebuilds++;
  // k_rank has packed these positions for the new list
  c->packed_pos = pos_dev;
  c->packed_gen = c->rebuilds;
  return P2A_OK;
}

// prepared cell for this box, on the host (fallback kernels take it by value)
// and on the device (the pair kernel reads it for its FP64 cut decisions);
// the device copy is written by a kernel that takes it as an argument, so
// a new box costs no host wait
static int upload_pbc(p2a_coord* c, const double* box9) {
  int rc;
  if (c->pbc_valid && std::memcmp(c->pbc_box, box9, sizeof(c->pbc_box)) == 0 && c->pbc_dev.p) return P2A_OK;
  if ((rc = c->pbc_dev.reserve(1))) return rc;
  pbc_setup(box9, c->pbc);
  std::memcpy(c->pbc_box, box9, sizeof(c->pbc_box));
  c->pbc_valid = true;
  fill_pbc_arg(c->pbc, c->pbc_stage);
  hipLaunchKernelGGL(k_store<PbcArg>, dim3(1), dim3(64), 0, c->stream, c->pbc_stage, c->pbc_dev.p);
  return launch_check("cell upload");
}

// A kept neighbour list under a new cell (NLIST / NLISTCELLS between two
// rebuilds, as NeighborList keeps its pair indices across box changes,
// NeighborList.cpp:433-456): the packed positions and the entry offsets take
// the lattice vectors of the new cell with the integer images chosen at the
// rebuild.  For a pair closer than D_MAX that image is the minimum image of
// the new cell, since every cell width stays above twice the list radius
// (choose_path), which is what Pbc::distance finds for the reference.
// Whether the kept list, imaged for box9, still holds every pair of the
// reference's list that comes within D_MAX.  A listed pair is measured as
// x_j - x_i + k.a with integers k of at most 2 max_wrap + 1 per component
// (wrapping of both atoms plus the cluster image); it is the minimum image of
// the new cell whenever it is shorter than D_MAX (the cell stays wider than
// twice the list radius), and a pair whose minimum image now lies within
// D_MAX was within D_MAX + 2 displacement + |k.(a' - a)| at the rebuild.
// The cell change may use a quarter of NL_CUTOFF - D_MAX for the last term;
// beyond that the list is rebuilt.
static bool reimage_exact(const p2a_coord* c, const double* box9) {
  const double margin = c->spec.nl_cutoff - c->spec.sw.dmax;
  if (!(margin > 0.0)) return false;
  double drift = 0.0;
  for (int r = 0; r < 3; r++) {
    double q = 0.0;
    for (int k = 0; k < 3; k++) {
      const double t = box9[3 * r + k] - c->box_at_rebuild[3 * r + k];
      q += t * t;
    }
    drift += std::sqrt(q);
  }
  return (2.0 * c->max_wrap + 1.0) * drift <= 0.25 * margin;
}

static int reimage(p2a_coord* c, const double* box9) {
  hipStream_t s = c->stream;
  const int ngroups = c->spec.nb > 0 ? 2 : 1;
  BoxArg B;
  std::memcpy(B.a, box9, sizeof(B.a));
  for (int gi = 0; gi < ngroups; gi++) {
    Group& G = c->g[gi];
    SysArg S = G.S;  // the cell grid of the rebuild stays; only the lattice changes
    sys_cell(box9, c->rlist, S);
    hipLaunchKernelGGL(k_store<SysArg>, dim3(1), dim3(64), 0, s, S, G.sys.p);
    G.S_dev = S;
  }
  const int wpb = 256 / WAVE;
  for (int d = 0; d < c->ndir; d++) {
    Dir& D = c->dir[d];
    Group& GI = c->g[D.I];
    Group& GJ = c->g[D.J];
    if (GI.ncl == 0) continue;
    hipLaunchKernelGGL(k_reimage, dim3(grid1(GI.ncl, wpb)), dim3(256), 0, s, GI.ncl, (const int*)D.estart.p,
                       (const int*)D.ecount.p, (int)D.ents.n, (const double4*)GI.origin.p,
                       (const double4*)GJ.origin.p, B, pack_scale(c->spec.sw), D.ents.p);
  }
  std::memcpy(c->box_at_build, box9, sizeof(c->box_at_build));
  return launch_check("reimage");
}

// value / virial / pair count from nred rows of c->partial, in one workgroup
// and a fixed order; the same launch also forms the derivatives of the first
// ngather directions
static int reduce_partials(p2a_coord* c, int nred, double* value_dev, double* virial_dev,
                           int ngather = 0, double* deriv_dev = nullptr, bool with_stats = true,
                           const int* skip = nullptr) {
  hipStream_t s = c->stream;
  Two<GatherSide> T;
  std::memset(&T, 0, sizeof(T));
  int nb[2] = {0, 0};
  for (int d = 0; d < ngather; d++) {
    Dir& D = c->dir[d];
    Group& GI = c->g[D.I];
    nb[d] = grid1((size_t)GI.ncl * CL * 3, 256);
    T.s[d] = GatherSide{GI.ncl, nullptr, GI.p.p, D.istart.p, (int)D.items.n, D.fpart.p};
  }
  T.n0 = nb[0];
  RedArgs R;
  std::memset(&R, 0, sizeof(R));
  R.nred = nred;
  R.partial = c->partial.p;
  R.value = value_dev;
  R.virial = virial_dev;
  R.stats = with_stats ? c->stats.p : nullptr;
  R.skip = skip;
  hipLaunchKernelGGL(k_gather_reduce, dim3(nb[0] + nb[1] + 1), dim3(256), 0, s, T, deriv_dev, 1, R);
  return P2A_OK;
}

// FP32 cluster positions and boxes of this step's positions, unless the
// skin test already packed them for the list in use
static void pack_positions(p2a_coord* c, const double* pos_dev) {
  const bool ahead = c->packed_pos == pos_dev && c->packed_gen == c->rebuilds;
  c->packed_pos = nullptr;
  if (ahead) return;
  const int ngroups = c->spec.nb > 0 ? 2 : 1;
  Two<PackSide> T;
  std::memset(&T, 0, sizeof(T));
  int nb[2] = {0, 0};
  for (int gi = 0; gi < ngroups; gi++) {
    Group& G = c->g[gi];
    T.s[gi] = PackSide{G.ncl * CL, G.slot_loc.p, G.slot_img.p, G.off, G.sys.p, G.origin.p, G.p.p, G.bb.p};
    nb[gi] = G.ncl > 0 ? grid1((size_t)G.ncl * CL, 256) : 0;
  }
  T.n0 = nb[0];
  if (nb[0] + nb[1] > 0)
    hipLaunchKernelGGL(k_pack_bbox, dim3(nb[0] + nb[1]), dim3(256), 0, c->stream, T, pos_dev, pack_scale(c->spec.sw));
}

// skip: a device flag; when it reads nonzero at run time the pair and
// reduction kernels do nothing (a pass queued before the skin test's answer)
static int run_pairs(p2a_coord* c, const double* box9, const double* pos_dev, double* value_dev, double* deriv_dev,
                     double* virial_dev, bool value_only, const int* skip = nullptr) {
  int rc;
  hipStream_t s = c->stream;
  const int ngroups = c->spec.nb > 0 ? 2 : 1;
  pack_positions(c, pos_dev);
  PairArgs A;
  std::memset(&A, 0, sizeof(A));
  A.share = ngroups == 2 && !c->distinct;
  pair_args_switch(c->spec.sw, A);
  if ((rc = upload_pbc(c, box9))) return rc;
  A.pbc = c->pbc_dev.p;
  A.cl_sys = nullptr;
  A.pos64 = pos_dev;
  A.skip = skip;
  A.item_partials = 0;  // value / virial / pair count per workgroup
  // value only: the counting direction (the first) holds every counted pair
  const int ndir_run = value_only ? 1 : c->ndir;
  int grids[2] = {0, 0}, nred = 0;
  for (int d = 0; d < ndir_run; d++) {
    Dir& D = c->dir[d];
    if (D.nitems == 0) continue;
    grids[d] = pair_grid(c, D.nitems);
    nred += grids[d];
  }
  if ((rc = c->partial.reserve(8 * (size_t)std::max(nred, 1)))) return rc;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  const bool rec = c->profiling && (c->prof_calls++ % c->prof_every) == 0;
  if (rec) {
    if (c->ev_pool.size() < 2) {
      hipEvent_t a, b;
      P2A_HIP(hipEventCreate(&a));
      P2A_HIP(hipEventCreate(&b));
      c->ev_pool.push_back(a);
      c->ev_pool.push_back(b);
    }
    e1 = c->ev_pool.back();
    c->ev_pool.pop_back();
    e0 = c->ev_pool.back();
    c->ev_pool.pop_back();
    P2A_HIP(hipEventRecord(e0, s));
  }
  Two<PairSide> T;
  std::memset(&T, 0, sizeof(T));
  T.n0 = grids[0];
  int off = 0;
  for (int d = 0; d < ndir_run; d++) {
    Dir& D = c->dir[d];
    if (grids[d] == 0) continue;
    Group& GI = c->g[D.I];
    Group& GJ = c->g[D.J];
    const int* wave_start = nullptr;
    if (c->tune.blocks_per_cu > 0) {
      // a persistent grid takes contiguous item ranges of balanced cost
      const int nw = grids[d] * (PAIR_BLOCK / WAVE);
      if (D.sched_waves != nw || D.sched_gen != c->rebuilds) {
        if ((rc = D.wave_start.reserve((size_t)nw + 1))) return rc;
        hipLaunchKernelGGL(k_wave_sched, dim3(grid1(std::max(D.nitems, 1), 256)), dim3(256), 0, s, D.nitems,
                           (const int*)nullptr, (int)D.items.n, (const int4*)D.items.p, nw, D.wave_start.p);
        D.sched_waves = nw;
        D.sched_gen = c->rebuilds;
      }
      wave_start = D.wave_start.p;
    }
    T.s[d] = PairSide{grids[d], D.nitems, nullptr,  (int)D.items.n, (int)D.ents.n, wave_start,       D.items.p, D.ents.p,
                      GI.p.p,   GJ.p.p,   GI.bb.p,  GJ.bb.p,        GI.twin_slot.p, D.fpart.p,
                      c->partial.p + 8 * (size_t)off};
    off += grids[d];
  }
  if (off > 0) launch_pairs<true>(A, T, s, value_only, c->tune.chunk);
  if (rec) {
    P2A_HIP(hipEventRecord(e1, s));
    c->pending.emplace_back(e0, e1);
  }
  if ((rc = launch_check("pair kernel"))) return rc;
  // the derivatives go with the reduction
  if ((rc = reduce_partials(c, nred, value_dev, virial_dev, value_only ? 0 : c->ndir, deriv_dev, true, skip))) return rc;
  return launch_check("finalize");
}

static int run_fallback(p2a_coord* c, const double* box9, const double* pos_dev, double* value_dev,
                        double* deriv_dev, double* virial_dev) {
  hipStream_t s = c->stream;
  int rc0;
  if ((rc0 = upload_pbc(c, box9))) return rc0;
  const PbcArg& P = c->pbc_stage;
  const int nA = (int)c->spec.na, nB = (int)c->spec.nb;
  int nblocks;
  int rc;
  if (c->path == 2) {
    nblocks = grid1(nA, 256);
    if ((rc = c->partial.reserve(8 * (size_t)std::max(nblocks, 1)))) return rc;
    hipLaunchKernelGGL(k_pairmode, dim3(std::max(nblocks, 1)), dim3(256), 0, s, nA, c->spec.pbc, P, c->spec.sw,
                       pos_dev, c->abs_dev.p, deriv_dev, c->partial.p);
  } else {
    if ((rc = c->partial.reserve(8 * (size_t)kMaxBlocks64))) return rc;
    nblocks = launch_pairs64(s, nA, nB, c->spec.pbc, P, c->spec.sw, pos_dev,
                             c->distinct ? nullptr : (const long long*)c->abs_dev.p, deriv_dev, c->partial.p);
  }
  if ((rc = launch_check("fp64 pair kernel"))) return rc;
  if ((rc = reduce_partials(c, std::max(nblocks, 1), value_dev, virial_dev))) return rc;
  return launch_check("finalize");
}

// LinkCells grid of the reference's cells branch for this cell and these
// positions (LinkCells::setupCells / createCells, LinkCells.cpp:49-122): the
// given cell, or, when the box is all zero, an orthorhombic box of whole
// NL_CUTOFF multiples around the atoms (whose extent needs the positions on
// the host: this rare case waits for a copy)
static int cell_grid(p2a_coord* c, const double* box9, const double* pos_dev, CellGrid& G) {
  std::memset(&G, 0, sizeof(G));
  const double cut = c->spec.nl_cutoff;
  double box[9];
  bool zero = true;
  for (int k = 0; k < 9; k++) zero = zero && box9[k] == 0.0;
  if (zero) {
    const size_t n3 = 3 * (size_t)c->natoms;
    std::vector<double> x(n3);
    P2A_HIP(hipMemcpyAsync(x.data(), pos_dev, n3 * sizeof(double), hipMemcpyDeviceToHost, c->stream));
    P2A_HIP(hipStreamSynchronize(c->stream));
    std::memset(box, 0, sizeof(box));
    for (int k = 0; k < 3; k++) {
      double lo = x[k], hi = x[k];
      for (int i = 1; i < c->natoms; i++) {
        if (x[3 * (size_t)i + k] > hi) hi = x[3 * (size_t)i + k];
        if (x[3 * (size_t)i + k] < lo) lo = x[3 * (size_t)i + k];
      }
      box[4 * k] = cut < std::sqrt(DBL_MAX) ? cut * (1 + std::ceil((hi - lo) / cut)) : hi - lo + 1;
      G.origin[k] = (lo + hi) / 2;
    }
    G.shift_origin = 1;
  } else {
    std::memcpy(box, box9, sizeof(box));
  }
  PbcHost h;
  pbc_setup(box, h);
  if (h.type == 0 && !zero) return fail(P2A_ERR_ARG, "cell lists cannot be built for a box with null volume");
  std::memcpy(G.inv, h.inv, sizeof(G.inv));
  for (int k = 0; k < 3; k++) {
    // reciprocal row k = column k of the inverse
    const double len = std::sqrt(h.inv[k] * h.inv[k] + h.inv[3 + k] * h.inv[3 + k] + h.inv[6 + k] * h.inv[6 + k]);
    const int n = (int)std::floor(1.0 / len / cut);
    G.nc[k] = n == 0 ? 1 : n;
  }
  G.use_pbc = c->spec.pbc ? 1 : 0;
  return P2A_OK;
}

// The FP64 path with NLIST / NLISTCELLS: the reference's candidate pairs are
// listed on the first step and every NL_STRIDE steps (NeighborList::prepare,
// NeighborList.cpp:433-456) and evaluated, with the current positions and
// cell, until the next rebuild.  Classic: pairs with |d|^2 <= NL_CUTOFF^2
// from Pbc::distance (NeighborList.cpp:237-308); cells: the pairs of atoms
// whose link cells are within one stencil (NeighborList.cpp:177-236).
// build: list the pairs at these positions first; value_dev null: no evaluation
static int run_fallback_nl(p2a_coord* c, bool build, const double* box9, const double* pos_dev,
                           double* value_dev, double* deriv_dev, double* virial_dev) {
  hipStream_t s = c->stream;
  int rc;
  if ((rc = upload_pbc(c, box9))) return rc;
  const PbcArg& P = c->pbc_stage;
  const int nA = (int)c->spec.na, nB = (int)c->spec.nb;
  const int natoms = c->natoms;
  const double cut2 = c->spec.nl_cutoff * c->spec.nl_cutoff;
  const int use_pbc = c->spec.pbc ? 1 : 0;
  if (build || !c->nl_valid) {
    if (c->spec.pair) {
      if ((rc = c->nl_count.reserve(std::max(nA, 1)))) return rc;
      hipLaunchKernelGGL(k_nl_pairs_keep, dim3(grid1(std::max(nA, 1), 256)), dim3(256), 0, s, nA, use_pbc, P, cut2,
                         pos_dev, c->nl_count.p);
    } else {
      CellGrid G;
      std::memset(&G, 0, sizeof(G));
      const int mode = c->spec.nl_mode;
      if ((rc = c->nl_count.reserve(natoms)) || (rc = c->nl_start.reserve((size_t)natoms + 1)) ||
          (rc = c->nl_total.reserve(1)))
        return rc;
      if (mode == P2A_NL_CELLS) {
        if ((rc = cell_grid(c, box9, pos_dev, G))) return rc;
        if ((rc = c->nl_cell.reserve(3 * (size_t)natoms))) return rc;
        hipLaunchKernelGGL(k_nl_cells, dim3(grid1(natoms, 256)), dim3(256), 0, s, natoms, G, pos_dev, c->nl_cell.p);
      }
      launch_nl_atoms<0>(s, nA, nB, mode == P2A_NL_CELLS, use_pbc, P, cut2, G, pos_dev, c->nl_cell.p, c->nl_count.p,
                         nullptr, nullptr);
      hipLaunchKernelGGL(k_scan_small, dim3(1), dim3(1024), 0, s, natoms, (const int*)c->nl_count.p, c->nl_start.p,
                         c->nl_total.p);
      long long total = 0;
      P2A_HIP(hipMemcpyAsync(c->host_ro + 40, c->nl_total.p, sizeof(long long), hipMemcpyDeviceToHost, s));
      P2A_HIP(hipStreamSynchronize(s));
      std::memcpy(&total, c->host_ro + 40, sizeof(total));
      if (total > INT32_MAX) return fail(P2A_ERR_UNSUPPORTED, "neighbour list too long for the FP64 path");
      if ((rc = c->nl_nbr.reserve(std::max<long long>(total, 1)))) return rc;
      c->nl_entries = total;
      launch_nl_atoms<1>(s, nA, nB, mode == P2A_NL_CELLS, use_pbc, P, cut2, G, pos_dev, c->nl_cell.p, nullptr,
                         c->nl_start.p, c->nl_nbr.p);
    }
    if ((rc = launch_check("FP64 neighbour list"))) return rc;
    c->nl_valid = true;
    c->rebuilds++;
  }
  if (!value_dev) return P2A_OK;
  int nblocks;
  if (c->spec.pair) {
    nblocks = grid1(nA, 256);
    if ((rc = c->partial.reserve(8 * (size_t)std::max(nblocks, 1)))) return rc;
    hipLaunchKernelGGL(k_pairmode, dim3(std::max(nblocks, 1)), dim3(256), 0, s, nA, c->spec.pbc, P, c->spec.sw,
                       pos_dev, c->abs_dev.p, deriv_dev, c->partial.p, (const int*)c->nl_count.p);
  } else {
    if ((rc = c->partial.reserve(8 * (size_t)kMaxListBlocks64))) return rc;
    nblocks = launch_pairs64(s, nA, nB, c->spec.pbc, P, c->spec.sw, pos_dev,
                             c->distinct ? nullptr : (const long long*)c->abs_dev.p, deriv_dev, c->partial.p,
                             c->nl_start.p, c->nl_nbr.p, c->nl_entries);
  }
  if ((rc = launch_check("fp64 pair kernel"))) return rc;
  if ((rc = reduce_partials(c, std::max(nblocks, 1), value_dev, virial_dev))) return rc;
  return launch_check("finalize");
}

// COORDINATIONNUMBER rows of GROUPA over the environment (GROUPA itself, or
// GROUPB) on the cluster list, and with weights their vector-Jacobian
// product and box derivative
static int run_rows(p2a_coord* c, const double* box9, const double* pos_dev, double* rows_dev,
                    const double* weights_dev, double* vjp_dev, double* virial_dev) {
  int rc;
  hipStream_t s = c->stream;
  const int ngroups = c->spec.nb > 0 ? 2 : 1;
  pack_positions(c, pos_dev);
  PairArgs A;
  std::memset(&A, 0, sizeof(A));
  A.share = ngroups == 2 && !c->distinct;
  pair_args_switch(c->spec.sw, A);
  if ((rc = upload_pbc(c, box9))) return rc;
  A.pbc = c->pbc_dev.p;
  A.pos64 = pos_dev;
  const bool weighted = weights_dev != nullptr;
  if (weighted) {
    for (int gi = 0; gi < ngroups; gi++) {
      Group& G = c->g[gi];
      if (G.ncl == 0) continue;
      if ((rc = G.pw.reserve((size_t)G.maxcl * CL))) return rc;
      hipLaunchKernelGGL(k_row_weights, dim3(grid1((size_t)G.ncl * CL, 256)), dim3(256), 0, s, G.ncl * CL,
                         (int)c->spec.na, (const float4*)G.p.p, weights_dev, G.pw.p);
    }
  }
  // the rows come from the first direction (i = GROUPA); the weighted
  // product needs every direction for the derivatives of all atoms
  const int ndir_run = weighted ? c->ndir : 1;
  int grids[2] = {0, 0}, nred = 0;
  for (int d = 0; d < ndir_run; d++) {
    Dir& D = c->dir[d];
    if (D.nitems == 0) continue;
    int grid = grid1(D.nitems, PAIR_BLOCK / WAVE);
    if (c->tune.blocks_per_cu > 0) grid = std::min(grid, c->tune.blocks_per_cu * c->cu_count);
    grids[d] = grid;
    nred += grid;
  }
  if ((rc = c->partial.reserve(8 * (size_t)std::max(nred, 1)))) return rc;
  int off = 0;
  for (int d = 0; d < ndir_run; d++) {
    Dir& D = c->dir[d];
    if (grids[d] == 0) continue;
    Group& GI = c->g[D.I];
    Group& GJ = c->g[D.J];
    if ((rc = D.rpart.reserve((size_t)CL * std::max(D.nitems, 1)))) return rc;
    A.nitems = D.nitems;
    A.items_cap = (int)D.items.n;
    A.ent_cap = (int)D.ents.n;
    launch_rows(A, weighted, grids[d], s, D.items.p, D.ents.p, GI.p.p, GJ.p.p, GI.pw.p, GJ.pw.p, GI.bb.p, GJ.bb.p,
                GI.twin_slot.p, D.rpart.p, D.fpart.p, c->partial.p + 8 * (size_t)off);
    off += grids[d];
  }
  if ((rc = launch_check("row kernel"))) return rc;
  {
    Dir& D = c->dir[0];
    Group& GI = c->g[D.I];
    if (GI.ncl > 0 && D.nitems > 0)
      hipLaunchKernelGGL(k_gather_rows, dim3(grid1((size_t)GI.ncl * CL, 256)), dim3(256), 0, s, GI.ncl * CL, GI.p.p,
                         (const int*)D.istart.p, (int)D.items.n, (const double*)D.rpart.p, (int)c->spec.na,
                         rows_dev);
    else
      hipLaunchKernelGGL(k_fill_double, dim3(grid1((size_t)c->spec.na, 256)), dim3(256), 0, s, rows_dev,
                         (size_t)c->spec.na);
  }
  if (!weighted) return launch_check("rows");
  if ((rc = c->out_buf.reserve(16))) return rc;
  double* wdev = virial_dev ? virial_dev : c->out_buf.p + 1;
  if ((rc = reduce_partials(c, nred, c->out_buf.p, wdev, c->ndir, vjp_dev, false))) return rc;
  return launch_check("row derivatives");
}

// The cluster list for this step: NeighborList::prepare (NeighborList.cpp:
// 433-456) rebuilds on the first step and every NL_STRIDE steps.  Without a
// neighbour list every step, or, with a skin, when some atom has moved more
// than skin/2 since the build: every pair within D_MAX now was within D_MAX +
// skin then, so the pairs evaluated are those of a list rebuilt now.
// The skin test on the device: moved = 1 when some atom has moved more than
// skin/2 since the build; the flag is copied to host_ro[32] and moved_ev
// recorded after the copy.
static int launch_moved_test(p2a_coord* c, const double* pos_dev) {
  int rc;
  if ((rc = c->moved.reserve(1))) return rc;
  if (!c->moved_ev) P2A_HIP(hipEventCreateWithFlags(&c->moved_ev, hipEventDisableTiming));
  const double half = 0.5 * c->skin_active;
  hipLaunchKernelGGL(k_fill_int, dim3(1), dim3(64), 0, c->stream, c->moved.p, 1, 0);
  hipLaunchKernelGGL(k_moved, dim3(grid1((size_t)c->natoms, 256)), dim3(256), 0, c->stream, c->natoms, pos_dev,
                     (const double*)c->pos_ref.p, half * half, c->moved.p);
  P2A_HIP(hipMemcpyAsync(c->host_ro + 32, c->moved.p, sizeof(int), hipMemcpyDeviceToHost, c->stream));
  P2A_HIP(hipEventRecord(c->moved_ev, c->stream));
  return launch_check("skin test");
}

// A list that the skin test may keep: no neighbour list, a skin in use, a
// list built on an earlier call in this same cell.
static bool skin_kept_candidate(p2a_coord* c, const double* box9) {
  return c->spec.nl_mode == P2A_NL_NONE && c->skin_active > 0.0 && c->built && !c->firsttime &&
         std::memcmp(c->box_at_build, box9, sizeof(c->box_at_build)) == 0;
}

static int prepare_cluster_list(p2a_coord* c, int64_t step, const double* box9, const double* pos_dev) {
  int rc;
  bool need = !c->built || c->firsttime;
  const bool new_cell = !need && std::memcmp(c->box_at_build, box9, sizeof(c->box_at_build)) != 0;
  if (c->spec.nl_mode == P2A_NL_NONE) {
    // the skin test measures motion in one cell: a new cell rebuilds
    if (new_cell) need = true;
    if (!need && c->skin_active > 0.0) {
      if ((rc = launch_moved_test(c, pos_dev))) return rc;
      // the positions are packed for the kept list while the host waits for
      // the answer (a rebuild packs them again)
      pack_positions(c, pos_dev);
      c->packed_pos = pos_dev;
      c->packed_gen = c->rebuilds;
      P2A_HIP(hipEventSynchronize(c->moved_ev));
      need = c->host_ro[32] != 0;
    } else {
      need = true;
    }
  } else if (c->spec.nl_stride <= 1 || step % c->spec.nl_stride == 0) {
    need = true;
  }
  c->firsttime = false;
  if (!need && new_cell && !reimage_exact(c, box9)) need = true;
  if (need) {
    if ((rc = rebuild(c, box9, pos_dev))) return rc;
  } else if (new_cell) {
    if ((rc = reimage(c, box9))) return rc;
  }
  return P2A_OK;
}

static int calc_device(p2a_coord* c, int64_t step, const double* box9, const double* pos_dev, double* value_dev,
                       double* deriv_dev, double* virial_dev) {
  int rc;
  if (!box9) return fail(P2A_ERR_ARG, "box is required");
  // positions packed ahead count only within the call that packed them (the
  // same address may hold other positions at a later call)
  c->packed_pos = nullptr;
  if (!c->stats.p) {
    if ((rc = c->stats.reserve(8))) return rc;
    hipLaunchKernelGGL(k_fill_double, dim3(1), dim3(64), 0, c->stream, c->stats.p, (size_t)8);
  }
  // no derivative and no virial requested: the cheaper value-only kernel
  const bool value_only = (deriv_dev == nullptr && virial_dev == nullptr);
  double* vdev = value_dev;
  double* wdev = virial_dev;
  double* ddev = deriv_dev;
  if (!vdev || !wdev) {
    if ((rc = c->out_buf.reserve(16))) return rc;
    if (!vdev) vdev = c->out_buf.p;
    if (!wdev) wdev = c->out_buf.p + 1;
  }
  if (!ddev) {
    if ((rc = c->deriv_buf.reserve(3 * (size_t)std::max(c->natoms, 1)))) return rc;
    ddev = c->deriv_buf.p;
  }
  int path = choose_path(c, box9);
  if (path != c->path) {
    // the list of the other path is not carried over: rebuild now
    c->built = false;
    c->nl_valid = false;
  }
  c->path = path;
  if (path != 0) {
    if (c->spec.nl_mode != P2A_NL_NONE) {
      const bool build = c->spec.nl_stride <= 1 || step % c->spec.nl_stride == 0;
      return run_fallback_nl(c, build, box9, pos_dev, vdev, ddev, wdev);
    }
    return run_fallback(c, box9, pos_dev, vdev, ddev, wdev);
  }
  if (skin_kept_candidate(c, box9)) {
    // The pass on the kept list is queued behind the displacement test and
    // does nothing on the device if the test finds an atom that moved too far;
    // the host waits only for the test's answer, while the pass runs.
    if ((rc = launch_moved_test(c, pos_dev))) return rc;
    if ((rc = run_pairs(c, box9, pos_dev, vdev, ddev, wdev, value_only, c->moved.p))) return rc;
    P2A_HIP(hipEventSynchronize(c->moved_ev));
    if (c->host_ro[32] == 0) return P2A_OK;
    if ((rc = rebuild(c, box9, pos_dev))) return rc;
    return run_pairs(c, box9, pos_dev, vdev, ddev, wdev, value_only);
  }
  if ((rc = prepare_cluster_list(c, step, box9, pos_dev))) return rc;
  return run_pairs(c, box9, pos_dev, vdev, ddev, wdev, value_only);
}

static void collect_profile(p2a_coord* c) {
  for (auto& pr : c->pending) {
    float ms = 0.f;
    if (hipEventElapsedTime(&ms, pr.first, pr.second) == hipSuccess) {
      c->prof_ms += ms;
      c->prof_launches++;
    }
    c->ev_pool.push_back(pr.first);
    c->ev_pool.push_back(pr.second);
  }
  c->pending.clear();
}

// COORDINATIONNUMBER rows: cn[k] = sum over env atoms j of the contact
// matrix element of (rows[k], j), ContactMatrix::calculateWeight
// (src/adjmat/ContactMatrix.h:95-121): nothing when |r|^2 < DBL_EPSILON (the
// diagonal, or two atoms at one place), s(r) zeroed below DBL_EPSILON.  FP64,
// WIDE: a wave per row, the environment over its lanes; else a thread per row.  An
// index outside [0, natoms) makes that row NaN instead of being read.
template <bool WIDE>
__global__ __launch_bounds__(256) void k_cn_rows(int natoms, int nrows, const int* __restrict__ rows, int nenv,
                                                 const int* __restrict__ env, int use_pbc, PbcArg P, p2a_switch sw,
                                                 const double* __restrict__ pos, double* __restrict__ cn) {
  const int lane = WIDE ? threadIdx.x & 63 : 0;
  const int k = WIDE ? blockIdx.x * 4 + (threadIdx.x >> 6) : blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nrows) return;
  const int i = rows[k];
  if (i < 0 || i >= natoms) {
    if (lane == 0) cn[k] = __builtin_nan("");
    return;
  }
  const double* xi = pos + 3 * (size_t)i;
  double sum = 0.0;
  for (int q = lane; q < nenv; q += WIDE ? WAVE : 1) {
    const int j = env[q];
    if (j < 0 || j >= natoms) {
      sum = __builtin_nan("");
      break;
    }
    const double* xj = pos + 3 * (size_t)j;
    double d[3];
    if (use_pbc) pbc_distance(P, xi, xj, d);
    else { d[0] = xj[0] - xi[0]; d[1] = xj[1] - xi[1]; d[2] = xj[2] - xi[2]; }
    const double mod2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
    if (mod2 < DBL_EPSILON) continue;
    double df;
    const double v = switch_calc_sqr(sw, mod2, df);
    if (v < DBL_EPSILON) continue;
    sum += v;
  }
  if constexpr (WIDE) sum = wave_sum_d(sum);
  if (lane == 0) cn[k] = sum;
}

// A thread per row takes about 0.5 us an environment atom while the rows do not
// fill the chip, a wave per row about 0.5 us a thousand rows while its lanes hold
// the environment: a thread per row from 1,000 rows an environment atom on, and
// for rows that fill the chip as threads (a row's environment is then read by
// all lanes together).  Thread / wave: 16,000 rows x 16 atoms 12 / 11 us, 100,000 x
// 64 36 / 51, 500,000 x 1 7 / 266, 500,000 x 256 314 / 542, 4,000 x 256 153 / 8.
static void launch_cn_rows(hipStream_t s, int natoms, int nrows, const int* rows, int nenv, const int* env,
                           int use_pbc, const PbcArg& P, const p2a_switch& sw, const double* pos, double* cn) {
  if (nrows >= (1 << 18) || nrows >= 1000 * (int64_t)nenv)
    hipLaunchKernelGGL(k_cn_rows<false>, dim3(grid1((size_t)nrows, 256)), dim3(256), 0, s, natoms, nrows, rows, nenv,
                       env, use_pbc, P, sw, pos, cn);
  else
    hipLaunchKernelGGL(k_cn_rows<true>, dim3(grid1((size_t)nrows, 4)), dim3(256), 0, s, natoms, nrows, rows, nenv,
                       env, use_pbc, P, sw, pos, cn);
}

// Scratch of the allocation-free entry point: the per-workgroup partials of
// k_allpairs that k_finalize sums (8 doubles for each of kMaxBlocks64).  Each
// device holds its own copy for the life of the process; its address is
// looked up once per device and kept in g_scratch_dev.
constexpr int kNoAllocMaxAtoms = 1 << 18;
static __device__ __align__(256) double scratch[8 * kMaxBlocks64];

constexpr int kMaxDevices = 64;
static std::mutex g_scratch_mu;
static double* g_scratch_dev[kMaxDevices] = {};

// device address of `scratch` on the current device (hipGetSymbolAddress,
// once per device); the host-side name is not a device address
static int noalloc_scratch(int device, double** out) {
  if (device < 0 || device >= kMaxDevices) return fail(P2A_ERR_ARG, "device index out of range");
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch_dev[device]) {
    void* ptr = nullptr;
    hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr)
      return fail(P2A_ERR_HIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
    g_scratch_dev[device] = static_cast<double*>(ptr);
  }
  *out = g_scratch_dev[device];
  return P2A_OK;
}

}  // namespace p2a

using namespace p2a;

extern "C" {

int p2a_device_count(void) {
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess) return 0;
  return n;
}

int p2a_coord_create(p2a_coord** out, int device, const p2a_coord_spec* spec) {
  if (!out || !spec) return fail(P2A_ERR_ARG, "null argument");
  *out = nullptr;
  if (spec->na <= 0) return fail(P2A_ERR_ARG, "GROUPA should contain at least one atom");
  if (spec->pair && spec->na != spec->nb)
    return fail(P2A_ERR_ARG, "when using PAIR the two groups should have the same number of atoms");
  if (spec->nl_mode != P2A_NL_NONE && (spec->nl_cutoff <= 0.0 || spec->nl_stride <= 0))
    return fail(P2A_ERR_ARG, "NL_CUTOFF and NL_STRIDE should be explicitly specified and positive");
  if (spec->na + spec->nb > (int64_t)1 << 29) return fail(P2A_ERR_UNSUPPORTED, "more than 2^29 atoms");
  if (spec->pair && spec->nl_mode == P2A_NL_CELLS)
    return fail(P2A_ERR_ARG, "Cell list should not be active with a Pair NL");
  if (spec->nl_mode != P2A_NL_NONE && spec->sw.dmax > spec->nl_cutoff)
    return fail(P2A_ERR_UNSUPPORTED,
                "D_MAX larger than NL_CUTOFF: the stale neighbour list of the reference would drop pairs; "
                "use D_MAX <= NL_CUTOFF");
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) return fail(P2A_ERR_HIP, "no HIP device available");
  if (device < 0 || device >= ndev) return fail(P2A_ERR_ARG, "device index out of range");
  P2A_HIP(hipSetDevice(device));
  auto* c = new p2a_coord();
  c->device = device;
  c->spec = *spec;
  c->spec.groupa = nullptr;
  c->spec.groupb = nullptr;
  c->natoms = (int)(spec->na + spec->nb);
  c->abs.resize(c->natoms);
  for (int64_t i = 0; i < spec->na; i++) c->abs[i] = spec->groupa[i];
  for (int64_t i = 0; i < spec->nb; i++) c->abs[spec->na + i] = spec->groupb[i];
  std::vector<int64_t> sorted[2];
  for (int gi = 0; gi < 2; gi++) {
    const int64_t* g = gi == 0 ? spec->groupa : spec->groupb;
    std::vector<int64_t>& v = sorted[gi];
    v.assign(g, g + (gi == 0 ? spec->na : spec->nb));
    if (!std::is_sorted(v.begin(), v.end())) std::sort(v.begin(), v.end());
    if (std::adjacent_find(v.begin(), v.end()) != v.end()) c->has_duplicates = true;
  }
  c->distinct = !c->has_duplicates;
  for (auto a = sorted[0].begin(), b = sorted[1].begin(); c->distinct && a != sorted[0].end() && b != sorted[1].end();) {
    if (*a == *b) c->distinct = false;
    else if (*a < *b) ++a;
    else ++b;
  }
  int ncu = 0;
  if (hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, device) == hipSuccess && ncu > 0)
    c->cu_count = ncu;
  if (hipStreamCreateWithFlags(&c->own_stream, hipStreamNonBlocking) != hipSuccess) {
    delete c;
    return fail(P2A_ERR_HIP, "hipStreamCreate failed");
  }
  c->stream = c->own_stream;
  if (hipHostMalloc((void**)&c->host_ro, 64 * sizeof(int), hipHostMallocDefault) != hipSuccess) {
    c->host_ro = nullptr;
    p2a_coord_destroy(c);
    return fail(P2A_ERR_HIP, "hipHostMalloc failed");
  }
  int rc;
  if ((rc = c->abs_dev.reserve(c->natoms))) {
    p2a_coord_destroy(c);
    return rc;
  }
  if (!c->distinct && !c->has_duplicates && c->spec.nb > 0) {
    // (duplicates within a group take the FP64 path)
    std::vector<std::pair<int64_t, int>> by[2];
    std::vector<int> twin(c->natoms, -2);
    for (int gi = 0; gi < 2; gi++) {
      const int off = gi == 0 ? 0 : (int)spec->na, n = (int)(gi == 0 ? spec->na : spec->nb);
      for (int k = 0; k < n; k++) by[gi].push_back({c->abs[off + k], off + k});
      std::sort(by[gi].begin(), by[gi].end());
    }
    for (size_t a = 0, b = 0; a < by[0].size() && b < by[1].size();) {
      if (by[0][a].first == by[1][b].first) {
        twin[by[0][a].second] = by[1][b].second;
        twin[by[1][b].second] = by[0][a].second;
        a++;
        b++;
      } else if (by[0][a].first < by[1][b].first) {
        a++;
      } else {
        b++;
      }
    }
    if ((rc = c->twin_dev.reserve(c->natoms))) {
      p2a_coord_destroy(c);
      return rc;
    }
    if (hipMemcpy(c->twin_dev.p, twin.data(), twin.size() * sizeof(int), hipMemcpyHostToDevice) != hipSuccess) {
      p2a_coord_destroy(c);
      return fail(P2A_ERR_HIP, "hipMemcpy of the shared atoms failed");
    }
  }
  std::vector<long long> ab(c->abs.begin(), c->abs.end());
  if (hipMemcpy(c->abs_dev.p, ab.data(), ab.size() * sizeof(long long), hipMemcpyHostToDevice) != hipSuccess) {
    p2a_coord_destroy(c);
    return fail(P2A_ERR_HIP, "hipMemcpy of atom indices failed");
  }
  *out = c;
  g_last_error.clear();
  return P2A_OK;
}

int p2a_coord_destroy(p2a_coord* c) {
  if (!c) return P2A_OK;
  (void)hipSetDevice(c->device);
  if (c->stream) (void)hipStreamSynchronize(c->stream);
  for (auto& pr : c->pending) {
    c->ev_pool.push_back(pr.first);
    c->ev_pool.push_back(pr.second);
  }
  for (auto e : c->ev_pool) (void)hipEventDestroy(e);
  if (c->moved_ev) (void)hipEventDestroy(c->moved_ev);
  if (c->own_stream) (void)hipStreamDestroy(c->own_stream);
  if (c->host_ro) (void)hipHostFree(c->host_ro);
  delete c;
  return P2A_OK;
}

int p2a_coord_set_stream(p2a_coord* c, void* stream) {
  if (!c) return fail(P2A_ERR_ARG, "null context");
  // NULL selects the default (null) stream, which orders with every blocking stream
  c->stream = (hipStream_t)stream;
  return P2A_OK;
}

int p2a_coord_set_tuning(p2a_coord* c, int chunk, int blocks_per_cu) {
  if (!c) return fail(P2A_ERR_ARG, "null context");
  if (chunk != 32 && chunk != 64) return fail(P2A_ERR_ARG, "chunk must be 32 or 64");
  if (blocks_per_cu < 0 || blocks_per_cu > 64) return fail(P2A_ERR_ARG, "blocks_per_cu must be in [0, 64]");
  // the work items depend on the chunk: the next call rebuilds them
  if (chunk != c->tune.chunk) c->built = false;
  c->tune.chunk = chunk;
  c->tune.blocks_per_cu = blocks_per_cu;
  return P2A_OK;
}

int p2a_coord_calculate_device(p2a_coord* c, int64_t step, const double* box9, const double* pos_dev,
                               double* value_dev, double* deriv_dev, double* virial_dev) {
  if (!c || !pos_dev) return fail(P2A_ERR_ARG, "null argument");
  P2A_HIP(hipSetDevice(c->device));
  return calc_device(c, step, box9, pos_dev, value_dev, deriv_dev, virial_dev);
}

int p2a_coord_backward_device(p2a_coord* c, const double* box9, const double* pos_dev, double* deriv_dev,
                              double* virial_dev) {
  if (!c || !pos_dev || !box9 || !deriv_dev) return fail(P2A_ERR_ARG, "null argument");
  P2A_HIP(hipSetDevice(c->device));
  c->packed_pos = nullptr;  // packed ahead by an earlier call: pack again
  int rc;
  if ((rc = c->out_buf.reserve(16))) return rc;
  double* wdev = virial_dev ? virial_dev : c->out_buf.p + 1;
  if (c->path != 0 || choose_path(c, box9) != 0) {
    // the pairs of the last listing (a neighbour list is kept as the forward left it)
    if (c->spec.nl_mode != P2A_NL_NONE) return run_fallback_nl(c, false, box9, pos_dev, c->out_buf.p, deriv_dev, wdev);
    return run_fallback(c, box9, pos_dev, c->out_buf.p, deriv_dev, wdev);
  }
  if (!c->built || std::memcmp(c->box_at_build, box9, sizeof(c->box_at_build)) != 0)
    return fail(P2A_ERR_ARG, "backward needs the neighbour structure of a forward call on the same box");
  return run_pairs(c, box9, pos_dev, c->out_buf.p, deriv_dev, wdev, false);
}

int p2a_coord_calculate_noalloc(void* stream, const p2a_switch* sw, const double* box9, int use_pbc, int64_t na,
                                int64_t nb, const int64_t* absidx_dev, const double* pos_dev, double* value_dev,
                                double* deriv_dev, double* virial_dev) {
  if (!sw || !pos_dev || !value_dev || !deriv_dev || !virial_dev) return fail(P2A_ERR_ARG, "null argument");
  if (na <= 0) return fail(P2A_ERR_ARG, "GROUPA should contain at least one atom");
  if (nb < 0) return fail(P2A_ERR_ARG, "GROUPB cannot have a negative size");
  if (na + nb > kNoAllocMaxAtoms)
    return fail(P2A_ERR_ARG, "p2a_coord_calculate_noalloc handles at most " + std::to_string(kNoAllocMaxAtoms) +
                                 " atoms");
  if (use_pbc && !box9) return fail(P2A_ERR_ARG, "box is required with periodic boundaries");
  int dev = 0;
  P2A_HIP(hipGetDevice(&dev));
  if (stream) {
    int sdev = -1;
    P2A_HIP(hipStreamGetDevice((hipStream_t)stream, &sdev));
    if (sdev != dev) return fail(P2A_ERR_ARG, "the stream belongs to another device than the current one");
  }
  double* part = nullptr;
  int rc;
  if ((rc = noalloc_scratch(dev, &part))) return rc;
  PbcArg P;
  std::memset(&P, 0, sizeof(P));
  if (use_pbc) {
    PbcHost h;
    pbc_setup(box9, h);
    if (h.type == 0) return fail(P2A_ERR_ARG, "the box is singular");
    fill_pbc_arg(h, P);
  }
  hipStream_t s = (hipStream_t)stream;
  // every workgroup writes its 8 partials, so nothing in scratch needs clearing
  const int nblocks = launch_pairs64(s, (int)na, (int)nb, use_pbc ? 1 : 0, P, *sw, pos_dev,
                                     (const long long*)absidx_dev, deriv_dev, part);
  hipLaunchKernelGGL(k_finalize, dim3(1), dim3(128), 0, s, nblocks, (const double*)part, value_dev, virial_dev,
                     (double*)nullptr);
  return launch_check("p2a_coord_calculate_noalloc");
}

int p2a_coord_list_generation(p2a_coord* c, int64_t* gen) {
  if (!c || !gen) return fail(P2A_ERR_ARG, "null argument");
  // the host counts the rebuilds it enqueues: no synchronisation
  *gen = c->rebuilds;
  return P2A_OK;
}

int p2a_coord_rebuild_device(p2a_coord* c, const double* box9, const double* pos_dev) {
  if (!c || !box9 || !pos_dev) return fail(P2A_ERR_ARG, "null argument");
  P2A_HIP(hipSetDevice(c->device));
  int rc;
  if (!c->stats.p) {
    if ((rc = c->stats.reserve(8))) return rc;
    hipLaunchKernelGGL(k_fill_double, dim3(1), dim3(64), 0, c->stream, c->stats.p, (size_t)8);
  }
  const int path = choose_path(c, box9);
  if (path != c->path) {
    c->built = false;
    c->nl_valid = false;
  }
  c->path = path;
  if (path != 0) {
    // without a neighbour list the FP64 kernels keep no pair structure
    if (c->spec.nl_mode == P2A_NL_NONE) return P2A_OK;
    return run_fallback_nl(c, true, box9, pos_dev, nullptr, nullptr, nullptr);
  }
  c->firsttime = false;
  return rebuild(c, box9, pos_dev);
}

int p2a_coord_calculate(p2a_coord* c, int64_t step, const double* box9, const double* pos, double* value,
                        double* deriv, double* virial) {
  if (!c || !pos) return fail(P2A_ERR_ARG, "null argument");
  P2A_HIP(hipSetDevice(c->device));
  int rc;
  const size_t n3 = 3 * (size_t)c->natoms;
  if ((rc = c->pos_buf.reserve(n3)) || (rc = c->deriv_buf.reserve(n3)) || (rc = c->out_buf.reserve(16))) return rc;
  P2A_HIP(hipMemcpyAsync(c->pos_buf.p, pos, n3 * sizeof(double), hipMemcpyHostToDevice, c->stream));
  if ((rc = calc_device(c, step, box9, c->pos_buf.p, c->out_buf.p, deriv ? c->deriv_buf.p : nullptr,
                        (deriv || virial) ? c->out_buf.p + 1 : nullptr)))
    return rc;
  double out[10];
  P2A_HIP(hipMemcpyAsync(out, c->out_buf.p, 10 * sizeof(double), hipMemcpyDeviceToHost, c->stream));
  if (deriv) P2A_HIP(hipMemcpyAsync(deriv, c->deriv_buf.p, n3 * sizeof(double), hipMemcpyDeviceToHost, c->stream));
  P2A_HIP(hipStreamSynchronize(c->stream));
  if (value) *value = out[0];
  if (virial) std::memcpy(virial, out + 1, 9 * sizeof(double));
  return P2A_OK;
}

int p2a_coord_set_skin(p2a_coord* c, double skin) {
  if (!c) return fail(P2A_ERR_ARG, "null argument");
  if (!(skin >= 0.0) || !std::isfinite(skin)) return fail(P2A_ERR_ARG, "the skin must be a finite distance >= 0");
  c->skin = skin;
  c->path_cached = -1;  // the radius decides whether the cell is wide enough
  c->built = false;
  return P2A_OK;
}

int p2a_coord_get_stats(p2a_coord* c, p2a_coord_stats* st) {
  if (!c || !st) return fail(P2A_ERR_ARG, "null argument");
  P2A_HIP(hipSetDevice(c->device));
  P2A_HIP(hipStreamSynchronize(c->stream));
  std::memset(st, 0, sizeof(*st));
  st->natoms = c->natoms;
  if (c->stats.p) {
    double d[2];
    P2A_HIP(hipMemcpy(d, c->stats.p, 2 * sizeof(double), hipMemcpyDeviceToHost));
    st->contributing_pairs = (int64_t)d[0];
    st->total_contributing_pairs = (int64_t)d[1];
  }
  const int ngroups = c->spec.nb > 0 ? 2 : 1;
  st->clusters_i = c->g[0].ncl;
  st->clusters_j = c->g[ngroups - 1].ncl;
  st->list_entries = c->nentries;
  st->rebuilds = c->rebuilds;
  st->path = c->path;
  collect_profile(c);
  st->pair_kernel_ms = c->prof_ms;
  st->pair_kernel_launches = c->prof_launches;
  return P2A_OK;
}

int p2a_coord_set_profiling(p2a_coord* c, int on) {
  if (!c) return fail(P2A_ERR_ARG, "null context");
  P2A_HIP(hipSetDevice(c->device));
  P2A_HIP(hipStreamSynchronize(c->stream));
  collect_profile(c);
  if (on < 0) return fail(P2A_ERR_ARG, "the profiling interval must be >= 0");
  c->profiling = on != 0;
  if (on) {
    c->prof_every = on;
    c->prof_calls = 0;
    c->prof_ms = 0.0;
    c->prof_launches = 0;
    if (c->stats.p) {
      hipLaunchKernelGGL(k_fill_double, dim3(1), dim3(64), 0, c->stream, c->stats.p + 1, (size_t)1);
      P2A_HIP(hipStreamSynchronize(c->stream));
    }
  }
  return P2A_OK;
}

int p2a_coord_rows_device(p2a_coord* c, int64_t step, const double* box9, const double* pos_dev, double* rows_dev,
                          const double* weights_dev, double* vjp_dev, double* virial_dev) {
  if (!c || !box9 || !pos_dev || !rows_dev) return fail(P2A_ERR_ARG, "null argument");
  if (weights_dev && !vjp_dev) return fail(P2A_ERR_ARG, "weights need an output for their derivatives");
  if (c->spec.pair) return fail(P2A_ERR_UNSUPPORTED, "PAIR gives no per-atom rows");
  P2A_HIP(hipSetDevice(c->device));
  c->packed_pos = nullptr;  // packed ahead by an earlier call: pack again
  int rc;
  if (!c->stats.p) {
    if ((rc = c->stats.reserve(8))) return rc;
    hipLaunchKernelGGL(k_fill_double, dim3(1), dim3(64), 0, c->stream, c->stats.p, (size_t)8);
  }
  const int path = choose_path(c, box9);
  if (path != c->path) {
    c->built = false;
    c->nl_valid = false;
  }
  c->path = path;
  if (path != 0) {
    if (weights_dev)
      return fail(P2A_ERR_UNSUPPORTED,
                  "derivatives of per-atom coordination numbers need the cluster path (a periodic cell wider than "
                  "twice the list radius, distinct atoms)");
    // every environment atom of every row, in FP64
    const int na = (int)c->spec.na, nb = (int)c->spec.nb;
    const int nenv = nb > 0 ? nb : na;
    if ((rc = c->cn_rows.reserve(na)) || (rc = c->cn_env.reserve(nenv))) return rc;
    std::vector<int> r(na), e(nenv);
    for (int k = 0; k < na; k++) r[k] = k;
    for (int k = 0; k < nenv; k++) e[k] = nb > 0 ? na + k : k;
    P2A_HIP(hipMemcpyAsync(c->cn_rows.p, r.data(), na * sizeof(int), hipMemcpyHostToDevice, c->stream));
    P2A_HIP(hipMemcpyAsync(c->cn_env.p, e.data(), nenv * sizeof(int), hipMemcpyHostToDevice, c->stream));
    if ((rc = upload_pbc(c, box9))) return rc;
    launch_cn_rows(c->stream, c->natoms, na, c->cn_rows.p, nenv, c->cn_env.p, c->spec.pbc ? 1 : 0, c->pbc_stage,
                   c->spec.sw, pos_dev, rows_dev);
    // the host vectors are read by the copies above before they return
    P2A_HIP(hipStreamSynchronize(c->stream));
    return launch_check("coordination numbers");
  }
  if ((rc = prepare_cluster_list(c, step, box9, pos_dev))) return rc;
  return run_rows(c, box9, pos_dev, rows_dev, weights_dev, vjp_dev, virial_dev);
}

int p2a_coordination_numbers_device(void* stream, const p2a_switch* sw, const double* box9, int use_pbc,
                                    int64_t natoms, int64_t nrows, const int* rows_dev, int64_t nenv,
                                    const int* env_dev, const double* pos_dev, double* cn_dev) {
  if (!sw) return fail(P2A_ERR_ARG, "null argument");
  if (natoms < 0 || nrows < 0 || nenv < 0 || natoms > INT32_MAX || nrows > INT32_MAX || nenv > INT32_MAX)
    return fail(P2A_ERR_ARG, "sizes must lie in [0, 2^31)");
  // no rows: nothing to write (an empty output may have a null address)
  if (nrows == 0) return P2A_OK;
  if (!pos_dev || !cn_dev || !rows_dev || (nenv > 0 && !env_dev)) return fail(P2A_ERR_ARG, "null argument");
  if (use_pbc && !box9) return fail(P2A_ERR_ARG, "box is required with periodic boundaries");
  PbcArg P;
  std::memset(&P, 0, sizeof(P));
  if (use_pbc) {
    PbcHost h;
    pbc_setup(box9, h);
    fill_pbc_arg(h, P);
  }
  launch_cn_rows((hipStream_t)stream, (int)natoms, (int)nrows, rows_dev, (int)nenv, env_dev, use_pbc ? 1 : 0, P, *sw,
                 pos_dev, cn_dev);
  return launch_check("coordination numbers");
}

}  // extern "C"
