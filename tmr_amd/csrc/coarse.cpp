// Plan and set-up of the coarsest level's direct solve (kernels in
// dense.hip).  Every independent component of the coarsest level is either
// one dense block with an explicit inverse, or is substructured: its node
// graph is bisected by coordinates into leaves D_i and one separator S, and
// the solve goes through D_i^-1, W_i = D_i^-1 E_i and the inverse of the
// Schur complement of S:
//   t_i = D_i^-1 b_i,  g = b_s - sum_i W_i^T b_i,  x_s = S^-1 g,
//   x_i = t_i - W_i x_s.
// An explicit inverse costs n^2 words per solve and n^3 work per set-up; the
// parts of a 9,441-dof level hold a sixth of the words.
#include <algorithm>
#include <cmath>
#include <cstring>

#include "problem.h"

namespace tmrx {

#define HIPCHK(x)                                                       \
  do {                                                                  \
    hipError_t e_ = (x);                                                \
    if (e_ == hipSuccess) e_ = take_launch_error();                     \
    if (e_ != hipSuccess) {                                             \
      last_error = std::string("HIP error: ") + hipGetErrorString(e_) + \
                   " at " + #x;                                         \
      return -1;                                                        \
    }                                                                   \
  } while (0)

namespace {

// Components from this many dofs are substructured: below it one launch
// over the explicit inverse (1,974 dofs: 15.6 MB in FP32, 7 us) beats three
// launches over the parts.
constexpr int SCHUR_MIN = 2048;
constexpr int DB = 64;

int padded(int n) { return (n + DB - 1) / DB * DB; }

struct Partition {
  std::vector<std::vector<int>> leaves;  // nodes
  std::vector<int> sep;
};

// Vertex bisection: the nodes up to the median coordinate of the longest
// axis against the rest, and as separator those of the first part next to
// the second.  Recursion to `depth`; every separator goes to part.sep.
void bisect(std::vector<int> nodes, int depth, const std::vector<double> &X,
            const std::vector<int> &ptr, const std::vector<int> &col, std::vector<int> &side,
            int &stamp, Partition &part) {
  if (depth == 0 || nodes.size() < 2) {
    if (!nodes.empty()) part.leaves.push_back(std::move(nodes));
    return;
  }
  double lo[3], hi[3];
  for (int d = 0; d < 3; d++) lo[d] = hi[d] = X[3 * (size_t)nodes[0] + d];
  for (int i : nodes)
    for (int d = 0; d < 3; d++) {
      lo[d] = std::min(lo[d], X[3 * (size_t)i + d]);
      hi[d] = std::max(hi[d], X[3 * (size_t)i + d]);
    }
  int ax = 0;
  for (int d = 1; d < 3; d++)
    if (hi[d] - lo[d] > hi[ax] - lo[ax]) ax = d;
  std::vector<double> c;
  for (int i : nodes) c.push_back(X[3 * (size_t)i + ax]);
  std::nth_element(c.begin(), c.begin() + c.size() / 2, c.end());
  const double cut = c[c.size() / 2];
  std::vector<int> a, b, s;
  const int sb = ++stamp;  // marks the second part
  for (int i : nodes)
    if (X[3 * (size_t)i + ax] > cut) {
      b.push_back(i);
      side[i] = sb;
    }
  for (int i : nodes) {
    if (X[3 * (size_t)i + ax] > cut) continue;
    bool edge = false;
    for (int q = ptr[i]; q < ptr[i + 1] && !edge; q++) edge = side[col[q]] == sb;
    (edge ? s : a).push_back(i);
  }
  if (a.empty() || b.empty()) {
    part.leaves.push_back(std::move(nodes));
    return;
  }
  part.sep.insert(part.sep.end(), s.begin(), s.end());
  bisect(std::move(a), depth - 1, X, ptr, col, side, stamp, part);
  bisect(std::move(b), depth - 1, X, ptr, col, side, stamp, part);
}

}  // namespace

int Problem::build_coarse_plan() {
  const int last = (int)levels_.size() - 1;
  Level &L = levels_[last];
  if (!L.has_bsr && build_bsr(last)) return -1;
  const std::vector<int> &ptr = L.bsr_ptr_h, &col = L.bsr_col_h;
  const int n = (int)L.ndof, nn = L.n_nodes;
  CoarsePlan &cp = cplan_;
  // node coordinates (the nodes' numbers where a forest has none)
  std::vector<double> X(3 * (size_t)nn, 0.0);
  {
    const std::vector<double> &P = L.forest->points();
    const size_t nd = (size_t)L.forest->num_dep_nodes();
    for (int i = 0; i < nn; i++) {
      if (P.size() >= 3 * (nd + (size_t)nn))
        for (int d = 0; d < 3; d++) X[3 * (size_t)i + d] = P[3 * (nd + (size_t)i) + d];
      else
        X[3 * (size_t)i] = i;
    }
  }
  struct Comp {
    int sg;
    Partition part;
  };
  std::vector<Comp> schur;
  std::vector<int> direct;
  std::vector<int> side(nn, 0);
  int stamp = 0;
  for (int sg = 0; sg < nseg_; sg++) {
    const int n0 = L.seg_node0[sg], n1 = L.seg_node0[sg + 1];
    const int64_t m = 3 * (int64_t)(n1 - n0);
    if (m == 0) continue;
    if (m < SCHUR_MIN) {
      direct.push_back(sg);
      continue;
    }
    std::vector<int> all(n1 - n0);
    for (int i = n0; i < n1; i++) all[i - n0] = i;
    // the depth of least time: what the solves of one set-up read (about 25
    // V-cycles) at 4 TB/s, the inversion steps at 20 us and 52 ns a block (of
    // the lower triangle, over a matrix's own steps) and the products with the
    // couplings at 10 ns a block product, zero ones counted.  Set-up in ms at
    // depths 2 to 5 (the rest of it included): 4,131 dofs 1.50, 1.26, 1.45,
    // 2.27; 9,441 dofs 7.9, 5.9, 7.1, 11.4; 13,923 dofs 16.4, 6.1, 7.3, 13.7;
    // 35,067 dofs 226, 68, 52, 118.  The model takes depths 3, 3, 3 and 4.
    auto blocks = [](int64_t d) { return (double)(padded((int)d) / DB); };
    auto inverse_s = [&](int64_t d) {
      const double nb = blocks(d);
      return 0.5 * nb * (nb + 1.0) * nb * 52e-9;
    };
    auto steps_s = [&](int64_t largest) { return blocks(largest) * 20e-6; };
    const double word_s = 25.0 * 8.0 / 4e12;
    double best = word_s * (double)m * (double)m + inverse_s(m) + steps_s(m);
    Partition keep;
    for (int depth = 1; depth <= 8 && (m >> depth) >= DB; depth++) {
      Partition p;
      bisect(all, depth, X, ptr, col, side, stamp, p);
      std::vector<int> leaf_of(n1 - n0, -1);
      for (size_t k = 0; k < p.leaves.size(); k++)
        for (int i : p.leaves[k]) leaf_of[i - n0] = (int)k;
      std::vector<int64_t> nb(p.leaves.size(), 0);
      for (int i : p.sep) {
        std::vector<int> seen;
        for (int q = ptr[i]; q < ptr[i + 1]; q++) {
          const int k = leaf_of[col[q] - n0];
          if (k >= 0 && std::find(seen.begin(), seen.end(), k) == seen.end()) {
            seen.push_back(k);
            nb[k] += 3;
          }
        }
      }
      const int64_t ms = 3 * (int64_t)p.sep.size();
      double words = (double)ms * (double)ms, s = inverse_s(ms) + steps_s(ms);
      int64_t nmax = 0;
      for (size_t k = 0; k < p.leaves.size(); k++) {
        const int64_t ni = 3 * (int64_t)p.leaves[k].size();
        words += (double)ni * (double)(ni + 2 * nb[k]);
        s += inverse_s(ni) + blocks(nb[k]) * blocks(ni) * (blocks(ni) + blocks(nb[k])) * 10e-9;
        nmax = std::max(nmax, ni);
      }
      s += steps_s(nmax) + word_s * words;
      if (s < best) {
        best = s;
        keep = std::move(p);
      }
    }
    if (keep.sep.empty())
      direct.push_back(sg);
    else
      schur.push_back({sg, std::move(keep)});
  }
  // Dense matrices of the first inversion (whole components and leaves) and
  // of the second (Schur complements), largest first: a step works on the
  // matrices that still have a block for it, a prefix of the list.
  struct Mat {
    int n;
    int64_t off;
    int comp, leaf;  // leaf -1: whole component (comp an index into direct)
  };
  std::vector<Mat> set[2];
  for (size_t k = 0; k < direct.size(); k++)
    set[0].push_back({3 * (L.seg_node0[direct[k] + 1] - L.seg_node0[direct[k]]), 0, (int)k, -1});
  for (size_t c = 0; c < schur.size(); c++) {
    for (size_t k = 0; k < schur[c].part.leaves.size(); k++)
      set[0].push_back({3 * (int)schur[c].part.leaves[k].size(), 0, (int)c, (int)k});
    set[1].push_back({3 * (int)schur[c].part.sep.size(), 0, (int)c, 0});
  }
  int64_t na = 0;
  for (int s = 0; s < 2; s++) {
    std::stable_sort(set[s].begin(), set[s].end(), [](const Mat &a, const Mat &b) { return a.n > b.n; });
    CoarseSet &cs = cp.set[s];
    std::vector<GJProb> pr;
    std::vector<int> tile0{0};
    for (Mat &m : set[s]) {
      const int nb = padded(m.n) / DB;
      m.off = na;
      pr.push_back({m.n, nb, na});
      na += (int64_t)padded(m.n) * padded(m.n);
      tile0.push_back(tile0.back() + nb * (nb + 1) / 2);
    }
    cs.nprob = (int)pr.size();
    cs.active.clear();
    cs.tiles.clear();
    for (int k = 0; !pr.empty() && k < pr[0].nblk; k++) {
      int a = 0;
      while (a < cs.nprob && pr[a].nblk > k) a++;
      cs.active.push_back(a);
      cs.tiles.push_back(tile0[a]);
    }
    if (pr.empty()) pr.push_back({0, 0, 0});
    if (cs.prob.upload(reinterpret_cast<const char *>(pr.data()), pr.size() * sizeof(GJProb)) ||
        cs.tile0.upload(tile0) || cs.fac.alloc((size_t)4 * DB * DB * std::max(1, cs.nprob))) {
      last_error = "coarse: device allocation failed";
      return -1;
    }
  }
  // where every node sits: kind 0 whole component, 1 leaf, 2 separator;
  // matrix (offset, leading dimension, local index)
  std::vector<int8_t> kind(nn, 0);
  std::vector<int> local(nn, 0), comp(nn, 0), leaf(nn, -1);
  std::vector<int64_t> moff(nn, 0);
  std::vector<int> mld(nn, 0);
  auto place = [&](int i, int kd, int c, int lf, int loc, const Mat &m) {
    kind[i] = (int8_t)kd;
    comp[i] = c;
    leaf[i] = lf;
    local[i] = loc;
    moff[i] = m.off;
    mld[i] = padded(m.n);
  };
  for (const Mat &m : set[0]) {
    if (m.leaf < 0) {
      const int n0 = L.seg_node0[direct[m.comp]], n1 = L.seg_node0[direct[m.comp] + 1];
      for (int i = n0; i < n1; i++) place(i, 0, m.comp, -1, i - n0, m);
    } else {
      const auto &nodes = schur[m.comp].part.leaves[m.leaf];
      for (size_t k = 0; k < nodes.size(); k++) place(nodes[k], 1, m.comp, m.leaf, (int)k, m);
    }
  }
  for (const Mat &m : set[1]) {
    const auto &nodes = schur[m.comp].part.sep;
    for (size_t k = 0; k < nodes.size(); k++) place(nodes[k], 2, m.comp, -1, (int)k, m);
  }
  // separator nodes next to each leaf, couplings, products
  struct Leaf {
    std::vector<int> bnd;  // separator nodes, in separator order
    std::vector<int> loc;  // [separator node] -> place in bnd
    int np, mq;
    int64_t et, wt, c;
    const Mat *m;
  };
  std::vector<std::vector<Leaf>> leaves(schur.size());
  int64_t net = 0, nw = 0, nc = 0;
  std::vector<GemmProb> g1, g2;
  std::vector<int> t1{0}, t2{0};
  for (size_t c = 0; c < schur.size(); c++) leaves[c].resize(schur[c].part.leaves.size());
  for (const Mat &m : set[0]) {
    if (m.leaf < 0) continue;
    Leaf &lf = leaves[m.comp][m.leaf];
    const Partition &p = schur[m.comp].part;
    lf.m = &m;
    lf.loc.assign(p.sep.size(), -1);
    for (size_t k = 0; k < p.sep.size(); k++) {
      const int i = p.sep[k];
      for (int q = ptr[i]; q < ptr[i + 1]; q++)
        if (kind[col[q]] == 1 && comp[col[q]] == m.comp && leaf[col[q]] == m.leaf) {
          lf.loc[k] = (int)lf.bnd.size();
          lf.bnd.push_back((int)k);
          break;
        }
    }
    lf.np = padded(m.n);
    lf.mq = padded(3 * (int)lf.bnd.size());
    lf.et = net;
    lf.wt = nw;
    net += (int64_t)lf.np * lf.mq;
    nw += (int64_t)lf.np * lf.mq;
    lf.c = nc;
    nc += (int64_t)lf.mq * lf.mq;
  }
  for (auto &lv : leaves)
    for (Leaf &lf : lv) {
      if (lf.mq == 0) continue;
      // W^T = E^T D^-1 (and W), C = E^T W
      g1.push_back({lf.mq, lf.np, lf.np, lf.et, lf.m->off, lf.wt, lf.wt});
      t1.push_back(t1.back() + lf.mq / DB * (lf.np / DB));
      g2.push_back({lf.mq, lf.mq, lf.np, lf.et, lf.wt, lf.c, -1});
      t2.push_back(t2.back() + lf.mq / DB * (lf.mq / DB));
    }
  // where every block of the level's matrix goes
  std::vector<uint8_t> which(L.nnzb, 255);
  std::vector<int64_t> dst(L.nnzb, 0);
  std::vector<int> ld(L.nnzb, 0);
  for (int i = 0; i < nn; i++)
    for (int q = ptr[i]; q < ptr[i + 1]; q++) {
      const int j = col[q];
      if (kind[i] == 2 && kind[j] == 1) {  // E^T
        const Leaf &lf = leaves[comp[j]][leaf[j]];
        which[q] = 2;
        dst[q] = lf.et + 3 * (int64_t)lf.loc[local[i]] * lf.np + 3 * local[j];
        ld[q] = lf.np;
      } else if (kind[i] == kind[j]) {  // inside a matrix (leaves do not touch)
        which[q] = (mld[i] / DB) & 1;
        dst[q] = moff[i] + 3 * (int64_t)local[i] * mld[i] + 3 * local[j];
        ld[q] = mld[i];
      }
    }
  // rows of the solve
  std::vector<int> col0(n, 0), nb(n, 0), idx;
  std::vector<int64_t> aoff(n, 0);
  bool any_direct = false;
  for (int i = 0; i < nn; i++) {
    if (kind[i] != 0) continue;
    any_direct = true;
    const int n0 = L.seg_node0[direct[comp[i]]], n1 = L.seg_node0[direct[comp[i]] + 1];
    for (int d = 0; d < 3; d++) {
      col0[3 * i + d] = 3 * n0;
      nb[3 * i + d] = 3 * (n1 - n0);
      aoff[3 * i + d] = moff[i] + (3 * (int64_t)local[i] + d) * mld[i];
    }
  }
  std::vector<CoarseRow> rows[3];
  std::vector<CoarseSeg> segs;
  const int64_t wt0 = na, w0 = na + nw;  // W^T and W follow the inverses
  int ntmp = 0, nxs = 0;
  std::vector<std::vector<int>> lidx(schur.size()), bidx(schur.size());
  std::vector<int> xs0(schur.size()), sidx(schur.size());
  for (size_t c = 0; c < schur.size(); c++) {
    const Partition &p = schur[c].part;
    xs0[c] = nxs;
    nxs += 3 * (int)p.sep.size();
    for (size_t k = 0; k < p.leaves.size(); k++) {
      lidx[c].push_back((int)idx.size());  // dofs of the leaf
      for (int i : p.leaves[k])
        for (int d = 0; d < 3; d++) idx.push_back(3 * i + d);
      bidx[c].push_back((int)idx.size());  // separator unknowns next to it
      for (int s : leaves[c][k].bnd)
        for (int d = 0; d < 3; d++) idx.push_back(xs0[c] + 3 * s + d);
    }
  }
  for (size_t c = 0; c < schur.size(); c++) {
    const Partition &p = schur[c].part;
    for (size_t k = 0; k < p.leaves.size(); k++) {
      const Leaf &lf = leaves[c][k];
      const int ni = 3 * (int)p.leaves[k].size();
      for (int r = 0; r < ni; r++) {
        const int s0 = (int)segs.size();
        segs.push_back({lf.m->off + (int64_t)r * lf.np, ni, lidx[c][k]});
        rows[0].push_back({s0, s0 + 1, -1, ntmp});
        const int dof = 3 * p.leaves[k][r / 3] + r % 3, s1 = (int)segs.size();
        if (!lf.bnd.empty())
          segs.push_back({w0 + lf.wt + (int64_t)r * lf.mq, 3 * (int)lf.bnd.size(), bidx[c][k]});
        rows[2].push_back({s1, (int)segs.size(), dof, ntmp});
        ntmp++;
      }
    }
    const int g0 = ntmp, m = 3 * (int)p.sep.size();
    sidx[c] = (int)idx.size();
    for (int r = 0; r < m; r++) idx.push_back(g0 + r);
    const Mat *S = nullptr;
    for (const Mat &mm : set[1])
      if (mm.comp == (int)c) S = &mm;
    for (int r = 0; r < m; r++) {
      const int dof = 3 * p.sep[r / 3] + r % 3, s0 = (int)segs.size();
      for (size_t k = 0; k < p.leaves.size(); k++) {
        const Leaf &lf = leaves[c][k];
        const int lo = lf.loc[r / 3];
        if (lo >= 0)
          segs.push_back({wt0 + lf.wt + (int64_t)(3 * lo + r % 3) * lf.np,
                          3 * (int)p.leaves[k].size(), lidx[c][k]});
      }
      rows[0].push_back({s0, (int)segs.size(), dof, ntmp});
      const int s1 = (int)segs.size();
      segs.push_back({S->off + (int64_t)r * padded(S->n), m, sidx[c]});
      rows[1].push_back({s1, s1 + 1, dof, xs0[c] + r});
      ntmp++;
    }
  }
  // the sums over leaves of the Schur complements
  cp.schur.clear();
  std::vector<int> loc;
  std::vector<int64_t> coff;
  std::vector<int> ldc;
  for (size_t c = 0; c < schur.size(); c++) {
    const Mat *S = nullptr;
    for (const Mat &mm : set[1])
      if (mm.comp == (int)c) S = &mm;
    CoarsePlan::Sum sm;
    sm.m = S->n;
    sm.ld = padded(S->n);
    sm.buf = (padded(S->n) / DB) & 1;
    sm.off = S->off;
    sm.nleaf = (int)leaves[c].size();
    sm.loc0 = loc.size();
    sm.leaf0 = coff.size();
    for (const Leaf &lf : leaves[c]) {
      loc.insert(loc.end(), lf.loc.begin(), lf.loc.end());
      coff.push_back(lf.c);
      ldc.push_back(lf.mq);
    }
    cp.schur.push_back(sm);
  }
  auto up = [](DevArray<char> &d, const void *p, size_t bytes) {
    const char z[8] = {0};
    return bytes ? d.upload(static_cast<const char *>(p), bytes) : d.upload(z, 8);
  };
  if (loc.empty()) loc.push_back(0);
  if (coff.empty()) coff.push_back(0);
  if (ldc.empty()) ldc.push_back(0);
  if (idx.empty()) idx.push_back(0);
  cp.na = na;
  cp.nw = nw;
  cp.ng1 = (int)g1.size();
  cp.nt1 = t1.back();
  cp.nt2 = t2.back();
  cp.any_direct = any_direct;
  cp.any_schur = !schur.empty();
  if (up(cp.g1, g1.data(), g1.size() * sizeof(GemmProb)) ||
      up(cp.g2, g2.data(), g2.size() * sizeof(GemmProb)) || cp.t1.upload(t1) || cp.t2.upload(t2) ||
      up(cp.segs, segs.data(), segs.size() * sizeof(CoarseSeg)) ||
      up(cp.rows[0], rows[0].data(), rows[0].size() * sizeof(CoarseRow)) ||
      up(cp.rows[1], rows[1].data(), rows[1].size() * sizeof(CoarseRow)) ||
      up(cp.rows[2], rows[2].data(), rows[2].size() * sizeof(CoarseRow)) || cp.idx.upload(idx) ||
      cp.loc.upload(loc) || cp.coff.upload(coff) || cp.ldc.upload(ldc) || cp.which.upload(which) ||
      cp.dst.upload(dst) || cp.ld.upload(ld) || cb_col0_.upload(col0) || cb_nb_.upload(nb) ||
      cb_aoff_.upload(aoff) || Ainv_.alloc((size_t)(na + 2 * nw)) || cp.A1.alloc((size_t)na) ||
      cp.Et.alloc((size_t)net) || cp.C.alloc((size_t)nc) || (chk_.n == 0 && chk_.alloc(1))) {
    last_error = "coarse: device allocation failed";
    return -1;
  }
  cp.net = net;
  coarse_.n = n;
  for (int s = 0; s < 3; s++) {
    coarse_.nrow[s] = (int)rows[s].size();
    coarse_.row[s] = reinterpret_cast<const CoarseRow *>(cp.rows[s].p);
  }
  coarse_.seg = reinterpret_cast<const CoarseSeg *>(cp.segs.p);
  coarse_.idx = cp.idx.p;
  coarse_.ntmp = ntmp;
  coarse_.nxs = nxs;
  coarse_.direct = any_direct;
  coarse_.col0 = cb_col0_.p;
  coarse_.nb = cb_nb_.p;
  coarse_.aoff = cb_aoff_.p;
  cp.built = true;
  gen_++;
  return 0;
}

// work vectors of the substructured solve for nrhs right-hand sides
int Problem::ensure_coarse_work(int nrhs) {
  const size_t need = (size_t)nrhs * (size_t)(coarse_.ntmp + coarse_.nxs);
  if (need > 0 && cplan_.work.n < need) {
    if (cplan_.work.alloc(need)) {
      last_error = "coarse: device allocation failed";
      return -1;
    }
    gen_++;
  }
  coarse_.tmp = cplan_.work.p;
  coarse_.xs = cplan_.work.p + (size_t)nrhs * (size_t)coarse_.ntmp;
  return 0;
}

// K of the coarsest level (identity rows and columns on clamped dofs) as a
// BSR matrix assembled on the device from its element matrices (K_E of the
// Galerkin product, or the scaled element stiffness), scattered into the
// plan's dense matrices and inverted
int Problem::coarse_factor() {
  const int last = (int)levels_.size() - 1;
  Level &L = levels_[last];
  const bool nodal = design_mode_ == 1;
  const bool gal = galerkin_ && levels_.size() > 1;
  CoarsePlan &cp = cplan_;
  if (!cp.built && build_coarse_plan()) return -1;
  if (ensure_coarse_work(std::max(1, batch_cap_))) return -1;
  if (!gal) {
    if ((L.KE.n < 576 * (size_t)L.n_elem && L.KE.alloc(576 * (size_t)L.n_elem)) ||
        (nodal && Kgd_.n == 0 && Kgd_.upload(Kgh_))) {
      last_error = "coarse: device allocation failed";
      return -1;
    }
    launch_elem_matrices(L.n_elem, L.d_cls.p, nodal ? L.sg64.p : L.s64.p,
                         nodal ? Kgd_.p : K0d_.p, nodal, L.KE.p, st_);
  }
  launch_bsr_assemble(bsr<double>(last), L.bt_ptr.p, L.bt_code.p, L.bt_w.p, L.bsr_row.p, L.KE.p,
                      L.bsr64.p, st_);
  double *A0 = Ainv_.p, *A1 = cp.A1.p, *Wt = Ainv_.p + cp.na, *W = Wt + cp.nw;
  launch_fill<int>(1, 0, chk_.p, st_);
  launch_fill<double>(cp.na, 0.0, A0, st_);
  launch_fill<double>(cp.na, 0.0, A1, st_);
  launch_fill<double>(cp.net, 0.0, cp.Et.p, st_);
  launch_coarse_scatter(L.nnzb, L.bsr64.p, cp.which.p, cp.dst.p, cp.ld.p, A0, A1, cp.Et.p, st_);
  auto invert = [&](CoarseSet &cs) {
    launch_gj_inverse(reinterpret_cast<const GJProb *>(cs.prob.p), cs.tile0.p, cs.nprob,
                      cs.active.data(), cs.tiles.data(), (int)cs.active.size(), A0, A1, cs.fac.p,
                      chk_.p, st_);
  };
  invert(cp.set[0]);
  if (cp.any_schur) {
    launch_gemm_nt(cp.ng1, cp.nt1, reinterpret_cast<const GemmProb *>(cp.g1.p), cp.t1.p, cp.Et.p,
                   A0, Wt, W, st_);
    launch_gemm_nt(cp.ng1, cp.nt2, reinterpret_cast<const GemmProb *>(cp.g2.p), cp.t2.p, cp.Et.p,
                   Wt, cp.C.p, nullptr, st_);
    for (const auto &s : cp.schur)
      launch_schur_sum(s.m, s.ld, s.nleaf, cp.loc.p + s.loc0, cp.coff.p + s.leaf0,
                       cp.ldc.p + s.leaf0, cp.C.p, (s.buf ? A1 : A0) + s.off, st_);
    invert(cp.set[1]);
  }
  int bad = 0;
  HIPCHK(hipMemcpyAsync(&bad, chk_.p, sizeof(int), hipMemcpyDeviceToHost, st_));
  HIPCHK(hipStreamSynchronize(st_));
  if (bad) {
    last_error = "coarse solve: the coarsest-level matrix is not positive definite "
                 "(missing boundary conditions?)";
    return -1;
  }
  coarse_.Ainv = Ainv_.p;
  // FP32 V-cycles read an FP32 copy (half the bytes of every coarse solve)
  coarse_.Ainv32 = nullptr;
  if (setup_prec_pending_ == 1) {
    const size_t words = (size_t)(cp.na + 2 * cp.nw);
    if (Ainv32_.n < words) {
      if (Ainv32_.alloc(words)) {
        last_error = "coarse: device allocation failed";
        return -1;
      }
      gen_++;
    }
    launch_convert<double, float>((int64_t)words, Ainv_.p, Ainv32_.p, st_);
    coarse_.Ainv32 = Ainv32_.p;
  }
  return 0;
}

}  // namespace tmrx
