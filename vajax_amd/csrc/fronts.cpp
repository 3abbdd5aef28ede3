// Front program of the sparse LU on the host: singletons, elimination tree,
// amalgamation, assembly maps, stages, and the CPU execution that the GPU
// kernels (fronts.hip) match bit for bit.
#include "fronts.h"

#include "symbolic.h"

#include <algorithm>
#include <cmath>

namespace vjx {

void find_singletons(int n, const int32_t* indptr, const int32_t* indices, const double* vals,
                     double pivot_tol, Singletons& out) {
  out = Singletons();
  std::vector<int32_t> ccount(n, 0), crow(n, -1);
  std::vector<double> cmax(n, 0.0);
  for (int r = 0; r < n; ++r)
    for (int e = indptr[r]; e < indptr[r + 1]; ++e) {
      ++ccount[indices[e]];
      crow[indices[e]] = r;
    }
  std::vector<char> row_used(n, 0), col_used(n, 0);
  // columns with one entry: no L entry, so no fill
  for (int c = 0; c < n; ++c) {
    if (ccount[c] != 1) continue;
    const int r = crow[c];
    if (row_used[r] || indptr[r + 1] - indptr[r] == 1) continue;
    row_used[r] = 1;
    col_used[c] = 1;
    out.sc.push_back(c);
    out.sr.push_back(r);
  }
  // rows with one entry: no U entry.  The pivot must pass the threshold test
  // of its column, as the pivots chosen by the factorisation do.
  for (int r = 0; r < n; ++r)
    if (!row_used[r])
      for (int e = indptr[r]; e < indptr[r + 1]; ++e)
        cmax[indices[e]] = std::max(cmax[indices[e]], std::fabs(vals[e]));
  for (int r = 0; r < n; ++r) {
    if (indptr[r + 1] - indptr[r] != 1 || row_used[r]) continue;
    const int c = indices[indptr[r]];
    const double a = std::fabs(vals[indptr[r]]);
    if (col_used[c] || !(a > 0.0) || !(a >= pivot_tol * cmax[c])) continue;
    row_used[r] = 1;
    col_used[c] = 1;
    out.rc.push_back(c);
    out.rr.push_back(r);
  }
}

namespace {

// Time of one front on one wavefront (us), the amalgamation's and the stages'
// yardstick: assembly and hand-over, a dependent chain per pivot, and the
// update blocks moved.
double front_cost(int k, int s) { return 0.9 + 0.13 * k + 0.01 * (double)s * s / 64.0; }

struct Tree {
  std::vector<int32_t> piv;   // pivots, in elimination order
  std::vector<int32_t> kids;  // fronts by id
  int top = -1;               // last pivot, whose structure is the front's
  double below = 0.0;         // time of the slowest chain below
  double time = 0.0;          // ... and through this front
  bool gone = false;          // merged into its parent
};

}  // namespace

bool plan_fronts(int n, int n_single, const std::vector<int64_t>& lptr,
                 const std::vector<int32_t>& lidx, const std::vector<int64_t>& uptr,
                 const std::vector<int32_t>& uidx, FrontPlan& plan, std::vector<int32_t>& np) {
  plan.ok = false;
  // U by rows (later columns of every pivot row)
  std::vector<int32_t> rcnt(n + 1, 0);
  for (int j = n_single; j < n; ++j)
    for (int64_t e = uptr[j]; e < uptr[j + 1]; ++e)
      if (uidx[e] != j) ++rcnt[uidx[e] + 1];
  for (int i = 0; i < n; ++i) rcnt[i + 1] += rcnt[i];
  std::vector<int32_t> rcol(rcnt[n]);
  {
    std::vector<int32_t> fill(rcnt.begin(), rcnt.end() - 1);
    for (int j = n_single; j < n; ++j)
      for (int64_t e = uptr[j]; e < uptr[j + 1]; ++e)
        if (uidx[e] != j) rcol[fill[uidx[e]]++] = j;
  }
  // symmetric structure of every pivot, closed under elimination
  std::vector<std::vector<int32_t>> st(n);
  std::vector<int32_t> head(n, -1), next(n, -1), stamp(n, -1);
  int64_t lu_nnz = (int64_t)(lidx.size() + uidx.size()), sym_nnz = 0;
  std::vector<std::vector<int32_t>> kids_of(n);
  for (int k = n_single; k < n; ++k) {
    auto& s = st[k];
    stamp[k] = k;
    auto add = [&](int i) {
      if (i > k && stamp[i] != k) {
        stamp[i] = k;
        s.push_back(i);
      }
    };
    for (int64_t e = lptr[k]; e < lptr[k + 1]; ++e) add(lidx[e]);
    for (int e = rcnt[k]; e < rcnt[k + 1]; ++e) add(rcol[e]);
    for (int c : kids_of[k])
      for (int i : st[c]) add(i);
    if ((int)s.size() >= kFrontMax) return false;
    std::sort(s.begin(), s.end());
    if (!s.empty()) kids_of[s.front()].push_back(k);
    sym_nnz += 2 * (int64_t)s.size() + 1;
  }
  if (sym_nnz > 2 * lu_nnz + 64) return false;
  // Amalgamation, bottom up: a pivot's front takes in a child front when that
  // does not lengthen the slowest chain through it by more than a fraction of
  // the front saved (a child off the chain lengthens it by its pivots), does
  // not need a larger lane grid for mostly padding, and stays within
  // kFrontMax.  The slowest child is offered first.
  std::vector<Tree> fr(n);
  std::vector<int32_t> front_of(n, -1);
  std::vector<int32_t> kids;
  for (int k = n_single; k < n; ++k) {
    Tree& t = fr[k];
    t.top = k;
    t.piv.assign(1, k);
    t.kids.clear();
    for (int c : kids_of[k]) t.kids.push_back(front_of[c]);
    const int s = (int)st[k].size();
    auto slowest = [&](const std::vector<int32_t>& v, int skip) {
      double m = 0.0;
      for (int f : v)
        if (f != skip) m = std::max(m, fr[f].time);
      return m;
    };
    std::sort(t.kids.begin(), t.kids.end(), [&](int a, int b) {
      return fr[a].time != fr[b].time ? fr[a].time > fr[b].time : a < b;
    });
    kids = t.kids;
    for (int c : kids) {
      const int kc = (int)fr[c].piv.size(), sc = (int)st[fr[c].top].size();
      const int k0 = (int)t.piv.size(), k1 = k0 + kc;
      if (k1 + s > kFrontMax) continue;
      const double before = slowest(t.kids, -1) + front_cost(k0, s);
      const double after = std::max(slowest(t.kids, c), fr[c].below) + front_cost(k1, s);
      const int64_t zeros = (int64_t)kc * (k0 + s - sc);
      const int64_t area = (int64_t)k1 * (k1 + 2 * s);
      if (zeros > 0 && (after > before + 0.35 || 2 * zeros > area + 64)) continue;
      std::vector<int32_t> p = fr[c].piv;
      p.insert(p.end(), t.piv.begin(), t.piv.end());
      t.piv.swap(p);
      t.kids.erase(std::find(t.kids.begin(), t.kids.end(), c));
      t.kids.insert(t.kids.end(), fr[c].kids.begin(), fr[c].kids.end());
      fr[c].gone = true;
      fr[c].kids.clear();
    }
    t.below = slowest(t.kids, -1);
    t.time = t.below + front_cost((int)t.piv.size(), s);
    front_of[k] = k;
  }
  // postorder; children of a front by decreasing time (the slow chain first)
  std::vector<int32_t> roots, order, stack;
  std::vector<char> has_parent(n, 0);
  for (int k = n_single; k < n; ++k)
    if (!fr[k].gone)
      for (int c : fr[k].kids) has_parent[c] = 1;
  for (int k = n_single; k < n; ++k)
    if (!fr[k].gone && !has_parent[k]) roots.push_back(k);
  std::vector<size_t> at(n, 0);
  for (int r : roots) {
    stack.assign(1, r);
    while (!stack.empty()) {
      const int f = stack.back();
      if (at[f] == 0)
        std::sort(fr[f].kids.begin(), fr[f].kids.end(), [&](int a, int b) {
          return fr[a].time != fr[b].time ? fr[a].time > fr[b].time : a < b;
        });
      if (at[f] < fr[f].kids.size()) {
        stack.push_back(fr[f].kids[at[f]++]);
      } else {
        stack.pop_back();
        order.push_back(f);
      }
    }
  }
  np.assign(n, 0);
  for (int k = 0; k < n_single; ++k) np[k] = k;
  int pos = n_single;
  for (int f : order)
    for (int p : fr[f].piv) np[p] = pos++;
  // descriptors
  plan = FrontPlan();
  const int nf = (int)order.size();
  plan.fronts.resize(nf);
  plan.parent.assign(nf, -1);
  plan.rows_below.assign(nf, 0);
  std::vector<int32_t> id(n, -1);
  for (int q = 0; q < nf; ++q) id[order[q]] = q;
  int64_t fac = 0;
  std::vector<int32_t> s_list;
  for (int q = 0; q < nf; ++q) {
    const Tree& t = fr[order[q]];
    FrontDesc& d = plan.fronts[q];
    d = FrontDesc{};
    d.k = (int)t.piv.size();
    const int s = (int)st[t.top].size();
    d.m = d.k + s;
    d.nt = (d.m + 7) / 8;
    d.r0 = np[t.piv.front()];
    d.fac = (int32_t)fac;
    fac += (int64_t)d.k * (d.m + s);
    d.idx = (int32_t)plan.idx.size();
    s_list.clear();
    for (int i : st[t.top]) s_list.push_back(np[i]);
    std::sort(s_list.begin(), s_list.end());
    plan.idx.insert(plan.idx.end(), s_list.begin(), s_list.end());
    plan.rows_below[q] += d.k;
    for (int c : t.kids) plan.parent[id[c]] = q;
  }
  for (int q = 0; q < nf; ++q)
    if (plan.parent[q] >= 0) plan.rows_below[plan.parent[q]] += plan.rows_below[q];
  // Update blocks and solve contributions: the children of a front lie next
  // to each other, so the front reads them as one run.  Its wavefront adds 64
  // consecutive values at a time; a child whose first values would meet an
  // earlier child's on one position within such a group starts on the next.
  std::vector<std::vector<int32_t>> kid(nf);
  for (int q = 0; q < nf; ++q)
    if (plan.parent[q] >= 0) kid[plan.parent[q]].push_back(q);
  int64_t cb = 0, cv = 0;
  std::vector<int32_t> lpos(n, -1);
  std::vector<uint16_t> pp;
  std::vector<int32_t> count;  // children's values so far per position
  for (int q = 0; q < nf; ++q) {
    FrontDesc& d = plan.fronts[q];
    const int ld = front_ld(d.nt), s = d.m - d.k;
    auto local = [&](int row) {
      if (row < d.r0 + d.k) return row - d.r0;
      const int32_t* b = &plan.idx[d.idx];
      return d.k + (int)(std::lower_bound(b, b + s, row) - b);
    };
    d.c0 = (int32_t)cb;
    d.cpos = (int32_t)plan.cpos.size();
    d.v0 = (int32_t)cv;
    d.vtab = (int32_t)plan.vtab.size();
    count.assign((size_t)front_lds(d.nt), 0);
    std::vector<std::vector<uint16_t>> contrib(d.m);
    for (int c : kid[q]) {
      FrontDesc& e = plan.fronts[c];
      const int sc = e.m - e.k;
      std::vector<int32_t> map(sc);
      for (int i = 0; i < sc; ++i) map[i] = local(plan.idx[e.idx + i]);
      pp.clear();
      for (int j = 0; j < sc; ++j)
        for (int i = 0; i < sc; ++i) pp.push_back((uint16_t)(map[i] + map[j] * ld));
      // values so far in the open group of 64
      const size_t have = plan.cpos.size() - d.cpos, open = have % 64;
      bool clash = false;
      for (size_t a = have - open; a < have && !clash; ++a) {
        const uint16_t x = plan.cpos[d.cpos + a];
        for (size_t b = 0; b < std::min(pp.size(), 64 - open) && !clash; ++b)
          clash = x != kNoPos && (x & kPosMask) == pp[b];
      }
      if (clash)
        for (size_t a = open; a < 64; ++a) {
          plan.cpos.push_back(kNoPos);
          ++cb;
        }
      e.cb = (int32_t)cb;
      cb += (int64_t)sc * sc;
      for (uint16_t x : pp) {
        const int nth = count[x]++;
        d.rounds = std::max(d.rounds, std::min(nth, kMaxRounds) + 1);
        plan.cpos.push_back((uint16_t)(x | std::min(nth, kMaxRounds - 1) << kPosBits));
      }
      e.cv = (int32_t)cv;
      for (int i = 0; i < sc; ++i) contrib[map[i]].push_back((uint16_t)(cv - d.v0 + i));
      cv += sc;
    }
    d.nc = (int32_t)(plan.cpos.size() - d.cpos);
    if (cv - d.v0 >= kNoPos) return false;
    size_t depth = 0;
    for (const auto& v : contrib) depth = std::max(depth, v.size());
    d.nv = (int32_t)depth;
    for (size_t c = 0; c < depth; ++c)
      for (int i = 0; i < d.m; ++i)
        plan.vtab.push_back(c < contrib[i].size() ? contrib[i][c] : kNoPos);
  }
  if (fac > INT32_MAX || cb > INT32_MAX) return false;
  plan.n_fac = (int32_t)fac;
  plan.n_cb = (int32_t)cb;
  plan.n_cv = (int32_t)cv;
  plan.ok = true;
  return true;
}

void plan_entries(const std::vector<int32_t>& rows, const std::vector<int32_t>& cols,
                  const std::vector<int32_t>& ids, FrontPlan& plan) {
  const int nf = (int)plan.fronts.size();
  int n = 0;
  for (const auto& d : plan.fronts) n = std::max(n, d.r0 + d.k);
  std::vector<int32_t> owner(n, -1);
  for (int q = 0; q < nf; ++q)
    for (int i = 0; i < plan.fronts[q].k; ++i) owner[plan.fronts[q].r0 + i] = q;
  std::vector<int32_t> cnt(nf + 1, 0);
  for (size_t e = 0; e < ids.size(); ++e) ++cnt[owner[std::min(rows[e], cols[e])] + 1];
  for (int q = 0; q < nf; ++q) {
    plan.fronts[q].a0 = cnt[q];
    plan.fronts[q].na = cnt[q + 1];
    cnt[q + 1] += cnt[q];
  }
  plan.apos.assign(ids.size(), kNoPos);
  plan.asrc.assign(ids.size(), -1);
  for (size_t e = 0; e < ids.size(); ++e) {
    const int q = owner[std::min(rows[e], cols[e])];
    const FrontDesc& d = plan.fronts[q];
    const int32_t* b = plan.idx.data() + d.idx;
    auto local = [&](int row) {
      if (row < d.r0 + d.k) return row - d.r0;
      return d.k + (int)(std::lower_bound(b, b + (d.m - d.k), row) - b);
    };
    const int at = cnt[q]++;
    plan.apos[at] = (uint16_t)(local(rows[e]) + local(cols[e]) * front_ld(d.nt));
    plan.asrc[at] = ids[e];
  }
}

void assemble_program(const std::vector<const FrontPlan*>& plans, const std::vector<int32_t>& kind,
                      const std::vector<int32_t>& row0,
                      const std::vector<std::vector<int32_t>>& entry, int n, FrontProgram& out) {
  out = FrontProgram();
  const int np = (int)plans.size();
  std::vector<int32_t> f0(np), a0(np);
  for (int p = 0; p < np; ++p) {
    const FrontPlan& P = *plans[p];
    f0[p] = (int32_t)out.fronts.size();
    a0[p] = (int32_t)out.apos.size();
    for (FrontDesc d : P.fronts) {
      d.idx += (int32_t)out.idx.size();
      d.a0 += a0[p];
      d.cpos += (int32_t)out.cpos.size();
      d.vtab += (int32_t)out.vtab.size();
      out.fronts.push_back(d);
    }
    out.idx.insert(out.idx.end(), P.idx.begin(), P.idx.end());
    out.apos.insert(out.apos.end(), P.apos.begin(), P.apos.end());
    out.cpos.insert(out.cpos.end(), P.cpos.begin(), P.cpos.end());
    out.vtab.insert(out.vtab.end(), P.vtab.begin(), P.vtab.end());
  }
  // Stages of each plan.  Stage 0: whole subtrees of up to R0 pivots, about
  // two workgroups per compute unit on a large circuit, of fronts that fit
  // the one-wavefront kernel (32 rows).  What remains has fronts of 20 to 64
  // rows, too few at a time to fill the device: by height, a workgroup each.
  int n_blocks = 0, n_fronts = 0, most_nt = 0;  // blocks that have fronts
  for (int32_t k : kind) {
    n_blocks += plans[k]->fronts.empty() ? 0 : 1;
    n_fronts += (int)plans[k]->fronts.size();
    for (const auto& d : plans[k]->fronts) most_nt = std::max(most_nt, d.nt);
  }
  const bool one = n_blocks == 1 && n_fronts <= kTinyFronts && most_nt <= 4;
  const int R0 = one ? n : std::min(384, std::max(48, n / 512));
  struct PlanTasks {
    std::vector<std::vector<std::pair<int32_t, int32_t>>> stage;  // {first level, levels}
    std::vector<int32_t> nt;
  };
  std::vector<PlanTasks> pt(np);
  std::vector<int32_t> uses(np, 0);  // instances of each plan
  for (int32_t k : kind) ++uses[k];
  out.level.assign(1, 0);
  for (int p = 0; p < np; ++p) {
    const FrontPlan& P = *plans[p];
    const int nf = (int)P.fronts.size();
    std::vector<int32_t> stage(nf, -1), root(nf, -1), height(nf, 0);
    std::vector<int32_t> load(nf, 0), big(nf, 0);
    for (int q = 0; q < nf; ++q) big[q] = P.fronts[q].nt > 4;
    for (int q = 0; q < nf; ++q) {
      load[q] += P.fronts[q].k;
      const int a = P.parent[q];
      if (a >= 0) {
        load[a] += load[q];
        big[a] |= big[q];
      }
    }
    for (int q = nf - 1; q >= 0; --q) {
      const int a = P.parent[q];
      const bool whole = a >= 0 && stage[a] == 0;  // inside its parent's piece
      if (!whole && (load[q] > R0 || big[q])) continue;
      stage[q] = 0;
      root[q] = whole ? root[a] : q;
    }
    std::vector<int32_t> below(nf, 0), only(nf, -1);  // children left, and one of them
    for (int q = 0; q < nf; ++q) {
      if (stage[q] != 0) {
        if (below[q] == 1) {  // continues its child's chain
          stage[q] = stage[only[q]];
          root[q] = root[only[q]];
        } else {
          root[q] = q;
          if (stage[q] < 0) stage[q] = 1;
        }
        const int a = P.parent[q];
        if (a >= 0) {
          ++below[a];
          only[a] = q;
          stage[a] = std::max(stage[a], stage[q] + 1);
        }
      }
    }
    int ns = 0;
    for (int q = 0; q < nf; ++q) ns = std::max(ns, stage[q] + 1);
    pt[p].stage.resize(ns);
    pt[p].nt.assign(ns, 1);
    std::vector<std::vector<int32_t>> members(nf);
    for (int q = 0; q < nf; ++q) {
      members[root[q]].push_back(q);
      pt[p].nt[stage[q]] = std::max(pt[p].nt[stage[q]], P.fronts[q].nt);
      const int a = P.parent[q];
      if (a >= 0 && root[a] == root[q]) height[a] = std::max(height[a], height[q] + 1);
    }
    // Tasks.  Stage 0: pieces packed into workgroups, level by level (the
    // pieces' fronts of one height run together), pieces of equal height
    // first.  A task takes pieces up to the stage's share of one of the
    // workgroups that fit the device at a time (four per compute unit),
    // between 8 and 60 us of front time: on the 65k-gate circuit most of the
    // 10 500 pieces are single fronts, and one workgroup each left three of
    // four wavefronts idle (138 us against 41 packed).
    std::vector<double> piece(nf, 0.0);
    std::vector<std::vector<int32_t>> roots(ns);
    std::vector<double> total(ns, 0.0);
    for (int q = 0; q < nf; ++q) {
      const double c = front_cost(P.fronts[q].k, P.fronts[q].m - P.fronts[q].k);
      piece[root[q]] += c;
      total[stage[q]] += c * uses[p];
      if (root[q] == q) roots[stage[q]].push_back(q);
    }
    for (int g = 0; g < ns; ++g) {
      auto& rs = roots[g];
      std::stable_sort(rs.begin(), rs.end(), [&](int a, int b) {
        return height[a] != height[b] ? height[a] > height[b] : piece[a] > piece[b];
      });
      const double share =
          one ? 1e30 : g > 0 ? 0.0 : std::min(60.0, std::max(8.0, total[g] / 1024.0));
      for (size_t i = 0; i < rs.size();) {
        std::vector<int32_t> v;
        double load_us = 0.0;
        do {
          v.insert(v.end(), members[rs[i]].begin(), members[rs[i]].end());
          load_us += piece[rs[i]];
          ++i;
        } while (i < rs.size() && load_us + piece[rs[i]] <= share);
        std::stable_sort(v.begin(), v.end(), [&](int a, int b) {
          if (height[a] != height[b]) return height[a] < height[b];
          const double ca = front_cost(P.fronts[a].k, P.fronts[a].m - P.fronts[a].k);
          const double cb = front_cost(P.fronts[b].k, P.fronts[b].m - P.fronts[b].k);
          return ca > cb;
        });
        const int l0 = (int)out.level.size() - 1;
        for (size_t j = 0; j < v.size(); ++j) {
          out.order.push_back(f0[p] + v[j]);
          if (j + 1 == v.size() || height[v[j + 1]] != height[v[j]])
            out.level.push_back((int32_t)out.order.size());
        }
        pt[p].stage[g].push_back({l0, (int)out.level.size() - 1 - l0});
      }
    }
  }
  // instances
  int64_t fac = 0, cb = 0, cv = 0;
  for (size_t c = 0; c < kind.size(); ++c) {
    const FrontPlan& P = *plans[kind[c]];
    FrontInst I{};
    I.row = row0[c];
    I.fac = (int32_t)fac;
    I.cb = (int32_t)cb;
    I.cv = (int32_t)cv;
    I.asrc = (int32_t)out.asrc.size() - a0[kind[c]];
    fac += P.n_fac;
    cb += P.n_cb;
    cv += P.n_cv;
    for (int32_t e : P.asrc) out.asrc.push_back(entry[c][e]);
    out.inst.push_back(I);
  }
  out.n_fac = (int32_t)fac;
  out.n_cb = (int32_t)cb;
  out.n_cv = (int32_t)cv;
  size_t ns = 0;
  for (const auto& t : pt) ns = std::max(ns, t.stage.size());
  out.stage_task.assign(1, 0);
  for (size_t g = 0; g < ns; ++g) {
    int nt = 1;
    for (size_t c = 0; c < kind.size(); ++c) {
      const PlanTasks& t = pt[kind[c]];
      if (g >= t.stage.size()) continue;
      nt = std::max(nt, t.nt[g]);
      for (const auto& x : t.stage[g])
        for (int32_t v : {(int32_t)c, x.first, x.second, out.level[x.first]}) out.task.push_back(v);
    }
    out.stage_task.push_back((int32_t)(out.task.size() / 4));
    out.stage_nt.push_back(nt);
  }
  out.tiny.total = one && out.task.size() == 4 ? 1 : 0;  // see tiny_layout
}

void tiny_layout(FrontProgram& F, int n_rows) {
  FrontProgram::Tiny t = {};
  if (F.tiny.total == 0) return;
  F.tiny = t;
  t.n_fronts = (int32_t)F.order.size();
  t.n_level = F.task[2] + 1;
  t.n_idx = (int32_t)F.idx.size();
  t.n_vtab = (int32_t)F.vtab.size();
  t.n_a = (int32_t)F.apos.size();
  t.n_c = (int32_t)F.cpos.size();
  t.n_fac = F.n_fac;
  t.n_rows = n_rows;
  t.lds_wave = front_lds(F.stage_nt[0]);
  int64_t at = 0;
  auto take = [&](int64_t bytes) {
    const int64_t p = at;
    at = (at + bytes + 15) & ~(int64_t)15;
    return (int32_t)p;
  };
  t.desc = take((int64_t)t.n_fronts * sizeof(FrontDesc));
  t.level = take(4 * (int64_t)t.n_level);
  t.idx = take(4 * (int64_t)t.n_idx);
  t.vtab = take(2 * (int64_t)t.n_vtab);
  t.apos = take(2 * (int64_t)t.n_a);
  t.cpos = take(2 * (int64_t)t.n_c);
  t.av = take(8 * (int64_t)t.n_a);
  t.fac = take(8 * (int64_t)t.n_fac);
  t.sg = take(8 * (int64_t)F.sg_src.size());
  t.cb = take(8 * (int64_t)F.n_cb);
  t.cv = take(8 * (int64_t)F.n_cv);
  t.y = take(8 * (int64_t)n_rows);
  t.z = take(8 * (int64_t)n_rows);
  t.front = take(8 * (int64_t)t.lds_wave * kTinyWaves);
  // 160 KiB a workgroup, less the kernel's own tables
  if (at > 152 * 1024) return;
  t.total = (int32_t)at;
  F.tiny = t;
}

void front_slot_map(const LuSymbolic& s, std::vector<int32_t>& map) {
  const FrontProgram& F = s.front;
  const int n = s.n;
  map.assign(s.col.size(), -1);
  // owner front of every permuted row, and its instance's bases
  std::vector<int32_t> owner(n, -1), inst(n, -1);
  const int ntask = (int)F.task.size() / 4;
  for (int t = 0; t < ntask; ++t) {
    const int c = F.task[4 * t];
    const int l0 = F.task[4 * t + 1], nl = F.task[4 * t + 2];
    for (int o = F.level[l0]; o < F.level[l0 + nl]; ++o) {
      const FrontDesc& d = F.fronts[F.order[o]];
      for (int i = 0; i < d.k; ++i) {
        owner[F.inst[c].row + d.r0 + i] = F.order[o];
        inst[F.inst[c].row + d.r0 + i] = c;
      }
    }
  }
  // what the singletons hold: {row, kind} -> value
  std::vector<int32_t> cs(n, -1), rs(n, -1);
  for (size_t i = 0; i < F.col_single.size() / 4; ++i) cs[F.col_single[4 * i]] = (int)i;
  for (size_t i = 0; i < F.row_single.size() / 2; ++i) rs[F.row_single[2 * i]] = (int)i;
  auto local = [&](const FrontDesc& d, int row0, int row) {
    const int r = row - row0;
    if (r < d.r0 + d.k) return r - d.r0;
    const int32_t* b = F.idx.data() + d.idx;
    return d.k + (int)(std::lower_bound(b, b + (d.m - d.k), r) - b);
  };
  for (int i = 0; i < n; ++i) {
    int us = cs[i] >= 0 ? F.col_single[4 * cs[i] + 2] : 0;
    int re = owner[i] >= 0 ? F.rs_ptr[i] : 0;
    for (int e = s.rowptr[i]; e < s.rowptr[i + 1]; ++e) {
      const int j = s.col[e];
      if (cs[i] >= 0) {  // a column singleton's row: its pivot and U entries
        map[e] = F.n_fac + (j == i ? F.col_single[4 * cs[i] + 1] : us++);
      } else if (rs[i] >= 0) {
        map[e] = F.n_fac + F.row_single[2 * rs[i] + 1];
      } else if (rs[j] >= 0) {  // L entry in a row singleton's column
        map[e] = F.n_fac + re++;
      } else {
        const int lo = std::min(i, j);
        const FrontDesc& d = F.fronts[owner[lo]];
        const FrontInst& I = F.inst[inst[lo]];
        const int a = local(d, I.row, i), b = local(d, I.row, j);
        map[e] = I.fac + d.fac +
                 (b < d.k ? b * d.m + a : d.k * d.m + (b - d.k) * d.k + a);
      }
    }
  }
}

bool check_fronts(const LuSymbolic& s, std::string& err) {
  const FrontProgram& F = s.front;
  const int n = s.n;
  auto fail = [&](const char* what) {
    err = std::string("front program: ") + what;
    return false;
  };
  std::vector<int32_t> map;
  front_slot_map(s, map);
  std::vector<char> used((size_t)F.storage(), 0);
  for (int32_t m : map) {
    if (m < 0 || (int64_t)m >= F.storage()) return fail("an LU entry has no place");
    if (used[m]) return fail("two LU entries share a place");
    used[m] = 1;
  }
  // every matrix entry is read once, by a front or as a singleton's value
  std::vector<int32_t> seen(s.nnz_a, 0);
  for (int32_t e : F.asrc) {
    if (e < 0 || e >= s.nnz_a) return fail("matrix entry out of range");
    ++seen[e];
  }
  for (int32_t e : F.sg_src) {
    if (e < 0 || e >= s.nnz_a) return fail("singleton entry out of range");
    ++seen[e];
  }
  for (int32_t c : seen)
    if (c != 1) return fail("a matrix entry is not read exactly once");
  // walk the tasks: every front once per instance, after its children, whose
  // rows it holds; children in the same task at a lower level
  const int ntask = (int)F.task.size() / 4;
  std::vector<int32_t> row_stage(n, -1), row_task(n, -1), row_level(n, -1);
  for (size_t g = 0; g + 1 < F.stage_task.size(); ++g)
    for (int t = F.stage_task[g]; t < F.stage_task[g + 1]; ++t) {
      const FrontInst& I = F.inst[F.task[4 * t]];
      const int l0 = F.task[4 * t + 1], nl = F.task[4 * t + 2];
      for (int l = l0; l < l0 + nl; ++l)
        for (int o = F.level[l]; o < F.level[l + 1]; ++o) {
          const FrontDesc& d = F.fronts[F.order[o]];
          if (d.nt > F.stage_nt[g] || d.m > kFrontMax || d.m > 8 * d.nt)
            return fail("front larger than its stage");
          for (int i = 0; i < d.k; ++i) {
            const int r = I.row + d.r0 + i;
            if (r < 0 || r >= n || row_stage[r] >= 0) return fail("row in two fronts");
            row_stage[r] = (int)g;
            row_task[r] = t;
            row_level[r] = l;
          }
          for (int e = 0; e < d.nc; ++e) {
            const int x = F.cpos[d.cpos + e] & kPosMask;
            if (F.cpos[d.cpos + e] != kNoPos && (x % front_ld(d.nt) >= d.m || x / front_ld(d.nt) >= d.m))
              return fail("update position outside the front");
          }
          for (int e = 0; e < d.na; ++e) {
            const int x = F.apos[d.a0 + e];
            if (x % front_ld(d.nt) >= d.m || x / front_ld(d.nt) >= d.m)
              return fail("entry position outside the front");
          }
          // one position per group of 64 values
          for (int b = 0; b < d.nc; b += 64) {
            std::vector<uint16_t> v(F.cpos.begin() + d.cpos + b,
                                    F.cpos.begin() + d.cpos + std::min(d.nc, b + 64));
            v.erase(std::remove(v.begin(), v.end(), kNoPos), v.end());
            for (uint16_t& x : v) x &= kPosMask;
            std::sort(v.begin(), v.end());
            if (std::unique(v.begin(), v.end()) != v.end())
              return fail("a group adds to one position twice");
          }
          // rounds: every position's values numbered in their order
          {
            std::vector<int32_t> seen((size_t)front_lds(d.nt), 0);
            for (int e = 0; e < d.nc; ++e) {
              const uint16_t x = F.cpos[d.cpos + e];
              if (x != kNoPos &&
                  (x >> kPosBits) != std::min(seen[x & kPosMask]++, kMaxRounds - 1))
                return fail("a position's values are misnumbered");
              if (x != kNoPos && (x >> kPosBits) >= d.rounds) return fail("a value past the rounds");
            }
            if (*std::max_element(seen.begin(), seen.end()) > kMaxRounds && d.rounds <= kMaxRounds)
              return fail("more values on a position than rounds");
          }
          if (g > 0 && F.level[l + 1] - F.level[l] != 1) return fail("two fronts in a later stage's level");
          if (d.c0 + (int64_t)d.nc > (int64_t)F.n_cb - I.cb ||
              d.v0 < 0 || d.cv + (d.m - d.k) > F.n_cv - I.cv)
            return fail("update block outside the storage");
        }
    }
  (void)ntask;
  for (size_t i = 0; i < F.col_single.size() / 4; ++i) row_stage[F.col_single[4 * i]] = 1 << 20;
  for (size_t i = 0; i < F.row_single.size() / 2; ++i) row_stage[F.row_single[2 * i]] = 1 << 20;
  for (int r = 0; r < n; ++r)
    if (row_stage[r] < 0) return fail("a row belongs to no front");
  for (int t = 0; t < ntask; ++t) {
    const FrontInst& I = F.inst[F.task[4 * t]];
    const int l0 = F.task[4 * t + 1], nl = F.task[4 * t + 2];
    for (int l = l0; l < l0 + nl; ++l)
      for (int o = F.level[l]; o < F.level[l + 1]; ++o) {
        const FrontDesc& d = F.fronts[F.order[o]];
        const int self = I.row + d.r0;
        for (int i = 0; i < d.m - d.k; ++i) {
          const int r = I.row + F.idx[d.idx + i];
          if (r < self + d.k || r >= n || row_task[r] < 0) return fail("update row before its front");
          const bool later = row_stage[r] > row_stage[self] ||
                             (row_task[r] == row_task[self] && row_level[r] > row_level[self]);
          if (!later) return fail("a front runs before one that updates it");
        }
      }
  }
  return true;
}

template <typename T>
void fronts_refactor_host(const LuSymbolic& s, const double* a, T* fac) {
  const FrontProgram& F = s.front;
  std::vector<T> cb((size_t)F.n_cb, (T)0), M;
  for (size_t i = 0; i < F.sg_src.size(); ++i) {
    T v = (T)a[F.sg_src[i]];
    if (F.sg_div[i] >= 0) v = v / (T)a[F.sg_div[i]];
    fac[F.n_fac + i] = v;
  }
  const int ntask = (int)F.task.size() / 4;
  for (int t = 0; t < ntask; ++t) {
    const FrontInst& I = F.inst[F.task[4 * t]];
    const int l0 = F.task[4 * t + 1], nl = F.task[4 * t + 2];
    for (int o = F.level[l0]; o < F.level[l0 + nl]; ++o) {
      const FrontDesc& d = F.fronts[F.order[o]];
      const int ld = front_ld(d.nt), k = d.k, m = d.m, ns = m - k;
      M.assign((size_t)front_lds(d.nt), (T)0);
      for (int e = 0; e < d.na; ++e) M[F.apos[d.a0 + e]] = (T)a[F.asrc[d.a0 + I.asrc + e]];
      for (int e = 0; e < d.nc; ++e) {
        const uint16_t p = F.cpos[d.cpos + e];
        if (p != kNoPos) M[p & kPosMask] += cb[(size_t)I.cb + d.c0 + e];
      }
      for (int p = 0; p < k; ++p) {
        const T piv = M[p + (size_t)p * ld];
        for (int i = p + 1; i < m; ++i) M[i + (size_t)p * ld] /= piv;
        for (int j = p + 1; j < m; ++j) {
          const T u = M[p + (size_t)j * ld];
          for (int i = p + 1; i < m; ++i) {
            T& x = M[i + (size_t)j * ld];
            x = std::fma(-M[i + (size_t)p * ld], u, x);
          }
        }
      }
      T* out = fac + I.fac + d.fac;
      for (int j = 0; j < k; ++j)
        for (int i = 0; i < m; ++i) out[j * m + i] = M[i + (size_t)j * ld];
      for (int j = k; j < m; ++j) {
        for (int i = 0; i < k; ++i) out[k * m + (j - k) * k + i] = M[i + (size_t)j * ld];
        for (int i = k; i < m; ++i)
          cb[(size_t)I.cb + d.cb + (size_t)(j - k) * ns + (i - k)] = M[i + (size_t)j * ld];
      }
    }
  }
}

template <typename T>
void fronts_solve_host(const LuSymbolic& s, const T* fac, const double* b, double* x) {
  const FrontProgram& F = s.front;
  const int n = s.n;
  const T* sg = fac + F.n_fac;
  std::vector<T> y(n), z(n), cv((size_t)F.n_cv), v;
  const int ntask = (int)F.task.size() / 4;
  for (int t = 0; t < ntask; ++t) {
    const FrontInst& I = F.inst[F.task[4 * t]];
    const int l0 = F.task[4 * t + 1], nl = F.task[4 * t + 2];
    for (int o = F.level[l0]; o < F.level[l0 + nl]; ++o) {
      const FrontDesc& d = F.fronts[F.order[o]];
      const T* f = fac + I.fac + d.fac;
      v.assign(d.m, (T)0);
      for (int i = 0; i < d.k; ++i) {
        const int r = I.row + d.r0 + i;
        v[i] = (T)b[s.p[r]];
        for (int e = F.rs_ptr[r]; e < F.rs_ptr[r + 1]; ++e)
          v[i] = std::fma(-sg[e], (T)b[F.rs_rhs[e]], v[i]);
      }
      for (int c = 0; c < d.nv; ++c)
        for (int i = 0; i < d.m; ++i) {
          const uint16_t q = F.vtab[d.vtab + c * d.m + i];
          if (q != kNoPos) v[i] += cv[(size_t)I.cv + d.v0 + q];
        }
      for (int p = 0; p < d.k; ++p)
        for (int i = p + 1; i < d.m; ++i) v[i] = std::fma(-f[p * d.m + i], v[p], v[i]);
      for (int i = 0; i < d.k; ++i) y[I.row + d.r0 + i] = v[i];
      for (int i = d.k; i < d.m; ++i) cv[(size_t)I.cv + d.cv + i - d.k] = v[i];
    }
  }
  for (int t = ntask - 1; t >= 0; --t) {
    const FrontInst& I = F.inst[F.task[4 * t]];
    const int l0 = F.task[4 * t + 1], nl = F.task[4 * t + 2];
    for (int o = F.level[l0 + nl] - 1; o >= F.level[l0]; --o) {
      const FrontDesc& d = F.fronts[F.order[o]];
      const T* f = fac + I.fac + d.fac;
      const int k = d.k, m = d.m;
      v.assign(m, (T)0);
      for (int i = 0; i < k; ++i) v[i] = y[I.row + d.r0 + i];
      for (int j = k; j < m; ++j) v[j] = z[I.row + F.idx[d.idx + j - k]];
      for (int j = m - 1; j >= k; --j)
        for (int i = 0; i < k; ++i) v[i] = std::fma(-f[k * m + (j - k) * k + i], v[j], v[i]);
      for (int j = k - 1; j >= 0; --j) {
        v[j] /= f[j * m + j];
        for (int i = 0; i < j; ++i) v[i] = std::fma(-f[j * m + i], v[j], v[i]);
      }
      for (int i = 0; i < k; ++i) z[I.row + d.r0 + i] = v[i];
    }
  }
  for (int i = 0; i < n; ++i) x[s.q[i]] = (double)z[i];
  for (size_t i = 0; i < F.row_single.size() / 2; ++i) {
    const int r = F.row_single[2 * i];
    x[s.q[r]] = (double)((T)b[s.p[r]] / sg[F.row_single[2 * i + 1]]);
  }
  // the column singletons' rows in chunks, each as a 256-lane sum
  for (size_t i = 0; i < F.col_single.size() / 4; ++i) {
    const int32_t* c = &F.col_single[4 * i];
    T acc = (T)0;
    for (int e0 = c[2]; e0 < c[3]; e0 += kHubChunk) {
      const int e1 = std::min(c[3], e0 + kHubChunk);
      T part[kReduceLanes];
      for (int l = 0; l < kReduceLanes; ++l) {
        T a = (T)0;
        for (int e = e0 + l; e < e1; e += kReduceLanes)
          a = std::fma(sg[e], (T)x[F.us_col[e - F.us_first]], a);
        part[l] = a;
      }
      for (int w = kReduceLanes / 2; w > 0; w >>= 1)
        for (int l = 0; l < w; ++l) part[l] += part[l + w];
      acc += part[0];
    }
    x[s.q[c[0]]] = (double)(((T)b[s.p[c[0]]] - acc) / sg[c[1]]);
  }
}

template void fronts_refactor_host<double>(const LuSymbolic&, const double*, double*);
template void fronts_refactor_host<float>(const LuSymbolic&, const double*, float*);
template void fronts_solve_host<double>(const LuSymbolic&, const double*, const double*, double*);
template void fronts_solve_host<float>(const LuSymbolic&, const float*, const double*, double*);

}  // namespace vjx
