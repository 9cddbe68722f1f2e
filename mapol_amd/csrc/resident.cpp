#include "resident.hpp"

#include <algorithm>
#include <utility>

namespace bpf {

namespace {

struct Task {
  int kind, target, piv;
  int first, n;                          // its words in the pool
};

int pow2_at_least(int x) {
  int g = 1;
  while (g < x) g <<= 1;
  return g;
}

}  // namespace

void build_resident(const Symbolic &S, int cap_top, int cap, ResidentPlan &R) {
  R = ResidentPlan();
  const int nb = S.nb;
  std::vector<std::vector<int>> st(nb), low(nb);   // column structure; L rows
  std::vector<int> parent(nb, -1), lev(nb, 0);
  for (int k = 0; k < nb; k++) {
    st[k].assign(S.lcol.begin() + S.ldiag[k] + 1, S.lcol.begin() + S.lrow[k + 1]);
    low[k].assign(S.lcol.begin() + S.lrow[k], S.lcol.begin() + S.ldiag[k]);
    if (!st[k].empty()) {
      parent[k] = st[k].front();
      lev[parent[k]] = std::max(lev[parent[k]], lev[k] + 1);
    }
  }
  std::vector<char> tail(nb, 0);
  for (int k : S.tail_piv) tail[k] = 1;
  auto pos = [&](int r, int c) {
    const auto b = S.lcol.begin() + S.lrow[r], e = S.lcol.begin() + S.lrow[r + 1];
    return (int)(std::lower_bound(b, e, c) - S.lcol.begin());
  };
  // ---- parts ---------------------------------------------------------------
  std::vector<int> cost(nb), sub(nb, 0);
  std::vector<std::vector<int>> child(nb);
  std::vector<int> roots;
  for (int k = 0; k < nb; k++) {
    cost[k] = (int)st[k].size() + 1;
    if (cost[k] > std::min(cap, cap_top)) return;
    if (tail[k]) continue;
    sub[k] += cost[k];
    const int p = parent[k];
    if (p >= 0 && !tail[p]) {
      sub[p] += sub[k];
      child[p].push_back(k);
    } else {
      roots.push_back(k);
    }
  }
  struct Part { std::vector<int> piv; int stage; };
  std::vector<Part> parts;
  std::vector<int> leaves;                         // subtrees that fit whole
  bool ok = true;
  // the upper levels of the trees at `xs` as one part: down to the highest
  // level below which every subtree fits a part by itself, or as far as fits
  auto cut = [&](auto &self, const std::vector<int> &xs, int room) -> int {
    std::vector<int> all(xs);
    for (size_t q = 0; q < all.size(); q++)
      all.insert(all.end(), child[all[q]].begin(), child[all[q]].end());
    int top = 0;
    for (int k : all) top = std::max(top, lev[k]);
    std::vector<int> at(top + 2, 0), big(top + 2, 0);
    for (int k : all) {
      at[lev[k]] += cost[k];
      big[lev[k]] = std::max(big[lev[k]], sub[k]);
    }
    int L = top + 1, held = 0;
    while (L > 0 && held + at[L - 1] <= room) {
      bool fits = true;                            // everything below L fits whole
      for (int l = 0; l < L; l++) fits = fits && big[l] <= cap;
      if (fits && L <= top) break;
      L--;
      held += at[L];
    }
    Part p;
    p.stage = 0;
    std::vector<int> below;
    for (int k : all) {
      if (lev[k] >= L) p.piv.push_back(k);
      else if (parent[k] < 0 || tail[parent[k]] || lev[parent[k]] >= L) below.push_back(k);
    }
    if (p.piv.empty()) ok = false;                 // a level wider than a part
    for (int k : ok ? below : std::vector<int>()) {
      if (sub[k] <= cap) {
        leaves.push_back(k);
        p.stage = std::max(p.stage, 1);
      } else {
        p.stage = std::max(p.stage, 1 + self(self, {k}, cap));
      }
    }
    parts.push_back(p);
    return p.stage;
  };
  long total = 0;
  for (int k : roots) total += sub[k];
  if (std::max(cap, cap_top) > RES_SLOT_MASK) return;
  if (total <= std::min(cap, cap_top)) {
    Part p;
    p.stage = 0;
    for (int k = 0; k < nb; k++) if (!tail[k]) p.piv.push_back(k);
    parts.push_back(p);
  } else {
    cut(cut, roots, cap_top);
    if (!ok) return;
    // the whole subtrees packed into parts, largest first into the least
    // filled
    long rest = 0;
    for (int k : leaves) rest += sub[k];
    std::stable_sort(leaves.begin(), leaves.end(), [&](int x, int y) { return sub[x] > sub[y]; });
    int nbins = (int)((rest + cap - 1) / cap);
    std::vector<Part> bins(nbins);
    std::vector<int> fill(nbins, 0);
    for (int k : leaves) {
      int b = (int)(std::min_element(fill.begin(), fill.end()) - fill.begin());
      if (fill[b] + sub[k] > cap) {
        bins.push_back({});
        fill.push_back(0);
        b = (int)bins.size() - 1;
      }
      fill[b] += sub[k];
      std::vector<int> all(1, k);
      for (size_t q = 0; q < all.size(); q++)
        all.insert(all.end(), child[all[q]].begin(), child[all[q]].end());
      bins[b].piv.insert(bins[b].piv.end(), all.begin(), all.end());
    }
    for (auto &b : bins) {
      b.stage = 0;
      if (!b.piv.empty()) parts.push_back(b);
    }
  }
  std::stable_sort(parts.begin(), parts.end(), [](const Part &x, const Part &y) { return x.stage < y.stage; });
  const int np = (int)parts.size(), nst = parts.back().stage + 1;
  R.stage.assign(nst + 1, np);
  for (int p = np - 1; p >= 0; p--) R.stage[parts[p].stage] = p;
  if (R.stage[nst] - R.stage[nst - 1] != 1) return;
  // ---- slots ---------------------------------------------------------------
  std::vector<char> in_jac(S.lcol.size(), 0);      // symmetric, like the pattern
  for (int q : S.jac_lu) in_jac[q] = 1;
  auto start = [&](int r, int c) {
    const int q = pos(r, c);
    return q | (in_jac[q] ? 0 : RES_FILL);
  };
  // rows nb stands for the right-hand side, the last entry of every column
  std::vector<int> part_of(nb, np), slot0(nb, -1), local(nb, -1);
  const int first_rhs = (int)S.lcol.size();
  for (int p = 0; p < np; p++) {
    auto &pv = parts[p].piv;
    std::sort(pv.begin(), pv.end());
    R.part.insert(R.part.end(), {R.nslots, 0, 0, 0, 0, 0, 0, 0});
    int at = 1;                                    // local 0: the zero slot
    for (int k : pv) {
      part_of[k] = p;
      local[k] = at;
      slot0[k] = R.nslots;
      const int keep = lev[k] == 0 && S.l0_chunks > 0 ? RES_KEEP : 0;
      for (int r : st[k]) {
        R.slot_pos.push_back(start(r, k) | keep);
        R.slot_pos.push_back(pos(k, r));
      }
      R.slot_pos.push_back(S.ldiag[k] | keep);
      R.slot_pos.push_back(first_rhs + k);
      at += cost[k];
      R.nslots += cost[k];
    }
    R.part[8 * p + 1] = R.nslots;
    if (at - 1 > (p == np - 1 ? cap_top : cap)) return;
  }
  // local slot of (k, r), r = nb the right-hand side
  auto slot = [&](int k, int r) {
    if (r == nb) return local[k] + (int)st[k].size();
    return local[k] + (int)(std::lower_bound(st[k].begin(), st[k].end(), r) - st[k].begin());
  };
  // ---- rounds --------------------------------------------------------------
  // tasks (pivots first) into waves of one lane-group size, `per` waves a
  // round, with the words per lane that cost least: measured on MI355X a wave
  // issues about 120 instructions a round and 22 per word (4.45 cycles each on
  // one of four SIMDs), 8 per halving of a lane group (40 beyond 16 lanes), and
  // a word reads four 16-byte LDS gathers of 10 cycles;
  // a round's chain is about 350 cycles and 130 per word, of which a
  // workgroup that shares its compute unit with four others shows 0.3
  bool fits = true;
  std::vector<uint32_t> pool;
  std::vector<int> ix, cut_at;
  auto pack = [&](const std::vector<Task> &ts, bool level, int per) {
    if (ts.empty()) return;
    int np1 = 0;
    for (auto &t : ts) np1 += t.kind == RES_PIVOT;
    // longest first within pivots and others, so that lane groups shrink
    ix.resize(ts.size());
    for (size_t q = 0; q < ts.size(); q++) ix[q] = (int)q;
    auto longer = [&](int x, int y) { return ts[x].n > ts[y].n; };
    std::stable_sort(ix.begin(), ix.begin() + np1, longer);
    std::stable_sort(ix.begin() + np1, ix.end(), longer);
    auto group = [&](int q, int J) { return pow2_at_least((ts[ix[q]].n + J - 1) / J); };
    // waves as ends in ix; pw: those of the pivots
    int pw = 0;
    auto order = [&](int J) {
      cut_at.assign(1, 0);
      int g = 0, used = 64;
      for (int q = 0; q < (int)ix.size(); q++) {
        const int gq = group(q, J);
        if (q > 0 && (gq != g || used + gq > 64 || q == np1)) { cut_at.push_back(q); used = 0; }
        if (q == np1) pw = (int)cut_at.size() - 1;
        if (q == 0) used = 0;
        g = gq;
        used += gq;
      }
      cut_at.push_back((int)ix.size());
      if (np1 == (int)ix.size()) pw = (int)cut_at.size() - 1;
    };
    // words per lane of a wave: its tasks share one group size, longest first
    auto words = [&](int w, int J) {
      const int g = group(cut_at[w], J);
      return (ts[ix[cut_at[w]]].n + g - 1) / g;
    };
    auto padded = [](int j) { return j > 4 ? 8 : j > 2 ? 4 : j; };
    const double alone = per == RES_TOP_LANES / 64 ? 1.0 : 0.3;
    int best = 0;
    double least = 0;
    for (int J = 1; J <= RES_J; J *= 2) {
      order(J);
      const int nw = (int)cut_at.size() - 1;
      bool in = true;
      double c = 0;
      for (int w = 0; w < nw; w += per) {
        int jm = 0;
        for (int x = w; x < std::min(nw, w + per); x++) {
          const int j = padded(words(x, J)), g = group(cut_at[x], J);
          in = in && g <= 64;
          jm = std::max(jm, j);
          int lg = 0;
          while ((1 << lg) < g) lg++;
          c += 133 + 42 * j + 9 * lg + 36 * std::max(0, lg - 4);
        }
        c += (350 + 130 * jm) * alone;
      }
      if (in && (best == 0 || c < least)) { best = J; least = c; }
    }
    if (best == 0) { fits = false; return; }
    const int J = best;
    order(J);
    const int nwaves = (int)cut_at.size() - 1;
    const int nr = (nwaves + per - 1) / per;
    for (int r = 0; r < nr; r++) {
      const int w0 = r * per, w1 = std::min(nwaves, w0 + per);
      int bar = 0;
      if (pw > w0 && pw <= w1) bar |= RES_MID;
      if (level && r == nr - 1) bar |= RES_END;
      for (int w = w0; w < w0 + per; w++) {
        if (w >= w1) {
          R.wave.insert(R.wave.end(), {0, 0, bar, 0});
          continue;
        }
        const int g = group(cut_at[w], J), jw = padded(words(w, J));
        if (jw > 1) while (R.word.size() % jw) R.word.push_back(0u);   // vector loads
        int lg = 0;
        while ((1 << lg) < g) lg++;
        const int wb = (int)R.word.size(), db = (int)R.desc.size();
        R.word.resize(wb + (size_t)64 * jw, 0u);
        R.desc.resize(db + (size_t)64, 0u);
        const int kind = ts[ix[cut_at[w]]].kind;
        const int all = kind == RES_PIVOT ? RES_PIV : kind >= RES_UPD_PAIR ? RES_UPD : 0;
        R.wave.insert(R.wave.end(), {wb, db, jw | lg << 4 | RES_RUN | all | bar, 0});
        int lane = 0;
        for (int q = cut_at[w]; q < cut_at[w + 1]; q++) {
          const Task &t = ts[ix[q]];
          // word n of the task: lane n % g of its group, step n / g
          for (int n = 0; n < t.n; n++)
            R.word[wb + (size_t)jw * (lane + n % g) + n / g] = pool[t.first + n];
          R.desc[db + (size_t)lane] = (uint32_t)t.kind << RES_KIND_SHIFT |
                                      (uint32_t)t.piv << RES_SLOT_BITS | (uint32_t)t.target;
          lane += g;
        }
      }
    }
  };
  // target (r, c) as one key, with the updates for it (c = nb: right-hand side)
  auto key = [&](int r, int c) { return (uint64_t)r * (nb + 1) + c; };
  std::vector<std::pair<uint64_t, int>> updates;
  std::vector<std::pair<uint64_t, uint32_t>> sums;
  std::vector<int> count, at;
  std::vector<int> plev(nb, 0);
  for (int p = 0; p < np; p++) {
    const auto &pv = parts[p].piv;
    const int per = (p == np - 1 ? RES_TOP_LANES : RES_SMALL_LANES) / 64;
    R.part[8 * p + 7] = per;
    while (R.word.size() % 4) R.word.push_back(0u);
    R.part[8 * p + 5] = (int)R.word.size();
    R.part[8 * p + 6] = (int)R.desc.size();
    R.part[8 * p + 2] = R.part[8 * p + 3] = (int)R.wave.size() / 4;
    int top = -1;
    for (int k : pv) {
      for (int c : child[k])
        if (part_of[c] == p) plev[k] = std::max(plev[k], plev[c] + 1);
      top = std::max(top, plev[k]);
    }
    // level by level; the pivots the fill may have finished come first
    for (int l = -1; l <= top; l++) {
      std::vector<Task> ts, rest;
      pool.clear();
      for (int k : pv) {
        const bool filled = lev[k] == 0;
        if (l < 0 ? !filled : (filled || plev[k] != l)) continue;
        // words of the pivot (entry 0), of each slot (k, r) and of the
        // right-hand side: counted, then written in the order of low[k]
        const int ns = (int)st[k].size();
        count.assign(ns + 2, 0);
        for (int pass = 0; pass < 2; pass++) {
          if (pass) {
            at.assign(ns + 3, (int)pool.size());
            for (int q = 0; q < ns + 2; q++) at[q + 1] = at[q] + count[q];
            pool.resize(at[ns + 2]);
            ts.push_back({RES_PIVOT, slot(k, nb), 0, at[0], count[0]});
            for (int q = 0; q < ns; q++)
              rest.push_back({RES_PAIR, local[k] + q, slot(k, nb), at[q + 1], count[q + 1]});
            if (count[ns + 1]) rest.push_back({RES_RHS, slot(k, nb), 0, at[ns + 1], count[ns + 1]});
          }
          auto put = [&](int q, uint32_t w) {
            if (pass) pool[at[q]++] = w; else count[q]++;
          };
          for (int m : low[k]) {
            if (part_of[m] != p) continue;
            const int x = slot(m, k) - local[m];
            const uint32_t a = (uint32_t)(local[m] + x);
            put(0, a | a << 16);
            // the rest of m's structure lies in k's
            for (int y = x + 1, q = 0; y < (int)st[m].size(); y++, q++) {
              while (st[k][q] != st[m][y]) q++;
              put(q + 1, a | (uint32_t)(local[m] + y) << 16);
            }
            put(ns + 1, a | (uint32_t)slot(m, nb) << 16);
          }
        }
      }
      ts.insert(ts.end(), rest.begin(), rest.end());
      pack(ts, true, per);
      if (l < 0 && S.l0_chunks > 0) R.part[8 * p + 3] = (int)R.wave.size() / 4;
    }
    // the sums for later parts and the tail
    sums.clear();
    for (int m : pv) {
      const int n = (int)st[m].size();
      for (int x = 0; x < n; x++) {
        const int r = st[m][x];
        if (part_of[r] == p) continue;
        const uint32_t a = (uint32_t)(local[m] + x);
        for (int y = x; y < n; y++)
          if (part_of[st[m][y]] != p)
            sums.push_back({key(r, st[m][y]), a | (uint32_t)(local[m] + y) << 16});
        if (!tail[r]) sums.push_back({key(r, nb), a | (uint32_t)slot(m, nb) << 16});
      }
    }
    std::stable_sort(sums.begin(), sums.end(),
                     [](auto &x, auto &y) { return x.first < y.first; });
    std::vector<Task> ts;
    pool.clear();
    for (size_t q = 0; q < sums.size();) {
      const uint64_t w = sums[q].first;
      const int r = (int)(w / (nb + 1)), c = (int)(w % (nb + 1)), f = (int)pool.size();
      for (; q < sums.size() && sums[q].first == w; q++) pool.push_back(sums[q].second);
      // the right-hand side shares the diagonal's update, formed just before
      // in this part (c ascends within r)
      if (c == r) at.assign(1, R.nupd);
      const int u = c == nb ? at[0] : R.nupd++;
      if (c != nb) updates.push_back({w, u});
      ts.push_back({c == nb ? RES_UPD_RHS : c == r ? RES_UPD_DIAG : RES_UPD_PAIR, u, 0, f,
                    (int)pool.size() - f});
    }
    pack(ts, false, per);
    if (!fits) return;
    R.part[8 * p + 4] = (int)R.wave.size() / 4;
  }
  R.part.insert(R.part.end(), {0, 0, 0, 0, 0, (int)R.word.size(), (int)R.desc.size(), 0});
  // ---- where the updates go --------------------------------------------------
  std::stable_sort(updates.begin(), updates.end(), [](auto &x, auto &y) { return x.first < y.first; });
  auto append = [&](int k, int r, std::vector<int> &to) {
    const uint64_t w = key(k, r);
    auto it = std::lower_bound(updates.begin(), updates.end(), w,
                               [](const std::pair<uint64_t, int> &x, uint64_t y) { return x.first < y; });
    for (; it != updates.end() && it->first == w; ++it) to.push_back(it->second);
  };
  R.upd_ptr.assign(1, 0);
  for (int p = 0; p < np; p++)
    for (int k : parts[p].piv)
      for (size_t q = 0; q <= st[k].size(); q++) {
        if (p >= R.stage[1]) append(k, q < st[k].size() ? st[k][q] : k, R.upd);
        R.upd_ptr.push_back((int)R.upd.size());
      }
  R.tail_ptr.assign(1, 0);
  std::vector<int> loc(nb, -1);
  for (int a = 0; a < S.tail_n; a++) loc[S.tail_piv[a]] = a;
  for (int k : S.tail_piv)
    for (size_t q = 0; q <= st[k].size(); q++) {
      const int r = q < st[k].size() ? st[k][q] : k;
      R.tail.insert(R.tail.end(), {start(r, k), r == k ? -1 : pos(k, r), loc[k], loc[r]});
      append(k, r, R.tail_upd);
      R.tail_ptr.push_back((int)R.tail_upd.size());
    }
  R.word.resize(R.word.size() + 8, 0u);    // the kernels load four words at a time
  R.ok = R.nupd < 1 << RES_KIND_SHIFT;
}

}  // namespace bpf
