// The plan of the LDS-resident factorization, run step by step on the CPU.
//
// A random block matrix of the case's pattern (diagonally dominant) and a
// random right-hand side are factored twice: by a plain block elimination,
// and by executing the plan as the kernels do: per part a slot array of at
// most the cap of slots loaded from the factor storage less the updates of earlier
// parts, rounds of at most the part's waves with their words per lane and lane groups,
// updates kept for later parts, the slots stored back, the tail assembled.
// Checked besides the values:
// * a word names a slot of its part whose value is final when it is read;
// * a pivot inverse is read only after a barrier that follows its round;
// * within a wave the groups are aligned and of the wave's size;
// * every update is formed once, in a part of an earlier stage than its user;
// * with and without level 0 finished by the Jacobian fill.
//
// Reads "n m ordering tail cap_top cap", n bus types and m branch end pairs from
// stdin; prints "ok, stages parts slots rounds" (exit 0) or the first
// violation (exit 1).
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <string>
#include <vector>

#include "../../mapol_amd/csrc/resident.hpp"

using namespace bpf;

struct Blk { double a = 0, b = 0, c = 0, d = 0; };
static Blk mul(const Blk &x, const Blk &y) {
  return {x.a * y.a + x.b * y.c, x.a * y.b + x.b * y.d, x.c * y.a + x.d * y.c, x.c * y.b + x.d * y.d};
}
static void add(Blk &x, const Blk &y, double f) { x.a += f * y.a; x.b += f * y.b; x.c += f * y.c; x.d += f * y.d; }
static Blk inv(const Blk &x) {
  const double r = 1 / (x.a * x.d - x.b * x.c);
  return {x.d * r, -x.b * r, -x.c * r, x.a * r};
}
static double off(const Blk &x, const Blk &y) {
  return std::fabs(x.a - y.a) + std::fabs(x.b - y.b) + std::fabs(x.c - y.c) + std::fabs(x.d - y.d);
}
static double rnd() { return rand() / (double)RAND_MAX - 0.5; }
static int fail(const char *what, int a = 0, int b = 0) {
  printf("FAIL %s (%d, %d)\n", what, a, b);
  return 1;
}

int main() {
  int n, m, ordering, tail, cap_top, cap_small;
  if (scanf("%d %d %d %d %d %d", &n, &m, &ordering, &tail, &cap_top, &cap_small) != 6) return 2;
  std::vector<int> ty(n), f(m), t(m);
  for (int i = 0; i < n; i++) if (scanf("%d", &ty[i]) != 1) return 2;
  for (int b = 0; b < m; b++) if (scanf("%d %d", &f[b], &t[b]) != 2) return 2;
  AnalysisParams prm;
  prm.ordering = ordering;
  prm.tail_limit = tail;
  Symbolic S;
  std::string err;
  if (!analyse(n, m, f.data(), t.data(), ty.data(), S, &err, prm)) return 2;
  ResidentPlan R;
  build_resident(S, cap_top, cap_small, R);
  if (!R.ok) return fail("no plan");
  const int nb = S.nb, nz = (int)S.lcol.size(), np = (int)R.part.size() / 8 - 1;
  auto pos = [&](int r, int c) {
    for (int p = S.lrow[r]; p < S.lrow[r + 1]; p++) if (S.lcol[p] == c) return p;
    return -1;
  };
  // the matrix: Jacobian blocks random, fill zero, right-hand sides after it
  std::vector<Blk> J(nz + nb);
  srand(1);
  for (int p : S.jac_lu) J[p] = {rnd(), rnd(), rnd(), rnd()};
  for (int k = 0; k < nb; k++) { J[S.ldiag[k]].a += 8; J[S.ldiag[k]].d += 8; }
  for (int k = 0; k < nb; k++) { J[nz + k].a = rnd(); J[nz + k].c = rnd(); }
  // plain elimination: pivots inverted, L scaled, U as is, y in the tail rows left
  std::vector<char> intail(nb, 0);
  std::vector<int> loc(nb, -1);
  for (int a = 0; a < S.tail_n; a++) { intail[S.tail_piv[a]] = 1; loc[S.tail_piv[a]] = a; }
  std::vector<Blk> W = J;
  for (int k = 0; k < nb; k++) {
    if (intail[k]) continue;
    W[S.ldiag[k]] = inv(W[S.ldiag[k]]);
    for (int x = S.ldiag[k] + 1; x < S.lrow[k + 1]; x++) {
      const int r = S.lcol[x], pl = S.mirror[x];
      W[pl] = mul(W[pl], W[S.ldiag[k]]);
      for (int y = S.ldiag[k] + 1; y < S.lrow[k + 1]; y++) add(W[pos(r, S.lcol[y])], mul(W[pl], W[y]), -1);
      if (!intail[r]) add(W[nz + r], mul(W[pl], W[nz + k]), -1);
    }
  }
  const int s = S.tail_n;
  std::vector<int> lev0(nz + nb, 0);
  for (int filled = 0; filled < (S.l0_chunks > 0 ? 2 : 1); filled++) {
    std::vector<Blk> A(nz + nb, Blk{7, -3, 5, 11});   // fill-in is not cleared
    for (int p : S.jac_lu) A[p] = J[p];
    for (int k = 0; k < nb; k++) A[nz + k] = J[nz + k];
    if (filled)                          // what the Jacobian fill leaves of level 0
      for (size_t r = 0; r < S.jac_lu.size(); r++) {
        if (S.jac_l0[r] == -2) A[S.jac_lu[r]] = inv(J[S.jac_lu[r]]);
        else if (S.jac_l0[r] >= 0) A[S.jac_lu[r]] = mul(J[S.jac_lu[r]], inv(J[S.jac_lu[S.jac_l0[r]]]));
      }
    std::vector<Blk> UPD(2 * (size_t)R.nupd);
    std::vector<int> made(R.nupd, 0), made_by(R.nupd, -1);
    std::vector<int> stage_of(np, 0);
    for (int q = 0; q + 1 < (int)R.stage.size(); q++)
      for (int p = R.stage[q]; p < R.stage[q + 1]; p++) stage_of[p] = q;
    if (R.stage.back() != np || R.stage[R.stage.size() - 2] != np - 1) return fail("stages");
    std::vector<char> stored(nz + nb, 0);
    for (int p = 0; p < np; p++) {
      const int *P = &R.part[8 * p];
      const int ns = P[1] - P[0];
      const int W = P[7];
      if (W != (p == np - 1 ? RES_TOP_LANES : RES_SMALL_LANES) / 64) return fail("waves of a part", p, W);
      if (ns > (p == np - 1 ? cap_top : cap_small)) return fail("part above its capacity", p, ns);
      // per slot part and side: the round after whose barrier the value is final
      std::vector<Blk> L(ns + 1), U(ns + 1);
      std::vector<int> finL(ns + 1, 1 << 30), finU(ns + 1, 1 << 30);
      finL[0] = finU[0] = -1;
      for (int q = 0; q < ns; q++) {
        const int *sp = &R.slot_pos[2 * (size_t)(P[0] + q)];
        if (!(sp[0] & RES_FILL)) {
          L[q + 1] = A[sp[0] & RES_POS];
          U[q + 1] = A[sp[1]];
        }
        for (int e = R.upd_ptr[P[0] + q]; e < R.upd_ptr[P[0] + q + 1]; e++) {
          const int u = R.upd[e];
          if (!made[u] || stage_of[made_by[u]] >= stage_of[p]) return fail("update not ready", p, u);
          add(L[q + 1], UPD[2 * u], -1);
          add(U[q + 1], UPD[2 * u + 1], -1);
        }
        if ((sp[0] & RES_KEEP) && filled) finL[q + 1] = -1;
        // a U part or y without a task of its own is final as loaded
      }
      std::vector<char> taskU(ns + 1, 0);
      const int r0 = filled ? P[3] : P[2];
      for (int r = r0; r < P[4]; r += W)
        for (int w = 0; w < W; w++) {
          const int *wt = &R.wave[4 * ((size_t)r + w)];
          for (int l = 0; (wt[2] & RES_RUN) && l < 64; l++) {
            const uint32_t d = R.desc[(size_t)(wt[1] + l)];
            const int kind = (int)(d >> RES_KIND_SHIFT);
            if (kind == RES_PAIR || kind == RES_RHS) taskU[d & RES_SLOT_MASK] = 1;
          }
        }
      for (int q = 1; q <= ns; q++) if (!taskU[q]) finU[q] = -1;
      int epoch = 0;                     // barriers passed
      for (int r = r0; r < P[4]; r += W) {
        const int bar = R.wave[4 * ((size_t)r) + 2] & (RES_MID | RES_END);
        struct Out { int kind, slot, piv; Blk l, u; };
        std::vector<Out> outs;
        for (int w = 0; w < W; w++) {
          const int *wt = &R.wave[4 * ((size_t)r + w)];
          if ((wt[2] & (RES_MID | RES_END)) != bar) return fail("barriers differ", r, w);
          if (!(wt[2] & RES_RUN)) continue;
          const int jw = wt[2] & 15, g = 1 << ((wt[2] >> 4) & 7);
          if ((jw > 2 && jw != 4 && jw != 8) || g > 64 || (jw && wt[0] % std::min(jw, 4))) return fail("wave shape", r, w);
          if (wt[0] + 64 * (size_t)jw + 8 > R.word.size() || (size_t)wt[1] + 64 > R.desc.size())
            return fail("tables too short", r, w);
          for (int l0 = 0; l0 < 64; l0 += g) {
            const uint32_t d = R.desc[(size_t)(wt[1] + l0)];
            for (int x = 1; x < g; x++)
              if (R.desc[(size_t)(wt[1] + l0 + x)]) return fail("misaligned group", r, w);
            const int kind = (int)(d >> RES_KIND_SHIFT);
            if (!kind) continue;
            if ((kind == RES_PIVOT) != !!(wt[2] & RES_PIV) || (kind >= RES_UPD_PAIR) != !!(wt[2] & RES_UPD))
              return fail("kinds of a wave", r, w);
            const int target = (int)(kind >= RES_UPD_PAIR ? d & ((1u << RES_KIND_SHIFT) - 1) : d & RES_SLOT_MASK);
            Out o{kind, target, (int)(d >> RES_SLOT_BITS) & RES_SLOT_MASK, {}, {}};
            for (int j = 0; j < jw; j++)
              for (int x = 0; x < g; x++) {
                const uint32_t wd = R.word[wt[0] + (size_t)jw * (l0 + x) + j];
                const int a = wd & 0xFFFF, b = wd >> 16;
                if (a > ns || b > ns) return fail("word outside the part", r, w);
                // both orders of a pair are read; the unused sums may be anything
                if (finL[a] > epoch || finU[b] > epoch) return fail("operand not final", r, w);
                if ((kind == RES_PAIR || kind == RES_UPD_PAIR) && (finL[b] > epoch || finU[a] > epoch)) return fail("operand not final", r, w);
                add(o.u, mul(L[a], U[b]), 1);
                add(o.l, mul(L[b], U[a]), 1);
              }
            outs.push_back(o);
          }
        }
        for (auto &o : outs)
          if (o.kind == RES_PIVOT) {
            Blk v = L[o.slot];
            add(v, o.u, -1);
            L[o.slot] = inv(v);
            finL[o.slot] = epoch + 1;
          }
        if (bar & RES_MID) epoch++;
        for (auto &o : outs) {
          if (o.kind == RES_PAIR) {
            if (finL[o.piv] > epoch) return fail("pivot not final", r);
            Blk v = L[o.slot];
            add(v, o.l, -1);
            L[o.slot] = mul(v, L[o.piv]);
            add(U[o.slot], o.u, -1);
            finL[o.slot] = finU[o.slot] = epoch + 1;
          } else if (o.kind == RES_RHS) {
            add(U[o.slot], o.u, -1);
            finU[o.slot] = epoch + 1;
          } else if (o.kind == RES_UPD_PAIR) {
            UPD[2 * o.slot] = o.l; UPD[2 * o.slot + 1] = o.u;
          } else if (o.kind == RES_UPD_DIAG) {
            UPD[2 * o.slot] = o.u;
          } else if (o.kind == RES_UPD_RHS) {
            UPD[2 * o.slot + 1] = o.u;
          }
          if (o.kind == RES_UPD_PAIR || o.kind == RES_UPD_DIAG) {
            if (made[o.slot]++) return fail("update formed twice", o.slot);
            made_by[o.slot] = p;
          }
        }
        if (bar & RES_END) epoch++;
      }
      for (int q = 0; q < ns; q++) {
        const int *sp = &R.slot_pos[2 * (size_t)(P[0] + q)];
        if (finL[q + 1] == 1 << 30 || finU[q + 1] == 1 << 30) return fail("slot never finished", p, q);
        if (stored[sp[0] & RES_POS]++ || stored[sp[1]]++) return fail("stored twice", p, q);
        if ((sp[0] & RES_KEEP) && filled) continue;
        A[sp[0] & RES_POS] = L[q + 1];
        A[sp[1]] = U[q + 1];
      }
    }
    double worst = 0;
    for (int k = 0; k < nb; k++) {
      if (intail[k]) continue;
      for (int x = S.ldiag[k]; x < S.lrow[k + 1]; x++) {
        worst = std::fmax(worst, off(A[x], W[x]));
        worst = std::fmax(worst, off(A[S.mirror[x]], W[S.mirror[x]]));
      }
      worst = std::fmax(worst, off(A[nz + k], W[nz + k]));
    }
    if ((int)R.tail.size() / 4 + 1 != (int)R.tail_ptr.size()) return fail("tail lists");
    for (size_t e = 0; e + 1 < R.tail_ptr.size(); e++) {
      const int *te = &R.tail[4 * e];
      Blk l, u;
      if (!(te[0] & RES_FILL)) {
        l = A[te[0]];
        if (te[1] >= 0) u = A[te[1]];
      }
      for (int q = R.tail_ptr[e]; q < R.tail_ptr[e + 1]; q++) {
        add(l, UPD[2 * R.tail_upd[q]], -1);
        add(u, UPD[2 * R.tail_upd[q] + 1], -1);
      }
      worst = std::fmax(worst, off(l, W[te[0] & RES_POS]));
      if (te[1] >= 0) worst = std::fmax(worst, off(u, W[te[1]]));
      const int r = S.tail_piv[te[2]], c = S.tail_piv[te[3]];
      if (pos(c, r) != (te[0] & RES_POS) || (te[1] >= 0 && pos(r, c) != te[1])) return fail("tail positions", (int)e);
    }
    if (!(worst < 1e-10)) { printf("FAIL values differ by %g (level 0 %s)\n", worst, filled ? "filled" : "here"); return 1; }
  }
  (void)s;
  printf("ok, %d stages %d parts %d slots %d wave rounds %zu words %d updates\n", (int)R.stage.size() - 1, np,
         R.nslots, (int)R.wave.size() / 4, R.word.size(), R.nupd);
  return 0;
}
