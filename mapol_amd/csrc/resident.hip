// LDS-resident factorization (kernels of the plan in resident.hpp).
//
// A compute unit gathers a 16-byte block from LDS in a sixth of the time it
// takes from L1 or L2 (a wave's gather: 10 against 64 cycles, one cache line a
// cycle), and a product of the elimination reads two blocks.  So the tree
// below the dense tail is cut into parts whose blocks fit LDS: a workgroup
// loads its part, eliminates it there level by level, leaves the sums that
// later parts need (updates) and stores the part once.  No product touches
// memory.  Parts of one stage run side by side: one instance fills 36 compute
// units at 9241 buses, and 200 instances keep five workgroups of 256 lanes on
// every compute unit, whose barriers and LDS round trips overlap.
//
// What bounds it now: a round's chain of LDS read, lane-group sum, pivot
// inverse, two barriers (about 2000 cycles, 17 to 36 rounds a part) while few
// instances are active; with many, the instructions a wave spends per round
// (lists are short: 109 k words in 500 k lane slots at 9241 buses).
// Factorization at 9241 buses in FP32: one instance 188 -> 117 us, average
// over a 200-instance solve's launches 443 -> 293 us; FP64 271 -> 167 and
// 660 -> 580 us; 1354 buses, one instance 71 -> 60 us.  Parts of 1024 lanes and
// 158 KB took 115 and 428 us (one workgroup a compute unit overlaps nothing).
#include "resident.hpp"

namespace bpf {

struct ResPlan {
  const int4 *part, *wave;               // two per part; one per round and wave
  const int2 *slot_pos;
  const int *upd_ptr, *upd;
  const unsigned *word, *desc;
  int nupd;                              // updates of one instance
  int tn, ntail;                         // dense tail: pivots, entry pairs
  const int4 *tail;
  const int *tail_ptr, *tail_upd;
};

// four words of a lane at any word's alignment
struct Words4 { unsigned x, y, z, w; };
struct ResFetch {
  int fl;
  unsigned d;
  Words4 a, b;
};

template <typename T>
struct ResSlot { B4<T> l, u; };

// sums of the updates upd[e0..e1) out of the L and U blocks
template <typename T>
__device__ __forceinline__ void sub_updates(const int *list, int e0, int e1, const B4<T> *UPD,
                                            B4<T> &l, B4<T> &u) {
  constexpr int EU = 2;                  // requested together
  for (int e = e0; e < e1; e += EU) {
    int id[EU];
    B4<T> a[EU], b[EU];
#pragma unroll
    for (int x = 0; x < EU; x++) id[x] = list[min(e + x, e1 - 1)];
#pragma unroll
    for (int x = 0; x < EU; x++) {
      a[x] = UPD[2 * (size_t)id[x]];
      b[x] = UPD[2 * (size_t)id[x] + 1];
    }
#pragma unroll
    for (int x = 0; x < EU; x++)
      if (e + x < e1) {
        l.a -= a[x].a; l.b -= a[x].b; l.c -= a[x].c; l.d -= a[x].d;
        u.a -= b[x].a; u.b -= b[x].b; u.c -= b[x].c; u.d -= b[x].d;
      }
  }
}

template <typename T>
__device__ __forceinline__ void blk_fma(B4<T> &acc, const B4<T> &l, const B4<T> &u) {
  acc.a = fma(l.b, u.c, fma(l.a, u.a, acc.a));
  acc.b = fma(l.b, u.d, fma(l.a, u.b, acc.b));
  acc.c = fma(l.d, u.c, fma(l.c, u.a, acc.c));
  acc.d = fma(l.d, u.d, fma(l.c, u.b, acc.d));
}

// One part: slots in, rounds, slots out.  A word {a, b} of a lane adds
// L(a) U(b) and L(b) U(a), so one index pair serves both blocks of a slot; a
// lane group's sums meet in its first lane (DPP), which finishes the slot.
// The next round's words and descriptors are requested as soon as this
// round's are read, and stay in flight over the sums and barriers.
template <typename T, int NL>
__device__ __forceinline__ void res_part(const ResPlan &R, int part, bool l0, bool upd_in,
                                         B4<T> *A, B4<T> *UPD, ResSlot<T> *S, int &sing) {
  constexpr int NW = NL / 64;
  const int4 pa = R.part[2 * part], pb = R.part[2 * part + 1];
  const int s0 = pa.x, ns = pa.y - pa.x, r0 = l0 ? pa.w : pa.z, r1 = pb.x;
  const int tid = (int)threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  if (tid == 0) {
    S[0].l = blk_zero<T>();
    S[0].u = blk_zero<T>();
  }
  // The plan's words and descriptors are read once per launch, and a launch
  // starts with a cold L2: a first touch takes longer than a round.  One lane
  // per 128-byte line brings the part's lists into L2 beside the slots.
  {
    const int4 pc = R.part[2 * part + 3];
    int touch = 0;
    for (int q = pb.y + 32 * tid; q < pc.y; q += 32 * NL) touch ^= (int)R.word[q];
    for (int q = pb.z + 32 * tid; q < pc.z; q += 32 * NL) touch ^= (int)R.desc[q];
    asm volatile("" ::"v"(touch));
  }
  constexpr int LU_ = sizeof(T) == 4 ? 4 : 2;   // slots of a lane requested together
  for (int q0 = tid; q0 < ns; q0 += LU_ * NL) {
    int2 ps[LU_];
    B4<T> l[LU_], u[LU_];
#pragma unroll
    for (int x = 0; x < LU_; x++) ps[x] = R.slot_pos[s0 + min(q0 + x * NL, ns - 1)];
#pragma unroll
    for (int x = 0; x < LU_; x++) {
      l[x] = A[ps[x].x & RES_POS];
      u[x] = A[ps[x].y];
    }
#pragma unroll
    for (int x = 0; x < LU_; x++) {
      const bool fill = ps[x].x & RES_FILL;
      l[x] = blk_sel(fill, blk_zero<T>(), l[x]);
      u[x] = blk_sel(fill, blk_zero<T>(), u[x]);
    }
    if (upd_in) {
#pragma unroll
      for (int x = 0; x < LU_; x++) {
        const int q = s0 + min(q0 + x * NL, ns - 1);
        sub_updates(R.upd, R.upd_ptr[q], R.upd_ptr[q + 1], UPD, l[x], u[x]);
      }
    }
#pragma unroll
    for (int x = 0; x < LU_; x++)
      if (q0 + x * NL < ns) {
        S[1 + q0 + x * NL].l = l[x];
        S[1 + q0 + x * NL].u = u[x];
      }
  }
  __syncthreads();
  // the wave's table entries of 64 rounds, one per lane, read with v_readlane:
  // a wave without work in a round spends a few instructions on it
  int4 tab;
  const int nr = (r1 - r0) / NW;
  auto load_tab = [&](int i) {
    tab = R.wave[r0 + min(i + lane, nr - 1) * NW + wv];
    __builtin_amdgcn_s_waitcnt(WAIT_VMCNT0);
  };
  // round i's words and descriptor: requested with no register of another set
  // involved (a copy of a loaded register would wait for the load)
  auto fetch = [&](int i, ResFetch &f) {
    f.fl = __builtin_amdgcn_readlane(tab.z, i & 63);
    if (f.fl & RES_RUN) {
      const unsigned *wp = R.word + __builtin_amdgcn_readlane(tab.x, i & 63);
      const int jw = f.fl & 15;
      f.d = R.desc[__builtin_amdgcn_readlane(tab.y, i & 63) + lane];
      f.a = *(const Words4 *)(wp + jw * lane);
      if (jw > 4) f.b = *(const Words4 *)(wp + jw * lane + 4);
    }
  };
  auto round = [&](int i, const ResFetch &f, ResFetch &next) {
    const int fl = f.fl;
    unsigned d = 0;
    int piv = 0, slot = 0;
    B4<T> aL = blk_zero<T>(), aU = aL, oL, oU;
    if (fl & RES_RUN) {
      __builtin_amdgcn_s_waitcnt(WAIT_VMCNT0);
      const int jw = fl & 15, g = 1 << ((fl >> 4) & 7);
      d = f.d;
      slot = d & RES_SLOT_MASK;
      piv = (d >> RES_SLOT_BITS) & RES_SLOT_MASK;
      if (!(fl & RES_UPD)) {
        oL = S[slot].l;
        oU = S[slot].u;
      }
      auto word = [&](unsigned v) {
        const ResSlot<T> p = S[v & 0xFFFF], q = S[v >> 16];
        blk_fma(aU, p.l, q.u);
        blk_fma(aL, q.l, p.u);
      };
      auto words = [&](unsigned v, unsigned x) {   // two words' reads together
        if constexpr (sizeof(T) == 8) {              // (FP64 has not the registers)
          word(v);
          word(x);
          return;
        }
        const ResSlot<T> p = S[v & 0xFFFF], q = S[v >> 16], k = S[x & 0xFFFF], m = S[x >> 16];
        blk_fma(aU, p.l, q.u);
        blk_fma(aL, q.l, p.u);
        blk_fma(aU, k.l, m.u);
        blk_fma(aL, m.l, k.u);
      };
      if (jw == 1) word(f.a.x);
      if (jw > 1) words(f.a.x, f.a.y);
      if (jw > 2) words(f.a.z, f.a.w);
      if (jw > 4) { words(f.b.x, f.b.y); words(f.b.z, f.b.w); }
      group_sum4x2_first(aU, aL, g);
    }
    if (i + 1 < nr) {
      if (((i + 1) & 63) == 0) load_tab(i + 1);
      fetch(i + 1, next);
    }
    if (fl & RES_PIV) {
      if (d >> RES_KIND_SHIFT) {
        B4<T> v = oL, inv;
        v.a -= aU.a; v.b -= aU.b; v.c -= aU.c; v.d -= aU.d;
        if (blk_inv(v, inv)) sing = 1;
        S[slot].l = inv;
      }
    }
    if (fl & RES_MID) __syncthreads();
    if ((fl & (RES_RUN | RES_PIV | RES_UPD)) == RES_RUN) {
      const int kind = (int)(d >> RES_KIND_SHIFT);
      if (kind) {
        oU.a -= aU.a; oU.b -= aU.b; oU.c -= aU.c; oU.d -= aU.d;
        S[slot].u = oU;
        if (kind == RES_PAIR) {
          const B4<T> D = S[piv].l;
          oL.a -= aL.a; oL.b -= aL.b; oL.c -= aL.c; oL.d -= aL.d;
          S[slot].l = blk_mul(oL, D);
        }
      }
    } else if (fl & RES_UPD) {
      const int kind = (int)(d >> RES_KIND_SHIFT);
      B4<T> *to = UPD + 2 * (size_t)(d & ((1u << RES_KIND_SHIFT) - 1));
      if (kind == RES_UPD_PAIR) {
        to[0] = aL;
        to[1] = aU;
      } else if (kind) {
        to[kind == RES_UPD_RHS ? 1 : 0] = aU;
      }
    }
    if (fl & RES_END) __syncthreads();
  };
  if (nr > 0) {
    ResFetch fa, fb;
    load_tab(0);
    fetch(0, fa);
    for (int i = 0; i < nr; i += 2) {
      round(i, fa, fb);
      if (i + 1 < nr) round(i + 1, fb, fa);
    }
  }
  for (int q = tid; q < ns; q += NL) {
    const int2 ps = R.slot_pos[s0 + q];
    if (l0 && (ps.x & RES_KEEP)) continue;
    A[ps.x & RES_POS] = S[1 + q].l;
    A[ps.y] = S[1 + q].u;
  }
}

// the parts p0 .. p0 + np - 1 of one stage: workgroup b takes part b mod np
// of instance b / np, so that a part's index lists stay in few L2s; a
// singular pivot sets jsing[t], which the last stage reports
template <typename T>
__global__ void __launch_bounds__(RES_SMALL_LANES, 4)
k_res_parts(DevTopo g, const InstState *st, ResPlan R, int p0, int np, int l0, int upd_in,
            B4<T> *LU, B4<T> *UPD, int *jsing) {
  __shared__ __align__(32) char lds[RES_SMALL_LDS];
  __shared__ int sing;
  const int t = (int)blockIdx.x / np, p = (int)blockIdx.x - t * np;
  if (st[t].done) return;
  if (threadIdx.x == 0) sing = 0;
  res_part<T, RES_SMALL_LANES>(R, p0 + p, l0 != 0, upd_in != 0, LU + (size_t)t * g.nnzLU,
              UPD + (size_t)t * 2 * R.nupd, (ResSlot<T> *)lds, sing);
  __syncthreads();
  if (threadIdx.x == 0 && sing) jsing[t] = 1;
}

// the last part, then the dense tail: its Schur complement from the Jacobian
// less the parts' updates, inverted on the matrix cores
template <typename T>
__global__ void __launch_bounds__(RES_TOP_LANES)
k_res_top(DevTopo g, InstState *st, int count_iter, ResPlan R, int part, int l0, int upd_in,
          B4<T> *LU, B4<T> *TL, B4<T> *UPD, int *jsing) {
  __shared__ __align__(32) char lds[RES_TOP_LDS];
  __shared__ int sing;
  static_assert(sizeof(B4<T>) * TAIL_MAX * TAIL_MAX + sizeof(TailQuads<T>) <= RES_TOP_LDS,
                "the dense tail takes the slots' LDS");
  const int t = (int)blockIdx.x;
  if (st[t].done) return;
  if (threadIdx.x == 0) {
    sing = jsing[t];
    jsing[t] = 0;
  }
  B4<T> *A = LU + (size_t)t * g.nnzLU, *U = UPD + (size_t)t * 2 * R.nupd;
  res_part<T, RES_TOP_LANES>(R, part, l0 != 0, upd_in != 0, A, U, (ResSlot<T> *)lds, sing);
  // this part's updates are read by other waves below
  __builtin_amdgcn_s_waitcnt(WAIT_VMCNT0);
  __syncthreads();
  const int s = R.tn, ss = s * s;
  if (s > 0) {
    B4<T> *D = (B4<T> *)lds;
    TailQuads<T> &mq = *(TailQuads<T> *)(lds + sizeof(B4<T>) * TAIL_MAX * TAIL_MAX);
    for (int q = threadIdx.x; q < ss; q += RES_TOP_LANES) D[q] = blk_zero<T>();
    __syncthreads();
    for (int q = threadIdx.x; q < R.ntail; q += RES_TOP_LANES) {
      const int4 te = R.tail[q];
      const bool fill = te.x & RES_FILL;
      B4<T> l = blk_sel(fill, blk_zero<T>(), A[te.x & RES_POS]);
      B4<T> u = blk_sel(fill, blk_zero<T>(), A[max(te.y, 0)]);
      sub_updates(R.tail_upd, R.tail_ptr[q], R.tail_ptr[q + 1], U, l, u);
      D[te.w * s + te.z] = l;
      if (te.y >= 0) D[te.z * s + te.w] = u;
    }
    __syncthreads();
    tail_inverse_mfma<T>(D, s, (s + 1) / 2, mq, TL + (size_t)t * ss, sing);
  }
  if (threadIdx.x == 0 && sing) {
    InstState x = st[t];
    x.done = 1;
    x.verdict = BPF_V_SINGULAR;
    x.it_round += count_iter;
    x.it_total += count_iter;
    st[t] = x;
  }
}

}  // namespace bpf
