// Wave-subtree kernels of linear transients (kg_ws.h): one system per block of
// NW waves. The level-scheduled and LDS-resident kernels put every
// elimination level behind a block barrier, and a level costs two dependent
// LDS round trips plus the serial tail of its long rows. Here a wave owns
// whole subtrees of the elimination forest, so that its levels are ordered by
// its own LDS operations alone; a row takes its entries level by level, with
// addresses and factors in registers, so that a level is one round trip of
// independent LDS reads and two multiply-adds; and the block meets twice per
// step, around the few top rows that wave 0 solves.
//
// Bound by latency: a level costs about 140 cycles (an LDS round trip and two
// dependent FP64 multiply-adds), a step about 0.5 us more for its right-hand
// side, companion update and source value, and 0.5 us for the top rows.
// Measured per trapezoidal step, 256 ladders, against the LDS-resident kernel:
// 52 unknowns 0.85 us (2.4), 202: 1.6 us (3.7), 602: 2.3 us (4.6), 1538: 4.2 us
// (8.8). Sixteen waves (128 registers a lane) spilled and took 10 us at 1538.
#include "kg_device.h"
#include "kg_ws.h"

namespace kg {

namespace {

// Orders a wave's LDS operations for the compiler; the hardware executes
// those of one wave in order.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// a with its sign flipped where sign's top bit is set
__device__ __forceinline__ double flip(double a, uint32_t sign) {
  return __hiloint2double(__double2hiint(a) ^ (int)sign, __double2loint(a));
}

// One row's share of both triangular solves, in registers.
template <int NP_>
struct WsRow {
  static constexpr int NP = NP_;
  uint32_t row, xrow, rx;  // places in y and x; codes beyond two: first | count << 16
  uint32_t pa[NP], pb[NP], ua, ub, ra, rb, sa, sb;  // columns of the pairs and upper entries; histories and signs
  double pv[2 * NP], uv0, uv1, dv, acc;

  // rec: slot record (null: a lane without a row, which reads zeros and
  // writes the unread slots); v: factors (v[nnz] = 0)
  __device__ __forceinline__ void take(const uint16_t* rec, const uint16_t* pairs, const uint16_t* codes,
                                       const double* v, int n, int ytrash, int zero_hist) {
    row = (uint32_t)ytrash;
    xrow = (uint32_t)n + 1;
    ua = ub = (uint32_t)n;
    ra = rb = (uint32_t)zero_hist;
    rx = sa = sb = 0;
    uv0 = uv1 = dv = acc = 0.0;
#pragma unroll
    for (int k = 0; k < NP; k++) {
      pa[k] = pb[k] = (uint32_t)n;
      pv[2 * k] = pv[2 * k + 1] = 0.0;
    }
    if (!rec) return;
    row = rec[WSR_ROW];
    if (row < (uint32_t)n) xrow = row;
    const int lev = rec[WSR_LEV];
    const uint16_t* q = pairs + 4 * (int)rec[WSR_PAIR];
#pragma unroll
    for (int k = 0; k < NP; k++)
      if (k < lev) {
        pa[k] = q[4 * k];
        pb[k] = q[4 * k + 2];
        pv[2 * k] = v[q[4 * k + 1]];
        pv[2 * k + 1] = v[q[4 * k + 3]];
      }
    ua = rec[WSR_UC0];
    ub = rec[WSR_UC1];
    uv0 = v[rec[WSR_US0]];
    uv1 = v[rec[WSR_US1]];
    dv = v[rec[WSR_DIAG]];
    const int nr = rec[WSR_NRHS], r0 = rec[WSR_RHS];
    if (nr > 0) {
      ra = codes[r0] >> 1;
      sa = (uint32_t)codes[r0] << 31;
    }
    if (nr > 1) {
      rb = codes[r0 + 1] >> 1;
      sb = (uint32_t)codes[r0 + 1] << 31;
    }
    if (nr > 2) rx = (uint32_t)(r0 + 2) | ((uint32_t)(nr - 2) << 16);
  }
};

// Both triangular solves of one system: x := (LU)^-1 b, or (TR) (LU)^-T b.
template <int NW, int R, bool TR>
struct WsSolve {
  static constexpr int TPS = 64 * NW;
  static constexpr int O = ws_cols(NW, R);  // krets columns per lane
  const uint16_t* codes;  // LDS list
  int n, nh, lane, w, nl, ntop, top_nl;
  bool more;
  double *x, *y, *hist, *sbuf, *td;
  uint32_t* ti;
  WsRow<ws_pairs(0)> r0;
  WsRow<ws_pairs(1)> r1;
  WsRow<ws_pairs(2)> r2;
  WsRow<ws_pairs(3)> r3;

  template <class F>
  __device__ __forceinline__ void each(F&& f) {
    f(r0, 0);
    if constexpr (R > 1) f(r1, 1);
    if constexpr (R > 2) f(r2, 2);
    if constexpr (R > 3) f(r3, 3);
  }

  // LDS carve-up and plan lists; returns the factors' place.
  __device__ __forceinline__ double* carve(const uint16_t* plan, char* smem) {
    const int t = threadIdx.x;
    const WsHdr* H = reinterpret_cast<const WsHdr*>(plan);
    lane = t & 63;
    w = __builtin_amdgcn_readfirstlane(t >> 6);
    n = H->n;
    nh = H->ndyn + H->nsrc;
    ntop = H->ntop;
    top_nl = H->top_nl;
    more = H->more != 0;
    uint16_t* q = reinterpret_cast<uint16_t*>(smem + 64);
    for (int i = t; i < H->nrhs; i += TPS) q[i] = plan[H->o_rhs + i];
    codes = q;
    const WsLds l = ws_lds(*H);
    x = reinterpret_cast<double*>(smem + 64 + ws_list_bytes(*H));
    y = x + l.y;
    hist = x + l.hist;
    sbuf = x + l.sbuf;
    td = x + l.top;
    ti = reinterpret_cast<uint32_t*>(td + WS_TOP_D * ntop);
    if (t == 0) x[H->nnz] = 0.0;  // the factors' zero entry
    return x;
  }

  // Stamps and factors the matrix into v (us: scratch); returns the
  // static-pivot guard's bound. flag: LDS status word, 28 free bytes after it.
  __device__ __forceinline__ double factorise(const PatDev& P, const double* prm, const double* eb, const TranArgs& ta,
                                              double* v, int* flag) {
    const int t = threadIdx.x;
    double* us = v + P.nnz + 1;
    StampArgs sa{AK_TRAN, 0.0, ta.h, ta.alpha, 0.0, -1, 0.0};
    unsigned long long* gw = reinterpret_cast<unsigned long long*>(flag + 2);  // ||A||, m, |||L||U|||
    if (t == 0) gw[0] = gw[1] = gw[2] = 0ull;
    stamp_matrix<double, double, TPS>(P, v, prm, eb, sa, nullptr, t, true);
    __syncthreads();
    double anp = 0.0;
    factor<double, TPS, true>(P, v, t, true, flag, &anp);
    __syncthreads();
    block_max_to(anp, &gw[0]);
    block_max_to(pivot_guard_rows<TPS>(P, v, us, t, true), &gw[1]);
    __syncthreads();
    block_max_to(pivot_guard_lu<TPS>(P, v, us, t, true), &gw[2]);
    __syncthreads();
    const double bnd = pivot_guard_bound(__longlong_as_double((long long)gw[2]), __longlong_as_double((long long)gw[0]),
                                         __longlong_as_double((long long)gw[1]));
    if (t == 0 && *flag == KG_OK && !(bnd <= KG_GUARD_STATIC)) *flag = KG_DECOMPOSITION;
    return bnd;
  }

  // Takes every lane's rows from the plan and the factors v, which the step's
  // arrays then overwrite. A barrier inside; the caller puts another before
  // the first step.
  __device__ __forceinline__ void rows(const uint16_t* plan, const double* v) {
    const WsHdr* H = reinterpret_cast<const WsHdr*>(plan);
    const uint16_t *pairs = plan + H->o_pair, *wr = plan + H->o_wave + w * WS_WAVE, *slot = plan + H->o_slot;
    const uint16_t* rh = plan + H->o_rhs;
    const int s0 = wr[WSW_S0], s1 = wr[WSW_S1], ytrash = n + H->npart + 2;
    nl = __builtin_amdgcn_readfirstlane((int)wr[WSW_NL]);
    each([&](auto& row, int r) __attribute__((always_inline)) {
      const int q = s0 + r * 64 + lane;
      row.take(q < s1 ? slot + q * WS_SLOT : nullptr, pairs, rh, v, n, ytrash, nh);
      if (TR && row.row > (uint32_t)n) row.dv = 1.0;  // partial sums are not divided
    });
    WsRow<WS_TOP_PAIRS> tp;
    const bool is_top = w == 0 && lane < ntop;
    const uint16_t* rec = plan + H->o_top + lane * WS_SLOT;
    if (NW > 1) tp.take(is_top ? rec : nullptr, pairs, rh, v, n, ytrash, nh);
    __syncthreads();  // every lane has its factors
    if (NW > 1 && is_top) {
      double* d = td + lane;
      uint32_t* q = ti + lane;
#pragma unroll
      for (int k = 0; k < WS_TOP_PAIRS; k++) {
        d[(2 * k) * ntop] = tp.pv[2 * k];
        d[(2 * k + 1) * ntop] = tp.pv[2 * k + 1];
        q[k * ntop] = tp.pa[k] | (tp.pb[k] << 16);
      }
      d[(2 * WS_TOP_PAIRS) * ntop] = tp.uv0;
      d[(2 * WS_TOP_PAIRS + 1) * ntop] = tp.uv1;
      d[(2 * WS_TOP_PAIRS + 2) * ntop] = tp.dv;
      q += WS_TOP_PAIRS * ntop;
      q[0] = tp.ua | (tp.ub << 16);
      q[ntop] = tp.ra | (tp.rb << 16);
      q[2 * ntop] = (tp.sa >> 31) | (tp.sb >> 30);
      q[3 * ntop] = tp.row | ((uint32_t)rec[WSR_COL] << 16);
      q[4 * ntop] = (uint32_t)rec[WSR_PART] | ((uint32_t)rec[WSR_NPART] << 16);
      q[5 * ntop] = tp.rx;
    }
    if (threadIdx.x == 0) x[n] = y[n] = y[ytrash - 1] = hist[nh] = 0.0;
  }

  __device__ __forceinline__ double more_rhs(uint32_t rx) const {
    double a = 0.0;
    for (uint32_t k = rx & 0xFFFF, e = k + (rx >> 16); k < e; k++)
      a += flip(hist[codes[k] >> 1], (uint32_t)codes[k] << 31);
    return a;
  }
  // Lower level L on, within the wave.
  template <int L>
  __device__ __forceinline__ void lower() {
    if constexpr (L < ws_pairs(0)) {
      if (L >= nl) return;
      double a[R], b[R];
      each([&](auto& q, int r) __attribute__((always_inline)) {
        if constexpr (L < std::remove_reference_t<decltype(q)>::NP) {
          a[r] = y[q.pa[L]];
          b[r] = y[q.pb[L]];
        }
      });
      each([&](auto& q, int r) __attribute__((always_inline)) {
        if constexpr (L < std::remove_reference_t<decltype(q)>::NP) {
          q.acc -= q.pv[2 * L] * a[r];
          q.acc -= q.pv[2 * L + 1] * b[r];
          y[q.row] = TR ? q.acc * q.dv : q.acc;
        }
      });
      wave_sync();
      lower<L + 1>();
    }
  }
  // Upper level L and below, within the wave.
  template <int L>
  __device__ __forceinline__ void upper() {
    if constexpr (L >= 0) {
      if (L <= nl) {
        double a[R], b[R];
        each([&](auto& q, int r) __attribute__((always_inline)) {
          if constexpr (L <= std::remove_reference_t<decltype(q)>::NP) {
            a[r] = x[q.ua];
            b[r] = x[q.ub];
          }
        });
        each([&](auto& q, int r) __attribute__((always_inline)) {
          if constexpr (L <= std::remove_reference_t<decltype(q)>::NP) {
            const double t = q.acc - q.uv0 * a[r] - q.uv1 * b[r];
            x[q.xrow] = TR ? t : t * q.dv;  // the diagonal holds its reciprocal
          }
        });
        wave_sync();
      }
      upper<L - 1>();
    }
  }
  // The top rows, by wave 0 (lanes past the last repeat it): right-hand sides
  // (add: what a row has besides its histories), the waves' partials and both
  // solves. Returns the lane's solution; row, col: its row and krets column.
  template <int L>
  __device__ __forceinline__ void top_lower(double& acc, double dv, const double* pv, const uint32_t* pc,
                                            uint32_t row) {
    if constexpr (L < WS_TOP_PAIRS) {
      if (L >= top_nl) return;
      acc -= pv[2 * L] * y[pc[L] & 0xFFFF];
      acc -= pv[2 * L + 1] * y[pc[L] >> 16];
      y[row] = TR ? acc * dv : acc;
      wave_sync();
      top_lower<L + 1>(acc, dv, pv, pc, row);
    }
  }
  __device__ __forceinline__ double top(double add, uint32_t* row, uint32_t* col) {
    int l = min(lane, ntop - 1);
    asm volatile("" : "+v"(l));  // the addresses below are formed here, not kept in registers by every wave
    const double* d = td + l;
    const uint32_t* q = ti + l;
    double pv[2 * WS_TOP_PAIRS];
    uint32_t pc[WS_TOP_PAIRS];
#pragma unroll
    for (int k = 0; k < WS_TOP_PAIRS; k++) {
      pv[2 * k] = d[(2 * k) * ntop];
      pv[2 * k + 1] = d[(2 * k + 1) * ntop];
      pc[k] = q[k * ntop];
    }
    const double uv0 = d[(2 * WS_TOP_PAIRS) * ntop], uv1 = d[(2 * WS_TOP_PAIRS + 1) * ntop];
    const double dv = d[(2 * WS_TOP_PAIRS + 2) * ntop];
    q += WS_TOP_PAIRS * ntop;
    const uint32_t uc = q[0], rw = q[3 * ntop], pp = q[4 * ntop], pn = pp >> 16;
    *row = rw & 0xFFFF;
    *col = rw >> 16;
    const double* part = y + n + 1 + (pp & 0xFFFF);
    double acc = add + top_hist(l);
    for (uint32_t k = 0; k < pn; k++) acc += part[k];
    y[*row] = TR ? acc * dv : acc;
    wave_sync();
    top_lower<0>(acc, dv, pv, pc, *row);
    if (TR) acc *= dv;
    double xv = 0.0;
    for (int lv = top_nl; lv >= 0; lv--) {
      const double t = acc - uv0 * x[uc & 0xFFFF] - uv1 * x[uc >> 16];
      xv = TR ? t : t * dv;
      x[*row] = xv;
      wave_sync();
    }
    return xv;
  }
  // the histories of top row l
  __device__ __forceinline__ double top_hist(int l) const {
    const uint32_t* q = ti + WS_TOP_PAIRS * ntop + l;
    const uint32_t rc = q[ntop], sg = q[2 * ntop];
    double a = flip(hist[rc & 0xFFFF], (sg & 1u) << 31) + flip(hist[rc >> 16], (sg & 2u) << 30);
    if (more) a += more_rhs(q[5 * ntop]);
    return a;
  }

  // The solve, from the histories; every row's right-hand side is init(r)
  // more. at_top(): wave 0 solves the top; between(): what the other waves do
  // meanwhile (they may still read the solution before, except its top rows).
  template <class I, class T, class F>
  __device__ __forceinline__ void solve(I&& init, T&& at_top, F&& between) {
    each([&](auto& q, int r) __attribute__((always_inline)) {
      q.acc = init(r, flip(hist[q.ra], q.sa) + flip(hist[q.rb], q.sb));
    });
    if (more) each([&](auto& q, int) __attribute__((always_inline)) { q.acc += more_rhs(q.rx); });
    each([&](auto& q, int) __attribute__((always_inline)) { y[q.row] = TR ? q.acc * q.dv : q.acc; });
    wave_sync();
    lower<0>();
    if (TR) each([&](auto& q, int) __attribute__((always_inline)) { q.acc *= q.dv; });
    if constexpr (NW > 1) __syncthreads();
    if (NW > 1 && w == 0 && ntop) at_top();
    if (NW == 1 || w > 0) between();
    if constexpr (NW > 1) __syncthreads();
    upper<ws_pairs(0)>();
  }
};

// The transient's step loop around the solve.
template <int NW, int R, int E>
struct WsSys : WsSolve<NW, R, false> {
  using S = WsSolve<NW, R, false>;
  using S::TPS, S::O, S::n, S::nh, S::lane, S::w, S::ntop, S::x, S::hist, S::sbuf;
  int ndyn, ntel, nsteps, nst1;
  bool with_state;
  double* tab;
  // a companion element: its unknowns, history and whether it is a capacitor
  struct Elem {
    uint32_t p, m, c, h;
    bool cap;
    double cf, ed, vo;
  };
  Elem el[E], tel;      // tel (wave 0): an element that several waves touch
  int nv, vhist, vsrc;  // this wave's sources; this lane's history and source
  int oc[O];            // rows of this lane's krets columns, -1: none

  // Source values of every step (global table; complete after a barrier).
  __device__ __forceinline__ void tabulate(const PatDev& P, const double* prm, const TranArgs& ta, double* srcv,
                                           int nsrc_max, int inst) {
    nsteps = ta.nsteps;
    nst1 = ta.nsteps + 1;
    tab = srcv ? srcv + (int64_t)inst * nsrc_max * nst1 : nullptr;
    const LinHdr* lh = reinterpret_cast<const LinHdr*>(P.lin);
    const uint16_t* src = P.lin + lh->o_src;
    const bool compat = ta.method == KG_BE_COMPAT;
    for (int i = threadIdx.x; i < lh->nsrc * nst1; i += TPS) {
      const int si = i / nst1, s = i - si * nst1;
      const double tn = (double)s * ta.h, tprev = (double)(s - 1) * ta.h;
      const double tsrc = compat ? tprev : tn;  // krets evaluates sources at the guess's time
      const double* pe = prm + (int)src[si * LIN_SRC + 1] * KG_NPARAM;
      tab[i] = s == 0 ? 0.0 : (src[si * LIN_SRC] == KG_V ? wave_value(pe, tsrc) : pe[0]);
    }
  }

  // Takes every lane's rows, elements and sources; x0 (krets numbering,
  // cpos_all its rows) becomes the solution before the first step. Barriers
  // inside.
  __device__ __forceinline__ void take(const uint16_t* plan, const double* v, const double* prm, const TranArgs& ta,
                                       const uint16_t* cpos_all, const double* x0) {
    const WsHdr* H = reinterpret_cast<const WsHdr*>(plan);
    const uint16_t *wr = plan + H->o_wave + w * WS_WAVE, *er = plan + H->o_elem, *cp = plan + H->o_cpos;
    const uint16_t* sr = plan + H->o_src;
    const int e0 = wr[WSW_E0], e1 = wr[WSW_E1], v0 = wr[WSW_V0];
    ndyn = H->ndyn;
    ntel = H->ntel;
    with_state = ta.alpha != 1.0;
    nv = __builtin_amdgcn_readfirstlane((int)wr[WSW_V1]) - v0;
    vhist = lane < nv ? (int)sr[(v0 + lane) * WS_SRC] : -1;
    vsrc = lane < nv ? (int)sr[(v0 + lane) * WS_SRC + 1] : 0;
#pragma unroll
    for (int r = 0; r < E; r++) {
      const int q = e0 + r * 64 + lane;
      element(q < e1 ? er + q * WS_ELEM : nullptr, prm, ta, el[r]);
    }
    const int last = plan[H->o_wave + (NW - 1) * WS_WAVE + WSW_E1];
    element(w == 0 && lane < ntel ? er + (last + lane) * WS_ELEM : nullptr, prm, ta, tel);
    const int ow = NW == 1 ? 0 : w - 1;
#pragma unroll
    for (int k = 0; k < O; k++) {
      const int j = lane + 64 * (ow + k * (NW == 1 ? 1 : NW - 1));
      oc[k] = ow >= 0 && j < n && cp[j] < n ? (int)cp[j] : -1;
    }
    S::rows(plan, v);
    for (int j = threadIdx.x; j < n; j += TPS) x[cpos_all[j]] = x0[j];
    __syncthreads();
  }
  __device__ __forceinline__ void element(const uint16_t* e, const double* prm, const TranArgs& ta, Elem& q) {
    q.p = q.m = q.c = (uint32_t)n;
    q.h = (uint32_t)nh + 1;  // never read
    q.cap = false;
    q.cf = q.ed = q.vo = 0.0;
    if (!e) return;
    q.p = e[WSE_P];
    q.m = e[WSE_M];
    q.c = e[WSE_C];
    q.h = e[WSE_HIST];
    q.cap = e[WSE_KIND] == 1;
    q.cf = ta.alpha * (prm[(int)e[WSE_E] * KG_NPARAM] / ta.h);
  }

  // History of the step after the solution in x: a capacitor's companion
  // current -(alpha C/h) v - i, an inductor's -(alpha L/h) i - v (the state
  // terms for the trapezoidal rule only). first: x is the initial state
  // (capacitor currents 0).
  __device__ __forceinline__ void companion(Elem& q, bool first) {
    const double vn = x[q.p] - x[q.m], xb = x[q.c];
    double ieq = -q.cf * (q.cap ? vn : xb);
    if (with_state) {
      const double e = q.cf * (vn - q.vo) - q.ed;  // 2C/h == alpha C/h for alpha = 2
      q.ed = first ? 0.0 : e;
      q.vo = vn;
      ieq -= q.cap ? q.ed : vn;
    }
    hist[q.h] = ieq;
  }
  // Histories of step s from the solution before it: this wave's elements and
  // sources. Source values come from the table 64 steps at a time (a table
  // read per step would cost its latency in every step).
  __device__ __forceinline__ void update(int s, bool first) {
#pragma unroll
    for (int r = 0; r < E; r++) companion(el[r], first);
    if (nv) {
      if (first || (s & 63) == 0) {
        const int s0 = (s & ~63) + lane;
        for (int k = 0; k < nv; k++) {
          const int src = __shfl(vsrc, k);
          sbuf[64 * src + lane] = s0 <= nsteps ? tab[(int64_t)src * nst1 + s0] : 0.0;
        }
        wave_sync();
      }
      if (vhist >= 0) hist[vhist] = sbuf[64 * vsrc + (s & 63)];
    }
  }

  // The solution's rows below the top to o (krets numbering), by the waves
  // that do not solve the top; OBJ: returns sum_j c_j x_j over them.
  template <bool OBJ>
  __device__ __forceinline__ double store(double* o, const double* c) const {
    const int j = lane + 64 * (NW == 1 ? 0 : w - 1), stride = 64 * (NW == 1 ? 1 : NW - 1);
    double a = 0.0;
#pragma unroll
    for (int k = 0; k < O; k++)
      if (oc[k] >= 0) {
        const double xv = x[oc[k]];
        o[j + k * stride] = xv;
        if (OBJ) a += c[k] * xv;
      }
    return a;
  }
};

// Fixed-step linear transient (k_tran semantics, FP64). ws: each instance's
// wave-subtree plan (nw == NW, rows <= R, elems <= E). OBJ: the discrete
// adjoint's forward pass: out is the trajectory ([instance][nsteps + 1][n],
// krets numbering, at out_off as a transient's), and Jout receives sum_s w_s
// c.x_s (trapezoid weights).
template <int NW, int R, int E, bool OBJ>
__global__ void __launch_bounds__(64 * NW) k_tran_ws(BatchDev B, int kind_slot, const uint16_t* const* ws, TranArgs ta,
                                                     const double* xop, const int64_t* xop_off, double* out,
                                                     const int64_t* out_off, int32_t* status, int32_t* iters,
                                                     double* err, double* srcv, int nsrc_max, const double* cvec,
                                                     double* Jout) {
  extern __shared__ __align__(16) char smem[];
  const int t = threadIdx.x;
  const int nslot = B.inst_list ? B.n_list : B.n_instances;
  const int64_t slot = xcd_block();
  if (slot >= nslot) return;
  const int inst = B.inst_list ? B.inst_list[slot] : (int)slot;
  const PatDev& P = B.pats[B.inst_pat[kind_slot * B.n_instances + inst]];
  if (status[inst] != KG_OK) {  // failed operating point or no plan: nothing to integrate
    if (t == 0 && err) err[inst] = 0.0;
    return;
  }
  const uint16_t* plan = ws[inst];
  const WsHdr* H = reinterpret_cast<const WsHdr*>(plan);
  if (plan == nullptr || H->nw != NW || H->rows > R || H->elems > E || (srcv == nullptr && nsrc_max > 0)) {
    if (t == 0) status[inst] = KG_UNEXPECTED;  // launched only where it fits
    return;
  }
  WsSys<NW, R, E> S;
  int* flags = reinterpret_cast<int*>(smem);
  double* v = S.carve(plan, smem);
  if (t == 0) flags[0] = KG_OK;
  __syncthreads();
  const double* prm = B.params + B.eoff[inst] * KG_NPARAM;
  S.tabulate(P, prm, ta, srcv, nsrc_max, inst);
  const double bnd = S.factorise(P, prm, B.ebase + B.eoff[inst], ta, v, &flags[0]);
  const double* x0 = xop + xop_off[inst];
  double* o = out + out_off[inst];
  for (int j = t; j < S.n; j += 64 * NW) o[j] = x0[j];
  int32_t* its = iters ? iters + (int64_t)inst * (ta.nsteps + 1) : nullptr;
  if (t == 0 && its) its[0] = 0;
  __syncthreads();
  if (flags[0] != KG_OK) {
    if (t == 0) {
      status[inst] = flags[0];
      if (err) err[inst] = bnd;
    }
    return;
  }
  if (its)
    for (int s = 1 + t; s <= ta.nsteps; s += 64 * NW) its[s] = 1;
  S.take(plan, v, prm, ta, P.lin + reinterpret_cast<const LinHdr*>(P.lin)->o_cpos, x0);
  S.update(1, true);
  double cv[OBJ ? S.O : 1], jsum = 0.0, ctop = 0.0;  // cv: this lane's columns; ctop: its top row's
  if constexpr (OBJ) {
#pragma unroll
    for (int k = 0; k < S.O; k++) {
      const int j = S.lane + 64 * ((NW == 1 ? 0 : S.w - 1) + k * (NW == 1 ? 1 : NW - 1));
      cv[k] = S.oc[k] >= 0 ? cvec[j] : 0.0;
    }
    if (S.w == 0 && S.lane < S.ntop) ctop = cvec[plan[H->o_top + S.lane * WS_SLOT + WSR_COL]];
    for (int j = t; j < S.n; j += 64 * NW) jsum += 0.5 * ta.h * cvec[j] * x0[j];
  }
  wave_sync();
  for (int s = 1; s <= ta.nsteps; s++) {
    S.solve([](int, double b) __attribute__((always_inline)) { return b; },
            [&]() __attribute__((always_inline)) {
              if (S.ntel) {
                S.companion(S.tel, s == 1);
                wave_sync();
              }
              uint32_t row, col;
              const double xv = S.top(0.0, &row, &col);
              o[(int64_t)s * S.n + col] = xv;
              if (OBJ) jsum += (s == ta.nsteps ? 0.5 * ta.h : ta.h) * ctop * xv;
            },
            [&]() __attribute__((always_inline)) {
              if (s == 1) return;
              const double a = S.template store<OBJ>(o + (int64_t)(s - 1) * S.n, cv);
              if (OBJ) jsum += ta.h * a;
            });
    S.update(s + 1, false);
    wave_sync();
  }
  if (ta.nsteps > 0) {
    __syncthreads();
    if (NW == 1 || S.w > 0) {
      const double a = S.template store<OBJ>(o + (int64_t)ta.nsteps * S.n, cv);
      if (OBJ) jsum += 0.5 * ta.h * a;
    }
  }
  if constexpr (OBJ) {
    for (int k = 32; k > 0; k >>= 1) jsum += __shfl_xor(jsum, k);
    __syncthreads();
    if (S.lane == 0) S.y[S.w] = jsum;
    __syncthreads();
    if (t == 0) {
      for (int k = 1; k < NW; k++) jsum += S.y[k];
      Jout[inst] = jsum;
    }
  }
  if (t == 0) {
    status[inst] = flags[0];
    if (err) err[inst] = bnd;
  }
}

// Backward pass of the discrete adjoint of a linear transient (k_adj_bwd
// semantics, FP64) over the stored trajectory ([instance][nsteps + 1][n],
// krets numbering, traj_stride per instance), by wave subtrees of the
// transposed factors. Per step: the adjoint loads (the objective's weight and
// the histories of the elements' adjoint states), lambda = A^-T load, then
// every element's share, in its own lane's registers: with z = (the
// difference of lambda across it) - (its adjoint state), a capacitor's
// gradient takes z (alpha/h) (d0 - d1) of its voltages at both ends of the
// step, its adjoint state becomes z and its load on the step before is
// alpha C/h (z + state); an inductor's take -z and the load -alpha L/h z on
// its branch; a resistor's z d1 / R^2. States are read one step ahead, a row
// of the trajectory at a time, through LDS. Bound by the same levels as the
// transient: 1.6 us a step at 202 unknowns and 401 elements, where the
// LDS-resident pass (atomic adjoint loads, block barriers) took 5.2 us, after
// 1.3 us a step of recomputation. xbar0 receives dJ/dx_0 for the
// operating-point term; grad: [instance][ne].
template <int NW, int R, int E>
__global__ void __launch_bounds__(64 * NW) k_adj_ws_bwd(BatchDev B, int kind_slot, const uint16_t* const* ws,
                                                        TranArgs ta, const double* cvec, const double* traj,
                                                        int64_t traj_stride, double* grad, int64_t grad_stride,
                                                        double* xbar0, const int64_t* xop_off, int32_t* status) {
  extern __shared__ __align__(16) char smem[];
  constexpr int TPS = 64 * NW;
  const int t = threadIdx.x, inst = (int)xcd_block();
  if (inst >= B.n_instances || status[inst] != KG_OK) return;
  const PatDev& P = B.pats[B.inst_pat[kind_slot * B.n_instances + inst]];
  const uint16_t* plan = ws[inst];
  const WsHdr* H = reinterpret_cast<const WsHdr*>(plan);
  if (plan == nullptr || !H->adjoint || H->nw != NW || H->rows > R || H->elems > E) {
    if (t == 0) status[inst] = KG_UNEXPECTED;  // launched only where it fits
    return;
  }
  WsSolve<NW, R, true> S;
  int* flags = reinterpret_cast<int*>(smem);
  double* v = S.carve(plan, smem);
  if (t == 0) flags[0] = KG_OK;
  __syncthreads();
  const double* prm = B.params + B.eoff[inst] * KG_NPARAM;
  S.factorise(P, prm, B.ebase + B.eoff[inst], ta, v, &flags[0]);
  double* g = grad + (int64_t)inst * grad_stride;
  for (int e = t; e < P.ne; e += TPS) g[e] = 0.0;
  __syncthreads();
  if (flags[0] != KG_OK) {
    if (t == 0) status[inst] = flags[0];
    return;
  }
  S.rows(plan, v);
  const int n = S.n, lane = S.lane, w = S.w, N = ta.nsteps;
  const bool trap = ta.alpha != 1.0;
  const double h = ta.h, ah = ta.alpha / ta.h;
  // objective coefficients of this lane's rows and top row
  double cr[R], ctop = 0.0;
  int rcol[R], tcol = -1;
  {
    const uint16_t* wr = plan + H->o_wave + w * WS_WAVE;
#pragma unroll
    for (int r = 0; r < R; r++) {
      const int q = (int)wr[WSW_S0] + r * 64 + lane;
      const uint16_t* rec = plan + H->o_slot + q * WS_SLOT;
      rcol[r] = q < (int)wr[WSW_S1] && rec[WSR_ROW] < n ? (int)rec[WSR_COL] : -1;
      cr[r] = rcol[r] >= 0 ? cvec[rcol[r]] : 0.0;
    }
    if (NW > 1 && w == 0 && S.ntop) {
      tcol = plan[H->o_top + min(lane, S.ntop - 1) * WS_SLOT + WSR_COL];
      ctop = cvec[tcol];
    }
  }
  // elements
  struct Elem {
    uint32_t a, b, p, m, h1, h2;
    bool cap;
    double f1, f2, a1, a0, sb, d1, gr;
    int e;
  } el[E];
  double* X = S.sbuf;  // two rows of the trajectory, n + 1 each
  const double* tr = traj + (int64_t)inst * traj_stride;
  for (int j = t; j < n; j += TPS) {
    X[(N & 1) * (n + 1) + j] = tr[(int64_t)N * n + j];
    X[((N - 1) & 1) * (n + 1) + j] = tr[(int64_t)(N - 1) * n + j];
  }
  if (t < 2) X[t * (n + 1) + n] = 0.0;
  for (int k = t; k < S.nh + 2; k += TPS) S.hist[k] = 0.0;
  __syncthreads();
  {
    const uint16_t *wr = plan + H->o_wave + w * WS_WAVE, *er = plan + H->o_elem;
    const double* X1 = X + (N & 1) * (n + 1);
#pragma unroll
    for (int r = 0; r < E; r++) {
      const int q = (int)wr[WSW_E0] + r * 64 + lane;
      Elem& q_ = el[r];
      q_.a = q_.b = q_.p = q_.m = (uint32_t)n;
      q_.h1 = q_.h2 = (uint32_t)S.nh + 1;
      q_.cap = false;
      q_.f1 = q_.f2 = q_.a1 = q_.a0 = q_.sb = q_.d1 = q_.gr = 0.0;
      q_.e = -1;
      if (q < (int)wr[WSW_E1]) {
        const uint16_t* rec = er + q * WS_AELEM;
        const int kind = rec[WSA_KIND];
        const double val = prm[(int)rec[WSA_E] * KG_NPARAM], cf = ta.alpha * (val / h);
        q_.a = rec[WSA_A], q_.b = rec[WSA_B], q_.p = rec[WSA_P], q_.m = rec[WSA_M];
        q_.h1 = rec[WSA_H1], q_.h2 = rec[WSA_H2];
        q_.cap = kind == 1;
        if (kind == 0) q_.a1 = 1.0 / (val * val);
        if (kind == 1) q_.f1 = trap ? 2.0 * cf : cf, q_.a1 = -ah, q_.a0 = ah;
        if (kind == 2) q_.f1 = trap ? -1.0 : 0.0, q_.f2 = -cf, q_.a1 = ah, q_.a0 = -ah;
        if (rec[WSA_GRAD]) q_.e = rec[WSA_E];
        q_.d1 = X1[q_.p] - X1[q_.m];
      }
    }
  }
  __syncthreads();
  // rows of the trajectory ahead of their step: columns of the waves that do not solve the top
  const int j0 = lane + 64 * (NW == 1 ? 0 : w - 1), js = 64 * (NW == 1 ? 1 : NW - 1);
  double pre[S.O];
  auto fetch = [&](int s) __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < S.O; k++) {
      const int j = j0 + k * js;
      pre[k] = s >= 0 && j0 >= 0 && j < n ? tr[(int64_t)s * n + j] : 0.0;
    }
  };
  fetch(N - 2);
  for (int s = N - 1; s >= 0; s--) {
    const double wt = s + 1 == N ? 0.5 * h : h;
    S.solve([&](int r, double b) __attribute__((always_inline)) { return wt * cr[r] + b; },
            [&]() __attribute__((always_inline)) {
              uint32_t row, col;
              S.top(wt * ctop, &row, &col);
            },
            [&]() __attribute__((always_inline)) {
              if (s == 0) return;
              double* Xn = X + ((s - 1) & 1) * (n + 1);
#pragma unroll
              for (int k = 0; k < S.O; k++)
                if (j0 + k * js < n) Xn[j0 + k * js] = pre[k];
              fetch(s - 2);
            });
    const double* Xs = X + (s & 1) * (n + 1);
#pragma unroll
    for (int r = 0; r < E; r++) {
      Elem& q = el[r];
      const double z = S.x[q.a] - S.x[q.b] - q.sb, d0 = Xs[q.p] - Xs[q.m];
      q.gr += z * (q.a1 * q.d1 + q.a0 * d0);
      if (s == 0 && q.cap && trap) q.f1 *= 0.5;  // no state before the first step
      S.hist[q.h1] = z * q.f1;
      S.hist[q.h2] = z * q.f2;
      if (trap && q.cap) q.sb = z;
      q.d1 = d0;
    }
    wave_sync();
  }
#pragma unroll
  for (int r = 0; r < E; r++)
    if (el[r].e >= 0) g[el[r].e] = el[r].gr;
  // dJ/dx_0: the loads that the first step leaves
  double* xo = xbar0 + xop_off[inst];
  S.each([&](auto& q, int r) __attribute__((always_inline)) {
    double b = 0.5 * h * cr[r] + flip(S.hist[q.ra], q.sa) + flip(S.hist[q.rb], q.sb);
    if (S.more) b += S.more_rhs(q.rx);
    if (rcol[r] >= 0) xo[rcol[r]] = b;
  });
  __syncthreads();
  if (tcol >= 0) xo[tcol] = 0.5 * h * ctop + S.top_hist(min(lane, S.ntop - 1));
  if (t == 0) status[inst] = flags[0];
}

template <class K, class... Args>
hipError_t launch(K fn, dim3 g, dim3 b, size_t lds, hipStream_t st, Args... args) {
  hipError_t e = hipFuncSetAttribute((const void*)fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(fn, g, b, lds, st, args...);
  return hipGetLastError();
}

}  // namespace

// Compiled (waves, rows, elements per lane); more registers per lane than a
// block of so many waves may have would spill.
#define KG_WS_SHAPES(X)                                                        \
  X(1, 1, 1) X(1, 2, 2) X(1, 4, 4) X(2, 1, 1) X(2, 2, 2) X(2, 4, 3) X(2, 4, 4) \
  X(4, 1, 1) X(4, 2, 2) X(4, 4, 3) X(4, 4, 4) X(8, 1, 1) X(8, 2, 2) X(8, 4, 3)
#define KG_WS_ADJ_SHAPES(X)                                                    \
  X(1, 1, 2) X(1, 2, 4) X(1, 4, 7) X(2, 1, 2) X(2, 2, 4) X(2, 4, 7)            \
  X(4, 1, 2) X(4, 2, 4) X(4, 4, 7) X(8, 1, 2) X(8, 2, 4)

bool ws_round(int nw, bool adjoint, int* r, int* e) {
#define KG_WS(NW, RR, EE)                 \
  if (nw == NW && *r <= RR && *e <= EE) { \
    *r = RR, *e = EE;                     \
    return true;                          \
  }
  if (adjoint) {
    KG_WS_ADJ_SHAPES(KG_WS)
  } else {
    KG_WS_SHAPES(KG_WS)
  }
#undef KG_WS
  return false;
}

hipError_t run_tran_ws(int nw, int r, int e, dim3 g, size_t lds, hipStream_t st, BatchDev B, int kind_slot,
                       const uint16_t* const* ws, TranArgs ta, const double* xop, const int64_t* xop_off, double* out,
                       const int64_t* out_off, int32_t* status, int32_t* iters, double* err, double* srcv,
                       int nsrc_max, const double* cvec, double* Jout) {
#define KG_WS(NW, RR, EE)                                                                                           \
  if (nw == NW && r == RR && e == EE)                                                                               \
    return cvec ? launch(k_tran_ws<NW, RR, EE, true>, g, dim3(64 * NW), lds, st, B, kind_slot, ws, ta, xop, xop_off, \
                         out, out_off, status, iters, err, srcv, nsrc_max, cvec, Jout)                              \
                : launch(k_tran_ws<NW, RR, EE, false>, g, dim3(64 * NW), lds, st, B, kind_slot, ws, ta, xop,        \
                         xop_off, out, out_off, status, iters, err, srcv, nsrc_max, cvec, Jout);
  KG_WS_SHAPES(KG_WS)
#undef KG_WS
  return hipErrorInvalidValue;
}

hipError_t run_adj_ws_bwd(int nw, int r, int e, dim3 g, size_t lds, hipStream_t st, BatchDev B, int kind_slot,
                          const uint16_t* const* ws, TranArgs ta, const double* cvec, const double* traj,
                          int64_t traj_stride, double* grad, int64_t grad_stride, double* xbar0,
                          const int64_t* xop_off, int32_t* status) {
#define KG_WS(NW, RR, EE)                                                                                         \
  if (nw == NW && r == RR && e == EE)                                                                             \
    return launch(k_adj_ws_bwd<NW, RR, EE>, g, dim3(64 * NW), lds, st, B, kind_slot, ws, ta, cvec, traj,          \
                  traj_stride, grad, grad_stride, xbar0, xop_off, status);
  KG_WS_ADJ_SHAPES(KG_WS)
#undef KG_WS
  return hipErrorInvalidValue;
}

}  // namespace kg
