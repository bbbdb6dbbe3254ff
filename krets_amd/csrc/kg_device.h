// Device helpers of the gfx950 kernels: scalar types, device models, stamps,
// the level-scheduled factorisation and solves, and the accuracy guards.
#pragma once
#include <hip/hip_runtime.h>

#include <cfloat>
#include <cmath>
#include <cstdint>

#include "kg_launch.h"

namespace kg {

// ------------------------------------------------------------ scalar types
template <class R>
struct cplx {
  R re, im;
};
using c64 = cplx<float>;
using c128 = cplx<double>;

template <class R>
__device__ __forceinline__ cplx<R> operator+(cplx<R> a, cplx<R> b) { return {a.re + b.re, a.im + b.im}; }
template <class R>
__device__ __forceinline__ cplx<R> operator-(cplx<R> a, cplx<R> b) { return {a.re - b.re, a.im - b.im}; }
template <class R>
__device__ __forceinline__ cplx<R> operator-(cplx<R> a) { return {-a.re, -a.im}; }
template <class R>
__device__ __forceinline__ cplx<R> operator*(cplx<R> a, cplx<R> b) {
  return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re};
}
template <class R>
__device__ __forceinline__ cplx<R> operator*(R s, cplx<R> a) { return {s * a.re, s * a.im}; }
template <class R>
__device__ __forceinline__ cplx<R>& operator+=(cplx<R>& a, cplx<R> b) { a = a + b; return a; }
template <class R>
__device__ __forceinline__ cplx<R>& operator-=(cplx<R>& a, cplx<R> b) { a = a - b; return a; }

template <class S> struct Traits;
template <> struct Traits<double> { using R = double; static constexpr bool cx = false; };
template <> struct Traits<float> { using R = float; static constexpr bool cx = false; };
template <> struct Traits<c128> { using R = double; static constexpr bool cx = true; };
template <> struct Traits<c64> { using R = float; static constexpr bool cx = true; };

template <class S> __device__ __forceinline__ S mk(double re, double im);
template <> __device__ __forceinline__ double mk<double>(double re, double) { return re; }
template <> __device__ __forceinline__ float mk<float>(double re, double) { return (float)re; }
template <> __device__ __forceinline__ c128 mk<c128>(double re, double im) { return {re, im}; }
template <> __device__ __forceinline__ c64 mk<c64>(double re, double im) { return {(float)re, (float)im}; }

__device__ __forceinline__ double re_of(double a) { return a; }
__device__ __forceinline__ double re_of(float a) { return a; }
__device__ __forceinline__ double re_of(c128 a) { return a.re; }
__device__ __forceinline__ double re_of(c64 a) { return a.re; }
__device__ __forceinline__ double im_of(double) { return 0.0; }
__device__ __forceinline__ double im_of(float) { return 0.0; }
__device__ __forceinline__ double im_of(c128 a) { return a.im; }
__device__ __forceinline__ double im_of(c64 a) { return a.im; }

template <class D, class S>
__device__ __forceinline__ D cvt(S a) { return mk<D>(re_of(a), im_of(a)); }

// modulus used for pivot checks and norms
__device__ __forceinline__ double absv(double a) { return fabs(a); }
__device__ __forceinline__ double absv(float a) { return fabsf(a); }
__device__ __forceinline__ double absv(c128 a) { return sqrt(a.re * a.re + a.im * a.im); }
__device__ __forceinline__ double absv(c64 a) { return sqrt((double)a.re * a.re + (double)a.im * a.im); }

// reciprocal; complex via Smith's scaled division
__device__ __forceinline__ double rcp(double a) { return 1.0 / a; }
__device__ __forceinline__ float rcp(float a) { return 1.0f / a; }
template <class R>
__device__ __forceinline__ cplx<R> rcp(cplx<R> b) {
  if (fabs(b.re) >= fabs(b.im)) {
    R r = b.im / b.re, d = b.re + b.im * r;
    return {R(1) / d, -r / d};
  }
  R r = b.re / b.im, d = b.re * r + b.im;
  return {r / d, R(-1) / d};
}
__device__ __forceinline__ bool finite_v(double a) { return isfinite(a); }
__device__ __forceinline__ bool finite_v(float a) { return isfinite(a); }
template <class R>
__device__ __forceinline__ bool finite_v(cplx<R> a) { return isfinite(a.re) && isfinite(a.im); }
__device__ __forceinline__ double scal(double s, double a) { return s * a; }
__device__ __forceinline__ c128 scal(double s, c128 a) { return {s * a.re, s * a.im}; }

// ------------------------------------------------------- device maths
// constants.rs:1-4
__device__ constexpr double KG_VT = 1.380649e-23 * 300.0 / 1.602176634e-19;
__device__ constexpr double KG_PI = 3.14159265358979323846;

// Pulse::value_at / Sinusoidal::value_at (voltage_source.rs:50-93) and
// transient_value_at (243-252).
__device__ double wave_value(const double* p, double t) {
  int kind = (int)p[2];
  const double* w = p + 3;
  if (kind == KG_WAVE_PULSE) {
    double v1 = w[0], v2 = w[1], td = w[2], tr = w[3], tf = w[4], pw = w[5], per = w[6];
    if (t < td) return v1;
    double tt = fmod(t - td, per);
    if (tt < tr) return v1 + (v2 - v1) * (tt / tr);
    if (tt < tr + pw) return v2;
    if (tt < tr + pw + tf) return v2 + (v1 - v2) * ((tt - tr - pw) / tf);
    return v1;
  }
  if (kind == KG_WAVE_SIN) {
    double vo = w[0], va = w[1], f = w[2], td = w[3], th = w[4], ph = w[5];
    if (t < td) return vo;
    double om = 2.0 * KG_PI * f;
    double phr = ph * (KG_PI / 180.0);
    double tt = t - td;
    return vo + va * exp(-th * tt) * sin(om * tt + phr);
  }
  return p[0];
}

// Diode companion (elements/diode.rs:24-71). compat: krets' semantics, where
// the exponent limit is n*Vt*ln(DBL_MAX*n*Vt/Is) (infinite for any practical
// Is) and Ieq uses the unlimited voltage. clean: SPICE3 pnjlim on the
// junction voltage against the previous iterate, consistent linearisation.
struct DiodeLin {
  double g, ieq, vd;
  bool limited;
};
__device__ DiodeLin diode_eval(double vd, double is, double n, bool compat, double vold) {
  double nvt = n * KG_VT;
  DiodeLin r;
  r.limited = false;
  if (compat) {
    double vcrit = nvt * log(DBL_MAX * n * KG_VT / is);
    double vl = fmin(fmax(vd, -vcrit), vcrit);
    double ex = exp(vl / nvt);
    r.g = (is / nvt) * ex;
    double i = is * (ex - 1.0);
    r.ieq = i - r.g * vd;
    r.vd = vd;
    return r;
  }
  double vcrit = nvt * log(nvt / (1.4142135623730951 * is));
  double v = vd;
  if (v > vcrit && fabs(v - vold) > nvt + nvt) {
    if (vold > 0) {
      double arg = 1.0 + (v - vold) / nvt;
      v = arg > 0 ? vold + nvt * log(arg) : vcrit;
    } else {
      v = nvt * log(v / nvt);
    }
    r.limited = true;
  }
  double ex = exp(v / nvt);
  r.g = is / nvt * ex;
  r.ieq = is * (ex - 1.0) - r.g * v;
  r.vd = v;
  return r;
}

// Junction charge of a diode at junction voltage v (opt-in diode parasitics;
// SPICE2 model, Nagel 1975): depletion charge with parameters CJO, VJ, M, FC
// from the record pe ([2..5]),
//   q = CJO VJ / (1 - M) (1 - (1 - v/VJ)^(1-M)),  c = CJO (1 - v/VJ)^-M
// below FC VJ, continued linearly in c above it, plus the diffusion charge
// TT i (pe[6]) with i and its conductance g the diode's current at v.
struct JQ {
  double q, c;
};
__device__ __forceinline__ bool has_jq(const double* pe) { return pe[2] != 0.0 || pe[6] != 0.0; }
__device__ JQ junction_charge(double v, const double* pe, double i, double g) {
  const double cjo = pe[2], vj = pe[3], m = pe[4], fc = pe[5], tt = pe[6];
  JQ r{tt * i, tt * g};
  if (cjo != 0.0) {
    const double fcv = fc * vj;
    if (v < fcv) {
      const double a = 1.0 - v / vj, s = pow(a, -m);
      r.q += cjo * vj * (1.0 - a * s) / (1.0 - m);
      r.c += cjo * s;
    } else {
      const double f1 = vj * (1.0 - pow(1.0 - fc, 1.0 - m)) / (1.0 - m);
      const double f2 = pow(1.0 - fc, 1.0 + m), f3 = 1.0 - fc * (1.0 + m);
      r.q += cjo * (f1 + (f3 * (v - fcv) + m / (2.0 * vj) * (v * v - fcv * fcv)) / f2);
      r.c += cjo / f2 * (f3 + m * v / vj);
    }
  }
  return r;
}

// Diode current and conductance at v without limiting (junction charge of
// the previous step).
__device__ __forceinline__ void diode_iv(double v, double is, double n, double& i, double& g) {
  const double nvt = n * KG_VT, ex = exp(v / nvt);
  i = is * (ex - 1.0);
  g = is / nvt * ex;
}

// Workgroups are dispatched round-robin over the 8 XCDs of an MI355X, each
// with its own L2. Remapping gives every XCD a contiguous range of logical
// blocks, so systems that share an instance's element data (consecutive
// logical blocks) hit the same L2.
__device__ __forceinline__ int64_t xcd_block() {
  const int64_t nb = gridDim.x, b = blockIdx.x;
  const int64_t q = nb / 8, r = nb % 8, x = b % 8, k = b / 8;
  return (x < r ? x * (q + 1) : r * (q + 1) + (x - r) * q) + k;
}

// Largest block of a level-scheduled kernel with TPS threads per system:
// one wave (64 / TPS systems) below 64 threads per system, else one system.
// Declared as the kernels' launch bound, so that the register allocator
// budgets for it instead of for a 1024-thread block (128 VGPRs, which made
// the transient kernels spill about 300 bytes per lane).
#define KG_LB(TPS) __launch_bounds__((TPS) < 64 ? 64 : (TPS))

// Per-point stamp parameters.
struct StampArgs {
  int ak;            // AnalysisKind
  double freq;       // AC frequency (krets computes 2*PI*f*value left to right)
  double h;          // transient step
  double alpha;      // 1 = backward Euler, 2 = trapezoidal
  double tsrc;       // transient source time
  int sweep_e;       // DC-swept element or -1
  double sweep_val;  // its value at this point
};


// Contribution `code` of an element of type ty whose entry in the value table
// (1/R for plain resistors, the element's value otherwise) is ev.
template <class A>
__device__ __forceinline__ A mat_value(int32_t code, int ty, double ev, const StampArgs& sa, const double* ed) {
  const int e = code >> 3, k = code & 7;
  if (k == CK_YP || k == CK_YN) {
    A y = mk<A>(0.0, 0.0);
    if (ty == KG_R) y = mk<A>(ev, 0.0);
    else if (ty == KG_C) y = sa.ak == AK_AC ? mk<A>(0.0, 2.0 * KG_PI * sa.freq * ev) : mk<A>(sa.alpha * (ev / sa.h), 0.0);
    else if (ty == KG_D)  // AC: conductance and junction capacitance at the operating point
      y = mk<A>(ed[e * ESTRIDE], sa.ak == AK_AC ? 2.0 * KG_PI * sa.freq * ed[e * ESTRIDE + 1] : 0.0);
    return k == CK_YP ? y : -y;
  }
  if (k == CK_ONEP) return mk<A>(1.0, 0.0);
  if (k == CK_ONEN) return mk<A>(-1.0, 0.0);
  if (k == CK_KP) return mk<A>(ev, 0.0);
  if (k == CK_KN) return mk<A>(-ev, 0.0);
  if (ty == KG_L)
    return sa.ak == AK_AC ? mk<A>(-0.0, -(2.0 * KG_PI * sa.freq * ev)) : mk<A>(-(sa.alpha * (ev / sa.h)), 0.0);
  if (ty == KG_R) return mk<A>(-ev, 0.0);
  return mk<A>(1.0, 0.0);
}

template <class A>
__device__ __forceinline__ A mat_contrib(int32_t code, const PatDev& P, const double* prm, const double* eb,
                                         const StampArgs& sa, const double* ed) {
  return mat_value<A>(code, P.etype[code >> 3], eb[code >> 3], sa, ed);
}

// xp: previous-step solution (permuted numbering) for companion models.
template <class A>
__device__ __forceinline__ A rhs_contrib(int32_t code, const PatDev& P, const double* prm, const StampArgs& sa,
                                         const double* ed, const double* xp) {
  int e = code >> 3, k = code & 7;
  const double* pe = prm + e * KG_NPARAM;
  switch (k) {
    case RK_SRC: {
      if (e == sa.sweep_e) return mk<A>(sa.sweep_val, 0.0);
      if (P.etype[e] == KG_V) {
        if (sa.ak == AK_AC) return mk<A>(pe[1], 0.0);
        if (sa.ak == AK_TRAN) return mk<A>(wave_value(pe, sa.tsrc), 0.0);
      }
      return mk<A>(pe[0], 0.0);
    }
    case RK_DP: return mk<A>(-ed[e * ESTRIDE + 1], 0.0);
    case RK_DM: return mk<A>(ed[e * ESTRIDE + 1], 0.0);
    case RK_CP:
    case RK_CM: {
      int p = P.ep[e], m = P.em[e];
      double vprev = (p >= 0 ? xp[p] : 0.0) - (m >= 0 ? xp[m] : 0.0);
      // krets: i_eq = -(C/h) * v_prev; RHS[p] += -i_eq, RHS[m] += i_eq
      double ieq = -(sa.alpha * (pe[0] / sa.h)) * vprev;
      if (sa.alpha != 1.0) ieq -= ed[e * ESTRIDE];
      return mk<A>(k == RK_CP ? -ieq : ieq, 0.0);
    }
    default: {  // RK_IND: -(L/h) * i_prev (krets), minus v_prev for TRAP
      int c = P.ec[e];
      double r = -(sa.alpha * (pe[0] / sa.h)) * xp[c];
      if (sa.alpha != 1.0) r -= ed[e * ESTRIDE];
      return mk<A>(r, 0.0);
    }
  }
}

// ------------------------------------------------------------- phases
// All phase helpers are executed by every thread of the block; t is the
// thread's index within its system. Work is skipped when `act` is false but
// barriers are always reached.

// A slot's value is a chain of dependent loads (list bounds, stamp code,
// element type and value), about 800 cycles each from the L2. Each thread
// takes four slots and up to three contributions of each at a time, so that
// the chains overlap (1002 unknowns, 512 threads: 37k cycles one by one).
template <class F, class A, int TPS>
__device__ void stamp_matrix(const PatDev& P, F* v, const double* prm, const double* eb, const StampArgs& sa,
                             const double* ed, int t, bool act) {
  constexpr bool wide = TPS >= 64 && !std::is_same<F, float>::value;  // (the FP32 transients would spill)
  constexpr int U = wide ? 4 : 1, C = wide ? 3 : 1;
  if (!wide || !P.ncr) {  // small systems and staged plans: one slot at a time
    if (act)
      for (int s = t; s < P.nnz; s += TPS) {
        A acc = mk<A>(0.0, 0.0);
        for (int q = P.scon_ptr[s]; q < P.scon_ptr[s + 1]; q++) acc += mat_contrib<A>(P.scon[q], P, prm, eb, sa, ed);
        v[s] = cvt<F>(acc);
      }
    return;
  }
  if (act)
    for (int s0 = t; s0 < P.nnz; s0 += U * TPS) {
      int q0[U], q1[U], most = 0;
      A acc[U];
#pragma unroll
      for (int u = 0; u < U; u++) {
        const int s = s0 + u * TPS, sc = s < P.nnz ? s : P.nnz - 1;
        q0[u] = P.scon_ptr[sc];
        q1[u] = P.scon_ptr[sc + 1];
        acc[u] = mk<A>(0.0, 0.0);
      }
#pragma unroll
      for (int u = 0; u < U; u++) {
        if (s0 + u * TPS >= P.nnz) q1[u] = q0[u];
        if (q1[u] - q0[u] > most) most = q1[u] - q0[u];
      }
      for (int r0 = 0; r0 < most; r0 += C) {
        int32_t code[U][C];
        int ty[U][C];
        double ev[U][C];
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
          for (int r = 0; r < C; r++) code[u][r] = P.scon[q0[u] + r0 + r < q1[u] ? q0[u] + r0 + r : 0];
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
          for (int r = 0; r < C; r++) {
            ty[u][r] = P.etype[code[u][r] >> 3];
            ev[u][r] = eb[code[u][r] >> 3];
          }
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
          for (int r = 0; r < C; r++)
            if (q0[u] + r0 + r < q1[u]) acc[u] += mat_value<A>(code[u][r], ty[u][r], ev[u][r], sa, ed);
      }
#pragma unroll
      for (int u = 0; u < U; u++)
        if (s0 + u * TPS < P.nnz) v[s0 + u * TPS] = cvt<F>(acc[u]);
    }
}

template <class A, int TPS>
__device__ void stamp_rhs(const PatDev& P, A* b, const double* prm, const StampArgs& sa, const double* ed,
                          const double* xp, int t, bool act) {
  if (act)
    for (int i = t; i < P.n; i += TPS) {
      A acc = mk<A>(0.0, 0.0);
      for (int q = P.rcon_ptr[i]; q < P.rcon_ptr[i + 1]; q++) acc += rhs_contrib<A>(P.rcon[q], P, prm, sa, ed, xp);
      b[i] = acc;
    }
}

// ||A||_inf's part of this thread's rows, for the static-pivot guard.
template <int TPS>
__device__ double row_sums(const PatDev& P, const double* v, int t, bool act) {
  double m = 0.0;
  if (act)
    for (int i = t; i < P.n; i += TPS) {
      double s = 0.0;
      for (int p = P.row_ptr[i]; p < P.row_ptr[i + 1]; p++) s += fabs(v[p]);
      m = fmax(m, s);
    }
  return m;
}

// Factorisation by pivot levels: each slot is a dot product over final factors
// (the subtractions of the row-by-row elimination below in their order, so the
// same bits), and a level's slots are independent. Row by row, a thread updated
// its row in LDS one multiplier after the other, 630 dependent updates on the
// 1002 unknowns of a 1000-section ladder (83k cycles with 512 threads); the
// longest dot products of its 11 levels add up to 106 terms.
// FWD: w holds the right-hand side and receives L^-1 w (the substitution of a
// level's rows runs beside its slots).
// V, I: pointers to the values and to the plan (LdsPtr where the caller knows
// them to be in LDS: the compiler does not, and its loads through generic
// pointers take half as long again).
template <class T>
using LdsPtr = __attribute__((address_space(3))) T*;

template <class F, int TPS, bool FWD, class V, class I>
__device__ void factor_levels(const PatDev& P, V v, V w, I lvl, I ent, I pair, I scale, int t, bool act, int* stat) {
  for (int l = 0; l < P.ncr; l++) {
    const int e0 = lvl[3 * l], e2 = FWD ? lvl[3 * l + 3] : lvl[3 * l + 1], s0 = lvl[3 * l + 2], s1 = lvl[3 * l + 5];
    if (act)
      for (int e = e0 + t; e < e2; e += TPS) {
        const int x = ent[2 * e], end = ent[2 * e + 3], s = x & 0xffff;
        int p = ent[2 * e + 1];
        V at = !FWD || s < P.nnz ? v + s : w + (s - P.nnz);
        F acc = *at;
        for (; p + 4 <= end; p += 4) {
          F a[4], b[4];
#pragma unroll
          for (int u = 0; u < 4; u++) {
            const uint32_t q = (uint32_t)pair[p + u];
            const int o = q >> 16;
            V bt = FWD && o >= P.nnz ? w + (o - P.nnz) : v + o;
            a[u] = v[q & 0xffff];
            b[u] = *bt;
          }
#pragma unroll
          for (int u = 0; u < 4; u++) acc -= a[u] * b[u];
        }
        for (; p < end; p++) {
          const uint32_t q = (uint32_t)pair[p];
          const int o = q >> 16;
          V bt = FWD && o >= P.nnz ? w + (o - P.nnz) : v + o;
          const F a = v[q & 0xffff], b = *bt;
          acc -= a * b;
        }
        if (x & 0x10000) {  // the pivot
          if (!(absv(acc) > 0.0) || !finite_v(acc)) *stat = KG_DECOMPOSITION;
          acc = rcp(acc);
        }
        *at = acc;
      }
    __syncthreads();
    if (act)
      for (int e = s0 + t; e < s1; e += TPS) {
        const uint32_t x = (uint32_t)scale[e];
        const F a = v[x & 0xffff], d = v[x >> 16];
        v[x & 0xffff] = a * d;
      }
    __syncthreads();
  }
}

// anorm (NORM, FP64): the largest row sum of |A| among the rows this thread
// takes, before their elimination (the static-pivot guard's ||A||_inf without
// re-gathering the stamps).
template <class F, int TPS, bool NORM = false>
__device__ void factor(const PatDev& P, F* v, int t, bool act, int* stat, double* anorm = nullptr) {
  if constexpr (TPS >= 64 && !std::is_same<F, float>::value) {  // (the FP32 transients would spill)
    if (P.ncr) {
      if constexpr (NORM) {
        *anorm = fmax(*anorm, row_sums<TPS>(P, v, t, act));
        __syncthreads();
      }
      factor_levels<F, TPS, false, F*>(P, v, (F*)nullptr, P.cr_lvl, P.cr_ent, P.cr_pair, P.cr_scale, t, act, stat);
      return;
    }
  }
  auto row = [&](int i) {
    if constexpr (NORM) {
      double s = 0.0;
      for (int p = P.row_ptr[i]; p < P.row_ptr[i + 1]; p++) s += fabs(v[p]);
      *anorm = fmax(*anorm, s);
    }
    const int32_t* fp = P.fprog + P.fprog_ptr[i];
    int nk = *fp++;
    for (int kk = 0; kk < nk; kk++) {
      int sik = fp[0], sdk = fp[1], nu = fp[2];
      fp += 3;
      F lik = v[sik] * v[sdk];
      v[sik] = lik;
      for (int u = 0; u < nu; u++) {
        v[fp[0]] -= lik * v[fp[1]];
        fp += 2;
      }
    }
    F piv = v[P.diag[i]];
    double a = absv(piv);
    if (!(a > 0.0) || !finite_v(piv)) *stat = KG_DECOMPOSITION;
    v[P.diag[i]] = rcp(piv);
  };
  if constexpr (TPS == 1) {
    if (act)
      for (int i = 0; i < P.n; i++) row(i);
  } else {
    for (int l = 0; l < P.nlev; l++) {
      if (act)
        for (int q = P.lvl_ptr[l] + t; q < P.lvl_ptr[l + 1]; q += TPS) row(P.lvl_rows[q]);
      __syncthreads();
    }
  }
}

// Level-scheduled substitution over rows' entries [from(i), to(i)): the next
// level's first row, its first two entries and (back substitution) its
// reciprocal pivot are read before the barrier, so that a level costs one round
// trip to the solution vector.
template <class F, int TPS, bool BACK>
__device__ void lu_levels(const PatDev& P, const F* v, F* w, int t, bool act) {
  const int nl = BACK ? P.nblev : P.nlev;
  const int32_t *ptr = BACK ? P.blvl_ptr : P.lvl_ptr, *rows = BACK ? P.blvl_rows : P.lvl_rows;
  auto from = [&](int i) { return BACK ? P.diag[i] + 1 : P.row_ptr[i]; };
  auto to = [&](int i) { return BACK ? P.row_ptr[i + 1] : P.diag[i]; };
  int i = -1, p0 = 0, p1 = 0, c0 = 0, c1 = 0;
  F f0{}, f1{}, fd{};
  auto ahead = [&](int q, int hi) {
    i = -1;
    if (!act || q >= hi) return;
    i = rows[q];
    p0 = from(i);
    p1 = to(i);
    if (p0 < p1) {
      c0 = P.col[p0];
      f0 = v[p0];
    }
    if (p0 + 1 < p1) {
      c1 = P.col[p0 + 1];
      f1 = v[p0 + 1];
    }
    if (BACK) fd = v[p0 - 1];
  };
  int lo = nl > 0 ? ptr[0] : 0, hi = nl > 0 ? ptr[1] : 0;  // nl = 0: no plan, no pointers either
  ahead(lo + t, hi);
  for (int l = 0; l < nl; l++) {
    if (i >= 0) {
      F s = w[i];
      if (p0 < p1) s -= f0 * w[c0];
      if (p0 + 1 < p1) s -= f1 * w[c1];
      for (int p = p0 + 2; p < p1; p++) s -= v[p] * w[P.col[p]];
      w[i] = BACK ? s * fd : s;
    }
    if (act)
      for (int q = lo + t + TPS; q < hi; q += TPS) {
        const int r = rows[q], b = from(r), e = to(r);
        F s = w[r];
        for (int p = b; p < e; p++) s -= v[p] * w[P.col[p]];
        w[r] = BACK ? s * v[b - 1] : s;
      }
    lo = hi;
    if (l + 1 < nl) {
      hi = ptr[l + 2];
      ahead(lo + t, hi);
    }
    __syncthreads();
  }
}

// Solves (LU) w = w in place.
template <class F, int TPS>
__device__ void lu_solve(const PatDev& P, const F* v, F* w, int t, bool act) {
  if constexpr (TPS == 1) {
    if (act) {
      for (int i = 0; i < P.n; i++) {
        F s = w[i];
        for (int p = P.row_ptr[i]; p < P.diag[i]; p++) s -= v[p] * w[P.col[p]];
        w[i] = s;
      }
      for (int i = P.n - 1; i >= 0; i--) {
        F s = w[i];
        const int d = P.diag[i];
        for (int p = d + 1; p < P.row_ptr[i + 1]; p++) s -= v[p] * w[P.col[p]];
        w[i] = s * v[d];
      }
    }
  } else if (TPS < 64 || std::is_same<F, float>::value || !P.ncr) {  // (the FP32 transients would spill)
    for (int l = 0; l < P.nlev; l++) {
      if (act)
        for (int q = P.lvl_ptr[l] + t; q < P.lvl_ptr[l + 1]; q += TPS) {
          const int i = P.lvl_rows[q];
          F s = w[i];
          for (int p = P.row_ptr[i]; p < P.diag[i]; p++) s -= v[p] * w[P.col[p]];
          w[i] = s;
        }
      __syncthreads();
    }
    for (int l = 0; l < P.nblev; l++) {
      if (act)
        for (int q = P.blvl_ptr[l] + t; q < P.blvl_ptr[l + 1]; q += TPS) {
          const int i = P.blvl_rows[q], d = P.diag[i];
          F s = w[i];
          for (int p = d + 1; p < P.row_ptr[i + 1]; p++) s -= v[p] * w[P.col[p]];
          w[i] = s * v[d];
        }
      __syncthreads();
    }
  } else if constexpr (TPS >= 64 && !std::is_same<F, float>::value) {
    lu_levels<F, TPS, false>(P, v, w, t, act);
    lu_levels<F, TPS, true>(P, v, w, t, act);
  }
}

// Solves (LU)^T w = w in place: U^T forward, then L^T backward.
template <class F, int TPS>
__device__ void lu_solve_t(const PatDev& P, const F* v, F* w, int t, bool act) {
  auto fwd = [&](int i) {
    F s = w[i];
    for (int q = P.ut_ptr[i]; q < P.ut_ptr[i + 1]; q += 2) s -= v[P.ut[q + 1]] * w[P.ut[q]];
    w[i] = s * v[P.diag[i]];
  };
  auto bwd = [&](int i) {
    F s = w[i];
    for (int q = P.lt_ptr[i]; q < P.lt_ptr[i + 1]; q += 2) s -= v[P.lt[q + 1]] * w[P.lt[q]];
    w[i] = s;
  };
  if constexpr (TPS == 1) {
    if (act) {
      for (int i = 0; i < P.n; i++) fwd(i);
      for (int i = P.n - 1; i >= 0; i--) bwd(i);
    }
  } else {
    for (int l = 0; l < P.ntlev; l++) {
      if (act)
        for (int q = P.tlvl_ptr[l] + t; q < P.tlvl_ptr[l + 1]; q += TPS) fwd(P.tlvl_rows[q]);
      __syncthreads();
    }
    for (int l = 0; l < P.ntblev; l++) {
      if (act)
        for (int q = P.tblvl_ptr[l] + t; q < P.tblvl_ptr[l + 1]; q += TPS) bwd(P.tblvl_rows[q]);
      __syncthreads();
    }
  }
}

// Max-reduction of a non-negative double over the TPS threads of a system.
template <int TPS>
__device__ double sys_max(double v, double* red, int ls, int t) {
  if constexpr (TPS == 1) {
    return v;
  } else {
    red[ls * TPS + t] = v;
    __syncthreads();
    for (int s = TPS / 2; s > 0; s >>= 1) {
      if (t < s) red[ls * TPS + t] = fmax(red[ls * TPS + t], red[ls * TPS + t + s]);
      __syncthreads();
    }
    double r = red[ls * TPS];
    __syncthreads();
    return r;
  }
}

// Full solve of A x = b given the factored v. FP64 (F == A): x := LU \ b.
// Mixed: x := LU \ b followed by `refine` steps of FP64 iterative refinement
// with A re-gathered in FP64. Returns the normwise size of the last
// correction relative to x (0 for FP64).
template <class F, class A, int TPS>
__device__ double solve_refine(const PatDev& P, const F* v, const A* b, A* x, F* w, const double* prm,
                               const double* eb, const StampArgs& sa, const double* ed, int refine, double* red,
                               int ls, int t, bool act, A* rbuf = nullptr) {
  if constexpr (std::is_same<F, A>::value) {
    if (act)
      for (int i = t; i < P.n; i += TPS) x[i] = b[i];
    __syncthreads();
    lu_solve<F, TPS>(P, v, x, t, act);
    return 0.0;
  } else {
    if (act)
      for (int i = t; i < P.n; i += TPS) w[i] = cvt<F>(b[i]);
    __syncthreads();
    lu_solve<F, TPS>(P, v, w, t, act);
    if (act)
      for (int i = t; i < P.n; i += TPS) x[i] = cvt<A>(w[i]);
    __syncthreads();
    double est = 0.0, dprev = 0.0;
    for (int it = 0; it < refine; it++) {
      // r = b - A x in FP64 (A gathered in FP64), kept in rbuf
      double rmax = 0.0;
      if (act)
        for (int i = t; i < P.n; i += TPS) {
          A r = b[i];
          for (int p = P.row_ptr[i]; p < P.row_ptr[i + 1]; p++) {
            int q0 = P.scon_ptr[p], q1 = P.scon_ptr[p + 1];
            if (q0 == q1) continue;
            A a = mk<A>(0.0, 0.0);
            for (int q = q0; q < q1; q++) a += mat_contrib<A>(P.scon[q], P, prm, eb, sa, ed);
            r -= a * x[P.col[p]];
          }
          rmax = fmax(rmax, absv(r));
          rbuf[i] = r;
        }
      double s = sys_max<TPS>(rmax, red, ls, t);
      // scaled FP32 correction right-hand side (keeps the residual in range)
      if (act && s > 0.0) {
        double inv = 1.0 / s;
        for (int i = t; i < P.n; i += TPS) w[i] = cvt<F>(scal(inv, rbuf[i]));
      }
      __syncthreads();
      lu_solve<F, TPS>(P, v, w, t, act && s > 0.0);  // barriers are reached by every system
      double dmax = 0.0, xmax = 0.0;
      if (act && s > 0.0)
        for (int i = t; i < P.n; i += TPS) {
          A d = scal(s, cvt<A>(w[i]));
          x[i] += d;
          dmax = fmax(dmax, absv(d));
          xmax = fmax(xmax, absv(x[i]));
        }
      __syncthreads();
      double dm = sys_max<TPS>(dmax, red, ls, t);
      double xm = sys_max<TPS>(xmax, red, ls, t);
      // remaining error ~ contraction ratio * last correction (geometric
      // convergence of refinement); the last correction itself bounds it
      double rho = (it > 0 && dprev > 0.0) ? fmin(dm / dprev, 1.0) : 1.0;
      est = xm > 0.0 ? rho * dm / xm : 0.0;
      dprev = dm;
    }
    return est;
  }
}

__device__ __forceinline__ void atomic_max_nonneg(double* addr, double v) {
  atomicMax(reinterpret_cast<unsigned long long*>(addr), (unsigned long long)__double_as_longlong(v));
}

// Entry norm of the backward-error guard: |re| + |im|.
__device__ __forceinline__ double c1(double a) { return fabs(a); }
__device__ __forceinline__ double c1(c128 a) { return fabs(a.re) + fabs(a.im); }

// Componentwise backward error of an FP64 solve (Oettli-Prager), omega =
// max_i |b - A x|_i / ((|A| |x| + |b|)_i + u ||b||_inf) with |z| = |re| + |im|
// and A re-gathered in FP64 from the stamps (the system's v holds its
// factors); it bounds the normwise backward error. The floor u ||b||_inf
// (perturbations of b allowed down to FP64's resolution of its largest
// entry) keeps rows whose solution has decayed towards underflow measurable:
// a long RC ladder at high frequency attenuates its node voltages into the
// subnormal range, where the plain componentwise ratio is rounding noise of
// order 1 even for a partial-pivoting solve. Reached by every thread.
template <class A, int TPS>
__device__ double guard_omega(const PatDev& P, const A* b, const A* x, const double* prm, const double* eb,
                              const StampArgs& sa, const double* ed, double* red, int ls, int t, bool act) {
  double bm = 0.0;
  if (act)
    for (int i = t; i < P.n; i += TPS) bm = fmax(bm, c1(b[i]));
  const double floor_b = 0x1p-53 * sys_max<TPS>(bm, red, ls, t);
  double om = 0.0;
  if (act)
    for (int i = t; i < P.n; i += TPS) {
      A r = b[i];
      double dr = c1(b[i]);
      for (int p = P.row_ptr[i]; p < P.row_ptr[i + 1]; p++) {
        int q0 = P.scon_ptr[p], q1 = P.scon_ptr[p + 1];
        if (q0 == q1) continue;
        A a = mk<A>(0.0, 0.0);
        for (int q = q0; q < q1; q++) a += mat_contrib<A>(P.scon[q], P, prm, eb, sa, ed);
        const A xj = x[P.col[p]];
        r -= a * xj;
        dr += c1(a) * c1(xj);
      }
      const double ri = c1(r);
      const double den = dr + floor_b;
      if (ri > 0.0) om = fmax(om, den > 0.0 ? ri / den : INFINITY);
    }
  return sys_max<TPS>(om, red, ls, t);
}

// Normwise backward error |b - A x| / (|A| |x| + |b|) of a solve returned by
// mixed precision refinement (infinity norms over |re| + |im|, A re-gathered
// in FP64 from the stamps). Reached by every thread.
template <class A, int TPS>
__device__ double guard_eta(const PatDev& P, const A* b, const A* x, const double* prm, const double* eb,
                            const StampArgs& sa, const double* ed, double* red, int ls, int t, bool act) {
  double rm = 0.0, am = 0.0, bm = 0.0, xm = 0.0;
  if (act)
    for (int i = t; i < P.n; i += TPS) {
      A r = b[i];
      double ar = 0.0;
      for (int p = P.row_ptr[i]; p < P.row_ptr[i + 1]; p++) {
        int q0 = P.scon_ptr[p], q1 = P.scon_ptr[p + 1];
        if (q0 == q1) continue;
        A a = mk<A>(0.0, 0.0);
        for (int q = q0; q < q1; q++) a += mat_contrib<A>(P.scon[q], P, prm, eb, sa, ed);
        r -= a * x[P.col[p]];
        ar += c1(a);
      }
      rm = fmax(rm, c1(r));
      am = fmax(am, ar);
      bm = fmax(bm, c1(b[i]));
      xm = fmax(xm, c1(x[i]));
    }
  rm = sys_max<TPS>(rm, red, ls, t);
  am = sys_max<TPS>(am, red, ls, t);
  bm = sys_max<TPS>(bm, red, ls, t);
  xm = sys_max<TPS>(xm, red, ls, t);
  const double den = am * xm + bm;
  return den > 0.0 ? rm / den : (rm > 0.0 ? INFINITY : 0.0);
}

// Static-pivot guard of the FP64 OP, DC sweep and transient factorisations
// (KG_GUARD_STATIC): the lane AC kernels' a-priori bound guard_bound_coeff(m)
// * rho, rho = || |L||U| ||_inf / ||A||_inf, formed after the fact from the
// factors in v (multipliers below the diagonal, the pivot's reciprocal on it,
// the upper factor unscaled), with ||A||_inf taken by factor<..., NORM> as
// it eliminates. This thread's parts over the rows t, t + TPS, ...:
// pivot_guard_rows returns the longest row m and writes the row sums of |U|
// into us; after a barrier, pivot_guard_lu returns the rows of |L||U|.
template <int TPS>
__device__ double pivot_guard_rows(const PatDev& P, const double* v, double* us, int t, bool act) {
  double m = 0.0;
  if (act)
    for (int i = t; i < P.n; i += TPS) {
      const int d = P.diag[i];
      double u = 1.0 / fabs(v[d]);
      for (int p = d + 1; p < P.row_ptr[i + 1]; p++) u += fabs(v[p]);
      us[i] = u;
      m = fmax(m, (double)(P.row_ptr[i + 1] - P.row_ptr[i]));
    }
  return m;
}

template <int TPS>
__device__ double pivot_guard_lu(const PatDev& P, const double* v, const double* us, int t, bool act) {
  double gm = 0.0;
  if (act)
    for (int i = t; i < P.n; i += TPS) {
      double g = us[i];
      for (int p = P.row_ptr[i]; p < P.diag[i]; p++) g += fabs(v[p]) * us[P.col[p]];
      gm = fmax(gm, g);
    }
  return gm;
}

__device__ __forceinline__ double pivot_guard_bound(double gm, double an, double m) {
  return gm > 0.0 ? (an > 0.0 ? guard_bound_coeff((int)m) * (gm / an) : INFINITY) : 0.0;
}

// Maxima of three values over the TPS threads of a system: shuffles inside
// the wave (a system's threads are consecutive lanes), then, for systems of
// several waves, one exchange through red (TPS doubles of the system) between
// two barriers. Reached by every thread of the block.
template <int TPS>
__device__ void sys_max3(double& a, double& b, double& c, double* red, int ls, int t) {
  constexpr int W = TPS < 64 ? TPS : 64;
  for (int o = W / 2; o > 0; o >>= 1) {
    a = fmax(a, __shfl_xor(a, o, W));
    b = fmax(b, __shfl_xor(b, o, W));
    c = fmax(c, __shfl_xor(c, o, W));
  }
  if constexpr (TPS > 64) {
    double* r = red + ls * TPS;
    if ((t & 63) == 0) {
      r[3 * (t / 64)] = a;
      r[3 * (t / 64) + 1] = b;
      r[3 * (t / 64) + 2] = c;
    }
    __syncthreads();
    for (int k = 0; k < TPS / 64; k++) {
      a = fmax(a, r[3 * k]);
      b = fmax(b, r[3 * k + 1]);
      c = fmax(c, r[3 * k + 2]);
    }
    __syncthreads();
  }
}

// Level-scheduled form, reached by every thread of the system; an: this
// thread's part of ||A||_inf from factor<..., NORM>; us: n doubles of scratch.
template <int TPS>
__device__ double pivot_guard(const PatDev& P, const double* v, double an, double* us, double* red, int ls, int t,
                              bool act) {
  double m = pivot_guard_rows<TPS>(P, v, us, t, act);
  __syncthreads();
  double gm = pivot_guard_lu<TPS>(P, v, us, t, act);
  sys_max3<TPS>(an, m, gm, red, ls, t);
  return pivot_guard_bound(gm, an, m);
}

// Block-wide maximum of non-negative values into a 64-bit LDS word that was
// zeroed before a barrier: a wave maximum, then one atomic per wave.
__device__ __forceinline__ void block_max_to(double v, unsigned long long* w) {
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o));
  if ((threadIdx.x & 63) == 0) atomicMax(w, (unsigned long long)__double_as_longlong(v));
}

// Queues system `sys` for k_ac_fix (queue words: [0] count, [1 + q] systems);
// a full queue marks the instance as failed instead.
__device__ __forceinline__ void fix_push(unsigned long long* fixq, int64_t cap, int64_t sys, int32_t* status,
                                         int inst) {
  const unsigned long long q = atomicAdd(fixq, 1ull);
  if (q < (unsigned long long)cap) fixq[1 + q] = (unsigned long long)sys;
  else atomicMax(&status[inst], KG_DECOMPOSITION);
}

// End of one AC solve (thread 0 of the system): a failed pivot, an FP64
// backward error above KG_GUARD_OMEGA or a mixed error estimate above
// KG_GUARD_MIXED queues the solve for k_ac_fix (when a queue is given);
// otherwise the status and the instance's error figure are published.
__device__ __forceinline__ void ac_finish(int32_t flag, double q, bool mixed, unsigned long long* fixq,
                                          int64_t fixcap, int64_t sys, int32_t* status, double* err, int inst) {
  const bool bad = flag != KG_OK || !(q <= (mixed ? KG_GUARD_MIXED : KG_GUARD_OMEGA));
  if (fixq && bad) {
    fix_push(fixq, fixcap, sys, status, inst);
    return;
  }
  if (flag != KG_OK) atomicMax(&status[inst], flag);
  if (err && q > 0.0) atomicMax(reinterpret_cast<unsigned long long*>(&err[inst]),
                                (unsigned long long)__double_as_longlong(q));
}

}  // namespace kg
