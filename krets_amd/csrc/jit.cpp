// Run-time specialisation of the AC sweep to one circuit topology.
//
// The host symbolic pass fixes, for a shared topology, every LU slot, the
// static pivot order and which element contributions land in each slot.
// Instead of interpreting that plan on the device (the level-scheduled
// kernels read it from memory), this file writes it out as straight-line
// HIP: one lane solves one (instance, frequency) system with the matrix, the
// factors and the solution in registers.
//
// Factorisation (row i in pivot order, up-looking as in the plan's factor
// program) keeps the upper factor scaled by the reciprocal pivot, U' =
// diag(U)^-1 U, and the forward-substitution vector scaled the same way, so
// that neither the lower factor nor the pivots outlive their row:
//   a_ij -= a_ik * U'_kj              (k < i in the row's pattern, j > k)
//   y_i   = b_i - sum_k a_ik * y'_k
//   U'_ij = a_ij / a_ii,  y'_i = y_i / a_ii
//   x_i   = y'_i - sum_j U'_ij x_j     (back substitution, i descending)
// This is the same LU (the same pivots, the same fill) as the plan's factor
// program, with the multiplier division moved onto the upper factor.
//
// Mixed precision repeats the factorisation in complex64 on every pass (it
// costs the same VALU work as re-reading stored factors would cost in
// registers this kernel does not have), with FP64 residuals b - A x from the
// FP64 stamps and FP64 accumulation of the corrections, as the generic
// kernels do.
#include "kg_jit.h"

#include <hip/hiprtc.h>

#include <algorithm>
#include <cstdio>
#include <functional>
#include <map>
#include <mutex>
#include <set>
#include <sstream>
#include <utility>
#include <vector>

namespace kg {
namespace {

struct View {
  int n = 0, nnz = 0, ne = 0;
  const int32_t *row_ptr, *col, *diag, *fprog_ptr, *fprog, *scon_ptr, *scon, *rcon_ptr, *rcon, *col_of, *etype;
};

View view(const PatLayout& L, const int32_t* b) {
  View v;
  v.n = L.n;
  v.nnz = L.nnz;
  v.ne = L.ne;
  v.row_ptr = b + L.o_row_ptr;
  v.col = b + L.o_col;
  v.diag = b + L.o_diag;
  v.fprog_ptr = b + L.o_fprog_ptr;
  v.fprog = b + L.o_fprog;
  v.scon_ptr = b + L.o_scon_ptr;
  v.scon = b + L.o_scon;
  v.rcon_ptr = b + L.o_rcon_ptr;
  v.rcon = b + L.o_rcon;
  v.col_of = b + L.o_col_of;
  v.etype = b + L.o_etype;
  return v;
}

const char* kPrelude = R"(typedef long long i64;
struct __attribute__((aligned(16))) Z { double re, im; };
struct __attribute__((aligned(8))) W { float re, im; };
__device__ __forceinline__ Z operator+(Z a, Z b) { return {a.re + b.re, a.im + b.im}; }
__device__ __forceinline__ Z operator-(Z a, Z b) { return {a.re - b.re, a.im - b.im}; }
__device__ __forceinline__ Z operator*(Z a, Z b) { return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re}; }
__device__ __forceinline__ W operator-(W a, W b) { return {a.re - b.re, a.im - b.im}; }
__device__ __forceinline__ W operator*(W a, W b) { return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re}; }
__device__ __forceinline__ Z cz(Z a) { return a; }
__device__ __forceinline__ Z cz(W a) { return {(double)a.re, (double)a.im}; }
__device__ __forceinline__ W cw(Z a) { return {(float)a.re, (float)a.im}; }
__device__ __forceinline__ Z scal(double s, Z a) { return {s * a.re, s * a.im}; }
// product with a factor known to be real (a stamp with no imaginary part that
// no elimination step has changed): two multiplications where the complex
// product spends four plus two additions (IEEE arithmetic keeps its
// 0 * x.im terms)
__device__ __forceinline__ Z rmul(double a, Z x) { return {a * x.re, a * x.im}; }
__device__ __forceinline__ W rmul(float a, W x) { return {a * x.re, a * x.im}; }
// z - a * b as two fused steps per component (one rounding fewer than the
// subtracted product)
__device__ __forceinline__ Z fms(Z z, Z a, Z b) {
  return {(z.re - a.re * b.re) + a.im * b.im, (z.im - a.re * b.im) - a.im * b.re};
}
__device__ __forceinline__ W fms(W z, W a, W b) {
  return {(z.re - a.re * b.re) + a.im * b.im, (z.im - a.re * b.im) - a.im * b.re};
}
__device__ __forceinline__ double m2(Z a) { return a.re * a.re + a.im * a.im; }
// running max norm over components, max(|re|, |im|), of complex64 values: one
// instruction per value, and no squares that could leave the FP32 range
__device__ __forceinline__ float cmax(float m, W a) {
  return __builtin_fmaxf(m, __builtin_fmaxf(__builtin_fabsf(a.re), __builtin_fabsf(a.im)));
}
__device__ __forceinline__ bool fin(Z a) { return __builtin_isfinite(a.re) && __builtin_isfinite(a.im); }
// |re| + |im|: the entry norm of the growth guard (submultiplicative, within
// a factor sqrt(2) of the modulus)
__device__ __forceinline__ double c1(Z a) { return __builtin_fabs(a.re) + __builtin_fabs(a.im); }
__device__ __forceinline__ double c1(W a) { return (double)__builtin_fabsf(a.re) + (double)__builtin_fabsf(a.im); }
// queues system `sys` for the dense partial-pivoting fixup (queue words: [0]
// count, [1 + q] systems); a full queue marks the instance instead
__device__ __forceinline__ void fix_push(unsigned long long* fixq, i64 cap, i64 sys, int* status, int inst) {
  const unsigned long long q = atomicAdd(fixq, 1ull);
  if (q < (unsigned long long)cap) fixq[1 + q] = (unsigned long long)sys;
  else atomicMax(&status[inst], 2);
}
// reciprocal of a pivot, conj(b) / |b|^2, without branches: an FP64 pivot is
// first scaled by the power of two of its larger component (exact), so
// |b|^2 cannot leave the FP64 range; an FP32 pivot's |b|^2 always fits FP64
__device__ __forceinline__ Z rcpF(Z b) {
  const int k = __builtin_amdgcn_frexp_exp(__builtin_fmax(__builtin_fabs(b.re), __builtin_fabs(b.im)));
  const double re = __builtin_amdgcn_ldexp(b.re, -k), im = __builtin_amdgcn_ldexp(b.im, -k);
  // m in [0.25, 2): hardware reciprocal estimate (off by e, at most 2^-24)
  // and the cubic step q (1 + e + e^2), which leaves e^3 (a shorter dependent
  // chain than two Newton steps or a correctly rounded division; ~1 ulp)
  const double m = re * re + im * im;
  double q = __builtin_amdgcn_rcp(m);
  const double e = 1.0 - m * q;
  q = q + q * (e + e * e);
  return {__builtin_amdgcn_ldexp(re * q, -k), __builtin_amdgcn_ldexp(-im * q, -k)};
}
// complex64 pivots: |b|^2 in FP64 (cannot leave its range) and the hardware
// reciprocal estimate as it is: its relative error (measured on gfx950: at
// most 4.6e-8, 2^-24.4) is that of the FP32 rounding that follows, and the
// refinement corrects the complex64 factorisation anyway (a Newton step
// costs two more dependent instructions per pivot and 1.5% of the kernel)
__device__ __forceinline__ W rcpF(W b) {
  const double re = b.re, im = b.im, m = re * re + im * im;
  const double q = __builtin_amdgcn_rcp(m);
  return {(float)(re * q), (float)(-im * q)};
}
// a pivot that can be divided by: not zero, finite
__device__ __forceinline__ bool piv_ok(Z b) { return m2(b) > 0.0 && fin(b); }
// complex64: |b|^2 in FP64 is zero, infinite or NaN only where the pivot is
__device__ __forceinline__ bool piv_ok(W b) {
  const double m = m2(cz(b));
#ifdef __AMDGCN__
  return __builtin_amdgcn_class(m, 0x180);  // positive, normal or subnormal
#else
  return m > 0.0 && m <= 1.7976931348623157e308;
#endif
}
// |1/b| of the growth guard, r = 1/b and c = c1(b) given
__device__ __forceinline__ double c1r(Z, Z r, double) { return c1(r); }
__device__ __forceinline__ double c1r(W b, W, double c) { return c * __builtin_amdgcn_rcp(m2(cz(b))); }
#ifdef __AMDGCN__
// 4 x 4 transposition within each quad of lanes: afterwards v_k of lane l is
// lane k's former v_l
template <int C> __device__ __forceinline__ void quad_swap(bool up, int& a, int& b) {
  const int ta = __builtin_amdgcn_mov_dpp(a, C, 0xf, 0xf, true), tb = __builtin_amdgcn_mov_dpp(b, C, 0xf, 0xf, true);
  a = up ? tb : a;
  b = up ? b : ta;
}
struct __attribute__((aligned(16))) I4 { int w[4]; };
// Stores unknowns c .. c + 3 of the quad's four systems, 64 contiguous bytes a
// store and system: one store per unknown and lane would put 64 requests of
// 16 bytes to the L2 where 16 of 64 carry the same data (4096 x 200 systems of
// 52 unknowns, mixed: 0.403 -> 0.322 ms; 1001 x 151 of 39, FP64: 45.6 -> 34 us).
// The rest of the kernel is VALU: without its stores it takes 0.255 ms, so the
// guard's figures cost as few conversions as its FP64 sums allow and products
// are subtracted in fused steps (0.322 -> 0.300 ms). q.o[k] is lane k's
// row, advanced by the lane's place in the quad.
struct Quad { Z* o[4]; bool u1, u2; };
template <int C> __device__ __forceinline__ i64 quad_bcast(i64 v) {
  const unsigned lo = (unsigned)__builtin_amdgcn_mov_dpp((int)v, C, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_mov_dpp((int)(v >> 32), C, 0xf, 0xf, true);
  return (i64)(((unsigned long long)(unsigned)hi << 32) | lo);
}
__device__ __forceinline__ Quad quad_rows(Z* out, i64 off) {
  const int l = threadIdx.x & 3;
  return {{out + (quad_bcast<0x00>(off) + l), out + (quad_bcast<0x55>(off) + l), out + (quad_bcast<0xaa>(off) + l),
           out + (quad_bcast<0xff>(off) + l)}, (l & 1) != 0, (l & 2) != 0};
}
__device__ __forceinline__ void st4(const Quad& q, int c, Z z0, Z z1, Z z2, Z z3) {
  I4 v0 = __builtin_bit_cast(I4, z0), v1 = __builtin_bit_cast(I4, z1), v2 = __builtin_bit_cast(I4, z2),
     v3 = __builtin_bit_cast(I4, z3);
  for (int i = 0; i < 4; i++) {
    quad_swap<0xb1>(q.u1, v0.w[i], v1.w[i]);
    quad_swap<0xb1>(q.u1, v2.w[i], v3.w[i]);
    quad_swap<0x4e>(q.u2, v0.w[i], v2.w[i]);
    quad_swap<0x4e>(q.u2, v1.w[i], v3.w[i]);
  }
  q.o[0][c] = __builtin_bit_cast(Z, v0);
  q.o[1][c] = __builtin_bit_cast(Z, v1);
  q.o[2][c] = __builtin_bit_cast(Z, v2);
  q.o[3][c] = __builtin_bit_cast(Z, v3);
}
#else  // lane by lane
struct Quad { Z* o; };
inline Quad quad_rows(Z* out, i64 off) { return {out + off}; }
inline void st4(const Quad& q, int c, Z z0, Z z1, Z z2, Z z3) {
  q.o[c] = z0;
  q.o[c + 1] = z1;
  q.o[c + 2] = z2;
  q.o[c + 3] = z3;
}
#endif
// block order that keeps consecutive systems (one instance) on one XCD
__device__ __forceinline__ i64 xcd_block() {
  const i64 nb = gridDim.x, b = blockIdx.x;
  const i64 q = nb / 8, r = nb % 8, x = b % 8, k = b / 8;
  return (x < r ? x * (q + 1) : r * (q + 1) + (x - r) * q) + k;
}
)";

// Emits straight-line code. Element values are loaded once per pass (a pass
// is a brace scope), `lookahead` rows before the row that first uses them, and
// an empty asm statement with a memory clobber after each row's loads keeps
// the compiler from hoisting every load of the kernel to its start (which
// would hold all element values in registers at once).

// refinement passes load x as well as element values: a shorter distance
// keeps the values in flight within the register budget
#ifndef KG_LANE_AHEAD_REFINE
#define KG_LANE_AHEAD_REFINE 4
#endif
#ifndef KG_LANE_AHEAD
#define KG_LANE_AHEAD 16
#endif
// rows between scheduling barriers in the forward (factor and forward
// substitution) and backward sweeps; 0: none (the mixed kernel then spills:
// 0.41 ms; 1, 2 or 3 rows: 0.307, 0.301, 0.304 ms on 4096 x 200 systems of 52
// unknowns, at 16 rows between load and use)
#ifndef KG_LANE_FWD_BARRIER
#define KG_LANE_FWD_BARRIER 2
#endif
#ifndef KG_LANE_BWD_BARRIER
#define KG_LANE_BWD_BARRIER 4
#endif
int LOOKAHEAD_REFINE = KG_LANE_AHEAD_REFINE;

// A double as a C++ literal that reads back to the same value.
std::string fmt_double(double v) {
  char b[40];
  std::snprintf(b, sizeof b, "%.17g", v);
  return b;
}

// rows of the four unknowns of group g as arguments
std::string st4_args(const std::vector<int>& row_of, int g, const char* name) {
  std::string a;
  for (int k = 0; k < 4; k++) a += std::string(", ") + name + std::to_string(row_of[4 * g + k]);
  return a;
}

// Systems whose upper factor does not fit in registers ran level by level, a
// block per system (64 ladders of 200 sections at 101 frequencies: 0.53 ms,
// the latency of some 15 levels per system at five systems per CU). A lane per
// system does the same elimination row by row; written out, its code would
// leave the instruction cache, so the rows that repeat along a chain become a
// loop: 45 us, a serial chain of about 400 cycles a row.
//
// Rows i0 .. i1 - 1 of D interleaved chains (row i couples to rows i - D and
// i + D only) whose stamps repeat with element numbers that advance by a
// constant: iteration t of a loop handles rows i0 + t D + c, c < D.
struct Run {
  int i0 = 0, i1 = 0, D = 1, nit = 0;
  std::vector<std::vector<std::pair<int, int>>> el;  // per chain: elements of its first row, and their step
  std::vector<int> col, cstep;                       // per chain: unknown of its first row, and its step
  bool has(int i) const { return i >= i0 && i < i1; }
};

// contributions of the three slots of a chain row as (slot, kind, type) and, apart from them, their elements
bool chain_row(const View& P, int i, int D, std::vector<int>& shape, std::vector<int>& els) {
  const int s0 = P.row_ptr[i];
  if (i < D || i + D >= P.n || P.row_ptr[i + 1] - s0 != 3) return false;
  if (P.col[s0] != i - D || P.col[s0 + 1] != i || P.col[s0 + 2] != i + D) return false;
  if (P.rcon_ptr[i + 1] != P.rcon_ptr[i]) return false;
  const int32_t* fp = P.fprog + P.fprog_ptr[i];  // one step: eliminate with row i - D, update the diagonal
  if (fp[0] != 1 || fp[1] != s0 || fp[3] != 1 || fp[4] != s0 + 1) return false;
  shape.clear();
  els.clear();
  for (int s = s0; s < s0 + 3; s++)
    for (int q = P.scon_ptr[s]; q < P.scon_ptr[s + 1]; q++) {
      const int e = P.scon[q] >> 3, k = P.scon[q] & 7;
      shape.insert(shape.end(), {s - s0, k, P.etype[e]});
      els.push_back(e);
    }
  return true;
}

// The longest run of D chains, its length in iterations a multiple of 4.
bool find_run(const View& P, int D, Run& best) {
  best.nit = 0;
  for (int i0 = D; i0 + 9 * D <= P.n; i0++) {
    Run r;
    r.i0 = i0;
    r.D = D;
    std::vector<std::vector<int>> shape(D), first(D), step(D), prev(D);
    int t = 0;
    for (bool go = true; go; t += go) {
      for (int c = 0; c < D && go; c++) {
        std::vector<int> sh, el;
        go = chain_row(P, i0 + t * D + c, D, sh, el);
        if (!go) break;
        el.push_back(P.col_of[i0 + t * D + c]);
        if (t == 0) {
          shape[c] = sh;
          first[c] = el;
        } else {
          go = sh == shape[c];
          if (go && t == 1)
            for (size_t q = 0; q < el.size(); q++) step[c].push_back(el[q] - first[c][q]);
          for (size_t q = 0; go && q < el.size(); q++) go = el[q] == prev[c][q] + step[c][q];
        }
        prev[c] = el;
      }
    }
    r.nit = t / 4 * 4;
    r.i1 = i0 + r.nit * D;
    if (r.nit <= best.nit) continue;
    bool ok = true;
    for (int c = 0; c < D; c++) {
      r.col.push_back(first[c].back());
      r.cstep.push_back(step[c].back());
      r.el.push_back({});
      for (size_t q = 0; q + 1 < first[c].size(); q++) {  // an element named twice advances alike
        const std::pair<int, int> v{first[c][q], step[c][q]};
        bool seen = false;
        for (auto& w : r.el[c]) {
          ok = ok && (w.first != v.first || w.second == v.second);
          seen |= w.first == v.first;
        }
        if (!seen) r.el[c].push_back(v);
      }
    }
    // nothing outside reads the run's rows but through its two ends
    for (int i = 0; i < P.n && ok; i++) {
      if (r.has(i)) continue;
      for (int s = P.row_ptr[i]; s < P.row_ptr[i + 1]; s++)
        ok = ok && !(i < r.i0 && P.col[s] >= r.i0 + D && P.col[s] < r.i1) &&
             !(i >= r.i1 && P.col[s] >= r.i0 && P.col[s] < r.i1 - D);
    }
    if (ok) best = r;
    if (t > 1) i0 += (t - 1) * D;  // a later start within this run is shorter
  }
  return best.nit >= 8;
}

struct Gen {
  const View& P;
  const Run* run = nullptr;  // rows handled by a loop, their state in memory
  int run_total = 0;         // its 16-byte entries per lane
  std::ostringstream out;         // kernel text
  std::ostringstream* cur = &out; // where statements go
  std::vector<std::string> loads; // loads first needed by the row being generated
  std::set<int> have_g, have_p, have_x;
  std::string why;
  bool track_bm = false;          // mixed precision: |b|_inf^2 for the correction scale
  // mixed precision with the solution split as x = x0 + dx: x0 (the complex64
  // first solution) in LDS, dx (complex64 sum of the corrections) in registers
  bool xsplit = false;
  // element values from the table blocked by 64 instances (entry
  // (inst / 64 * ne + e) * 64 + inst % 64), so that a wave of consecutive
  // instances reads one contiguous run per value
  bool emajor = false;
  int lookahead = KG_LANE_AHEAD;  // rows between a load and the row that first uses it
  // names of element-value loads
  std::string gname = "g", pname = "p";
  // growth guard (first pass): an = ||A||_inf and gm = || |L||U| ||_inf in
  // |re| + |im| entry norms, the latter bounded from above through
  // |l_ik| <= |v_ik| |1/u_kk| (c1 is submultiplicative)
  bool growth = false;
  std::function<void(std::ostringstream&, int)> on_result;
  explicit Gen(const View& v) : P(v) {}

  // Element values come from the per-instance value table (1/R for plain
  // resistors, the element value otherwise: C, L, G2 resistors, current
  // sources), whose small offsets fit the loads' immediate field; only the
  // AC magnitude of voltage sources is read from the parameter records.
  std::string g(int e) {
    std::string nm = gname + std::to_string(e);
    if (have_g.insert(e).second) {
      if (emajor)  // buffer load: the wave's block (scalar), the lane's offset, a constant per element
        loads.push_back("    const double " + nm + " = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(EBR, jl8, " +
                        std::to_string(512 * e) + ", 0));\n");
      else
        loads.push_back("    const double " + nm + " = EB[" + std::to_string(e) + "];\n");
    }
    return nm;
  }
  std::string p(int e, int k) {  // params[e][k]
    std::string nm = pname + std::to_string(e) + "_" + std::to_string(k);
    if (have_p.insert(e * KG_NPARAM + k).second)
      loads.push_back("    const double " + nm + " = PR[" + std::to_string(e * KG_NPARAM + k) + "];\n");
    return nm;
  }
  // FP64 value of LU slot s as (re, im) expressions; both empty when the slot
  // receives no contribution. Follows the stamp kinds of the plan's gather
  // lists (AC stamps, stampable.rs): +-y (1/R, j w C), +-1, branch diagonal,
  // +-k (controlled-source gains).
  bool slot(int s, std::string& re, std::string& im) {
    std::vector<std::string> R, I;
    for (int q = P.scon_ptr[s]; q < P.scon_ptr[s + 1]; q++) {
      int code = P.scon[q], e = code >> 3, k = code & 7, ty = P.etype[e];
      switch (k) {
        case CK_YP:
        case CK_YN: {
          const char* sg = k == CK_YN ? "-" : "";
          if (ty == KG_R) R.push_back(sg + g(e));
          else if (ty == KG_C) I.push_back(std::string(sg) + "(w * " + g(e) + ")");
          else if (ty == KG_D) { why = "diode small-signal stamps are not generated"; return false; }
          break;
        }
        case CK_ONEP: R.push_back("1.0"); break;
        case CK_ONEN: R.push_back("-1.0"); break;
        case CK_BR:
          if (ty == KG_L) I.push_back("-(w * " + g(e) + ")");
          else if (ty == KG_R) R.push_back("-" + g(e));
          else R.push_back("1.0");
          break;
        case CK_KP: R.push_back(g(e)); break;  // controlled-source gain
        case CK_KN: R.push_back("-" + g(e)); break;
        default: why = "unknown stamp kind"; return false;
      }
    }
    auto join = [](const std::vector<std::string>& v) {
      std::string s;
      for (size_t i = 0; i < v.size(); i++) s += (i ? " + " : "") + v[i];
      return s;
    };
    re = join(R);
    im = join(I);
    return true;
  }
  bool has_slot(int s) const { return P.scon_ptr[s + 1] > P.scon_ptr[s]; }
  // FP64 right-hand side of row i (AC excitation, ac.rs: V sources carry their
  // AC magnitude, current sources their DC value); empty when zero.
  bool rhs(int i, std::string& re) {
    std::vector<std::string> R;
    for (int q = P.rcon_ptr[i]; q < P.rcon_ptr[i + 1]; q++) {
      int code = P.rcon[q], e = code >> 3, k = code & 7, ty = P.etype[e];
      if (k != RK_SRC) { why = "only source excitations are generated"; return false; }
      R.push_back(ty == KG_V ? p(e, 1) : g(e));
    }
    re.clear();
    for (size_t t = 0; t < R.size(); t++) re += (t ? " + " : "") + R[t];
    return true;
  }
  static std::string zexpr(const std::string& re, const std::string& im) {
    return "Z{" + (re.empty() ? std::string("0.0") : re) + ", " + (im.empty() ? std::string("0.0") : im) + "}";
  }
  static std::string conv(const std::string& F, const std::string& zval) {
    return F == "Z" ? zval : "cw(" + zval + ")";
  }

  // a * b, with a's real part only when a is known to be real
  static std::string mul(bool a_real, const std::string& a, const std::string& b) {
    return a_real ? "rmul(" + a + ".re, " + b + ")" : a + " * " + b;
  }

  // z - a * b likewise
  static std::string sub(bool a_real, const std::string& z, const std::string& a, const std::string& b) {
    return a_real ? z + " - rmul(" + a + ".re, " + b + ")" : "fms(" + z + ", " + a + ", " + b + ")";
  }

  // FP64 x_j for a residual: a register, or (xsplit) x0_j read from LDS ahead
  // of its row plus dx_j
  std::string xref(int j) {
    if (!xsplit) return "x" + std::to_string(j);
    std::string nm = "xl" + std::to_string(j);
    if (have_x.insert(j).second) loads.push_back("    const W " + nm + " = xs[" + std::to_string(64 * j) + " + lane];\n");
    return "(cz(" + nm + ") + cz(dx" + std::to_string(j) + "))";
  }

  // The run's rows (FP64, right-hand side b): chain c's upper factor, y' and
  // growth weight of the row before are carried in cu, cy and cg; U' and y'
  // of each row go to memory (ws, one 16-byte entry per lane), element values
  // are loaded four iterations ahead.
  int run_words(int c, const std::vector<char>& yz) const { return yz[run->i0 + c] ? 1 : 2; }
  int run_entry(int c, const std::vector<char>& yz) const {  // entry of chain c within an iteration
    int e = 0;
    for (int k = 0; k < c; k++) e += run_words(k, yz);
    return e;
  }
  void run_forward(std::ostringstream& O, const std::vector<char>& real, const std::vector<char>& yz) {
    const Run& R = *run;
    const int D = R.D, ne = run_entry(D, yz);
    run_total = R.nit * ne;
    auto nm = [](const char* p, int j, int c, int e) {
      return std::string(p) + std::to_string(j) + "_" + std::to_string(c) + "_" + std::to_string(e);
    };
    auto each = [&](auto f) {
      for (int j = 0; j < 4; j++)
        for (int c = 0; c < D; c++)
          for (auto& v : R.el[c]) f(j, c, v.first, v.second);
    };
    auto at = [&](int e, int st, int j, const char* it) {
      return "EB[" + std::to_string(e + st * j) + " + " + std::to_string(st) + " * " + it + "]";
    };
    for (int c = 0; c < D; c++) {
      const int k = R.i0 + c - D, us = P.fprog[P.fprog_ptr[R.i0 + c] + 5];
      O << "    Z cu" << c << " = u" << us << ";\n    double cg" << c << " = gw" << k << ";\n";
      if (!yz[k]) O << "    Z cy" << c << " = y" << k << "s;\n";
    }
    each([&](int j, int c, int e, int st) { O << "    double " << nm("n", j, c, e) << " = " << at(e, st, j, "0") << ";\n"; });
    O << "#pragma clang loop unroll(disable)\n    for (int it = 0; it < " << R.nit << "; it += 4) {\n"
      << "      const int nx = it + 4 < " << R.nit << " ? it + 4 : it;\n";
    each([&](int j, int c, int e, int st) {
      O << "      const double " << nm("h", j, c, e) << " = " << nm("n", j, c, e) << ";\n      " << nm("n", j, c, e) << " = "
        << at(e, st, j, "nx") << ";\n";
    });
    O << "      asm volatile(\"\" ::: \"memory\");\n";
    for (int j = 0; j < 4; j++)
      for (int c = 0; c < D; c++) {
        const int i = R.i0 + c, s0 = P.row_ptr[i];
        const std::string C = std::to_string(c);
        O << "      {\n";
        for (auto& v : R.el[c]) O << "        const double g" << v.first << " = " << nm("h", j, c, v.first) << ";\n";
        const char* name[3] = {"vl", "vd", "vu"};
        for (int q = 0; q < 3; q++) {
          std::string re, im;
          slot(s0 + q, re, im);
          O << "        Z " << name[q] << " = " << zexpr(re, im) << ";\n";
        }
        O << "        an = fmax(an, c1(vl) + c1(vd) + c1(vu));\n        gsr = c1(vl) * cg" << C << ";\n"
          << "        vd = " << sub(real[s0], "vd", "vl", "cu" + C) << ";\n";
        if (!yz[i]) O << "        const Z y = Z{0, 0} - " << mul(real[s0], "vl", "cy" + C) << ";\n";
        O << "        bad |= !piv_ok(vd);\n        const Z rd = rcpF(vd);\n"
          << "        const double gd = c1(vd), gr = gd + c1(vu);\n        gm = fmax(gm, gsr + gr);\n"
          << "        cg" << C << " = c1r(vd, rd, gd) * gr;\n        cu" << C << " = " << mul(real[s0 + 2], "vu", "rd") << ";\n";
        const int ent = run_entry(c, yz);
        O << "        ws[(i64)(it + " << j << ") * " << 64 * ne << " + " << 64 * ent << "] = cu" << C << ";\n";
        if (!yz[i])
          O << "        cy" << C << " = y * rd;\n        ws[(i64)(it + " << j << ") * " << 64 * ne << " + " << 64 * (ent + 1)
            << "] = cy" << C << ";\n";
        O << "      }\n";
      }
    O << "    }\n";
    for (int c = 0; c < D; c++) {
      const int i = R.i1 - D + c;
      O << "    const Z u" << P.diag[i] + 1 << " = cu" << c << ";\n    const double gw" << i << " = cg" << c << ";\n";
      if (!yz[i]) O << "    const Z y" << i << "s = cy" << c << ";\n";
    }
  }
  void run_backward(std::ostringstream& O, const std::vector<char>& yz) {
    const Run& R = *run;
    const int D = R.D, ne = run_entry(D, yz);
    auto nm = [](const char* p, int j, int q) { return std::string(p) + std::to_string(j) + "_" + std::to_string(q); };
    auto each = [&](auto f) {
      for (int j = 3; j >= 0; j--)
        for (int q = 0; q < ne; q++) f(j, q);
    };
    auto at = [&](int j, int q, const std::string& it) {
      return "ws[(i64)(" + it + " + " + std::to_string(j) + ") * " + std::to_string(64 * ne) + " + " + std::to_string(64 * q) + "]";
    };
    for (int c = 0; c < D; c++) O << "    Z ct" << c << " = t" << R.i1 + c << ";\n";
    each([&](int j, int q) { O << "    Z " << nm("m", j, q) << " = " << at(j, q, std::to_string(R.nit - 4)) << ";\n"; });
    O << "#pragma clang loop unroll(disable)\n    for (int it = " << R.nit - 4 << "; it >= 0; it -= 4) {\n"
      << "      const int nx = it >= 4 ? it - 4 : it;\n";
    each([&](int j, int q) {
      O << "      const Z " << nm("l", j, q) << " = " << nm("m", j, q) << ";\n      " << nm("m", j, q) << " = " << at(j, q, "nx")
        << ";\n";
    });
    O << "      asm volatile(\"\" ::: \"memory\");\n";
    for (int j = 3; j >= 0; j--)
      for (int c = 0; c < D; c++) {
        const int ent = run_entry(c, yz);
        O << "      ct" << c << " = fms(" << (yz[R.i0 + c] ? std::string("Z{0, 0}") : nm("l", j, ent + 1)) << ", "
          << nm("l", j, ent) << ", ct" << c << ");\n      const Z " << nm("t", j, c) << " = ct" << c << ";\n";
      }
    for (int c = 0; c < D; c++) {
      if (R.cstep[c] == 1 || R.cstep[c] == -1) {
        const bool up = R.cstep[c] == 1;
        O << "      st4(oq, " << R.col[c] << (up ? " + it" : " - it - 3");
        for (int j = 0; j < 4; j++) O << ", " << nm("t", up ? j : 3 - j, c);
        O << ");\n";
      } else {
        for (int j = 0; j < 4; j++)
          O << "      o[" << R.col[c] << " + " << R.cstep[c] << " * (it + " << j << ")] = " << nm("t", j, c) << ";\n";
      }
    }
    O << "    }\n";
    for (int c = 0; c < D; c++) O << "    const Z t" << R.i0 + c << " = ct" << c << ";\n";
  }

  // One factorisation + forward + backward pass in type F ("Z" or "W"),
  // appended to `out`. mode 0: right-hand side b; mode 1: scaled FP64
  // residual b - A x. Row i's back-substitution result t<i> is handed to
  // on_result.
  bool pass(const std::string& F, int mode) {
    const int n = P.n;
    have_g.clear();
    have_p.clear();
    have_x.clear();
    std::vector<std::string> code(n);
    std::vector<std::vector<std::string>> rload(n);
    std::vector<char> yz(n, 1);  // y'_i structurally zero
    // slot value has no imaginary part: its stamp is real and no elimination
    // step has updated it yet (products with it take the real form)
    std::vector<char> real(P.nnz, 0);
    for (int i = 0; i < n; i++) {
      std::ostringstream o;
      loads.clear();
      const std::set<int> held = have_g;
      // gather row i
      for (int s = P.row_ptr[i]; s < P.row_ptr[i + 1]; s++) {
        std::string re, im;
        if (!slot(s, re, im)) return false;
        real[s] = im.empty();
        if (mode == 1 || (growth && F == "W")) {
          if (has_slot(s)) o << "    const Z a" << s << " = " << zexpr(re, im) << ";\n";
          o << "    " << F << " v" << s << " = "
            << (has_slot(s) ? conv(F, "a" + std::to_string(s)) : F + "{0, 0}") << ";\n";
        } else {
          o << "    " << F << " v" << s << " = " << conv(F, zexpr(re, im)) << ";\n";
        }
      }
      const bool gg = growth && mode == 0;
      if (gg) {  // ||A||_inf: this row's sum of |a|
        o << "    an = fmax(an, 0.0";
        for (int s = P.row_ptr[i]; s < P.row_ptr[i + 1]; s++)  // complex64: from the FP64 stamps
          if (has_slot(s)) o << " + c1(" << (F == "W" ? "a" : "v") << s << ")";
        o << ");\n    gsr = 0.0;\n";
      }
      // right-hand side of row i
      bool ynz = false;
      std::string b;
      if (!rhs(i, b)) return false;
      if (mode == 0) {
        if (!b.empty()) {
          o << "    " << F << " y" << i << " = " << conv(F, "Z{" + b + ", 0.0}") << ";\n";
          if (track_bm) o << "    bm2 = fmax(bm2, m2(Z{" << b << ", 0.0}));\n";
          ynz = true;
        }
      } else {
        o << "    Z r" << i << " = " << (b.empty() ? std::string("Z{0.0, 0.0}") : "Z{" + b + ", 0.0}") << ";\n";
        for (int s = P.row_ptr[i]; s < P.row_ptr[i + 1]; s++)
          if (has_slot(s))
            o << "    r" << i << " = "
              << sub(real[s], "r" + std::to_string(i), "a" + std::to_string(s), xref(P.col[s])) << ";\n";
        o << "    " << F << " y" << i << " = " << conv(F, "scal(inv_s, r" + std::to_string(i) + ")") << ";\n";
        ynz = true;
      }
      // factor row i: the plan's factor program for this row
      const int32_t* fp = P.fprog + P.fprog_ptr[i];
      int nk = *fp++;
      for (int kk = 0; kk < nk; kk++) {
        int sik = fp[0], k = P.col[sik], nu = fp[2];
        fp += 3;
        // |l_ik| (row sum of |U| row k) <= |v_ik| w_k, v_ik final here
        if (gg) o << "    gsr = gsr + c1(v" << sik << ") * gw" << k << ";\n";
        for (int u = 0; u < nu; u++, fp += 2) {
          int dst = fp[0], src = fp[1];
          if (!(src > P.diag[k] && src < P.row_ptr[k + 1])) { why = "factor program reads outside U"; return false; }
          o << "    v" << dst << " = " << sub(real[sik], "v" + std::to_string(dst), "v" + std::to_string(sik),
                                             "u" + std::to_string(src)) << ";\n";
          real[dst] = 0;
        }
        if (!yz[k]) {
          const std::string a = "v" + std::to_string(sik), b = "y" + std::to_string(k) + "s";
          if (!ynz) o << "    " << F << " y" << i << " = " << F << "{0, 0} - " << mul(real[sik], a, b) << ";\n";
          else o << "    y" << i << " = " << sub(real[sik], "y" + std::to_string(i), a, b) << ";\n";
          ynz = true;
        }
      }
      // pivot: decomposition check as the generic kernels (|piv| > 0, finite);
      // refinement passes repeat the first pass' factorisation exactly, so
      // only the first pass checks every pivot; they repeat the check of
      // their last pivot, whose only effect is on register allocation (with
      // no check at all in the refinement passes, the mixed kernel of the
      // 50-section RC ladder takes 512 registers and 596 B of scratch per
      // lane instead of 360 registers)
      int d = P.diag[i];
      if (mode == 0 || i == n - 1) o << "    bad |= !piv_ok(v" << d << ");\n";
      o << "    const " << F << " rd" << i << " = rcpF(v" << d << ");\n";
      if (gg) {  // row i of U: its sum of |u|, the diagonal term of |L||U|, and w_i = |1/u_ii| sum
        o << "    const double gd" << i << " = c1(v" << d << "), gr" << i << " = gd" << i;
        for (int s = d + 1; s < P.row_ptr[i + 1]; s++) o << " + c1(v" << s << ")";
        o << ";\n    gm = fmax(gm, gsr + gr" << i << ");\n    const double gw" << i << " = c1r(v" << d << ", rd" << i
          << ", gd" << i << ") * gr" << i << ";\n";
      }
      for (int s = d + 1; s < P.row_ptr[i + 1]; s++)
        o << "    const " << F << " u" << s << " = " << mul(real[s], "v" + std::to_string(s), "rd" + std::to_string(i))
          << ";\n";
      if (ynz) {
        o << "    const " << F << " y" << i << "s = y" << i << " * rd" << i << ";\n";
        yz[i] = 0;
      }
      if (run && run->has(i)) {  // the loop loads for itself
        have_g = held;
        continue;
      }
      code[i] = o.str();
      rload[i] = loads;
    }
    // rows with their loads issued `lookahead` rows early
    std::ostringstream& O = out;
    auto issue = [&](int r) {
      if (r >= n || rload[r].empty()) return;
      for (auto& l : rload[r]) O << l;
      O << "    asm volatile(\"\" ::: \"memory\");\n";
      rload[r].clear();
    };
    for (int r = 0; r < lookahead; r++) issue(r);
    for (int i = 0; i < n; i++) {
      if (run && i == run->i0) {
        run_forward(O, real, yz);
        i = run->i1;
        for (int r = 0; r < lookahead; r++) issue(i + r);
      }
      issue(i + lookahead);
      O << code[i];
      if (KG_LANE_FWD_BARRIER > 0 && (i + 1) % KG_LANE_FWD_BARRIER == 0) O << "    __builtin_amdgcn_sched_barrier(0);\n";
    }
    // back substitution
    for (int i = n - 1; i >= 0; i--) {
      if (run && i == run->i1 - 1) {
        run_backward(O, yz);
        i = run->i0 - 1;
        if (i < 0) break;
      }
      std::string acc = yz[i] ? F + "{0, 0}" : "y" + std::to_string(i) + "s";
      O << "    " << F << " t" << i << " = " << acc << ";\n";
      for (int s = P.diag[i] + 1; s < P.row_ptr[i + 1]; s++)
        O << "    t" << i << " = fms(t" << i << ", u" << s << ", t" << P.col[s] << ");\n";
      on_result(O, i);
      if (KG_LANE_BWD_BARRIER > 0 && i % KG_LANE_BWD_BARRIER == 0) O << "    __builtin_amdgcn_sched_barrier(0);\n";
    }
    return true;
  }
};

}  // namespace

const char* jit_ac_name(bool mixed, bool xsplit, bool looped) {
  return looped ? "kg_ac_lane_c128_loop" : !mixed ? "kg_ac_lane_c128" : xsplit ? "kg_ac_lane_c64_split" : "kg_ac_lane_c64";
}

bool jit_ac_source(const PatLayout& L, const int32_t* buf, bool mixed, bool xsplit, std::string& src,
                   std::string& why, int* loop_words) {
  View P = view(L, buf);
  const int n = P.n;
  const bool looped = loop_words != nullptr;
  if (L.status != KG_OK) { why = "structurally singular pattern"; return false; }
  if (L.has_diode) { why = "diode small-signal stamps are not generated"; return false; }
  Run run, two;
  if (looped) {
    const bool one = find_run(P, 1, run);
    if (find_run(P, 2, two) && (!one || 2 * two.nit > run.nit)) run = two;
    else if (!one) { why = "no chain of rows alike"; return false; }
  }
  int nu = 0, nr = 0;
  for (int i = 0; i < n; i++)
    if (!run.has(i)) nu += P.row_ptr[i + 1] - P.diag[i] - 1, nr++;
  // registers per lane held across a pass: U' and y' (and the FP64 solution
  // for mixed precision); the register file holds 512 per lane at one wave
  // per SIMD, and the pass needs a few dozen more for its temporaries
  // (xsplit: dx in registers, x0 in 512 * n bytes of LDS per 64-lane block;
  // looped: the rows outside the loop)
  int regs = !mixed ? 4 * (nu + nr) : 2 * (nu + n) + (xsplit ? 2 * n : 4 * n);
  if (mixed && xsplit && n > 78) { why = "x0 would not fit in LDS at four waves per CU"; return false; }
  if (regs > (looped ? 200 : 440)) { why = "per-lane state exceeds the register budget"; return false; }
  Gen G(P);
  if (looped) G.run = &run;
  G.xsplit = mixed && xsplit;
  G.emajor = mixed;
  std::ostringstream& o = G.out;
  o << kPrelude;
  o << "extern \"C\" __global__ void __launch_bounds__(64) " << jit_ac_name(mixed, xsplit, looped)
    << "(const double* __restrict__ prm,\n"
       "    const double* __restrict__ ebase, const double* __restrict__ freqs, int nf, i64 nsys,\n"
       "    double* __restrict__ out, int* __restrict__ status, double* __restrict__ err, int refine,\n"
       "    double stop, unsigned long long* __restrict__ fixq, i64 fixcap"
    << (looped ? ", Z* __restrict__ wsb" : "") << ") {\n";
  // looped: each block takes every gridDim-th group of 64 systems, its region of the workspace its own
  if (looped) o << "  for (i64 blk = xcd_block(); blk * 64 < nsys; blk += gridDim.x) {\n";
  o << "  const i64 sys0 = " << (looped ? "blk" : "xcd_block()") << " * 64 + threadIdx.x;\n";
  // lanes past the last system repeat it (identical values to the same
  // addresses; they queue nothing), so that the whole wave stays active for
  // the stores by quads and the error figure's wave reduction
  o << "  const bool live = sys0 < nsys;\n  const i64 sys = live ? sys0 : nsys - 1;\n";
  if (!mixed) {  // consecutive frequencies of one instance per wave (element loads shared by the wave)
    o << "  const int inst = (int)(sys / nf), fi = (int)(sys - (i64)inst * nf);\n";
  } else {
    // 64 instances at one frequency per wave: refinement converges alike
    // across the wave, so the adaptive stop applies to whole waves
    // (measured: 0.49 ms instead of 0.78 ms on the 4096 x 200 RC-ladder
    // sweep; the FP64 kernel is faster with the instance-major order)
    o << "  const i64 ni = nsys / nf, ib = sys / (64 * (i64)nf), rem = sys - ib * 64 * (i64)nf;\n"
         "  const int nbi = (int)(ni - ib * 64 < 64 ? ni - ib * 64 : 64);\n"
         "  const int fi = (int)(rem / nbi), inst = (int)(ib * 64 + rem % nbi);\n";
  }
  if (mixed) {
    // ib is uniform across the wave (64 * nf consecutive systems per group of
    // 64 instances): the group's block of values as a buffer resource
    // (descriptor word 3 of gfx9 raw buffers; reads past the block return 0)
    o << "  const __amdgpu_buffer_rsrc_t EBR = __builtin_amdgcn_make_buffer_rsrc((void*)(ebase + "
         "(i64)__builtin_amdgcn_readfirstlane((int)ib) * "
      << 64 * P.ne << "), (short)0, " << 512 * P.ne << ", 0x00020000);\n"
      << "  const int jl8 = (inst - (int)ib * 64) * 8;\n";
  }
  else o << "  const double* EB = ebase + (i64)inst * " << P.ne << ";\n";
  o << "  const double* PR = prm + (i64)inst * " << (int64_t)P.ne * KG_NPARAM << ";\n"
    << "  const double w = (2.0 * 3.14159265358979323846) * freqs[fi];\n"
    << "  const i64 orow = ((i64)inst * nf + fi) * " << n << ";\n  Z* o = reinterpret_cast<Z*>(out) + orow;\n"
    << "  bool bad = false;\n";
  // growth guard: computed during the first pass' factorisation
  G.growth = true;
  int mrow = 1;
  for (int i = 0; i < n; i++) mrow = std::max(mrow, (int)(P.row_ptr[i + 1] - P.row_ptr[i]));
  o << "  double an = 0.0, gm = 0.0, gsr = 0.0;\n";
  if (!mixed) {
    // results wait for the other three of their group of four consecutive unknowns
    std::vector<int> left(n / 4 + 1, 4), row_of(n);
    for (int i = 0; i < n; i++) row_of[P.col_of[i]] = i;
    G.on_result = [&](std::ostringstream& O, int i) {
      const int c = P.col_of[i], g = c / 4;
      if (4 * g + 4 > n) O << "    o[" << c << "] = t" << i << ";\n";
      else if (looped) O << "    o[" << c << "] = t" << i << ";\n";  // its group may be the loop's
      else if (--left[g] == 0) O << "    st4(oq, " << 4 * g << st4_args(row_of, g, "t") << ");\n";
    };
    o << "  const Quad oq = quad_rows(reinterpret_cast<Z*>(out), orow);\n";
    if (looped) o << "  Z* const ws = wsb + (i64)blockIdx.x * KG_LOOP_WORDS * 64 + threadIdx.x;\n";
    o << "  {\n";
    if (!G.pass("Z", 0)) { why = G.why; return false; }
    // rho = gm / an above KG_GUARD_GROWTH (or a failed pivot): re-solved by
    // the fixup; else the instance's figure is the backward-error bound
    // c_m rho of the solve
    // the figure is reduced over the wave first: its lanes hold one or two
    // instances (consecutive frequencies), and 64 atomics on one address
    // serialise (a segmented maximum over lanes of the same instance, then
    // one atomic per instance)
    o << "  }\n"
      << "  const bool queue = bad || !(gm <= " << fmt_double(KG_GUARD_GROWTH) << " * an);\n"
      << "  if (queue && live) fix_push(fixq, fixcap, (i64)inst * nf + fi, status, inst);\n"
      << "  if (err != nullptr) {\n"
      << "    const int lane = threadIdx.x;\n"
      << "    double ev = queue || !(gm > 0.0) ? 0.0 : " << fmt_double(guard_bound_coeff(mrow)) << " * (gm / an);\n"
      << "    for (int off = 1; off < 64; off <<= 1) {\n"
      << "      const double ov = __shfl_down(ev, off, 64);\n"
      << "      const int oi = __shfl_down(inst, off, 64);\n"
      << "      if (lane + off < 64 && oi == inst) ev = fmax(ev, ov);\n"
      << "    }\n"
      << "    const int pi = __shfl_up(inst, 1, 64);\n"
      << "    if ((lane == 0 || pi != inst) && ev > 0.0)\n"
      << "      atomicMax(reinterpret_cast<unsigned long long*>(&err[inst]), (unsigned long long)__double_as_longlong(ev));\n"
      << "  }\n"
      << (looped ? "  }\n}\n" : "}\n");
    src = o.str();
    if (looped) {
      *loop_words = G.run_total;
      src = "#define KG_LOOP_WORDS " + std::to_string(G.run_total) + "\n" + src;
    }
    return true;
  } else {
    if (G.xsplit) {
      o << "  extern __shared__ W xs[];\n  const int lane = threadIdx.x;\n";
      for (int i = 0; i < n; i++) o << "  W dx" << i << " = W{0.0f, 0.0f};\n";
    } else {
      for (int i = 0; i < n; i++) o << "  Z x" << i << ";\n";
    }
    o << "  double est = 0.0, d2prev = 0.0, d2last = 0.0, bm2 = 0.0;\n  float xmf = 0.0f;\n  int npass = 0;\n";
    // pass 0: complex64 solve of b; x = its FP64 copy (xsplit: x0 = it, dx = 0)
    // |x|_inf is taken from this first solution (the refinement changes it by
    // the FP32 solve error only); tracking it through the refinement passes
    // makes the compiler keep far more values live
    G.on_result = [&](std::ostringstream& O, int i) {
      if (G.xsplit) O << "    xs[" << 64 * i << " + lane] = t" << i << "; xmf = cmax(xmf, t" << i << ");\n";
      else O << "    x" << i << " = cz(t" << i << "); xmf = cmax(xmf, t" << i << ");\n";
    };
    G.track_bm = true;
    o << "  {\n";
    if (!G.pass("W", 0)) { why = G.why; return false; }
    // the growth verdict is taken here, so that only a lane mask stays live
    // through the refinement
    o << "  }\n  bad |= !(gm <= " << fmt_double(KG_GUARD_GROWTH) << " * an);\n";
    G.track_bm = false;
    // refinement: corrections scaled by |b|_inf stay in FP32 range
    o << "  const double s = sqrt(bm2), inv_s = s > 0.0 ? 1.0 / s : 0.0, xm2 = (double)xmf * (double)xmf;\n"
         "  const float sf = (float)s;\n";
    // refinement passes after the first run inside a run-time loop: the pass
    // body is compiled once, so its registers are allocated once (an unrolled
    // sequence of passes lets live ranges of neighbouring passes overlap)
    G.on_result = [&](std::ostringstream& O, int i) {
      // (xsplit: the correction is formed and accumulated in complex64, the
      // precision dx is kept in; FP64 here costs registers, not accuracy)
      if (G.xsplit)
        O << "    { const W d = W{sf * t" << i << ".re, sf * t" << i << ".im}; dx" << i << " = W{dx" << i << ".re + d.re, dx"
          << i << ".im + d.im}; dmf = cmax(dmf, t" << i << "); }\n";
      else
        O << "    x" << i << " = x" << i << " + scal(s, cz(t" << i << ")); dmf = cmax(dmf, t" << i << ");\n";
    };
    // the first pass is peeled off the loop: a wave-uniform branch around the
    // remaining passes (adaptive stop) leaves the loop itself unchanged,
    // while an exit inside it makes the compiler spill
    o << "  if (s > 0.0 && refine > 0) {\n  {\n    float dmf = 0.0f;\n";
    G.lookahead = LOOKAHEAD_REFINE;
    if (!G.pass("W", 1)) { why = G.why; return false; }
    // only the squared correction sizes of the last two passes are carried;
    // the estimate is formed after the loop (square roots and divisions in
    // the loop body make the compiler keep far more values live)
    o << "    d2prev = d2last;\n    d2last = s * (double)dmf * (s * (double)dmf);\n    npass = 1;\n  }\n";
    // adaptive stop (stop > 0): a wave leaves after the first pass once every
    // lane's predicted remaining error, the squared relative correction times
    // KG_REFINE_SAFETY (refinement contracts by about the relative size of
    // its correction), is at most `stop`
    o << "  if (refine > 1 && !(stop > 0.0 && __builtin_amdgcn_ballot_w64(" << KG_REFINE_SAFETY
      << " * d2last <= stop * xm2) == __builtin_amdgcn_read_exec()))\n"
         "#pragma clang loop unroll(disable)\n"
         "  for (int it = 1; it < refine; it++) {\n    float dmf = 0.0f;\n";
    if (!G.pass("W", 1)) { why = G.why; return false; }
    o << "    d2prev = d2last;\n    d2last = s * (double)dmf * (s * (double)dmf);\n    npass = it + 1;\n  }\n  }\n"
      << "  {\n    const double dm = sqrt(d2last), dp = sqrt(d2prev), xm = sqrt(xm2);\n"
      << "    const double rho = (npass > 1 && dp > 0.0) ? fmin(dm / dp, 1.0) : 1.0;\n"
      << "    est = xm > 0.0 ? (npass == 1 && stop > 0.0 ? " << KG_REFINE_SAFETY
      << " * d2last / xm2 : rho * dm / xm) : 0.0;\n  }\n";
    std::vector<int> row_of(n);
    for (int i = 0; i < n; i++) row_of[P.col_of[i]] = i;
    if (G.xsplit)
      for (int i = 0; i < n; i++) o << "#define x" << i << " (cz(xs[" << 64 * i << " + lane]) + cz(dx" << i << "))\n";
    o << "  const Quad oq = quad_rows(reinterpret_cast<Z*>(out), orow);\n";
    for (int g = 0; 4 * g + 4 <= n; g++) o << "  st4(oq, " << 4 * g << st4_args(row_of, g, "x") << ");\n";
    for (int c = n / 4 * 4; c < n; c++) o << "  o[" << c << "] = x" << row_of[c] << ";\n";
    // a solve whose complex64 factorisation grew (rho above
    // KG_GUARD_GROWTH), whose estimate stays above KG_GUARD_MIXED or whose
    // complex64 pivots failed is solved again in FP64 with partial pivoting
    // by the fixup
    o << "  if ((bad || !(est <= " << fmt_double(KG_GUARD_MIXED) << ")) && live)\n    fix_push(fixq, fixcap, (i64)inst * nf + fi, status, inst);\n"
         "  else if (live && err != nullptr && est > 0.0)\n"
         "    atomicMax(reinterpret_cast<unsigned long long*>(&err[inst]), (unsigned long long)__double_as_longlong(est));\n";
  }
  o << "}\n";
  src = o.str();
  return true;
}

namespace {
std::mutex g_mu;
std::map<std::pair<int, std::string>, std::pair<hipModule_t, JitFn>> g_cache;
}  // namespace

hipError_t jit_load(int device, const std::string& src, const char* name, JitFn& out, std::string& log) {
  std::lock_guard<std::mutex> lk(g_mu);
  auto key = std::make_pair(device, src + "\n//" + name);
  auto it = g_cache.find(key);
  if (it != g_cache.end()) {
    out = it->second.second;
    return hipSuccess;
  }
  hipDeviceProp_t prop;
  hipError_t e = hipGetDeviceProperties(&prop, device);
  if (e != hipSuccess) return e;
  std::string arch = std::string("--offload-arch=") + prop.gcnArchName;
  hiprtcProgram prog;
  if (hiprtcCreateProgram(&prog, src.c_str(), "kg_jit.hip", 0, nullptr, nullptr) != HIPRTC_SUCCESS) {
    log = "hiprtcCreateProgram failed";
    return hipErrorInvalidValue;
  }
  // packed FP32 instructions stay disabled, as for the prebuilt kernels
  const char* opts[] = {arch.c_str(), "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
                        "-packed-fp32-ops"};
  hiprtcResult rc = hiprtcCompileProgram(prog, 7, opts);
  size_t ls = 0;
  hiprtcGetProgramLogSize(prog, &ls);
  log.assign(ls, '\0');
  if (ls) hiprtcGetProgramLog(prog, &log[0]);
  if (rc != HIPRTC_SUCCESS) {
    hiprtcDestroyProgram(&prog);
    return hipErrorInvalidValue;
  }
  size_t cs = 0;
  hiprtcGetCodeSize(prog, &cs);
  std::vector<char> code(cs);
  hiprtcGetCode(prog, code.data());
  hiprtcDestroyProgram(&prog);
  hipModule_t mod;
  if ((e = hipModuleLoadData(&mod, code.data())) != hipSuccess) return e;
  JitFn f;
  if ((e = hipModuleGetFunction(&f.fn, mod, name)) != hipSuccess) return e;
  (void)hipFuncGetAttribute(&f.vgprs, HIP_FUNC_ATTRIBUTE_NUM_REGS, f.fn);
  (void)hipFuncGetAttribute(&f.scratch, HIP_FUNC_ATTRIBUTE_LOCAL_SIZE_BYTES, f.fn);
  g_cache[key] = {mod, f};
  out = f;
  return hipSuccess;
}

}  // namespace kg
