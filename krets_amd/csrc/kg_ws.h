// Wave-subtree plan of a linear system's triangular solves, shared by the
// host builder (wsplan.cpp) and the kernels.
//
// The rows of the elimination forest are cut into pieces: the top rows (at
// most 64, closed towards the root) and, below them, subtrees that are dealt
// out to the nw waves of a block. No row of one wave couples to a row of
// another, so a wave runs all its levels alone, ordered by its own LDS
// operations, and the block meets only before and after the top rows, which
// wave 0 solves. One lane owns up to R rows ("slots") for a whole step loop,
// with their factors in registers.
//
// A row's level is one more than the largest level of the rows it couples to
// from below (in either factor). Lower solve: a slot's entries are consumed
// level by level: pair l holds the (at most two) entries whose columns lie at
// level l, so that every level is one round trip for every row, however long
// the row. A pseudo slot sums a top row's entries in one wave and leaves the
// sum in a partial that wave 0 adds. Upper solve: levels downwards, at most
// two entries a row. Neither solve has branches: a slot takes part in every
// level up to its number of pairs, with zero factors where it has no entry,
// and rewrites its unknown at each; values written before a row's own level
// are never read as final, later ones repeat it. Systems whose rows couple to
// more rows of one level (meshes) do not take this form.
#pragma once
#include <cstdint>

#ifdef __HIP__
#define KG_WS_HD __host__ __device__
#else
#define KG_WS_HD
#endif

namespace kg {

constexpr int WS_TOP_MAX = 64;
constexpr int WS_R_MAX = 4;      // slots and elements per lane
constexpr int WS_AE_MAX = 7;     // elements per lane of the transposed plan
constexpr int WS_TOP_PAIRS = 4;  // pairs (levels) of a top row

// Pairs of slot r, and the highest level a row in it may have. Slots are dealt
// in order of decreasing level: on the nested-dissection order of a chain
// about 2/3 of a wave's rows over 2^l lie above level l, so only the first
// slots hold deep rows.
KG_WS_HD constexpr int ws_pairs(int r) { return r == 0 ? 9 : r == 1 ? 3 : 1; }

// Solution columns per lane of the waves that move them (all but wave 0,
// which solves the top rows meanwhile): enough for nw waves' slots, but the
// top rows come on top of these, so that a plan also needs n to stay within.
KG_WS_HD constexpr int ws_cols(int nw, int rows) { return nw == 1 ? rows : (rows * nw + nw - 2) / (nw - 1); }
KG_WS_HD constexpr int ws_cols_max(int nw, int rows) { return 64 * ws_cols(nw, rows) * (nw == 1 ? 1 : nw - 1); }

// The transposed plan (discrete adjoint) is the same over U^T and L^T: its
// lower solve divides by the diagonal. Its elements are all R, C and L; an
// element whose history rows of several waves read has an instance in each.
//
// Slot record (WS_SLOT words): row (n + 1 + k: pseudo, partial k), level, first
// pair (`level` of them), the upper entries' columns (n: none) and LU slots
// (nnz: none), diagonal slot (nnz: none), first right-hand side code, codes,
// column in krets numbering, and for top rows first partial and partials.
enum : int { WSR_ROW, WSR_LEV, WSR_PAIR, WSR_UC0, WSR_UC1, WSR_US0, WSR_US1, WSR_DIAG, WSR_RHS, WSR_NRHS, WSR_PART,
             WSR_NPART, WSR_COL, WS_SLOT = 13 };
// Pair (4 words): column, LU slot, column, LU slot (n, nnz where absent).
// Right-hand side code: history index << 1 | negate. Element record: history index, kind (1 C, 2 L), plus, minus,
// branch column (n where absent), element. Source record: history index,
// source.
enum : int { WSE_HIST, WSE_KIND, WSE_P, WSE_M, WSE_C, WSE_E, WS_ELEM = 6 };
constexpr int WS_SRC = 2;
// Element record of the transposed plan: kind (0 R, 1 C, 2 L), element, the
// rows whose adjoints differ across it (L: its branch row, n), the krets
// columns whose states differ across it (L: its branch, n; n: ground), the
// history its node columns read, the one its branch column reads (L), and
// whether this instance carries the gradient. Histories without a reader: the
// unread one.
enum : int { WSA_KIND, WSA_E, WSA_A, WSA_B, WSA_P, WSA_M, WSA_H1, WSA_H2, WSA_GRAD, WS_AELEM = 9 };
// Wave record: first and last slot, element and source (one source a lane),
// levels.
enum : int { WSW_S0, WSW_S1, WSW_E0, WSW_E1, WSW_V0, WSW_V1, WSW_NL, WS_WAVE = 7 };

// After the waves' elements come ntel more (at most 64) that several waves'
// unknowns touch: only top rows read their histories, and wave 0 updates them
// beside the top rows, when the solution before is complete.
// Header; o_*: offsets in 16-bit words from the start of the plan. Histories
// 0 .. ndyn - 1: the companion currents of capacitors and inductors in the
// compact plan's order; ndyn .. ndyn + nsrc - 1: source values; ndyn + nsrc:
// zero (transposed plan: ndyn histories, the elements' own numbering; nsrc 0).
// o_cpos: per krets column the row, or n for a top row.
struct WsHdr {
  int32_t n, nnz, ndyn, nsrc, nw, rows, elems, ntop;
  int32_t npart, o_wave, o_slot, o_top, o_elem, o_src, o_pair, o_rhs;
  int32_t o_cpos, nrhs, more, top_nl, ntel, words, adjoint, pad;  // more: some row has over two right-hand side codes
};

// LDS of one system, in doubles from its start: right-hand side codes; then
// the factors and a scratch vector, until the lanes have taken their entries,
// and over them the step's arrays: solution x (a zero at n, an unread slot at
// n + 1), lower solution y (a zero at n, the partials, a zero, an unread
// slot), histories (a zero, an unread slot), 64 steps of source values, and
// the top rows' factors and indices.
constexpr int WS_TOP_D = 2 * WS_TOP_PAIRS + 3, WS_TOP_I = WS_TOP_PAIRS + 6;  // doubles and 32-bit words per top row
struct WsLds {
  int y, hist, sbuf, top, total;  // x at 0
};
// The transposed plan: no sources; sbuf holds two states of the trajectory
// (krets numbering, a zero at n).
KG_WS_HD inline WsLds ws_lds(const WsHdr& h) {
  WsLds l;
  l.y = h.n + 2;
  l.hist = l.y + h.n + h.npart + 3;
  l.sbuf = l.hist + h.ndyn + h.nsrc + 2;
  l.top = l.sbuf + (h.adjoint ? 2 * (h.n + 1) : 64 * h.nsrc);
  l.total = l.top + (WS_TOP_D + WS_TOP_I / 2) * h.ntop;
  return l;
}
KG_WS_HD inline size_t ws_list_bytes(const WsHdr& h) { return (2 * (size_t)h.nrhs + 15) & ~size_t(15); }
KG_WS_HD inline size_t ws_bytes(const WsHdr& h) {
  const size_t fac = (size_t)h.nnz + h.n + 2, step = (size_t)ws_lds(h).total;
  return 64 + ws_list_bytes(h) + 8 * (fac > step ? fac : step);
}

}  // namespace kg
