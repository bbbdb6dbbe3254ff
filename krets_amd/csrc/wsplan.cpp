// Builds the wave-subtree plan (kg_ws.h) of a linear transient from the
// pattern's plan buffer and its compact plan.
#include <algorithm>
#include <cstring>
#include <queue>
#include <vector>

#include "kg_internal.h"
#include "kg_ws.h"

namespace kg {

namespace {

using Lists = std::vector<std::vector<std::pair<int, int>>>;  // row -> (column, LU slot)

uint16_t u16(int v) { return (uint16_t)v; }

}  // namespace

// nw: waves per block. Returns false when the system does not take this form
// (more than two couplings to one level, too many top rows, rows per wave,
// columns or levels, an element shared by two waves, or indices beyond 16 bits).
// adjoint: the transposed plan.
bool build_ws_plan(const PatLayout& L, const std::vector<int32_t>& b, const std::vector<uint16_t>& lin, int nw,
                   bool adjoint, std::vector<uint16_t>& out) {
  out.clear();
  if (L.status != KG_OK || lin.empty() || (nw != 1 && nw != 2 && nw != 4 && nw != 8)) return false;
  LinHdr lh;
  std::memcpy(&lh, lin.data(), sizeof lh);
  const int n = L.n, nnz = L.nnz;
  if (n > 64 * WS_R_MAX * nw + (nw > 1 ? WS_TOP_MAX : 0)) return false;  // more rows than lanes, whatever the cut
  const int32_t* rp = b.data() + L.o_row_ptr;
  const int32_t* col = b.data() + L.o_col;
  const int32_t* dg = b.data() + L.o_diag;
  {  // more than two upper entries in a row: declined below whatever the cut
    std::vector<uint8_t> nup(n, 0);
    for (int i = 0; i < n; i++)
      for (int p = rp[i]; p < rp[i + 1]; p++)
        if ((adjoint ? col[p] < i : col[p] > i) && ++nup[adjoint ? col[p] : i] > 2) return false;
  }
  Lists lo(n), up(n);
  for (int i = 0; i < n; i++)
    for (int p = rp[i]; p < rp[i + 1]; p++) {
      const int r = adjoint ? col[p] : i, c = adjoint ? i : col[p];
      if (c != r) (c < r ? lo[r] : up[r]).push_back({c, p});
    }
  // elimination forest of the symmetrised factor pattern
  std::vector<int> parent(n, n), size(n, 1);
  for (int i = 0; i < n; i++) {
    for (auto& e : lo[i]) parent[e.first] = std::min(parent[e.first], i);
    for (auto& e : up[i]) parent[i] = std::min(parent[i], e.first);
  }
  std::vector<std::vector<int>> kids(n + 1);
  for (int i = 0; i < n; i++) {
    kids[parent[i]].push_back(i);
    if (parent[i] < n) size[parent[i]] += size[i];
  }
  // cut: the largest subtree gives its root to the top until every subtree
  // is at most an even share (a tenth more, to keep near-equal halves whole)
  auto smaller = [&](int x, int y) { return size[x] != size[y] ? size[x] < size[y] : x < y; };
  std::priority_queue<int, std::vector<int>, decltype(smaller)> roots(smaller);
  for (int r : kids[n]) roots.push(r);
  std::vector<char> top(n, 0);
  int ntop = 0;
  const int share = (n + nw - 1) / nw, most = nw == 1 ? n : share + share / 10 + 1;
  while (!roots.empty() && size[roots.top()] > most) {
    const int r = roots.top();
    roots.pop();
    if (++ntop > WS_TOP_MAX) return false;
    top[r] = 1;
    for (int k : kids[r]) roots.push(k);
  }
  // deal the subtrees out, largest first, each to the least loaded wave
  std::vector<int> wave(n, -1), load(nw, 0);
  std::vector<int> piece;
  while (!roots.empty()) {
    piece.push_back(roots.top());
    roots.pop();
  }
  for (int r : piece) {
    const int w = (int)(std::min_element(load.begin(), load.end()) - load.begin());
    load[w] += size[r];
    wave[r] = w;
  }
  for (int i = n - 1; i >= 0; i--)
    if (!top[i] && wave[i] < 0) wave[i] = wave[parent[i]];
  // no coupling between waves, and the top only above its neighbours
  for (int i = 0; i < n; i++) {
    for (auto& e : lo[i])
      if (top[e.first] ? !top[i] : (!top[i] && wave[e.first] != wave[i])) return false;
    for (auto& e : up[i])
      if (top[i] ? !top[e.first] : (!top[e.first] && wave[e.first] != wave[i])) return false;
  }
  auto same = [&](int i, int j) { return top[i] ? top[j] != 0 : !top[j] && wave[i] == wave[j]; };
  std::vector<int> lev(n, 0);
  for (int i = 0; i < n; i++) {  // the rows below i are final by now
    for (auto& e : lo[i])
      if (same(i, e.first)) lev[i] = std::max(lev[i], lev[e.first] + 1);
    for (auto& e : up[i])
      if (same(i, e.first)) lev[e.first] = std::max(lev[e.first], lev[i] + 1);
  }

  // right-hand side codes per row, and each wave's element and source records
  if (n >= 0x7FFF || nnz >= 0xFFFF) return false;
  const uint16_t* lw = lin.data();
  const int32_t* col_of = b.data() + L.o_col_of;
  auto col_or = [&](uint16_t v) { return v == LIN_NONE ? n : (int)v; };
  auto below = [&](int row) { return row < n && !top[row]; };
  std::vector<std::vector<uint16_t>> codes(n), erec(nw), vrec(nw);
  std::vector<uint16_t> tel;
  int nh = 0;  // histories
  if (adjoint) {
    const uint16_t* ar = lw + lh.o_adj;
    for (int k = 0; k < lh.nadj; k++) {
      const uint16_t* r = ar + k * LIN_ADJ;
      const int kind = r[0] >> 14, e = r[0] & 0x3FFF, p = col_or(r[1]), m = col_or(r[2]), c = col_or(r[5]);
      const int ra = kind == 2 ? col_or(r[6]) : col_or(r[3]), rb = kind == 2 ? n : col_or(r[4]);
      const int xp = kind == 2 ? c : p, xm = kind == 2 ? n : m;
      // an instance in every wave whose rows read its histories, else in one that sees its adjoints
      std::vector<int> in;
      auto add = [&](int row) {
        if (below(row) && std::find(in.begin(), in.end(), wave[row]) == in.end()) in.push_back(wave[row]);
      };
      if (kind) add(p), add(m);
      if (kind == 2) add(c);
      if (in.empty()) add(ra), add(rb);
      if (in.empty()) in.push_back(0);
      if (!kind && in.size() > 1) return false;
      for (size_t q = 0; q < in.size(); q++) {
        const int w = in[q];
        for (int row : {ra, rb})
          if (below(row) && wave[row] != w) return false;
        int h[2] = {-1, -1};
        auto code = [&](int row, int x, int neg) {
          if (row < n && (top[row] ? q == 0 : wave[row] == w)) codes[row].push_back(u16((x << 1) | neg));
        };
        if (kind) h[0] = nh++, code(p, h[0], 0), code(m, h[0], 1);
        if (kind == 2) h[1] = nh++, code(c, h[1], 0);
        if (nh >= 0x3FFF) return false;
        erec[w].insert(erec[w].end(), {u16(kind), u16(e), u16(ra), u16(rb), u16(xp < n ? col_of[xp] : n),
                                       u16(xm < n ? col_of[xm] : n), u16(h[0]), u16(h[1]), u16(q == 0)});
      }
    }
    for (auto& v : erec)  // the unread history follows the zero
      for (size_t q = 0; q < v.size(); q += WS_AELEM)
        for (int k : {WSA_H1, WSA_H2})
          if (v[q + k] == 0xFFFF) v[q + k] = u16(nh + 1);
  } else {
    const uint16_t *rcp = lw + lh.o_rcon_ptr, *rc = lw + lh.o_rcon, *dyn = lw + lh.o_dyn;
    nh = lh.ndyn + lh.nsrc;
    if (nh >= 0x3FFF) return false;
    // each history's wave (-1: only top rows touch it; -2: several waves' unknowns, which only a top row may then
    // read: the element is wave 0's to update beside the top rows)
    std::vector<int> owner(nh, -1);
    std::vector<char> read(nh, 0);
    auto claim = [&](int h, int row) {
      if (below(row)) owner[h] = owner[h] == -1 || owner[h] == wave[row] ? wave[row] : -2;
    };
    for (int i = 0; i < n; i++)
      for (int q = rcp[i]; q < rcp[i + 1]; q++) {
        const int idx = rc[q] >> 2, k = rc[q] & 3;
        const int h = k == LK_SRC ? lh.ndyn + idx : idx;
        codes[i].push_back(u16((h << 1) | (k == LK_CP ? 1 : 0)));
        claim(h, i);
        if (!top[i]) read[h] = 1;
      }
    for (int d = 0; d < lh.ndyn; d++) {
      const uint16_t* r = dyn + d * LIN_DYN;
      const int kind = r[0] >> 14, e = r[0] & 0x3FFF, p = col_or(r[1]), m = col_or(r[2]);
      const int c = kind == 2 ? col_or(r[3]) : n;
      claim(d, p), claim(d, m), claim(d, c);
      if (owner[d] == -2 && read[d]) return false;
      auto& v = owner[d] == -2 ? tel : erec[std::max(owner[d], 0)];
      v.insert(v.end(), {u16(d), u16(kind), u16(p), u16(m), u16(c), u16(e)});
    }
    if (tel.size() > 64 * WS_ELEM) return false;
    for (int k = 0; k < lh.nsrc; k++) {
      const int h = lh.ndyn + k, w = owner[h];
      if (w == -2) return false;
      vrec[std::max(w, 0)].insert(vrec[std::max(w, 0)].end(), {u16(h), u16(k)});
    }
  }

  // slots
  struct Slot {
    int row, lev, part = 0, npart = 0;  // row: index into the solution buffer
    std::vector<std::pair<int, int>> ent;
  };
  std::vector<std::vector<Slot>> slots(nw);
  std::vector<Slot> tops;
  int npart = 0;
  for (int i = 0; i < n; i++) {
    Slot s{i, lev[i]};
    if (!top[i]) {
      s.ent = lo[i];
      slots[wave[i]].push_back(s);
      continue;
    }
    std::vector<Slot> ps(nw, Slot{n, 0});
    for (auto& e : lo[i])
      if (top[e.first]) {
        s.ent.push_back(e);
      } else {
        Slot& q = ps[wave[e.first]];
        q.ent.push_back(e);
        q.lev = std::max(q.lev, lev[e.first] + 1);
      }
    s.part = npart;
    for (int w = 0; w < nw; w++)
      if (!ps[w].ent.empty()) {
        ps[w].row = n + 1 + npart++;
        s.npart++;
        slots[w].push_back(ps[w]);
      }
    tops.push_back(s);
  }
  WsHdr h{};
  const int esz = adjoint ? WS_AELEM : WS_ELEM;
  int rows = 1, elems = 1, top_nl = 0;
  for (int w = 0; w < nw; w++) {
    rows = std::max(rows, ((int)slots[w].size() + 63) / 64);
    elems = std::max(elems, ((int)erec[w].size() / esz + 63) / 64);
    if (vrec[w].size() > 64 * WS_SRC) return false;
  }
  if (rows > WS_R_MAX || elems > (adjoint ? WS_AE_MAX : WS_R_MAX)) return false;
  if (n > ws_cols_max(nw, rows == 3 ? 4 : rows)) return false;  // (the kernels' rows per lane are 1, 2 or 4)
  bool fits = true;
  std::vector<uint16_t> wrec, srec, trec, pairs, rhs, evec, vvec;
  auto emit = [&](const Slot& s, int keep, std::vector<uint16_t>& rec) {
    uint16_t r[WS_SLOT];
    r[WSR_ROW] = u16(s.row);
    r[WSR_LEV] = u16(s.lev);
    if (s.lev > keep) fits = false;
    r[WSR_PAIR] = u16((int)pairs.size() / 4);
    std::vector<int> have(s.lev, 0);
    const size_t p0 = pairs.size();
    for (int l = 0; l < s.lev; l++) pairs.insert(pairs.end(), {u16(n), u16(nnz), u16(n), u16(nnz)});
    for (auto& e : s.ent) {
      const int l = lev[e.first], k = have[l]++;
      if (k > 1) {
        fits = false;
        break;
      }
      pairs[p0 + 4 * l + 2 * k] = u16(e.first);
      pairs[p0 + 4 * l + 2 * k + 1] = u16(e.second);
    }
    const bool real = s.row < n;
    r[WSR_UC0] = r[WSR_UC1] = u16(n);
    r[WSR_US0] = r[WSR_US1] = u16(nnz);
    r[WSR_DIAG] = real ? u16(dg[s.row]) : u16(nnz);
    r[WSR_RHS] = u16((int)rhs.size());
    r[WSR_NRHS] = 0;
    r[WSR_COL] = real ? u16(b[L.o_col_of + s.row]) : u16(0);
    if (real) {
      const auto& u = up[s.row];
      if (u.size() > 2) fits = false;
      for (int k = 0; k < std::min<int>(2, (int)u.size()); k++) {
        r[WSR_UC0 + k] = u16(u[k].first);
        r[WSR_US0 + k] = u16(u[k].second);
      }
      rhs.insert(rhs.end(), codes[s.row].begin(), codes[s.row].end());
      r[WSR_NRHS] = u16((int)codes[s.row].size());
      if (codes[s.row].size() > 2) h.more = 1;
    }
    r[WSR_PART] = u16(s.part);
    r[WSR_NPART] = u16(s.npart);
    rec.insert(rec.end(), r, r + WS_SLOT);
  };
  int ns = 0;
  for (int w = 0; w < nw; w++) {
    std::stable_sort(slots[w].begin(), slots[w].end(), [](const Slot& x, const Slot& y) { return x.lev > y.lev; });
    for (size_t q = 0; q < slots[w].size(); q++) emit(slots[w][q], ws_pairs((int)q / 64), srec);
    const int s0 = ns, e0 = (int)evec.size() / esz, v0 = (int)vvec.size() / WS_SRC;
    const int nl = slots[w].empty() ? 0 : slots[w][0].lev;
    ns += (int)slots[w].size();
    evec.insert(evec.end(), erec[w].begin(), erec[w].end());
    vvec.insert(vvec.end(), vrec[w].begin(), vrec[w].end());
    wrec.insert(wrec.end(), {u16(s0), u16(ns), u16(e0), u16((int)evec.size() / esz), u16(v0),
                             u16((int)vvec.size() / WS_SRC), u16(nl)});
  }
  evec.insert(evec.end(), tel.begin(), tel.end());  // after the waves' elements
  for (auto& s : tops) {
    emit(s, WS_TOP_PAIRS, trec);
    top_nl = std::max(top_nl, s.lev);
  }
  if (!fits || n + npart + 3 >= 0xFFFF || pairs.size() / 4 >= 0xFFFF || rhs.size() >= 0xFFFF || ns >= 0xFFFF ||
      evec.size() / esz >= 0xFFFF)
    return false;
  h.adjoint = adjoint ? 1 : 0;
  h.n = n, h.nnz = nnz, h.ndyn = adjoint ? nh : lh.ndyn, h.nsrc = adjoint ? 0 : lh.nsrc;
  h.nw = nw, h.rows = rows, h.elems = elems;
  h.ntop = ntop, h.npart = npart;
  h.nrhs = (int)rhs.size(), h.top_nl = top_nl;
  h.ntel = (int)tel.size() / WS_ELEM;
  std::vector<uint16_t> o(sizeof(WsHdr) / 2, 0);
  auto put = [&](const std::vector<uint16_t>& v) {
    while (o.size() % 4) o.push_back(0);
    const int at = (int)o.size();
    o.insert(o.end(), v.begin(), v.end());
    return at;
  };
  h.o_wave = put(wrec), h.o_slot = put(srec), h.o_top = put(trec), h.o_elem = put(evec), h.o_src = put(vvec);
  h.o_pair = put(pairs);
  h.o_rhs = put(rhs);
  std::vector<uint16_t> cpos(lw + lh.o_cpos, lw + lh.o_cpos + n);
  for (auto& c : cpos)
    if (top[c]) c = u16(n);
  h.o_cpos = put(cpos);
  while (o.size() % 8) o.push_back(0);
  h.words = (int)o.size();
  std::memcpy(o.data(), &h, sizeof h);
  out.swap(o);
  return true;
}

}  // namespace kg
