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
// (more than two couplings to one level, too many top rows, rows per wave or
// levels, an element shared by two waves, or indices beyond 16 bits).
bool build_ws_plan(const PatLayout& L, const std::vector<int32_t>& b, const std::vector<uint16_t>& lin, int nw,
                   std::vector<uint16_t>& out) {
  out.clear();
  if (L.status != KG_OK || lin.empty() || (nw != 1 && nw != 2 && nw != 4 && nw != 8)) return false;
  LinHdr lh;
  std::memcpy(&lh, lin.data(), sizeof lh);
  const int n = L.n, nnz = L.nnz;
  const int32_t* rp = b.data() + L.o_row_ptr;
  const int32_t* col = b.data() + L.o_col;
  const int32_t* dg = b.data() + L.o_diag;
  Lists lo(n), up(n);
  for (int i = 0; i < n; i++)
    for (int p = rp[i]; p < rp[i + 1]; p++)
      if (col[p] != i) (col[p] < i ? lo[i] : up[i]).push_back({col[p], p});
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

  // right-hand side codes per row, and each history's wave (-1: only top rows touch it)
  const uint16_t* lw = lin.data();
  const uint16_t *rcp = lw + lh.o_rcon_ptr, *rc = lw + lh.o_rcon, *dyn = lw + lh.o_dyn;
  const int nh = lh.ndyn + lh.nsrc;
  if (n >= 0x7FFF || nnz >= 0xFFFF || nh >= 0x3FFF) return false;
  // (-2: several, which only a top row may then read: the element is wave 0's to update beside the top rows)
  std::vector<int> owner(nh, -1);
  std::vector<char> below(nh, 0);
  auto claim = [&](int h, int row) {  // row: a row or column index of the permuted system
    if (row < n && !top[row]) owner[h] = owner[h] == -1 || owner[h] == wave[row] ? wave[row] : -2;
  };
  std::vector<std::vector<uint16_t>> codes(n);
  for (int i = 0; i < n; i++)
    for (int q = rcp[i]; q < rcp[i + 1]; q++) {
      const int idx = rc[q] >> 2, k = rc[q] & 3;
      const int h = k == LK_SRC ? lh.ndyn + idx : idx;
      codes[i].push_back(u16((h << 1) | (k == LK_CP ? 1 : 0)));
      claim(h, i);
      if (!top[i]) below[h] = 1;
    }
  struct El { int hist, kind, p, m, c, e; };
  std::vector<El> els;
  auto col_or = [&](uint16_t v) { return v == LIN_NONE ? n : (int)v; };
  for (int d = 0; d < lh.ndyn; d++) {
    const uint16_t* r = dyn + d * LIN_DYN;
    const El e{d, r[0] >> 14, col_or(r[1]), col_or(r[2]), (r[0] >> 14) == 2 ? col_or(r[3]) : n, r[0] & 0x3FFF};
    claim(d, e.p), claim(d, e.m), claim(d, e.c);
    els.push_back(e);
  }
  for (int k = 0; k < nh; k++)
    if (owner[k] == -2 && (below[k] || k >= lh.ndyn)) return false;

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
  std::vector<std::vector<El>> wel(nw);
  std::vector<El> tel;
  for (auto& e : els) (owner[e.hist] == -2 ? tel : wel[std::max(owner[e.hist], 0)]).push_back(e);
  if (tel.size() > 64) return false;
  std::vector<std::vector<int>> wsrc(nw);
  for (int k = 0; k < lh.nsrc; k++) wsrc[std::max(owner[lh.ndyn + k], 0)].push_back(k);
  int rows = 1, elems = 1, top_nl = 0;
  for (int w = 0; w < nw; w++) {
    rows = std::max(rows, ((int)slots[w].size() + 63) / 64);
    elems = std::max(elems, ((int)wel[w].size() + 63) / 64);
    if (wsrc[w].size() > 64) return false;
  }
  if (rows > WS_R_MAX || elems > WS_R_MAX) return false;
  bool fits = true;
  std::vector<uint16_t> wrec, srec, trec, erec, vrec, pairs, rhs;
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
  auto element = [&](const El& e) {
    erec.insert(erec.end(), {u16(e.hist), u16(e.kind), u16(e.p), u16(e.m), u16(e.c), u16(e.e)});
  };
  int ns = 0, ne = 0, nv = 0;
  for (int w = 0; w < nw; w++) {
    std::stable_sort(slots[w].begin(), slots[w].end(), [](const Slot& x, const Slot& y) { return x.lev > y.lev; });
    for (size_t q = 0; q < slots[w].size(); q++) emit(slots[w][q], ws_pairs((int)q / 64), srec);
    for (auto& e : wel[w]) element(e);
    for (int k : wsrc[w]) vrec.insert(vrec.end(), {u16(lh.ndyn + k), u16(k)});
    const int s0 = ns, e0 = ne, v0 = nv, nl = slots[w].empty() ? 0 : slots[w][0].lev;
    ns += (int)slots[w].size();
    ne += (int)wel[w].size();
    nv += (int)wsrc[w].size();
    wrec.insert(wrec.end(), {u16(s0), u16(ns), u16(e0), u16(ne), u16(v0), u16(nv), u16(nl)});
  }
  for (auto& e : tel) element(e);  // after the waves' elements
  for (auto& s : tops) {
    emit(s, WS_TOP_PAIRS, trec);
    top_nl = std::max(top_nl, s.lev);
  }
  if (!fits || n + npart + 3 >= 0xFFFF || pairs.size() / 4 >= 0xFFFF || rhs.size() >= 0xFFFF ||
      ns >= 0xFFFF)
    return false;
  h.n = n, h.nnz = nnz, h.ndyn = lh.ndyn, h.nsrc = lh.nsrc, h.nw = nw, h.rows = rows, h.elems = elems;
  h.ntop = ntop, h.npart = npart;
  h.nrhs = (int)rhs.size(), h.top_nl = top_nl;
  h.ntel = (int)tel.size();
  std::vector<uint16_t> o(sizeof(WsHdr) / 2, 0);
  auto put = [&](const std::vector<uint16_t>& v) {
    while (o.size() % 4) o.push_back(0);
    const int at = (int)o.size();
    o.insert(o.end(), v.begin(), v.end());
    return at;
  };
  h.o_wave = put(wrec), h.o_slot = put(srec), h.o_top = put(trec), h.o_elem = put(erec), h.o_src = put(vrec);
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
