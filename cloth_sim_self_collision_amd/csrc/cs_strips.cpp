// Strip plan of the triangular sweeps (see cs_strips.hpp).
#include "cs_strips.hpp"

#include <algorithm>
#include <climits>

namespace cs {

namespace {

// smallest strip that a component boundary may end: the strips of a mesh of
// many small components would otherwise each hold a few rows
constexpr int kCompRows = 256;

std::vector<int> level_of_row(const std::vector<int>& ptr, const std::vector<int>& rows, int np) {
  std::vector<int> l(np, 0);
  for (int k = 0; k + 1 < (int)ptr.size(); k++)
    for (int q = ptr[k]; q < ptr[k + 1]; q++) l[rows[q]] = k;
  return l;
}

// rows in sweep order: ascending for the forward sweep, descending for the
// backward one; a row's dependencies come before it
struct Order {
  const MeshSetup& s;
  bool fwd;
  int np;
  int at(int q) const { return fwd ? q : np - 1 - q; }
  int first(int i) const { return fwd ? s.rowptr[i] : s.diaind[i]; }
  int last(int i) const { return fwd ? s.diaind[i] : s.rowptr[i + 1]; }
};

// Strips: rows are taken in sweep order until one more would give some level
// kStripRows + 1 rows of the strip.  In a grid numbered along its columns that
// cuts it into bands of eight columns, whose sub-levels are the levels.
bool cut(const Order& o, const std::vector<int>& lvl, int nlev, StripSweep& w,
         std::vector<int>& sub_of) {
  const int np = o.np;
  std::vector<int> count(nlev, 0), seen(nlev, -1);
  std::vector<int> begin{0};  // first position (in sweep order) of each strip
  int strip = 0;
  for (int q = 0; q < np; q++) {
    const int i = o.at(q), l = lvl[i];
    const bool new_comp = q > 0 && o.s.comp[i] != o.s.comp[o.at(q - 1)];
    const int have = seen[l] == strip ? count[l] : 0;
    if (have == kStripRows || (new_comp && q - begin.back() >= kCompRows)) {
      begin.push_back(q);
      strip++;
    }
    if (seen[l] != strip) {
      seen[l] = strip;
      count[l] = 0;
    }
    count[l]++;
  }
  begin.push_back(np);
  const int ns = strip + 1;
  w.ptr.assign(1, 0);
  sub_of.assign(np, 0);
  w.slot.assign(np, 0);
  std::vector<int> order;
  long long nsub = 0;
  std::vector<std::vector<int>> rows_of(ns);
  for (int t = 0; t < ns; t++) {
    order.clear();
    for (int q = begin[t]; q < begin[t + 1]; q++) order.push_back(o.at(q));
    std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return lvl[a] < lvl[b]; });
    int sub = (int)nsub - 1, last = -1, in = 0;
    for (int i : order) {
      if (lvl[i] != last) {
        sub++;
        in = 0;
        last = lvl[i];
      }
      sub_of[i] = sub;
      w.slot[i] = sub * kStripRows + in++;
    }
    nsub = (sub + 1 + kStripGroup - 1) / kStripGroup * kStripGroup;
    if (nsub > INT_MAX / (4 * kStripRows) - kStripTail) return false;
    w.ptr.push_back((int)nsub);
  }
  w.nsub = (int)nsub;
  w.row.assign((size_t)(w.nsub + kStripTail) * kStripRows, -1);
  for (int i = 0; i < np; i++) w.row[w.slot[i]] = i;
  return true;
}

// Imports and ring offsets for a ring of `ring` sub-levels; false when a
// dependency is further back than the ring or a sub-level has no import slot
// in reach.
bool place(const Order& o, const std::vector<int>& sub_of, int k, int ring, StripSweep& w) {
  const size_t slots = w.row.size();
  w.col.assign(slots * k, 0);  // offset 0 is the zero entry
  w.import.assign(slots / kStripRows * kStripImports, -1);
  std::vector<int> used(slots / kStripRows, 0);
  std::vector<int> at(o.np, -1);  // import slot of a row in the current strip
  std::vector<int> mine;          // rows whose `at` is set
  const int mask = ring - 1;
  auto own_offset = [&](int slot) {
    return (unsigned short)(kStripZero + (slot / kStripRows & mask) * kStripSub +
                            slot % kStripRows * kStripEntry);
  };
  auto import_offset = [&](int at) {
    const int q = at % kStripImports;
    return (unsigned short)(kStripZero + (at / kStripImports & mask) * kStripSub +
                            (1 + q % 2 * 2) * kStripRows * kStripEntry + q / 2 * kStripEntry);
  };
  for (int t = 0; t + 1 < (int)w.ptr.size(); t++) {
    for (int i : mine) at[i] = -1;
    mine.clear();
    for (int sub = w.ptr[t]; sub < w.ptr[t + 1]; sub++)
      for (int q = 0; q < kStripRows; q++) {
        const int slot = sub * kStripRows + q, i = w.row[slot];
        if (i < 0) continue;
        const int b = o.first(i), e = o.last(i);
        for (int m = b; m < e; m++) {
          const int j = o.s.colind[m];
          const int js = sub_of[j];
          if (js >= w.ptr[t] && js < w.ptr[t + 1]) {  // swept by this strip
            if (js >= sub || sub - js >= ring) return false;
            w.col[(size_t)slot * k + (m - b)] = own_offset(w.slot[j]);
            continue;
          }
          if (at[j] < 0 || sub - at[j] / kStripImports >= ring) {
            // the latest free import slot not after this sub-level
            int u = sub;
            while (u >= w.ptr[t] && sub - u < ring && used[u] == kStripImports) u--;
            if (u < w.ptr[t] || sub - u >= ring) return false;
            if (at[j] < 0) mine.push_back(j);
            at[j] = u * kStripImports + used[u]++;
            w.import[at[j]] = j;
          }
          w.col[(size_t)slot * k + (m - b)] = import_offset(at[j]);
        }
      }
  }
  return true;
}

std::string check(const Order& o, const StripPlan& p, const StripSweep& w) {
  if (p.ring < 1 || p.ring > kStripMaxRing || (p.ring & (p.ring - 1))) return "ring size";
  const size_t slots = (size_t)(w.nsub + kStripTail) * kStripRows;
  if (w.row.size() != slots || w.import.size() != slots / kStripRows * kStripImports || w.col.size() != slots * p.k ||
      (int)w.slot.size() != o.np || w.ptr.empty() || w.ptr[0] != 0 || w.ptr.back() != w.nsub)
    return "array sizes";
  const int entries = (kStripZero + p.ring * kStripSub) / kStripEntry;
  std::vector<int> holds(entries, -1);
  std::vector<char> done(o.np, 0);
  for (int t = 0; t + 1 < (int)w.ptr.size(); t++) {
    if (w.ptr[t + 1] < w.ptr[t] || w.ptr[t] % kStripGroup) return "strip bounds";
    std::fill(holds.begin(), holds.end(), -1);
    std::vector<int> swept;
    for (int sub = w.ptr[t]; sub < w.ptr[t + 1]; sub++) {
      const int base = (kStripZero + (sub & (p.ring - 1)) * kStripSub) / kStripEntry;
      for (int q = 0; q < kStripImports; q++) {
        const int j = w.import[(size_t)sub * kStripImports + q];
        if (j < -1 || j >= o.np) return "import out of range";
        if (j >= 0 && !done[j]) return "a row imported from a strip that is not swept before";
        if (j >= 0) holds[base + (1 + q % 2 * 2) * kStripRows + q / 2] = j;
      }
      for (int q = 0; q < kStripRows; q++) {
        const size_t slot = (size_t)sub * kStripRows + q;
        const int i = w.row[slot];
        if (i < -1 || i >= o.np) return "row out of range";
        if (i >= 0 && w.slot[i] != (int)slot) return "slot of a row";
        const int n = i < 0 ? 0 : o.last(i) - o.first(i);
        if (n > p.k) return "row too wide";
        for (int m = 0; m < p.k; m++) {
          const int off = w.col[slot * p.k + m];
          if (off % kStripEntry || off / kStripEntry >= entries) return "ring offset";
          if (m >= n ? off != 0 : holds[off / kStripEntry] != o.s.colind[o.first(i) + m])
            return "a block reads another row's entry";
        }
      }
      for (int q = 0; q < kStripRows; q++) {
        holds[base + q] = w.row[(size_t)sub * kStripRows + q];
        if (holds[base + q] >= 0) swept.push_back(holds[base + q]);
      }
    }
    for (int i : swept) done[i] = 1;
  }
  for (int i = 0; i < o.np; i++)
    if (!done[i]) return "a row is not swept";
  for (size_t q = (size_t)w.nsub * kStripRows; q < slots; q++)
    if (w.row[q] != -1) return "the tail is not empty";
  for (size_t q = (size_t)w.nsub * kStripImports; q < w.import.size(); q++)
    if (w.import[q] != -1) return "the tail is not empty";
  return "";
}

}  // namespace

void build_strips(const MeshSetup& s, StripPlan& p) {
  p = StripPlan();
  const int k = std::max(s.kl, s.ku);
  if (s.kl <= 0 || k > kMaxBlocksPerRow) return;
  p.k = k;
  const Order f{s, true, s.np}, b{s, false, s.np};
  std::vector<int> fsub, bsub;
  if (!cut(f, level_of_row(s.lf_ptr, s.lf_rows, s.np), s.nlf, p.fwd, fsub) ||
      !cut(b, level_of_row(s.lb_ptr, s.lb_rows, s.np), s.nlb, p.bwd, bsub))
    return;
  for (p.ring = 8; p.ring <= kStripMaxRing; p.ring *= 2)
    if (place(f, fsub, k, p.ring, p.fwd) && place(b, bsub, k, p.ring, p.bwd)) {
      p.ok = true;
      return;
    }
  p.ring = 0;
}

std::string validate_strips(const MeshSetup& s, const StripPlan& p) {
  std::string e = check(Order{s, true, s.np}, p, p.fwd);
  if (!e.empty()) return "forward strips: " + e;
  e = check(Order{s, false, s.np}, p, p.bwd);
  return e.empty() ? e : "backward strips: " + e;
}

}  // namespace cs
