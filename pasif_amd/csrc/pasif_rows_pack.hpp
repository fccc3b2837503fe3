// Host side of the row kernel's layout (pasif_rows.hpp): the units of one
// side of one system and their wave-blocked program.
#pragma once

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <limits>
#include <vector>

#include "pasif_host.hpp"
#include "pasif_rows.hpp"
#include "pasif_tiles.hpp"

namespace pasif {

// Terms [t0, t1) of a row (numbered through its kinds in order).
struct RowUnit {
  uint32_t row = 0, t0 = 0, t1 = 0;
  uint32_t cnt[4] = {0, 0, 0, 0};
  bool owns = true;       // outputs the row's value itself
  bool first = true;      // carries the row's initial value and force
  uint32_t p0 = 0, p1 = 0;  // split row: its aux units
};

// The units of one side in the kernel's order, and the slot of every
// published row (kRowNone: a sink).
struct RowUnits {
  std::vector<RowUnit> main, aux;
  uint32_t pub = 0, pieces = 0;            // published units; pieces of multi-unit sinks
  std::vector<uint32_t> sink;              // {row, first piece, end} of each multi-unit sink
  std::vector<uint32_t> slot;              // [rows of the system]
};

// published rows of system s: those a term of its own side reads as a state
// factor and, for the forward side of an adjoint run, those an adjoint term
// reads as a set point
inline std::vector<uint8_t> row_published(const RowTerms& rt, uint32_t s, bool adjoint_side,
                                          const RowTerms* adj) {
  const uint32_t off = rt.off[s], n = rt.size[s];
  std::vector<uint8_t> pub(n, 0);
  for (int k = 0; k < 4; ++k) {
    const int nf = k + 1;
    const int own = adjoint_side ? 1 : nf;
    for (uint32_t e = rt.ptr[k][off]; e < rt.ptr[k][off + n]; ++e)
      for (int a = 0; a < own; ++a) pub[rt.idx[k][size_t(e) * nf + a] - off] = 1;
  }
  if (adj) {
    const uint32_t ao = adj->off[s], an = adj->size[s];
    for (int k = 1; k < 4; ++k) {
      const int nf = k + 1;
      for (uint32_t e = adj->ptr[k][ao]; e < adj->ptr[k][ao + an]; ++e)
        for (int a = 1; a < nf; ++a) pub[adj->idx[k][size_t(e) * nf + a] - off] = 1;
    }
  }
  return pub;
}

inline void row_unit_counts(const RowTerms& rt, uint32_t g, RowUnit& u) {
  uint32_t t = 0;
  for (int k = 0; k < 4; ++k) {
    const uint32_t c = rt.ptr[k][g + 1] - rt.ptr[k][g];
    const uint32_t b = std::max(t, u.t0), e = std::min(t + c, u.t1);
    u.cnt[k] = e > b ? e - b : 0;
    t += c;
  }
}

inline RowUnits row_units(const RowTerms& rt, uint32_t s, const std::vector<uint8_t>& pub) {
  const uint32_t off = rt.off[s], n = rt.size[s];
  RowUnits o;
  std::vector<RowUnit> sinks, pieces;
  for (uint32_t r = 0; r < n; ++r) {
    uint32_t nt = 0;
    for (int k = 0; k < 4; ++k) nt += rt.ptr[k][off + r + 1] - rt.ptr[k][off + r];
    RowUnit u;
    u.row = r;
    if (pub[r]) {
      if (nt <= kRowSplitTerms) {
        u.t1 = nt;
      } else {
        u.p0 = uint32_t(o.aux.size());
        for (uint32_t t = 0; t < nt; t += kRowPieceTerms) {
          RowUnit a;
          a.row = r;
          a.t0 = t;
          a.t1 = std::min(nt, t + kRowPieceTerms);
          row_unit_counts(rt, off + r, a);
          o.aux.push_back(a);
        }
        u.p1 = uint32_t(o.aux.size());
      }
      row_unit_counts(rt, off + r, u);
      o.main.push_back(u);
    } else if (nt <= kRowPieceTerms) {
      u.t1 = nt;
      row_unit_counts(rt, off + r, u);
      sinks.push_back(u);
    } else {
      const uint32_t p0 = uint32_t(pieces.size());
      for (uint32_t t = 0; t < nt; t += kRowPieceTerms) {
        RowUnit a;
        a.row = r;
        a.t0 = t;
        a.t1 = std::min(nt, t + kRowPieceTerms);
        a.owns = false;
        a.first = t == 0;
        row_unit_counts(rt, off + r, a);
        pieces.push_back(a);
      }
      o.sink.insert(o.sink.end(), {r, p0, uint32_t(pieces.size())});
    }
  }
  // units of equal trip counts next to each other: a wave runs to the
  // largest of its 64
  auto longer = [](const RowUnit& a, const RowUnit& b) {
    for (int k = 3; k >= 0; --k)
      if (a.cnt[k] != b.cnt[k]) return a.cnt[k] > b.cnt[k];
    return false;
  };
  std::stable_sort(o.main.begin(), o.main.end(), longer);
  std::stable_sort(sinks.begin(), sinks.end(), longer);
  o.pub = uint32_t(o.main.size());
  o.pieces = uint32_t(pieces.size());
  o.slot.assign(n, kRowNone);
  for (uint32_t u = 0; u < o.pub; ++u) o.slot[o.main[u].row] = u;
  o.main.insert(o.main.end(), pieces.begin(), pieces.end());
  o.main.insert(o.main.end(), sinks.begin(), sinks.end());
  return o;
}

// LDS values of an instance's buffers (RowInst): a slot more than published
// rows holds the 0 that padding terms read.
struct RowLds {
  uint32_t ys, xs, ps;
  size_t values() const { return row_lds_values(ys, xs, ps); }
};
inline RowLds row_lds(const RowUnits& f, const RowUnits* a) {
  RowLds l;
  l.ys = std::max(f.pub, a ? a->pub : 0u) + 1u;
  l.xs = a ? f.pub + 1u : 0u;
  size_t part = std::max<size_t>(f.aux.size(), f.pieces);
  if (a) part = std::max<size_t>(part, std::max<size_t>(a->aux.size(), a->pieces));
  l.ps = uint32_t(part);
  return l;
}

// Whether the kernel can hold an instance with these units: threads and
// slots, 16-bit LDS offsets and piece ranges, LDS size.
inline bool row_units_fit(const RowUnits& f, const RowUnits* a, size_t el) {
  const size_t most = size_t(kRowThreads) * kRowSlots;
  if (f.main.size() > most || (a && a->main.size() > most)) return false;
  if (f.aux.size() > 0xFFFF || (a && a->aux.size() > 0xFFFF)) return false;
  const RowLds l = row_lds(f, a);
  return size_t(l.ys) * el <= 0xFFFF && size_t(l.xs) * el <= 0xFFFF &&
         l.values() * el <= kMaxLdsBytes;
}

// Packed program arrays of many sides.
template <typename R>
struct RowPacked {
  std::vector<uint32_t> blk;  // [blocks][4]
  std::vector<R> val, init, force;
  std::vector<uint32_t> word, row, piece, sink;
};

// Append one side: `zero` is the slot holding 0 for state factors, `xslot`
// the slots of set-point factors (the side's own for a forward side) and
// `xzero` their zero slot.
template <typename R>
RowProg row_emit(RowPacked<R>& o, const RowTerms& rt, uint32_t s, const RowUnits& un, bool adjoint,
                 const std::vector<uint32_t>& xslot, uint32_t xoff, uint32_t zero,
                 uint32_t xzero) {
  const double eps = std::numeric_limits<R>::epsilon();
  const uint32_t off = rt.off[s];
  constexpr uint32_t EL = sizeof(R);
  RowProg p{};
  p.val = o.val.size();
  p.word = o.word.size();
  p.blk = o.blk.size() / 4;
  p.unit = o.init.size();
  p.sink = o.sink.size();
  p.units = uint32_t(un.main.size());
  p.pub = un.pub;
  p.aux = uint32_t(un.aux.size());
  p.nsink = uint32_t(un.sink.size() / 3);
  o.sink.insert(o.sink.end(), un.sink.begin(), un.sink.end());
  const uint32_t zs = zero * EL, zx = xzero * EL;
  auto blocks = [&](const std::vector<RowUnit>& units, bool main) {
    for (size_t b = 0; b < units.size(); b += 64) {
      const size_t e = std::min(units.size(), b + 64);
      uint32_t c[4] = {0, 0, 0, 0}, flags = 0;
      for (size_t u = b; u < e; ++u) {
        for (int k = 0; k < 4; ++k) c[k] = std::max(c[k], units[u].cnt[k]);
        if (main && units[u].p1 > units[u].p0) flags |= 1u << 29;
        if (main && !adjoint && units[u].first && std::fabs(rt.force[off + units[u].row]) > eps)
          flags |= 1u << 28;
      }
      c[0] = (c[0] + 1u) & ~1u;
      c[1] = (c[1] + 1u) & ~1u;
      const size_t v0 = o.val.size(), w0 = o.word.size();
      const uint32_t nv = c[0] + c[1] + c[2] + c[3];
      const uint32_t nw = c[0] / 2 + c[1] + 2 * c[2] + 2 * c[3];
      o.blk.insert(o.blk.end(), {uint32_t((v0 - p.val) / 64), uint32_t((w0 - p.word) / 64),
                                 c[0] | (c[1] << 7) | (c[2] << 14) | (c[3] << 21) | flags, 0u});
      o.val.resize(v0 + size_t(nv) * 64, R(0));
      o.word.resize(w0 + size_t(nw) * 64, 0u);
      for (uint32_t ln = 0; ln < 64; ++ln) {
        const RowUnit* u = b + ln < e ? &units[b + ln] : nullptr;
        size_t v = v0 + ln, w = w0 + ln;
        uint32_t first = 0;  // of this kind, within the row
        for (int k = 0; k < 4; ++k) {
          const int nf = k + 1;
          uint32_t cn = 0, e0 = 0;
          if (u) {
            const uint32_t g = off + u->row;
            const uint32_t lo = std::max(first, u->t0);
            cn = u->cnt[k];
            e0 = rt.ptr[k][g] + (lo - first);
            first += rt.ptr[k][g + 1] - rt.ptr[k][g];
          }
          for (uint32_t i = 0; i < c[k]; ++i) {
            uint32_t f[4] = {zs, zx, zx, zx};
            if (i < cn) {
              const uint32_t* ix = &rt.idx[k][size_t(e0 + i) * nf];
              o.val[v] = R(rt.val[k][e0 + i]);
              f[0] = un.slot[ix[0] - off] * EL;
              for (int a = 1; a < nf; ++a) f[a] = xslot[ix[a] - xoff] * EL;
            }
            v += 64;
            if (k == 0) {
              o.word[w] |= f[0] << (16 * (i & 1u));
              if (i & 1u) w += 64;
            } else {
              o.word[w] = f[0] | (f[1] << 16);
              w += 64;
              if (k >= 2) {
                o.word[w] = f[2] | ((k == 3 ? f[3] : zx) << 16);
                w += 64;
              }
            }
          }
        }
        if (main) {
          const bool live = u != nullptr;
          o.init.push_back(live && u->first ? R(rt.init[off + u->row]) : R(0));
          const double fr = live && !adjoint && u->first ? rt.force[off + u->row] : 0.0;
          o.force.push_back(std::fabs(fr) > eps ? R(fr) : R(0));
          o.row.push_back(live && u->owns ? u->row : kRowNone);
          o.piece.push_back(live ? (u->p0 | (u->p1 << 16)) : 0u);
        }
      }
    }
  };
  blocks(un.main, true);
  blocks(un.aux, false);
  return p;
}

}  // namespace pasif
