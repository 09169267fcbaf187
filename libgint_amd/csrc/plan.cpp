// Plans of the recurrences.
//
// ClassPlan: the (e0|f0) blocks of one class (la lb|lc ld) and the FLOPs of
// the reference chain for it: VRR, horizontal recurrence (HRR1 moves d onto
// c, HRR2 b onto a, as in reference src/plan.cpp:56-146, rec_add) and
// cartesian -> spherical transform.
//
// TypePlan: the union of the (e0|f0) blocks that the classes of one quartet
// type read, the Hermite sizes of the McMurchie-Davidson path that produces
// them, and the per-class bookkeeping (gates, contraction layout, checksum
// multipliers).
#include <algorithm>
#include <array>
#include <cstring>
#include <map>
#include <set>
#include <tuple>
#include <vector>

#include "device.hpp"

namespace gint {

// VRR FLOPs of the reference plan for one class: the recursion of reference
// src/plan.cpp:56-146 from the (e0|f0) targets at m = 0, with the m-ranges
// of each (a,c) block collapsed to [min m, max m] (src/plan.cpp:320-338) and
// weights per element VRR1 3, VRR2 8, VRR3 3, VRR4 8, VRR5 11, VRR6 6.
static int ref_vrr_flops(int la, int lb, int lc, int ld)
{
   std::map<std::pair<int, int>, std::pair<int, int>> mr;  // (a,c) -> (min m, max m)
   std::set<std::tuple<int, int, int>> seen;
   std::vector<std::tuple<int, int, int>> stack;
   for (int e = la; e <= la + lb; e++)
      for (int f = lc; f <= lc + ld; f++) stack.emplace_back(e, f, 0);
   while (!stack.empty()) {
      auto [a, c, m] = stack.back();
      stack.pop_back();
      if (a + c == 0 || !seen.insert({a, c, m}).second) continue;
      auto it = mr.find({a, c});
      if (it == mr.end()) mr[{a, c}] = {m, m};
      else it->second = {std::min(it->second.first, m), std::max(it->second.second, m)};
      if (c == 0) {
         stack.emplace_back(a - 1, 0, m);
         stack.emplace_back(a - 1, 0, m + 1);
         if (a > 1) {
            stack.emplace_back(a - 2, 0, m);
            stack.emplace_back(a - 2, 0, m + 1);
         }
      } else {
         stack.emplace_back(a, c - 1, m);
         stack.emplace_back(a, c - 1, m + 1);
         if (c > 1) {
            stack.emplace_back(a, c - 2, m);
            stack.emplace_back(a, c - 2, m + 1);
         }
         if (a > 0) stack.emplace_back(a - 1, c - 1, m + 1);
      }
   }
   long fl = 0;
   for (auto &kv : mr) {
      const int a = kv.first.first, c = kv.first.second;
      int w;
      if (c == 0) w = (a == 1) ? 3 : 8;
      else if (a == 0) w = (c == 1) ? 3 : 8;
      else w = (c == 1) ? 6 : 11;
      fl += (long)w * (kv.second.second - kv.second.first + 1) * nco(a) * nco(c);
   }
   return (int)fl;
}

ClassPlan make_plan(int la, int lb, int lc, int ld)
{
   ClassPlan p;
   std::memset(&p, 0, sizeof p);
   p.la = la; p.lb = lb; p.lc = lc; p.ld = ld;
   p.LA = la + lb;
   p.LC = lc + ld;
   p.L = p.LA + p.LC;
   p.Ns = nsph(la) * nsph(lb) * nsph(lc) * nsph(ld);

   // (e0|f0) blocks that feed the HRR, e outer, f inner
   for (int e = la; e <= p.LA; e++)
      for (int f = lc; f <= p.LC; f++) p.ncp += nco(e) * nco(f);

   p.fm_flops = 52 + 211 * (p.L + 1);
   p.vrr_flops = ref_vrr_flops(la, lb, lc, ld);
   // 2 per element of the HRR layers: ket layer dd of the blocks (e,c), then
   // bra layer bb of the blocks a
   const int ncd = nco(lc) * nco(ld);
   for (int dd = 1; dd <= ld; dd++)
      for (int e = la; e <= p.LA; e++)
         for (int c = lc; c <= p.LC - dd; c++) p.hrr_flops += 2 * nco(e) * nco(c) * nco(dd);
   for (int bb = 1; bb <= lb; bb++)
      for (int a = la; a <= p.LA - bb; a++) p.hrr_flops += 2 * nco(a) * nco(bb) * ncd;
   {
      int dims[4] = {nco(la), nco(lb), nco(lc), nco(ld)};
      const int ls[4] = {la, lb, lc, ld};
      int sf = 0;
      for (int s = 0; s < 4; s++) {
         const int k = dims[0], n = dims[1] * dims[2] * dims[3], m = nsph(ls[s]);
         sf += 2 * m * n * k;
         dims[0] = dims[1]; dims[1] = dims[2]; dims[2] = dims[3]; dims[3] = m;
      }
      p.sph_flops = sf;
   }
   return p;
}

// odd multiplier of a class in the survivor checksum (the oracle uses the
// same function)
uint64_t class_mult(int code)
{
   uint64_t z = 0xC1A55E5ULL + (uint64_t)code * 0x9E3779B97F4A7C15ULL;
   z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ULL;
   z = (z ^ (z >> 27)) * 0x94d049bb133111ebULL;
   z = z ^ (z >> 31);
   return z | 1ull;
}

// FLOPs of the Hermite recursion R^(n)_tuv, n = L-1..0, from the G_m ladder:
// an element whose recursion direction has component >= 2 costs 3 (one
// product with (t-1), one fused product-add), otherwise 1; plus the (-2 rho)^n
// scaling (2 per order) and the cell accumulation of the n = 0 layer.
static long long herm_flops(int L)
{
   long long f = 2LL * (L + 1);
   for (int n = L - 1; n >= 0; n--)
      for (int N = 1; N <= L - n; N++)
         for (int t = N; t >= 0; t--)
            for (int u = N - t; u >= 0; u--) {
               const int v = N - t - u;
               const int c = t > 0 ? t : (u > 0 ? u : v);
               f += c >= 2 ? 3 : 1;
            }
   return f + nherm(L);
}

void make_type_plan(TypePlan &tp)
{
   TypePlan p;
   std::memset(&p, 0, sizeof p);
   for (int t = 0; t < 4; t++) {
      p.nsh[t] = tp.nsh[t];
      for (int s = 0; s < tp.nsh[t]; s++) {
         p.l[t][s] = tp.l[t][s];
         p.nl[t][s] = tp.nl[t][s];
      }
   }
   int lmin[4], lmax[4];
   for (int t = 0; t < 4; t++) {
      lmin[t] = 99;
      lmax[t] = -1;
      for (int s = 0; s < p.nsh[t]; s++) {
         lmin[t] = std::min(lmin[t], p.l[t][s]);
         lmax[t] = std::max(lmax[t], p.l[t][s]);
      }
   }
   p.LA0 = lmin[0];
   p.LA = lmax[0] + lmax[1];
   p.LC0 = lmin[2];
   p.LC = lmax[2] + lmax[3];
   p.L = p.LA + p.LC;
   int off = 0;
   for (int f = p.LC0; f <= p.LC; f++) {
      p.kcoff[f] = off;
      off += nco(f);
   }
   p.nkc = off;
   off = 0;
   for (int e = p.LA0; e <= p.LA; e++) {
      p.bcoff[e] = off;
      off += nco(e);
   }
   p.ncp = off * p.nkc;
   p.nbh = nherm(p.LA);
   p.nh = nherm(p.L);
   p.has00 = (p.LA0 == 0 && p.LC0 == 0) ? 1 : 0;
   // ket components per pass of the transform: about 4 KB of [nbh][FC + 2]
   p.FC = std::max(4, std::min((p.nkc + 3) & ~3, (512 / p.nbh - 2) & ~3));
   auto nterms = [](int l0, int l1) {
      int n = 0;
      for (int l = l0; l <= l1; l++)
         for (int lx = l; lx >= 0; lx--)
            for (int ly = l - lx; ly >= 0; ly--) n += ((lx + 1) * (ly + 1) * (l - lx - ly + 1) + 1) & ~1;
      return n;
   };
   p.nkt = nterms(p.LC0, p.LC);
   p.nbt = nterms(p.LA0, p.LA);

   std::set<int> Lset;
   int k = 0;
   long long ref = 0;
   for (int sa = 0; sa < p.nsh[0]; sa++)
      for (int sb = 0; sb < p.nsh[1]; sb++)
         for (int sc = 0; sc < p.nsh[2]; sc++)
            for (int sd = 0; sd < p.nsh[3]; sd++, k++) {
               const int la = p.l[0][sa], lb = p.l[1][sb], lc = p.l[2][sc], ld = p.l[3][sd];
               const ClassPlan cp = make_plan(la, lb, lc, ld);
               p.cls_code[k] = class_code(la, lb, lc, ld);
               p.cls_sh[k] = sa | sb << 4 | sc << 8 | sd << 12;
               p.cls_nl[k] = p.nl[0][sa] * p.nl[1][sb] * p.nl[2][sc] * p.nl[3][sd];
               p.cls_ncp[k] = cp.ncp;
               p.cls_mult[k] = class_mult(p.cls_code[k]);
               p.mult_all += p.cls_mult[k];
               Lset.insert(cp.L);
               ref += cp.fm_flops + cp.vrr_flops;
            }
   p.nclass = k;
   for (int t = 0; t < 4; t++) {
      int f = 0;
      for (int s2 = 0; s2 < p.nsh[t]; s2++) {
         p.fun0[t][s2] = f;
         f += p.nl[t][s2] * nsph(p.l[t][s2]);
      }
      p.nfun[t] = f;
   }
   p.nL = 0;
   for (int L : Lset) p.Ls[p.nL++] = L;
   for (k = 0; k < p.nclass; k++) {
      const int c = p.cls_code[k];
      const int L = c / 64 + (c / 16) % 4 + (c / 4) % 4 + c % 4;
      for (int i = 0; i < p.nL; i++)
         if (p.Ls[i] == L) p.cls_gate[k] = i;
   }
   p.ref_slot_flops = ref;
   p.surv_flops = 52 + 211LL * (p.L + 1) + herm_flops(p.L);
   // Hermite -> cartesian: E coefficients (3 directions, 3 FLOPs per entry
   // on each side), then 3 FLOPs per term of the two contraction stages
   long long pf = 0;
   for (int e = 0; e <= p.LA; e++) pf += 3LL * 3 * (e + 1);
   for (int f = 0; f <= p.LC; f++) pf += 3LL * 3 * (f + 1);
   for (int N = 0; N <= p.LA; N++)
      for (int t = N; t >= 0; t--)
         for (int u = N - t; u >= 0; u--)
            for (int f = p.LC0; f <= p.LC; f++)
               for (int fx = f; fx >= 0; fx--)
                  for (int fy = f - fx; fy >= 0; fy--) pf += 3LL * (fx + 1) * (fy + 1) * (f - fx - fy + 1);
   for (int e = p.LA0; e <= p.LA; e++)
      for (int ex = e; ex >= 0; ex--)
         for (int ey = e - ex; ey >= 0; ey--) pf += 3LL * p.nkc * (ex + 1) * (ey + 1) * (e - ex - ey + 1);
   p.prim_flops = pf;
   tp = p;
}

// Tables of a type's Hermite -> cartesian transform: a component (ex,ey,ez)
// has the terms E^ex_a E^ey_b E^ez_d of its one-centre expansion.
//   items[0 .. nkt)  ket terms: entries e (e + 1) / 2 + a of the three
//                    directions' E (5 bits each), place << 15 (herm_place),
//                    bit 31: none, its coefficient is 0
//   then             nbt bra terms, the place a Hermite triple's index
//   then             nkc ket components, passes of FC, within a pass by
//                    falling number of terms: component | first term << 8 |
//                    terms << 20 (an even number, the last may be 0)
//   then             the bra components by falling number of terms, likewise
//   then             the places of the nbh bra Hermite triples
void make_type_items(const TypePlan &tp, std::vector<uint32_t> &items)
{
   // cartesian components of shell L in order: lx descending, then ly descending
   auto comps = [](int L) {
      std::vector<std::array<int, 3>> v;
      for (int lx = L; lx >= 0; lx--)
         for (int ly = L - lx; ly >= 0; ly--) v.push_back({lx, ly, L - lx - ly});
      return v;
   };
   auto entry = [](int e, int a) { return (uint32_t)(e * (e + 1) / 2 + a); };
   std::vector<std::array<int, 3>> ket, bra, herm;
   for (int f = tp.LC0; f <= tp.LC; f++)
      for (auto &c : comps(f)) ket.push_back(c);
   for (int e = tp.LA0; e <= tp.LA; e++)
      for (auto &c : comps(e)) bra.push_back(c);
   for (int N = 0; N <= tp.LA; N++)
      for (auto &h : comps(N)) herm.push_back(h);
   items.clear();
   std::vector<uint32_t> rec[2];
   for (int side = 0; side < 2; side++) {
      const size_t first = items.size();
      auto &cs = side == 0 ? ket : bra;
      for (size_t i = 0; i < cs.size(); i++) {
         const auto &c = cs[i];
         const size_t start = items.size() - first;
         for (int a = 0; a <= c[0]; a++)
            for (int b = 0; b <= c[1]; b++)
               for (int d = 0; d <= c[2]; d++) {
                  const int N = a + b + d;
                  const int place = side == 0 ? herm_place(tp.L, a, b, d)
                                              : N * (N + 1) * (N + 2) / 6 + (N - a) * (N - a + 1) / 2 + d;
                  items.push_back(entry(c[0], a) | entry(c[1], b) << 5 | entry(c[2], d) << 10 | (uint32_t)place << 15);
               }
         if ((items.size() - first - start) & 1) items.push_back(1u << 31);
         const size_t n = items.size() - first - start;
         rec[side].push_back((uint32_t)i | (uint32_t)start << 8 | (uint32_t)n << 20);
      }
   }
   auto more = [](uint32_t a, uint32_t b) { return a >> 20 > b >> 20; };
   for (size_t f0 = 0; f0 < ket.size(); f0 += tp.FC)
      std::stable_sort(rec[0].begin() + f0, rec[0].begin() + std::min(f0 + tp.FC, ket.size()), more);
   std::stable_sort(rec[1].begin(), rec[1].end(), more);
   for (auto &r : rec) items.insert(items.end(), r.begin(), r.end());
   for (auto &h : herm) items.push_back((uint32_t)herm_place(tp.L, h[0], h[1], h[2]));
}

// The matrix-core contraction of a type (k_eco): its classes of at least
// ECO_MIN_NQ contractions, one work item per 64 columns x 64 contractions of
// each, their places in a row of the contraction buffer and their columns
// among the type's.
void make_eco_plan(const TypePlan &tp, const std::vector<ClassPlan> &cps, EcoPlan &ep)
{
   ep = EcoPlan();
   ep.off.assign(tp.nclass, -1);
   ep.info.assign(2 * MAXTC, 0);
   for (int k = 0; k < tp.nclass; k++) {
      const int nq = tp.cls_nl[k], cols = tp.cls_ncp[k];
      if (nq < ECO_MIN_NQ) continue;
      ep.off[k] = (int)ep.row;
      ep.info[k] = (int)ep.srcmaps.size();
      ep.info[MAXTC + k] = (int)ep.row;
      ep.row += (size_t)nq * cols;
      const ClassPlan &cp = cps[k];
      for (int e = cp.la; e <= cp.LA; e++)
         for (int ie = 0; ie < nco(e); ie++)
            for (int f = cp.lc; f <= cp.LC; f++)
               for (int jf = 0; jf < nco(f); jf++)
                  ep.srcmaps.push_back((tp.bcoff[e] + ie) * tp.nkc + tp.kcoff[f] + jf);
      for (int jt0 = 0; jt0 * 16 < cols; jt0 += 4)
         for (int qb = 0; qb * 64 < nq; qb++) ep.items.push_back(EcoItem{(uint16_t)k, (uint16_t)jt0, (uint16_t)qb, 0});
   }
   // items in the order of the first type column they read: the classes
   // share the row's blocks (a block (e,f) serves every class with
   // la <= e <= la+lb, lc <= f <= lc+ld), so items that run together read
   // the same columns of a row that is larger than the caches
   auto first_col = [&](const EcoItem &it) { return ep.srcmaps[ep.info[it.k] + it.jt0 * 16]; };
   std::stable_sort(ep.items.begin(), ep.items.end(), [&](const EcoItem &a, const EcoItem &b) {
      const int ca = first_col(a), cb = first_col(b);
      return ca < cb || (ca == cb && (a.k < b.k || (a.k == b.k && a.qb < b.qb)));
   });
}

// Registers of a pair's transform: 0 without f shells, 1 with one whose
// transform is no larger than (dd|'s, 2 the others ((df|, (fd|, (ff|).
static int sq_group(int l1, int l2) { return l1 <= 2 && l2 <= 2 ? 0 : (l1 + l2 <= 4 ? 1 : 2); }

// One side of a type (bra: sets 0, 1; ket: sets 2, 3) in tiles of at most
// `max_row` rows and `max_fn` functions, of the shell pairs of register group
// `grp` (sq_group); single: one shell pair per tile.
static void make_sq_tiles(const TypePlan &tp, int side, int grp, int max_row, int max_fn, bool single, SqPlan &sp,
                          std::vector<int> &out)
{
   const int x = 2 * side, y = 2 * side + 1, low = side ? tp.LC0 : tp.LA0;
   auto below = [](int l) { return l * (l + 1) * (l + 2) / 6; };
   auto con0 = [&](int set, int s) {   // contractions of the set's shells before s
      int n = 0;
      for (int i = 0; i < s; i++) n += tp.nl[set][i];
      return n;
   };
   SqTile t{};
   int lo1 = 0, hi1 = 0, lo2 = 0, hi2 = 0, e0 = 0, e1 = 0;
   auto close = [&]() {
      if (!t.nrow) return;
      t.comp0 = (uint16_t)(below(e0) - below(low));
      t.ncomp = (uint16_t)(below(e1 + 1) - below(e0));
      t.r1 = (uint16_t)lo1;
      t.n1 = (uint16_t)(hi1 - lo1);
      t.r2 = (uint16_t)lo2;
      t.n2 = (uint16_t)(hi2 - lo2);
      t.row = (uint32_t)sp.rows.size();
      t.rc = (uint32_t)sp.rcs.size() / 2;
      t.fn = (uint32_t)sp.fns.size();
      int rc = 0;
      for (int i = 0; i < t.nsp; i++) {
         SqSp &q = sp.sps[t.sp + i];
         q.f1 = (int16_t)(tp.fun0[x][q.s1] - lo1);
         q.f2 = (int16_t)(tp.fun0[y][q.s2] - lo2);
         for (int c = q.c0; c < q.c0 + q.nc; c++, rc++) {
            const int i1 = c / q.n2, i2 = c % q.n2;
            const int c0 = below(q.l1) - below(e0), nr = below(q.l1 + q.l2 + 1) - below(q.l1);
            sp.rcs.push_back((uint32_t)(con0(x, q.s1) + i1) | (uint32_t)(con0(y, q.s2) + i2) << 8);
            sp.rcs.push_back((uint32_t)(q.row0 + (c - q.c0) * nr) | (uint32_t)c0 << 8 | (uint32_t)(c0 + nr) << 16);
            for (int r = 0; r < nr; r++) sp.rows.push_back((uint16_t)((c0 + r) | rc << 8));
            for (int s1 = 0; s1 < nsph(q.l1); s1++)
               for (int s2 = 0; s2 < nsph(q.l2); s2++)
                  sp.fns.push_back((uint32_t)(q.f1 + i1 * nsph(q.l1) + s1) | (uint32_t)(q.f2 + i2 * nsph(q.l2) + s2) << 8 |
                                   (uint32_t)i << 16);
         }
      }
      out.push_back((int)sp.tiles.size());
      sp.tiles.push_back(t);
      t = SqTile{};
   };
   // the first shells apart (their function ranges stay short) unless the
   // whole side is one tile
   int all = 0, all_fn = 0;
   for (int s1 = 0; s1 < tp.nsh[x]; s1++)
      for (int s2 = 0; s2 < tp.nsh[y]; s2++) {
         const int l1 = tp.l[x][s1], l2 = tp.l[y][s2], nc = tp.nl[x][s1] * tp.nl[y][s2];
         all += nc * (below(l1 + l2 + 1) - below(l1));
         all_fn += nc * nsph(l1) * nsph(l2);
      }
   const bool whole = all <= max_row && all_fn <= max_fn;
   for (int s1 = 0; s1 < tp.nsh[x]; s1++)
      for (int s2 = 0; s2 < tp.nsh[y]; s2++) {
         const int l1 = tp.l[x][s1], l2 = tp.l[y][s2];
         if (!whole && s2 == 0) close();
         if (sq_group(l1, l2) != grp) continue;
         const int nr = below(l1 + l2 + 1) - below(l1), nf = nsph(l1) * nsph(l2);
         const int nc = tp.nl[x][s1] * tp.nl[y][s2];
         if (single) close();
         for (int c = 0; c < nc; c++) {
            if (t.nrow && (t.nrow + nr > max_row || t.nfn + nf > max_fn || t.nrc + 1 > SQ_MAXRC)) close();
            if (!t.nrow) {
               t.sp = (uint32_t)sp.sps.size();
               lo1 = lo2 = 1 << 20;
               hi1 = hi2 = 0;
               e0 = 99;
               e1 = 0;
            }
            if (!t.nsp || sp.sps.back().s1 != s1 || sp.sps.back().s2 != s2) {
               SqSp q{};
               q.l1 = (uint8_t)l1;
               q.l2 = (uint8_t)l2;
               q.s1 = (uint8_t)s1;
               q.s2 = (uint8_t)s2;
               q.c0 = (uint8_t)c;
               q.n2 = (uint8_t)tp.nl[y][s2];
               q.row0 = t.nrow;
               q.fn0 = t.nfn;
               sp.sps.push_back(q);
               t.nsp++;
               e0 = std::min(e0, l1);
               e1 = std::max(e1, l1 + l2);
            }
            sp.sps.back().nc++;
            const int i1 = tp.fun0[x][s1] + c / tp.nl[y][s2] * nsph(l1), i2 = tp.fun0[y][s2] + c % tp.nl[y][s2] * nsph(l2);
            lo1 = std::min(lo1, i1);
            hi1 = std::max(hi1, i1 + nsph(l1));
            lo2 = std::min(lo2, i2);
            hi2 = std::max(hi2, i2 + nsph(l2));
            t.nrow += nr;
            t.nfn += nf;
            t.nrc++;
         }
      }
   close();
}

// The k_sq launch of the items of a type whose larger register group
// (sq_group) is `grp`, for nspin density matrices; eco: classes of at least
// ECO_MIN_NQ contractions take their contracted blocks from the contraction
// buffer (a tile is then part of one shell pair).
void make_sq_plan(const TypePlan &tp, const EcoPlan &ep, int grp, int nspin, bool eco, SqPlan &sp)
{
   sp = SqPlan();
   int lx = 0;
   for (int t = 0; t < 4; t++)
      for (int s = 0; s < tp.nsh[t]; s++) lx = std::max(lx, tp.l[t][s]);
   sp.lm = grp ? 2 + grp : (lx <= 1 ? 1 : 2);
   for (int t = 0; t < 4; t++)
      for (int s = 0; s < tp.nsh[t]; s++)
         for (int i = 0; i < tp.nl[t][s]; i++) sp.cons.push_back((uint16_t)(s | i << 8));
   std::vector<int> bra[3], ket[3];
   for (int f = 0; f <= grp; f++) {
      make_sq_tiles(tp, 0, f, 42, SQ_MAXFN, eco, sp, bra[f]);
      make_sq_tiles(tp, 1, f, 32, 30, eco, sp, ket[f]);
   }
   std::vector<SqItem> large;
   for (int fb = 0; fb <= grp; fb++)
      for (int fk = 0; fk <= grp; fk++) {
         if (std::max(fb, fk) != grp) continue;
         for (int bi : bra[fb])
            for (int ki : ket[fk]) {
               const SqTile &b = sp.tiles[bi], &k = sp.tiles[ki];
               SqItem it{};
               it.bt = (uint16_t)bi;
               it.kt = (uint16_t)ki;
               it.eco_off = -1;
               if (eco) {
                  const SqSp &qb = sp.sps[b.sp], &qk = sp.sps[k.sp];
                  const int c = ((qb.s1 * tp.nsh[1] + qb.s2) * tp.nsh[2] + qk.s1) * tp.nsh[3] + qk.s2;
                  it.eco_off = ep.off[c];
               }
               const int pk = 2 * nspin * (b.n1 + b.n2) * (k.n1 + k.n2);
               it.lds_k = pk <= 512 * nspin ? 1 : 0;
               int off = SQ_TAB_BYTES / 8;
               it.o_pk = off;
               off += it.lds_k ? pk : 0;
               it.o_c = off;
               off += b.nrow * (k.nrow | 1);
               const bool small = sp.lm == SQ_KERNELS && 8 * off <= SQ_SMALL_LDS;
               if (small) sp.lds_small = std::max(sp.lds_small, 8 * off);
               sp.lds_bytes = std::max(sp.lds_bytes, 8 * off);
               (small ? sp.items : large).push_back(it);
            }
      }
   sp.nsmall = (int)sp.items.size();
   sp.items.insert(sp.items.end(), large.begin(), large.end());
}

}  // namespace gint
