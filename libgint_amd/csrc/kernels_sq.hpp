// k_sq: from the primitive (e0|f0) blocks of a set quartet to its K updates,
// one wavefront per (set quartet, bra tile, ket tile).  A tile is a run of
// (shell pair, contraction pair) units of one side, so one item covers the
// classes of several shell pairs at once.  For each (n1,n2) row:
//
//   contraction      C[unit, e][col] = sum over the primitive quartets n of
//                    (K_a K_b)[n][unit] (K_c K_d)[n][col] A[n][e][f(col)]
//                    (reference src/compute_ECO.cpp:12-214) in FP64
//                    matrix-core tiles: 4 or 16 bra units x 16 (e, col) x 4
//                    primitive quartets; or a copy of the blocks k_eco
//                    contracted
//   ket transform    HRR d -> c and cartesian -> spherical of the ket pair
//                    (src/compute_HRR.cpp, src/compute_SPH.cpp:58-237), one
//                    (row, unit) per lane, in registers, C in place
//   bra transform    the same on the bra side, one (unit, ket function) per
//                    lane
//   K update         from the lane's integrals in registers (src/compute_KS.cpp:
//                    8-117): its sums over a or b go to the item's four K
//                    blocks in LDS, from there one atomic per element to K
//
// The transforms act on one side of the integral only, so the HRR is done
// for (components + function) vectors instead of the full four-index block,
// and every index and coefficient is a compile-time constant (the pair
// (l1,l2) is a template parameter, chosen by a uniform branch).  One
// wavefront per workgroup: the phases exchange data through LDS in program
// order, with no barrier and no wait for loads in flight.
//
// A wavefront or a workgroup per set quartet and class, with the four-index
// HRR in LDS, took 250 ms for 262 k set quartets (32 waters, 27 cells), items
// of several shell pairs 66.  What brought that to 34 (MI355X):
//   - the item's set-up: all of its loads that do not wait for each other at
//     once, instead of a load after another per shell (28 k -> 12 k cycles)
//   - the items of a set quartet on one XCD, so that its blocks come from one
//     L2 (xcd_run: 172 -> 57 GB from memory and 42.8 -> 32.2 ms; at 46 ms
//     runs of 16 items took 50, of 512 49; of k_sq<4>'s large items 16 are
//     better, 27.5 for 28.4 ms)
//   - tiles of at most 42 rows x 32 columns: whole matrix-core tiles of 16
//     columns, and LDS (16 KB at most with one spin, 20 with two, and the
//     coefficients) for eight wavefronts per CU or more (38 x 38: 45.7,
//     30 x 38: 44.0, 35 x 32: 42.1, but 34 for 29.6 ms in f shells)
//   - in the contraction four independent matrix-core chains, with the next
//     loads in flight (f shells: 58 -> 53 ms) and weights taken per column
//     from the coefficients, not from a table of the window
//   - large set quartets in parts and by falling work (SqSeg):
//     no launch ends on a few wavefronts; 93 -> 76 ms where the largest have
//     16384 primitive quartets
//   - matrix-core tiles of 4 rows for tiles of at most 8 units (39 -> 34 ms)
//   - the contraction's loads at a uniform base plus 32 bits per lane instead
//     of 64-bit addresses (K-build with s to f shells 96.5 -> 95.7 ms)
// Bound: latency and instruction issue, at 2.4 wavefronts per SIMD (k_sq<3>
// 1.9, k_sq<4> 1.2): waits in 44 to 49% of the wave cycles, VALU busy 21 to
// 42%, matrix cores 6 to 27%; 0.5 to 2.5 TB/s from memory.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>
#include <utility>

#include "c2s_table.h"
#include "device.hpp"
#include "gint_math.h"
#include "uniform.hpp"

namespace gint {
namespace sq {

__host__ __device__ constexpr int comp(int L, int i, int d)
{
   int n = 0;
   for (int lx = L; lx >= 0; lx--)
      for (int ly = L - lx; ly >= 0; ly--) {
         if (n == i) return d == 0 ? lx : (d == 1 ? ly : L - lx - ly);
         n++;
      }
   return 0;
}
__host__ __device__ constexpr int cidx(int L, int lx, int lz) { return (L - lx) * (L - lx + 1) / 2 + lz; }
__host__ __device__ constexpr int n_co(int l) { return (l + 1) * (l + 2) / 2; }
__host__ __device__ constexpr int co_below(int l) { return l * (l + 1) * (l + 2) / 6; }   // components of shells 0..l-1
__host__ __device__ constexpr int n_side(int l1, int l2) { return co_below(l1 + l2 + 1) - co_below(l1); }
__host__ __device__ constexpr double c2s(int l, int m, int k)
{
   constexpr double v[] = {GINT_C2S_VALUES};
   constexpr int off[4] = {GINT_C2S_OFF_0, GINT_C2S_OFF_1, GINT_C2S_OFF_2, GINT_C2S_OFF_3};
   return v[off[l] + m * n_co(l) + k];
}
__host__ __device__ constexpr int binom(int n, int k) { return (k == 0 || k == n) ? 1 : n; }   // n <= 3

template <int... I, class F>
__device__ __forceinline__ void for_seq(std::integer_sequence<int, I...>, F &&f)
{
   (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F &&f)
{
   for_seq(std::make_integer_sequence<int, N>{}, static_cast<F &&>(f));
}

__device__ __forceinline__ double rpow(double r, int n) { return n == 0 ? 1.0 : (n == 1 ? r : (n == 2 ? r * r : r * r * r)); }

// One side: from the components of shells l1 .. l1 + l2 on the first centre
// to the spherical pairs (s1 s2).  The HRR (x, y + 1_d| = (x + 1_d, y| + R_d
// (x, y|, R = AB or CD, unrolled:
//    (x y| = sum_{0 <= i <= y} prod_d C(y_d, i_d) R_d^(y_d - i_d) (x + i, 0|
// for one y at a time (few values live), then both c2s with their zeros
// left out.
template <int l1, int l2>
__device__ __forceinline__ void side_transform(const double *in, const double R[3], double *out)
{
   constexpr int N1 = n_co(l1), S1 = 2 * l1 + 1, S2 = 2 * l2 + 1;
#pragma unroll
   for (int s = 0; s < S1 * S2; s++) out[s] = 0.0;
   static_for<n_co(l2)>([&](auto Y) {
      constexpr int y = decltype(Y)::value;
      constexpr int y0 = comp(l2, y, 0), y1 = comp(l2, y, 1), y2 = comp(l2, y, 2);
      double v[N1];
#pragma unroll
      for (int x = 0; x < N1; x++) v[x] = 0.0;
      static_for<(y0 + 1) * (y1 + 1) * (y2 + 1)>([&](auto I) {
         constexpr int i = decltype(I)::value;
         constexpr int i2 = i % (y2 + 1), i1 = (i / (y2 + 1)) % (y1 + 1), i0 = i / ((y2 + 1) * (y1 + 1));
         constexpr int e = l1 + i0 + i1 + i2;
         constexpr double bin = (double)(binom(y0, i0) * binom(y1, i1) * binom(y2, i2));
         const double m = bin * rpow(R[0], y0 - i0) * rpow(R[1], y1 - i1) * rpow(R[2], y2 - i2);
         static_for<N1>([&](auto X) {
            constexpr int x = decltype(X)::value;
            constexpr int src = co_below(e) - co_below(l1) + cidx(e, comp(l1, x, 0) + i0, comp(l1, x, 2) + i2);
            if constexpr (i0 == y0 && i1 == y1 && i2 == y2) v[x] += in[src];
            else v[x] += m * in[src];
         });
      });
      static_for<S1>([&](auto A) {
         constexpr int s1 = decltype(A)::value;
         double t = 0.0;
         static_for<N1>([&](auto X) {
            constexpr int x = decltype(X)::value;
            constexpr double c = c2s(l1, s1, x);
            if constexpr (c == 1.0) t += v[x];
            else if constexpr (c != 0.0) t += c * v[x];
         });
         static_for<S2>([&](auto B) {
            constexpr int s2 = decltype(B)::value;
            constexpr double c = c2s(l2, s2, y);
            if constexpr (c == 1.0) out[s1 * S2 + s2] += t;
            else if constexpr (c != 0.0) out[s1 * S2 + s2] += c * t;
         });
      });
   });
}

// x / d for 0 <= x < 2^22, d >= 1
__device__ __forceinline__ int fdiv(int x, int d)
{
   int q = (int)((float)x * __builtin_amdgcn_rcpf((float)d));
   const int rem = x - q * d;
   if (rem < 0) q--;
   else if (rem >= d) q++;
   return q;
}

// Where coefficient i of a set quartet lies in the basis data: the sets'
// contractions follow each other, np coefficients each
struct CoefMap {
   const uint16_t *cons;
   const uint32_t *Kof;   // [4][MAXSH]
   int n0, n1, n2;        // first contraction of sets 1 to 3
   int ob, oc, od;        // their first coefficient
   int npa, npb, npc, npd;
};
__device__ __forceinline__ uint32_t coef_at(const CoefMap m, int i)
{
   const int tc = (i >= m.ob) + (i >= m.oc) + (i >= m.od);
   const int np = tc == 0 ? m.npa : (tc == 1 ? m.npb : (tc == 2 ? m.npc : m.npd));
   const int x = i - (tc == 0 ? 0 : (tc == 1 ? m.ob : (tc == 2 ? m.oc : m.od)));
   const int con = fdiv(x, np);
   const uint32_t c = m.cons[(tc == 0 ? 0 : (tc == 1 ? m.n0 : (tc == 2 ? m.n1 : m.n2))) + con];
   return m.Kof[tc * MAXSH + (int)(c & 255)] + (c >> 8) * (uint32_t)np + (uint32_t)(x - con * np);
}

// Where element e of an item's four blocks (ac, ad, bc, bd) lies in P and K
struct BlockMap {
   KsSet s;
   int NC, ND, oad, obc, obd;
   unsigned ra, rb, rc, rd;   // first function of the tiles on the four centres
};
__device__ __forceinline__ size_t block_at(const BlockMap m, int e)
{
   const bool bc = e >= m.obc, d = e >= (bc ? m.obd : m.oad);   // rows of b; columns of d
   const int nc = d ? m.ND : m.NC;
   const int x = e - (bc ? (d ? m.obd : m.obc) : (d ? m.oad : 0));
   const unsigned ld = ((bc ? m.s.ld23 : m.s.ld01) >> (d ? 16 : 0)) & 0xffff;
   const bool tr = (m.s.flags >> ((bc ? 2 : 0) + (d ? 1 : 0))) & 1;
   const int r = fdiv(x, nc), c = x - r * nc;
   const size_t base = bc ? (d ? m.s.base[3] : m.s.base[2]) : (d ? m.s.base[1] : m.s.base[0]);
   return base + (size_t)((bc ? m.rb : m.ra) + r) * (tr ? ld : 1) + (size_t)((d ? m.rd : m.rc) + c) * (tr ? 1 : ld);
}

struct GroupHead {   // the start of GroupRec
   uint32_t row0, row1, R[4];
};
struct Vec3 {
   double v[3];
};
struct Cell {
   double v[18];
};

__device__ __forceinline__ unsigned blk_at(bool T, unsigned ld, unsigned r, unsigned c) { return T ? r * ld + c : c * ld + r; }
__device__ __forceinline__ double symm_fac(uint32_t code)
{
   return code >= 4 ? 0.0 : (code == 0 ? 2.0 : (code == 1 ? 1.0 : (code == 2 ? 0.5 : 0.25)));
}

constexpr int SQ_EU = 4;   // components whose loads are in flight together in the contraction

typedef double dbl4 __attribute__((ext_vector_type(4)));

// What the K update of an item needs
struct Upd {
   const BatchDev &b;
   const KTargets &kt;
   const TypePlan &tp;
   const GroupRec &g;
   const SqSp *ksp;     // the ket tile's shell pairs
   double *Pl, *Kl;     // LDS: the four P and K blocks of the item, per spin [ac | ad | bc | bd]
   const uint32_t *fn;  // LDS: ket functions
   bool lds;            // through them, else straight to K or the integral output
   bool add;            // integral output: an earlier row wrote already
   int NA, NB, NC, ND;
};

// the updates of bra contraction cb of shell pair q with ket function f, by
// the K layout of the class: integral x (2 lb + 1) + y at I[(x (2 lb + 1) + y) is]
__device__ __forceinline__ void k_update_class(const double *I, int is, const Upd &u, const SqSp &q, int cb, int f)
{
   const int SA = 2 * q.l1 + 1, SB = 2 * q.l2 + 1;
   const uint32_t fe = u.fn[f];
   const SqSp &kq = u.ksp[fe >> 16];
   const TypePlan &tp = u.tp;
   const int k = ((q.s1 * tp.nsh[1] + q.s2) * tp.nsh[2] + kq.s1) * tp.nsh[3] + kq.s2;
   const KsGroup ks = group_ks(u.b, tp, u.g, k);
   const int nlb = tp.nl[1][q.s2], nlc = tp.nl[2][kq.s1], nld = tp.nl[3][kq.s2];
   const int nsc = 2 * kq.l1 + 1, nsd = 2 * kq.l2 + 1;
   const int cf = (int)(fe & 255) - kq.f1, df = (int)((fe >> 8) & 255) - kq.f2;
   const int ia = cb / nlb, ib = cb - ia * nlb, ic = cf / nsc, isc = cf - ic * nsc, id = df / nsd, isd = df - id * nsd;
   const int l = (cb * nlc + ic) * nld + id;
   if (l >= (int)ks_count(ks.flags)) return;
   if (ks.flags & KS_OUTPUT) {
      double *O = u.kt.out + ((size_t)ks.base[0] | (size_t)ks.base[1] << 32);
      for (int x = 0; x < SA; x++)
         for (int y = 0; y < SB; y++) {
            double &o = O[tra_index(ia, x, ib, y, ic, isc, id, isd, nlb, nlc, nld, SA, SB, nsc, nsd)];
            o = u.add ? o + I[(x * SB + y) * is] : I[(x * SB + y) * is];
         }
      return;
   }
   size_t off[4];
   uint32_t ld01 = ks.ld01, ld23 = ks.ld23, flags = ks.flags;
   if (flags & KS_EXPLICIT) {
      const KsRec x = u.b.ksx[ks.expl + l];
      for (int z = 0; z < 4; z++) off[z] = x.off[z];
      ld01 = x.ld01;
      ld23 = x.ld23;
      flags = x.flags;
   } else {
      off[0] = (size_t)((long long)ks.base[0] + (long long)ia * ks.step[0] + (long long)ic * ks.step[1]);
      off[1] = (size_t)((long long)ks.base[1] + (long long)ia * ks.step[2] + (long long)id * ks.step[3]);
      off[2] = (size_t)((long long)ks.base[2] + (long long)ib * ks.step[4] + (long long)ic * ks.step[5]);
      off[3] = (size_t)((long long)ks.base[3] + (long long)ib * ks.step[6] + (long long)id * ks.step[7]);
   }
   const double fac = -symm_fac((flags >> 4) & 7) * u.kt.hf_fac;
   if (fac == 0.0) return;
   const unsigned ldac = ld01 & 0xffff, ldad = ld01 >> 16, ldbc = ld23 & 0xffff, ldbd = ld23 >> 16;
   const bool Tac = flags & 1, Tad = flags & 2, Tbc = flags & 4, Tbd = flags & 8;
   for (int sp = 0; sp < u.kt.nspin; sp++) {
      const double *P = sp ? u.kt.P[1] : u.kt.P[0];
      double *K = sp ? u.kt.K[1] : u.kt.K[0];
      for (int x = 0; x < SA; x++) {
         double kc = 0.0, kd = 0.0;
         for (int y = 0; y < SB; y++) {
            kc += I[(x * SB + y) * is] * P[off[3] + blk_at(Tbd, ldbd, y, isd)];
            kd += I[(x * SB + y) * is] * P[off[2] + blk_at(Tbc, ldbc, y, isc)];
         }
         unsafeAtomicAdd(&K[off[0] + blk_at(Tac, ldac, x, isc)], fac * kc);
         unsafeAtomicAdd(&K[off[1] + blk_at(Tad, ldad, x, isd)], fac * kd);
      }
      for (int y = 0; y < SB; y++) {
         double kc = 0.0, kd = 0.0;
         for (int x = 0; x < SA; x++) {
            kc += I[(x * SB + y) * is] * P[off[1] + blk_at(Tad, ldad, x, isd)];
            kd += I[(x * SB + y) * is] * P[off[0] + blk_at(Tac, ldac, x, isc)];
         }
         unsafeAtomicAdd(&K[off[2] + blk_at(Tbc, ldbc, y, isc)], fac * kc);
         unsafeAtomicAdd(&K[off[3] + blk_at(Tbd, ldbd, y, isd)], fac * kd);
      }
   }
}

// the same through the item's blocks in LDS (set-level K layout): the sums
// over b go to K_ac and K_ad, those over a to K_bc and K_bd
template <int la, int lb>
__device__ __forceinline__ void k_update_lds(const double *I, const Upd &u, const SqSp &q, int cb, int f)
{
   constexpr int SA = 2 * la + 1, SB = 2 * lb + 1;
   const uint32_t fe = u.fn[f];
   const int c = fe & 255, d = (fe >> 8) & 255;
   const int ia = cb / q.n2, ib = cb - ia * q.n2;
   const int a0 = q.f1 + ia * SA, b0 = q.f2 + ib * SB;
   const int oad = u.NA * u.NC, obc = oad + u.NA * u.ND, obd = obc + u.NB * u.NC;
   const int nblk = obd + u.NB * u.ND;
   for (int sp = 0; sp < u.kt.nspin; sp++) {
      const double *P = u.Pl + sp * nblk;
      double *K = u.Kl + sp * nblk;
      {
         double pc[SB], pd[SB];
#pragma unroll
         for (int y = 0; y < SB; y++) {
            pc[y] = P[obc + (b0 + y) * u.NC + c];
            pd[y] = P[obd + (b0 + y) * u.ND + d];
         }
#pragma unroll
         for (int x = 0; x < SA; x++) {
            double kc = 0.0, kd = 0.0;
#pragma unroll
            for (int y = 0; y < SB; y++) {
               kc += I[x * SB + y] * pd[y];
               kd += I[x * SB + y] * pc[y];
            }
            atomicAdd(&K[(a0 + x) * u.NC + c], kc);
            atomicAdd(&K[oad + (a0 + x) * u.ND + d], kd);
         }
      }
      double qc[SA], qd[SA];
#pragma unroll
      for (int x = 0; x < SA; x++) {
         qc[x] = P[(a0 + x) * u.NC + c];
         qd[x] = P[oad + (a0 + x) * u.ND + d];
      }
#pragma unroll
      for (int y = 0; y < SB; y++) {
         double kc = 0.0, kd = 0.0;
#pragma unroll
         for (int x = 0; x < SA; x++) {
            kc += I[x * SB + y] * qd[x];
            kd += I[x * SB + y] * qc[x];
         }
         atomicAdd(&K[obc + (b0 + y) * u.NC + c], kc);
         atomicAdd(&K[obd + (b0 + y) * u.ND + d], kd);
      }
   }
}

// ket transform of the units of one shell pair in the rows of C (row stride
// ts), in place: a unit's functions end where its columns ended at the
// latest, and the lanes take (row, unit) in rising order, so nothing unread
// is overwritten
template <int l1, int l2>
__device__ __forceinline__ void ket_units(double *T, int ts, int nrow, const SqSp &q, const double R[3], int lane)
{
   constexpr int NIN = n_side(l1, l2), NOUT = (2 * l1 + 1) * (2 * l2 + 1);
   const int nc = q.nc, n = nrow * nc;
   for (int i = lane; i < n; i += 64) {
      const int r = fdiv(i, nc), u = i - r * nc;
      const double *c = T + r * ts + q.row0 + u * NIN;
      double in[NIN], out[NOUT];
#pragma unroll
      for (int x = 0; x < NIN; x++) in[x] = c[x];
      side_transform<l1, l2>(in, R, out);
      double *d = T + r * ts + q.fn0 + u * NOUT;
#pragma unroll
      for (int x = 0; x < NOUT; x++) d[x] = out[x];
   }
}

// bra transform and K update of the units of one shell pair: lanes over
// (unit, ket function)
template <int l1, int l2>
__device__ __forceinline__ void bra_units(double *D, int ds, int nfn, const SqSp &q, const double R[3], const Upd &u,
                                          int lane)
{
   constexpr int NIN = n_side(l1, l2), NOUT = (2 * l1 + 1) * (2 * l2 + 1);
   const int n = q.nc * nfn;
   for (int i = lane; i < n; i += 64) {
      const int c = fdiv(i, nfn), f = i - c * nfn;
      double *d = D + (q.row0 + c * NIN) * ds + f;
      double in[NIN], out[NOUT];
#pragma unroll
      for (int x = 0; x < NIN; x++) in[x] = d[x * ds];
      side_transform<l1, l2>(in, R, out);
      if (u.lds) {
         k_update_lds<l1, l2>(out, u, q, q.c0 + c, f);
      } else {
         // back in place: k_update_class takes them from there
#pragma unroll
         for (int x = 0; x < NOUT; x++) d[x * ds] = out[x];
      }
   }
}

// the shell pairs of kernel LM
template <int LM>
__device__ constexpr bool has_pair(int l1, int l2)
{
   return LM == 4 || (LM == 3 ? l1 + l2 <= 4 : (l1 <= LM && l2 <= LM));
}

template <int LM>
__device__ __forceinline__ void ket_transform(double *T, int ts, int nrow, const SqSp &q, const double R[3], int lane)
{
   switch (q.l1 * 4 + q.l2) {
#define GINT_SQ_KET(a_, b_)                                                                              \
   case a_ * 4 + b_:                                                                                     \
      if constexpr (has_pair<LM>(a_, b_)) ket_units<a_, b_>(T, ts, nrow, q, R, lane);                    \
      break;
      GINT_SQ_KET(0, 0) GINT_SQ_KET(0, 1) GINT_SQ_KET(0, 2) GINT_SQ_KET(0, 3)
      GINT_SQ_KET(1, 0) GINT_SQ_KET(1, 1) GINT_SQ_KET(1, 2) GINT_SQ_KET(1, 3)
      GINT_SQ_KET(2, 0) GINT_SQ_KET(2, 1) GINT_SQ_KET(2, 2) GINT_SQ_KET(2, 3)
      GINT_SQ_KET(3, 0) GINT_SQ_KET(3, 1) GINT_SQ_KET(3, 2) GINT_SQ_KET(3, 3)
#undef GINT_SQ_KET
   }
}

template <int LM>
__device__ __forceinline__ void bra_transform(double *D, int ds, int nfn, const SqSp &q, const double R[3],
                                              const Upd &u, int lane)
{
   switch (q.l1 * 4 + q.l2) {
#define GINT_SQ_BRA(a_, b_)                                                                              \
   case a_ * 4 + b_:                                                                                     \
      if constexpr (has_pair<LM>(a_, b_)) bra_units<a_, b_>(D, ds, nfn, q, R, u, lane);                  \
      break;
      GINT_SQ_BRA(0, 0) GINT_SQ_BRA(0, 1) GINT_SQ_BRA(0, 2) GINT_SQ_BRA(0, 3)
      GINT_SQ_BRA(1, 0) GINT_SQ_BRA(1, 1) GINT_SQ_BRA(1, 2) GINT_SQ_BRA(1, 3)
      GINT_SQ_BRA(2, 0) GINT_SQ_BRA(2, 1) GINT_SQ_BRA(2, 2) GINT_SQ_BRA(2, 3)
      GINT_SQ_BRA(3, 0) GINT_SQ_BRA(3, 1) GINT_SQ_BRA(3, 2) GINT_SQ_BRA(3, 3)
#undef GINT_SQ_BRA
   }
}

// Wavefronts per SIMD: three of the s, p, d kernels (two: 52 ms, four: 51.6
// for 45.5, spills), two of the f kernels (k_sq<3> 25.3 -> 23.8 ms from three,
// k_sq<4> 20.1 -> 16.5 from one)
template <int LM>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(LM >= 3 ? 2 : 3)))
void k_sq(const BatchDev *__restrict__ batches, const SqRef *__restrict__ refs, int nref, uint32_t item0, DevTables t,
          RunDev run, KTargets kt)
{
   extern __shared__ __align__(16) double lds[];
   const int lane = threadIdx.x;
   // the item's chunk: the first whose items end beyond it
   uint32_t item = item0 + xcd_run<LM == 4 ? 16 : 64>(blockIdx.x, gridDim.x);
   const uint32_t end = lane < nref ? refs[lane].end : 0xffffffffu;
   const int ri = __builtin_amdgcn_readfirstlane(__popcll(__ballot(end <= item)));
   if (ri > 0) item -= load_uniform(&refs[ri - 1].end);
   SqArgs y = load_uniform(&refs[ri].y);
   y.tiles = in_global(y.tiles);
   y.sps = in_global(y.sps);
   y.rows = in_global(y.rows);
   y.rcs = in_global(y.rcs);
   y.fns = in_global(y.fns);
   y.cons = in_global(y.cons);
   const BatchDev b = load_batch(batches, load_uniform(&refs[ri].batch), run);
   const TypePlan &tp = *b.tp;
   const int ncpt = load_uniform(&tp.ncp), nkc = load_uniform(&tp.nkc);
   const uint32_t nfix = min(in_global(run.fix)[b.id], b.fix_cap);
   char *tab = (char *)lds;
   uint16_t *tcol = (uint16_t *)tab;
   uint32_t *urb = (uint32_t *)(tab + SQ_TAB_URB), *urk = (uint32_t *)(tab + SQ_TAB_URK);
   uint32_t *tfn = (uint32_t *)(tab + SQ_TAB_FN);
   double *co = lds + y.o_co;   // the set quartet's coefficients, contraction by contraction
   const int m16 = lane & 15, k4 = lane >> 4;
   {
      SqSeg seg{b.g0 + item / (uint32_t)y.nitem, 0, 1};
      if (b.segs) seg = load_uniform(b.segs + item / (uint32_t)y.nitem);
      if (kt.out) {   // integrals of a row are written by one wavefront after the other's
         if (seg.part) return;
         seg.parts = 1;
      }
      const uint32_t gi = seg.group;
      const SqItem it = load_uniform(y.items + item % (uint32_t)y.nitem);
      const SqTile bt = load_uniform(y.tiles + it.bt), ktl = load_uniform(y.tiles + it.kt);
      const SqSp *bsp = y.sps + bt.sp, *ksp = y.sps + ktl.sp;
      const GroupRec &g = b.groups[gi];
      const int nfn = ktl.nfn, ncol = ktl.nrow, cs = ncol | 1;
      double *C = lds + it.o_c;
      lds_order();
      const GroupHead gh = load_uniform((const GroupHead *)&g);
      const bool eco = it.eco_off >= 0;   // contracted by k_eco: the parts take whole rows in turn
      if (eco && seg.part >= gh.row1 - gh.row0) return;
      const uint32_t np4 = load_uniform(&g.np4);
      // Tables of the ket tile, the units' coefficients, the set quartet's P
      // blocks: what does not depend on another load first and together, since
      // an item waited for its set-up longer than it took for most rows (28 k
      // cycles; the coefficients alone were a load after another per shell).
      const int npa = (np4 & 15) + 1, npb = ((np4 >> 4) & 15) + 1, npc = ((np4 >> 8) & 15) + 1, npd = ((np4 >> 12) & 15) + 1;
      const int n0 = y.ncon[0], n1 = n0 + y.ncon[1], n2 = n1 + y.ncon[2];
      // first coefficient of the sets: contraction after contraction
      const int ob = y.ncon[0] * npa, oc = ob + y.ncon[1] * npb, od = oc + y.ncon[2] * npc, oe = od + y.ncon[3] * npd;
      const bool uket = lane >= SQ_MAXRC;   // unit of the lane
      const int un0 = uket ? lane - SQ_MAXRC : lane;
      const bool uok = lane < 2 * SQ_MAXRC && un0 < (uket ? (int)ktl.nrc : (int)bt.nrc);
      const uint16_t vcol = lane < ncol ? y.rows[ktl.row + lane] : (uint16_t)0;
      const uint32_t vfn = lane < nfn ? y.fns[ktl.fn + lane] : 0u;
      const uint32_t vrc = uok ? y.rcs[2 * ((uket ? +ktl.rc : +bt.rc) + un0)] : 0u;
      // the units of the lane's matrix-core results (4 r + lane / 16): first
      // row less first component, and the components they have
      uint32_t vunit[4];
#pragma unroll
      for (int r = 0; r < 4; r++) vunit[r] = 4 * r + k4 < bt.nrc ? y.rcs[2 * (bt.rc + 4 * r + k4) + 1] : 0u;
      const CoefMap cm{y.cons, &g.Kof[0][0], n0, n1, n2, ob, oc, od, npa, npb, npc, npd};
      uint32_t cat[2];
#pragma unroll
      for (int z = 0; z < 2; z++) cat[z] = lane + 64 * z < oe ? coef_at(cm, lane + 64 * z) : 0u;
      double cv[2];
#pragma unroll
      for (int z = 0; z < 2; z++) cv[z] = lane + 64 * z < oe ? b.data[cat[z]] : 0.0;
      const bool setlevel = (load_uniform(&g.ksmode) & KS_SETLEVEL) != 0;
      Upd u{b, kt, tp, g, ksp, lds + it.o_pk, nullptr, tfn, it.lds_k && setlevel, false, bt.n1, bt.n2, ktl.n1, ktl.n2};
      const int nblk = (u.NA + u.NB) * (u.NC + u.ND);
      u.Kl = u.Pl + kt.nspin * nblk;
      double fac = 0.0;
      // where element e of the item's four blocks lies in P and K
      KsSet kss{};
      if (setlevel) {
         kss = load_uniform(b.kss + load_uniform(&g.ks));
         fac = -symm_fac((kss.flags >> 4) & 7) * kt.hf_fac;
         if (fac == 0.0) return;
      }
      const int oad = u.NA * u.NC, obc = oad + u.NA * u.ND, obd = obc + u.NB * u.NC;
      const BlockMap bm{kss, u.NC, u.ND, oad, obc, obd, bt.r1, bt.r2, ktl.r1, ktl.r2};
      double pv[2][2];
#pragma unroll
      for (int z = 0; z < 2; z++) {
         pv[z][0] = pv[z][1] = 0.0;
         if (u.lds && lane + 64 * z < nblk) {
            const size_t o = block_at(bm, lane + 64 * z);
            pv[z][0] = kt.P[0][o];
            if (kt.nspin > 1) pv[z][1] = kt.P[1][o];
         }
      }
      if (lane < ncol) tcol[lane] = vcol;
      for (int i = lane + 64; i < ncol; i += 64) tcol[i] = y.rows[ktl.row + i];
      if (lane < nfn) tfn[lane] = vfn;
      if (uok)
         (uket ? urk : urb)[un0] = (uint32_t)((uket ? oc : 0) + (int)(vrc & 255) * (uket ? npc : npa)) |
                                   (uint32_t)((uket ? od : ob) + (int)(vrc >> 8) * (uket ? npd : npb)) << 16;
      int urow[4];
      unsigned ulo[4], un_[4];
#pragma unroll
      for (int r = 0; r < 4; r++) {
         ulo[r] = (vunit[r] >> 8) & 255;
         un_[r] = (vunit[r] >> 16) - ulo[r];
         urow[r] = (int)(vunit[r] & 255) - (int)ulo[r];
      }
#pragma unroll
      for (int z = 0; z < 2; z++)
         if (lane + 64 * z < oe) co[lane + 64 * z] = cv[z];
      for (int i = lane + 128; i < oe; i += 64) co[i] = b.data[coef_at(cm, i)];
      if (u.lds) {
         for (int sp = 0; sp < kt.nspin; sp++)
            for (int e = lane; e < nblk; e += 64) u.Kl[sp * nblk + e] = 0.0;
#pragma unroll
         for (int z = 0; z < 2; z++)
            if (lane + 64 * z < nblk) {
               u.Pl[lane + 64 * z] = pv[z][0];
               if (kt.nspin > 1) u.Pl[nblk + lane + 64 * z] = pv[z][1];
            }
         for (int e = lane + 128; e < nblk; e += 64) {
            const size_t o = block_at(bm, e);
            u.Pl[e] = kt.P[0][o];
            if (kt.nspin > 1) u.Pl[nblk + e] = kt.P[1][o];
         }
      }
      lds_order();
      auto wbra = [&](int un, uint32_t ip) { return co[(urb[un] & 0xffff) + (ip & 15)] * co[(urb[un] >> 16) + ((ip >> 4) & 15)]; };
      auto wket = [&](int un, uint32_t ip) {
         return co[(urk[un] & 0xffff) + ((ip >> 8) & 15)] * co[(urk[un] >> 16) + ((ip >> 12) & 15)];
      };
      // minimum images of B and D
      const Vec3 Ra = load_uniform((const Vec3 *)(b.data + gh.R[0])), Rb = load_uniform((const Vec3 *)(b.data + gh.R[1])),
                 Rc = load_uniform((const Vec3 *)(b.data + gh.R[2])), Rd = load_uniform((const Vec3 *)(b.data + gh.R[3]));
      double ABs[3], CDs[3];
      {
         const Cell cell = load_uniform((const Cell *)t.cell);
         gint_pbc(Ra.v, Rb.v, cell.v, ABs);
         gint_pbc(Rc.v, Rd.v, cell.v, CDs);
      }
      // at most 8 units: matrix-core tiles of 4 rows, 16 cycles each where one
      // of 16 rows takes 64; the same lanes hold the same elements of theirs
      // and of rows 0 to 3 of that.  39.4 -> 33.7 ms for 32 waters, 72.0 ->
      // 56.9 with s to f shells; for at most 4 units only 34.2 and 57.5
      const bool few = bt.nrc <= 8;
      int ahead = seg.part;   // windows to the next one of the item's part
      const int parts = seg.parts;
      for (uint32_t r = gh.row0; r < gh.row1; r++) {
         const RowRec row = load_uniform(b.rows + r);
         const int nwin = ((int)row.n_prm + SQ_NW - 1) / SQ_NW, win = eco ? 0 : ahead;   // the first one in this row
         if (eco) {
            if (parts > 1 && (r - gh.row0) % (uint32_t)parts != seg.part) continue;
         } else if (parts > 1) {
            if (win >= nwin) {
               ahead -= nwin;
               continue;
            }
            ahead = win + fdiv(nwin - win + parts - 1, parts) * parts - nwin;
         }
         double AB[3], CD[3];
         {
            const Vec3 g1 = load_uniform((const Vec3 *)(t.neighs + 3 * (row.n12 & 0xffff))),
                       g2 = load_uniform((const Vec3 *)(t.neighs + 3 * (row.n12 >> 16)));
#pragma unroll
            for (int x = 0; x < 3; x++) {
               const double Bx = Ra.v[x] + ABs[x] + g1.v[x];
               const double Dx = Rc.v[x] + CDs[x] + g2.v[x];
               AB[x] = Ra.v[x] - Bx;
               CD[x] = Rc.v[x] - Dx;
            }
         }
         lds_order();
         if (eco) {
            // contracted on the matrix cores by k_eco: the units of the tile
            // are part of one class's contractions
            const SqSp qb = load_uniform(bsp), qk = load_uniform(ksp);
            const int nbra = bt.ncomp, nket = fdiv(ncol, qk.nc), ncp = nbra * nket;
            const int nck = tp.nl[2][qk.s1] * tp.nl[3][qk.s2];
            const double *E0 = b.eco + (size_t)(r - b.r0) * b.eco_row + it.eco_off;
            for (int cu = 0; cu < qb.nc; cu++) {
               const double *E = E0 + ((size_t)(qb.c0 + cu) * nck + qk.c0) * ncp;
               for (int i = lane; i < qk.nc * ncp; i += 64) {
                  const int c = fdiv(i, ncp), j = i - c * ncp, e = fdiv(j, nket);
                  C[(cu * nbra + e) * cs + c * nket + (j - e * nket)] = E[i];
               }
            }
         } else {
            const uint32_t *IP = b.prm_ip + row.prm_off;
            const double *A0 = b.ac0 + (size_t)(row.prm_off - b.p0) * ncpt + (size_t)bt.comp0 * nkc + ktl.comp0;
            // the lane's primitive quartet of each step of a window (past its
            // end: the last one, with weight 0)
            uint32_t ipn[4];
            auto exponents = [&](int w0) __attribute__((always_inline)) {
#pragma unroll
               for (int z = 0; z < 4; z++) ipn[z] = IP[min(w0 + 4 * z + k4, (int)row.n_prm - 1)];
            };
            const int wfirst = win * SQ_NW, wstep = parts * SQ_NW;
            exponents(wfirst);
            for (int w0 = wfirst; w0 < (int)row.n_prm; w0 += wstep) {
               const int nw = min(SQ_NW, (int)row.n_prm - w0);
               double wb[4], wb1[4];   // weights of the lane's bra unit; of its second one (few units)
               uint32_t ip[4];
               int no[4];
               {
                  auto weights = [&](double (&w)[4], int un) {
                     const uint32_t ub = urb[min(un, bt.nrc - 1)];
#pragma unroll
                     for (int z = 0; z < 4; z++) {
                        const double v = co[(ub & 0xffff) + (ip[z] & 15)] * co[(ub >> 16) + ((ip[z] >> 4) & 15)];
                        w[z] = (4 * z + k4 < nw && un < bt.nrc) ? v : 0.0;
                     }
                  };
#pragma unroll
                  for (int z = 0; z < 4; z++) {
                     ip[z] = ipn[z];
                     no[z] = min(4 * z + k4, nw - 1);
                  }
                  weights(wb, few ? lane & 3 : m16);
                  if (few && bt.nrc > 4) weights(wb1, 4 + (lane & 3));
               }
               if (w0 + wstep < (int)row.n_prm) exponents(w0 + wstep);
               const double *Aw = A0 + (size_t)w0 * ncpt;
               // 16 columns of a component at a time, SQ_EU components in a
               // step; the loads of a step are in flight during the one before
               auto tiles = [&](auto NZ, auto FEW) {
                  constexpr int nz = decltype(NZ)::value;
                  double a[SQ_EU][nz], an[SQ_EU][nz];
                  auto load = [&](double (&x)[SQ_EU][nz], int c0, int e0) {
                     const uint32_t f = (uint32_t)(tcol[min(c0 + m16, ncol - 1)] & 255);
#pragma unroll
                     for (int v = 0; v < SQ_EU; v++) {
                        const char *p = (const char *)(Aw + min(e0 + v, (int)bt.ncomp - 1) * nkc);
#pragma unroll
                        for (int z = 0; z < nz; z++) x[v][z] = *(const double *)(p + 8 * ((uint32_t)(no[z] * ncpt) + f));
                     }
                  };
                  load(a, 0, 0);
                  for (int c0 = 0; c0 < ncol; c0 += 16) {
                     const bool okc = c0 + m16 < ncol;
                     const uint32_t uk = urk[tcol[min(c0 + m16, ncol - 1)] >> 8];
                     double wc[nz];
#pragma unroll
                     for (int z = 0; z < nz; z++)
                        wc[z] = co[(uk & 0xffff) + ((ip[z] >> 8) & 15)] * co[(uk >> 16) + ((ip[z] >> 12) & 15)];
                     for (int e0 = 0; e0 < bt.ncomp; e0 += SQ_EU) {
                        const bool lastc = e0 + SQ_EU >= bt.ncomp;
                        if (!lastc || c0 + 16 < ncol) load(an, lastc ? c0 + 16 : c0, lastc ? 0 : e0 + SQ_EU);
                        // (past the last component: computed, not stored)
                        auto store = [&](int q, auto &&value) {
                           double *c = C + (urow[q] + e0) * cs + c0 + m16;
                           const unsigned n = okc ? un_[q] : 0u;
#pragma unroll
                           for (int v = 0; v < SQ_EU; v++)
                              if ((unsigned)(e0 + v) - ulo[q] < n) c[v * cs] = w0 != wfirst ? c[v * cs] + value(v) : value(v);
                        };
#pragma unroll
                        for (int v = 0; v < SQ_EU; v++)
#pragma unroll
                           for (int z = 0; z < nz; z++) a[v][z] *= wc[z];
                        if constexpr (decltype(FEW)::value) {
                           double acc[SQ_EU];
#pragma unroll
                           for (int v = 0; v < SQ_EU; v++) acc[v] = 0.0;
#pragma unroll
                           for (int z = 0; z < nz; z++)
#pragma unroll
                              for (int v = 0; v < SQ_EU; v++)
                                 acc[v] = __builtin_amdgcn_mfma_f64_4x4x4f64(wb[z], a[v][z], acc[v], 0, 0, 0);
                           store(0, [&](int v) { return acc[v]; });
                           if (bt.nrc > 4) {
#pragma unroll
                              for (int v = 0; v < SQ_EU; v++) acc[v] = 0.0;
#pragma unroll
                              for (int z = 0; z < nz; z++)
#pragma unroll
                                 for (int v = 0; v < SQ_EU; v++)
                                    acc[v] = __builtin_amdgcn_mfma_f64_4x4x4f64(wb1[z], a[v][z], acc[v], 0, 0, 0);
                              store(1, [&](int v) { return acc[v]; });
                           }
                        } else {
                           dbl4 acc[SQ_EU];
#pragma unroll
                           for (int v = 0; v < SQ_EU; v++) acc[v] = dbl4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
                           for (int z = 0; z < nz; z++)
#pragma unroll
                              for (int v = 0; v < SQ_EU; v++)
                                 acc[v] = __builtin_amdgcn_mfma_f64_16x16x4f64(wb[z], a[v][z], acc[v], 0, 0, 0);
#pragma unroll
                           for (int q = 0; q < 4; q++) {
                              if (4 * q >= bt.nrc) break;
                              store(q, [&](int v) { return acc[v][q]; });
                           }
                        }
#pragma unroll
                        for (int v = 0; v < SQ_EU; v++)
#pragma unroll
                           for (int z = 0; z < nz; z++) a[v][z] = an[v][z];
                     }
                  }
               };
               auto windows = [&](auto FEW) {
                  if (nw > 12) tiles(std::integral_constant<int, 4>{}, FEW);
                  else if (nw > 8) tiles(std::integral_constant<int, 3>{}, FEW);
                  else if (nw > 4) tiles(std::integral_constant<int, 2>{}, FEW);
                  else tiles(std::integral_constant<int, 1>{}, FEW);
               };
               if (few) windows(std::true_type{});
               else windows(std::false_type{});
            }
         }
         // slots of this row whose screening depends on the class
         for (uint32_t e = 0; e < nfix && win == 0; e++) {
            // (where its list begins is read again: kept, it costs registers that the rows need)
            const uint32_t *fe = in_global(run.fix) + FIX_HEAD + FIX_WORDS * (load_uniform(&batches[b.id].fix_at) + e);
            const uint32_t p = fe[0], word = fe[1];
            if (p == FIX_VOID || b.prm_row[p] != r) continue;
            lds_order();
            const uint32_t mask = (word >> 8) & 0xffff, ip = b.prm_ip[p];
            const double *src = in_global(run.fix_ws) + fe[2];
            const double *A = src + (size_t)bt.comp0 * nkc + ktl.comp0;
            for (int qb = 0; qb < bt.nsp; qb++)
               for (int qk = 0; qk < ktl.nsp; qk++) {
                  const SqSp sb = load_uniform(bsp + qb), sk = load_uniform(ksp + qk);
                  const int k = ((sb.s1 * tp.nsh[1] + sb.s2) * tp.nsh[2] + sk.s1) * tp.nsh[3] + sk.s2;
                  const int gate = tp.cls_gate[k];
                  const bool keep = (mask >> gate) & 1u;
                  if (!keep && (sb.l1 || sk.l1)) continue;
                  const int nr = sb.nc * (co_below(sb.l1 + sb.l2 + 1) - co_below(sb.l1));
                  const int nc = sk.nc * (co_below(sk.l1 + sk.l2 + 1) - co_below(sk.l1));
                  for (int i = lane; i < nr * nc; i += 64) {
                     const int rr = fdiv(i, nc), cl = sk.row0 + i - rr * nc;
                     const uint32_t tr = y.rows[bt.row + sb.row0 + rr], tc = tcol[cl];
                     // a screened slot keeps its Fm[0] in (00|00) (reference src/compute_VRR.cpp:384-385)
                     const double v = keep ? A[(tr & 255) * nkc + (tc & 255)]
                                           : ((tr & 255) + (tc & 255) + bt.comp0 + ktl.comp0 == 0 ? src[ncpt + gate] : 0.0);
                     C[(sb.row0 + rr) * cs + cl] += v * wbra(tr >> 8, ip) * wket(tc >> 8, ip);
                  }
               }
         }
         lds_order();
         for (int q = 0; q < ktl.nsp; q++) {
            const SqSp qk = load_uniform(ksp + q);
            if (qk.l1 + qk.l2 > 0 || qk.row0 != qk.fn0) ket_transform<LM>(C, cs, bt.nrow, qk, CD, lane);
         }
         lds_order();
         for (int q = 0; q < bt.nsp; q++) {
            const SqSp qb = load_uniform(bsp + q);
            bra_transform<LM>(C, cs, nfn, qb, AB, u, lane);
            if (u.lds) continue;
            lds_order();
            const int nbra = co_below(qb.l1 + qb.l2 + 1) - co_below(qb.l1);
            for (int i = lane; i < qb.nc * nfn; i += 64) {
               const int c = fdiv(i, nfn), f = i - c * nfn;
               k_update_class(C + (qb.row0 + c * nbra) * cs + f, cs, u, qb, qb.c0 + c, f);
            }
         }
         u.add = true;
      }
      lds_order();
      if (u.lds)
         for (int e = lane; e < nblk; e += 64) {
            const size_t o = block_at(bm, e);
            for (int sp = 0; sp < kt.nspin; sp++) {
               const double v = u.Kl[sp * nblk + e];
               if (v != 0.0) unsafeAtomicAdd(&(sp ? kt.K[1] : kt.K[0])[o], fac * v);
            }
         }
   }
}

}  // namespace sq

template <int LM>
int launch_sq_lm(const BatchDev *batches, const SqRef *refs, int nref, uint32_t item0, unsigned grid, size_t lds,
                 const DevTables &t, const RunDev &run, const KTargets &kt, void *stream);

}  // namespace gint
