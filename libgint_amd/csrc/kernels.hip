// gfx950 kernels of the K-build.  A launch covers one chunk of one quartet
// type (the shell structure of the four sets of a set quartet).
//
//   k_fm_r         one wavefront per primitive quartet (two when the cells
//                  fit half the lanes).  Lanes evaluate
//                  G_m(R,T) (or F_m) of 64 lattice cells at once and decide
//                  Fm[0] > 1e-12 for every class L of the type; surviving
//                  cells run the McMurchie-Davidson Hermite recursion
//                  R^(n)_tuv in LDS and the n = 0 layer is summed over cells
//                  in registers.  One Hermite -> cartesian transform per
//                  primitive quartet then gives the cell-summed (e0|f0)
//                  blocks of every class of the type.  Replaces, for all
//                  classes at once, reference src/compute_Fm.cpp (prepare,
//                  Fm, Vm), src/compute_VRR.cpp and the cell sum of
//                  src/compute_ECO.cpp:216-272.
//   k_fm_r<true,.> slots whose screening differs between the classes of the
//                  type (Fm[0] within rounding of 1e-12 at different L): the
//                  slot's blocks alone, added by the consumers to the classes
//                  that keep it.
//
// kernels_sq.hpp takes the blocks from there to K.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>

#include "device.hpp"
#include "gint_math.h"
#include "uniform.hpp"

namespace gint {

// ---------------------------------------------------------------------------
// cartesian and Hermite index tables, built at compile time
// ---------------------------------------------------------------------------
constexpr int NSHELL = 13;  // shells 0..12

struct CartTables {
   unsigned char comp[NSHELL][91][3];  // lx ly lz of component i of shell L
   unsigned char first[NSHELL][91];    // first non-zero direction
   signed char minus[NSHELL][91][3];   // index of i - 1_d in shell L-1, -1 if none
   signed char plus[7][28][3];         // index of i + 1_d in shell L+1
};

constexpr int cart_index(int L, int lx, int lz) { return (L - lx) * (L - lx + 1) / 2 + lz; }

constexpr CartTables make_cart_tables()
{
   CartTables t{};
   for (int L = 0; L < NSHELL; L++) {
      int i = 0;
      for (int lx = L; lx >= 0; lx--)
         for (int ly = L - lx; ly >= 0; ly--) {
            int lz = L - lx - ly;
            int v[3] = {lx, ly, lz};
            for (int d = 0; d < 3; d++) t.comp[L][i][d] = (unsigned char)v[d];
            t.first[L][i] = (unsigned char)(lx > 0 ? 0 : (ly > 0 ? 1 : 2));
            for (int d = 0; d < 3; d++) {
               if (v[d] > 0) {
                  int w[3] = {v[0], v[1], v[2]};
                  w[d]--;
                  t.minus[L][i][d] = (signed char)cart_index(L - 1, w[0], w[2]);
               } else {
                  t.minus[L][i][d] = -1;
               }
               if (L < 7) {
                  int u[3] = {v[0], v[1], v[2]};
                  u[d]++;
                  t.plus[L][i][d] = (signed char)cart_index(L + 1, u[0], u[2]);
               }
            }
            i++;
         }
   }
   return t;
}

// Hermite triples (t,u,v), ordered by N = t+u+v, then like the cartesian
// components of shell N; the first nherm(K) entries are those with N <= K.
struct HermEntry {
   short m1, m2;          // index of tuv - 1_dir and tuv - 2_dir (-1 if none)
   unsigned char dir;     // recursion direction: first non-zero of t, u, v
   unsigned char coef;    // component along dir, minus one
   unsigned char N, pad;
};
struct HermTables {
   HermEntry e[MAXHERM];
   unsigned char tuv[MAXHERM][3];
   short idx[NSHELL][NSHELL][NSHELL];
};

constexpr HermTables make_herm_tables()
{
   HermTables h{};
   int n = 0;
   for (int N = 0; N < NSHELL; N++)
      for (int t = N; t >= 0; t--)
         for (int u = N - t; u >= 0; u--) {
            const int v = N - t - u;
            h.tuv[n][0] = (unsigned char)t;
            h.tuv[n][1] = (unsigned char)u;
            h.tuv[n][2] = (unsigned char)v;
            h.idx[t][u][v] = (short)n;
            n++;
         }
   for (int i = 0; i < n; i++) {
      const int t = h.tuv[i][0], u = h.tuv[i][1], v = h.tuv[i][2];
      HermEntry e{};
      e.N = (unsigned char)(t + u + v);
      e.m1 = e.m2 = -1;
      if (t + u + v > 0) {
         const int d = t > 0 ? 0 : (u > 0 ? 1 : 2);
         int w[3] = {t, u, v};
         const int c = w[d];
         e.dir = (unsigned char)d;
         e.coef = (unsigned char)(c - 1);
         w[d]--;
         e.m1 = h.idx[w[0]][w[1]][w[2]];
         if (c >= 2) {
            w[d]--;
            e.m2 = h.idx[w[0]][w[1]][w[2]];
         }
      }
      h.e[i] = e;
   }
   return h;
}

__constant__ CartTables c_cart = make_cart_tables();
__constant__ HermTables c_herm = make_herm_tables();
__device__ __forceinline__ int d_nco(int l) { return (l + 1) * (l + 2) / 2; }
__device__ __forceinline__ int d_nherm(int L) { return (L + 1) * (L + 2) * (L + 3) / 6; }

// ---------------------------------------------------------------------------
// per-primitive quantities, in the order of reference
// src/compute_Fm.cpp:66-159 and 202-210, 281-290 (no contraction: these
// feed the Fm[0] > 1e-12 decision)
// ---------------------------------------------------------------------------
struct PrimGeo {
   double P[3], Q[3], PA[3], QC[3];
   double Kfac, zab, zcd, rho, Rr;
   double i2ab, i2cd;
};

__device__ void prim_prepare(const double *Ao, const double *Bo, const double *Co, const double *Do,
                             double za, double zb, double zc, double zd, int n1, int n2,
                             const DevTables &t, PrimGeo &g)
{
   GINT_NO_CONTRACT
   const double *neighs = t.neighs;
   const double zab = za + zb;
   const double inv_zab = 1. / zab;
   const double zcd = zc + zd;
   const double inv_zcd = 1. / zcd;
   const double z = zab + zcd;
   const double inv_z = 1. / z;
   double A[3], B[3], C[3], D[3], bimg[3], dimg[3], qimg[3], kshift[3], Cn[3], Dn[3], P[3], Q[3];
   gint_pbc(Ao, Bo, t.cell, bimg);
   A[0] = Ao[0]; A[1] = Ao[1]; A[2] = Ao[2];
   B[0] = Ao[0] + bimg[0] + neighs[n1 * 3 + 0];
   B[1] = Ao[1] + bimg[1] + neighs[n1 * 3 + 1];
   B[2] = Ao[2] + bimg[2] + neighs[n1 * 3 + 2];
   P[0] = (za * A[0] + zb * B[0]) * inv_zab;
   P[1] = (za * A[1] + zb * B[1]) * inv_zab;
   P[2] = (za * A[2] + zb * B[2]) * inv_zab;
   gint_pbc(Co, Do, t.cell, dimg);
   C[0] = Co[0]; C[1] = Co[1]; C[2] = Co[2];
   D[0] = Co[0] + dimg[0] + neighs[n2 * 3 + 0];
   D[1] = Co[1] + dimg[1] + neighs[n2 * 3 + 1];
   D[2] = Co[2] + dimg[2] + neighs[n2 * 3 + 2];
   Q[0] = (zc * C[0] + zd * D[0]) * inv_zcd;
   Q[1] = (zc * C[1] + zd * D[1]) * inv_zcd;
   Q[2] = (zc * C[2] + zd * D[2]) * inv_zcd;
   gint_pbc(Q, P, t.cell, qimg);
   kshift[0] = P[0] - Q[0] - qimg[0];
   kshift[1] = P[1] - Q[1] - qimg[1];
   kshift[2] = P[2] - Q[2] - qimg[2];
   const double pref = GINT_TWO_PI_52 * inv_zab * inv_zcd;
   double dx = A[0] - B[0], dy = A[1] - B[1], dz = A[2] - B[2];
   const double ab2 = dx * dx + dy * dy + dz * dz;
   const double eab = -(za * zb) / (za + zb) * ab2;
   dx = C[0] - D[0]; dy = C[1] - D[1]; dz = C[2] - D[2];
   const double cd2 = dx * dx + dy * dy + dz * dz;
   const double ecd = -(zc * zd) / (zc + zd) * cd2;
   const double rsz = 1. / sqrt(z);
   g.Kfac = rsz * pref * gint_exp(eab + ecd);
   Cn[0] = Co[0] + kshift[0];
   Cn[1] = Co[1] + kshift[1];
   Cn[2] = Co[2] + kshift[2];
   Dn[0] = Co[0] + dimg[0] + neighs[n2 * 3 + 0] + kshift[0];
   Dn[1] = Co[1] + dimg[1] + neighs[n2 * 3 + 1] + kshift[1];
   Dn[2] = Co[2] + dimg[2] + neighs[n2 * 3 + 2] + kshift[2];
   Q[0] = (zc * Cn[0] + zd * Dn[0]) * inv_zcd;
   Q[1] = (zc * Cn[1] + zd * Dn[1]) * inv_zcd;
   Q[2] = (zc * Cn[2] + zd * Dn[2]) * inv_zcd;
   for (int k = 0; k < 3; k++) {
      g.P[k] = P[k];
      g.Q[k] = Q[k];
      g.PA[k] = P[k] - A[k];
      g.QC[k] = Q[k] - Cn[k];
   }
   g.zab = zab;
   g.zcd = zcd;
   g.rho = zab * zcd * inv_z;
   g.Rr = t.R_cut * sqrt(g.rho);
   g.i2ab = 0.5 * inv_zab;
   g.i2cd = 0.5 * inv_zcd;
}

// order-independent survivor checksum, same function as the oracle's
__device__ __forceinline__ unsigned long long mix64(unsigned long long z)
{
   z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ULL;
   z = (z ^ (z >> 27)) * 0x94d049bb133111ebULL;
   return z ^ (z >> 31);
}

__device__ __forceinline__ unsigned long long slot_hash(uint32_t set_ij, uint32_t set_kl, int n1, int n2, uint32_t ip,
                                                        int n3)
{
   const unsigned long long w0 = ((unsigned long long)(set_ij & 0xffff) << 32) | (set_ij >> 16);
   const unsigned long long w1 = ((unsigned long long)(set_kl & 0xffff) << 32) | (set_kl >> 16);
   const unsigned long long w2 = ((unsigned long long)n1 << 24) | ((unsigned long long)n2 << 16);
   const unsigned long long pk = ((ip & 15) << 12) | (((ip >> 4) & 15) << 8) | (((ip >> 8) & 15) << 4) | ((ip >> 12) & 15);
   const unsigned long long w3 = (pk << 8) | (unsigned long long)n3;
   unsigned long long z = mix64(w0 + 0x9E3779B97F4A7C15ULL);
   z = mix64(z ^ w1);
   z = mix64(z ^ w2);
   z = mix64(z ^ w3);
   return z;
}

// sum_j T2_j sum_{l<14-j} T1_l c[jl]: the operations of gint_cheb_sum in the
// same order (so the value is bitwise the host's), with T2_j produced by
// the recurrence of gint_cheb14 inside the loop to keep few values live
__device__ __forceinline__ double d_cheb_sum(const double *__restrict__ c, const double *T1, double x2)
{
   GINT_NO_CONTRACT
   double tmp = 0.0, tm1 = 0.0, tm2 = 0.0;
   int jl = 0;
#pragma unroll 7
   for (int j = 0; j < 14; j++) {
      double t2;
      if (j == 0) t2 = 1.0;
      else if (j == 1) t2 = GINT_SQRT2 * x2;
      else if (j == 2) t2 = 2. * x2 * tm1 - GINT_SQRT2;
      else t2 = 2. * x2 * tm1 - tm2;
      double dot = 0.0;
#pragma unroll
      for (int l = 0; l < 14; l++)
         if (l < 14 - j) dot += T1[l] * c[jl + l];
      tmp += dot * t2;
      jl += 14 - j;
      tm2 = tm1;
      tm1 = t2;
   }
   return tmp;
}

// ---------------------------------------------------------------------------
// K1: G_m -> Hermite R -> cell sum -> (e0|f0), one wavefront per primitive
// quartet.  FIX: one wavefront per listed (primitive, cell) slot, no
// screening, blocks and per-L Fm[0] into the fix-up workspace.
// ---------------------------------------------------------------------------
constexpr int GEO = 24;   // doubles of the primitive geometry at the start of LDS
enum { G_P = 0, G_Q = 3, G_PA = 6, G_QC = 9, G_KFAC = 12, G_RHO = 13, G_RR = 14, G_I2AB = 15, G_I2CD = 16 };

static FmLayout fm_layout(const TypePlan &tp, bool fix, bool pair = false)
{
   FmLayout y;
   const int L = tp.L, nh = tp.nh;
   const int geo = pair ? 2 * GEO : GEO;   // one geometry record per primitive quartet of the wavefront
   y.o_fmv = geo;
   y.o_sv = geo + 64 * (L + 1);
   y.o_R = y.o_sv + 320;
   // the Hermite batch fills what is left of a 10 KB budget: small enough
   // that 4 wavefronts per SIMD fit in LDS
   int SB = fix ? 1 : (1280 - y.o_R) / (2 * nh);
   SB = std::max(1, std::min(16, SB));
   y.SB = SB;
   const int cell_phase = y.o_R + 2 * SB * nh;
   const int e_phase = geo + nh + 6 * 28 + tp.nbh * tp.nkc;
   const int dbl = std::max(cell_phase, e_phase);
   y.o_int = 8 * dbl;
   y.bytes = y.o_int + 4 * 128;
   return y;
}

// at most 128 VGPRs (4 wavefronts per SIMD, with the LDS budget above): the
// kernel waits on memory half of its time, so wavefronts in flight pay more
// than the few values it then keeps in scratch
//
// PAIR (at most 32 cells, at most 256 Hermite functions): two primitive
// quartets per wavefront.  Lanes 0-31 take the cells of the first, lanes
// 32-63 those of the second; their survivors share the G_m and Hermite
// batches and each quartet keeps its own cell sum and transform.
//
// One launch takes the chunks of a list, one after the other in the
// numbering of its units (primitive quartets or pairs of them): a launch per
// type left the chip to the slowest wavefronts of each, and small systems to
// launch after launch of a few workgroups.
template <bool FIX, bool PAIR>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4)))
void k_fm_r(const BatchDev *__restrict__ batches, const WorkRef *__restrict__ refs, int nref, DevTables t, RunDev run)
{
   static_assert(!(FIX && PAIR), "the fix-up takes one slot per wavefront");
   constexpr int NPR = PAIR ? 2 : 1;      // primitive quartets per wavefront
   constexpr int NACC = PAIR ? 4 : 8;     // Hermite functions per lane and quartet, / 64
   extern __shared__ double lds[];
   const int lane = threadIdx.x;
   const int half = PAIR ? lane >> 5 : 0;   // the lane's quartet
   uint32_t ubase = 0;
   const uint32_t nfix = FIX ? min(run.fix_count[0], run.fix_cap) : 0;
   // (the fix-up: one entry per turn, each with its own chunk)
   for (uint32_t turn = FIX ? blockIdx.x : 0; turn < (FIX ? nfix : (uint32_t)nref); turn += FIX ? gridDim.x : 1) {
   const BatchDev b = load_batch(batches, FIX ? (uint32_t)__builtin_amdgcn_readfirstlane((int)(run.fix[2 * turn + 1] >> 24))
                                              : load_uniform(&refs[turn].batch), run);
   const TypePlan &tp = *b.tp;
   const FmLayout lay = FIX ? b.fix_fm : b.fm;
   const int L = load_uniform(&tp.L), nh = load_uniform(&tp.nh), Lp1 = L + 1;
   const int SB = lay.SB;
   double *G = lds + GEO * half;      // geometry of the lane's quartet
   double *fmv = lds + lay.o_fmv;     // [64][L+1]
   double *sv = lds + lay.o_sv;       // [64][5]
   double *Rb = lds + lay.o_R;        // [2][SB][nh]
   int *svi = (int *)((char *)lds + lay.o_int);
   int *svl = svi + 64;
   const uint32_t nwork = FIX ? turn + 1 : b.p1 - b.p0;
   const uint32_t *__restrict__ e1 = b.e1, *__restrict__ e2 = b.e2;
   // the first unit of the chunk that is this workgroup's
   const uint32_t skip = ubase % gridDim.x;
   const uint32_t u0 = FIX ? turn : (blockIdx.x >= skip ? blockIdx.x - skip : blockIdx.x + gridDim.x - skip);
   if (!FIX) ubase = load_uniform(&refs[turn].end);

   for (uint32_t w0 = u0 * NPR; w0 < nwork; w0 += gridDim.x * NPR) {
      const uint32_t w = w0 + half;
      const bool hvalid = w < nwork;                    // the lane's quartet exists
      const int nprim = (int)min((uint32_t)NPR, nwork - w0);
      uint32_t p;
      int fix_n3 = 0;
      if (FIX) {
         p = b.fix[2 * w];
         fix_n3 = (int)(b.fix[2 * w + 1] & 0xff);
      } else {
         p = b.p0 + (hvalid ? w : w0);
      }
      const uint32_t r = b.prm_row[p];
      const RowRec row = b.rows[r];
      const GroupRec &g = b.groups[row.group];
      const uint32_t ip = b.prm_ip[p];
      const int n1 = row.n12 & 0xffff, n2 = row.n12 >> 16;
      if ((lane & (64 / NPR - 1)) == 0 && hvalid) {
         const double *data = b.data;
         PrimGeo geo;
         prim_prepare(data + g.R[0], data + g.R[1], data + g.R[2], data + g.R[3], data[g.Z[0] + (ip & 15)],
                      data[g.Z[1] + ((ip >> 4) & 15)], data[g.Z[2] + ((ip >> 8) & 15)],
                      data[g.Z[3] + ((ip >> 12) & 15)], n1, n2, t, geo);
         for (int k = 0; k < 3; k++) {
            G[G_P + k] = geo.P[k];
            G[G_Q + k] = geo.Q[k];
            G[G_PA + k] = geo.PA[k];
            G[G_QC + k] = geo.QC[k];
         }
         G[G_KFAC] = geo.Kfac;
         G[G_RHO] = geo.rho;
         G[G_RR] = geo.Rr;
         G[G_I2AB] = geo.i2ab;
         G[G_I2CD] = geo.i2cd;
      }
      __syncthreads();
      double acc[NPR][NACC];
#pragma unroll
      for (int q = 0; q < NPR; q++)
#pragma unroll
         for (int i = 0; i < NACC; i++) acc[q][i] = 0.0;
      double quirk = 0.0;
      unsigned long long n_surv = 0, csum = 0, n_any = 0;
      bool any_surv[NPR];
#pragma unroll
      for (int q = 0; q < NPR; q++) any_surv[q] = false;
      const unsigned all = (1u << tp.nL) - 1u;
      const int ncell = FIX ? 1 : t.Ng;

      for (int base = 0; base < ncell; base += 64) {
         const int n3 = FIX ? fix_n3 : base + (PAIR ? (lane & 31) : lane);
         const bool valid = FIX ? (lane == 0) : (hvalid && n3 < t.Ng);
         int status = 0;  // 1 kept by every class, 2 screened by every class, 3 class-dependent
         unsigned mask = 0;
         double *myf = fmv + lane * Lp1;
         if (valid) {
            const double Kfac = G[G_KFAC], rho = G[G_RHO];
            double X[3], T, Fm0 = 0.0, tg1 = 0.0, tg2 = 0.0;
            int br, patch = 0;
            {
               GINT_NO_CONTRACT
               X[0] = G[G_P + 0] - G[G_Q + 0] - t.neighs[n3 * 3 + 0];
               X[1] = G[G_P + 1] - G[G_Q + 1] - t.neighs[n3 * 3 + 1];
               X[2] = G[G_P + 2] - G[G_Q + 2] - t.neighs[n3 * 3 + 2];
               const double rpq2 = X[0] * X[0] + X[1] * X[1] + X[2] * X[2];
               T = rho * rpq2;
            }
            br = t.truncated ? gint_tcg_locate(G[G_RR], T, t.grid_lo, t.grid_hi, t.bw, &patch, &tg1, &tg2) : GINT_G_BOYS;
            if (br == GINT_G_PATCH) {
               double T1[14];
               gint_cheb14(tg1, T1);
               {
                  GINT_NO_CONTRACT
                  Fm0 = d_cheb_sum(t.C0 + (size_t)t.ld_C0 * patch, T1, tg2) * Kfac;
               }
               myf[0] = Fm0;
            } else if (br == GINT_G_BOYS) {
               gint_boys(L, T, myf, t.ftable, Kfac);
               Fm0 = myf[0];
            }
            const bool lsens = br == GINT_G_BOYS && T >= 1.e-13 && T < 12.;   // F_0 depends on the start order
            if (br == GINT_G_ZERO) {
               status = 2;
            } else {
               mask = Fm0 > 1.e-12 ? all : 0u;
               // F_0 of the downward recursion depends on the starting order
               // by rounding only; decide each class L exactly this close to
               // the threshold
               if (lsens && tp.nL > 1 && fabs(Fm0 - 1.e-12) <= 1.e-20) {
                  mask = 0u;
                  for (int i = 0; i < tp.nL; i++) {
                     gint_boys(tp.Ls[i], T, myf, t.ftable, Kfac);
                     if (myf[0] > 1.e-12) mask |= 1u << i;
                  }
                  gint_boys(L, T, myf, t.ftable, Kfac);
               }
               status = mask == all ? 1 : (mask == 0u ? 2 : 3);
            }
            if (FIX) {
               // per-L Fm[0] of the slot, for the classes that screen it
               double *f0 = b.fix_ws + (size_t)w * b.fix_stride + tp.ncp;
               for (int i = 0; i < tp.nL; i++) {
                  double v = Fm0;
                  if (lsens) {
                     gint_boys(tp.Ls[i], T, myf, t.ftable, Kfac);
                     v = myf[0];
                  }
                  f0[i] = v;
               }
               if (lsens) gint_boys(L, T, myf, t.ftable, Kfac);
               status = br == GINT_G_ZERO ? 2 : 1;
            } else if (b.force_fix && status == 1) {
               status = 3;
            }
            if (!FIX) {
               if (status == 2) {
                  if (tp.has00) quirk += Fm0;
               } else {
                  if (b.stats) {
                     const unsigned long long h = slot_hash(g.set_ij, g.set_kl, n1, n2, ip, n3);
                     if (mask == all) {
                        n_surv += (unsigned long long)tp.nclass;
                        csum += h * tp.mult_all;
                     } else {
                        unsigned long long cm = 0;
                        for (int k = 0; k < tp.nclass; k++)
                           if ((mask >> tp.cls_gate[k]) & 1u) {
                              n_surv++;
                              cm += tp.cls_mult[k];
                           }
                        csum += h * cm;
                     }
                  }
                  if (status == 3) {
                     const uint32_t idx = atomicAdd(&b.fix_count[0], 1u);
                     if (idx < b.fix_cap) {
                        b.fix[2 * idx] = p;
                        b.fix[2 * idx + 1] = (uint32_t)n3 | (mask << 8) | (b.id << 24);
                     } else {
                        // list full: every class keeps the slot (its G_0 is
                        // within rounding of the 1e-12 threshold)
                        atomicAdd(&b.fix_count[1], 1u);
                        status = 1;
                        n_any++;
                     }
                  } else {
                     n_any++;
                  }
               }
            }
            if (status == 1) {
               sv[lane * 5 + 0] = X[0];
               sv[lane * 5 + 1] = X[1];
               sv[lane * 5 + 2] = X[2];
               sv[lane * 5 + 3] = br == GINT_G_PATCH ? tg1 : T;
               sv[lane * 5 + 4] = tg2;
               svi[lane] = br | (patch << 2);
            }
         }
         // survivors of this pass, in lane order
         const unsigned long long smask = __ballot(status == 1);
         const int nsv = __popcll(smask);
         const int nsv0 = PAIR ? __popcll(smask & 0xffffffffull) : nsv;   // survivors of the first quartet
         if (status == 1) svl[__popcll(smask & ((1ull << lane) - 1ull))] = lane;
         __syncthreads();
         if (nsv == 0) continue;
         any_surv[0] = any_surv[0] || nsv0 > 0;
         if (PAIR) any_surv[NPR - 1] = any_surv[NPR - 1] || nsv > nsv0;
         // G_1..G_L of the patch survivors, one (survivor, order) per lane
         {
            for (int idx = lane; idx < nsv * L; idx += 64) {
               const int s = idx / L, m = idx - s * L + 1;
               const int ln = svl[s];
               const double Kfac = lds[GEO * (PAIR ? ln >> 5 : 0) + G_KFAC];
               const int info = svi[ln];
               if ((info & 3) == GINT_G_PATCH) {
                  double T1[14];
                  gint_cheb14(sv[ln * 5 + 3], T1);
                  const double *c = t.C0 + (size_t)t.ld_C0 * (info >> 2) + m * TCG_NCOEF;
                  fmv[ln * Lp1 + m] = d_cheb_sum(c, T1, sv[ln * 5 + 4]) * Kfac;
               }
            }
         }
         __syncthreads();
         {
            for (int idx = lane; idx < nsv * Lp1; idx += 64) {
               const int s = idx / Lp1, m = idx - s * Lp1;
               const int ln = svl[s];
               const double m2rho = -2.0 * lds[GEO * (PAIR ? ln >> 5 : 0) + G_RHO];
               double pw = 1.0;
               for (int k = 0; k < m; k++) pw *= m2rho;
               fmv[ln * Lp1 + m] *= pw;
            }
         }
         __syncthreads();
         // Hermite recursion R^(n)_tuv = coef R^(n+1)_{tuv-2d} + X_d R^(n+1)_{tuv-d}
         for (int s0 = 0; s0 < nsv; s0 += SB) {
            const int nb = min(SB, nsv - s0);
            double *prv = Rb, *cur = Rb + SB * nh;
            if (lane < nb) prv[lane * nh] = fmv[svl[s0 + lane] * Lp1 + L];
            __syncthreads();
            for (int n = L - 1; n >= 1; n--) {
               const int mn = d_nherm(L - n);
               for (int h = lane; h < mn; h += 64) {
                  if (h == 0) {
                     for (int s = 0; s < nb; s++) cur[s * nh] = fmv[svl[s0 + s] * Lp1 + n];
                  } else {
                     const HermEntry e = c_herm.e[h];
                     const double cf = (double)e.coef;
                     for (int s = 0; s < nb; s++) {
                        double v = sv[svl[s0 + s] * 5 + e.dir] * prv[s * nh + e.m1];
                        if (e.m2 >= 0) v += cf * prv[s * nh + e.m2];
                        cur[s * nh + h] = v;
                     }
                  }
               }
               __syncthreads();
               double *tmp = prv;
               prv = cur;
               cur = tmp;
            }
            // the n = 0 layer goes straight into the cell sum of its quartet
#pragma unroll
            for (int i = 0; i < NACC; i++) {
               const int h = lane + 64 * i;
               if (h < nh) {
                  double a0 = acc[0][i], a1 = acc[NPR - 1][i];
                  if (h == 0) {
                     for (int s = 0; s < nb; s++) {
                        const double v = fmv[svl[s0 + s] * Lp1];
                        if (!PAIR || s0 + s < nsv0) a0 += v;
                        else a1 += v;
                     }
                  } else {
                     const HermEntry e = c_herm.e[h];
                     const double cf = (double)e.coef;
                     for (int s = 0; s < nb; s++) {
                        double v = sv[svl[s0 + s] * 5 + e.dir] * prv[s * nh + e.m1];
                        if (e.m2 >= 0) v += cf * prv[s * nh + e.m2];
                        if (!PAIR || s0 + s < nsv0) a0 += v;
                        else a1 += v;
                     }
                  }
                  acc[0][i] = a0;
                  if (PAIR) acc[NPR - 1][i] = a1;
               }
            }
            __syncthreads();
         }
      }

      // ---- Hermite -> cartesian, once per primitive quartet ----
      double *sR = lds + lay.o_fmv;      // [nh]
      double *Ex = sR + nh;              // [3][28] bra E^{e0}_t
      double *Fk = Ex + 84;              // [3][28] ket (-1)^tau E^{f0}_tau
      double *W = Fk + 84;               // [nbh][nkc]
      // screened slots' Fm[0], summed per quartet (lane 0, and lane 32 for the second)
      for (int off = 32 / NPR; off > 0; off >>= 1) quirk += __shfl_down(quirk, off, 64 / NPR);
      double qsum[NPR];
#pragma unroll
      for (int q = 0; q < NPR; q++) qsum[q] = __shfl(quirk, 32 * q, 64);
#pragma unroll
      for (int q = 0; q < NPR; q++) {
         if (q >= nprim) break;
         const double *Gq = lds + GEO * q;
         double *dst = FIX ? b.fix_ws + (size_t)w * b.fix_stride : b.ac0 + (size_t)(w0 + q) * tp.ncp;
         // calibration of the mixed-precision routing: the largest block
         // element of each set quartet (a positive double orders as its bits)
         unsigned long long *gm = nullptr;
         if (!FIX && b.gmag) gm = (unsigned long long *)(b.gmag + b.rows[b.prm_row[b.p0 + w0 + q]].group);
         if (!FIX && !any_surv[q]) {
            // no cell survives: the blocks are zero but for the screened
            // slots' Fm[0] in (00|00)
            for (int j = lane; j < tp.ncp; j += 64) dst[j] = (j == 0 && tp.has00) ? qsum[q] : 0.0;
            if (gm && lane == 0 && tp.has00) atomicMax(gm, (unsigned long long)__double_as_longlong(fabs(qsum[q])));
            __syncthreads();
            continue;
         }
         __syncthreads();
#pragma unroll
         for (int i = 0; i < NACC; i++) {
            const int h = lane + 64 * i;
            if (h < nh) sR[h] = acc[q][i];
         }
         if (lane < 6) {
            const int d = lane % 3;
            const bool ket = lane >= 3;
            const int Lm = ket ? tp.LC : tp.LA;
            const double x = ket ? Gq[G_QC + d] : Gq[G_PA + d];
            const double i2 = ket ? Gq[G_I2CD] : Gq[G_I2AB];
            double *E = (ket ? Fk : Ex) + d * 28;
            E[0] = 1.0;
            for (int e = 0; e < Lm; e++) {
               const double *Ee = E + e * (e + 1) / 2;
               double *En = E + (e + 1) * (e + 2) / 2;
               for (int tt = 0; tt <= e + 1; tt++) {
                  double v = 0.0;
                  if (tt > 0) v += i2 * Ee[tt - 1];
                  if (tt <= e) v += x * Ee[tt];
                  if (tt + 1 <= e) v += (double)(tt + 1) * Ee[tt + 1];
                  En[tt] = v;
               }
            }
            if (ket)
               for (int e = 0; e <= Lm; e++)
                  for (int tt = 1; tt <= e; tt += 2) E[e * (e + 1) / 2 + tt] = -E[e * (e + 1) / 2 + tt];
         }
         __syncthreads();
         const int nkc = tp.nkc;
         // W[tuv][f] = sum E^f_tau E^f_nu E^f_phi R[t+tau, u+nu, v+phi]
         for (int idx = lane; idx < tp.nbh * nkc; idx += 64) {
            const uint32_t it = e1[idx];
            const int tt = it & 7, uu = (it >> 3) & 7, vv = (it >> 6) & 7;
            const int fx = (it >> 9) & 7, fy = (it >> 12) & 7, fz = (it >> 15) & 7;
            const double *Fx = Fk + fx * (fx + 1) / 2, *Fy = Fk + 28 + fy * (fy + 1) / 2, *Fz = Fk + 56 + fz * (fz + 1) / 2;
            double s = 0.0;
            for (int a = 0; a <= fx; a++)
               for (int c = 0; c <= fy; c++) {
                  const double cxy = Fx[a] * Fy[c];
                  const int t1 = tt + a, u1 = uu + c;
                  for (int d = 0; d <= fz; d++) {
                     const int v1 = vv + d, N = t1 + u1 + v1;
                     const int H = N * (N + 1) * (N + 2) / 6 + (N - t1) * (N - t1 + 1) / 2 + v1;
                     s += cxy * Fz[d] * sR[H];
                  }
               }
            W[it >> 18] = s;
         }
         __syncthreads();
         // (e0|f0) = sum E^e_t E^e_u E^e_v W[tuv][f]
         double vmax = 0.0;
         for (int j = lane; j < tp.ncp; j += 64) {
            const uint32_t it = e2[j];
            const int ex = it & 7, ey = (it >> 3) & 7, ez = (it >> 6) & 7, col = (int)((it >> 9) & 127);
            const double *Ea = Ex + ex * (ex + 1) / 2, *Eb = Ex + 28 + ey * (ey + 1) / 2, *Ec = Ex + 56 + ez * (ez + 1) / 2;
            double s = 0.0;
            for (int a = 0; a <= ex; a++)
               for (int c = 0; c <= ey; c++) {
                  const double cxy = Ea[a] * Eb[c];
                  for (int d = 0; d <= ez; d++) {
                     const int N = a + c + d;
                     const int H = N * (N + 1) * (N + 2) / 6 + (N - a) * (N - a + 1) / 2 + d;
                     s += cxy * Ec[d] * W[H * nkc + col];
                  }
               }
            const int jd = (int)(it >> 16);
            if (!FIX && jd == 0 && tp.has00) s += qsum[q];
            dst[jd] = s;
            vmax = fmax(vmax, fabs(s));
         }
         if (gm) {
            for (int off = 32; off > 0; off >>= 1) vmax = fmax(vmax, __shfl_xor(vmax, off, 64));
            if (lane == 0) atomicMax(gm, (unsigned long long)__double_as_longlong(vmax));
         }
         __syncthreads();
      }

      if (!FIX && b.stats) {
         for (int off = 32; off > 0; off >>= 1) {
            n_surv += __shfl_down(n_surv, off, 64);
            csum += __shfl_down(csum, off, 64);
            n_any += __shfl_down(n_any, off, 64);
         }
         if (lane == 0) {
            // per-workgroup partials spread over STATS_SLOTS counters: one
            // address hit by every workgroup of the chip serialises them
            unsigned long long *st = b.stats + 3 * (blockIdx.x & (STATS_SLOTS - 1));
            if (n_surv) {
               atomicAdd(&st[0], n_surv);
               atomicAdd(&st[1], csum);
            }
            // algorithmic FLOPs: the reference chain's Fm and VRR of every
            // (slot, class) pair kept (reference src/compute_Fm.cpp,
            // src/compute_VRR.cpp; summed over the type's classes)
            atomicAdd(&st[2], n_any * (unsigned long long)tp.ref_slot_flops);
         }
      }
   }
   __syncthreads();   // the next chunk's layout of LDS
   }
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
static constexpr size_t LDS_LIMIT = 64 * 1024;

size_t fm_r_lds_bytes(const TypePlan &tp)
{
   const FmLayout y = fm_layout(tp, false);
   return (size_t)y.bytes <= LDS_LIMIT ? (size_t)y.bytes : 0;
}

void fm_layouts(const TypePlan &tp, int Ng, FmLayout &main, FmLayout &fix, bool *pair)
{
   // two primitive quartets per wavefront when each takes at most half of
   // the lanes' cells and its cell sum fits 4 values per lane
   const FmLayout yp = fm_layout(tp, false, true);
   *pair = Ng <= 32 && tp.nh <= 256 && (size_t)yp.bytes <= LDS_LIMIT;
   main = *pair ? yp : fm_layout(tp, false);
   fix = fm_layout(tp, true);
}

int launch_fm_r(const BatchDev *batches, const WorkRef *refs, int nref, uint32_t units, bool pair, size_t lds,
                const DevTables &t, const RunDev &run, void *stream)
{
   if (!units) return 0;
   if (lds > LDS_LIMIT) return -3;
   // workgroups stay resident and stride over the units
   const unsigned grid = std::min(units, 16384u);
   if (pair)
      hipLaunchKernelGGL((k_fm_r<false, true>), dim3(grid), dim3(64), lds, (hipStream_t)stream, batches, refs, nref, t, run);
   else
      hipLaunchKernelGGL((k_fm_r<false, false>), dim3(grid), dim3(64), lds, (hipStream_t)stream, batches, refs, nref, t, run);
   return hipGetLastError() == hipSuccess ? 0 : -1;
}

int launch_fixup(const BatchDev *batches, size_t lds, const DevTables &t, const RunDev &run, uint32_t n_fix, void *stream)
{
   if (lds > LDS_LIMIT) return -3;
   const unsigned grid = std::max(1u, std::min(n_fix, 4096u));
   hipLaunchKernelGGL((k_fm_r<true, false>), dim3(grid), dim3(64), lds, (hipStream_t)stream, batches,
                      (const WorkRef *)nullptr, 0, t, run);
   return hipGetLastError() == hipSuccess ? 0 : -1;
}

// ---------------------------------------------------------------------------
// scratch of the no-allocation executor: one array per GPU, held for the
// life of the process.  In host code `scratch` only names the symbol; its
// device address comes from hipGetSymbolAddress, per device.
// ---------------------------------------------------------------------------
static __device__ __align__(256) double scratch[NOALLOC_BYTES / sizeof(double)];

static constexpr int NOALLOC_MAX_DEVICES = 64;
static std::mutex g_scratch_mu;
static void *g_scratch_ptr[NOALLOC_MAX_DEVICES];

void *noalloc_scratch()
{
   int dev = 0;
   if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= NOALLOC_MAX_DEVICES) return nullptr;
   std::lock_guard<std::mutex> lock(g_scratch_mu);
   if (!g_scratch_ptr[dev]) {
      void *ptr = nullptr;
      if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess) return nullptr;
      g_scratch_ptr[dev] = ptr;
   }
   return g_scratch_ptr[dev];
}

__global__ void k_zero_u32(uint32_t *p, int n)
{
   const int i = blockIdx.x * blockDim.x + threadIdx.x;
   if (i < n) p[i] = 0u;
}

// max |P| over n elements into *out (a positive double orders as its bits;
// *out starts at 0)
__global__ void k_absmax(const double *__restrict__ P, size_t n, unsigned long long *out)
{
   double m = 0.0;
   for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
      m = fmax(m, fabs(P[i]));
   for (int off = 32; off > 0; off >>= 1) m = fmax(m, __shfl_xor(m, off, 64));
   if ((threadIdx.x & 63) == 0) atomicMax(out, (unsigned long long)__double_as_longlong(m));
}

// The mixed-precision route of each set quartet of a chunk: single
// precision when its bound  max|block element| x max|coefficient|^4 x
// primitive quartets  times max|P| is below tau.  count[0] += flagged.
__global__ void k_mixed_flags(const BatchDev *__restrict__ batch, RunDev run, const unsigned long long *__restrict__ pmax,
                              double tau, unsigned long long *count)
{
   const double *gmag = load_uniform(&batch->gmag);
   const BatchDev b = load_batch(batch, 0, run);
   const TypePlan &tp = *b.tp;
   const double maxP = __longlong_as_double((long long)*pmax);
   for (uint32_t gi = b.g0 + blockIdx.x * blockDim.x + threadIdx.x; gi < b.g1; gi += gridDim.x * blockDim.x) {
      const GroupRec &g = b.groups[gi];
      double c4 = 1.0;
      for (int t = 0; t < 4; t++) {
         const int np = ((g.np4 >> (4 * t)) & 15) + 1;
         double cm = 0.0;
         for (int sh = 0; sh < tp.nsh[t]; sh++)
            for (int i = 0; i < tp.nl[t][sh] * np; i++) cm = fmax(cm, fabs(b.data[g.Kof[t][sh] + i]));
         c4 *= cm;
      }
      double npr = 0.0;
      for (uint32_t r = g.row0; r < g.row1; r++) npr += (double)b.rows[r].n_prm;
      const bool f32 = gmag[gi] * c4 * npr * maxP < tau;
      b.gflag[gi] = f32 ? 1u : 0u;
      if (f32) atomicAdd(count, 1ull);
   }
}

int launch_absmax(const double *P, size_t n, unsigned long long *out, bool zero, void *stream)
{
   if (zero) hipLaunchKernelGGL(k_zero_u32, dim3(1), dim3(64), 0, (hipStream_t)stream, (uint32_t *)out, 2);
   const unsigned grid = (unsigned)std::min<size_t>((n + 255) / 256, 2048);
   hipLaunchKernelGGL(k_absmax, dim3(std::max(grid, 1u)), dim3(256), 0, (hipStream_t)stream, P, n, out);
   return hipGetLastError() == hipSuccess ? 0 : -1;
}

int launch_mixed_flags(const BatchDev *batch, const RunDev &run, uint32_t ng, const unsigned long long *pmax, double tau,
                       unsigned long long *count, void *stream)
{
   if (!ng) return 0;
   const unsigned grid = std::min<unsigned>((ng + 255) / 256, 4096);
   hipLaunchKernelGGL(k_mixed_flags, dim3(grid), dim3(256), 0, (hipStream_t)stream, batch, run, pmax, tau, count);
   return hipGetLastError() == hipSuccess ? 0 : -1;
}

__global__ void k_zero_f64(double *p, size_t n)
{
   for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = 0.0;
}

void launch_zero_f64(double *p, size_t n, void *stream)
{
   if (!n) return;
   const unsigned grid = (unsigned)std::min<size_t>((n + 255) / 256, 4096);
   hipLaunchKernelGGL(k_zero_f64, dim3(grid), dim3(256), 0, (hipStream_t)stream, p, n);
}

int launch_zero_u32(uint32_t *p, int n, void *stream)
{
   if (n <= 0) return 0;
   hipLaunchKernelGGL(k_zero_u32, dim3((n + 255) / 256), dim3(256), 0, (hipStream_t)stream, p, n);
   return hipGetLastError() == hipSuccess ? 0 : -1;
}

// ---------------------------------------------------------------------------
// self-test of the screening arithmetic (bitwise comparison with the host)
// ---------------------------------------------------------------------------
__global__ void k_math_selftest(const double *x, const double *y, int n, double *out)
{
   GINT_NO_CONTRACT
   const int i = blockIdx.x * blockDim.x + threadIdx.x;
   if (i >= n) return;
   const double a = x[i], c = y[i];
   out[4 * i + 0] = gint_exp(a);
   out[4 * i + 1] = sqrt(fabs(a));
   out[4 * i + 2] = 1. / a;
   out[4 * i + 3] = a * c / (a + c);
}

int device_math_selftest(const double *x, const double *y, int n, double *out)
{
   double *dx = nullptr, *dy = nullptr, *dout = nullptr;
   int rc = 0;
   if (hipMalloc(&dx, sizeof(double) * n) != hipSuccess || hipMalloc(&dy, sizeof(double) * n) != hipSuccess ||
       hipMalloc(&dout, sizeof(double) * 4 * n) != hipSuccess)
      rc = -1;
   if (!rc && (hipMemcpy(dx, x, sizeof(double) * n, hipMemcpyHostToDevice) != hipSuccess ||
               hipMemcpy(dy, y, sizeof(double) * n, hipMemcpyHostToDevice) != hipSuccess))
      rc = -1;
   if (!rc) {
      hipLaunchKernelGGL(k_math_selftest, dim3((n + 255) / 256), dim3(256), 0, 0, dx, dy, n, dout);
      if (hipGetLastError() != hipSuccess) rc = -1;
   }
   if (!rc && hipMemcpy(out, dout, sizeof(double) * 4 * n, hipMemcpyDeviceToHost) != hipSuccess) rc = -1;
   if (dx) (void)hipFree(dx);
   if (dy) (void)hipFree(dy);
   if (dout) (void)hipFree(dout);
   return rc;
}

}  // namespace gint
