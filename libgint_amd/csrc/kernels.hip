// gfx950 kernels of the K-build.  A launch covers the chunks of a launch set,
// each of one quartet type (the shell structure of the four sets of a set
// quartet).
//
//   k_fm_r         one wavefront per run of primitive quartets.  Lanes evaluate
//                  G_m(R,T) (or F_m) of 64 (quartet, cell) slots at once and decide
//                  Fm[0] > 1e-12 for every class L of the type; surviving
//                  cells run the McMurchie-Davidson Hermite recursion
//                  R^(n)_tuv in LDS and the n = 0 layer is summed over cells
//                  in registers.  One Hermite -> cartesian transform per
//                  primitive quartet then gives the cell-summed (e0|f0)
//                  blocks of every class of the type.  Replaces, for all
//                  classes at once, reference src/compute_Fm.cpp (prepare,
//                  Fm, Vm), src/compute_VRR.cpp and the cell sum of
//                  src/compute_ECO.cpp:216-272.
//   k_fm_r<true>   slots whose screening differs between the classes of the
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
// Hermite index tables, built at compile time
// ---------------------------------------------------------------------------
constexpr int NSHELL = 13;  // shells 0..12

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

__constant__ HermTables c_herm = make_herm_tables();
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

// sum_j T2_j sum_{l<14-j} T1_l c[jl]: the operations of reference
// src/t_c_g0_n.cpp:163-178 in the same order (so the value is bitwise the
// oracle's), with T2_j produced by the recurrence of gint_cheb14 inside the
// loop to keep few values live
__device__ __forceinline__ double d_cheb_sum(const double *c, const double *T1, double x2)
{
   GINT_NO_CONTRACT
   double tmp = 0.0, tm1 = 0.0, tm2 = 0.0;
   int jl = 0;
#pragma unroll
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

// the same sum, from the table in coefficient pairs (c: the order's first
// pair, ld: doubles from one pair to the next).  Not fused either: where G_m
// is small against its terms, a slot's orders carry the rounding of this
// order of operations, which far images' integrals amplify
__device__ __forceinline__ double d_cheb_pairs(const double *c, int ld, const double *T1, double x2)
{
   GINT_NO_CONTRACT
   double tmp = 0.0, tm1 = 0.0, tm2 = 0.0, odd = 0.0;
   int jl = 0;
#pragma unroll
   for (int j = 0; j < 14; j++) {
      double t2;
      if (j == 0) t2 = 1.0;
      else if (j == 1) t2 = GINT_SQRT2 * x2;
      else if (j == 2) t2 = 2. * x2 * tm1 - GINT_SQRT2;
      else t2 = 2. * x2 * tm1 - tm2;
      double dot = 0.0;
#pragma unroll
      for (int l = 0; l < 14; l++)
         if (l < 14 - j) {
            const int k = jl + l;
            double ck = odd;
            if (k % 2 == 0) {
               const double2 v = *(const double2 *)(c + (size_t)(k / 2) * ld);
               ck = v.x;
               odd = v.y;
            }
            dot += T1[l] * ck;
         }
      tmp += dot * t2;
      jl += 14 - j;
      tm2 = tm1;
      tm1 = t2;
   }
   return tmp;
}

// A value whose uses stay where they are: what is unpacked from it is not
// kept in registers over the loops around
__device__ __forceinline__ uint32_t here(uint32_t v)
{
   asm volatile("" : "+v"(v));
   return v;
}

// ---------------------------------------------------------------------------
// K1: G_m -> Hermite R -> cell sum -> (e0|f0).  FIX: one wavefront per listed
// (primitive, cell) slot, no screening, blocks and per-L Fm[0] into the
// fix-up workspace.
// ---------------------------------------------------------------------------
constexpr int GEO = 14;   // doubles of a primitive quartet's geometry, at the start of LDS
enum { G_PQ = 0, G_PA = 3, G_QC = 6, G_KFAC = 9, G_RHO = 10, G_RR = 11, G_I2AB = 12, G_I2CD = 13 };
constexpr int EXP1 = 28;  // doubles of one direction's expansion, E^e_t at e (e + 1) / 2 + t
constexpr int FM_CAND = 128;   // slots listed for evaluation

// two doubles, stored at once
struct __attribute__((packed, aligned(8))) Pair {
   double a, b;
};

static FmLayout fm_layout(const TypePlan &tp, bool fix)
{
   FmLayout y;
   const int L = tp.L, nbr = tp.ncp / tp.nkc;
   // the geometries, survivors and blocks of about 8 KB (L = 5) to 16 KB
   // ((dd|dd)-like) per wavefront; beyond that the transform's tables rule
   y.NB = fix ? 1 : (L <= 6 ? 16 : 8);
   y.SV = fix ? 1 : (L <= 6 ? 24 : 16);
   const int places = herm_places(L);
   y.SB = fix ? 1 : std::max(1, std::min(4, places / tp.nh));
   y.o_quirk = GEO * y.NB;
   y.o_sv = y.o_quirk + y.NB;
   y.o_fm = y.o_sv + 5 * y.SV;
   y.o_R = y.o_fm + (L + 1) * y.SV;
   y.o_e = y.o_R + std::max(places, y.SB * tp.nh);
   y.o_c = y.o_e + 6 * EXP1;
   y.o_W = (y.o_c + tp.nkt + tp.nbt + 1) & ~1;   // read two doubles at a time
   y.o_int = 8 * (y.o_W + tp.nbh * (tp.FC + 2));
   const int words = 2 * y.SV + tp.nkc + nbr;
   const int shorts = FM_CAND + 2 * (tp.nkt + tp.nbt) + tp.nbh;
   y.bytes = (y.o_int + 4 * words + 2 * shorts + 15) & ~15;
   return y;
}

// A wavefront takes NB consecutive primitive quartets of a type:
//   - their geometries, one lane each;
//   - all their (quartet, cell) slots, 64 at a time: those within the
//     truncation radius are listed, and G_0 and the screening decision of 64
//     listed ones are taken at once, one lane each;
//   - G_1..G_L of the survivors, one lane per (survivor, order);
//   - quartet by quartet, the Hermite recursion of its survivors in place in
//     LDS (a shell's values before those of the shells below, so one buffer
//     does), their sum in registers, and the transform to (e0|f0) in two
//     passes over LDS, four results per lane.
// About one slot per quartet survives (of 27 to 256 cells), so what it costs
// is the work per quartet, and the serial parts of it: the geometry is 700
// operations, the G sums are loads from a table, and both leave most lanes
// idle when a wavefront has one quartet or two.  Taking 16 (8 of the largest
// types, for LDS) and four results per lane in the transform brought 5.0
// million quartets in 27 cells from 53.7 to 19.5 ms, 6.1 million with s to f
// shells in 125 cells from 81 to 24.4, a cluster of 1.1 million from 9.8 to
// 2.9.  What bounds it now is latency: a wavefront waits in 59 to 64% of its
// cycles, and the vector units are busy 14 (NACC 8) to 40% (NACC 1).
//
// At most 168 VGPRs (3 wavefronts per SIMD): with 128 more values go to
// scratch in the loops, 23.2 instead of 19.5 ms.
//
// NACC: Hermite functions per lane, for types of at most 64 NACC.  Their
// table and sums stay in registers; with those of the largest type for all
// they went to scratch, and each reload waited for the blocks' stores.
//
// One launch takes the chunks of a list, one after the other in the
// numbering of its units (NB primitive quartets): a launch per type left the
// chip to the slowest wavefronts of each, and small systems to launch after
// launch of a few workgroups.
template <bool FIX, int NACC>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(3)))
void k_fm_r(const BatchDev *__restrict__ batches, const WorkRef *__restrict__ refs, int nref, DevTables t, RunDev run)
{
   extern __shared__ double lds[];
   const int lane = threadIdx.x;
   const unsigned long long below = (1ull << lane) - 1ull;
   uint32_t ubase = 0;
   // the fix-up: one entry per turn, those of the set's chunks (nref) one
   // after the other; lane c holds where chunk c's entries end
   uint32_t nfix = 0, fix_end = 0;
   if (FIX) {
      fix_end = lane < nref ? run.fix[lane] : 0u;
      if (!__ballot(fix_end != 0u)) return;
      if (lane < nref) fix_end = min(fix_end, batches[lane].fix_cap);
      for (int off = 1; off < 64; off <<= 1) {
         const uint32_t v = __shfl_up(fix_end, off, 64);
         if (lane >= off) fix_end += v;
      }
      nfix = __shfl(fix_end, 63, 64);
   }
   for (uint32_t turn = FIX ? blockIdx.x : 0; turn < (FIX ? nfix : (uint32_t)nref); turn += FIX ? gridDim.x : 1) {
   uint32_t u0 = turn, nunit = turn + 1, id = 0;
   if (FIX) {
      id = (uint32_t)__builtin_amdgcn_readfirstlane(__popcll(__ballot(fix_end <= turn)));
      if (id) u0 -= (uint32_t)__builtin_amdgcn_readfirstlane((int)__shfl(fix_end, (int)id - 1, 64));
      nunit = u0 + 1;
   } else {
      // the first unit of the chunk that is this workgroup's
      const WorkRef ref = load_uniform(refs + turn);
      const uint32_t skip = ubase % gridDim.x;
      u0 = blockIdx.x >= skip ? blockIdx.x - skip : blockIdx.x + gridDim.x - skip;
      nunit = ref.end - ubase;
      ubase = ref.end;
      id = ref.batch;
      if (u0 >= nunit) continue;
   }
   const BatchDev b = load_batch(batches, id, run);
   const TypePlan &tp = *b.tp;
   const FmLayout lay = FIX ? b.fix_fm : b.fm;
   const int L = load_uniform(&tp.L), nh = load_uniform(&tp.nh), Lp1 = L + 1;
   const int nkc = load_uniform(&tp.nkc), ncp = load_uniform(&tp.ncp), nbh = load_uniform(&tp.nbh);
   const int FC = load_uniform(&tp.FC), FW = FC + 2, nkt = load_uniform(&tp.nkt), nterm = nkt + load_uniform(&tp.nbt);
   const int has00 = load_uniform(&tp.has00), nL = load_uniform(&tp.nL), nbr = ncp / nkc;
   const int LA = load_uniform(&tp.LA), LC = load_uniform(&tp.LC);
   const int NB = lay.NB, SV = lay.SV, SB = lay.SB;
   double *quirk = lds + lay.o_quirk;   // [NB]
   double *sv = lds + lay.o_sv;         // [SV][5]
   double *fm = lds + lay.o_fm;         // [SV][L+1]
   double *R = lds + lay.o_R;
   double *E1 = lds + lay.o_e;          // [2][3][EXP1]: x y z; bra, ket
   double *cf = lds + lay.o_c;          // [nkt], [nbt]
   double *W = lds + lay.o_W;
   int *svi = (int *)((char *)lds + lay.o_int);           // [SV] branch | patch << 2
   int *svq = svi + SV;                                   // [SV] quartet
   uint32_t *rec = (uint32_t *)(svq + SV);                // [nkc] ket components, then bra
   uint16_t *cand = (uint16_t *)(rec + nkc + nbr);        // [FM_CAND] quartet << 8 | cell
   uint16_t *pos = cand + FM_CAND;                        // bytes of the terms' places, [nkt], [nbt]
   uint16_t *ent = pos + nterm;                           // the terms' entries of E, 5 bits each; bit 15: none
   uint16_t *hpos = ent + nterm;                          // [nbh]
   const uint32_t *__restrict__ items = b.items;
   const unsigned all = (1u << nL) - 1u;
   const int Ng = FIX ? 1 : t.Ng;
   // exact quotients of the small numbers that they divide
   const uint32_t qNg = (1u << 24) / (uint32_t)Ng + 1u, qL = 65536u / (uint32_t)max(L, 1) + 1u;
   const int nblk = (nbh + 3) >> 2;
   const uint32_t qblk = 65536u / (uint32_t)nblk + 1u;

   // the type's tables
   lds_order();
   for (int i = lane; i < nterm; i += 64) {
      const uint32_t it = items[i];
      pos[i] = (uint16_t)(((it >> 15) & 1023) * (i < nkt ? 8 : 8 * FW));
      ent[i] = (uint16_t)((it & 0x7fff) | (it >> 31) << 15);
   }
   for (int i = lane; i < nkc + nbr; i += 64) rec[i] = items[nterm + i];
   for (int i = lane; i < nbh; i += 64) hpos[i] = (uint16_t)(items[nterm + nkc + nbr + i] * 8);
   // the lane's Hermite functions h = lane + 64 i: R_h = X_dir R_m1 + coef R_m2
   uint32_t hent[NACC], hplace[NACC];
#pragma unroll
   for (int i = 0; i < NACC; i++) {
      const int h = lane + 64 * i;
      hent[i] = hplace[i] = 0;
      if (h < nh) {
         const HermEntry e = c_herm.e[h];
         if (h) hent[i] = (uint32_t)e.m1 | (uint32_t)(e.m2 >= 0 ? e.m2 : 0) << 9 | (uint32_t)e.dir << 18 | (uint32_t)e.coef << 20;
         hplace[i] = (uint32_t)herm_place(L, c_herm.tuv[h][0], c_herm.tuv[h][1], c_herm.tuv[h][2]);
      }
   }

   for (uint32_t u = u0; u < nunit; u += FIX ? 1u : gridDim.x) {
      // ---- geometry, one lane per quartet ----
      const uint32_t w0 = FIX ? u : u * (uint32_t)NB;
      const int nq = FIX ? 1 : (int)min((uint32_t)NB, b.p1 - b.p0 - w0);
      uint32_t pfirst = b.p0 + w0;
      int fix_n3 = 0;
      double *fix_out = nullptr;
      if (FIX) {
         const uint32_t *fe = in_global(run.fix) + FIX_HEAD + FIX_WORDS * (b.fix_at + u);
         pfirst = fe[0];
         if (pfirst == FIX_VOID) continue;
         fix_n3 = (int)(fe[1] & 0xff);
         fix_out = in_global(run.fix_ws) + fe[2];
      }
      lds_order();
      if (lane < nq) {
         const uint32_t p = pfirst + lane;
         const RowRec row = b.rows[b.prm_row[p]];
         const GroupRec &g = b.groups[row.group];
         const uint32_t ip = b.prm_ip[p];
         const double *data = b.data;
         PrimGeo geo;
         prim_prepare(data + g.R[0], data + g.R[1], data + g.R[2], data + g.R[3], data[g.Z[0] + (ip & 15)],
                      data[g.Z[1] + ((ip >> 4) & 15)], data[g.Z[2] + ((ip >> 8) & 15)],
                      data[g.Z[3] + ((ip >> 12) & 15)], row.n12 & 0xffff, row.n12 >> 16, t, geo);
         double *G = lds + GEO * lane;
         for (int k = 0; k < 3; k++) {
            GINT_NO_CONTRACT
            G[G_PQ + k] = geo.P[k] - geo.Q[k];
            G[G_PA + k] = geo.PA[k];
            G[G_QC + k] = geo.QC[k];
         }
         G[G_KFAC] = geo.Kfac;
         G[G_RHO] = geo.rho;
         G[G_RR] = geo.Rr;
         G[G_I2AB] = geo.i2ab;
         G[G_I2CD] = geo.i2cd;
         quirk[lane] = 0.0;
      }
      lds_order();
      double acc[NACC];
      unsigned long long n_surv = 0, csum = 0, n_any = 0;
      const int nslot = nq * Ng;
      int ncand = 0, s0 = 0;        // listed slots; the next slot to look at
      int cur = -1, next = 0;       // the quartet being summed; the first one without its blocks
      for (bool last = false; !last;) {
         // ---- list the slots that are not beyond truncation ----
         while (ncand < 64 && s0 < nslot) {
            const int slot = s0 + lane;
            int q = 0, n3 = 0;
            bool keep = slot < nslot;
            if (keep) {
               q = (int)(((uint32_t)slot * qNg) >> 24);
               n3 = FIX ? fix_n3 : slot - q * Ng;
               if (t.truncated && !FIX) {
                  GINT_NO_CONTRACT
                  const double *G = lds + GEO * q;
                  const double x = G[G_PQ + 0] - t.neighs[n3 * 3 + 0];
                  const double y = G[G_PQ + 1] - t.neighs[n3 * 3 + 1];
                  const double z = G[G_PQ + 2] - t.neighs[n3 * 3 + 2];
                  const double rpq2 = x * x + y * y + z * z;
                  const double Rr = G[G_RR];
                  keep = !(G[G_RHO] * rpq2 > Rr * Rr + 11.0 * Rr + 50.0);
               }
            }
            const unsigned long long m = __ballot(keep);
            if (keep) cand[ncand + __popcll(m & below)] = (uint16_t)(q << 8 | n3);
            ncand += __popcll(m);
            s0 += 64;
         }
         lds_order();
         const int ncd = min(ncand, 64);
         // ---- G_0 and the decision of up to 64 listed slots ----
         int status = 0;  // 1 kept by every class, 2 screened by every class, 3 class-dependent
         int q = 0, br = 0, patch = 0;
         double X[3] = {0.0, 0.0, 0.0}, Fm0 = 0.0, tg1 = 0.0, tg2 = 0.0;
         if (lane < ncd) {
            const int c = cand[lane], n3 = c & 255;
            q = c >> 8;
            const double *G = lds + GEO * q;
            const double Kfac = G[G_KFAC];
            unsigned mask = 0;
            double T;
            {
               GINT_NO_CONTRACT
               X[0] = G[G_PQ + 0] - t.neighs[n3 * 3 + 0];
               X[1] = G[G_PQ + 1] - t.neighs[n3 * 3 + 1];
               X[2] = G[G_PQ + 2] - t.neighs[n3 * 3 + 2];
               const double rpq2 = X[0] * X[0] + X[1] * X[1] + X[2] * X[2];
               T = G[G_RHO] * rpq2;
            }
            br = t.truncated ? gint_tcg_locate(G[G_RR], T, t.grid_lo, t.grid_hi, t.bw, &patch, &tg1, &tg2) : GINT_G_BOYS;
            if (br == GINT_G_PATCH) {
               GINT_NO_CONTRACT
               double T1[14];
               gint_cheb14(tg1, T1);
               Fm0 = d_cheb_sum(t.C0 + (size_t)t.ld_C0 * patch, T1, tg2) * Kfac;
            } else if (br == GINT_G_BOYS) {
               Fm0 = gint_boys_f0(L, T, t.ftable, Kfac);
               tg1 = T;
            }
            const bool lsens = br == GINT_G_BOYS && T >= 1.e-13 && T < 12.;   // F_0 depends on the start order
            if (br == GINT_G_ZERO) {
               status = 2;
            } else {
               mask = Fm0 > 1.e-12 ? all : 0u;
               // F_0 of the downward recursion depends on the starting order
               // by rounding only; decide each class L exactly this close to
               // the threshold
               if (lsens && nL > 1 && fabs(Fm0 - 1.e-12) <= 1.e-20) {
                  mask = 0u;
                  for (int i = 0; i < nL; i++)
                     if (gint_boys_f0(tp.Ls[i], T, t.ftable, Kfac) > 1.e-12) mask |= 1u << i;
               }
               status = mask == all ? 1 : (mask == 0u ? 2 : 3);
            }
            if (FIX) {
               // per-L Fm[0] of the slot, for the classes that screen it
               double *f0 = fix_out + ncp;
               for (int i = 0; i < nL; i++) f0[i] = lsens ? gint_boys_f0(tp.Ls[i], T, t.ftable, Kfac) : Fm0;
               status = br == GINT_G_ZERO ? 2 : 1;
            } else if (b.force_fix && status == 1) {
               status = 3;
            }
            if (!FIX) {
               if (status == 2) {
                  if (has00) atomicAdd(&quirk[q], Fm0);
               } else {
                  if (b.stats) {
                     const uint32_t p = pfirst + q;
                     const RowRec row = b.rows[b.prm_row[p]];
                     const GroupRec &g = b.groups[row.group];
                     const unsigned long long h = slot_hash(g.set_ij, g.set_kl, row.n12 & 0xffff, row.n12 >> 16, b.prm_ip[p], n3);
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
                     // (the list's place read here: kept, it costs registers)
                     const BatchDev *bd = in_global(batches) + here(id);
                     const uint32_t idx = atomicAdd(run.fix + id, 1u);
                     bool room = idx < bd->fix_cap;
                     if (room) {
                        const unsigned long long at =
                            atomicAdd((unsigned long long *)(run.fix + FIX_USED), (unsigned long long)(ncp + 16));
                        room = at + (unsigned long long)(ncp + 16) <= run.fix_doubles;
                        uint32_t *fe = in_global(run.fix) + FIX_HEAD + FIX_WORDS * (bd->fix_at + idx);
                        fe[0] = room ? pfirst + q : FIX_VOID;
                        fe[1] = (uint32_t)n3 | (mask << 8);
                        fe[2] = (uint32_t)at;
                     }
                     if (!room) {
                        // every class keeps the slot (its G_0 is within
                        // rounding of the 1e-12 threshold)
                        atomicAdd(run.fix + FIX_LOST, 1u);
                        status = 1;
                        n_any++;
                     }
                  } else {
                     n_any++;
                  }
               }
            }
         }
         // the listed slots that are left move to the front
         ncand -= ncd;
         if (lane < ncand) cand[lane] = cand[64 + lane];
         last = ncand == 0 && s0 >= nslot;
         // ---- the survivors, in the order of the quartets, SV at a time ----
         const unsigned long long smask = __ballot(status == 1);
         const int nsv = __popcll(smask), rank = __popcll(smask & below);
         int k0 = 0;
         do {
            const int np = min(SV, nsv - k0);
            const int r = rank - k0;
            lds_order();
            if (status == 1 && r >= 0 && r < SV) {
               sv[r * 5 + 0] = X[0];
               sv[r * 5 + 1] = X[1];
               sv[r * 5 + 2] = X[2];
               sv[r * 5 + 3] = tg1;
               sv[r * 5 + 4] = tg2;
               fm[r * Lp1] = Fm0;
               svi[r] = br | patch << 2;
               svq[r] = q;
            }
            lds_order();
            // (-2 rho)^m G_m, one (survivor, order) per lane
            for (int idx = lane; idx < np * L; idx += 64) {
               const int s = (int)(((uint32_t)idx * qL) >> 16), m = idx - s * L + 1;
               const int info = svi[s];
               if ((info & 3) != GINT_G_PATCH) continue;
               const double *G = lds + GEO * svq[s];
               const double m2rho = -2.0 * G[G_RHO];
               double pw = G[G_KFAC];
               for (int k = 0; k < m; k++) pw *= m2rho;
               const double *c = t.Cm + ((size_t)(info >> 2) * CM_PAIRS * t.ldm + (m - 1)) * 2;
               double T1[14];
               gint_cheb14(sv[s * 5 + 3], T1);
               fm[s * Lp1 + m] = d_cheb_pairs(c, 2 * t.ldm, T1, sv[s * 5 + 4]) * pw;
            }
            if (lane < np && (svi[lane] & 3) == GINT_G_BOYS) {
               const double *G = lds + GEO * svq[lane];
               double *f = fm + lane * Lp1;
               gint_boys(L, sv[lane * 5 + 3], f, t.ftable, G[G_KFAC]);
               const double m2rho = -2.0 * G[G_RHO];
               double pw = 1.0;
               for (int m = 1; m <= L; m++) {
                  pw *= m2rho;
                  f[m] *= pw;
               }
            }
            lds_order();

            for (int s = 0;;) {
               int qs;
               if (s < np) qs = __builtin_amdgcn_readfirstlane(svq[s]);
               else if (last && k0 + np >= nsv) qs = nq;   // the end: what is left to write
               else break;
               if (qs != cur) {
                  if (cur >= 0) {
                     // ---- Hermite -> cartesian of the quartet `cur` ----
                     const double *G = lds + GEO * cur;
                     const int ln = (int)here((uint32_t)lane);
                     lds_order();
#pragma unroll
                     for (int i = 0; i < NACC; i++)
                        if (ln + 64 * i < nh) R[here(hplace[i])] = acc[i];
                     // E^{e+1}_t = E^e_{t-1} / (2 zeta) + x E^e_t + (t + 1) E^e_{t+1}, one
                     // direction per lane (ket: (-1)^t E).  The recursion as such: the
                     // errors of its steps cancel in the horizontal recurrence, those
                     // of a closed form do not
                     if (ln < 6) {
                        const bool ket = ln >= 3;
                        const double x = G[(ket ? G_QC - 3 : G_PA) + ln], i2 = ket ? G[G_I2CD] : G[G_I2AB];
                        const int lm = ket ? LC : LA;
                        double *E = E1 + EXP1 * ln;
                        double e0[8] = {1.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
                        E[0] = 1.0;
#pragma unroll
                        for (int e = 0; e < 6; e++) {
                           if (e >= lm) break;
                           double below_ = 0.0;   // E^e_{t-1}
#pragma unroll
                           for (int tt = 0; tt <= e + 1; tt++) {
                              double v = 0.0;
                              if (tt > 0) v += i2 * below_;
                              if (tt <= e) v += x * e0[tt];
                              if (tt + 1 <= e) v += (double)(tt + 1) * e0[tt + 1];
                              below_ = e0[tt];
                              e0[tt] = v;
                              E[(e + 1) * (e + 2) / 2 + tt] = ket && (tt & 1) ? -v : v;
                           }
                        }
                     }
                     lds_order();
                     for (int i = ln; i < nterm; i += 64) {
                        const uint32_t it = ent[i];
                        const double *e = E1 + (i < nkt ? 3 * EXP1 : 0);
                        const double v = e[it & 31] * e[EXP1 + ((it >> 5) & 31)] * e[2 * EXP1 + ((it >> 10) & 31)];
                        cf[i] = it >> 15 ? 0.0 : v;
                     }
                     double *dst = FIX ? fix_out : b.ac0 + (size_t)(w0 + cur) * ncp;
                     const double qsum = !FIX && has00 ? quirk[cur] : 0.0;
                     double vmax = 0.0;
                     for (int f0 = 0; f0 < nkc; f0 += FC) {
                        const int nf = min(FC, nkc - f0);
                        lds_order();
                        // W[tuv][f] = sum of the ket component's terms over R[tuv + term]
                        for (int idx = ln; idx < nf * nblk; idx += 64) {
                           const int fi = (int)(((uint32_t)idx * qblk) >> 16), hb = idx - fi * nblk;
                           const uint32_t rc = rec[f0 + fi];
                           const int n = (int)(rc >> 20);
                           const double *ck = cf + ((rc >> 8) & 0xfff);
                           const uint16_t *pk = pos + ((rc >> 8) & 0xfff);
                           const char *r0 = (const char *)R + hpos[hb];
                           const char *r1 = (const char *)R + hpos[min(hb + nblk, nbh - 1)];
                           const char *r2 = (const char *)R + hpos[min(hb + 2 * nblk, nbh - 1)];
                           const char *r3 = (const char *)R + hpos[min(hb + 3 * nblk, nbh - 1)];
                           double s0_ = 0.0, s1_ = 0.0, s2_ = 0.0, s3_ = 0.0;
                           for (int k = 0; k < n; k += 2) {
                              const double ca = ck[k], cb = ck[k + 1];
                              const int pa = pk[k], pb = pk[k + 1];
                              s0_ += ca * *(const double *)(r0 + pa);
                              s1_ += ca * *(const double *)(r1 + pa);
                              s2_ += ca * *(const double *)(r2 + pa);
                              s3_ += ca * *(const double *)(r3 + pa);
                              s0_ += cb * *(const double *)(r0 + pb);
                              s1_ += cb * *(const double *)(r1 + pb);
                              s2_ += cb * *(const double *)(r2 + pb);
                              s3_ += cb * *(const double *)(r3 + pb);
                           }
                           double *w = W + hb * FW + (int)(rc & 0xff) - f0;
                           w[0] = s0_;
                           if (hb + nblk < nbh) w[nblk * FW] = s1_;
                           if (hb + 2 * nblk < nbh) w[2 * nblk * FW] = s2_;
                           if (hb + 3 * nblk < nbh) w[3 * nblk * FW] = s3_;
                        }
                        lds_order();
                        // (e0|f0) = sum of the bra component's terms over W[tuv][f]
                        const int nfb = (nf + 3) >> 2;
                        const uint32_t qfb = 65536u / (uint32_t)nfb + 1u;
                        for (int idx = ln; idx < nbr * nfb; idx += 64) {
                           const int ei = (int)(((uint32_t)idx * qfb) >> 16), fb = idx - ei * nfb;
                           const uint32_t rc = rec[nkc + ei];
                           const int n = (int)(rc >> 20), e = (int)(rc & 0xff);
                           const double *ck = cf + nkt + ((rc >> 8) & 0xfff);
                           const uint16_t *pk = pos + nkt + ((rc >> 8) & 0xfff);
                           const char *w = (const char *)(W + 4 * fb);
                           double s0_ = 0.0, s1_ = 0.0, s2_ = 0.0, s3_ = 0.0;
                           for (int k = 0; k < n; k += 2) {
                              const double ca = ck[k], cb = ck[k + 1];
                              const double2 *wa = (const double2 *)(w + pk[k]), *wb = (const double2 *)(w + pk[k + 1]);
                              const double2 a0 = wa[0], a1 = wa[1], b0 = wb[0], b1 = wb[1];
                              s0_ += ca * a0.x;
                              s1_ += ca * a0.y;
                              s2_ += ca * a1.x;
                              s3_ += ca * a1.y;
                              s0_ += cb * b0.x;
                              s1_ += cb * b0.y;
                              s2_ += cb * b1.x;
                              s3_ += cb * b1.y;
                           }
                           const int f = f0 + 4 * fb;
                           double *o = dst + e * nkc + f;
                           if (e == 0 && f == 0) s0_ += qsum;
                           if (f + 3 < nkc) {
                              *(Pair *)o = Pair{s0_, s1_};
                              *(Pair *)(o + 2) = Pair{s2_, s3_};
                           } else {
                              o[0] = s0_;
                              if (f + 1 < nkc) o[1] = s1_;
                              else s1_ = 0.0;
                              if (f + 2 < nkc) o[2] = s2_;
                              else s2_ = 0.0;
                              s3_ = 0.0;
                           }
                           vmax = fmax(vmax, fmax(fmax(fabs(s0_), fabs(s1_)), fmax(fabs(s2_), fabs(s3_))));
                        }
                     }
                     // calibration of the mixed-precision routing: the largest block
                     // element of each set quartet (a positive double orders as its bits)
                     if (!FIX && b.gmag) {
                        for (int off = 32; off > 0; off >>= 1) vmax = fmax(vmax, __shfl_xor(vmax, off, 64));
                        if (lane == 0)
                           atomicMax((unsigned long long *)(b.gmag + b.rows[b.prm_row[pfirst + cur]].group),
                                     (unsigned long long)__double_as_longlong(vmax));
                     }
                     next = cur + 1;
                  }
                  // quartets without a surviving cell: zero but for the
                  // screened slots' Fm[0] in (00|00)
                  for (; !FIX && next < qs; next++) {
                     double *dst = b.ac0 + (size_t)(w0 + next) * ncp;
                     const double qsum = has00 ? quirk[next] : 0.0;
                     for (int j = lane; j < ncp; j += 64) dst[j] = j == 0 ? qsum : 0.0;
                     if (b.gmag && lane == 0 && has00)
                        atomicMax((unsigned long long *)(b.gmag + b.rows[b.prm_row[pfirst + next]].group),
                                  (unsigned long long)__double_as_longlong(fabs(qsum)));
                  }
                  cur = qs;
                  if (qs == nq) break;
#pragma unroll
                  for (int i = 0; i < NACC; i++) acc[i] = 0.0;
               }
               // ---- Hermite recursion of the quartet's survivors ----
               //    R^(n)_tuv = coef R^(n+1)_{tuv-2d} + X_d R^(n+1)_{tuv-d}
               const int nb = min(SB, (int)__popcll(__ballot(lane >= s && lane < np && svq[min(lane, SV - 1)] == qs)));
               const double *xs = sv + 5 * s, *fs = fm + Lp1 * s;
               lds_order();
               const int ln = (int)here((uint32_t)lane);
               if (ln < nb) R[ln * nh] = fs[ln * Lp1 + L];
               for (int n = L - 1; n >= 1; n--) {
                  const int mn = d_nherm(L - n);
#pragma unroll
                  for (int i = NACC - 1; i >= 0; i--) {
                     if (64 * i >= mn) continue;
                     lds_order();
                     const int h = lane + 64 * i;
                     if (h >= mn) continue;
                     const uint32_t he = here(hent[i]);
                     const int m1 = he & 511, m2 = (he >> 9) & 511, dir = (he >> 18) & 3;
                     const double c = (double)(he >> 20);
                     for (int k = 0; k < nb; k++) {
                        double *Rk = R + k * nh;
                        double v = xs[5 * k + dir] * Rk[m1] + c * Rk[m2];
                        if (h == 0) v = fs[k * Lp1 + n];
                        Rk[h] = v;
                     }
                  }
               }
               // the n = 0 layer goes straight into the cell sum
               lds_order();
#pragma unroll
               for (int i = 0; i < NACC; i++) {
                  if (64 * i >= nh) continue;
                  const uint32_t he = here(hent[i]);
                  const int m1 = he & 511, m2 = (he >> 9) & 511, dir = (he >> 18) & 3;
                  const double c = (double)(he >> 20);
                  for (int k = 0; k < nb; k++) {
                     const double *Rk = R + k * nh;
                     double v = xs[5 * k + dir] * Rk[m1] + c * Rk[m2];
                     if (i == 0 && lane == 0) v = fs[k * Lp1];
                     acc[i] += v;
                  }
               }
               s += nb;
            }
            k0 += SV;
         } while (k0 < nsv);
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
   }
}

// orders 1 .. ldm of the caller's table, as d_cheb_pairs reads them: the
// orders of one coefficient pair side by side, so that the lanes of a
// survivor read one or two cache lines
__global__ void k_pack_c0(const double *__restrict__ C0, int ld_C0, int ldm, double *__restrict__ Cm)
{
   const int n = TCG_NPATCH * CM_PAIRS * ldm;
   for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
      const int m = i % ldm, k = i / ldm % CM_PAIRS, p = i / ldm / CM_PAIRS;
      const double *c = C0 + (size_t)ld_C0 * p + (m + 1) * TCG_NCOEF + 2 * k;
      Cm[2 * i] = c[0];
      Cm[2 * i + 1] = 2 * k + 1 < TCG_NCOEF ? c[1] : 0.0;
   }
}

int launch_pack_c0(const double *C0, int ld_C0, int ldm, double *Cm, void *stream)
{
   hipLaunchKernelGGL(k_pack_c0, dim3(512), dim3(256), 0, (hipStream_t)stream, C0, ld_C0, ldm, Cm);
   return hipGetLastError() == hipSuccess ? 0 : -1;
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

void fm_layouts(const TypePlan &tp, FmLayout &main, FmLayout &fix)
{
   main = fm_layout(tp, false);
   fix = fm_layout(tp, true);
}

int launch_fm_r(const BatchDev *batches, const WorkRef *refs, int nref, uint32_t units, int nacc, size_t lds,
                const DevTables &t, const RunDev &run, void *stream)
{
   if (!units) return 0;
   if (lds > LDS_LIMIT) return -3;
   // workgroups stay resident and stride over the units
   const dim3 grid(std::min(units, 16384u)), block(64);
   hipStream_t st = (hipStream_t)stream;
   switch (nacc) {
      case 1: hipLaunchKernelGGL((k_fm_r<false, 1>), grid, block, lds, st, batches, refs, nref, t, run); break;
      case 3: hipLaunchKernelGGL((k_fm_r<false, 3>), grid, block, lds, st, batches, refs, nref, t, run); break;
      case 8: hipLaunchKernelGGL((k_fm_r<false, 8>), grid, block, lds, st, batches, refs, nref, t, run); break;
      default: return -3;
   }
   return hipGetLastError() == hipSuccess ? 0 : -1;
}

int launch_fixup(const BatchDev *batches, int nbatch, size_t lds, const DevTables &t, const RunDev &run, uint32_t n_fix,
                 void *stream)
{
   if (nbatch > MAX_LAUNCH_CHUNKS) return -4;
   if (lds > LDS_LIMIT) return -3;
   const unsigned grid = std::max(1u, std::min(n_fix, 4096u));
   hipLaunchKernelGGL((k_fm_r<true, 8>), dim3(grid), dim3(64), lds, (hipStream_t)stream, batches,
                      (const WorkRef *)nullptr, nbatch, t, run);
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

// The mixed-precision flag of each set quartet of a chunk, for k_eco (where
// k_sq contracts it, it is counted and no more): its bound  max|block
// element| x max|coefficient|^4 x primitive quartets  times max|P| is below
// tau.  count[0] += flagged.
__global__ void k_mixed_flags(const BatchDev *__restrict__ batch, RunDev run, const unsigned long long *__restrict__ pmax,
                              double tau, unsigned long long *count)
{
   const double *gmag = in_global(load_uniform(&batch->gmag));
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
