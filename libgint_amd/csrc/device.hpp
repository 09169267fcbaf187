// Interface between the host engine (engine.cpp, built with g++ -fopenmp)
// and the gfx950 kernels (kernels.hip, built with hipcc): record layouts in
// HBM, the per-type and per-class plans, and the launchers.  Plain types
// only.
//
// Work is organised by quartet *type*: the shell structure (l and number of
// contractions of every shell) of the four sets of a set quartet.  All
// shells of a set share its exponents, so the primitive work of a
// (primitive quartet, lattice cell) slot is done once for every
// angular-momentum class of the set quartet.
#pragma once
#include <stdint.h>
#include <stddef.h>

#include <vector>

#if defined(__HIPCC__)
#define GINT_HDI __host__ __device__ inline
#else
#define GINT_HDI inline
#endif

namespace gint {

constexpr int MAXL = 3;          // highest angular momentum of a shell (f)
constexpr int MAXLL = 4 * MAXL;  // highest total angular momentum of a class
constexpr int MAXNL = 4;         // contractions per shell
constexpr int MAXNP = 16;        // primitives per set
constexpr int MAXNG = 256;       // lattice vectors
constexpr int NCLASS = 256;      // (la,lb,lc,ld), each 0..3
constexpr int MAXSH = 4;         // shells per set (distinct l)
constexpr int MAXTC = MAXSH * MAXSH * MAXSH * MAXSH;  // classes per type
constexpr int MAXHERM = 455;     // Hermite triples t+u+v <= 12

inline constexpr int nco(int l) { return (l + 1) * (l + 2) / 2; }
inline constexpr int nsph(int l) { return 2 * l + 1; }
inline constexpr int nherm(int L) { return (L + 1) * (L + 2) * (L + 3) / 6; }
inline constexpr int class_code(int la, int lb, int lc, int ld) { return ((la * 4 + lb) * 4 + lc) * 4 + ld; }

// One row: a set quartet at bra/ket images (n1,n2) with its primitive
// quartets (one libgint_add_shell call).  Its contracted blocks sit at
// (row - first row of the chunk) * eco_row in the contraction buffer.
struct RowRec {
   uint32_t prm_off;   // first primitive quartet of the row
   uint32_t n_prm;
   uint32_t group;     // its set quartet
   uint32_t n12;       // n1 | n2 << 16
};
static_assert(sizeof(RowRec) == 16, "RowRec layout");

// One set quartet (the work between two libgint_add_set calls).
struct GroupRec {
   uint32_t row0, row1;       // its rows
   uint32_t R[4], Z[4];       // centre and exponent offsets in the basis data
   uint32_t Kof[4][MAXSH];    // normalised coefficients of shell s of centre t (nl x np)
   uint32_t np4;              // np-1 of the four sets, 4-bit fields
   uint32_t set_ij, set_kl;   // set indices, 16-bit fields (survivor checksum only)
   uint32_t ks;               // KS_SETLEVEL: its KsSet; else its first KsGroup (nclass of them)
   uint32_t ksmode;           // KS_SETLEVEL or 0
   uint32_t pad;
};
static_assert(sizeof(GroupRec) == 128, "GroupRec layout");

// Where the contracted quartets of one (set quartet, class) go in K: the
// add_qrtt calls of the class compressed to offsets affine in the
// contraction indices (inla, inlb, inlc, inld), or a reference to an
// explicit list when the caller's offsets are not affine.
struct KsGroup {
   uint32_t base[4];   // ac ad bc bd block offsets of the first call
   int32_t step[8];    // ac: by inla, inlc; ad: by inla, inld; bc: by inlb, inlc; bd: by inlb, inld
   uint32_t ld01;      // ld_ac | ld_ad << 16
   uint32_t ld23;      // ld_bc | ld_bd << 16
   uint32_t flags;     // bits 0-3 transposes, 4-6 symmetry code, bit 8 explicit, bits 16-24 calls
   uint32_t expl;      // first explicit record when bit 8 is set
};
static_assert(sizeof(KsGroup) == 64, "KsGroup layout");

constexpr uint32_t KS_EXPLICIT = 1u << 8;
// integral output instead of a K update: the class's spherical integrals go
// to the output array at base[0] | base[1] << 32, ordered
// [ila, isa, ilb, isb, ilc, isc, ild, isd] (reference src/compute_TRA.cpp:36-47)
constexpr uint32_t KS_OUTPUT = 1u << 9;
GINT_HDI uint32_t ks_count(uint32_t flags) { return flags >> 16; }

// Every add_qrtt call of one set quartet at once, when the caller lays out
// its P / K blocks per pair of sets (the layout of CP2K's block matrices):
// function f of set x and function g of set y sit at
// base + (T ? f ld + g : g ld + f) of the (x,y) pair block, with the
// functions of a set ordered shell by shell, contraction by contraction,
// 2l+1 each.  Every class of the set quartet has all its contraction
// combinations, and they share leading dimensions, transposes and the
// symmetry code.  The KsGroup of each class follows from it (ks_from_set).
struct KsSet {
   uint32_t base[4];   // ac ad bc bd pair blocks: element of (function 0, function 0)
   uint32_t ld01;      // ld_ac | ld_ad << 16
   uint32_t ld23;      // ld_bc | ld_bd << 16
   uint32_t flags;     // bits 0-3 transposes, 4-6 symmetry code
   uint32_t pad;
};
static_assert(sizeof(KsSet) == 32, "KsSet layout");

constexpr uint32_t KS_SETLEVEL = 1u;   // GroupRec::ksmode

// one add_qrtt call, kept when a (set quartet, class) is not affine
struct KsRec {
   uint32_t off[4];
   uint32_t ld01, ld23, flags, pad;
};
static_assert(sizeof(KsRec) == 32, "KsRec layout");

// One angular-momentum class: its blocks and what its recurrences cost.
struct ClassPlan {
   int la, lb, lc, ld;
   int L, LA, LC;
   int ncp;                  // its (e0|f0) block set, e in [la,LA], f in [lc,LC], e outer
   int Ns;                   // spherical integrals
   // algorithmic FLOPs of the reference chain for this class
   int fm_flops;             // 52 + 211 (L+1) per surviving slot
   int vrr_flops;            // reference plan VRR (weights 3/8/3/8/11/6 per element)
   int hrr_flops;            // 2 per HRR element
   int sph_flops;            // 2 m n k over the four stages
};

// Plan of one quartet type.  The blocks (e0|f0) with e in [LA0,LA], f in
// [LC0,LC] are produced per primitive quartet, summed over lattice cells, as
// one matrix: bra components (shell e outer) x ket components (shell f
// outer); each class reads a rectangle of it.
struct TypePlan {
   int nsh[4];
   int l[4][MAXSH];
   int nl[4][MAXSH];
   int nclass;               // nsh0*nsh1*nsh2*nsh3, sa outer
   int LA0, LA, LC0, LC, L;
   int ncp;
   int bcoff[7];             // first bra component of shell e
   int nkc;                  // ket cartesian components, f in [LC0,LC]
   int kcoff[7];             // first of shell f among them
   int nbh;                  // bra Hermite triples t+u+v <= LA
   int nh;                   // Hermite triples t+u+v <= L
   // Hermite -> cartesian transform (make_type_items)
   int FC;                   // ket components per pass, a multiple of 4
   int nkt, nbt;             // terms of the ket and of the bra expansion
   int has00;                // LA0 == 0 && LC0 == 0
   int nL;                   // distinct class L values
   int Ls[16];
   int cls_code[MAXTC];      // class_code(la,lb,lc,ld) of class k
   int cls_sh[MAXTC];        // sa | sb<<4 | sc<<8 | sd<<12
   int cls_gate[MAXTC];      // index into Ls
   int cls_nl[MAXTC];        // nla*nlb*nlc*nld
   int cls_ncp[MAXTC];
   int fun0[4][MAXSH];       // first spherical function of shell s within set t (sets list shells in order)
   int nfun[4];              // spherical functions of set t
   unsigned long long cls_mult[MAXTC];   // checksum multiplier of class k (odd)
   unsigned long long mult_all;          // sum of cls_mult
   // algorithmic FLOPs of this library's kernels (Hermite path)
   long long surv_flops;     // per slot that survives for some class: G_m and the R recursion
   long long prim_flops;     // per primitive quartet: Hermite -> cartesian transform
   long long ref_slot_flops; // per slot, summed over classes: the reference's Fm + VRR
};

// Place of Hermite triple (t,u,v), t+u+v <= L, in the cell sum of a type:
// additive, so that the place of a sum of two triples is the sum of theirs,
// and different for different triples (found by search up to L = 12)
GINT_HDI int herm_place(int L, int t, int u, int v) { return t + u * (L + 1) + v * (L * (L + 1) + 1); }
GINT_HDI int herm_places(int L) { return L * (L * (L + 1) + 1) + 1; }

// The KsGroup of class k of a set quartet stored as a KsSet: offsets of
// contraction (ia,ib,ic,id) are base + ia step[0] + ic step[1] (ac), ...
GINT_HDI KsGroup ks_from_set(const KsSet &s, const TypePlan &tp, int k)
{
   KsGroup g;
   const int sh = tp.cls_sh[k], code = tp.cls_code[k];
   const int sa = sh & 15, sb = (sh >> 4) & 15, sc = (sh >> 8) & 15, sd = (sh >> 12) & 15;
   const long long nsa = 2 * (code / 64) + 1, nsb = 2 * ((code / 16) % 4) + 1, nsc = 2 * ((code / 4) % 4) + 1,
                   nsd = 2 * (code % 4) + 1;
   const long long fa = tp.fun0[0][sa], fb = tp.fun0[1][sb], fc = tp.fun0[2][sc], fd = tp.fun0[3][sd];
   const long long ld[4] = {s.ld01 & 0xffff, s.ld01 >> 16, s.ld23 & 0xffff, s.ld23 >> 16};
   // element (row r, column c) of pair block q: rows of a (ac, ad) or b (bc, bd)
   auto pos = [&](int q, long long r, long long c) { return ((s.flags >> q) & 1) ? r * ld[q] + c : c * ld[q] + r; };
   g.base[0] = (uint32_t)(s.base[0] + pos(0, fa, fc));
   g.base[1] = (uint32_t)(s.base[1] + pos(1, fa, fd));
   g.base[2] = (uint32_t)(s.base[2] + pos(2, fb, fc));
   g.base[3] = (uint32_t)(s.base[3] + pos(3, fb, fd));
   g.step[0] = (int32_t)pos(0, nsa, 0);
   g.step[1] = (int32_t)pos(0, 0, nsc);
   g.step[2] = (int32_t)pos(1, nsa, 0);
   g.step[3] = (int32_t)pos(1, 0, nsd);
   g.step[4] = (int32_t)pos(2, nsb, 0);
   g.step[5] = (int32_t)pos(2, 0, nsc);
   g.step[6] = (int32_t)pos(3, nsb, 0);
   g.step[7] = (int32_t)pos(3, 0, nsd);
   g.ld01 = s.ld01;
   g.ld23 = s.ld23;
   g.flags = (s.flags & 0x7fu) | (uint32_t)tp.cls_nl[k] << 16;
   g.expl = 0;
   return g;
}

// Device-resident constant tables.
struct DevTables {
   const double *C0;          // [patch][ld_C0]: the caller's table
   int ld_C0;
   const double *Cm;          // orders 1 .. ldm of it as [patch][coefficient pair][order][2] (launch_pack_c0)
   int ldm;
   const int *grid_lo, *grid_hi;
   const double *bw;
   const double *ftable;
   const double *cell;
   const double *neighs;
   int Ng;
   int truncated;
   double R_cut;
};

// LDS of k_fm_r for a type: offsets in doubles, of the tables in bytes.
struct FmLayout {
   int NB;      // primitive quartets per wavefront
   int SV;      // surviving slots kept at once
   int SB;      // of them in one Hermite recursion
   int o_quirk; // [NB] screened slots' Fm[0] (behind the geometry)
   int o_sv;    // [SV] X Y Z of P-Q-g, TG1 (or T), TG2
   int o_fm;    // [SV][L+1] (-2 rho)^m G_m
   int o_R;     // Hermite layers [SB][nh]; then the cell sum at its additive places
   int o_e;     // one-dimensional expansions E of both sides, [2][3][28]
   int o_c;     // the transform's coefficients: ket terms, bra terms
   int o_W;     // [nbh][FC + 2]
   int o_int;   // byte offset of the slot lists and the type's tables
   int bytes;
};

// Part `part` of `parts` of a set quartet for k_sq: every parts-th window of
// SQ_NW primitive quartets, counted through its rows
struct SqSeg {
   uint32_t group;
   uint16_t part, parts;
};

// One chunk of one type's work.  Primitive, row and group indices are
// absolute within the type's arrays; ac0 and eco are indexed from the
// chunk's first primitive and first row.  The records of a launch sequence's
// chunks lie in device memory; a kernel takes a list of them (so that one
// launch covers many types) and adds the execution's buffers (RunDev).
struct BatchDev {
   const TypePlan *tp;        // device copy
   const SqSeg *segs;         // the chunk's set quartets for k_sq, in parts, by falling work (null: whole, as stored)
   const uint32_t *rorder;    // its rows by falling work, absolute, for k_eco (null: as stored)
   const uint32_t *items;     // the type's Hermite -> cartesian tables (make_type_items)
   const RowRec *rows;
   const GroupRec *groups;
   const uint32_t *prm_row;   // row of each primitive quartet
   const uint32_t *prm_ip;    // ipa | ipb << 4 | ipc << 8 | ipd << 12
   const KsGroup *ksg;        // per class of the groups that are not KS_SETLEVEL (GroupRec::ks)
   const KsSet *kss;          // KS_SETLEVEL groups
   const KsRec *ksx;
   uint64_t ac_off, eco_off;  // the chunk's blocks and contraction buffer rows in the work buffer, doubles
   size_t eco_row;            // doubles per row of the contraction buffer (k_eco); 0: none
   double *gmag;              // calibration: max |block element| per set quartet (nullable; absolute group index)
   uint32_t *gflag;           // mixed precision: 1 = single-precision contraction for the set quartet (nullable)
   uint32_t p0, p1;           // primitives of the chunk
   uint32_t r0, r1;           // rows
   uint32_t g0, g1;           // groups
   uint32_t fix_at, fix_cap;  // its entries of the fix-up list: the first, how many there may be
   FmLayout fm, fix_fm;       // k_fm_r: the chunk's own pass, the fix-up
   // set from RunDev by the kernels
   const double *data;
   double *ac0;               // [primitive - p0][ncp]
   double *eco;
   unsigned long long *stats; // STATS_SLOTS x {surviving (slot, class) pairs, checksum, K1 FLOPs} (nullable)
   int force_fix;             // route every surviving slot through the fix-up path (test hook)
   uint32_t id;               // the chunk's number in the launch
};

// Buffers of an execution.
struct RunDev {
   double *work;
   const double *data;
   unsigned long long *stats;
   uint32_t *fix;         // fix-up list: FIX_HEAD words, then the entries
   double *fix_ws;        // its workspace
   uint32_t fix_doubles;  // doubles of it
   int force_fix;
   int mixed;   // 0 off, 1 calibrate (gmag), 2 route (gflag)
};

constexpr int MAX_LAUNCH_CHUNKS = 64;   // of one launch

// The fix-up list of a launch set, of the slots that some classes keep and
// others screen: each chunk has room for FIX_CAP entries of its own
// (NOALLOC_FIX in the static scratch), and all of them share a workspace that
// holds as many of the set's largest type.  A slot that finds no room is kept
// by every class and counted.  An entry: primitive (FIX_VOID: none, the
// workspace was full), n3 | mask of the classes' L << 8, its first double of
// ncp + 16 in the workspace.
constexpr uint32_t FIX_CAP = 4096, FIX_WORDS = 3, FIX_VOID = 0xffffffffu;
// The words before the entries: [0..63] entries of the set's chunks (may
// exceed their room), [64, 65] doubles taken, cleared for each set; [66]
// slots without an entry, cleared when the host has read it
constexpr int FIX_USED = MAX_LAUNCH_CHUNKS, FIX_CLEAR = FIX_USED + 2, FIX_LOST = FIX_CLEAR, FIX_HEAD = 128;

// A chunk's part of a launch: its units of work end at `end` of the launch's
// numbering, where the next one's begin.
struct WorkRef {
   uint32_t batch, end;
};

// One work item of the matrix-core contraction (k_eco) of a row: class k,
// column tiles jt0 .. jt0 + 3 (16 columns each), contractions qb * 64 ..
struct EcoItem {
   uint16_t k, jt0, qb, pad;
};

struct EcoArgs {
   const EcoItem *items;      // the items of one row (the same for every row of the type)
   int n_items;
   const int *srcmaps;        // the type's class column maps (make_eco_plan)
   const int *src_off;        // [MAXTC] first entry of class k's map
   const int *eco_off;        // [MAXTC] class k's offset in a row of the contraction buffer
   size_t row_doubles;        // contraction buffer doubles per row
};

// Work of k_sq (kernels_sq.hpp).  A side (bra or ket) of a type is cut into
// tiles: runs of (shell pair, contraction pair) units.  A unit has the
// Hermite-expanded components of shells l1 .. l1 + l2 as its rows (ket:
// columns) before and (2 l1 + 1)(2 l2 + 1) functions after the transform.
struct SqSp {             // the units of one shell pair in a tile
   uint8_t l1, l2;
   uint8_t s1, s2;        // its shells on the two centres
   uint8_t c0, nc;        // its contraction pairs c0 .. c0 + nc - 1 (i1 n2 + i2)
   uint8_t n2;            // contractions of the second shell
   uint8_t pad;
   uint16_t row0, fn0;    // first row and function in the tile
   int16_t f1, f2;        // first function of the shells, from the start of the tile's function ranges
};
struct SqTile {
   uint16_t nrow, nfn, nrc, nsp;
   uint16_t comp0, ncomp;           // its components among the type's
   uint16_t r1, n1, r2, n2;         // its function ranges on the two centres (start, count)
   uint32_t sp, row, rc, fn;        // first entries in the tables
};
struct SqItem {           // one (bra tile, ket tile)
   uint16_t bt, kt;
   uint16_t lds_k, pad;   // its P and K blocks fit in LDS
   int32_t eco_off;       // its class's place in a row of the contraction buffer, or -1: own contraction
   int32_t o_pk, o_c;     // LDS offsets, doubles
};
constexpr int SQ_NW = 16;      // primitive quartets per window (four matrix-core steps)
constexpr int SQ_MAXROW = 80, SQ_MAXRC = 16, SQ_MAXFN = 56;   // of a tile
// LDS tables of an item, bytes: ket columns, coefficient offsets of the
// units, ket functions
constexpr int SQ_TAB_URB = 2 * SQ_MAXROW, SQ_TAB_URK = SQ_TAB_URB + 4 * SQ_MAXRC,
              SQ_TAB_FN = SQ_TAB_URK + 4 * SQ_MAXRC, SQ_TAB_BYTES = (SQ_TAB_FN + 4 * SQ_MAXFN + 15) & ~15;
struct SqArgs {
   const SqItem *items;
   const SqTile *tiles;
   const SqSp *sps;
   const uint16_t *rows;   // component (from comp0) | unit << 8
   const uint32_t *rcs;    // unit, two words: contraction of the two sets, 8 bits each;
                           // first row | first component << 8 | last + 1 << 16
   const uint32_t *fns;    // function: c | d << 8 (from the tile's ranges) | shell pair << 16
   const uint16_t *cons;   // contraction of a set (set after set): shell | contraction of it << 8
   int nitem;
   int ncon[4];            // contractions of the four sets
   int o_co;               // LDS offset, doubles, of the coefficients
};
struct SqRef {            // a chunk's part of a k_sq launch
   uint32_t batch, end;    // items
   SqArgs y;
};
struct SqPlan {
   std::vector<SqItem> items;
   std::vector<SqTile> tiles;
   std::vector<SqSp> sps;
   std::vector<uint16_t> rows, cons;
   std::vector<uint32_t> rcs, fns;
   int lm = 0;
   int nsmall = 0;         // items that need at most SQ_SMALL_LDS, the first ones
   int lds_small = 0, lds_bytes = 0;   // LDS of those and of all
   char *dev = nullptr;    // all tables on the device, one after the other
   size_t off[7] = {};
};

// the K layout of class k of group g
GINT_HDI KsGroup group_ks(const BatchDev &b, const TypePlan &tp, const GroupRec &g, int k)
{
   if (g.ksmode & KS_SETLEVEL) return ks_from_set(b.kss[g.ks], tp, k);
   return b.ksg[(size_t)g.ks + k];
}

struct KTargets {
   const double *P[2];
   double *K[2];
   int nspin;
   double hf_fac;
   double *out;   // integral output (KS_OUTPUT groups)
};

// position in a class's output block of integral (isa,isb,isc,isd) of
// contraction (ia,ib,ic,id): the reference's TRA order
GINT_HDI size_t tra_index(int ia, int isa, int ib, int isb, int ic, int isc, int id, int isd, int nlb, int nlc, int nld,
                          int nsa, int nsb, int nsc, int nsd)
{
   (void)nsa;
   return ((((((size_t)ia * nsa + isa) * nlb + ib) * nsb + isb) * nlc + ic) * nsc + isc) * (size_t)(nld * nsd) +
          (size_t)id * nsd + isd;
}

// The no-allocation executor (libgint_amd_plan_execute_noalloc) takes all
// its device scratch from one static array of NOALLOC_BYTES per GPU:
//   fix-up list                   its counters, NOALLOC_FIX entries for each chunk of a launch set
//   fix-up workspace              NOALLOC_FIX x (MAX_NCP + 16) doubles, shared by them
//   primitive blocks (ac0)        the rest, NOALLOC_AC0_BYTES
constexpr size_t NOALLOC_BYTES = 177ull << 20;
constexpr int MAX_NCP = 84 * 84;              // (e0|f0) doubles of an (f f|f f) type
constexpr size_t NOALLOC_FIX = 256;
constexpr size_t NOALLOC_OFF_FIXWS = (4 * (FIX_HEAD + FIX_WORDS * NOALLOC_FIX * MAX_LAUNCH_CHUNKS) + 255) & ~(size_t)255;
constexpr size_t NOALLOC_OFF_AC0 = NOALLOC_OFF_FIXWS + ((NOALLOC_FIX * (MAX_NCP + 16) * 8 + 255) & ~(size_t)255);
constexpr size_t NOALLOC_AC0_BYTES = NOALLOC_BYTES - NOALLOC_OFF_AC0;
static_assert(NOALLOC_AC0_BYTES >= (162ull << 20), "no-allocation scratch layout");
constexpr unsigned STATS_SLOTS = 4096;   // counter triples the kernels spread their statistics over

// address of the no-allocation scratch array on the current device, looked
// up (hipGetSymbolAddress) once per device; null if the lookup failed
void *noalloc_scratch();

// launchers (kernels.hip), asynchronous on `stream`; 0 or a negative code
// zeroes n words (a kernel, not a memset node, so that the launch sequence
// can be captured in a graph)
int launch_zero_u32(uint32_t *p, int n, void *stream);
// k_fm_r over the chunks of a list (a unit: FmLayout::NB primitive quartets),
// and the fix-up of the listed slots of the set's nbatch chunks
int launch_fm_r(const BatchDev *batches, const WorkRef *refs, int nref, uint32_t units, int nacc, size_t lds,
                const DevTables &t, const RunDev &run, void *stream);
// Hermite functions per lane that k_fm_r takes for a type of nh: 1, 3 or 8
inline int fm_nacc(int nh) { return nh <= 64 ? 1 : (nh <= 192 ? 3 : 8); }
int launch_fixup(const BatchDev *batches, int nbatch, size_t lds, const DevTables &t, const RunDev &run, uint32_t n_fix,
                 void *stream);
// the LDS layouts of a type for k_fm_r and for the fix-up
void fm_layouts(const TypePlan &tp, FmLayout &main, FmLayout &fix);
// orders 1 .. ldm of the caller's table in the order that k_fm_r reads them
constexpr int CM_PAIRS = 53;   // of the 105 coefficients, the last one with a 0
int launch_pack_c0(const double *C0, int ld_C0, int ldm, double *Cm, void *stream);
// from the chunks' blocks to K (kernels_sq.hpp)
int launch_sq(const BatchDev *batches, const SqRef *refs, int nref, uint32_t items, int lm, size_t lds,
              const DevTables &t, const RunDev &run, const KTargets &kt, void *stream);
// contraction of primitive blocks on the matrix cores (kernels_eco.hip) for
// classes with at least this many contractions
constexpr int ECO_MIN_NQ = 8;
struct EcoPlan {
   std::vector<EcoItem> items;
   std::vector<int> off;       // per class: its place in a row of the contraction buffer, or -1
   std::vector<int> info;      // [MAXTC] first entry of the class's column map, [MAXTC] off
   std::vector<int> srcmaps;   // class column -> type column
   size_t row = 0;             // doubles per row of the buffer
};
void make_eco_plan(const TypePlan &tp, const std::vector<ClassPlan> &cps, EcoPlan &ep);
void make_sq_plan(const TypePlan &tp, const EcoPlan &ep, int grp, int nspin, bool eco, SqPlan &sp);
// k_sq<4>'s items of at most this much LDS (bytes, without the coefficients)
// are launched apart: a launch takes the LDS of its largest item (48 KB of an
// (ff|ff) class), three times the mean.  64 molecules in f shells: 20.1 ->
// 17.0 ms.  Not so the other kernels, whose items come to 16.3 KB at most (20.3
// with two spins): apart they read a set quartet's blocks twice, 47.5 -> 53.2
// ms with s to f shells.
constexpr int SQ_SMALL_LDS = 18 * 1024;
// Types of at most this much LDS with the coefficients are launched apart in
// k_sq<1..3>: twelve wavefronts per CU, what the registers of k_sq<1> and <2>
// allow.  k_sq<3>'s allow eight; a line of its own there (20 KB) is no
// different, K-builds with f shells 51.4 for 51.5 ms, s to f 94.0 for 94.0.
constexpr size_t SQ_TYPE_LDS = 13 * 1024 + 256;
constexpr int SQ_GROUPS = 3;   // register groups of k_sq's items
constexpr int SQ_KERNELS = 4;  // k_sq<1..4>: s and p shells; and d; and f with a transform no larger than (dd|'s; any
int launch_eco(const BatchDev *batch, const RunDev &run, uint32_t nrow, const EcoArgs &e, void *stream);
// mixed precision: max |P| (*out, zeroed first) and the route of each set
// quartet of a chunk from its calibrated magnitude
int launch_absmax(const double *P, size_t n, unsigned long long *out, bool zero, void *stream);
int launch_mixed_flags(const BatchDev *batch, const RunDev &run, uint32_t ng, const unsigned long long *pmax, double tau,
                       unsigned long long *count, void *stream);
// D (16 x 16, row-major) = A (16 x 4) B (4 x 16) through the matrix-core
// tile the contraction uses, with its lane layout; 0 or -1
int mfma_selftest(const double *A, const double *B, double *D, int prec);
// LDS bytes of the fused kernel for a type (0 if it does not fit)
size_t fm_r_lds_bytes(const TypePlan &tp);

ClassPlan make_plan(int la, int lb, int lc, int ld);
// fills everything from nsh, l and nl
void make_type_plan(TypePlan &tp);
// item descriptors of the Hermite -> cartesian transform of a type
void make_type_items(const TypePlan &tp, std::vector<uint32_t> &items);
uint64_t class_mult(int code);
void boys_table(double *ftable);
int device_math_selftest(const double *x, const double *y, int n, double *out);

}  // namespace gint
