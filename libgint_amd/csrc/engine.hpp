// Host engine behind the libgint_* C-ABI (one object per handle, i.e. per
// OpenMP thread of the caller).  Mirrors the state and call protocol of the
// reference class libGint (reference src/libGint.h:53-229,
// src/libGint.cpp), with its own batching and device layout:
//
//  * work is grouped by quartet type (shell structure of the four sets);
//    one row per add_shell call keeps its primitive list once for every
//    class of the set quartet;
//  * the add_qrtt calls of a (set quartet, class) are compressed to offsets
//    affine in the contraction indices (or kept as an explicit list);
//  * pending work is uploaded and run when it exceeds the memory budget or
//    at dispatch / get_K, or, in plan mode, kept resident on the device and
//    run again for every new density.
#pragma once
#include <stdint.h>

#include <algorithm>
#include <array>
#include <cstring>
#include <map>
#include <unordered_map>
#include <vector>

#include "device.hpp"
#include "tcg_patches.h"

namespace gint {

// Append-only store of basis data (positions, exponents, coefficients) with
// exact deduplication: equal arrays share one copy (hash then compare; the
// reference's src/UniqueArray.cpp:60-92 trusts the hash alone).
class DataStore {
 public:
   uint32_t add(const double *v, int n);
   const std::vector<double> &data() const { return buf_; }
   uint64_t version() const { return version_; }

 private:
   std::vector<double> buf_;
   std::unordered_multimap<uint64_t, std::pair<uint32_t, int>> index_;
   uint64_t version_ = 0;
};

struct SetInfo {
   uint32_t R = 0, Z = 0;
   int np = 0;
   std::vector<int> l, nl;
   std::vector<uint32_t> K;
   int sig = -1;   // shell-structure id, -1 until needed
};

// host-side pending work of one quartet type
struct TypeQueue {
   std::vector<RowRec> rows;
   std::vector<uint32_t> prm_ip, prm_row;
   std::vector<GroupRec> groups;
   std::vector<KsGroup> ksg;
   std::vector<KsSet> kss;
   std::vector<KsRec> ksx;
   bool empty() const { return groups.empty(); }
   void release();
};

struct Chunk {
   uint32_t g0, g1, r0, r1, p0, p1;
   uint32_t s0, s1;   // its parts of set quartets in TypeDev::segs
   double k3_flops, eco_flops;
};

// The arrays of all types of a dispatch in one device allocation and one
// copy: seven to nine copies per type took most of a small dispatch (16 types
// of two or three molecules: 2.7 of 3.7 ms).  Put them, then send.  Work of
// more than MAX bytes goes array by array: there the copies are the time, and
// gathering it first would be a second one.
struct UploadArena {
   static constexpr size_t MAX = 8 << 20;
   char *dev = nullptr;
   size_t cap = 0;
   std::vector<char> host;
   std::vector<std::pair<void **, size_t>> at;   // pointers to set, offsets
   template <class T>
   void put(T *&ptr, const std::vector<T> &v)
   {
      host.resize((host.size() + 15) & ~(size_t)15);
      at.emplace_back((void **)&ptr, host.size());
      const char *p = (const char *)v.data();
      host.insert(host.end(), p, p + sizeof(T) * v.size());
   }
   void send();      // the arrays of the last send must no longer be in use
   void release();
};

// one type's work on the device
struct TypeDev {
   int type = -1;
   RowRec *rows = nullptr;
   GroupRec *groups = nullptr;
   uint32_t *prm_ip = nullptr, *prm_row = nullptr;
   KsGroup *ksg = nullptr;
   KsSet *kss = nullptr;
   KsRec *ksx = nullptr;
   SqSeg *segs = nullptr;                 // set quartets of each chunk in parts, by falling work
   uint32_t *rorder = nullptr;            // rows of each chunk by falling work (eco)
   size_t cap[9] = {};                    // allocated elements of each array
   bool ordered = false;                  // segs (and rorder) are this work's
   bool in_arena = false;                 // the arrays lie in an UploadArena, which frees them
   size_t n_rows = 0, n_groups = 0, n_prm = 0, n_ksx = 0, n_ksg = 0, n_kss = 0;
   size_t max_group_bytes = 0;            // largest set quartet's primitive blocks
   std::vector<Chunk> chunks;
   std::vector<Chunk> chunks_na;          // the same work in chunks that fit the no-allocation scratch
   bool na_fit = true;                    // every set quartet fits it
   int max_np = 1;                        // most primitives of a set
   bool used = false;                     // some set quartet has calls
   bool eco = false;                      // its contraction runs on the matrix cores
   double *gmag = nullptr;      // mixed precision: calibrated max |block element| per set quartet
   uint32_t *gflag = nullptr;   // mixed precision: route per set quartet (1 single precision)
   void release();
};

struct TypeInfo {
   std::array<int, 4> sig;
   TypePlan plan;
   UploadArena tables;                    // what the pointers to device memory below lie in
   TypePlan *d_plan = nullptr;
   std::vector<uint32_t> items;           // Hermite -> cartesian tables
   uint32_t *d_items = nullptr;
   std::vector<ClassPlan> cplans;
   // from the blocks to K: [nspin - 1][0 own contraction, 1 k_eco][register group]
   SqPlan sq[2][2][SQ_GROUPS];
   // matrix-core contraction (k_eco), for types with many primitive
   // quartets per row
   EcoPlan eco;
   int *d_srcmaps = nullptr;
   EcoItem *d_eco_items = nullptr;
   int *d_eco_info = nullptr;
};

// k_fm_r launches of a set: by the Hermite functions per lane of the types
// (fm_nacc), the largest in two lists, since a launch takes the LDS of its
// largest type and wavefronts per CU follow from it (13 to 44 KB).  A set of
// few primitive quartets does not fill the chip and pays for the launches
// instead: 5783 in 27 cells 0.69 ms in one launch, 0.9 in four.
constexpr uint64_t FM_ONE_LAUNCH = 16384;   // a set of at most this many primitive quartets: one launch
constexpr int FM_LARGE_LDS = 26 * 1024;
constexpr int FM_BUCKETS = 4;
// wavefronts that a set should give k_fm_r before one takes more than one
// primitive quartet: a K-build of 5783 takes 0.5 ms with one to a wavefront,
// 0.7 with 16; 5 million are done in 19.5 ms by sixteens, in 53.7 by twos
constexpr uint64_t FM_UNITS = 8192;

// Types of at most this many primitive quartets are not put in order: their
// kernels are over before an order shows, and it is one more copy per type.
// 64 molecules and 8 centres with s to f shells, ordered: k_eco 54.5 -> 20.2
// ms, k_sq 103 -> 93; 32 molecules 42.9 -> 40.4
constexpr size_t ORDER_MIN_PRM = 2048;
// primitive quartets of a set quartet's part, for those of more than two
// parts: a part of 256 is 16 windows, ten times its set-up and K update; with
// set quartets of up to 16384 whole, 76.5 ms for the same took 93
constexpr uint32_t SEG_PRM = 256;

// One launch of a launch set: its list of chunks among the set's tables
struct ListRef {
   size_t off = 0;       // bytes from the start of the tables
   int n = 0;
   uint32_t units = 0;   // units of work of all of them
   size_t lds = 0;       // the most LDS one needs
};
// Chunks of any types that share the work buffer and are launched together
struct LaunchSet {
   std::vector<std::pair<int, int>> chunks;   // (index among the types' devs, chunk)
   uint32_t b0 = 0;                           // first BatchDev of the set in the tables
   size_t doubles = 0;                        // of the work buffer
   size_t n_prm = 0;
   ListRef fm[FM_BUCKETS];                    // k_fm_r
   int fm_nacc[FM_BUCKETS] = {0, 0, 0, 0};
   ListRef sq[2][SQ_KERNELS][2];              // k_sq: [nspin - 1][kernel - 1][large items, small items]
   size_t fix_lds = 0;
   size_t n_fix = 0, fix_doubles = 0;         // fix-up entries; workspace of all of them
};
// The launch sequence of an execution and its tables on the device
struct LaunchPlan {
   std::vector<LaunchSet> sets;
   char *dev = nullptr;
   size_t cap = 0, ncp_max = 0, doubles = 0, n_fix = 0, fix_doubles = 0;
   bool valid = false;
   uint64_t key = 0;   // launch_key it was built for
   void release();
};

// device buffers of an execution's kernels
struct RunBufs {
   RunDev run;
   bool count;   // host counters and timing events
};

struct Timing {
   double ms[5] = {0, 0, 0, 0, 0};        // fm_r, none, sq, fixup, eco (matrix-core contraction)
   uint64_t launches[5] = {0, 0, 0, 0, 0};
   double flops[5] = {0, 0, 0, 0, 0};     // host-counted algorithmic FLOPs of sq [2] and eco [4]
};

class Engine {
 public:
   Engine();
   ~Engine();
   void init();
   void set_potential_truncated(double R_cut, const double *C0, int ld_C0, int C0_size);
   void set_hf_fac(double f) { hf_fac_ = f; }
   void set_max_mem(int max_mem_MiB);
   void set_P(const double *P, int n);
   void set_P(const double *Pa, const double *Pb, int n);
   void set_K(const double *K, int n);
   void set_K(const double *Ka, const double *Kb, int n);
   void get_K(double *K);
   void get_K(double *Ka, double *Kb);
   void set_cell(const double *h, const double *hinv);
   void set_neighs(const double *g, int n);
   void set_atom(int i, const double *R, const double *Z, int np);
   void set_atom_L(int i, int l, int nl, const double *K_normalised);
   void add_prm(int ipa, int ipb, int ipc, int ipd);
   void add_shell(int i, int j, int k, int l, int n1, int n2);
   void add_qrt(int la, int lb, int lc, int ld, int nla, int nlb, int nlc, int nld);
   void add_qrtt(double symm_fac, int la, int lb, int lc, int ld, int inla, int inlb, int inlc, int inld,
                 int ld_ac, int ld_ad, int ld_bc, int ld_bd, unsigned off_ac, unsigned off_ad, unsigned off_bc,
                 unsigned off_bd, bool Tac, bool Tad, bool Tbc, bool Tbd);
   void add_set();
   // extension: every add_qrt / add_qrtt call of the current set quartet at
   // once, for K blocks laid out per pair of sets (KsSet)
   void add_set_blocks(double symm_fac, const int ld[4], const unsigned off[4], const bool T[4]);
   // extension: integral output (the reference's TRA layout) in place of K
   void set_output(double *out, uint64_t n);
   void add_tra(int la, int lb, int lc, int ld, uint64_t dest);
   void get_output();
   void dispatch_all();
   void synchronize();

   // extensions (not in the reference ABI)
   void enable_stats(bool on) { stats_on_ = on; }
   void stats(uint64_t out[8]);
   void enable_timing(bool on) { timing_on_ = on; }
   Timing timing();
   void timing_detail(int cat, double out[256]);
   void reset_counters();
   void set_debug(int flags)
   {
      debug_ = flags;
      na_lost_new_ = true;
   }
   void set_graph(bool on) { graph_on_ = on; }
   void set_autotune(bool) {}
   void set_mixed_precision(double tau) { mixed_tau_ = tau > 0.0 ? tau : 0.0; }
   void mixed_info(double out[4]);
   // no schedule is timed any more (the kernels are chosen by a rule): the
   // classes of the plan on the workgroup kernel's own and on the matrix-core contraction
   void tune_info(double out[5]) const;
   void tune_detail(double ms[256], int pick[256]) const
   {
      for (int i = 0; i < 256; i++) {
         ms[i] = 0.0;
         pick[i] = 0;
      }
   }
   void graph_info(uint64_t out[4]) const
   {
      out[0] = graph_on_ ? 1 : 0;
      out[1] = graph_captures_;
      out[2] = graph_replays_;
      out[3] = graph_exec_ ? 1 : 0;
   }
   void plan_begin();
   void plan_end();
   void plan_execute();
   // extension: the resident plan into caller-owned device P / K, with every
   // scratch buffer in the library's static no-allocation array; 0 or < 0
   int plan_execute_noalloc(const double *Pa, const double *Pb, double *Ka, double *Kb, uint64_t n);
   void plan_clear();
   void plan_info(uint64_t out[6]);
   // serving (server.cpp)
   void use_private_stream();
   void *stream() const { return stream_; }
   uint64_t device_bytes() const;       // device memory held now (plan, work buffers, tables, basis)
   uint64_t plan_host_bytes() const;    // the evicted plan's host copy
   uint64_t work_estimate() const;      // work buffers an execution of the resident plan allocates
   uint64_t plan_max_index() const { return plan_max_index_; }
   bool plan_evicted() const { return evicted_; }
   void plan_evict();                   // plan records and work buffers off the device, host copy kept
   void plan_restore();
   void plan_execute_into(const double *P0, const double *P1, double *K0, double *K1, int nspin, uint64_t n);
   void queue_info(uint64_t out[8]);
   int queue_types(uint64_t *out, int max_types);
   int np_of(int i) const { return i < (int)sets_.size() ? sets_[i].np : 0; }
   const double *exponents_of(int i) const { return &store_.data()[sets_[i].Z]; }

 private:
   int type_of(int i, int j, int k, int l);
   int set_sig(int i);
   KsGroup compress(std::vector<KsRec> &calls, const TypePlan &tp, int k, std::vector<KsRec> &ksx);
   bool set_level(const KsGroup *g, const TypePlan &tp, KsSet &s) const;
   void upload(std::vector<TypeQueue> &qs, std::vector<TypeDev> &devs, bool release_host, UploadArena &arena);
   void execute(std::vector<TypeDev> &devs, uint64_t max_index);
   bool prepare_exec(std::vector<TypeDev> &devs, LaunchPlan &lp, uint64_t max_index, RunBufs &w, KTargets &kt, uint64_t n);
   void build_launches(std::vector<TypeDev> &devs, bool na, LaunchPlan &lp);
   void launch_all(std::vector<TypeDev> &devs, const LaunchPlan &lp, const RunBufs &w, const KTargets &kt);
   void run_set(std::vector<TypeDev> &devs, const LaunchPlan &lp, const LaunchSet &ls, const RunBufs &w, const KTargets &kt,
                bool na);
   void replay_graph(const RunBufs &w, const KTargets &kt);
   void drop_graph();
   static uint64_t graph_bits(double x)
   {
      uint64_t u;
      std::memcpy(&u, &x, 8);
      return u;
   }
   bool use_eco(const TypeInfo &ti, const TypeDev &td, bool forced) const;
   DevTables dev_tables() const;
   void ensure_work(const LaunchPlan &lp);
   void take_fix_lost(uint32_t *word);
   // what the launch lists depend on beside the work: forced contractions (the
   // static scratch's chunks are cut for the rule, so not there) and every
   // slot through the fix-up
   uint64_t launch_key(bool na) const
   {
      return na ? 0 : (uint64_t)(debug_ & 25) | (debug_ & 1 ? (uint64_t)neighs_.size() << 32 : 0);
   }
   void ensure_tables();
   void upload_data();
   void harvest_events();
   void ev_begin(int cat, void *stream);
   void ev_end(int cat, void *stream);
   void ensure_side();
   int my_thr_ = 0, nomp_ = 1;
   void *stream_ = nullptr;
   // the kernels that take the blocks to K only add into it: those of the
   // types without d shells and of the classes with f shells run on a side
   // stream, and stream_ waits for it before the blocks are overwritten
   void *side_ = nullptr;
   void *ev_join_[2] = {};   // blocks ready, side stream done

   // geometry, potential
   double cell_[18];
   std::vector<double> neighs_;
   bool truncated_ = false;
   double R_cut_ = 0.0;
   std::vector<double> C0_;
   int ld_C0_ = 0;
   int nder_ = -1;   // highest derivative order of the C0 table
   double hf_fac_ = 1.0;
   bool tables_dirty_ = true;

   // basis
   DataStore store_;
   std::vector<SetInfo> sets_;
   std::map<std::pair<std::vector<int>, std::vector<int>>, int> sig_ids_;
   std::map<std::array<int, 4>, int> type_ids_;
   std::vector<TypeInfo> types_;
   uint64_t data_version_dev_ = ~0ull;
   std::array<int, 4> last_sets_ = {-1, -1, -1, -1};
   int last_type_ = -1;

   // ingestion
   std::vector<uint32_t> prm_tmp_;
   std::vector<TypeQueue> q_;
   int cur_type_ = -1;
   std::array<int, 4> cur_sets_ = {-1, -1, -1, -1};
   std::vector<KsRec> pend_[NCLASS];
   std::vector<int> touched_;
   KsSet blocks_{};            // add_set_blocks of the open set quartet
   bool have_blocks_ = false;
   std::vector<std::pair<int, uint64_t>> pend_out_;   // (class code, destination) of the open set quartet
   double *h_out_ = nullptr;   // caller's output array (set_output)
   double *d_out_ = nullptr;
   uint64_t out_n_ = 0;
   size_t pend_bytes_ = 0;
   uint64_t max_index_ = 0;   // highest P / K element the pending calls reach
   uint64_t plan_max_index_ = 0;
   size_t budget_bytes_ = 0;
   bool recording_ = false;
   int debug_ = 0;

   // device
   std::vector<TypeDev> stream_dev_, plan_dev_;
   UploadArena stream_arena_, plan_arena_;
   LaunchPlan stream_lp_, plan_lp_, plan_na_lp_;   // the plan's with allocated and with the static scratch
   double *d_data_ = nullptr;
   size_t d_data_cap_ = 0;
   double *d_C0_ = nullptr, *d_Cm_ = nullptr;
   int cm_orders() const { return std::min(nder_, 12); }   // an (ff|ff) quartet needs order 12
   size_t cm_size() const { return (size_t)TCG_NPATCH * CM_PAIRS * 2 * cm_orders(); }
   int *d_grid_ = nullptr;
   double *d_bw_ = nullptr, *d_ftab_ = nullptr, *d_cell_ = nullptr, *d_neighs_ = nullptr;
   size_t d_neighs_cap_ = 0;
   double *d_work_ = nullptr;   // ac0 + eco of one chunk
   size_t work_bytes_ = 0;
   uint32_t *d_fix_ = nullptr;
   double *d_fix_ws_ = nullptr;
   size_t fix_cap_ = 0, fix_ws_cap_ = 0;
   void *noalloc_scratch_ = nullptr;   // this device's static scratch array (init)
   unsigned long long *d_stats_ = nullptr;   // [0..2] kernel statistics, [3] unused
   // the static scratch's lost entries to be read by the next synchronize: once
   // for a plan and its tables, since its slots do not depend on the density
   bool na_lost_new_ = true, na_lost_read_ = false;
   uint64_t fix_overflow_ = 0;                // slots without a fix-up entry so far (kept by every class)
   bool stats_on_ = false;
   uint64_t n_slots_ = 0, n_prmc_ = 0, n_q_ = 0, n_rows_ = 0;

   // P and K: shared by the team (reference src/libGint.cpp:441-447,558-562)
   int nspin_ = 0;
   size_t FP_size_ = 0;
   double *d_P_[2] = {nullptr, nullptr};
   double *d_K_[2] = {nullptr, nullptr};

   // Primitive quartets per row of a type from which k_eco contracts it.  The
   // line was put where all types of the K-builds with spdf centres gain and
   // is no crossover: that lies by the contractions.  K-build ms with k_eco
   // and with k_sq's own contraction, mean primitive quartets per row:
   //   s to f shells of 4 to 1 contractions  9: 2.8 / 2.3   28: 3.0 / 5.6
   //                                         105: 2.6 / 8.7   1059: 22.6 / 156
   //   O 3s2p1d, H 2s1p                      21: 0.66 / 0.46   129: 0.56 / 0.44
   //                                         205: 1.5 / 1.1
   //   O 4s3p2d1f, H 3s2p1d                  25: 1.6 / 1.4   102: 1.2 / 1.0
   //                                         544: 10.2 / 9.2
   static constexpr double ECO_MIN_PRM = 96.0;

   // mixed precision (plans): set quartets whose calibrated bound times
   // max |P| is below tau take the single-precision contraction
   double mixed_tau_ = 0.0;
   bool mixed_calibrated_ = false;
   unsigned long long *d_mix_ = nullptr;   // [0] max |P| bits, [1] set quartets below tau
   void ensure_mixed();

   bool own_stream_ = false;
   bool evicted_ = false;
   std::vector<TypeQueue> plan_host_;

   // the resident plan as a HIP graph (plan_execute)
   bool graph_on_ = true;
   void *graph_exec_ = nullptr;
   uint64_t graph_key_[32] = {};
   uint64_t graph_counts_[2] = {0, 0};
   double graph_flops_[2] = {0, 0};
   uint64_t graph_captures_ = 0, graph_replays_ = 0;

   bool timing_on_ = false;
   Timing timing_;
   struct EvRec {
      int cat;
      void *e0, *e1;
      int key;
   };
   int ev_key_ = 0;
   std::array<std::array<double, 256>, 5> detail_{};   // ms per category and key (type L / class code)
   std::vector<void *> ev_pool_;
   std::vector<EvRec> ev_live_;
   size_t ev_used_ = 0;
   void *ev_open_ = nullptr;
};

void fatal(const char *what, long long code);

}  // namespace gint
