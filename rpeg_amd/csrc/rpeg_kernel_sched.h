// rpeg_kernel_sched.h - the list scheduler of the one-plan-per-wavefront kernel (device only).
//
// A wavefront schedules one plan.  Its parts, functions of their own (inside the kernel the register allocator would
// have to find room for them among the launch record and the cost model, and spill in their loops):
//   kp_ranks        ranks of the lowered nodes
//   kp_positions    from them every node's position in the order that breaks ties
//   kp_lanes        the scheduler for graphs of at most 192 nodes: every node has a lane of its own, or a third of one
//   kp_list         the scheduler for larger graphs: every waiting node has a lane, the others live in LDS
//   kp_plain        the textbook form, for a graph whose waiting nodes outgrow a wavefront in kp_list
//
// Order.  The key of the reference's heap is (est, comm_prio, topo_idx, -rank, tie).  (comm_prio, topo_idx, -rank) is
// fixed once the ranks are known: the node's position.  Nodes that agree in all three share it; where they can be in the
// heap together (nodes of one quantile chain cannot: they follow each other) the position is marked `shared`.
//
// A decision.  Every node knows the availability of the devices it reserves (raised at each dispatch), so a waiting node
// knows its true start time e = max(key, availability).  The heap pops stale entries (key < e) in key order and pushes
// each back with e and a fresh tie until the minimum is current; what it then dispatches is the minimum of
// (e, position, tie).  For a node whose position no other node has, neither key nor tie of a push-back is ever looked
// at again: max(key, availability) is the same before and after it.  So push-backs are carried out only for the waiting
// nodes of shared position: those whose old (key, position, tie) is below the dispatched entry's final one take their
// true time as key and fresh ties in the order of their old (key, tie), and where several entries share the smallest
// (e, position), current ones come first, by tie, then stale ones, by old (key, tie).
//
// Bound: one wavefront's instructions, one after the other.  Measured on gfx950, clocks: a vector or scalar instruction 4.6
// where it does not need the one before it, 8.2 where it does; a step of a reduction over the lanes 16; a branch that
// falls through 12, a taken one 24; v_readlane of a lane number in a register 8.6, v_readfirstlane 4.9; a comparison to
// the scalar side and back 32; an LDS read 52.  A decision without live entries of shared position takes 310-330 clocks
// (one node to a lane), 400 (two), 600 (three) and 1,060-1,110 (kp_list); where such entries wait 100-500 more, and each
// one pushed back among others of its position 120-260.
// Before that form (a node's key and the availability of its devices kept apart, the candidates' registers selected and
// read behind the reduction, four branches): 470, 750, and kp_list beyond 128 nodes.  150 plans in one launch, a plan's
// scheduling before -> now, mean: DPO 9.4 -> 7.0 us, PPO (K = 4) of 65-128 nodes 37 -> 22, of 129-192 73 -> 48, AC-share of
// those sizes 51 -> 34 and 82 -> 65.
#ifndef RPEG_KERNEL_SCHED_H
#define RPEG_KERNEL_SCHED_H

#include "rpeg_kernel_eval.h"

namespace rpeg {

constexpr int KP_PAIR_NODES = 128;   // up to here kp_lanes has at most two nodes to a lane
constexpr int KP_LANE_NODES = 192;   // largest graph of kp_lanes: five nodes to a lane were tried, 300-node graphs 150 -> 205 us

#if defined(__HIPCC__)

template <int CTRL, int ROWS>
__device__ inline int kp_dpp(int v) { return __builtin_amdgcn_update_dpp(v, v, CTRL, ROWS, 0xF, false); }

struct KpMax { __device__ double operator()(double a, double b) const { return __builtin_fmax(a, b); } };

template <int CTRL, int ROWS, class OP>
__device__ inline double kp_step(double v, OP op) {
  const int lo = kp_dpp<CTRL, ROWS>(__double2loint(v)), hi = kp_dpp<CTRL, ROWS>(__double2hiint(v));
  return op(v, __hiloint2double(hi, lo));
}
// reduction over the 64 lanes (all must be active); the result is uniform
template <class OP>
__device__ inline double kp_wave_reduce(double v, OP op) {
  v = kp_step<0xB1, 0xF>(v, op);    // lanes 1,0,3,2 of each quad
  v = kp_step<0x4E, 0xF>(v, op);    // lanes 2,3,0,1 of each quad
  v = kp_step<0x124, 0xF>(v, op);   // row rotated by 4
  v = kp_step<0x128, 0xF>(v, op);   // row rotated by 8: every lane holds its row's result
  v = kp_step<0x142, 0xA>(v, op);   // last lane of rows 0 and 2 into rows 1 and 3
  v = kp_step<0x143, 0xC>(v, op);   // last lane of row 1 into rows 2 and 3: row 3 holds the result
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), 63), __builtin_amdgcn_readlane(__double2loint(v), 63));
}
// minimum of an unsigned word over the 64 lanes; the neutral element fills the lanes a step does not
// write, so that each step is one instruction (the lane move folds into the minimum)
template <int CTRL, int ROWS>
__device__ inline uint32_t kp_ustep(uint32_t v) {
  const uint32_t o = (uint32_t)__builtin_amdgcn_update_dpp((int)0xFFFFFFFFu, (int)v, CTRL, ROWS, 0xF, false);
  return o < v ? o : v;
}
__device__ inline uint32_t kp_wave_umin(uint32_t v) {
  v = kp_ustep<0xB1, 0xF>(v);
  v = kp_ustep<0x4E, 0xF>(v);
  v = kp_ustep<0x124, 0xF>(v);
  v = kp_ustep<0x128, 0xF>(v);
  v = kp_ustep<0x142, 0xA>(v);
  v = kp_ustep<0x143, 0xC>(v);
  return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}
__device__ inline double kp_readlane(double v, int l) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l), __builtin_amdgcn_readlane(__double2loint(v), l));
}

// max of two non-NaN doubles in one instruction (the library's fmax quiets its operands first)
__device__ inline double kp_vmax(double a, double b) {
  double r;
  asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ inline double kp_vmin(double a, double b) {   // (of a quiet NaN and a number the number)
  double r;
  asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
// the second operand from scalar registers, which no vector instruction has written in the two wait states before
__device__ inline double kp_vmax_s(double a, double uniform) {
  double r;
  asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "s"(uniform));
  return r;
}
__device__ inline bool kp_in(unsigned long long mask) { return __builtin_amdgcn_inverse_ballot_w64(mask); }   // this lane's bit of a uniform mask
// mask bit of this lane ? a : b.  (In the compiler's hands: a vector instruction that reads a mask another one has just
// written needs two wait states between them, which inline assembly does not get.)
__device__ inline uint32_t kp_sel(unsigned long long mask, uint32_t a, uint32_t b) { return kp_in(mask) ? a : b; }
__device__ inline double kp_sel(unsigned long long mask, double a, double b) {
  return __hiloint2double((int)kp_sel(mask, (uint32_t)__double2hiint(a), (uint32_t)__double2hiint(b)),
                          (int)kp_sel(mask, (uint32_t)__double2loint(a), (uint32_t)__double2loint(b)));
}
// Masks of 64 lanes by vector instructions, as two words (two 32-bit shifts: no 64-bit one whose amount could lie in the last
// register of the allocation, blocked_mask).
struct KpMask { uint32_t lo, hi; };
__device__ inline KpMask kp_bit(uint32_t l) {   // (none for 64 and more)
  const uint32_t b = 1u << (l & 31u);
  return {l < 32u ? b : 0u, l - 32u < 32u ? b : 0u};
}
__device__ inline KpMask kp_lanes_from_to(uint32_t a, uint32_t b) {   // a <= b < 64
  auto word = [](int a, int b) { return b < 0 || a > 31 ? 0u : (0xFFFFFFFFu << (a < 0 ? 0 : a)) & (0xFFFFFFFFu >> (b > 31 ? 0 : 31 - b)); };
  return {word((int)a, (int)b), word((int)a - 32, (int)b - 32)};
}
__device__ inline double kp_settled(double uniform) {   // (for kp_vmax_s)
  asm("s_nop 1" : "+s"(uniform));
  return uniform;
}
// v minus the mask's bit of this lane (the mask as the operand of kp_vmax_s)
__device__ inline uint32_t kp_dec(unsigned long long mask, uint32_t v) {
  uint32_t r;
  asm("v_subb_co_u32 %0, vcc, %1, 0, %2" : "=v"(r) : "v"(v), "s"(mask) : "vcc");
  return r;
}

enum KpTrace { KP_NO_TRACE = 0, KP_TIMES = 1, KP_TIMES_ORDER = 2 };   // what of the schedule is kept: nothing, start and
                                                                       // finish of every node, the dispatch order too
typedef unsigned long long mask64;

// (Pointers into LDS and into the class pool, typed as such: the functions below are not inlined, and an untyped pointer
// would make every access of theirs a flat one.)
#if defined(__HIP_DEVICE_COMPILE__)
#define KP_LDS __attribute__((address_space(3)))
#else
#define KP_LDS
#endif

constexpr uint32_t KP_AT_SHARED = 1u << 10;
__device__ inline uint32_t kp_at_place(uint32_t at) { return at & 0x3FFu; }
__device__ inline uint32_t kp_at_size(uint32_t at) { return (at >> 11) & 0x1FFu; }
__device__ inline uint32_t kp_at_pos(uint32_t at) { return at >> 20; }
struct KpState {        // a node's state in kp_list until it is ready
  double ready;         // largest finish time of its predecessors so far
  uint32_t left;        // predecessors to go | reserved vertices << 8 | duration slot << 14 | vertices whose allocations overlap the
                        // reserved ones << 22 | shared position << 31
  uint32_t word;        // position << 16 | level place
};
// LDS areas of the scheduler.
struct KpLds {
  const KP_LDS double* dur;   // per slot
  KP_LDS LevelRec* rec;       // by level place; in kp_list then its successor words (four to a node), then its times
  KP_LDS double* rank;        // by level place, one neutral element behind; at the end the finish times by node
  KP_LDS double* rk;          // by order place; at the end the start times by node.  (In between both are kp_list's states)
  KP_LDS uint32_t* at;        // position -> level place | shared << 10 | positions that agree << 11 | the first of them << 20 (kp_at_*)
  KP_LDS uint16_t* q;         // level place -> position, one neutral element behind
  // over the two maps, once the nodes are where the scheduler wants them:
  KP_LDS uint16_t* order;     // nodes in dispatch order (KP_TIMES_ORDER)
  KP_LDS uint16_t* node;      // level place -> node, successors of it (kp_list)
  KP_LDS uint8_t* n_succ;
};
__device__ inline uint32_t kp_scalar(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }   // a value of all lanes, in a scalar register
__device__ inline uint64_t kp_scalar64(uint64_t v) { return (uint64_t)kp_scalar((uint32_t)v) | ((uint64_t)kp_scalar((uint32_t)(v >> 32)) << 32); }

// The class tables of a blob in the constant address space.
struct KpClass {
  uint64_t base;
  template <class T>
  __device__ const KP_CONST T* at(uint32_t off) const { return (const KP_CONST T*)(base + off); }
  __device__ const KP_CONST ClassHdr* hdr() const { return at<ClassHdr>(0); }
};
// within a wavefront: what one lane wrote to LDS another may read (a wavefront's LDS instructions execute in order)
__device__ inline void kp_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
// NW wavefronts work on a plan: with one the barrier is kp_sync
template <int NW>
__device__ inline void kp_barrier() {
  if (NW == 1) kp_sync();
  else __syncthreads();
}

// Places of a node's successors, from the first-th on.
template <class VISIT>
__device__ inline void kp_more_places(const KpClass& T, uint32_t node, uint32_t first, VISIT&& visit) {
  const KP_CONST ClassHdr* h = T.hdr();
  const uint64_t rec = T.at<uint64_t>(h->off_node)[node];   // (NodeRec: succ_begin, n_succ)
  const uint32_t sb = (uint32_t)rec & 0xFFFFu, n_succ = (uint32_t)(rec >> 16) & 0xFFu;
  for (uint32_t j = first; j < n_succ; ++j) visit(kp_scalar(T.at<uint16_t>(h->off_place)[T.at<uint16_t>(h->off_succ)[sb + j]]));
}
// Reserved vertices of a node, and (second byte) the vertices whose allocations overlap one of them: its devices are busy
// until the largest finish time of the dispatched nodes whose reserved vertices meet those (the relation is symmetric).
__device__ inline uint32_t kp_reserved(uint32_t blocked, uint32_t cond, uint64_t ovl, uint64_t dpne) {
  NodeRec nr;
  nr.blocked = (uint8_t)blocked; nr.cond = (uint8_t)cond;
  const unsigned b = blocked_mask(nr, dpne);
  uint32_t touch = 0u;
#pragma unroll
  for (int v = 0; v < RPEG_MAX_V; ++v)
    if ((b >> v) & 1u) touch |= mask_row(ovl, v);
  return b | (touch << 8);
}

// What the rank pass reads of the class beside the level records, in LDS over the ranks by order place: where the levels end, the
// chains and, by level place, their members.
struct KpRankTables {
  KP_LDS uint16_t* ends;     // lbeg
  KP_LDS uint32_t* group;    // GroupRec: begin | count << 16
  KP_LDS uint16_t* member;
};
__device__ inline KpRankTables kp_rank_tables(const KpLds& M, uint32_t n_levels, uint32_t n_groups) {   // (2 n + 2, 4 n and 2 n bytes at most)
  KpRankTables t;
  t.ends = (KP_LDS uint16_t*)M.rk;
  t.group = (KP_LDS uint32_t*)(t.ends + ((n_levels + 2u) & ~1u));
  t.member = (KP_LDS uint16_t*)(t.group + n_groups);
  return t;
}
// These and the level records go to LDS.
__device__ inline void kp_stage(const uint8_t* blob, const KpLds& M) {
  const int lane = (int)__lane_id();
  const KpClass T{kp_scalar64((uint64_t)blob)};
  const KP_CONST ClassHdr* h = T.hdr();
  const int n = (int)h->n_nodes, n_levels = (int)h->n_levels, n_groups = (int)h->n_groups, n_members = (int)h->n_gmembers;
  const KP_CONST uint4* src = T.at<uint4>(h->off_lrec);
  const KP_CONST uint16_t* lbeg = T.at<uint16_t>(h->off_lbeg);
  const KP_CONST uint32_t* group = T.at<uint32_t>(h->off_group);
  const KP_CONST uint16_t* gm = T.at<uint16_t>(h->off_glvl);
  const KpRankTables t = kp_rank_tables(M, (uint32_t)n_levels, (uint32_t)n_groups);
  for (int v = lane; v - lane < n; v += KE_WAVE) {   // (one round trip for all of a stretch)
    uint4 rec;
    uint32_t g = 0u;
    uint16_t e = 0, m = 0;
    if (v < n) rec = src[v];
    if (v <= n_levels) e = lbeg[v];
    if (v < n_groups) g = group[v];
    if (v < n_members) m = gm[v];
    if (v < n) ((KP_LDS uint4*)M.rec)[v] = rec;
    if (v <= n_levels) t.ends[v] = e;
    if (v < n_groups) t.group[v] = g;
    if (v < n_members) t.member[v] = m;
  }
  if (n_levels == n && n % KE_WAVE == 0 && lane == 0) t.ends[n] = lbeg[n];   // (a chain of a whole number of wavefronts: one more end)
}

// Ranks (scheduler.py:71-100), level by level from the nodes without successors; then chain inheritance (scheduler.py:367-378):
// the sub-nodes of one split vertex share the chain's top rank.
// Bound: the latency of a level, one LDS trip for its successors' ranks.  So nothing else stands in it: records are read two levels
// ahead, durations and addresses one, lanes without a node write where nobody reads, and what only few graphs have (more than 62
// levels, a level of more than 64 nodes, a node of more than four successors) is a loop of its own.  What it reads of the class is in
// LDS before (kp_stage).  (With ballots, a duration and branches in every level, and ends, chains and their members from memory:
// PPO graphs of 82-117 nodes 6.2 us, now 4.4; AC-share of 92-300 9.0, now 7.3; 4,096 PPO plans 136 -> 130 us a step.)
__device__ __attribute__((noinline)) void kp_ranks(uint64_t blob, const KpLds M) {
  const int lane = (int)__lane_id();
  const KpClass T{kp_scalar64(blob)};
  const KP_CONST ClassHdr* h = T.hdr();
  const int n = (int)h->n_nodes, n_levels = (int)h->n_levels;
  const uint32_t n_groups = h->n_groups;
  const KpRankTables t = kp_rank_tables(M, (uint32_t)n_levels, n_groups);
  const KP_LDS uint16_t* const lbeg = t.ends;
  const KP_LDS uint32_t* const group = t.group;
  const KP_LDS uint16_t* const gm = t.member;
  KP_LDS double* const nowhere = (KP_LDS double*)M.at;   // written by lanes without a node
  constexpr int MEMBERS = 8;
  uint32_t ends = lbeg[lane + 1 <= n_levels ? lane + 1 : n_levels];   // lane l: where level l ends
  const uint32_t g0 = (uint32_t)lane < n_groups ? group[lane] : 1u << 16;
  uint32_t member[MEMBERS];
#pragma unroll
  for (int j = 0; j < MEMBERS; ++j) {   // (behind a chain's last member that one again)
    const uint32_t count = g0 >> 16;
    member[j] = n_groups ? gm[(g0 & 0xFFFFu) + ((uint32_t)j < count ? (uint32_t)j : count - 1u)] : 0u;
  }
  if (lane == 0) M.rank[n] = 0.0;
  kp_sync();
  const KP_LDS uint4* const recs = (const KP_LDS uint4*)M.rec;   // succ[0..3]; node | slot << 16 | ..; .. | n_succ << 16 | ..
  const int before = __shfl_up((int)ends, 1);
  mask64 odd = __ballot(lane < n_levels && (int)ends - (lane ? before : 0) > KE_WAVE);
  for (int i = lane; i < n; i += KE_WAVE) odd |= __ballot(((recs[i].w >> 16) & 0xFFu) > 4u);
  if (__builtin_expect(n_levels <= KE_WAVE - 2 && __ballot(odd != 0ull) == 0ull, 1)) {
    auto end_of = [&](int l) { return __builtin_amdgcn_readlane((int)ends, l); };   // (n behind the last level)
    auto at = [&](int i) { return recs[i < n ? i : n - 1]; };
    int begin = 0, end = end_of(0), end1 = end_of(1);
    uint4 rec = at(lane), rec1 = at(end + lane);
    double d = M.dur[(rec.z >> 16) & 0xFFu];
    for (int l = 0; l < n_levels; ++l) {
      const double r0 = M.rank[rec.x & 0xFFFFu], r1 = M.rank[rec.x >> 16], r2 = M.rank[rec.y & 0xFFFFu], r3 = M.rank[rec.y >> 16];
      const double d1 = M.dur[(rec1.z >> 16) & 0xFFu];
      const uint4 rec2 = at(end1 + lane);
      const int i = begin + lane, end2 = end_of(l + 2);
      *(i < end ? M.rank + i : nowhere) = d + kp_vmax(kp_vmax(r0, r1), kp_vmax(r2, r3));
      begin = end;
      end = end1;
      end1 = end2;
      rec = rec1;
      rec1 = rec2;
      d = d1;
    }
  } else {   // the record and the duration of the next level are read while this one's ranks are computed
    int i = lane;
    LevelRec rec = M.rec[i < n ? i : 0];
    double d = M.dur[rec.slot];
    for (int l = 0; l < n_levels; ++l) {
      if ((l & 63) == 0) ends = lbeg[l + lane + 1 <= n_levels ? l + lane + 1 : n_levels];
      const int end = __builtin_amdgcn_readlane((int)ends, l & 63);
      const int nx = end + lane < n ? end + lane : 0;
      const LevelRec rec2 = M.rec[nx];
      for (;;) {   // (a level of more than 64 nodes goes round more than once)
        const double r0 = M.rank[rec.succ[0]], r1 = M.rank[rec.succ[1]], r2 = M.rank[rec.succ[2]], r3 = M.rank[rec.succ[3]];
        double best = kp_vmax(kp_vmax(r0, r1), kp_vmax(r2, r3));
        if (i < end && rec.n_succ > 4) {
          const uint32_t sb = T.at<uint16_t>(h->off_node + rec.node * 8u)[0];
          for (uint32_t j = 4; j < rec.n_succ; ++j) best = kp_vmax(best, M.rank[T.at<uint16_t>(h->off_place)[T.at<uint16_t>(h->off_succ)[sb + j]]]);
        }
        if (i < end) M.rank[i] = d + best;
        i += 64;
        if (__builtin_expect(__ballot(i < end) == 0ull, 1)) break;
        rec = M.rec[i < n ? i : 0];
        d = M.dur[rec.slot];
      }
      i = end + lane;
      rec = rec2;
      d = M.dur[rec.slot];
    }
  }
  kp_sync();
  if (n_groups) {
    if ((uint32_t)lane < n_groups) {
      double r[MEMBERS], top;
#pragma unroll
      for (int j = 0; j < MEMBERS; ++j) r[j] = M.rank[member[j]];
      top = r[0];
#pragma unroll
      for (int j = 1; j < MEMBERS; ++j) top = r[j] > top ? r[j] : top;
      const uint32_t begin = g0 & 0xFFFFu, count = g0 >> 16;
      for (uint32_t j = MEMBERS; j < count; ++j) {   // (a chain of more)
        const double x = M.rank[gm[begin + j]];
        top = x > top ? x : top;
      }
#pragma unroll
      for (int j = 0; j < MEMBERS; ++j) M.rank[member[j]] = top;
      for (uint32_t j = MEMBERS; j < count; ++j) M.rank[gm[begin + j]] = top;
    }
    for (uint32_t g = (uint32_t)lane + KE_WAVE; g < n_groups; g += KE_WAVE) {   // (more chains than lanes)
      const uint32_t begin = group[g] & 0xFFFFu, count = group[g] >> 16;
      double top = M.rank[gm[begin]];
      for (uint32_t j = 1; j < count; ++j) {
        const double r = M.rank[gm[begin + j]];
        top = r > top ? r : top;
      }
      for (uint32_t j = 0; j < count; ++j) M.rank[gm[begin + j]] = top;
    }
    kp_sync();
  }
}

__device__ inline uint64_t kp_order_rec(const ClassView& cv, int place) {   // (OrderRec)
  return ((const uint64_t*)cv.orec)[place < (int)cv.h->n_nodes ? place : 0];
}
// Positions: within its tie-break class a node comes behind those of larger rank.  Nodes that agree have the same position
// and are told apart by the order in which they counted themselves there (of one chain: by their place in it); `shared`
// where they are more than the node's own chain.  NW wavefronts share the nodes.
// Bound: instruction issue.  A wavefront goes through the classes of its 64 nodes rank by rank, all lanes the same one: two
// instructions for 64 comparisons.  With the equal ranks counted along, the nodes of shared position going through their class
// once more, and every lane at its own node's class, it took twice that and more (sixteen wavefronts on a compute unit, 300
// nodes: 44 us, now 18; 92 nodes 10, now 6.  4,096 PPO plans 170 -> 165 us a step).
// w0: this lane's first record, kp_order_rec, which is fetched ahead of the ranks.
template <int NW>
__device__ __attribute__((noinline)) void kp_positions(uint64_t blob, int wave, const uint64_t w0, const KpLds M) {
  const int first = wave * KE_WAVE + (int)__lane_id();
  constexpr int STEP = NW * KE_WAVE;
  const KpClass T{kp_scalar64(blob)};
  const KP_CONST ClassHdr* h = T.hdr();
  const int n = (int)h->n_nodes;
  const KP_CONST uint64_t* orec = T.at<uint64_t>(h->off_orec);
  KP_LDS uint32_t* const count = M.at;                    // by position: the nodes that have it
  KP_LDS uint32_t* const found = (KP_LDS uint32_t*)M.rank;   // by node of this order: its position | its turn there << 10 | nodes that have it << 20 (over the ranks by level place)
  {
    uint64_t w = w0;
    for (int p = first; p < n; p += STEP) {
      const uint64_t next = orec[p + STEP < n ? p + STEP : 0];
      M.rk[p] = M.rank[w & 0xFFFFu];
      count[p] = 0u;
      w = next;
    }
  }
  kp_barrier<NW>();
  uint64_t oword = w0;
  for (int p = first; p - (int)__lane_id() < n; p += STEP) {
    const uint64_t next = orec[p + STEP < n ? p + STEP : 0];
    const bool ok = p < n;
    const double rk = M.rk[ok ? p : 0];
    const int b0 = ok ? (int)((oword >> 16) & 0xFFFFu) : n, b1 = ok ? (int)((oword >> 32) & 0xFFFFu) : n;
    const int c0 = p - (int)__lane_id(), last = c0 + KE_WAVE < n ? c0 + KE_WAVE : n;
    uint32_t pos = 0u;
    for (int b = __builtin_amdgcn_readfirstlane(b0); b < last;) {   // the classes of these lanes' nodes
      const int e = __builtin_amdgcn_readlane(b1, b < c0 ? 0 : b - c0);
      uint32_t before[2] = {(uint32_t)b, 0u};
      int j = b;
      for (; j + 8 <= e; j += 8) {
        double r[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) r[k] = M.rk[j + k];
#pragma unroll
        for (int k = 0; k < 8; ++k) before[k & 1] += r[k] > rk ? 1u : 0u;
      }
      for (; j < e; ++j) before[0] += M.rk[j] > rk ? 1u : 0u;
      pos = kp_sel(__ballot(b0 == b), before[0] + before[1], pos);
      b = e;
    }
    if (ok) found[p] = pos | (__hip_atomic_fetch_add(&count[pos], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) << 10);
    oword = next;
  }
  kp_barrier<NW>();
  for (int p = first; p < n; p += STEP) {   // (the counters make room for the map)
    const uint32_t f = found[p];
    found[p] = f | (count[f & 0x3FFu] << 20);
  }
  kp_barrier<NW>();
  oword = w0;
  for (int p = first; p < n; p += STEP) {
    const uint64_t next = orec[p + STEP < n ? p + STEP : 0];
    const uint32_t f = found[p], pos = f & 0x3FFu, same = f >> 20, chain_n = (uint32_t)(oword >> 48) & 0xFFu, chain_i = (uint32_t)(oword >> 56);
    const bool sh = same > chain_n;
    const uint32_t q = pos + (sh ? (f >> 10) & 0x3FFu : chain_i);
    M.at[q] = (uint32_t)(oword & 0x3FFu) | (sh ? KP_AT_SHARED : 0u) | (same << 11) | (pos << 20);
    M.q[oword & 0xFFFFu] = (uint16_t)q;
    oword = next;
  }
  if (first == 0) M.q[n] = 0xFFFFu;
  kp_barrier<NW>();
}

// The head of a round of kp_lanes, written out because the order of its instructions is what it costs: the smallest high word h
// over the 64 lanes (ghi), the lanes that have it (m), and the words of the lowest of them, read with the others switched
// off (v_readlane of a lane number takes twice as long); differ: lanes of m with another first word.  A step of the
// reduction needs what the step before it wrote two instructions later, a value that goes to the scalar side and back two
// as well: other work stands in between where there is some, the slots of a lane being merged (in the lanes of `pick` the
// first's words).  The lanes are all on before and after.
#define KP_DPP_QUAD1 " quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
#define KP_DPP_QUAD2 " quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
#define KP_DPP_ROR4 " row_ror:4 row_mask:0xf bank_mask:0xf\n\t"
#define KP_DPP_ROR8 " row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
#define KP_DPP_ROW15 " row_bcast:15 row_mask:0xa bank_mask:0xf\n\t"
#define KP_DPP_ROW31 " row_bcast:31 row_mask:0xc bank_mask:0xf\n\t"
struct KpHead {
  uint32_t ghi;
  mask64 m, differ;
};
__device__ inline KpHead kp_head(uint32_t h, double e, double dur, const uint32_t (&a)[7], double* f, uint32_t (&w)[7]) {   // *f = e + dur; a[1], a[2] are not read: f's words
  KpHead o;
  uint32_t t;
  double fm;
  asm("v_add_f64 %[f], %[e], %[d]\n\t"
      "s_nop 0\n\t"
      "v_min_u32_dpp %[t], %[h], %[h]" KP_DPP_QUAD1
      "s_nop 1\n\t"
      "v_min_u32_dpp %[t], %[t], %[t]" KP_DPP_QUAD2
      "s_nop 1\n\t"
      "v_min_u32_dpp %[t], %[t], %[t]" KP_DPP_ROR4
      "s_nop 1\n\t"
      "v_min_u32_dpp %[t], %[t], %[t]" KP_DPP_ROR8
      "s_nop 1\n\t"
      "v_min_u32_dpp %[t], %[t], %[t]" KP_DPP_ROW15
      "s_nop 1\n\t"
      "v_min_u32_dpp %[t], %[t], %[t]" KP_DPP_ROW31
      "s_nop 1\n\t"
      "v_readlane_b32 %[ghi], %[t], 63\n\t"
      "s_nop 1\n\t"
      "v_cmp_eq_u32 %[m], %[ghi], %[h]"
      : [t] "=&v"(t), [f] "=&v"(fm), [ghi] "=&s"(o.ghi), [m] "=&s"(o.m)
      : [h] "v"(h), [e] "v"(e), [d] "v"(dur));
  const uint32_t f0 = (uint32_t)__double2loint(fm), f1 = (uint32_t)__double2hiint(fm);
  asm("s_mov_b64 exec, %[m]\n\t"
      "v_readfirstlane_b32 %[w0], %[a0]\n\t"
      "v_readfirstlane_b32 %[w3], %[a3]\n\t"
      "v_readfirstlane_b32 %[w4], %[a4]\n\t"
      "v_cmp_ne_u32 %[differ], %[w0], %[a0]\n\t"
      "v_readfirstlane_b32 %[w1], %[a1]\n\t"
      "v_readfirstlane_b32 %[w2], %[a2]\n\t"
      "v_readfirstlane_b32 %[w5], %[a5]\n\t"
      "v_readfirstlane_b32 %[w6], %[a6]\n\t"
      "s_mov_b64 exec, -1\n\t"
      "s_nop 0"
      : [differ] "=&s"(o.differ), [w0] "=&s"(w[0]), [w1] "=&s"(w[1]), [w2] "=&s"(w[2]), [w3] "=&s"(w[3]), [w4] "=&s"(w[4]), [w5] "=&s"(w[5]), [w6] "=&s"(w[6])
      : [m] "s"(o.m), [a0] "v"(a[0]), [a1] "v"(f0), [a2] "v"(f1), [a3] "v"(a[3]), [a4] "v"(a[4]), [a5] "v"(a[5]), [a6] "v"(a[6]));
  *f = fm;
  return o;
}
__device__ inline KpHead kp_head(uint32_t h, const uint32_t (&v)[4], uint32_t (&w)[4]) {
  KpHead o;
  uint32_t t;
  asm("s_nop 1\n\t"
      "v_min_u32_dpp %[t], %[h], %[h]" KP_DPP_QUAD1
      "s_nop 1\n\t"
      "v_min_u32_dpp %[t], %[t], %[t]" KP_DPP_QUAD2
      "s_nop 1\n\t"
      "v_min_u32_dpp %[t], %[t], %[t]" KP_DPP_ROR4
      "s_nop 1\n\t"
      "v_min_u32_dpp %[t], %[t], %[t]" KP_DPP_ROR8
      "s_nop 1\n\t"
      "v_min_u32_dpp %[t], %[t], %[t]" KP_DPP_ROW15
      "s_nop 1\n\t"
      "v_min_u32_dpp %[t], %[t], %[t]" KP_DPP_ROW31
      "s_nop 1\n\t"
      "v_readlane_b32 %[ghi], %[t], 63\n\t"
      "s_nop 1\n\t"
      "v_cmp_eq_u32 %[m], %[ghi], %[h]\n\t"
      "s_mov_b64 exec, %[m]\n\t"
      "v_readfirstlane_b32 %[w3], %[v3]\n\t"
      "v_readfirstlane_b32 %[w0], %[v0]\n\t"
      "v_readfirstlane_b32 %[w1], %[v1]\n\t"
      "v_readfirstlane_b32 %[w2], %[v2]\n\t"
      "v_cmp_ne_u32 %[differ], %[w0], %[v0]\n\t"
      "s_mov_b64 exec, -1\n\t"
      "s_nop 0"
      : [t] "=&v"(t), [ghi] "=&s"(o.ghi), [m] "=&s"(o.m), [differ] "=&s"(o.differ), [w0] "=&s"(w[0]), [w1] "=&s"(w[1]), [w2] "=&s"(w[2]), [w3] "=&s"(w[3])
      : [h] "v"(h), [v0] "v"(v[0]), [v1] "v"(v[1]), [v2] "v"(v[2]), [v3] "v"(v[3]));
  return o;
}
__device__ inline KpHead kp_head(uint32_t h, mask64 pick, const uint32_t (&a)[11], const uint32_t (&b)[11], uint32_t (&v)[11], uint32_t (&w)[11]) {
  KpHead o;
  uint32_t t;
  asm("s_nop 1\n\t"
      "v_min_u32_dpp %[t], %[h], %[h]" KP_DPP_QUAD1
      "s_nop 0\n\t"
      "v_cndmask_b32 %[v0], %[b0], %[a0], %[p]\n\t"
      "v_min_u32_dpp %[t], %[t], %[t]" KP_DPP_QUAD2
      "v_cndmask_b32 %[v1], %[b1], %[a1], %[p]\n\t"
      "v_cndmask_b32 %[v2], %[b2], %[a2], %[p]\n\t"
      "v_min_u32_dpp %[t], %[t], %[t]" KP_DPP_ROR4
      "v_cndmask_b32 %[v3], %[b3], %[a3], %[p]\n\t"
      "v_cndmask_b32 %[v4], %[b4], %[a4], %[p]\n\t"
      "v_min_u32_dpp %[t], %[t], %[t]" KP_DPP_ROR8
      "v_cndmask_b32 %[v5], %[b5], %[a5], %[p]\n\t"
      "v_cndmask_b32 %[v6], %[b6], %[a6], %[p]\n\t"
      "v_min_u32_dpp %[t], %[t], %[t]" KP_DPP_ROW15
      "v_cndmask_b32 %[v7], %[b7], %[a7], %[p]\n\t"
      "v_cndmask_b32 %[v8], %[b8], %[a8], %[p]\n\t"
      "v_min_u32_dpp %[t], %[t], %[t]" KP_DPP_ROW31
      "v_cndmask_b32 %[v9], %[b9], %[a9], %[p]\n\t"
      "v_cndmask_b32 %[v10], %[b10], %[a10], %[p]\n\t"
      "v_readlane_b32 %[ghi], %[t], 63\n\t"
      "s_nop 1\n\t"
      "v_cmp_eq_u32 %[m], %[ghi], %[h]"
      : [t] "=&v"(t), [ghi] "=&s"(o.ghi), [m] "=&s"(o.m), [v0] "=&v"(v[0]), [v1] "=&v"(v[1]), [v2] "=&v"(v[2]), [v3] "=&v"(v[3]), [v4] "=&v"(v[4]),
        [v5] "=&v"(v[5]), [v6] "=&v"(v[6]), [v7] "=&v"(v[7]), [v8] "=&v"(v[8]), [v9] "=&v"(v[9]), [v10] "=&v"(v[10])
      : [h] "v"(h), [p] "s"(pick), [a0] "v"(a[0]), [a1] "v"(a[1]), [a2] "v"(a[2]), [a3] "v"(a[3]), [a4] "v"(a[4]), [a5] "v"(a[5]), [a6] "v"(a[6]),
        [a7] "v"(a[7]), [a8] "v"(a[8]), [a9] "v"(a[9]), [a10] "v"(a[10]), [b0] "v"(b[0]), [b1] "v"(b[1]), [b2] "v"(b[2]), [b3] "v"(b[3]),
        [b4] "v"(b[4]), [b5] "v"(b[5]), [b6] "v"(b[6]), [b7] "v"(b[7]), [b8] "v"(b[8]), [b9] "v"(b[9]), [b10] "v"(b[10]));
  asm("s_mov_b64 exec, %[m]\n\t"
      "v_readfirstlane_b32 %[w0], %[v0]\n\t"
      "v_readfirstlane_b32 %[w3], %[v3]\n\t"
      "v_readfirstlane_b32 %[w4], %[v4]\n\t"
      "v_cmp_ne_u32 %[differ], %[w0], %[v0]\n\t"
      "v_readfirstlane_b32 %[w1], %[v1]\n\t"
      "v_readfirstlane_b32 %[w2], %[v2]\n\t"
      "v_readfirstlane_b32 %[w5], %[v5]\n\t"
      "v_readfirstlane_b32 %[w6], %[v6]\n\t"
      "v_readfirstlane_b32 %[w7], %[v7]\n\t"
      "v_readfirstlane_b32 %[w8], %[v8]\n\t"
      "v_readfirstlane_b32 %[w9], %[v9]\n\t"
      "v_readfirstlane_b32 %[w10], %[v10]\n\t"
      "s_mov_b64 exec, -1\n\t"
      "s_nop 0"
      : [differ] "=&s"(o.differ), [w0] "=&s"(w[0]), [w1] "=&s"(w[1]), [w2] "=&s"(w[2]), [w3] "=&s"(w[3]), [w4] "=&s"(w[4]), [w5] "=&s"(w[5]),
        [w6] "=&s"(w[6]), [w7] "=&s"(w[7]), [w8] "=&s"(w[8]), [w9] "=&s"(w[9]), [w10] "=&s"(w[10])
      : [m] "s"(o.m), [v0] "v"(v[0]), [v1] "v"(v[1]), [v2] "v"(v[2]), [v3] "v"(v[3]), [v4] "v"(v[4]), [v5] "v"(v[5]), [v6] "v"(v[6]), [v7] "v"(v[7]),
        [v8] "v"(v[8]), [v9] "v"(v[9]), [v10] "v"(v[10]));
  return o;
}

// A graph of at most 64 * NS nodes: the nodes are dealt to the lanes by position (q: lane q / NS, slot q % NS), so that
// among the waiting nodes of smallest true start time the one to dispatch is in the lowest lane of a ballot, and there in
// the lowest slot.  All control flow is uniform.  Returns the makespan, or -1 where a node was never ready (a cycle) or a
// start time was infinite.
//
// What bounds it is the number of instructions of a round.  So a node has ONE time, the largest finish time of its
// predecessors and of the nodes dispatched on its devices: once the node is ready that is its true start time, and the heap's
// key is kept beside it for the nodes of shared position alone.  A dispatched node brings the lanes whose time it raises and
// the lanes of its successors as masks (three nodes to a lane: the latter from LDS, the former by their reservations), and
// the slots of a lane are merged in the waits of the reduction.  Everything that is about ties stands behind one branch.
template <int NS, int TR>
__device__ __attribute__((noinline)) double kp_lanes(uint64_t blob, uint64_t ovl_, uint64_t dpne_, const KpLds M, unsigned long long* stamp) {
  const int lane = (int)__lane_id();
  const KpClass T{kp_scalar64(blob)};
  const uint64_t ovl = kp_scalar64(ovl_), dpne = kp_scalar64(dpne_);
  const int n = (int)kp_scalar(T.hdr()->n_nodes);
  constexpr bool WIDE = NS > 2;   // the lanes of a node's successors are kept in LDS
  // ---- the nodes in their lanes
  double e[NS], dur[NS], key[NS], start[NS];
  uint32_t deg[NS], node[NS], tie[NS], pos[NS], seq[NS], res[NS];   // res: kp_reserved | q << 16
  uint32_t mate_lo[NS], mate_hi[NS];                     // the other lanes that hold nodes of equal position
  KpMask raise_lane[NS][NS], succ_lane[NS][NS];          // by slot: the lanes of the nodes whose time this one raises, and of its successors and itself
  mask64 shm[NS];                                        // nodes of shared position
  mask64 any_shared = 0ull;
  bool order_pushes = false;                             // nodes of equal position may be successors of one node
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    const int x = lane * NS + s;
    const bool ok = x < n;
    const uint32_t at = M.at[ok ? x : 0];
    const LevelRec r = M.rec[kp_at_place(at)];
    uint32_t before[4];
    auto succeeds = [&](uint32_t q) {   // (no successor: all ones)
      const KpMask b = kp_bit(ok ? q / NS : 64u);
#pragma unroll
      for (int t = 0; t < NS; ++t) {
        succ_lane[s][t].lo |= q % NS == (uint32_t)t ? b.lo : 0u;
        succ_lane[s][t].hi |= q % NS == (uint32_t)t ? b.hi : 0u;
      }
    };
#pragma unroll
    for (int t = 0; t < NS; ++t) succ_lane[s][t] = KpMask{0u, 0u};
    succeeds((uint32_t)x);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t q = M.q[r.succ[j]];
      succeeds(q);
      before[j] = j < r.n_succ ? kp_at_pos(M.at[q]) : 0xFFFFFFFFu - (uint32_t)j;
#pragma unroll
      for (int i = 0; i < j; ++i) order_pushes = order_pushes || __ballot(ok && before[i] == before[j]) != 0ull;
    }
    if (__builtin_expect(__ballot(ok && r.n_succ > 4) != 0ull, 0)) {
      order_pushes = true;
      const KP_CONST ClassHdr* h = T.hdr();
      const uint32_t sb = T.at<uint16_t>(h->off_node + r.node * 8u)[0];
      for (uint32_t j = 4; ok && j < r.n_succ; ++j) succeeds(M.q[T.at<uint16_t>(h->off_place)[T.at<uint16_t>(h->off_succ)[sb + j]]]);
    }
    res[s] = ok ? kp_reserved(r.blocked, r.cond, ovl, dpne) | ((uint32_t)x << 16) : 0u;
    node[s] = r.node;
    deg[s] = ok ? (uint32_t)r.indeg : 0xFFFFFFFFu;
    dur[s] = M.dur[r.slot];
    e[s] = start[s] = 0.0;
    key[s] = ok && r.indeg == 0 ? 0.0 : __builtin_inf();
    tie[s] = seq[s] = 0u;
    pos[s] = kp_at_pos(at);
    shm[s] = __ballot(ok && (at & KP_AT_SHARED));
    {
      const uint32_t p0 = kp_at_pos(at), p1 = p0 + kp_at_size(at);
      const KpMask g = kp_lanes_from_to(p0 / NS, (p1 > p0 ? p1 - 1u : p0) / NS), own = kp_bit((uint32_t)lane);
      mate_lo[s] = g.lo & ~own.lo;
      mate_hi[s] = g.hi & ~own.hi;
    }
    any_shared |= shm[s];
  }
  KP_LDS mask64* const row = (KP_LDS mask64*)M.rec;   // (WIDE; over the records and the ranks) by position: the lanes of the successors and the node's own
  if constexpr (WIDE) {
    kp_sync();
#pragma unroll
    for (int s = 0; s < NS; ++s)
      if (lane * NS + s < n) {
#pragma unroll
        for (int t = 0; t < NS; ++t) row[(lane * NS + s) * NS + t] = (mask64)succ_lane[s][t].lo | ((mask64)succ_lane[s][t].hi << 32);
      }
    kp_sync();
  } else {
#pragma unroll
    for (int t = 0; t < NS; ++t) {   // nodes that conflict: this one's reserved vertices among those that overlap the other's
#pragma unroll
      for (int s = 0; s < NS; ++s) raise_lane[s][t] = succ_lane[s][t];   // (the node itself among them: it has devices of its own)
#pragma unroll
      for (int v = 0; v < RPEG_MAX_V; ++v) {
        const mask64 overlaps = __ballot((res[t] >> (8 + v)) & 1u);
#pragma unroll
        for (int s = 0; s < NS; ++s) {
          raise_lane[s][t].lo |= (res[s] >> v) & 1u ? (uint32_t)overlaps : 0u;
          raise_lane[s][t].hi |= (res[s] >> v) & 1u ? (uint32_t)(overlaps >> 32) : 0u;
        }
      }
    }
  }
  mask64 twins = 0ull;   // lanes two of whose slots hold nodes of equal position (neighbours, then)
#pragma unroll
  for (int s = 0; s + 1 < NS; ++s) twins |= __ballot(pos[s] == pos[s + 1]);
  // ties of the nodes without predecessors, in the reference's node order
  uint32_t ctr = 0;   // (ties: a push's number << 8 | order among those of one push-back)
  if (any_shared) {
    const KP_CONST ClassHdr* h = T.hdr();
    for (uint32_t i = 0; i < h->n_init; ++i) {
      const uint32_t x = kp_scalar(M.q[T.at<uint16_t>(h->off_place)[T.at<uint16_t>(h->off_init)[i]]]);
#pragma unroll
      for (int s = 0; s < NS; ++s) tie[s] = (uint32_t)s == x % NS && (uint32_t)lane == x / NS ? ctr : tie[s];
      ctr += 256u;
    }
  }
  if (stamp) stamp[4] = wall_clock64();

  // ---- list scheduling (scheduler.py:399-546): one node per round.  A node waits while it has no predecessors left
  // (deg 0); dispatched, it is its own successor (deg -1)
  uint32_t ghi = 0u;
  mask64 last_m = 0ull, last_pick[NS];   // m and pick of the round before
#pragma unroll
  for (int s = 0; s < NS; ++s) last_pick[s] = 0ull;
  for (int round = 0; round < n; ++round) {
    // a lane's candidate: its waiting node of smallest start time, of several the one in the lowest slot.  Non-negative
    // doubles order like their bit patterns: the smallest high word first, then -- where the candidates that have it
    // differ in the low word, which is rare: they were released by one finish, or wait for one device -- that
    constexpr int NM = WIDE ? 4 : 3 + 4 * NS;
    uint32_t mine[NM], w[NM];   // of the lane's candidate: low word of its start time, finish time, lanes of its successors, lanes it raises (WIDE: its reservations and position); of the one to dispatch
    auto words = [&](int s, uint32_t (&x)[NM]) {
      const double f = e[s] + dur[s];
      x[0] = (uint32_t)__double2loint(e[s]);
      x[1] = (uint32_t)__double2loint(f);
      x[2] = (uint32_t)__double2hiint(f);
      if constexpr (WIDE) x[3] = res[s];
      else
#pragma unroll
      for (int t = 0; t < NS; ++t) {
        x[3 + 2 * t] = succ_lane[s][t].lo;
        x[4 + 2 * t] = succ_lane[s][t].hi;
        x[3 + 2 * NS + 2 * t] = raise_lane[s][t].lo;
        x[4 + 2 * NS + 2 * t] = raise_lane[s][t].hi;
      }
    };
    mask64 rm[NS], ls[NS], pick[NS];
    uint32_t eh[NS], h = 0xFFFFFFFFu;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      rm[s] = __ballot(deg[s] == 0u);
      eh[s] = kp_sel(rm[s], (uint32_t)__double2hiint(e[s]), 0xFFFFFFFFu);
      h = eh[s] < h ? eh[s] : h;
    }
    KpHead head;
    if constexpr (NS == 1) {
      double f;
      pick[0] = ~0ull;
      words(0, mine);
      head = kp_head(h, e[0], dur[0], mine, &f, w);
      mine[1] = (uint32_t)__double2loint(f);
      mine[2] = (uint32_t)__double2hiint(f);
    } else if constexpr (NS == 2) {
      pick[0] = rm[0] & (__ballot(e[0] <= e[1]) | ~rm[1]);
      pick[1] = ~pick[0];
      uint32_t a[NM], b[NM];
      words(0, a);
      words(1, b);
      head = kp_head(h, pick[0], a, b, mine, w);
    } else {
      double em = e[NS - 1];
      mask64 some = rm[NS - 1];
      words(NS - 1, mine);
      pick[NS - 1] = ~0ull;
#pragma unroll
      for (int s = NS - 2; s >= 0; --s) {
        const mask64 p = rm[s] & (__ballot(e[s] <= em) | ~some);
        some |= rm[s];
        if (s > 0) em = kp_sel(p, e[s], em);
        uint32_t a[NM];
        words(s, a);
#pragma unroll
        for (int k = 0; k < NM; ++k) mine[k] = kp_sel(p, a[k], mine[k]);
#pragma unroll
        for (int t = s + 1; t < NS; ++t) pick[t] &= ~p;
        pick[s] = p;
      }
      head = kp_head(h, mine, w);
    }
    ghi = head.ghi;
    mask64 rare = head.differ;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      ls[s] = rm[s] & shm[s];
      rare |= ls[s];
    }
    mask64 m = head.m;
    if (__builtin_expect(rare != 0ull, 0)) {
      // Nodes of shared position wait, or the candidates differ.  A node the last round made ready is pushed: its key is its
      // time now (the key of those that have not been ready yet is infinite), its tie the number of the push
      mask64 fresh[NS];
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        const double ew = __hiloint2double((int)eh[s], __double2loint(e[s]));   // (no number where the node does not wait)
        fresh[s] = __ballot(key[s] > ew);
        tie[s] = kp_sel(fresh[s], ctr, tie[s]);
        key[s] = kp_vmin(key[s], ew);
      }
      ctr += 256u;
      // (x[s]: met[s] the lanes of those that meet another one, of equal position, among all of them, and perhaps of others)
      auto meet = [&](const mask64 (&x)[NS], mask64 (&met)[NS]) {
        mask64 all = 0ull;
#pragma unroll
        for (int s = 0; s < NS; ++s) all |= x[s];
#pragma unroll
        for (int s = 0; s < NS; ++s) met[s] = x[s] & __ballot((((uint32_t)all & mate_lo[s]) | ((uint32_t)(all >> 32) & mate_hi[s])) != 0u);
        if (NS > 1) {   // (within a lane)
          mask64 one = 0ull, two = 0ull;
#pragma unroll
          for (int s = 0; s < NS; ++s) {
            two |= one & x[s];
            one |= x[s];
          }
#pragma unroll
          for (int s = 0; s < NS; ++s) met[s] |= x[s] & two & twins;
        }
      };
      if (__builtin_expect(order_pushes, 0)) {   // nodes of equal position among one node's successors: in their order
        mask64 x[NS], met[NS], any = 0ull;
#pragma unroll
        for (int s = 0; s < NS; ++s) x[s] = fresh[s] & shm[s];
        meet(x, met);
#pragma unroll
        for (int s = 0; s < NS; ++s) any |= met[s];
        if (any != 0ull) {
          const int ll = __builtin_ctzll(last_m);
          uint32_t v = (uint32_t)__builtin_amdgcn_readlane((int)node[0], ll);
#pragma unroll
          for (int s = 1; s < NS; ++s) {
            const uint32_t y = (uint32_t)__builtin_amdgcn_readlane((int)node[s], ll);
            v = (last_pick[s] >> ll) & 1ull ? y : v;
          }
          kp_more_places(T, v, 0u, [&](uint32_t p) {
            const uint32_t q = kp_scalar(M.q[p]);
#pragma unroll
            for (int s = 0; s < NS; ++s) tie[s] = kp_sel(q % NS == (uint32_t)s ? x[s] & (1ull << (q / NS & 63u)) : 0ull, ctr, tie[s]);
            ctr += 256u;
          });
        }
      }
      // back: stale entries -- their devices are busy beyond their key -- the heap may meet on the way; rivals: the lanes of
      // entries of the dispatched one's position that could be dispatched as well
      double gk = __hiloint2double((int)ghi, (int)w[0]);
      int wl = __builtin_ctzll(m);
      const mask64 bit = 1ull << wl;
      uint32_t w_lo = mate_lo[NS - 1], w_hi = mate_hi[NS - 1];
#pragma unroll
      for (int s = NS - 2; s >= 0; --s) {
        w_lo = kp_sel(pick[s], mate_lo[s], w_lo);
        w_hi = kp_sel(pick[s], mate_hi[s], w_hi);
      }
      mask64 rivals = m & ((mask64)(uint32_t)__builtin_amdgcn_readlane((int)w_lo, wl) | ((mask64)(uint32_t)__builtin_amdgcn_readlane((int)w_hi, wl) << 32));
      if constexpr (NS == 2) rivals |= bit & twins & ls[0] & ls[1] & __ballot(e[0] == e[1]);
      else if constexpr (NS > 2) {   // (two nodes of its lane wait, and nodes of its lane share a position)
        mask64 one = 0ull;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
          rivals |= bit & twins & one & ls[s];
          one |= ls[s];
        }
      }
      mask64 stale[NS], back[NS], any_back = 0ull;
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        stale[s] = ls[s] & __ballot(e[s] > key[s]);
        back[s] = stale[s] & __ballot(key[s] <= gk) & ~(pick[s] & bit);
        any_back |= back[s];
      }
      if ((head.differ | rivals | any_back) != 0ull) {
        mask64 d_stale = 0ull;
        if ((head.differ | rivals) != 0ull) {
          if (head.differ) {
            const uint32_t glo = kp_wave_umin(kp_sel(m, mine[0], 0xFFFFFFFFu));
            wl = __builtin_ctzll(m & __ballot(mine[0] == glo));
            gk = __hiloint2double((int)ghi, (int)glo);
          }
          int ws = 0;
#pragma unroll
          for (int s = NS - 1; s > 0; --s) ws = (pick[s] >> wl) & 1ull ? s : ws;
          uint32_t pd = (uint32_t)__builtin_amdgcn_readlane((int)pos[0], wl);
#pragma unroll
          for (int s = 1; s < NS; ++s) {
            const uint32_t x = (uint32_t)__builtin_amdgcn_readlane((int)pos[s], wl);
            pd = s == ws ? x : pd;
          }
          mask64 c[NS], current[NS], any_current = 0ull;
          int members = 0;
#pragma unroll
          for (int s = 0; s < NS; ++s) {
            back[s] = stale[s] & __ballot(key[s] <= gk);
            c[s] = rm[s] & __ballot(e[s] == gk) & __ballot(pos[s] == pd);
            members += __builtin_popcountll(c[s]);
            current[s] = c[s] & ~back[s];   // (of the entries of true start time gk the stale ones are those of a smaller key)
            any_current |= current[s];
          }
          if (members > 1) {   // current entries first, by tie; else stale ones, by old key and tie
            bool first = true;
            double bk = 0.0;
            uint32_t bt = 0u;
#pragma unroll
            for (int s = 0; s < NS; ++s) {
              mask64 todo = any_current ? current[s] : c[s];
              while (todo) {
                const int j = __builtin_ctzll(todo);
                todo &= todo - 1ull;
                const uint32_t tj = (uint32_t)__builtin_amdgcn_readlane((int)tie[s], j);
                const double kj = any_current ? 0.0 : kp_readlane(key[s], j);
                if (first || kj < bk || (kj == bk && tj < bt)) { first = false; bk = kj; bt = tj; ws = s; wl = j; }
              }
            }
            ws = (int)kp_scalar((uint32_t)ws);
            wl = (int)kp_scalar((uint32_t)wl);
          }
          m = 1ull << wl;
          any_back = 0ull;
#pragma unroll
          for (int s = 0; s < NS; ++s) {   // (its lane may have had another candidate)
            const mask64 here = s == ws ? m : 0ull;
            d_stale |= back[s] & here;
            back[s] &= ~here;
            any_back |= back[s];
            if (NS > 1) {
              uint32_t a[NM];
              words(s, a);
              pick[s] = (pick[s] & ~m) | here;
#pragma unroll
              for (int k = 1; k < NM; ++k) mine[k] = kp_sel(here, a[k], mine[k]);
            }
          }
#pragma unroll
          for (int k = 1; k < NM; ++k) w[k] = (uint32_t)__builtin_amdgcn_readlane((int)mine[k], wl);
        } else {
#pragma unroll
          for (int s = 0; s < NS; ++s) d_stale |= stale[s] & pick[s] & bit;
        }
        mask64 level = 0ull;
#pragma unroll
        for (int s = 0; s < NS; ++s) level |= back[s] & __ballot(key[s] == gk);
        if (__builtin_expect(level != 0ull, 0)) {
          // a stale entry of key gk is met only if its position and tie are below the dispatched one's (of which, if that was
          // stale, the tie is a fresh one)
          uint32_t pd = (uint32_t)__builtin_amdgcn_readlane((int)pos[0], wl), td = (uint32_t)__builtin_amdgcn_readlane((int)tie[0], wl);
#pragma unroll
          for (int s = 1; s < NS; ++s) {
            const uint32_t p = (uint32_t)__builtin_amdgcn_readlane((int)pos[s], wl), t = (uint32_t)__builtin_amdgcn_readlane((int)tie[s], wl);
            const bool here = (pick[s] >> wl) & 1ull;
            pd = here ? p : pd;
            td = here ? t : td;
          }
          td = d_stale ? 0xFFFFFFFFu : td;
          any_back = 0ull;
#pragma unroll
          for (int s = 0; s < NS; ++s) {
            back[s] &= __ballot(key[s] < gk) | __ballot(pos[s] < pd) | (__ballot(pos[s] == pd) & __ballot(tie[s] < td));
            any_back |= back[s];
          }
        }
        if (any_back != 0ull) {
          // fresh ties; only among entries of equal position is their order ever looked at.  They are pushed back in the
          // order of their old keys and ties: entries that were pushed back together the last time, and have equal keys
          // since, keep theirs (the low byte of the ties of one push-back tells it)
          uint32_t t2[NS];
          mask64 met[NS], any_met = 0ull, apart = 0ull;
          meet(back, met);
#pragma unroll
          for (int s = 0; s < NS; ++s) {
            any_met |= met[s];
            t2[s] = ctr | (tie[s] & 0xFFu);
          }
          if (any_met != 0ull) {
            double k1 = 0.0;
            uint32_t t1 = 0u;
#pragma unroll
            for (int s = NS - 1; s >= 0; --s)
              if (met[s] != 0ull) {
                const int j = __builtin_ctzll(met[s]);
                k1 = kp_readlane(key[s], j);
                t1 = (uint32_t)__builtin_amdgcn_readlane((int)tie[s], j);
              }
#pragma unroll
            for (int s = 0; s < NS; ++s) apart |= met[s] & (__ballot(key[s] != k1) | __ballot(((tie[s] ^ t1) >> 8) != 0u));
            if (apart != 0ull) {
#pragma unroll
              for (int s = 0; s < NS; ++s) t2[s] = ctr;
#pragma unroll
              for (int s = 0; s < NS; ++s) {
                mask64 todo = met[s];
                while (todo) {
                  const int j = __builtin_ctzll(todo);
                  todo &= todo - 1ull;
                  const double kj = kp_readlane(key[s], j);
                  const uint32_t tj = (uint32_t)__builtin_amdgcn_readlane((int)tie[s], j);
#pragma unroll
                  for (int t = 0; t < NS; ++t) t2[t] += ((kj < key[t]) | ((kj == key[t]) & (tj < tie[t]))) ? 1u : 0u;
                }
              }
            }
          }
#pragma unroll
          for (int s = 0; s < NS; ++s) {
            key[s] = kp_sel(kp_scalar64(back[s]), e[s], key[s]);
            tie[s] = kp_sel(kp_scalar64(back[s]), t2[s], tie[s]);
          }
          ctr += 256u;
        }
      }
    }

    // ---- dispatch
#pragma unroll
    for (int k = 1; k < NM; ++k) asm("" : "+s"(w[k]));   // (they are in scalar registers, whichever way they came)
    const double fin = __hiloint2double((int)w[2], (int)w[1]);
    last_m = m;
    mask64 sm[NS], raised[NS];
    if constexpr (WIDE) {
      const KP_LDS mask64* const r = row + (w[3] >> 16) * NS;
      mask64 x[NS];
#pragma unroll
      for (int s = 0; s < NS; ++s) x[s] = r[s];
      const uint32_t reserved = (w[3] & 0x3Fu) << 8;
#pragma unroll
      for (int s = 0; s < NS; ++s) raised[s] = __ballot((res[s] & reserved) != 0u);
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        sm[s] = kp_scalar64(x[s]);
        raised[s] |= sm[s];
      }
    } else {
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        sm[s] = (mask64)w[3 + 2 * s] | ((mask64)w[4 + 2 * s] << 32);
        raised[s] = (mask64)w[3 + 2 * NS + 2 * s] | ((mask64)w[4 + 2 * NS + 2 * s] << 32);
      }
    }
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      last_pick[s] = pick[s];
      if (TR) {   // (its finish time is the sum, again)
        const mask64 won = pick[s] & m & (0ull - m);
        start[s] = kp_sel(won, e[s], start[s]);
        if (TR == KP_TIMES_ORDER) seq[s] = kp_sel(won, (uint32_t)round, seq[s]);
      }
      deg[s] = WIDE ? deg[s] - (kp_in(sm[s]) ? 1u : 0u) : kp_dec(sm[s], deg[s]);
      e[s] = kp_sel(raised[s], kp_vmax_s(e[s], fin), e[s]);
    }
  }
  mask64 never = 0ull;
#pragma unroll
  for (int s = 0; s < NS; ++s) never |= __ballot(deg[s] != 0xFFFFFFFFu);
  if (never != 0ull || ghi >= 0x7FF00000u) return -1.0;   // (the smallest start time only grows)
  // every node raised its own time to its finish time, with the others on its devices: the makespan is the largest
  double last = e[0];
#pragma unroll
  for (int s = 1; s < NS; ++s) last = kp_vmax(last, e[s]);
  if (TR) {   // from position to node
    kp_sync();
#pragma unroll
    for (int s = 0; s < NS; ++s)
      if (lane * NS + s < n) {
        M.rank[node[s]] = start[s] + dur[s];
        M.rk[node[s]] = start[s];
        if (TR == KP_TIMES_ORDER) M.order[seq[s]] = (uint16_t)node[s];
      }
    kp_sync();
  }
  return kp_wave_reduce(last, KpMax());
}


// A graph of any size: a lane for every waiting node, whichever is free; the nodes that wait for predecessors live in LDS
// (a state of sixteen bytes, sixteen bytes of static data, four successor words).  A decision costs the same whatever
// the size of the graph: two LDS round trips (the successor words of the dispatched node, then the states of up to four
// successors side by side, each handled by the free lane that will hold it if it becomes ready), hidden behind the
// bookkeeping of the dispatch.  Availability by reserved set: lane m keeps it for the set of vertices with bit pattern m,
// a node that becomes ready takes it from there.  (`order` lies over the maps' first half, `node` over their second.)
// Returns the makespan, -1 as kp_lanes, -2 where the waiting nodes outgrew the lanes.
template <int TR>
__device__ __attribute__((noinline)) double kp_list(uint64_t blob, uint64_t ovl_, uint64_t dpne_, const KpLds M, unsigned long long* stamp) {
  const int lane = (int)__lane_id();
  const KpClass T{kp_scalar64(blob)};
  const uint64_t ovl = kp_scalar64(ovl_), dpne = kp_scalar64(dpne_);
  const int n = (int)kp_scalar(T.hdr()->n_nodes);
  KP_LDS KpState* const state = (KP_LDS KpState*)M.rank;
  KP_LDS uint32_t* const words = (KP_LDS uint32_t*)M.rec;    // successor word: place | reserved vertices << 16 | duration slot << 24, or all ones
  KP_LDS double* const times = (KP_LDS double*)M.rec;        // finish and start of a dispatched node, over its words
  constexpr uint32_t NONE = 0xFFFFFFFFu;
  const double inf = __builtin_inf();

  // ---- the nodes in LDS
  for (int p = lane; p - lane < n; p += KE_WAVE) {
    const bool ok = p < n;
    const LevelRec r = M.rec[ok ? p : 0];
    const uint32_t at = M.at[M.q[ok ? p : 0]];
    KpState st;
    st.ready = 0.0;
    const uint32_t rt = kp_reserved(r.blocked, r.cond, ovl, dpne);
    st.left = r.indeg | ((rt & 0x3Fu) << 8) | ((uint32_t)r.slot << 14) | (((rt >> 8) & 0x3Fu) << 22) | ((at & KP_AT_SHARED) << 21);
    st.word = (kp_at_pos(at) << 16) | (uint32_t)p;
    if (ok) state[p] = st;   // (the ranks are not needed any more)
  }
  kp_sync();
  for (int p = lane; p - lane < n; p += KE_WAVE) {
    const bool ok = p < n;
    const LevelRec r = M.rec[ok ? p : 0];
    uint4 w;
    auto successor = [&](int j) {
      const uint32_t sp = j < r.n_succ ? (uint32_t)r.succ[j] : (uint32_t)p;
      const uint32_t x = state[ok ? sp : 0].left;
      return j < r.n_succ ? sp | (((x >> 8) & 0x3Fu) << 16) | (((x >> 14) & 0xFFu) << 24) : NONE;
    };
    w.x = successor(0); w.y = successor(1); w.z = successor(2); w.w = successor(3);
    if (ok) {
      ((KP_LDS uint4*)words)[p] = w;   // (every lane has read its own record, and reads no other's; the maps are done with)
      M.node[p] = r.node;
      M.n_succ[p] = r.n_succ;
    }
  }
  kp_sync();
  double e = inf, key = inf, dur = 0.0, dvm = 0.0;   // e: the node's true start time (infinite: none); key: the heap's, where its position is shared
  uint32_t word = NONE, res = 0u, tie = 0u, ctr = 0u, mate_lo = 0u, mate_hi = 0u;
  // the lanes whose node shares the position of one that has just come to lane b: each other's mates from now on (of a
  // lane that has been given to another node since, a bit may be left standing: it costs time, no more)
  auto meet = [&](mask64 shared_lanes, int b) {
    const mask64 g = shared_lanes & __ballot((word >> 16) == (uint32_t)__builtin_amdgcn_readlane((int)(word >> 16), b)), bit = 1ull << b, others = g & ~bit;
    mate_lo = kp_sel(bit, (uint32_t)others, kp_sel(others, mate_lo | (uint32_t)bit, mate_lo));
    mate_hi = kp_sel(bit, (uint32_t)(others >> 32), kp_sel(others, mate_hi | (uint32_t)(bit >> 32), mate_hi));
  };
  mask64 free_lanes, shl = 0ull;   // lanes without a node; lanes whose node shares its position
  {
    const KP_CONST ClassHdr* h = T.hdr();
    const int ni = (int)kp_scalar(h->n_init);
    if (ni > 60) return -2.0;
    const bool ok = lane < ni;
    const uint32_t p = T.at<uint16_t>(h->off_place)[T.at<uint16_t>(h->off_init)[ok ? lane : 0]];
    const KpState st = state[p];
    if (ok) {
      e = key = 0.0;
      dur = M.dur[(st.left >> 14) & 0xFFu];
      word = st.word;
      res = st.left;
      tie = (uint32_t)lane;
    }
    ctr = (uint32_t)ni;
    free_lanes = ~((1ull << ni) - 1ull);
    shl = __ballot(ok && (res & 0x80000000u));
    for (mask64 todo = shl; todo; todo &= todo - 1ull) meet(shl, __builtin_ctzll(todo));
  }
  if (stamp) stamp[4] = wall_clock64();

  uint32_t ghi = 0u;
  for (int done = 0; done < n; ++done) {
    const uint32_t eh = (uint32_t)__double2hiint(e), el = (uint32_t)__double2loint(e);
    ghi = kp_wave_umin(eh);
    mask64 m = __ballot(eh == ghi);
    int wl = __builtin_ctzll(m);
    uint32_t glo = (uint32_t)__builtin_amdgcn_readlane((int)el, wl);
    if (__builtin_expect((m & (m - 1ull)) != 0ull, 1)) {
      if (__builtin_expect((m & __ballot(el != glo)) != 0ull, 0)) {
        glo = kp_wave_umin(kp_sel(m, el, NONE));
        m &= __ballot(el == glo);
      }
      const uint32_t w = kp_sel(m, word, NONE);   // (the position leads; the place behind it tells the nodes apart)
      wl = __builtin_ctzll(__ballot(w == kp_wave_umin(w)));
    }

    // ---- ties among waiting nodes of equal position, and the push-backs they depend on (as in kp_lanes)
    const mask64 ls = shl & ~free_lanes;
    if (__builtin_expect(ls != 0ull, 0)) {
      const double gk = __hiloint2double((int)ghi, (int)glo);
      mask64 back = ls & __ballot(e > key) & __ballot(key <= gk);
      const mask64 rivals = m & ls;
      if (back != 0ull || (rivals & (rivals - 1ull)) != 0ull) {
        const uint32_t pd = (uint32_t)__builtin_amdgcn_readlane((int)(word >> 16), wl), pos = word >> 16;
        if ((rivals & (rivals - 1ull)) != 0ull) {
          const mask64 c = m & __ballot(pos == pd), current = c & ~back;
          if ((c & (c - 1ull)) != 0ull) {   // current entries first, by tie; else stale ones, by old key and tie
            bool first = true;
            double bk = 0.0;
            uint32_t bt = 0u;
            mask64 todo = current ? current : c;
            while (todo) {
              const int j = __builtin_ctzll(todo);
              todo &= todo - 1ull;
              const uint32_t tj = (uint32_t)__builtin_amdgcn_readlane((int)tie, j);
              const double kj = current ? 0.0 : kp_readlane(key, j);
              if (first || kj < bk || (kj == bk && tj < bt)) { first = false; bk = kj; bt = tj; wl = j; }
            }
          }
        }
        const mask64 d_stale = (back >> wl) & 1ull;
        back &= ~(1ull << wl);
        if (__builtin_expect((back & __ballot(key == gk)) != 0ull, 0)) {
          const uint32_t td = d_stale ? NONE : (uint32_t)__builtin_amdgcn_readlane((int)tie, wl);
          back &= __ballot(key < gk) | __ballot(pos < pd) | (__ballot(pos == pd) & __ballot(tie < td));
        }
        if (back) {
          uint32_t fresh = ctr;
          mask64 todo = back & __ballot((((uint32_t)back & mate_lo) | ((uint32_t)(back >> 32) & mate_hi)) != 0u);
          while (todo) {   // (only among entries of equal position is the order of their ties ever looked at)
            const int j = __builtin_ctzll(todo);
            todo &= todo - 1ull;
            const double kj = kp_readlane(key, j);
            const uint32_t tj = (uint32_t)__builtin_amdgcn_readlane((int)tie, j);
            fresh += ((kj < key) | ((kj == key) & (tj < tie))) ? 1u : 0u;
          }
          key = kp_sel(back, e, key);
          tie = kp_sel(back, fresh, tie);
          ctr += (uint32_t)__builtin_popcountll(back);
        }
      }
    }

    // ---- dispatch: its successor words are on their way while the lanes take note of it
    uint32_t place = (uint32_t)__builtin_amdgcn_readlane((int)word, wl) & 0xFFFFu;
    place = place < (uint32_t)n ? place : (uint32_t)n - 1u;   // (a lane without a node, where nothing is ready: the class lowering flags such graphs)
    const mask64 bit = 1ull << wl;
    free_lanes |= bit;
    const uint32_t k = __builtin_amdgcn_mbcnt_hi((uint32_t)(free_lanes >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)free_lanes, 0u));
    const bool mine = kp_in(free_lanes) && k < 4u;    // this lane takes the k-th successor
    const uint32_t sw = words[place * 4u + (k & 3u)];
    const double f = e + dur;
    const double fin = kp_settled(kp_readlane(f, wl));
    const uint32_t rd = (uint32_t)__builtin_amdgcn_readlane((int)res, wl);
    e = kp_sel(bit, inf, e);
    word = kp_sel(bit, NONE, word);
    shl &= ~bit;
    {
      const double r = kp_vmax_s(e, fin), rm = kp_vmax_s(dvm, fin);
      e = (res & ((rd & 0x3F00u) << 14)) ? r : e;
      dvm = ((uint32_t)lane & ((rd >> 22) & 0x3Fu)) ? rm : dvm;
    }
    if (TR) {
      if (lane == 0) {
        times[2 * place] = fin;
        times[2 * place + 1] = __hiloint2double((int)ghi, (int)glo);
        if (TR == KP_TIMES_ORDER) M.order[done] = (uint16_t)place;
      }
    }
    const bool has = mine && sw != NONE;
    const uint32_t sp = sw & 0xFFFFu;
    if (__builtin_expect(__ballot(has) != 0ull, 1)) {
      const uint32_t spx = has ? sp : 0u;
      const KpState st = state[spx];
      const double du = M.dur[has ? sw >> 24 : 0u];
      const int from = (int)((sw >> 14) & 0xFCu);   // (any lane of the 64 where there is no successor)
      const double dv = __hiloint2double(__builtin_amdgcn_ds_bpermute(from, __double2hiint(dvm)), __builtin_amdgcn_ds_bpermute(from, __double2loint(dvm)));
      const double ready = kp_vmax_s(st.ready, fin);
      const uint32_t left = st.left - 1u;
      const mask64 now = __ballot(has && (left & 0xFFu) == 0u);
      if (has) {
        state[sp].ready = ready;
        state[sp].left = left;
      }
      e = kp_sel(now, kp_vmax(ready, dv), e);
      dur = kp_sel(now, du, dur);
      word = kp_sel(now, st.word, word);
      res = kp_sel(now, left, res);
      free_lanes &= ~now;
      const mask64 now_shared = now & __ballot((res & 0x80000000u) != 0u);
      if (__builtin_expect(now_shared != 0ull, 0)) {
        shl |= now_shared;
        key = kp_sel(now, e, key);
        tie = kp_sel(now, ctr + k, tie);
        ctr += 4u;
        for (mask64 todo = now_shared; todo; todo &= todo - 1ull) meet(shl, __builtin_ctzll(todo));
      }
      if (__builtin_expect(__builtin_popcountll(free_lanes) < 4, 0)) {
        if (done + 1 < n) return -2.0;
      }
      // more than four successors: one after the other, each to the first free lane
      if (__builtin_expect((__ballot(has && k == 3u)) != 0ull, 0)) {
        const uint32_t ns = kp_scalar(M.n_succ[place]);
        if (ns > 4u) {
          bool full = false;
          kp_more_places(T, kp_scalar(M.node[place]), 4u, [&](uint32_t p) {
            const KpState s2 = state[p];
            const double ready2 = kp_vmax_s(s2.ready, fin);
            const uint32_t left2 = s2.left - 1u;
            const int from2 = (int)(((s2.left >> 8) & 0x3Fu) << 2);
            const double dv2 = __hiloint2double(__builtin_amdgcn_ds_bpermute(from2, __double2hiint(dvm)), __builtin_amdgcn_ds_bpermute(from2, __double2loint(dvm)));
            kp_sync();
            if (lane == 0) { state[p].ready = ready2; state[p].left = left2; }
            kp_sync();
            if ((kp_scalar(left2) & 0xFFu) == 0u) {
              if (!free_lanes) { full = true; return; }
              const mask64 b = free_lanes & (0ull - free_lanes);
              e = kp_sel(b, kp_vmax(ready2, dv2), e);
              key = kp_sel(b, e, key);
              dur = kp_sel(b, M.dur[(s2.left >> 14) & 0xFFu], dur);
              word = kp_sel(b, s2.word, word);
              res = kp_sel(b, left2, res);
              tie = kp_sel(b, ctr, tie);
              ++ctr;
              free_lanes &= ~b;
              if (kp_scalar(left2) & 0x80000000u) {
                shl |= b;
                meet(shl, __builtin_ctzll(b));
              }
            }
          });
          if (full || (__builtin_popcountll(free_lanes) < 4 && done + 1 < n)) return -2.0;
        }
      }
    }
  }
  if (n > 0 && ghi >= 0x7FF00000u) return -1.0;
  const double makespan = kp_readlane(dvm, 63);   // (the set of all vertices: every node reserves one)
  if (TR) {   // from place to node; the states are not needed any more
    kp_sync();
    for (int p = lane; p < n; p += KE_WAVE) {
      const uint32_t node = M.node[p];
      M.rank[node] = times[2 * p];
      M.rk[node] = times[2 * p + 1];
    }
    if (TR == KP_TIMES_ORDER)
      for (int k = lane; k < n; k += KE_WAVE) M.order[k] = M.node[M.order[k]];
    kp_sync();
  }
  return makespan;
}

// The scheduler in its plain form (list_schedule of rpeg_class.h, the function the host build runs too) on LDS arrays, all
// lanes doing the same: where more than sixty nodes wait at once (horizons of dozens of steps).
struct KpPlainMem {
  const KP_LDS double* d;
  KP_LDS double *t, *r, *f, *s;    // ready time and rank; finish and start by node
  KP_LDS uint16_t *rd, *ord;
  KP_LDS uint8_t* deg;
  int seq;
  bool with_order;
  __device__ KP_LDS double& time(int i) { return t[i]; }
  __device__ KP_LDS double& rank(int i) { return r[i]; }
  __device__ KP_LDS uint8_t& indeg(int i) { return deg[i]; }
  __device__ double dur(int k) const { return d[k]; }
  __device__ KP_LDS uint16_t& rd_node(int j) { return rd[j]; }
  __device__ void on_schedule(int v, double start, double fin) {
    f[v] = fin;
    s[v] = start;
    if (with_order) ord[seq] = (uint16_t)v;
    ++seq;
  }
};
template <int TR>
__device__ __attribute__((noinline)) double kp_plain(uint64_t blob, uint64_t ovl_, uint64_t dpne_, const KpLds M) {
  const ClassView cv = class_view((const uint8_t*)kp_scalar64(blob));
  const uint64_t ovl = kp_scalar64(ovl_), dpne = kp_scalar64(dpne_);
  const int n = (int)cv.h->n_nodes;
  KpPlainMem mem;
  mem.d = M.dur;
  mem.t = (KP_LDS double*)M.rec; mem.r = mem.t + n;
  mem.f = M.rank; mem.s = M.rk;
  mem.rd = M.node; mem.ord = M.order;
  mem.deg = M.n_succ;
  mem.seq = 0;
  mem.with_order = TR == KP_TIMES_ORDER;
  uint8_t rows[RPEG_MAX_V];
  for (int x = 0; x < RPEG_MAX_V; ++x) rows[x] = (uint8_t)mask_row(ovl, x);
  bool error = false;
  const double ms = list_schedule(cv, mem, rows, dpne, RPEG_MAX_V, n + 1, &error);
  kp_sync();
  return error ? -1.0 : ms;
}

// The schedule of a plan whose nodes have their positions, on this wavefront: makespan, or a negative number where there
// is none.
template <int TR>
__device__ inline double kp_schedule(const uint8_t* blob, int n, uint64_t ovl, uint64_t dpne, const KpLds& M, unsigned long long* stamp) {
  const uint64_t b = (uint64_t)blob;
  if (n <= 64) return kp_lanes<1, TR>(b, ovl, dpne, M, stamp);
  if (n <= KP_PAIR_NODES) return kp_lanes<2, TR>(b, ovl, dpne, M, stamp);
  if (n <= KP_LANE_NODES) return kp_lanes<3, TR>(b, ovl, dpne, M, stamp);
  const double ms = kp_list<TR>(b, ovl, dpne, M, stamp);
  return ms == -2.0 ? kp_plain<TR>(b, ovl, dpne, M) : ms;
}

#endif  // __HIPCC__

}  // namespace rpeg
#endif
