// rpeg_kernel_sched.h - the list scheduler of the one-plan-per-wavefront kernel (device only).
//
// A wavefront schedules one plan.  Its parts, functions of their own (inside the kernel the register allocator would
// have to find room for them among the launch record and the cost model, and spill in their loops):
//   kp_ranks        ranks of the lowered nodes
//   kp_positions    from them every node's position in the order that breaks ties
//   kp_lanes        the scheduler for graphs of at most 128 nodes: every node has a lane of its own
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
// Bound: instruction issue of one wavefront.  On gfx950 an instruction costs it ~4.4 clocks however simple, a branch
// that falls through 12, a taken one 25, a value crossing from the vector to the scalar side and back 15 more, an LDS
// read 50-64.  With every waiting node's push-backs carried out in the reference's order a decision took 1,700 clocks;
// now it takes 790-890 (28-45 nodes, one to a lane), 860-1,140 (75-107 nodes, two to a lane) and 1,290-1,470 (130 nodes
// and more, kp_list), 330-610 ns at 2.4 GHz, by how many positions are shared.
// Measured, a plan's scheduling alone on its SIMD, 150 plans in one launch, before and after: PPO (K = 4) mean 72 ->
// 41 us, slowest 133 -> 76; 161-node AC-share graphs 90 us, of 300 nodes 440 -> 228 us.
#ifndef RPEG_KERNEL_SCHED_H
#define RPEG_KERNEL_SCHED_H

#include "rpeg_kernel_eval.h"

namespace rpeg {

constexpr int KP_LANE_NODES = 128;   // largest graph of kp_lanes: beyond two nodes to a lane its decisions are the slower ones

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
__device__ inline double kp_vmax_s(double a, double uniform) {   // the second operand from the scalar registers
  double r;
  asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "s"(uniform));
  return r;
}
// mask bit of this lane ? a : b.  (Written out: of a choice between two elements of a register array the compiler makes
// an indexed load from scratch memory.)
__device__ inline uint32_t kp_sel(unsigned long long mask, uint32_t a, uint32_t b) {
  uint32_t r;
  asm("v_cndmask_b32 %0, %1, %2, %3" : "=v"(r) : "v"(b), "v"(a), "s"(mask));
  return r;
}
__device__ inline double kp_sel(unsigned long long mask, double a, double b) {
  return __hiloint2double((int)kp_sel(mask, (uint32_t)__double2hiint(a), (uint32_t)__double2hiint(b)),
                          (int)kp_sel(mask, (uint32_t)__double2loint(a), (uint32_t)__double2loint(b)));
}
__device__ inline bool kp_in(unsigned long long mask) { return __builtin_amdgcn_inverse_ballot_w64(mask); }   // this lane's bit of a uniform mask

enum KpTrace { KP_NO_TRACE = 0, KP_TIMES = 1, KP_TIMES_ORDER = 2 };   // what of the schedule is kept: nothing, start and
                                                                       // finish of every node, the dispatch order too
typedef unsigned long long mask64;

// (Pointers into LDS and into the class pool, typed as such: the functions below are not inlined, and an untyped pointer
// would make every access of theirs a flat one.)
#if defined(__HIP_DEVICE_COMPILE__)
#define KP_LDS __attribute__((address_space(3)))
#define KP_CONST __attribute__((address_space(4)))
#else
#define KP_LDS
#define KP_CONST
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

// Places of the fifth successor on of the node at level place `at`.
template <class VISIT>
__device__ inline void kp_more_places(const KpClass& T, uint32_t node, uint32_t n_succ, VISIT&& visit) {
  const KP_CONST ClassHdr* h = T.hdr();
  const uint32_t sb = T.at<uint16_t>(h->off_node + node * 8u)[0];   // (NodeRec::succ_begin)
  for (uint32_t j = 4; j < n_succ; ++j) visit(kp_scalar(T.at<uint16_t>(h->off_place)[T.at<uint16_t>(h->off_succ)[sb + j]]));
}
template <class VISIT>
__device__ inline void kp_more(const KpClass& T, const KpLds& M, uint32_t at, VISIT&& visit) {   // their positions
  const uint32_t node = kp_scalar(M.rec[at].node), ns = kp_scalar(M.rec[at].n_succ);
  kp_more_places(T, node, ns, [&](uint32_t p) { visit(kp_scalar(M.q[p])); });
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

// The class's level records go to LDS.
__device__ inline void kp_stage(const uint8_t* blob, const KpLds& M) {
  const int lane = (int)__lane_id();
  const KpClass T{kp_scalar64((uint64_t)blob)};
  const KP_CONST ClassHdr* h = T.hdr();
  const int n = (int)h->n_nodes;
  const KP_CONST uint4* src = T.at<uint4>(h->off_lrec);
  for (int v = lane; v < n; v += KE_WAVE) ((KP_LDS uint4*)M.rec)[v] = src[v];
}

// Ranks.
__device__ __attribute__((noinline)) void kp_ranks(uint64_t blob, const KpLds M) {
  const int lane = (int)__lane_id();
  const KpClass T{kp_scalar64(blob)};
  const KP_CONST ClassHdr* h = T.hdr();
  const int n = (int)h->n_nodes, n_levels = (int)h->n_levels;
  if (lane == 0) M.rank[n] = 0.0;
  kp_sync();

  // ---- ranks (scheduler.py:71-100), level by level from the nodes without successors; the record and the duration of
  // the next level are read while this one's ranks are computed (the levels follow each other in this order)
  {
    const KP_CONST uint16_t* lbeg = T.at<uint16_t>(h->off_lbeg);
    uint32_t ends = 0;
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
        if (__builtin_expect(__ballot(i < end && rec.n_succ > 4) != 0ull, 0)) {
          if (i < end && rec.n_succ > 4) {
            const uint32_t sb = T.at<uint16_t>(h->off_node + rec.node * 8u)[0];
            for (uint32_t j = 4; j < rec.n_succ; ++j) best = kp_vmax(best, M.rank[T.at<uint16_t>(h->off_place)[T.at<uint16_t>(h->off_succ)[sb + j]]]);
          }
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
  // chain inheritance (scheduler.py:367-378): the sub-nodes of one split vertex share the chain's top rank
  {
    const KP_CONST uint32_t* group = T.at<uint32_t>(h->off_group);   // GroupRec: begin | count << 16
    const KP_CONST uint16_t* gm = T.at<uint16_t>(h->off_glvl);
    for (uint32_t g = lane; g < h->n_groups; g += KE_WAVE) {
      const uint32_t begin = group[g] & 0xFFFFu, count = group[g] >> 16;
      double top = M.rank[gm[begin]];
      for (uint32_t j = 1; j < count; ++j) {
        const double r = M.rank[gm[begin + j]];
        top = r > top ? r : top;
      }
      for (uint32_t j = 0; j < count; ++j) M.rank[gm[begin + j]] = top;
    }
  }
  kp_sync();
}

// Positions: within its tie-break class a node comes behind those of larger rank.  Nodes that agree are told apart by
// their place in the order; `shared` where they are more than the node's own chain.  NW wavefronts share the nodes (the
// counting is a pass over the class for each: 34 us of one wavefront's time on a graph of 300 nodes).
template <int NW>
__device__ __attribute__((noinline)) void kp_positions(uint64_t blob, int wave, const KpLds M) {
  const int first = wave * KE_WAVE + (int)__lane_id();
  constexpr int STEP = NW * KE_WAVE;
  const KpClass T{kp_scalar64(blob)};
  const KP_CONST ClassHdr* h = T.hdr();
  const int n = (int)h->n_nodes;
  const KP_CONST uint64_t* orec = T.at<uint64_t>(h->off_orec);
  const uint64_t w0 = orec[first < n ? first : 0];   // the records by tie-break class
  {
    uint64_t w = w0;
    for (int p = first; p < n; p += STEP) {
      const uint64_t next = orec[p + STEP < n ? p + STEP : 0];
      M.rk[p] = M.rank[w & 0xFFFFu];
      w = next;
    }
  }
  kp_barrier<NW>();
  uint64_t oword = w0;
  for (int p = first; p - (int)__lane_id() < n; p += STEP) {
    const uint64_t next = orec[p + STEP < n ? p + STEP : 0];
    const bool ok = p < n;
    const double rk = M.rk[ok ? p : 0];
    const int b0 = (int)((oword >> 16) & 0xFFFFu), b1 = ok ? (int)((oword >> 32) & 0xFFFFu) : b0;
    const uint32_t chain_n = (uint32_t)(oword >> 48) & 0xFFu, chain_i = (uint32_t)(oword >> 56);
    uint32_t before = 0u, same = 0u;
    int j = b0;
    for (; j + 4 <= b1; j += 4) {   // four independent LDS reads in flight
      const double r0 = M.rk[j], r1 = M.rk[j + 1], r2 = M.rk[j + 2], r3 = M.rk[j + 3];
      before += (r0 > rk ? 1u : 0u) + (r1 > rk ? 1u : 0u) + (r2 > rk ? 1u : 0u) + (r3 > rk ? 1u : 0u);
      same += (r0 == rk ? 1u : 0u) + (r1 == rk ? 1u : 0u) + (r2 == rk ? 1u : 0u) + (r3 == rk ? 1u : 0u);
    }
    for (; j < b1; ++j) {
      const double r = M.rk[j];
      before += r > rk ? 1u : 0u;
      same += r == rk ? 1u : 0u;
    }
    const bool sh = ok && same > chain_n;
    uint32_t among = chain_i;
    if (__ballot(sh)) {
      if (sh) {
        among = 0u;
        for (int u = b0; u < p; ++u) among += M.rk[u] == rk ? 1u : 0u;
      }
    }
    const uint32_t pos = (uint32_t)b0 + before, q = pos + among;
    if (ok) {
      M.at[q] = (uint32_t)(oword & 0x3FFu) | (sh ? KP_AT_SHARED : 0u) | (same << 11) | (pos << 20);
      M.q[oword & 0xFFFFu] = (uint16_t)q;
    }
    oword = next;
  }
  if (first == 0) M.q[n] = 0xFFFFu;
  kp_barrier<NW>();
}

// A graph of at most 64 * NS nodes: the nodes are dealt to the lanes by position (q: register slot q >> 6, lane q & 63),
// so that among the waiting nodes of smallest true start time the one to dispatch is the lowest set bit of a ballot.  All
// control flow is uniform.  Returns the makespan, or -1 where nothing was ready (a cycle) or a start time was infinite.
template <int NS, int TR>
__device__ __attribute__((noinline)) double kp_lanes(uint64_t blob, uint64_t ovl_, uint64_t dpne_, const KpLds M, unsigned long long* stamp) {
  const int lane = (int)__lane_id();
  const KpClass T{kp_scalar64(blob)};
  const uint64_t ovl = kp_scalar64(ovl_), dpne = kp_scalar64(dpne_);
  const int n = (int)kp_scalar(T.hdr()->n_nodes);

  // ---- the nodes in their lanes
  double key[NS], dvc[NS], dur[NS];
  uint32_t deg[NS], res[NS], sx01[NS], sx23[NS], tie[NS], pos[NS], mate_lo[NS], mate_hi[NS];   // res: kp_reserved | place << 16 | more than four successors << 31
  mask64 rm[NS], shm[NS];                                            // waiting nodes; nodes of shared position
  mask64 any_shared = 0ull;
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    const int x = s * 64 + lane;
    const bool ok = x < n;
    const uint32_t at = M.at[ok ? x : 0];
    const LevelRec r = M.rec[kp_at_place(at)];
    sx01[s] = (uint32_t)M.q[r.succ[0]] | ((uint32_t)M.q[r.succ[1]] << 16);
    sx23[s] = (uint32_t)M.q[r.succ[2]] | ((uint32_t)M.q[r.succ[3]] << 16);
    res[s] = ok ? (kp_reserved(r.blocked, r.cond, ovl, dpne) | (kp_at_place(at) << 16) | (r.n_succ > 4 ? 0x80000000u : 0u)) : 0u;
    deg[s] = ok ? (uint32_t)r.indeg : 0xFFFFu;
    dur[s] = M.dur[r.slot];
    key[s] = 0.0;
    dvc[s] = 0.0;
    tie[s] = 0u;
    pos[s] = kp_at_pos(at);
    rm[s] = __ballot(ok && r.indeg == 0);
    shm[s] = __ballot(ok && (at & KP_AT_SHARED));
    {   // the lanes of the other nodes of equal position (all lanes, its own too, where they lie in two slots)
      const int lo = (int)kp_at_pos(at) - s * 64, hi = lo + (int)kp_at_size(at);
      mask64 g = ~0ull;
      if (lo >= 0 && hi <= 64) g = ((hi - lo > 63 ? ~0ull : (1ull << (hi - lo)) - 1ull) << lo) & ~(1ull << lane);
      mate_lo[s] = (uint32_t)g;
      mate_hi[s] = (uint32_t)(g >> 32);
    }
    any_shared |= shm[s];
  }
  // ties of the nodes without predecessors, in the reference's node order
  uint32_t ctr = 0;
  if (any_shared) {
    const KP_CONST ClassHdr* h = T.hdr();
    for (uint32_t i = 0; i < h->n_init; ++i) {
      const int x = (int)kp_scalar(M.q[T.at<uint16_t>(h->off_place)[T.at<uint16_t>(h->off_init)[i]]]);
#pragma unroll
      for (int s = 0; s < NS; ++s) tie[s] = s == (x >> 6) && lane == (x & 63) ? ctr : tie[s];
      ++ctr;
    }
  }
  if (stamp) stamp[4] = wall_clock64();

  // ---- list scheduling (scheduler.py:399-546): one node per round.  The rare cases are kept out of line: a branch that
  // falls through costs three instructions, a taken one six.
  double makespan = 0.0;
  uint32_t ghi = 0u;
  for (int done = 0; done < n; ++done) {
    double e[NS];
    uint32_t eh[NS], h = 0xFFFFFFFFu;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      e[s] = kp_vmax(key[s], dvc[s]);
      eh[s] = kp_sel(rm[s], (uint32_t)__double2hiint(e[s]), 0xFFFFFFFFu);
      h = eh[s] < h ? eh[s] : h;
    }
    // non-negative doubles order like their bit patterns: the smallest high word, then -- where the waiting nodes that
    // have it differ in the low word, which is rare: they were released by one finish, or wait for one device -- that
    ghi = kp_wave_umin(h);
    mask64 m[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) m[s] = __ballot(eh[s] == ghi);
    // (a register of the winner's slot: in a lane of m[0] slot 0's, else in a lane of m[1] slot 1's, ...)
    auto of_slot = [&](auto&& get) {
      uint32_t v = get(NS - 1);
#pragma unroll
      for (int s = NS - 2; s >= 0; --s) v = kp_sel(m[s], get(s), v);
      return v;
    };
    mask64 mw = m[NS - 1];
#pragma unroll
    for (int s = NS - 2; s >= 0; --s) mw = m[s] ? m[s] : mw;
    int wl = __builtin_ctzll(mw);
    uint32_t glo;
    {
      const uint32_t lo0 = (uint32_t)__builtin_amdgcn_readlane((int)of_slot([&](int s) { return (uint32_t)__double2loint(e[s]); }), wl);
      mask64 differ = 0ull;
      glo = lo0;
#pragma unroll
      for (int s = 0; s < NS; ++s) differ |= m[s] & __ballot((uint32_t)__double2loint(e[s]) != lo0);
      if (__builtin_expect(differ != 0ull, 0)) {
        uint32_t l = 0xFFFFFFFFu;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
          const uint32_t x = kp_sel(m[s], (uint32_t)__double2loint(e[s]), 0xFFFFFFFFu);
          l = x < l ? x : l;
        }
        glo = kp_wave_umin(l);
#pragma unroll
        for (int s = 0; s < NS; ++s) m[s] &= __ballot((uint32_t)__double2loint(e[s]) == glo);
        mw = m[NS - 1];
#pragma unroll
        for (int s = NS - 2; s >= 0; --s) mw = m[s] ? m[s] : mw;
        wl = __builtin_ctzll(mw);
      }
    }

    // ---- ties among waiting nodes of equal position, and the push-backs they depend on
    mask64 ls[NS], live_shared = 0ull;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      ls[s] = rm[s] & shm[s];
      live_shared |= ls[s];
    }
    if (__builtin_expect(live_shared != 0ull, 0)) {
      const double gk = __hiloint2double((int)ghi, (int)glo);
      // back: stale entries the heap may have met on the way (a stale entry of key gk only if its position and tie are
      // below the dispatched one's); rivals: entries of shared position that could be dispatched now
      mask64 back[NS], any_back = 0ull;
      int n_rivals = 0;
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        back[s] = ls[s] & __ballot(dvc[s] > key[s]) & __ballot(key[s] <= gk);
        any_back |= back[s];
        n_rivals += __builtin_popcountll(m[s] & ls[s]);
      }
      if (any_back != 0ull || n_rivals > 1) {
        int ws = 0;
#pragma unroll
        for (int s = NS - 1; s >= 0; --s)
          if (m[s]) ws = s;
        uint32_t pd = (uint32_t)__builtin_amdgcn_readlane((int)of_slot([&](int s) { return pos[s]; }), wl);
        if (n_rivals > 1) {
          mask64 c[NS], current[NS], any_current = 0ull;
          int members = 0;
#pragma unroll
          for (int s = 0; s < NS; ++s) {
            c[s] = m[s] & __ballot(pos[s] == pd);
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
#pragma unroll
            for (int s = 0; s < NS; ++s) m[s] = s == ws ? 1ull << wl : 0ull;
          }
        }
        mask64 level = 0ull;
        int members = 0;
        mask64 d_stale = 0ull;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
          if (s == ws) {
            d_stale = (back[s] >> wl) & 1ull;
            back[s] &= ~(1ull << wl);
          }
          level |= back[s] & __ballot(key[s] == gk);
        }
        if (__builtin_expect(level != 0ull, 0)) {
          // (a stale entry that is dispatched was pushed back with a fresh tie)
          const uint32_t td = d_stale ? 0xFFFFFFFFu : (uint32_t)__builtin_amdgcn_readlane((int)of_slot([&](int s) { return tie[s]; }), wl);
#pragma unroll
          for (int s = 0; s < NS; ++s)
            back[s] &= __ballot(key[s] < gk) | __ballot(pos[s] < pd) | (__ballot(pos[s] == pd) & __ballot(tie[s] < td));
        }
#pragma unroll
        for (int s = 0; s < NS; ++s) members += __builtin_popcountll(back[s]);
        if (members) {
          // fresh ties; only among entries of equal position is their order ever looked at
          uint32_t fresh[NS];
          mask64 mated[NS], any_mated = 0ull;
#pragma unroll
          for (int s = 0; s < NS; ++s) {
            fresh[s] = ctr;
            mated[s] = back[s] & __ballot((((uint32_t)back[s] & mate_lo[s]) | ((uint32_t)(back[s] >> 32) & mate_hi[s])) != 0u);
            any_mated |= mated[s];
          }
          if (any_mated) {
#pragma unroll
            for (int s = 0; s < NS; ++s) {
              mask64 todo = mated[s];
              while (todo) {
                const int j = __builtin_ctzll(todo);
                todo &= todo - 1ull;
                const double kj = kp_readlane(key[s], j);
                const uint32_t tj = (uint32_t)__builtin_amdgcn_readlane((int)tie[s], j);
#pragma unroll
                for (int t = 0; t < NS; ++t) fresh[t] += ((kj < key[t]) | ((kj == key[t]) & (tj < tie[t]))) ? 1u : 0u;
              }
            }
          }
#pragma unroll
          for (int s = 0; s < NS; ++s) {
            key[s] = kp_sel(back[s], dvc[s], key[s]);
            tie[s] = kp_sel(back[s], fresh[s], tie[s]);
          }
          ctr += (uint32_t)members;
        }
      }
    }

    // ---- dispatch
    double f[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) f[s] = e[s] + dur[s];
    const uint32_t flo = of_slot([&](int s) { return (uint32_t)__double2loint(f[s]); }), fhi = of_slot([&](int s) { return (uint32_t)__double2hiint(f[s]); });
    const uint32_t info = (uint32_t)__builtin_amdgcn_readlane((int)of_slot([&](int s) { return res[s]; }), wl);
    const uint32_t s01 = (uint32_t)__builtin_amdgcn_readlane((int)of_slot([&](int s) { return sx01[s]; }), wl);
    const uint32_t s23 = (uint32_t)__builtin_amdgcn_readlane((int)of_slot([&](int s) { return sx23[s]; }), wl);
    const double fin = __hiloint2double(__builtin_amdgcn_readlane((int)fhi, wl), __builtin_amdgcn_readlane((int)flo, wl));
    {
      const mask64 bit = 1ull << wl;
      mask64 left = bit;   // (of the slots that hold candidates, the first is the winner's)
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        rm[s] &= ~(s + 1 < NS && !m[s] ? 0ull : left);
        left = m[s] ? 0ull : left;
      }
      if (TR) {   // start and finish by position
        if (kp_in(bit)) {
          uint32_t q = (uint32_t)((NS - 1) * 64 + lane);
#pragma unroll
          for (int s = NS - 2; s >= 0; --s) q = kp_sel(m[s], (uint32_t)(s * 64 + lane), q);
          M.rank[q] = __hiloint2double((int)fhi, (int)flo);
          M.rk[q] = __hiloint2double((int)ghi, (int)glo);
          if (TR == KP_TIMES_ORDER) M.order[done] = (uint16_t)((info >> 16) & 0x7FFFu);
        }
      }
    }
    makespan = kp_vmax_s(makespan, fin);
    const uint32_t reserved = (info & 0xFFu) << 8;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const double r = kp_vmax_s(dvc[s], fin);
      dvc[s] = (res[s] & reserved) ? r : dvc[s];
    }
    // successors; a node whose last predecessor this was becomes ready.  (What waits for the devices of a ready node is
    // in its availability: only a node of shared position needs it in its key, and its place in the order of pushes.)
    if (__builtin_expect((s01 & 0xFFFFu) != 0xFFFFu, 1)) {
      mask64 sm[NS];
#pragma unroll
      for (int s = 0; s < NS; ++s) sm[s] = 0ull;
      auto mark = [&](const uint32_t x) {
        const mask64 bit = 1ull << (x & 63u);
#pragma unroll
        for (int s = 0; s < NS; ++s) sm[s] |= NS == 1 || s == (int)(x >> 6) ? bit : 0ull;
      };
      mark(s01 & 0xFFFFu);
      if (__builtin_expect((s01 >> 16) != 0xFFFFu, 0)) {
        mark(s01 >> 16);
        if ((s23 & 0xFFFFu) != 0xFFFFu) {
          mark(s23 & 0xFFFFu);
          if ((s23 >> 16) != 0xFFFFu) mark(s23 >> 16);
        }
        if (__builtin_expect((info & 0x80000000u) != 0u, 0)) {   // more than four successors
          kp_more(T, M, (info >> 16) & 0x7FFFu, mark);
        }
      }
      mask64 now[NS], now_shared = 0ull;
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        const double k = kp_vmax_s(key[s], fin);
        key[s] = kp_sel(sm[s], k, key[s]);
        deg[s] -= kp_in(sm[s]) ? 1u : 0u;
        now[s] = sm[s] & __ballot(deg[s] == 0u);
        rm[s] |= now[s];
        now_shared |= now[s] & shm[s];
      }
      if (__builtin_expect(now_shared != 0ull, 0)) {
        uint32_t j = 0u;
        auto push = [&](const uint32_t x) {
          const mask64 bit = 1ull << (x & 63u);
#pragma unroll
          for (int s = 0; s < NS; ++s)
            if (NS == 1 || s == (int)(x >> 6)) {
              const mask64 b = bit & now[s];
              key[s] = kp_sel(b, kp_vmax(key[s], dvc[s]), key[s]);
              tie[s] = kp_sel(b, ctr + j, tie[s]);
            }
          ++j;
        };
        push(s01 & 0xFFFFu);
        if ((s01 >> 16) != 0xFFFFu) {
          push(s01 >> 16);
          if ((s23 & 0xFFFFu) != 0xFFFFu) {
            push(s23 & 0xFFFFu);
            if ((s23 >> 16) != 0xFFFFu) push(s23 >> 16);
          }
        }
        if (info & 0x80000000u) {
          kp_more(T, M, (info >> 16) & 0x7FFFu, push);
        }
        ctr += j;
      }
    }
  }
  // (nothing was ready -- a cycle, which the class lowering flags -- or a start time was infinite: it stays so to the end)
  if (n > 0 && ghi >= 0x7FF00000u) return -1.0;
  if (TR) {   // from position to node; the dispatch order so far names places
    double tf[NS], ts[NS];
    uint32_t node[NS];
    kp_sync();
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const int x = s * 64 + lane < n ? s * 64 + lane : 0;
      tf[s] = M.rank[x];
      ts[s] = M.rk[x];
      node[s] = (uint32_t)M.rec[(res[s] >> 16) & 0x7FFFu].node;
    }
    kp_sync();
#pragma unroll
    for (int s = 0; s < NS; ++s)
      if (s * 64 + lane < n) {
        M.rank[node[s]] = tf[s];
        M.rk[node[s]] = ts[s];
      }
    if (TR == KP_TIMES_ORDER)
      for (int k = lane; k < n; k += KE_WAVE) M.order[k] = M.rec[M.order[k]].node;
    kp_sync();
  }
  return makespan;
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
  double key = inf, dvc = 0.0, dur = 0.0, dvm = 0.0;
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
      key = 0.0;
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

  double makespan = 0.0;
  uint32_t ghi = 0u;
  for (int done = 0; done < n; ++done) {
    const double e = kp_vmax(key, dvc);
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
      mask64 back = ls & __ballot(dvc > key) & __ballot(key <= gk);
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
          key = kp_sel(back, dvc, key);
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
    const double fin = kp_readlane(f, wl);
    const uint32_t rd = (uint32_t)__builtin_amdgcn_readlane((int)res, wl);
    key = kp_sel(bit, inf, key);
    word = kp_sel(bit, NONE, word);
    shl &= ~bit;
    makespan = kp_vmax_s(makespan, fin);
    {
      const double r = kp_vmax_s(dvc, fin), rm = kp_vmax_s(dvm, fin);
      dvc = (res & ((rd & 0x3F00u) << 14)) ? r : dvc;
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
      key = kp_sel(now, kp_vmax(ready, dv), key);
      dvc = kp_sel(now, dv, dvc);
      dur = kp_sel(now, du, dur);
      word = kp_sel(now, st.word, word);
      res = kp_sel(now, left, res);
      free_lanes &= ~now;
      const mask64 now_shared = now & __ballot((res & 0x80000000u) != 0u);
      if (__builtin_expect(now_shared != 0ull, 0)) {
        shl |= now_shared;
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
          kp_more_places(T, kp_scalar(M.node[place]), ns, [&](uint32_t p) {
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
              key = kp_sel(b, kp_vmax(ready2, dv2), key);
              dvc = kp_sel(b, dv2, dvc);
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
  if (n <= KP_LANE_NODES) return kp_lanes<2, TR>(b, ovl, dpne, M, stamp);
  const double ms = kp_list<TR>(b, ovl, dpne, M, stamp);
  return ms == -2.0 ? kp_plain<TR>(b, ovl, dpne, M) : ms;
}

#endif  // __HIPCC__

}  // namespace rpeg
#endif
