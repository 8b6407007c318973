// rpeg_kernel_quad.h - two or four lanes per plan, 32 or 16 plans of one class per wavefront (device only).
//
// The kernel of large batches.  The ready set of a plan lives in the REGISTERS of its QL lanes, SL entries each
// (two, four or six, by what the class needs), unordered.  An entry:
//
//   e     true start time: the larger of the node's key and the availability of the devices it reserves, raised at every
//         dispatch that reserves one of them
//   key   the key the reference's heap holds for it, where its position is shared (below); KQ_NO_TIME elsewhere
//   word  position << 16 | tie
//   meta  node id | duration slot | reserved vertices | vertices whose allocations overlap those
//
// Order.  The heap's key is (est, comm_prio, topo_idx, -rank, tie) (scheduler.py:427); (comm_prio, topo_idx, -rank) is
// replaced by the node's position, equal for nodes that agree in all three.  The heap pops stale entries (key < e) in key
// order and pushes each back with e and a fresh tie (scheduler.py:437-443) until the minimum is current: what it then
// dispatches is the minimum of (e, position, tie).  Where no other node has a node's position, neither key nor tie of its
// push-backs is ever looked at: they are not carried out.  For shared positions they are: first the entries with a key
// below the smallest e (all of them stale) -- those that meet no other of their position side by side, the others one
// after the other in the heap's order --, then, at that key, the stale ones whose (position, tie) is below the dispatched
// one's.
//
// So every plan of a wavefront dispatches one node per round, and all of them end together: a class has one node count.
// (With every push-back carried out a round lasted as long as that of the plan with the most of them.)
//
// Per-plan state in LDS, interleaved by plan: a word of position, sharing and predecessors to go per node; the ready times
// of nodes with several predecessors, in rows that later nodes take over (QuadRec); durations by slot; reservations by
// type; availability by vertex.  What is the same for all plans comes with the successor's place (QuadRec).  A round is
// three LDS trips: the successors' places and the duration of the dispatched node; the state of up to four successors, each
// looked at by a lane that has room for it; the availability of their vertices.
//
// A plan with more entries ready at once than its lanes hold is not evaluated here: it is flagged (EvalLaunch::limit)
// and redone by the launch that ends the call, a plan per wavefront.  Its class then reports one entry more than there was
// room for (EvalLaunch::cneed), and the next call gives it the form above: without that a class stayed where it was and
// its plans were redone in every call (20,011 PPO plans, forms learned from other plans: 25 of them, 452 us a step; now
// 384).  Ranks go level by level with a node per lane of the plan, all plans together (kq_ranks).  A node's id is its place by tie-break class, so that
// counting the larger ranks of its class walks through consecutive rows.
//
// Bound: vector issue and, with few wavefronts in flight, the latency of a round (four lanes of four entries: 114 vector
// instructions in a round that looks at its successors once and files some, 47 more where entries are pushed back; some 360 at
// first, then 270).  LDS bounds the wavefronts in flight: sixteen plans of 85 nodes and 40 slots take 13 KiB, 3 per
// SIMD (with a ready time, a word and an in-degree per node and plan, and all plans' ranks at once, 26 KiB and 1.5; 300
// nodes 28 against 70 KiB).
// Scheduling a wavefront: 42-node GRPO class 60 us, 92 nodes 130-190, 28-node DPO class 35.  The step, with the larger state
// against now: 131,072 GRPO plans 568 -> 486 us, 20,011 PPO plans 366 -> 320, 60,000 761 -> 578, 131,072 1,442 -> 1,075,
// 1,048,576 DPO plans 1,187 -> 1,015; GRPO 17,000 and 65,536 and DPO 65,536 within 8 %.
#ifndef RPEG_KERNEL_QUAD_H
#define RPEG_KERNEL_QUAD_H

#include "rpeg_kernel_eval.h"
#include "rpeg_kernel_sched.h"

namespace rpeg {

// Ties are counted for all plans of a wavefront together: a round takes one for its entries alone in their position, one for each of up to
// 24 others below the smallest start time and as many at it, and a lane each for successors that became ready, once for every node of
// every plan at most: 512 x 49 + 64 x 512 < 2^16.
constexpr uint32_t KQ_TIE_BITS = 16, KQ_TIE_MASK = (1u << KQ_TIE_BITS) - 1u;
constexpr uint32_t KQ_EMPTY = 0xFFFFFFFFu;
// High word of the times of a slot without an entry, whatever the low one is: larger than any start time that is evaluated here
// (a plan with a larger one is flagged and redone by the launch that ends the call).
constexpr uint32_t KQ_NO_TIME = 0x7FEFFFFFu;

// Positions are found for 1 / parts of a wavefront's plans at a time: all at once, or half or a quarter with two lanes a plan, a
// quarter or an eighth with four.
__host__ __device__ constexpr uint32_t kq_parts_least(uint32_t lanes) { return lanes == 2 ? 2u : 4u; }
// Graphs of up to this many nodes have their equal ranks counted along with the larger ones, larger graphs afterwards, by
// position: along, every pair of a class costs two instructions more, afterwards every node 25 and three LDS trips, and
// classes grow with the graph.  (Afterwards / along, us a step: 65,536 GRPO plans of 51 nodes 322 / 315, 65,536 DPO plans of 28
// 163 / 156; 65,536 AC-share plans of 152 1,520 / 1,625, 131,072 PPO plans of 98 1,010 / 1,045.)
constexpr int KQ_EQ_NODES = 60;
// What a launch's LDS is sized for: the largest of its classes in each respect.
struct QuadSize {
  uint32_t nodes = 0, slots = 0, rows = 0, types = 0, ranks = 0;   // (ranks: rows of the rank pass)
  uint32_t parts = 4;
  __host__ __device__ void fit(const QuadSize& o) {
    nodes = o.nodes > nodes ? o.nodes : nodes; slots = o.slots > slots ? o.slots : slots;
    rows = o.rows > rows ? o.rows : rows; types = o.types > types ? o.types : types;
    ranks = o.ranks > ranks ? o.ranks : ranks;
  }
};
// LDS of one wavefront.  Class tables: per node four successor words, its own, its level place's id and its place in its chain.
// Per plan [row][plan]: durations, availability by vertex with a row of zeros and one nobody reads, ready-time
// rows -- over these two, before they are needed, the rows and records of the rank pass, then the ranks of the plans whose
// positions are being found --, with the critical-chain masses finish
// and start times, a state word and a reservation each.
__host__ __device__ inline size_t kq_tab_bytes(uint32_t nodes) { return (20ull * nodes + 2 * 2ull * (nodes + 2) + 15) & ~size_t(15); }
__host__ __device__ inline size_t kq_union_bytes(uint32_t plans, const QuadSize& z) {
  const size_t rows = 8ull * plans * (z.rows + RPEG_MAX_V + 2), part = 8ull * (plans / z.parts) * (z.nodes + 1ull),
               ranks = z.parts == 1 ? 0 : 8ull * plans * z.ranks + sizeof(RankRec) * (z.nodes + 1ull);
  const size_t most = rows > part ? rows : part;
  return ((most > ranks ? most : ranks) + 15) & ~size_t(15);
}
// Ranks of one wavefront in memory, by part of the plans: [part][node id][plan of the part].
__host__ __device__ inline size_t kq_rank_doubles(uint32_t plans, const QuadSize& z) { return (size_t)plans * z.nodes; }
__host__ __device__ inline size_t kq_lds_bytes(uint32_t plans, const QuadSize& z, bool mass) {
  return (kq_tab_bytes(z.nodes) + (size_t)plans * (8ull * z.slots + (mass ? 16ull * z.nodes : 0ull) + 2ull * z.nodes + 2ull * z.types) +
          kq_union_bytes(plans, z) + 15) & ~size_t(15);
}

#if defined(__HIPCC__)

// (a permutation within quads reads lanes that are on, throughout: without a value for others the move needs no copy before it and
// folds into the instruction that uses it)
template <int CTRL>
__device__ inline uint32_t kq_dpp(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, CTRL, 0xF, 0xF, true);
}
template <int CTRL>
__device__ inline double kq_dpp(double v) {
  return __hiloint2double((int)kq_dpp<CTRL>((uint32_t)__double2hiint(v)), (int)kq_dpp<CTRL>((uint32_t)__double2loint(v)));
}
constexpr int KQ_XOR1 = 0xB1, KQ_XOR2 = 0x4E;   // quad_perm [1,0,3,2], [2,3,0,1]

// min of two non-NaN doubles in one instruction
__device__ inline double kq_vmin(double a, double b) {
  double r;
  asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ inline double kq_vmin(double a, double b, double c, double d) {
  double r, t;
  asm("v_min_f64 %0, %2, %3\n\tv_min_f64 %1, %4, %5\n\tv_min_f64 %0, %0, %1" : "=&v"(r), "=&v"(t) : "v"(a), "v"(b), "v"(c), "v"(d));
  return r;
}
// What changes in some lanes only, mostly for two slots at a time: the lanes of m0, those of m1, then all (a wavefront schedules with
// all of them on; the build refuses a listing in which one of these stands where some may be off: exec_check.py).  A move or a maximum
// each, where a select takes an instruction for every word and one for what it selects; the masks go to EXEC by scalar instructions,
// which other wavefronts' vector instructions overlap.  (us a step, selects / moves: 1,048,576 DPO plans 787 / 720, 262,144 AC-share
// 3,455 / 3,370, 131,072 PPO 838 / 810, GRPO 418 / 402, 65,536 GRPO 304 / 291, 20,011 PPO 297 / 284.)
// What is written here is written before the last of the other operands is read: early-clobber, also what is read itself.
// -- the larger of two times
__device__ inline void kq_raise(mask64 m0, mask64 m1, double& a, double& b, double t) {
  asm("s_mov_b64 exec, %2\n\tv_max_f64 %0, %0, %4\n\ts_mov_b64 exec, %3\n\tv_max_f64 %1, %1, %4\n\ts_mov_b64 exec, -1"
      : "+&v"(a), "+&v"(b) : "s"(m0), "s"(m1), "v"(t));
}
__device__ inline void kq_raise(mask64 m0, mask64 m1, mask64 m2, double& a, double& b, double& c, double t) {
  asm("s_mov_b64 exec, %3\n\tv_max_f64 %0, %0, %6\n\ts_mov_b64 exec, %4\n\tv_max_f64 %1, %1, %6\n\ts_mov_b64 exec, %5\n\tv_max_f64 %2, %2, %6\n\t"
      "s_mov_b64 exec, -1"
      : "+&v"(a), "+&v"(b), "+&v"(c) : "s"(m0), "s"(m1), "s"(m2), "v"(t));
}
// -- the smallest of some words
__device__ inline void kq_least(mask64 m0, uint32_t& least, uint32_t o0) {
  asm("s_mov_b64 exec, %1\n\tv_min_u32 %0, %2, %0\n\ts_mov_b64 exec, -1" : "+&v"(least) : "s"(m0), "v"(o0));
}
__device__ inline void kq_least(mask64 m0, mask64 m1, uint32_t& least, uint32_t o0, uint32_t o1) {
  asm("s_mov_b64 exec, %1\n\tv_min_u32 %0, %3, %0\n\ts_mov_b64 exec, %2\n\tv_min_u32 %0, %4, %0\n\ts_mov_b64 exec, -1"
      : "+&v"(least) : "s"(m0), "s"(m1), "v"(o0), "v"(o1));
}
// -- bits met so far, and those met twice
__device__ inline void kq_meet(mask64 m0, mask64 m1, uint32_t& seen, uint32_t& twice, uint32_t bit0, uint32_t bit1) {
  asm("s_mov_b64 exec, %2\n\tv_and_or_b32 %1, %0, %4, %1\n\tv_or_b32 %0, %4, %0\n\t"
      "s_mov_b64 exec, %3\n\tv_and_or_b32 %1, %0, %5, %1\n\tv_or_b32 %0, %5, %0\n\t"
      "s_mov_b64 exec, -1"
      : "+&v"(seen), "+&v"(twice) : "s"(m0), "s"(m1), "v"(bit0), "v"(bit1));
}
// -- an entry into its slot
__device__ inline void kq_put(mask64 m0, mask64 m1, double& e0, double& e1, double& s0, double& s1, uint32_t& o0, uint32_t& o1, uint32_t& w0, uint32_t& w1,
                              double e, double s, uint32_t o, uint32_t w) {
  asm("s_mov_b64 exec, %8\n\tv_mov_b64 %0, %10\n\tv_mov_b64 %2, %11\n\tv_mov_b32 %4, %12\n\tv_mov_b32 %6, %13\n\t"
      "s_mov_b64 exec, %9\n\tv_mov_b64 %1, %10\n\tv_mov_b64 %3, %11\n\tv_mov_b32 %5, %12\n\tv_mov_b32 %7, %13\n\t"
      "s_mov_b64 exec, -1"
      : "+&v"(e0), "+&v"(e1), "+&v"(s0), "+&v"(s1), "+&v"(o0), "+&v"(o1), "+&v"(w0), "+&v"(w1) : "s"(m0), "s"(m1), "v"(e), "v"(s), "v"(o), "v"(w));
}
// -- the dispatched entry out of it: a slot without times, free, its word in `out`
template <int U>
__device__ inline void kq_take(mask64 m0, mask64 m1, double& e0, double& e1, double& s0, double& s1, uint32_t& free_slots, uint32_t& out, uint32_t w0, uint32_t w1,
                               double none) {
  asm("s_mov_b64 exec, %6\n\tv_mov_b64 %0, %8\n\tv_mov_b64 %2, %8\n\tv_or_b32 %4, %11, %4\n\tv_mov_b32 %5, %9\n\t"
      "s_mov_b64 exec, %7\n\tv_mov_b64 %1, %8\n\tv_mov_b64 %3, %8\n\tv_or_b32 %4, %12, %4\n\tv_mov_b32 %5, %10\n\t"
      "s_mov_b64 exec, -1"
      : "+&v"(e0), "+&v"(e1), "+&v"(s0), "+&v"(s1), "+&v"(free_slots), "+&v"(out) : "s"(m0), "s"(m1), "s"(none), "v"(w0), "v"(w1), "n"(1 << U), "n"(2 << U));
}
// -- push-backs with ties from `tie` on (kq_again) or a word of their own
__device__ inline void kq_again(mask64 m0, mask64 m1, double& s0, double& s1, uint32_t& o0, uint32_t& o1, double e0, double e1, uint32_t tie_mask, uint32_t tie) {
  asm("s_mov_b64 exec, %4\n\tv_mov_b64 %0, %6\n\tv_bfi_b32 %2, %8, %9, %2\n\t"
      "s_mov_b64 exec, %5\n\tv_mov_b64 %1, %7\n\tv_bfi_b32 %3, %8, %9, %3\n\t"
      "s_mov_b64 exec, -1"
      : "+&v"(s0), "+&v"(s1), "+&v"(o0), "+&v"(o1) : "s"(m0), "s"(m1), "v"(e0), "v"(e1), "v"(tie_mask), "s"(tie));
}
__device__ inline void kq_again(mask64 m0, mask64 m1, double& s0, double& s1, uint32_t& o0, uint32_t& o1, double e0, double e1, uint32_t word) {
  asm("s_mov_b64 exec, %4\n\tv_mov_b64 %0, %6\n\tv_mov_b32 %2, %8\n\t"
      "s_mov_b64 exec, %5\n\tv_mov_b64 %1, %7\n\tv_mov_b32 %3, %8\n\t"
      "s_mov_b64 exec, -1"
      : "+&v"(s0), "+&v"(s1), "+&v"(o0), "+&v"(o1) : "s"(m0), "s"(m1), "v"(e0), "v"(e1), "v"(word));
}
// reductions over the lanes of a plan (two or four)
template <int QL>
__device__ inline uint32_t kq_or(uint32_t v) {
  v |= kq_dpp<KQ_XOR1>(v);
  if (QL == 4) v |= kq_dpp<KQ_XOR2>(v);
  return v;
}
template <int QL>
__device__ inline uint32_t kq_min(uint32_t v) {
  uint32_t o = kq_dpp<KQ_XOR1>(v);
  v = o < v ? o : v;
  if (QL == 4) {
    o = kq_dpp<KQ_XOR2>(v);
    v = o < v ? o : v;
  }
  return v;
}
template <int QL>
__device__ inline double kq_min(double v) {
  v = kq_vmin(v, kq_dpp<KQ_XOR1>(v));
  if (QL == 4) v = kq_vmin(v, kq_dpp<KQ_XOR2>(v));
  return v;
}

// Positions of nodes i, i + QR, ... of the tie-break class that takes ids b to e - 1, into their state words; with EQ also
// whether they are shared.
template <int QL, int QR, int NB, bool EQ>
__device__ inline void kq_count(const double* g_rank, const uint32_t* l_own, const uint16_t* l_chain, uint16_t* g_state, int i, int b, int e) {
  constexpr int RW = KE_WAVE / QL, RG = KE_WAVE / QR, AHEAD = NB == 1 ? 8 : 4;
  double rv[NB];
  uint32_t before[NB], same[NB];
#pragma unroll
  for (int t = 0; t < NB; ++t) {
    rv[t] = g_rank[(i + t * QR < e ? i + t * QR : b) * RG];
    before[t] = (uint32_t)b;
    same[t] = 0u;
  }
  int j = b;
  for (; j + AHEAD <= e; j += AHEAD) {
    double r[AHEAD];
#pragma unroll
    for (int k = 0; k < AHEAD; ++k) r[k] = g_rank[(j + k) * RG];
#pragma unroll
    for (int k = 0; k < AHEAD; ++k)
#pragma unroll
      for (int t = 0; t < NB; ++t) {
        before[t] += r[k] > rv[t] ? 1u : 0u;
        if (EQ) same[t] += r[k] == rv[t] ? 1u : 0u;
      }
  }
  for (; j < e; ++j) {
    const double r = g_rank[j * RG];
#pragma unroll
    for (int t = 0; t < NB; ++t) {
      before[t] += r > rv[t] ? 1u : 0u;
      if (EQ) same[t] += r == rv[t] ? 1u : 0u;
    }
  }
#pragma unroll
  for (int t = 0; t < NB; ++t) {
    const int it = i + t * QR;
    if (it < e) g_state[it * RW] = (uint16_t)(before[t] | (EQ && same[t] > (uint32_t)(l_chain[it] >> 8) ? 0x200u : 0u) | (((l_own[it] >> 3) & 0x3Fu) << 10));
  }
}
// The same for two nodes a lane of classes of `size` nodes each that follow one another, ids b to e - 1 together; per_size: 1 / size.
template <int QL, int QR, bool EQ>
__device__ inline void kq_count_run(const double* g_rank, const uint32_t* l_own, const uint16_t* l_chain, uint16_t* g_state, int i, int b, int e, int size, float per_size) {
  constexpr int RW = KE_WAVE / QL, RG = KE_WAVE / QR, NB = 2, AHEAD = 4;
  const double* from[NB];
  double rv[NB];
  uint32_t before[NB], same[NB];
#pragma unroll
  for (int t = 0; t < NB; ++t) {
    const int it = i + t * QR < e ? i + t * QR : b;
    before[t] = (uint32_t)(b + (int)(((float)(it - b) + 0.5f) * per_size) * size);   // (its class's first: exact, a half is far more than what is rounded)
    from[t] = g_rank + before[t] * RG;
    rv[t] = g_rank[it * RG];
    same[t] = 0u;
  }
  auto count = [&](int t, double r) {
    before[t] += r > rv[t] ? 1u : 0u;
    if (EQ) same[t] += r == rv[t] ? 1u : 0u;
  };
  int j = 0;
  for (; j + AHEAD <= size; j += AHEAD) {
    double r[NB][AHEAD];
#pragma unroll
    for (int t = 0; t < NB; ++t)
#pragma unroll
      for (int k = 0; k < AHEAD; ++k) r[t][k] = from[t][(j + k) * RG];
#pragma unroll
    for (int t = 0; t < NB; ++t)
#pragma unroll
      for (int k = 0; k < AHEAD; ++k) count(t, r[t][k]);
  }
  for (; j < size; ++j)
#pragma unroll
    for (int t = 0; t < NB; ++t) count(t, from[t][j * RG]);
#pragma unroll
  for (int t = 0; t < NB; ++t) {
    const int it = i + t * QR;
    if (it < e) g_state[it * RW] = (uint16_t)(before[t] | (EQ && same[t] > (uint32_t)(l_chain[it] >> 8) ? 0x200u : 0u) | (((l_own[it] >> 3) & 0x3Fu) << 10));
  }
}
// Positions of all nodes: one class after the other, up to four of its nodes to a lane, so that a rank read counts for all of them;
// of small classes (the iterations of an operator: five or eight nodes) as many of one size as follow one another, where one by one a
// class of five leaves eleven of sixteen lanes idle.  (us a step, one by one / together: 131,072 PPO plans 813 / 798, GRPO 401 / 398;
// 65,536 GRPO, 1,048,576 DPO and 262,144 AC-share within 0.2 %.)
template <int QL, int QR, bool EQ>
__device__ inline void kq_count_all(const double* g_rank, const uint32_t* l_own, const uint16_t* l_chain, uint16_t* g_state, uint32_t class_ends, int r_q, int n) {
  for (int b = 0, k = 0; b < n;) {
    int e = __builtin_amdgcn_readlane((int)class_ends, k++);
    const int size = e - b;
    if (size <= 2 * QR) {
      while (e < n && __builtin_amdgcn_readlane((int)class_ends, k) == e + size) {
        e += size;
        ++k;
      }
      if (e > b + size) {
        const float per_size = __builtin_amdgcn_rcpf((float)size);
        for (int i0 = b; i0 < e; i0 += 2 * QR) kq_count_run<QL, QR, EQ>(g_rank, l_own, l_chain, g_state, i0 + r_q, b, e, size, per_size);
        b = e;
        continue;
      }
    }
    int i0 = b;
    for (; e - i0 > 2 * QR; i0 += 4 * QR) kq_count<QL, QR, 4, EQ>(g_rank, l_own, l_chain, g_state, i0 + r_q, b, e);
    if (e - i0 > QR) kq_count<QL, QR, 2, EQ>(g_rank, l_own, l_chain, g_state, i0 + r_q, b, e);
    else if (e - i0 > 0) kq_count<QL, QR, 1, EQ>(g_rank, l_own, l_chain, g_state, i0 + r_q, b, e);
    b = e;
  }
}

// The largest rank among the successors from the fifth on of the node at level place i, or `best`; rank_at: by level place.
template <class AT>
__device__ inline double kq_more_successors(const ClassView& cv, int i, double best, AT&& rank_at) {
  const NodeRec nr = cv.node[cv.lrec[i].node];
  for (int j = 4; j < nr.n_succ; ++j) best = kp_vmax(best, rank_at(cv.place[cv.succ[nr.succ_begin + j]]));
  return best;
}

// Ranks of all plans of a wavefront (scheduler.py:71-100), level by level from the nodes without successors, a node per lane of
// the plan, out to `keep`.
// Bound: a trip (up to two or four nodes a plan) is some 35 vector instructions and one LDS round trip; records are read two trips
// ahead, durations one.  A rank takes eight bytes a node, more than all a plan keeps of it later, but is read back only by the
// few levels below: in LDS lie rows that nodes share (RankRec), and the ranks go through memory to the comparison of positions, which takes
// them a part of the plans at a time (1,048,576 DPO plans, 240 MB of ranks: by the counters all of them are written out and most read
// back from beyond the L2, the launch moves 769 MB, before 358; 262,144 AC-share plans, all schedulers, 1,555, before 845); where the launches'
// wavefronts find room together with all of their ranks those stay in LDS (kq_ranks_in_lds).  Before, the pass ran once for every part,
// with two to four times the lanes for levels of two or three nodes, and a part's ranks all lay in LDS.  us a step, before / now:
// 262,144 AC-share plans 4,196 / 3,953, 131,072 2,720 / 2,572, 65,536 1,550 / 1,430; 131,072 PPO 989 / 935, GRPO 490 / 442; 65,536
// GRPO 320 / 307; 1,048,576 DPO 971 / 971.
template <int QL>
__device__ inline void kq_ranks(const ClassView& cv, double* rows, uint32_t n_rows, uint32_t ends, const double* g_dur, double* keep, uint32_t parts, bool many) {
  constexpr int RW = KE_WAVE / QL;
  const int lane = threadIdx.x, p = lane / QL, q = lane % QL, n = (int)cv.h->n_nodes, n_levels = (int)cv.h->n_levels;
  double* const g_rank = rows + p;
  const uint2* const l_rec = (const uint2*)(rows + (size_t)n_rows * RW);
  // (bytes, of the nodes' ranks of a plan)
  const uint32_t rg = (uint32_t)__builtin_ctz(RW / parts) + 3u, out = (((uint32_t)p >> (rg - 3u)) * (uint32_t)n << rg) + (((uint32_t)p & (RW / parts - 1u)) << 3);
  int level = 0;
  auto end_of = [&](int l) {   // (asked for level by level)
    if (__builtin_expect(l && (l & 63) == 0, 0)) ends = cv.lbeg[l + lane + 1 <= n_levels ? l + lane + 1 : n_levels];
    return l < n_levels ? __builtin_amdgcn_readlane((int)ends, l & 63) : n;
  };
  // a trip: places at to end - 1, QL at most.  This one, the next, the one after that
  int at = 0, end = end_of(0), at1, end1, at2, end2;
  auto next = [&](int a, int e, int& a1, int& e1) {
    a1 = a + QL;
    e1 = e;
    if (a1 >= e) {
      a1 = e;
      e1 = end_of(++level);
    }
  };
  auto record = [&](int a, int e) { return l_rec[a + q < e ? a + q : n]; };
  next(at, end, at1, end1);
  uint2 rec = record(at, end), rec1 = record(at1, end1);
  double d = g_dur[((rec.y >> 8) & 0xFFu) * RW];
  while (at < n) {
    const double r0 = g_rank[(rec.x & 0xFFu) * RW], r1 = g_rank[((rec.x >> 8) & 0xFFu) * RW];
    double best;
    next(at1, end1, at2, end2);
    const uint2 rec2 = record(at2, end2);
    const double d1 = g_dur[((rec1.y >> 8) & 0xFFu) * RW];
    if (__ballot(rec.x > 0xFFFFu)) {
      const double r2 = g_rank[((rec.x >> 16) & 0xFFu) * RW], r3 = g_rank[(rec.x >> 24) * RW];
      best = kp_vmax(kp_vmax(r0, r1), kp_vmax(r2, r3));
      if (__builtin_expect(many, 0))
        if (at + q < end && (rec.y >> 31)) best = kq_more_successors(cv, at + q, best, [&](uint32_t to) { return g_rank[cv.rrec[to].row * RW]; });
    } else {
      best = kp_vmax(r0, r1);
    }
    const double rank = d + best;
    g_rank[(rec.y & 0xFFu) * RW] = rank;
    if (at + q < end) *(double*)((uint8_t*)keep + (out + (((rec.y >> 16) & 0x1FFu) << rg))) = rank;
    rec = rec1;
    rec1 = rec2;
    d = d1;
    at = at1;
    end = end1;
    at1 = at2;
    end1 = end2;
  }
  __syncthreads();   // (the ranks are in memory: a wavefront reads its own)
}

// The same where the ranks of all plans stay in LDS, by node id: no rows, nor their records.  (With them, which take 3 KB more beside
// 33 of graphs of 152 nodes: 20,011 PPO plans 308 / 314 us a step.)
template <int QL>
__device__ inline void kq_ranks_in_lds(const ClassView& cv, double* ranks, const double* g_dur, const uint32_t* l_succ, const uint32_t* l_own,
                                       const uint16_t* l_id, uint32_t ends, bool many) {
  constexpr int RW = KE_WAVE / QL;
  const int lane = threadIdx.x, q = lane % QL, n = (int)cv.h->n_nodes, n_levels = (int)cv.h->n_levels;
  double* const g_rank = ranks + lane / QL;
  // A level waits for one LDS trip, that of its successors' ranks: words and durations of its nodes were read a level ahead,
  // their ids two levels.
  auto rank_at = [&](uint32_t to) { return g_rank[l_id[to] * RW]; };
  if (q == 0) g_rank[n * RW] = 0.0;
  __syncthreads();
  {
    auto end_of = [&](int l) { return l < n_levels ? __builtin_amdgcn_readlane((int)ends, l & 63) : n; };
    auto id_at = [&](int i) { return (int)l_id[i < n ? i : n - 1]; };
    int begin = 0;
    int end = end_of(0), id = id_at(q), id1 = id_at(end + q);
    uint4 sw = ((const uint4*)l_succ)[id];
    uint32_t own = l_own[id];
    double d = g_dur[((own >> 10) & 0xFFu) * RW];
    for (int l = 0; l < n_levels; ++l) {
      const double r0 = g_rank[(sw.x & 0x1FFu) * RW], r1 = g_rank[(sw.y & 0x1FFu) * RW], r2 = g_rank[(sw.z & 0x1FFu) * RW], r3 = g_rank[(sw.w & 0x1FFu) * RW];
      const uint4 sw1 = ((const uint4*)l_succ)[id1];
      const uint32_t own1 = l_own[id1];
      if (__builtin_expect((l & 63) == 63, 0)) ends = cv.lbeg[l + 1 + lane + 1 <= n_levels ? l + 1 + lane + 1 : n_levels];
      const int end1 = end_of(l + 1), id2 = id_at(end1 + q);
      double best = kp_vmax(kp_vmax(r0, r1), kp_vmax(r2, r3));
      int i = begin + q;
      if (__builtin_expect(many, 0))
        if (i < end && (own & 7u) > 4u) best = kq_more_successors(cv, i, best, rank_at);
      if (i < end) g_rank[id * RW] = d + best;
      for (i += QL; __builtin_expect(__ballot(i < end) != 0ull, 0); i += QL) {   // (more nodes than lanes)
        const int id_i = id_at(i);
        const uint4 w = ((const uint4*)l_succ)[id_i];
        const uint32_t o = l_own[id_i];
        best = kp_vmax(kp_vmax(g_rank[(w.x & 0x1FFu) * RW], g_rank[(w.y & 0x1FFu) * RW]), kp_vmax(g_rank[(w.z & 0x1FFu) * RW], g_rank[(w.w & 0x1FFu) * RW]));
        if (many && i < end && (o & 7u) > 4u) best = kq_more_successors(cv, i, best, rank_at);
        if (i < end) g_rank[id_i * RW] = g_dur[((o >> 10) & 0xFFu) * RW] + best;
      }
      d = g_dur[((own1 >> 10) & 0xFFu) * RW];
      begin = end;
      end = end1;
      id = id1;
      id1 = id2;
      sw = sw1;
      own = own1;
    }
  }
  __syncthreads();
}

// From the ranks the state words of all plans of a wavefront, a part of them at a time with as many times the lanes for each.  The
// next part's ranks are fetched while one's are compared with four lanes a plan; with two the sixteen registers this takes kept the
// memory model's launch off the compute units (1,048,576 DPO plans 982 us a step, without 971).
// Bound: instruction issue, two instructions for the comparison of up to 64 pairs of ranks.
template <int QL, uint32_t PARTS>
__device__ inline void kq_positions(const ClassView& cv, double* ranks, const double* keep, const uint32_t* l_own, const uint16_t* l_chain,
                                    uint32_t class_ends, bool shrink, uint16_t* states) {
  constexpr int RW = KE_WAVE / QL, QR = (int)PARTS * QL, RG = KE_WAVE / QR;   // lanes of a plan, plans at a time
  const int lane = threadIdx.x, r_q = lane % QR, n = (int)cv.h->n_nodes;
  const uint4* const from = (const uint4*)keep;
  uint4* const to = (uint4*)ranks;
  const int n4 = n * RG / 2;
  uint4 ahead0, ahead1, ahead2, ahead3;   // (an array would lie in scratch memory)
  auto fetch = [&](int part) {
    const uint4* const f = from + part * n4;
    auto at = [&](int k) { return f[lane + k * KE_WAVE < n4 ? lane + k * KE_WAVE : 0]; };
    ahead0 = at(0); ahead1 = at(1); ahead2 = at(2); ahead3 = at(3);
  };
  if (PARTS > 1 && QL == 4) fetch(0);
  for (int part = 0; part < (int)PARTS; ++part) {
    const int r_p = part * RG + lane / QR;
    double* const g_rank = ranks + lane / QR;
    if (PARTS > 1) {
      auto put = [&](int k, const uint4 w) { if (lane + k * KE_WAVE < n4) to[lane + k * KE_WAVE] = w; };
      if (QL == 2) fetch(part);
      put(0, ahead0); put(1, ahead1); put(2, ahead2); put(3, ahead3);
      for (int i = lane + 4 * KE_WAVE; i < n4; i += KE_WAVE) to[i] = from[part * n4 + i];
      __syncthreads();
      if (QL == 4 && part + 1 < (int)PARTS) fetch(part + 1);
    }
    // (the nodes of a chain have the chain's largest rank, which is the first one's where no duration is negative: a class
    // whose chains are not runs of ids, each node a successor of the one before, has no rows -- chains_in_sequence)
    if (cv.h->n_groups) {
      if (__builtin_expect(shrink, 0)) {
        for (int i = r_q; i < n; i += QR) {
          const int size = (l_chain[i] & 0xFFu) ? 1 : (int)(l_chain[i] >> 8);
          double top = g_rank[i * RG];
          for (int j = 1; j < size; ++j) top = kp_vmax(top, g_rank[(i + j) * RG]);
          if (size > 1) g_rank[i * RG] = top;
        }
        __syncthreads();
      }
      for (int i = r_q; i < n; i += QR) {
        const int in_chain = (int)(l_chain[i] & 0xFFu);
        if (in_chain) g_rank[i * RG] = g_rank[(i - in_chain) * RG];
      }
      __syncthreads();
    }
    // ---- positions: nodes before v in (comm_prio*8+topo_idx ascending, rank descending) = the nodes of lower tie-break
    // classes and the nodes of its own class with a larger rank; shared where more nodes than its own chain agree.  Equal ranks
    // are found by counting them along, in small graphs, or afterwards, by counting the nodes of a position.
    if (n <= KQ_EQ_NODES) {
      kq_count_all<QL, QR, true>(g_rank, l_own, l_chain, states + r_p, class_ends, r_q, n);
      __syncthreads();   // (these ranks are done with)
      continue;
    }
    kq_count_all<QL, QR, false>(g_rank, l_own, l_chain, states + r_p, class_ends, r_q, n);
    __syncthreads();   // (these ranks are done with: over them counters, by position)
    uint32_t* const g_count = (uint32_t*)(ranks + lane / QR);
    for (int i = r_q; i < n; i += QR) g_count[2 * i * RG] = 0u;
    __syncthreads();
    for (int i = r_q; i < n; i += QR) atomicAdd(&g_count[2 * (states[i * RW + r_p] & 0x1FFu) * RG], 1u);
    __syncthreads();
    for (int i = r_q; i < n; i += QR) {
      const uint32_t state = states[i * RW + r_p];
      if (g_count[2 * (state & 0x1FFu) * RG] > (uint32_t)(l_chain[i] >> 8)) states[i * RW + r_p] = (uint16_t)(state | 0x200u);
    }
    __syncthreads();   // (these ranks are done with)
  }
}

template <int QL, int SL>
__device__ inline void kq_eval_wave(const EvalLaunch& L, const QuadSize& Z, double* keep, uint64_t w, uint8_t* lds) {   // keep: ranks (kq_rank_doubles)
  constexpr int RW = KE_WAVE / QL;
  const int lane = threadIdx.x, p = lane / QL, q = lane % QL;
  constexpr int first_lane = 0;
  const rpeg_problem_t& P = *L.P;
  const ClassView cv = class_view(L.pool + (L.wave_cls[w] & ~KE_CLS_LDS));   // uniform
  const int n = (int)cv.h->n_nodes, n_slots = (int)cv.h->n_slots;
  const int n_rows = (int)cv.h->n_rows, n_types = (int)cv.h->n_types;

  // ---- LDS carve-up
  uint32_t* l_succ = (uint32_t*)lds;               // [node id][4]: id | the successor's QuadRec from bit 10 on (none: the neutral element's id, alone)
  uint32_t* l_own = l_succ + 4 * Z.nodes;          // [node id]: QuadRec
  uint16_t* l_id = (uint16_t*)(l_own + Z.nodes);   // level place -> id
  uint16_t* l_chain = l_id + (Z.nodes + 2);        // [node id]: place in its chain (whose nodes' ids follow each other) | nodes of the chain << 8
  double* rows = (double*)(lds + kq_tab_bytes(Z.nodes));
  double* g_dur = rows + p;
  rows += (size_t)Z.slots * RW;
  double* const ranks = rows;                      // [node id][plans at a time], before the two below are needed
  double* g_lf = rows + p;
  double* g_time = g_lf + (size_t)(RPEG_MAX_V + 2) * RW;   // [row]
  rows = (double*)((uint8_t*)rows + kq_union_bytes(RW, Z));
  double* g_fin = rows + p;                        // [node id], with L.mass
  double* g_start = g_fin + (size_t)Z.nodes * RW;
  if (L.mass) rows += 2 * (size_t)Z.nodes * RW;
  uint16_t* const states = (uint16_t*)rows;
  uint16_t* g_state = states + p;                  // [node id]: position | shared << 9 | predecessors to go << 10
  uint16_t* g_type = states + (size_t)Z.nodes * RW + p;   // [reservation]: reserved vertices | vertices that overlap them << 6

  // a place without a plan repeats the first one of the wavefront, without outputs: every lane is active throughout
  const uint32_t entry = L.perm[w * KE_WAVE + p];
  const bool idle = entry == KE_IDLE;
  const uint64_t pi = (uint64_t)(idle ? L.perm[w * KE_WAVE] : entry);
  __syncthreads();  // the previous task of this wavefront is done with LDS
  uint32_t class_ends = 0;   // lane k: where the ids of tie-break class k end
  for (int i = lane, k = 0; i - lane < n; i += KE_WAVE) {
    const OrderRec r = cv.orec[i < n ? i : 0];
    if (i < n) {
      l_id[r.at] = (uint16_t)i;
      l_chain[i] = (uint16_t)(r.chain_i | r.chain_n << 8);
    }
    for (mask64 last = __ballot(i < n && (int)r.b1 == i + 1); last; last &= last - 1ull, ++k) class_ends = lane == k ? (uint32_t)(i - lane + __builtin_ctzll(last) + 1) : class_ends;
  }
  if (lane == 0) l_id[n] = (uint16_t)n;
  __syncthreads();
  const uint32_t level_ends = cv.lbeg[lane + 1 <= (int)cv.h->n_levels ? lane + 1 : (int)cv.h->n_levels];
  if (Z.parts > 1) {   // what the rank pass reads, behind its rows
    uint2* const l_rec = (uint2*)(ranks + (size_t)Z.ranks * RW);
    for (int i = lane; i <= n; i += KE_WAVE) l_rec[i] = ((const uint2*)cv.rrec)[i];
    if (q == 0) ranks[p] = 0.0;
  }
  mask64 many = 0ull;   // some node has more than four successors
  for (int i = lane; i < n; i += KE_WAVE) {
    const LevelRec r = cv.lrec[i];
    const uint32_t id = l_id[i];
    l_own[id] = cv.qrec[i];
    many |= __ballot((cv.qrec[i] & 7u) > 4u);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint32_t at = r.succ[k];
      l_succ[4 * id + k] = (uint32_t)l_id[at] | (at < (uint32_t)n ? cv.qrec[at] & ~0x3FFu : 0u);
    }
  }
  KE_STAMP(0);

  // pair relations, penalty factor and gate bits of this plan and the durations of its class's slots (out of the table
  // of the slot universe) come from the prologue launches, by plan index
  const uint64_t ovl = L.aux_ovl[pi], dpne = L.aux_dpne[pi];
  const double pen = L.aux_pen ? L.aux_pen[pi] : 1.0;
  const uint8_t gates = L.aux_mask ? L.aux_mask[pi] : (uint8_t)(RPEG_MASK_VALID | RPEG_MASK_STALE_OK | RPEG_MASK_MEM_OK);
  KE_STAMP(1);
  bool err = cv.h->error != 0, shrink = false;   // shrink: some plan has a node that ends before it starts
  {   // a slot whose duration the reference could not compute (division by zero) is NaN; a share by each lane
    bool bad = false, shrinks = false;
    for (int s0 = q; s0 < n_slots; s0 += 4 * QL) {   // four rows in flight
      double d[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int s = s0 + k * QL;
        d[k] = L.dur[(size_t)cv.umap[s < n_slots ? s : s0] * L.dur_stride + pi];
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int s = s0 + k * QL;
        bad = bad || d[k] != d[k];
        shrinks = shrinks || d[k] < 0.0;
        if (s < n_slots) g_dur[s * RW] = d[k];
      }
    }
    err = err || kq_or<QL>(bad ? 1u : 0u) != 0u;
    shrink = __ballot(shrinks) != 0ull;
    if (err)   // (no NaN in the loops below)
      for (int s = q; s < n_slots; s += QL) g_dur[s * RW] = 0.0;
  }
  for (int t = q; t < n_types; t += QL) {
    const uint32_t bc = cv.type[t], bt = kp_reserved(bc & 0xFFu, bc >> 8, ovl, dpne);
    const uint32_t b6 = bt & 0x3Fu;
    g_type[t * RW] = (uint16_t)(b6 | (((bt >> 8) & 0x3Fu) << 6) | ((b6 ? 31u - (uint32_t)__builtin_clz(b6) : (uint32_t)RPEG_MAX_V) << 12));
  }
  __syncthreads();
  KE_STAMP(2);
  const bool stale_ok = (gates & RPEG_MASK_STALE_OK) != 0, mem_ok = (gates & RPEG_MASK_MEM_OK) != 0;

  const bool any_many = __ballot(many != 0ull) != 0ull;   // (lanes that left the loop early)
  if (Z.parts == 1) {
    kq_ranks_in_lds<QL>(cv, ranks, g_dur, l_succ, l_own, l_id, level_ends, any_many);
    KE_STAMP(3);
    kq_positions<QL, 1>(cv, ranks, keep, l_own, l_chain, class_ends, shrink, states);
  } else {
    kq_ranks<QL>(cv, ranks, Z.ranks, level_ends, g_dur, keep, Z.parts, any_many);
    KE_STAMP(3);
    if (Z.parts == kq_parts_least(QL)) kq_positions<QL, kq_parts_least(QL)>(cv, ranks, keep, l_own, l_chain, class_ends, shrink, states);
    else kq_positions<QL, 2 * kq_parts_least(QL)>(cv, ranks, keep, l_own, l_chain, class_ends, shrink, states);
  }
  for (int x = q; x <= RPEG_MAX_V; x += QL) g_lf[x * RW] = 0.0;
  for (int r = q; r < n_rows; r += QL) g_time[r * RW] = 0.0;
  __syncthreads();

  KE_STAMP(4);
  // ---- list scheduling (scheduler.py:399-546)
  const double no_time = __hiloint2double((int)KQ_NO_TIME, 0);
  auto no_time_in = [&](mask64 m, double x) {   // (in the lanes of m)
    return __hiloint2double((int)kp_sel(m, KQ_NO_TIME, (uint32_t)__double2hiint(x)), __double2loint(x));
  };
  uint32_t tie_mask;   // (in a register: as a constant it takes an instruction of its own with every use)
  asm("v_mov_b32 %0, %1" : "=v"(tie_mask) : "s"(KQ_TIE_MASK));
  double ek[SL], sk[SL];
  uint32_t eo[SL], em[SL];
#pragma unroll
  for (int u = 0; u < SL; ++u) { ek[u] = no_time; sk[u] = no_time; eo[u] = KQ_EMPTY; em[u] = 0u; }
  uint32_t tie = 0, free_slots = (1u << SL) - 1u;
  bool ovf = false;
  int live = 0, longest = 0;   // entries now and at most (one more than there is room for where one was lost)
  const unsigned group_shift = (unsigned)(lane & ~(QL - 1));
  const uint32_t below = (1u << q) - 1u;   // the lanes of this plan before this one
  // this lane keeps the availability of vertices q, q + QL, ... (where there are fewer: of the row behind the zeros)
  constexpr int NLF = (RPEG_MAX_V + QL - 1) / QL;
  double lf[NLF];
  uint32_t lf_bit[NLF];
  double* lf_row[NLF];
#pragma unroll
  for (int k = 0; k < NLF; ++k) {
    const int x = q + k * QL;
    lf[k] = 0.0;
    lf_bit[k] = x < RPEG_MAX_V ? 1u << (24 + x) : 0u;
    lf_row[k] = g_lf + (x < RPEG_MAX_V ? x : RPEG_MAX_V + 1) * RW;
  }
  const mask64 quads0 = QL == 4 ? 0x1111111111111111ull : 0x5555555555555555ull;   // the first lane of every plan
  // an entry into the first free slot of this lane, in the lanes of `take` (conditions are kept as masks of the lanes in
  // scalar registers: as booleans the compiler moves them through vector registers).  node: id | its QuadRec from bit 10 on
  auto file = [&](mask64 take, double key, uint32_t state, uint32_t node, uint32_t type, uint32_t t) {
    const uint32_t first = kp_sel(take, free_slots & (0u - free_slots), 0u);
    const uint32_t word = ((state & 0x1FFu) << KQ_TIE_BITS) | t, meta = (node & 0x3FDFFu) | (type << 18);
    const double heap_key = no_time_in(__ballot(state < 0x200u), key);
#pragma unroll
    for (int u = 0; u < SL; u += 2)
      kq_put(__ballot(first == (1u << u)), __ballot(first == (2u << u)), ek[u], ek[u + 1], sk[u], sk[u + 1], eo[u], eo[u + 1], em[u], em[u + 1], key, heap_key, word, meta);
    free_slots ^= first;
  };
  {
    const int n_init = (int)cv.h->n_init;
    ovf = n_init > QL * SL;
    for (int i0 = 0; i0 < n_init && i0 < QL * SL; i0 += QL) {
      const bool mine = i0 + q < n_init;
      const uint32_t v = l_id[cv.place[cv.init[mine ? i0 + q : 0]]], own = l_own[v];
      file(__ballot(mine), 0.0, g_state[v * RW], v | (own & ~0x3FFu), g_type[((own >> 18) & 0x3Fu) * RW], (uint32_t)(i0 + q));
    }
    tie = (uint32_t)n_init;
    live = longest = n_init;
  }
  double makespan = 0.0;
  uint32_t n_back = 0;
  mask64 lost = 0ull;                             // plans (all four lanes) with an entry that found no room
  // Lanes of this plan with room: before this one, all.  (Of two from one another; of four by a shift of 64 bits, which with these is
  // shorter than bits put together: AC-share 3,355 us a step, so 3,375.)
  auto count_room = [&](mask64 room, uint32_t& r, uint32_t& n_room) {
    if constexpr (QL == 2) {
      const uint32_t one = free_slots < 1u ? free_slots : 1u, other = kq_dpp<KQ_XOR1>(one);
      r = other & below;
      n_room = one + other;
    } else {
      const uint32_t in_plan = (uint32_t)(room >> group_shift) & ((1u << QL) - 1u);
      r = (uint32_t)__builtin_popcount(in_plan & below);
      n_room = (uint32_t)__builtin_popcount(in_plan);
    }
  };
  auto least = [&](const mask64 (&m)[SL]) {   // the smallest word of this lane's entries in m
    uint32_t o = kp_sel(m[0], eo[0], KQ_EMPTY);
    kq_least(m[1], o, eo[1]);
#pragma unroll
    for (int u = 2; u < SL; u += 2) kq_least(m[u], m[u + 1], o, eo[u], eo[u + 1]);
    return o;
  };
  auto key_min = [&](const double (&x)[SL]) {
    double k;
    if constexpr (SL == 2) k = kq_vmin(x[0], x[1]);
    else if constexpr (SL == 4) k = kq_vmin(x[0], x[1], x[2], x[3]);
    else k = kq_vmin(kq_vmin(x[0], x[1], x[2], x[3]), kq_vmin(x[SL - 2], x[SL - 1]));
    return kq_min<QL>(k);
  };
  // the entry of word o (of every plan: its own) is pushed back
  auto push_back = [&](uint32_t o) {
    const uint32_t fresh = (o & ~tie_mask) | tie;
#pragma unroll
    for (int u = 0; u < SL; u += 2) kq_again(__ballot(eo[u] == o), __ballot(eo[u + 1] == o), sk[u], sk[u + 1], eo[u], eo[u + 1], ek[u], ek[u + 1], fresh);
    ++tie;   // (also in a plan that pushed nothing back: only the order of ties is looked at)
  };
  for (int done = 0; done < n; ++done) {
    const double gk = key_min(ek);
    // push-backs of entries of shared position below the smallest true start time
    mask64 back[SL], more = 0ull;
#pragma unroll
    for (int u = 0; u < SL; ++u) {
      back[u] = __ballot(sk[u] < gk);
      more |= back[u];
    }
    if (more) {
      // positions (by their low five bits) that occur twice among them
      uint32_t bit[SL], seen = 0u, twice = 0u;
#pragma unroll
      for (int u = 0; u < SL; u += 2) {
        bit[u] = 1u << ((eo[u] >> KQ_TIE_BITS) & 31u);
        bit[u + 1] = 1u << ((eo[u + 1] >> KQ_TIE_BITS) & 31u);
        kq_meet(back[u], back[u + 1], seen, twice, bit[u], bit[u + 1]);
      }
      uint32_t other = kq_dpp<KQ_XOR1>(seen);
      twice |= (seen & other) | kq_dpp<KQ_XOR1>(twice);
      if (QL == 4) {
        seen |= other;
        other = kq_dpp<KQ_XOR2>(seen);
        twice |= (seen & other) | kq_dpp<KQ_XOR2>(twice);
      }
      more = 0ull;
      mask64 alone[SL];
#pragma unroll
      for (int u = 0; u < SL; ++u) {
        const mask64 mates = back[u] & __ballot((bit[u] & twice) != 0u);
        alone[u] = back[u] & ~mates;
        more |= mates;
      }
#pragma unroll
      for (int u = 0; u < SL; u += 2) kq_again(alone[u], alone[u + 1], sk[u], sk[u + 1], eo[u], eo[u + 1], ek[u], ek[u + 1], tie_mask, tie);
      ++tie;
      while (more) {
        ++n_back;
        const double k = key_min(sk);
        more = __ballot(k < gk);
        mask64 at_k[SL];
#pragma unroll
        for (int u = 0; u < SL; ++u) at_k[u] = __ballot(sk[u] == k);
        push_back(kp_sel(more, kq_min<QL>(least(at_k)), KQ_EMPTY - 1u));   // (no entry has that word)
        if constexpr (QL == 2) {   // the last one of every plan needs not be looked for (four lanes a plan, AC-share: 3,472 us a step, with this 3,510)
          mask64 left[SL], several = 0ull;
          more = 0ull;
#pragma unroll
          for (int u = 0; u < SL; ++u) {
            left[u] = __ballot(sk[u] < gk);
            several |= more & left[u];
            more |= left[u];
          }
          if (!more) break;
          several |= more & (more >> 1) & quads0;
          if (several == 0ull) {
#pragma unroll
            for (int u = 0; u < SL; u += 2) kq_again(left[u], left[u + 1], sk[u], sk[u + 1], eo[u], eo[u + 1], ek[u], ek[u + 1], tie_mask, tie);
            ++tie;
            break;
          }
        } else {
          more = 0ull;
#pragma unroll
          for (int u = 0; u < SL; ++u) more |= __ballot(sk[u] < gk);
        }
      }
    }
    mask64 at_gk[SL], level = 0ull;
#pragma unroll
    for (int u = 0; u < SL; ++u) {
      at_gk[u] = __ballot(ek[u] == gk);
      level |= __ballot(sk[u] == gk) & ~at_gk[u];
    }
    uint32_t bo = kq_min<QL>(least(at_gk));
    // push-backs of entries with that key that come before the one to dispatch
    if (__builtin_expect(level != 0ull, 0)) {
      for (;;) {
        mask64 stale[SL];
#pragma unroll
        for (int u = 0; u < SL; ++u) stale[u] = __ballot(sk[u] == gk) & __ballot(ek[u] > gk);
        const uint32_t o = kq_min<QL>(least(stale));
        const mask64 act = __ballot(o < bo);
        if (!act) break;
        push_back(kp_sel(act, o, KQ_EMPTY - 1u));
      }
    }
    const mask64 alive = __ballot(gk < no_time);   // (nothing waits: an entry was lost, or a start time is as good as infinite: flagged)
    lost |= ~alive;
    bo = kp_sel(alive, bo, KQ_EMPTY - 1u);
    uint32_t bm = 0;
#pragma unroll
    for (int u = 0; u < SL; u += 2) {   // the dispatched entry leaves its slot (what an emptied slot keeps of one is no other's word)
      const mask64 hit0 = __ballot(eo[u] == bo), hit1 = __ballot(eo[u + 1] == bo);
      if (u == 0) kq_take<0>(hit0, hit1, ek[0], ek[1], sk[0], sk[1], free_slots, bm, em[0], em[1], no_time);
      if constexpr (SL > 2) if (u == 2) kq_take<2>(hit0, hit1, ek[2], ek[3], sk[2], sk[3], free_slots, bm, em[2], em[3], no_time);
      if constexpr (SL > 4) if (u == 4) kq_take<4>(hit0, hit1, ek[4], ek[5], sk[4], sk[5], free_slots, bm, em[4], em[5], no_time);
    }
    bm = kq_or<QL>(bm);
    mask64 room = __ballot(free_slots != 0u);
    uint32_t r, n_room;
    count_room(room, r, n_room);
    const uint32_t place = bm & 0x1FFu;
    const uint32_t first_succ = l_succ[4 * place + r];   // (r < QL)
    uint32_t n_succ = l_own[place] & 7u;
    uint32_t slot = (bm >> 10) & 0xFFu;
    asm("" : "+v"(slot));   // (a field, then its address: two instructions, where the compiler shifts, masks and adds)
    const double fin = gk + g_dur[slot * RW];
    if (L.mass) {
      if (kp_in(alive & quads0)) {
        g_fin[place * RW] = fin;
        g_start[place * RW] = gk;
      }
    }
    makespan = kp_vmax(makespan, fin);
    auto reserved = [&](int k) { return __ballot((bm & lf_bit[k]) != 0u); };
    static_assert(NLF == 2 || NLF == 3, "");
    if constexpr (NLF == 2) kq_raise(reserved(0), reserved(1), lf[0], lf[1], fin);
    else kq_raise(reserved(0), reserved(1), reserved(2), lf[0], lf[1], lf[2], fin);
#pragma unroll
    for (int k = 0; k < NLF; ++k) lf_row[k][0] = lf[k];
    --live;
    const uint32_t touched = (bm >> 6) & (0x3Fu << 18);
#pragma unroll
    for (int u = 0; u < SL; u += 2) kq_raise(__ballot((em[u] & touched) != 0u), __ballot((em[u + 1] & touched) != 0u), ek[u], ek[u + 1], fin);
    // successors: the lanes with room look at one each; those that became ready are filed where they were looked at
    // (scheduler.py:540-546: ties in successor order)
    if (__builtin_expect(any_many, 0)) n_succ = n_succ == 7u ? (uint32_t)cv.node[cv.lrec[cv.orec[place].at].node].n_succ : n_succ;
    mask64 mine = room & alive & __ballot(r < n_succ);
    uint32_t j0 = n_room, node = first_succ;   // (in lanes that have none to look at: another's, or the neutral element, which are read alone)
    while (mine) {
      const uint32_t row = node >> 24;   // (a node of one predecessor: the row that stays zero)
      uint32_t at = node & 0x1FFu, type_at = (node >> 18) & 0x3Fu;
      asm("" : "+v"(at), "+v"(type_at));
      const uint32_t state = g_state[at * RW], left = state - 0x400u;
      uint32_t type = g_type[type_at * RW];
      double t = kp_vmax(g_time[row * RW], fin);
      const mask64 ready = mine & __ballot(left < 0x400u);
      if (kp_in(mine & ~ready)) {
        g_time[row * RW] = t;
        g_state[at * RW] = (uint16_t)left;
      }
      if (ready) {
        if (__builtin_expect(shrink, 0)) {   // (a later node of the row may be ready before what this one leaves there)
          if (kp_in(ready)) g_time[row * RW] = 0.0;
        }
        asm("" : "+v"(type));   // (all of the register: not narrowed to 16 bits again)
        // one vertex or two (none: the row of zeros)
        const uint32_t v1 = (uint32_t)__builtin_ctz((type & 0x3Fu) | (1u << RPEG_MAX_V)), v2 = type >> 12;
        t = kp_vmax(t, kp_vmax(g_lf[v1 * RW], g_lf[v2 * RW]));
        uint32_t before, filed;
        if constexpr (QL == 2) {
          const uint32_t one = kp_sel(ready, 1u, 0u), other = kq_dpp<KQ_XOR1>(one);
          before = other & below;
          filed = one + other;
        } else {
          const uint32_t rdy = (uint32_t)(ready >> group_shift) & ((1u << QL) - 1u);
          before = (uint32_t)__builtin_popcount(rdy & below);
          filed = (uint32_t)__builtin_popcount(rdy);
        }
        file(ready, t, left, node, type, tie + before);
        tie += (uint32_t)QL;
        live += (int)filed;
        longest = live > longest ? live : longest;
      }
      const mask64 again = alive & __ballot(j0 < n_succ);
      if (__builtin_expect(again == 0ull, 1)) break;
      room = __ballot(free_slots != 0u);
      count_room(room, r, n_room);
      const mask64 full = again & __ballot(n_room == 0u);
      lost |= full;
      longest = (int)kp_sel(full, (uint32_t)(QL * SL + 1), (uint32_t)longest);   // (an entry without room is not counted in `live`: the class moves up a form)
      j0 = kp_sel(full, n_succ, j0);
      mine = again & room & __ballot(j0 + r < n_succ);
      node = 0;
      if (kp_in(mine)) {
        const uint32_t j = j0 + r;
        if (j < 4u) {
          node = l_succ[4 * place + j];
        } else {
          const uint32_t to = cv.place[cv.succ[cv.node[cv.lrec[cv.orec[place].at].node].succ_begin + j]];
          node = (uint32_t)l_id[to] | (cv.qrec[to] & ~0x3FFu);
        }
      }
      j0 += n_room;
    }
  }
  ovf = ovf || kp_in(lost);
  err = err || ovf;
  if (ovf && q == 0 && !idle) ke_flag_limit(L, pi, L.wave_cls[w] & ~KE_CLS_LDS);
  if (L.need) {   // the longest ready set of the wavefront, folded into one of the running maxima
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      const int o = __shfl_xor(longest, off);
      longest = o > longest ? o : longest;
    }
    uint32_t* slot = L.need + (blockIdx.x & (KE_NEED_SHARDS - 1));
    if (lane == 0 && (uint32_t)longest > *slot) atomicMax(slot, (uint32_t)longest);
    if (lane == 0 && L.cneed && (uint32_t)longest > L.cneed[cv.h->id]) atomicMax(&L.cneed[cv.h->id], (uint32_t)longest);
  }
  KE_STAMP(5);
  if (L.prof && lane == 0) L.prof[w * 8 + 7] = ((unsigned long long)n << 32) | (unsigned long long)(n + n_back);

  // ---- outputs
  uint8_t mask = RPEG_MASK_VALID;
  if (stale_ok) mask |= RPEG_MASK_STALE_OK;
  if (mem_ok) mask |= RPEG_MASK_MEM_OK;
  double out_makespan, out_score;
  if (err || makespan == 0.0) {
    out_makespan = out_score = __builtin_nan("");
    mask |= RPEG_MASK_ERROR;
    if (ovf) mask |= RPEG_MASK_LIMIT;
  } else {
    double score = P.score_num / makespan;
    if (!mem_ok) score = score * pen;
    if ((L.flags & RPEG_GATE_STALE) && !stale_ok) score = 0.0;
    out_makespan = makespan;
    out_score = score;
  }
  if (q == 0 && !idle) {
    if (L.makespan) L.makespan[pi] = out_makespan;   // (the peak is the prologue launch's output)
    if (L.score) L.score[pi] = out_score;
    if (L.mask) L.mask[pi] = mask;
    if (L.mass) {
      double m[RPEG_MAX_V];
      if (err) {
#pragma unroll
        for (int x = 0; x < RPEG_MAX_V; ++x) m[x] = __builtin_nan("");
      } else {
        critical_mass(cv, [&](int i) { return g_fin[l_id[cv.place[i]] * RW]; }, [&](int i) { return g_start[l_id[cv.place[i]] * RW]; }, m);
      }
#pragma unroll
      for (int x = 0; x < RPEG_MAX_V; ++x) L.mass[pi * RPEG_MAX_V + x] = m[x];
    }
  }
  KE_STAMP(6);
}

#endif  // __HIPCC__

}  // namespace rpeg
#endif
