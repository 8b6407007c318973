// rpeg_kernel_plan.h - the evaluation kernel of small batches, of the smallest classes and of the largest graphs (device
// only): ONE PLAN PER WAVEFRONT, or per block of four.
//
// The lanes share the plan's work instead of each carrying a plan of its own:
//   cost model      lane = duration slot of the class (NodeCostModel.time of one node variant each)
//   memory model    lane = template vertex, then lane = vertex subset (candidate device class)
//   ranks           level by level from the nodes without successors, lane = node of the level (scheduler.py:71-100)
//   positions       lane = node, which counts the nodes of its tie-break class with a larger rank
//   list scheduler  rpeg_kernel_sched.h: up to 192 nodes every node in a lane, one to three to each, dealt by position; beyond
//                   that a lane for every waiting node, the others in LDS.  All control flow is uniform
//   outputs         lane = node for the predecessors of the critical chain, lane = set of allocations for the utilisation
//
// Device availability: a node waits for max(avail[d]) over the devices it reserves, i.e. for the largest finish time of
// any dispatched node whose reserved vertices intersect its own.  Every lane keeps that maximum for its nodes and raises
// it at each dispatch (max is exact, so the order does not matter).
//
// As a task of a full batch durations, pair relations, penalty factor and gate bits come from the prologue launches; in a batch that
// gets a wavefront per plan throughout the durations do (EvalLaunch::dur without ::aux_ovl).
#ifndef RPEG_KERNEL_PLAN_H
#define RPEG_KERNEL_PLAN_H

#include "rpeg_kernel_sched.h"

namespace rpeg {

constexpr int KP_MAX_NS = 6;                    // nodes per lane: classes of up to 384 nodes
constexpr uint32_t KP_SKIP = 0xFFFFFFFFu;        // task -> class blob offset of a task that is skipped (offsets stay below 2^31)
constexpr int KP_PLAN_I16 = 80;                 // plan fields in LDS (60 used; pair tests may read past them)

// LDS of one wavefront: plan fields, per-vertex memory terms, the areas of the scheduler (KpLds: level records, two doubles
// per node and a neutral element each, the two maps between level place and position, over which the dispatch order and
// the critical chain's tables lie), durations per slot; for the utilisation busy time by allocation set (64 doubles).
__host__ __device__ inline size_t kp_lds_bytes(uint32_t nodes, uint32_t slots) {
  const size_t fixed = (size_t)KP_PLAN_I16 * 2 + (size_t)RPEG_MAX_V * 4 * 8 + 64 * 8 + 8ull * slots;
  return (fixed + 16ull * nodes + 16ull * (nodes + 1) + 4ull * nodes + 2ull * (nodes + 1) + 15) & ~size_t(15);
}

#if defined(__HIPCC__)

// Critical-chain mass per template vertex (critical_mass of rpeg_class.h; moves.py:590-642) for one plan.  What the walk
// needs at a node -- the predecessor it goes on to (the first one, in edge order, of largest finish time) and the vertex
// the node counts for -- is found for all nodes at once, a node per lane, and left in LDS; the walk itself, one hop after
// the other from the first node of largest finish time, then reads LDS only.  KpHop: what the class says of a node,
// which a wavefront that has nothing else to do fetches while the plan is scheduled.
struct KpHop {
  uint32_t begin = 0, end = 0, first = 0, vx = 0xFF;   // predecessors, the first of them; vertex
};
__device__ inline KpHop kp_hop_of(const ClassView& cv, int v) {
  KpHop p;
  p.begin = cv.pbeg[v]; p.end = cv.pbeg[v + 1];
  p.first = cv.pred[p.begin < p.end ? p.begin : 0];
  const SlotDesc sd = cv.slot[cv.node[v].slot];
  p.vx = sd.type <= SLOT_OP_SUB ? sd.a : 0xFFu;
  return p;
}
__device__ inline void kp_hop(const ClassView& cv, int v, const KpHop& p, const double* l_fin, uint16_t* l_next, uint8_t* l_vx) {
  uint32_t nx = 0xFFFFu;
  if (p.begin != p.end) {
    nx = p.first;
    double b = l_fin[nx];
    for (uint32_t j = p.begin + 1; j < p.end; ++j) {
      const uint32_t q = cv.pred[j];
      const double fq = l_fin[q];
      if (fq > b) { b = fq; nx = q; }
    }
  }
  l_next[v] = (uint16_t)nx;
  l_vx[v] = (uint8_t)p.vx;
}
// Lane x < RPEG_MAX_V returns the mass of vertex x, summed in the order of the walk.  scratch: sixteen bytes a node.
// Bound: the walk, a dependent LDS trip a hop.  So it is done in steps of eight hops -- where those lead is found for all nodes at
// once by doubling --, every lane then walks one of these stretches, and the sums read the chain from consecutive places.  (Hop by
// hop: chains of PPO graphs of 77-153 nodes, with the outputs, 3.6 us, now 3.0.)
__device__ inline double kp_critical_mass(const int n, const int lane, const double* l_fin, const double* l_start,
                                          const uint16_t* l_next, const uint8_t* l_vx, uint8_t* scratch) {
  double bf = -1.0;
  uint32_t bi = 0xFFFFFFFFu;
  for (int v = lane; v < n; v += KE_WAVE) {
    const double f = l_fin[v];
    if (f > bf) { bf = f; bi = (uint32_t)v; }
  }
  const double top = kp_wave_reduce(bf, KpMax());
  int cur = (int)kp_wave_umin(bf == top ? bi : 0xFFFFFFFFu);
  double m = 0.0;
  constexpr int STEP = 8, FEW = 32;   // (a graph of at most FEW nodes has no room for the stretches, nor use for them)
  static_assert(STEP * KE_WAVE >= KE_WAVE * KP_MAX_NS, "a stretch for every lane");
  if (n <= FEW) {
    for (int hops = 0; hops <= n; ++hops) {   // a chain visits a node at most once
      const int vx = l_vx[cur];
      const double d = l_fin[cur] - l_start[cur];
      const int nx = __builtin_amdgcn_readfirstlane((int)l_next[cur]);
      if (lane == vx) m += d;
      if (nx == 0xFFFF) break;
      cur = nx;
    }
    return m;
  }
  const int places = (n + STEP - 1) & ~(STEP - 1);
  double* const time = (double*)scratch;                       // of the chain, by place
  uint8_t* const vertex = scratch + 8 * (size_t)places;
  uint16_t *const twice = (uint16_t*)(vertex + places), *const four = twice + n;   // where two, four and, over the first, eight hops lead
  auto after = [&](const uint16_t* from, const uint16_t* by, uint16_t* to) {
    for (int v = lane; v < n; v += KE_WAVE) {
      const uint32_t x = from[v];
      const uint16_t y = by[x < (uint32_t)n ? x : 0u];
      to[v] = x < (uint32_t)n ? y : (uint16_t)0xFFFFu;
    }
    kp_sync();
  };
  after(l_next, l_next, twice);
  after(twice, twice, four);
  after(four, four, twice);
  int n_stretch = 0;
  uint32_t at = 0xFFFFu;   // lane k: where stretch k begins
  for (;;) {
    const int nx = __builtin_amdgcn_readfirstlane((int)twice[cur]);
    at = lane == n_stretch ? (uint32_t)cur : at;
    ++n_stretch;
    if (nx == 0xFFFF || n_stretch * STEP >= places) break;
    cur = nx;
  }
  for (int j = 0; j < STEP; ++j) {
    const uint32_t v = at < (uint32_t)n ? at : 0u;
    const double d = l_fin[v] - l_start[v];
    const uint8_t vx = l_vx[v];
    const uint32_t nx = l_next[v];
    if (lane < n_stretch) {
      time[lane * STEP + j] = at < (uint32_t)n ? d : 0.0;
      vertex[lane * STEP + j] = at < (uint32_t)n ? vx : (uint8_t)0xFFu;
    }
    at = at < (uint32_t)n ? nx : 0xFFFFu;
  }
  kp_sync();
  for (int k = 0; k < n_stretch; ++k) {
    const uint64_t vx = *(const uint64_t*)(vertex + k * STEP);
    double d[STEP];
#pragma unroll
    for (int j = 0; j < STEP; ++j) d[j] = time[k * STEP + j];
#pragma unroll
    for (int j = 0; j < STEP; ++j) m += (int)((vx >> (8 * j)) & 0xFFu) == lane ? d[j] : 0.0;   // (no sum is a negative zero: zero leaves it as it is)
  }
  return m;
}

// Pair relations and vertex sets of one plan by POSITION in the order of first appearance (bit 8i+j of a
// 64-bit word: positions i and j; bit i of a 32-bit word: position i).
struct KpOrdered {
  unsigned long long ovl, eq, same_model, train_same;
  unsigned train, trainable;
  bool coresident;
};
__device__ inline unsigned kp_row(unsigned long long m, int i) { return (unsigned)(m >> (8 * i)) & 0xFFu; }

__device__ inline bool kp_maximal_clique(int nv, unsigned long long ovl, unsigned M) {
  bool clique = true, maximal = true;
#pragma unroll
  for (int i = 0; i < RPEG_MAX_V; ++i) {
    if (i >= nv) break;
    const bool in = (M >> i) & 1u;
    const bool fits = (M & ~kp_row(ovl, i)) == 0;
    clique = clique && !(in && !fits);
    maximal = maximal && !(!in && fits);
  }
  return clique && maximal;
}

// device_class_peak of rpeg_core.h on position-indexed masks; vm[i * 4 + f] holds w_shard, mem_w, opt and
// extra of the vertex at position i.  M is uniform, so is the control flow; every loop runs over the
// compile-time bound and nothing is indexed dynamically.
__device__ inline double kp_class_peak(const rpeg_problem_t& P, const rpeg_struct_t& st, const uint8_t* order, int nv,
                                       const KpOrdered& om, const double* vm, unsigned M) {
  double persistent = 0.0;
  int groups = 0;
#pragma unroll
  for (int i = 0; i < RPEG_MAX_V; ++i) {   // distinct (model, allocation) worker keys
    if (!((M >> i) & 1u)) continue;
    if ((kp_row(om.eq, i) & M & kp_row(om.same_model, i) & ((1u << i) - 1u)) == 0) ++groups;
  }
  if (om.coresident) {   // the co-resident sum model, as in device_class_peak (vm[i * 4 + 2] carries dp)
    double stat = 0.0, transient = 0.0;
#pragma unroll
    for (int i = 0; i < RPEG_MAX_V; ++i) {
      if (!((M >> i) & 1u)) continue;
      transient = dmax(transient, vm[i * 4 + 3]);
      const unsigned same = M & kp_row(om.same_model, i);
      if (same & ((1u << i) - 1u)) continue;
      double wmax = 0.0, dp = vm[i * 4 + 2];
      bool trained = false;
#pragma unroll
      for (int q = 0; q < RPEG_MAX_V; ++q) {
        if (!((same >> q) & 1u)) continue;
        wmax = dmax(wmax, vm[q * 4 + 0]);
        if ((om.train >> q) & 1u) { trained = true; dp = vm[q * 4 + 2]; }
      }
      const double sbw = (double)P.model[st.vertex[order[i]].model].sb * wmax;
      double x = sbw;
      if (trained) x = (sbw + 12.0 * wmax / (P.optimizer_stage >= 1 ? dp : 1.0)) + sbw / (P.optimizer_stage >= 2 ? dp : 1.0);
      stat += x;
    }
    double peak = ((double)groups * P.group_overhead + stat) + transient;
    if (P.max_groups > 0 && groups > P.max_groups) peak = __builtin_inf();
    return peak;
  }
#pragma unroll
  for (int i = 0; i < RPEG_MAX_V; ++i)     // optimizer shards of the training vertices
    if (((M & om.train & om.trainable) >> i) & 1u) persistent += vm[i * 4 + 2];
  unsigned serving = 0;                    // serving shards: one per worker key that is not a training worker
#pragma unroll
  for (int i = 0; i < RPEG_MAX_V; ++i) {
    if (!(((M & om.trainable & ~om.train) >> i) & 1u)) continue;
    const unsigned same_key = kp_row(om.eq, i) & M & kp_row(om.same_model, i);
    if (same_key & kp_row(om.train_same, i)) continue;
    const bool first = (same_key & serving) == 0;
    serving |= 1u << i;
    if (!first) continue;
    double ws = 0.0;
#pragma unroll
    for (int q = 0; q < RPEG_MAX_V; ++q)
      if (((same_key & ~om.train) >> q) & 1u) ws = dmax(ws, vm[q * 4 + 0]);
    persistent += (double)P.model[st.vertex[order[i]].model].sb * ws;
  }
#pragma unroll
  for (int i = 0; i < RPEG_MAX_V; ++i) {   // frozen weights: one entry per model, its largest shard
    if (!(((M & ~om.trainable) >> i) & 1u)) continue;
    const unsigned same = M & kp_row(om.same_model, i);
    if (same & ((1u << i) - 1u)) continue;
    double wb = 0.0;
#pragma unroll
    for (int q = 0; q < RPEG_MAX_V; ++q)
      if ((same >> q) & 1u) wb = dmax(wb, vm[q * 4 + 1]);
    persistent += wb;
  }
  double top = 0.0;
#pragma unroll
  for (int i = 0; i < RPEG_MAX_V; ++i) {
    if (!((M >> i) & 1u)) continue;
    const bool resident = !((om.trainable >> i) & 1u) || (kp_row(om.eq, i) & serving & kp_row(om.same_model, i)) != 0;
    const double c = resident ? vm[i * 4 + 3] : vm[i * 4 + 1] + vm[i * 4 + 3];
    top = dmax(top, c);
  }
  double peak = (double)groups * P.group_overhead + persistent + top;
  if (P.max_groups > 0 && groups > P.max_groups) peak = __builtin_inf();   // memory.py:699-704
  (void)nv;
  return peak;
}

// Trace.utilization() (RPEG/schedule/trace.py:53-101) of the plan just scheduled: the mean over the devices that
// any node reserved of busy time / makespan, where a device's busy time is the measure of the union of the
// (start, finish) spans of the nodes whose reserved allocations hold it, merged in sorted order, and the mean is
// a running sum over the devices in the order in which the trace first met them (dispatch order of the nodes;
// within a node the source allocation before the destination; within an allocation rack-major) divided by
// their number.  The additions are done in exactly that order: the result equals the reference's bit for bit.
//
// All devices held by the same set of vertex allocations have the same spans, so the busy time is computed once
// per set (lane m takes the set with bit pattern m) over the nodes in dispatch order -- on one device that is
// the sorted order, because a node starts no earlier than the nodes dispatched before it on its devices ended.
// Then the vertices are taken in the order of their first reservation, and the devices of each allocation that
// no earlier one holds are added 64 at a time: the lanes find set and value of their device, one running sum
// takes the values in lane order.  l_start / l_fin: per node; l_order: node dispatched k-th; l_tab: 64 doubles;
// l_span / l_set: two doubles and a byte per node in dispatch order.
//
// Bound: one chain of compares and adds per node, whose operands are therefore brought into dispatch order first, a node
// per lane, and read four nodes at a time; values are added from constant lanes, zeros where there is no device.  (Class
// records fetched within the chain, and a loop over the devices found: outputs of an AC-share plan 50-70 us, now 21-25; a
// launch of 41 such plans of 92-300 nodes 298 -> 248 us, one evaluation of a PPO plan 264 -> 248.)
__device__ inline double kp_utilization(const ClassView& cv, const int n, const int lane, const int nv, const int16_t* l_plan,
                                        const uint64_t dpne, const double* l_start, const double* l_fin,
                                        const uint16_t* l_order, double* l_tab, double2* l_span, uint8_t* l_set, const double ms) {
  if (!(ms > 0.0) || n == 0) return 0.0;
  // vertices by first reservation, four bits each: of node number k, a transfer's source before its destination
  uint32_t first = 0xFFFFFFFFu;   // lane v: when vertex v is first reserved
  unsigned seen = 0u;
  for (int base = 0; base < n; base += KE_WAVE) {
    const int k = base + lane, i = (int)l_order[k < n ? k : base];
    NodeRec nr;
    const uint64_t bits = ((const uint64_t*)cv.node)[i];
    __builtin_memcpy(&nr, &bits, 8);
    const unsigned b = k < n ? blocked_mask(nr, dpne) : 0u;
    if (k < n) l_span[k] = make_double2(l_start[i], l_fin[i]);
    if (k < ((n + 3) & ~3)) l_set[k] = (uint8_t)b;
    for (int v = 0; v < nv; ++v) {
      const mask64 has = __ballot((b >> v) & 1u);
      if (!has || ((seen >> v) & 1u)) continue;
      const int at = __builtin_ctzll(has);
      const unsigned cond = (unsigned)__builtin_amdgcn_readlane((int)nr.cond, at);
      if (lane == v) first = (uint32_t)(base + at) << 4 | (cond && (cond - 1u) >> 3 == (unsigned)v ? 0u : (uint32_t)v + 1u);
      seen |= 1u << v;
    }
  }
  kp_sync();
  {
    const unsigned mine = (unsigned)lane;
    double merged = 0.0, cs = -1.0, ce = -1.0;   // (no span yet: one of no length)
    for (int k = 0; k < n; k += 4) {
      const uint32_t sets = *(const uint32_t*)(l_set + k);
#pragma unroll
      for (int j = 0; j < 4; ++j) {   // (behind the last node: sets without a vertex)
        const double2 t = l_span[k + j];
        const bool in = ((sets >> (8 * j)) & mine) != 0u;
        const double s = in ? t.x : -__builtin_inf(), f = in ? t.y : -__builtin_inf(), span = ce - cs;
        const bool apart = s > ce;
        merged = apart ? merged + span : merged;
        cs = apart ? s : cs;
        ce = apart || f > ce ? f : ce;
      }
    }
    merged += ce - cs;
    l_tab[lane] = merged / ms;
  }
  kp_sync();
  uint32_t order = 0u;
  const int n_ev = __builtin_popcount(seen);
  for (int v = 0; v < nv; ++v) {
    const uint32_t f = (uint32_t)__builtin_amdgcn_readlane((int)first, v);
    if ((seen >> v) & 1u) order |= (uint32_t)v << (4 * __builtin_popcountll(__ballot(first < f)));
  }
  double total = 0.0;
  int count = 0;
  unsigned earlier = 0u;
  for (int e = 0; e < n_ev; ++e) {
    const int v = (int)((order >> (4 * e)) & 15u);
    const int16_t* bx = l_plan + v * RPEG_FIELDS;
    const int ro = bx[4], qo = bx[5], go = bx[6], re = bx[7], qe = bx[8], ge = bx[9];
    const uint32_t ng = (uint32_t)(qe * ge), cnt = (uint32_t)re * ng;
    const uint32_t m_ng = 0xFFFFFFFFu / ng + 1u, m_g = 0xFFFFFFFFu / (uint32_t)ge + 1u;   // exact quotients below 2^16
    for (uint32_t base = 0; base < cnt; base += 64u) {
      const uint32_t idx = base + (uint32_t)lane;
      const uint32_t r = ng == 1u ? idx : __umulhi(idx, m_ng);
      const uint32_t rem = idx - r * ng;
      const uint32_t q = ge == 1 ? rem : __umulhi(rem, m_g);
      const int R = ro + (int)r, Q = qo + (int)q, G = go + (int)(rem - q * (uint32_t)ge);
      unsigned M = 0u;
#pragma unroll
      for (int x = 0; x < RPEG_MAX_V; ++x) {
        const int16_t* p = l_plan + x * RPEG_FIELDS;
        const bool in = x < nv && R >= p[4] && R < p[4] + p[7] && Q >= p[5] && Q < p[5] + p[8] && G >= p[6] && G < p[6] + p[9];
        M |= in ? 1u << x : 0u;
      }
      const double val = l_tab[M & 63u];
      const bool fresh = idx < cnt && (M & earlier) == 0u;
      const mask64 all = __ballot(fresh);
      const double add = fresh ? val : 0.0;   // (the sum is not negative: zero leaves it as it is)
      count += (int)__builtin_popcountll(all);
#pragma unroll
      for (int j0 = 0; j0 < 64; j0 += 16) {
        if (!((all >> j0) & 0xFFFFull)) continue;
#pragma unroll
        for (int j = j0; j < j0 + 16; ++j) total += kp_readlane(add, j);
      }
    }
    earlier |= 1u << v;
  }
  return count ? total / (double)count : 0.0;
}

// What wavefront 3 of a block finds out while the others go on, and flags of the durations.
struct KpShared {
  double peak, pen;
  uint32_t gates;      // RPEG_MASK_STALE_OK | RPEG_MASK_MEM_OK
  uint32_t err;        // bit w: wavefront w met a node the reference raises for
  uint32_t head, off;  // of the plan's record
};

// The fields of plan pi into LDS, by one wavefront: header bytes (structure, split, tau0, tau1).  rec: lane l < 32 holds
// word l of the plan's record where the launch has records.
__device__ inline uint32_t kp_load_plan(const EvalLaunch& L, const uint64_t pi, const uint32_t rec, const int nv, const int lane,
                                        int16_t* l_plan) {
  if (L.rec) {
    if (lane < KP_PLAN_I16 / 2) ((uint32_t*)l_plan)[lane] = lane < RPEG_MAX_V * RPEG_FIELDS / 2 ? rec : 0x00010001u;
    return (uint32_t)__builtin_amdgcn_readlane((int)rec, RPEG_MAX_V * RPEG_FIELDS / 2);
  }
  for (int x = lane; x < KP_PLAN_I16; x += KE_WAVE) l_plan[x] = x < nv * RPEG_FIELDS ? L.vert[(uint64_t)x * L.stride + pi] : (int16_t)1;
  const uint32_t b = L.head[(uint64_t)(lane & 3) * L.stride + pi];
  return (uint32_t)__builtin_amdgcn_readlane((int)b, 0) | (uint32_t)__builtin_amdgcn_readlane((int)b, 1) << 8 |
         (uint32_t)__builtin_amdgcn_readlane((int)b, 2) << 16 | (uint32_t)__builtin_amdgcn_readlane((int)b, 3) << 24;
}

// Memory model (memory.py:608-841) of the plan, by one wavefront, in the order of first appearance of the vertices among
// the lowered operator nodes (position i = vertex vorder[i]): that order fixes the order of the float sums.
// One vertex per lane (kp_memory_vertices), then one vertex subset per lane tests whether it is a device class (a maximal
// clique of the overlap graph); the few that are get evaluated one after the other with uniform control flow.
__device__ inline KpOrdered kp_memory_vertices(const rpeg_problem_t& P, const rpeg_struct_t& st, const ClassView& cv, const int lane,
                                               const int16_t* l_plan, double* l_vm) {
  const int nv = st.n_vertex;
  const uint8_t* order = cv.h->vorder;
  const bool coresident = struct_coresident(st);
  if (lane < nv) {
    const int v = order[lane];
    const VMem m = vertex_memory(P, st.vertex[v], ke_vplan<1>(l_plan, v), coresident);
    l_vm[lane * 4 + 0] = (double)m.w_shard;
    l_vm[lane * 4 + 1] = m.mem_w;
    l_vm[lane * 4 + 2] = m.opt;
    l_vm[lane * 4 + 3] = m.extra;
  }
  KpOrdered om;
  const int i = lane >> 3, j = lane & 7;
  const bool valid = i < nv && j < nv;
  const int vi = order[valid ? i : 0], vj = order[valid ? j : 0];
  const VPlan ai = ke_vplan<1>(l_plan, vi), aj = ke_vplan<1>(l_plan, vj);
  const rpeg_vertex_t &xi = st.vertex[vi], &xj = st.vertex[vj];
  om.ovl = __ballot(valid && !alloc_disjoint(ai, aj));
  om.eq = __ballot(valid && alloc_equal(ai, aj));
  om.same_model = __ballot(valid && xi.model == xj.model);
  om.train_same = __ballot(valid && xi.model == xj.model && xj.role == RPEG_ROLE_TRAIN);
  const unsigned long long t = __ballot(valid && j == 0 && xi.role == RPEG_ROLE_TRAIN),
                           tr = __ballot(valid && j == 0 && st.mem_trainable[xi.model] != 0);   // bit 8i: position i
  om.train = om.trainable = 0u;
  om.coresident = coresident;
#pragma unroll
  for (int q = 0; q < RPEG_MAX_V; ++q) {
    om.train |= (unsigned)((t >> (8 * q)) & 1ull) << q;
    om.trainable |= (unsigned)((tr >> (8 * q)) & 1ull) << q;
  }
  return om;
}
__device__ inline double kp_memory_peak(const rpeg_problem_t& P, const rpeg_struct_t& st, const ClassView& cv, const int lane,
                                        const KpOrdered& om, const double* l_vm) {
  const int nv = st.n_vertex;
  kp_sync();
  double peak = -1.0;
  const unsigned M = (unsigned)lane + 1u;
  unsigned long long classes = __ballot(M < (1u << nv) && kp_maximal_clique(nv, om.ovl, M));
  while (classes) {
    const unsigned Mu = (unsigned)__builtin_ctzll(classes) + 1u;
    classes &= classes - 1ull;
    const double p = kp_class_peak(P, st, cv.h->vorder, nv, om, l_vm, Mu);
    peak = p > peak ? p : peak;
  }
  return peak;
}

// One plan, evaluated by NW wavefronts (this is number `wave`).  pi: plan index (uniform).  head: its header bytes, with
// its fields in LDS.  TR (KpTrace): what the outputs of the launch need of the schedule -- nothing, the times for
// L.mass, the dispatch order too for L.util and L.trace.
//
// NW = 4, for launches whose plans all find a place at once: what one wavefront does one after the other for 13 us before
// its first rank is known is shared out by kind -- generation, other operators, transfers, the memory model -- because
// the kinds are branches of divergent code that a single wavefront walks through in turn; all four count positions; and
// three fetch what the critical chain needs of the class while the first one schedules.
// Measured, 150 PPO plans (K = 4) in one launch: to the first rank 14.7 -> 4.7 us, positions 5.6 -> 4.9 (300 nodes: 34 ->
// 14.5), a plan 73 -> 61 us on average, the launch 128 -> 110 us.
template <int TR, int NW>
__device__ inline void kp_eval_plan(const EvalLaunch& L, const uint64_t w, const uint64_t pi, const int wave, const uint32_t head,
                                    const ClassView cv, uint8_t* lds, KpShared& shared) {
  const int lane = (int)__lane_id();
  const rpeg_problem_t& P = *L.P;
  const int n = (int)cv.h->n_nodes, n_slots = (int)cv.h->n_slots;
  const int first_lane = NW == 1 || wave == 0 ? 0 : -1;

  int16_t* l_plan = (int16_t*)lds;
  double* l_vm = (double*)(lds + KP_PLAN_I16 * 2);
  LevelRec* l_rec = (LevelRec*)(l_vm + RPEG_MAX_V * 4);     // (sixteen-byte boundary, as the two areas behind it)
  double* l_rank = (double*)(l_rec + L.ws_nodes);
  double* l_start = l_rank + (L.ws_nodes + 1);
  double* l_dur = l_start + (L.ws_nodes + 1);
  double* l_tab = l_dur + L.ws_slots;
  uint32_t* l_at = (uint32_t*)(l_tab + 64);
  uint16_t* l_q = (uint16_t*)(l_at + L.ws_nodes);
  // over the two maps: dispatch order and node numbers, then, behind the schedule, the critical chain's predecessors; and
  // the vertex a node counts for
  uint16_t* l_ord = (uint16_t*)l_at;
  uint16_t* l_next = l_ord + L.ws_nodes;
  uint8_t* l_pt = (uint8_t*)l_q;
  const KpLds M{(const KP_LDS double*)l_dur, (KP_LDS LevelRec*)l_rec, (KP_LDS double*)l_rank, (KP_LDS double*)l_start,
                (KP_LDS uint32_t*)l_at, (KP_LDS uint16_t*)l_q, (KP_LDS uint16_t*)l_ord, (KP_LDS uint16_t*)l_next, (KP_LDS uint8_t*)l_pt};

  KE_STAMP(0);
  const rpeg_struct_t& st = P.st[cv.h->structure];
  const int nv = st.n_vertex;
  PlanMasks pm;
  pm.ovl = pm.eq = pm.dpne = 0;
  bool err = cv.h->error != 0, stale_ok = false, mem_ok = false;
  double peak = -1.0, pen = 1.0;
  if (NW == 1 && L.aux_ovl) {
    // a task of a laid-out batch: the prologue launches have left the durations of the slot universe, the pair
    // relations, the penalty factor and the gate bits by plan index (and written the peak themselves)
    const uint64_t sp = pi;
    bool bad = false;
    for (int s = lane; s < n_slots; s += KE_WAVE) {
      const double d = L.dur[(size_t)cv.umap[s] * L.dur_stride + sp];
      l_dur[s] = d;
      bad = bad || d != d;
    }
    err = err || __ballot(bad) != 0ull;
    pm.ovl = L.aux_ovl[sp];
    pm.dpne = L.aux_dpne[sp];
    pen = L.aux_pen ? L.aux_pen[sp] : 1.0;
    const uint8_t gates = L.aux_mask ? L.aux_mask[sp] : (uint8_t)(RPEG_MASK_VALID | RPEG_MASK_STALE_OK | RPEG_MASK_MEM_OK);
    stale_ok = (gates & RPEG_MASK_STALE_OK) != 0;
    mem_ok = (gates & RPEG_MASK_MEM_OK) != 0;
    kp_stage((const uint8_t*)cv.h, M);
    kp_sync();
    KE_STAMP(1);
    KE_STAMP(2);
  } else {
    PlanHead h;
    h.structure = (int)(head & 0xFFu); h.split = (int)((head >> 8) & 0xFFu);
    h.tau0 = (int)((head >> 16) & 0xFFu); h.tau1 = (int)(head >> 24);

    // ---- pair relations: lane 8u+v tests vertices u and v, the ballots are the masks
    {
      const int u = lane >> 3, v = lane & 7;
      const bool valid = u < nv && v < nv;
      const VPlan au = ke_vplan<1>(l_plan, valid ? u : 0), av = ke_vplan<1>(l_plan, valid ? v : 0);
      pm.ovl = __ballot(valid && !alloc_disjoint(au, av));
      pm.eq = 0;   // the memory model works on position-indexed masks of its own
      pm.dpne = __ballot(valid && au.dp != av.dp);
    }

    // ---- durations of the class's slots, one slot per lane
    if (NW == 1 && L.dur) {   // (the prologue launch has left those of the slot universe)
      bool bad = false;
      for (int s = lane; s < n_slots; s += KE_WAVE) {
        const double d = L.dur[(size_t)cv.umap[s] * L.dur_stride + pi];
        l_dur[s] = d;
        bad = bad || d != d;
      }
      err = err || __ballot(bad) != 0ull;
    } else if (NW == 1 || wave < 3) {
      bool zero_div = false;
      const int split = (int)cv.h->split;
      for (int s = lane; s < n_slots; s += KE_WAVE) {
        const SlotDesc sd = cv.slot[s];
        if (NW > 1) {
          const int mine = sd.type > SLOT_OP_SUB ? 2 : st.vertex[sd.a].role == RPEG_ROLE_GEN ? 0 : 1;
          if (mine != wave) continue;
        }
        l_dur[s] = ke_slot_duration<1>(P, st, split, sd, l_plan, &zero_div);
      }
      const bool bad = __ballot(zero_div) != 0ull;
      if (NW == 1) err = err || bad;
      else if (bad && lane == 0) atomicOr(&shared.err, 1u);
    }
    if (NW == 1 || wave == 2) kp_stage((const uint8_t*)cv.h, M);
    KpOrdered om;
    if (NW == 1 || wave == 3) om = kp_memory_vertices(P, st, cv, lane, l_plan, l_vm);
    kp_barrier<NW>();
    KE_STAMP(1);
    if (NW > 1) err = err || shared.err != 0u;
    if (NW == 1 || wave == 3) {
      peak = kp_memory_peak(P, st, cv, lane, om, l_vm);
      stale_ok = stale_layout_ok(st, h, pm.ovl);
      mem_ok = !(peak > P.cap);
      if (!mem_ok) pen = oom_penalty(peak, P.cap);
      if (NW > 1 && lane == 0) {
        shared.peak = peak;
        shared.pen = pen;
        shared.gates = (stale_ok ? RPEG_MASK_STALE_OK : 0u) | (mem_ok ? RPEG_MASK_MEM_OK : 0u);
      }
    }
    KE_STAMP(2);
  }
  unsigned long long* stamp = L.prof && lane == first_lane ? L.prof + w * 8 : nullptr;

  // ---- ranks, positions and list scheduling
  double makespan = 0.0;
  const uint64_t order_rec = kp_order_rec(cv, wave * KE_WAVE + lane);
  if (!err && (NW == 1 || wave == 0)) kp_ranks((uint64_t)cv.h, M);
  kp_barrier<NW>();
  if (stamp) stamp[3] = wall_clock64();
  if (!err) kp_positions<NW>((uint64_t)cv.h, wave, order_rec, M);
  if (NW > 1 && wave == 0) {
    peak = shared.peak;
    pen = shared.pen;
    stale_ok = (shared.gates & RPEG_MASK_STALE_OK) != 0u;
    mem_ok = (shared.gates & RPEG_MASK_MEM_OK) != 0u;
  }
  const bool chain = TR != KP_NO_TRACE && L.mass && !err;   // (uniform over the wavefronts, also where there is no schedule)
  if (NW > 1 && wave != 0) {
    if (!chain) return;
    const int v0 = (wave - 1) * KE_WAVE + lane;
    KpHop hop;
    if (v0 < n) hop = kp_hop_of(cv, v0);
    __syncthreads();   // the plan is scheduled
    if (v0 < n) kp_hop(cv, v0, hop, l_rank, l_next, l_pt);
    for (int v = v0 + (NW - 1) * KE_WAVE; v < n; v += (NW - 1) * KE_WAVE) kp_hop(cv, v, kp_hop_of(cv, v), l_rank, l_next, l_pt);
    __syncthreads();
    return;
  }
  if (!err) {
    makespan = kp_schedule<TR>((const uint8_t*)cv.h, n, pm.ovl, pm.dpne, M, stamp);
    err = makespan < 0.0;
  }
  KE_STAMP(5);
  if (L.prof && lane == 0) L.prof[w * 8 + 7] = ((unsigned long long)n << 32) | (unsigned long long)n;

  // ---- outputs
  uint8_t mask = RPEG_MASK_VALID;
  if (stale_ok) mask |= RPEG_MASK_STALE_OK;
  if (mem_ok) mask |= RPEG_MASK_MEM_OK;
  double out_makespan, out_score;
  if (err || makespan == 0.0) {
    out_makespan = out_score = __builtin_nan("");
    mask |= RPEG_MASK_ERROR;
  } else {
    double score = P.score_num / makespan;
    if (!mem_ok) score = score * pen;
    if ((L.flags & RPEG_GATE_STALE) && !stale_ok) score = 0.0;
    out_makespan = makespan;
    out_score = score;
  }
  kp_sync();
  if (TR == KP_TIMES_ORDER && L.trace && !err) {
    double* const t = L.trace;
    uint16_t* const d = (uint16_t*)(t + 2 * (size_t)L.ws_nodes);
    for (int i = lane; i < n; i += KE_WAVE) {
      t[i] = l_start[i];
      t[(size_t)L.ws_nodes + i] = l_rank[i];
      d[i] = l_ord[i];
    }
  }
  double util = 0.0;
  if (TR == KP_TIMES_ORDER && L.util)
    util = err ? __builtin_nan("") : kp_utilization(cv, n, lane, nv, l_plan, pm.dpne, l_start, l_rank, l_ord, l_tab, (double2*)l_rec, l_pt, makespan);
  double m = __builtin_nan("");   // lane x < RPEG_MAX_V: mass of vertex x
  if (chain) {
    if (NW > 1) {
      __syncthreads();
      __syncthreads();   // (the others leave what the walk needs at every node)
    } else {
      kp_sync();
      for (int v = lane; v < n; v += KE_WAVE) kp_hop(cv, v, kp_hop_of(cv, v), l_rank, l_next, l_pt);
      kp_sync();
    }
    if (!err) m = kp_critical_mass(n, lane, l_rank, l_start, l_next, l_pt, (uint8_t*)l_rec);
  }
  if (lane == 0) {
    if (TR == KP_TIMES_ORDER && L.util) L.util[pi] = util;
    if (L.makespan) L.makespan[pi] = out_makespan;
    if (L.peak && !L.aux_ovl) L.peak[pi] = peak;   // (where the memory model is a launch of its own the peak is its output)
    if (L.score) L.score[pi] = out_score;
    if (L.mask) L.mask[pi] = mask;
  }
  if (TR != KP_NO_TRACE && L.mass && lane < RPEG_MAX_V) L.mass[pi * RPEG_MAX_V + lane] = m;
  KE_STAMP(6);
}

#endif  // __HIPCC__

}  // namespace rpeg
#endif
