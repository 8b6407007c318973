// rpeg_kernel_prologue.h - the part of a plan's evaluation that is plain arithmetic, as launches of their own
// (device only).
//
// The list scheduler is a chain of dependent steps: the kernels that run it (rpeg_kernel_eval.h, _quad.h, _plan.h)
// keep one or two wavefronts on a SIMD and issue an instruction every ten clocks or so.  Inside those kernels the
// cost model (NodeCostModel.time of every duration slot, cost.py:66-686) and the memory model (per-device peaks,
// memory.py:608-887) cost the same ten clocks an instruction, a fifth to a quarter of a wavefront's time, although
// nothing in them waits for anything.
//
// Neither depends on the lowering class of a plan: a duration is a function of the plan fields and of which slot
// it is -- so every slot a class of the plan's structure COULD have (slot_universe) is evaluated, and a class picks
// its own through ClassView::umap --, and the vertex order that fixes the memory model's float sums follows from the
// plan (plan_vorder).  Both launches therefore run on the plans in the caller's own order, straight from the
// caller's tensors (coalesced), right behind the signature kernel: while the class totals are on their way to the
// host, which lays the batch out, i.e. off the critical path of the call.
//
//   k_prologue   one wavefront per (64 plans, row); a row is one slot of the universe, or the pair relations, or one
//                vertex's memory terms -- a wavefront holds one short piece of arithmetic, so that many are resident
//                dur[u][i]            duration of universe slot u for plan i (rows dur_stride apart), NaN where the
//                                     reference would raise ZeroDivisionError; not written for the phases a plan's
//                                     split variant does not have
//                aux_ovl / _eq / _dpne  pair relations (PlanMasks), per plan
//                vm[v * 4 + f][i]     per-vertex memory terms (kpro_vmem)
//   k_peaks      peak[i]              the call's own output: largest device peak
//                aux_pen[i]           factor of the soft OOM penalty (evaluate.py:396-401), 1.0 where the plan fits
//                aux_mask[i]          RPEG_MASK_VALID | _STALE_OK | _MEM_OK
#ifndef RPEG_KERNEL_PROLOGUE_H
#define RPEG_KERNEL_PROLOGUE_H

#include "rpeg_kernel_eval.h"

namespace rpeg {

constexpr int KPRO_PARTS = 6;                    // wavefronts that share the rows of a block of 64 plans, at least
constexpr uint32_t KPRO_INVALID = 0xFFFFFFFFu;   // class id of a plan that breaks an integer rule: not evaluated

// The tasks of a batch of a wavefront per plan: start (or null), [class * shards + shard], the first task of the class's plans of that
// shard; what a plan's own is, its class's blob and the plan go into the task.  Where *not_lowered there are none yet.
struct DealtTasks {
  const uint32_t *start, *kidx, *coff, *not_lowered;
  uint32_t shards;
  uint32_t *perm, *task_cls, *limit;
};

struct PrologueLaunch {
  const rpeg_problem_t* P;
  const int16_t* vert;         // the caller's plan tensors
  const uint8_t* head;
  uint64_t stride, n;
  const uint32_t* cid;         // per plan: KPRO_INVALID for a plan the gate rejected
  const SlotDesc* uni;         // [structure][RPEG_MAX_UNIVERSE]
  uint32_t n_uni[RPEG_MAX_STRUCT];
  uint32_t max_uni;            // rows: max_uni durations, one row of pair relations, then one per vertex
  uint32_t row_begin, row_end; // the rows of a launch of the first kind
  double* dur;
  uint64_t dur_stride;         // plans per row of dur and vm
  uint64_t* aux_ovl;
  uint64_t* aux_eq;
  uint64_t* aux_dpne;
  double* vm;                  // [vertex * 4 + field][plan]: memory terms of every vertex (kpro_vmem)
  double* aux_pen;
  uint8_t* aux_mask;
  double* peak;                // or null
  DealtTasks deal;             // beside durations for k_plan
};

#if defined(__HIPCC__)

__device__ inline VPlan kpro_vplan(const int16_t* p, uint64_t stride, int v) {
  p += (uint64_t)v * RPEG_FIELDS * stride;
  VPlan a;
  a.dp = p[0 * stride]; a.pp = p[1 * stride]; a.tp = p[2 * stride]; a.mb = p[3 * stride];
  a.o[0] = p[4 * stride]; a.o[1] = p[5 * stride]; a.o[2] = p[6 * stride];
  a.e[0] = p[7 * stride]; a.e[1] = p[8 * stride]; a.e[2] = p[9 * stride];
  return a;
}

// (the pieces are functions of their own, not inlined: each gets the registers it needs instead of the kernel holding
// the union of all of them, which costs it its residency)
// (NaN where the reference would raise ZeroDivisionError: a flag handed in by address would live in scratch memory)
__device__ __attribute__((noinline)) double kpro_op_time(const rpeg_problem_t& P, const rpeg_vertex_t& vx, const rpeg_opconst_t& oc,
                                                         const int16_t* pl, uint64_t stride, int v) {
  bool zero_div = false;
  const double t = op_time(ke_common(P), ke_common(vx), oc, kpro_vplan(pl, stride, v), &zero_div);   // (the constants: those of the lane's own split)
  return zero_div ? __builtin_nan("") : t;
}

__device__ inline double kpro_slot_duration(const rpeg_problem_t& P, const rpeg_struct_t& st, int split, const SlotDesc sd,
                                            const int16_t* pl, uint64_t stride) {
  switch (sd.type) {
    case SLOT_OP_UNSPLIT:
      return kpro_op_time(P, st.vertex[sd.a], st.vertex[sd.a].unsplit, pl, stride, sd.a);
    case SLOT_OP_SUB:
      return kpro_op_time(P, st.vertex[sd.a], st.vertex[sd.a].sub[split][sd.q], pl, stride, sd.a);
    case SLOT_COMM_DATA: {
      const rpeg_edge_t& e = st.edge[sd.a];
      const int64_t payload = sd.q == 0xFF ? e.full_bytes : e.sub_bytes[split][sd.q];
      return comm_time(P, kpro_vplan(pl, stride, e.src), kpro_vplan(pl, stride, e.dst), payload, e.is_weight != 0);
    }
    case SLOT_COMM_PUB: {
      const rpeg_pub_t& p = st.pub[sd.a];
      const VPlan s = kpro_vplan(pl, stride, p.src), d = kpro_vplan(pl, stride, p.dst);
      return comm_time(P, s, d, pub_payload(P, s, d, p.model), true);
    }
    default:
      return reshard_time(P, kpro_vplan(pl, stride, sd.a), sd.b);
  }
}

// (these take what they need by value: the address of the launch record would force a copy of it into scratch memory
// in every wavefront)
__device__ __attribute__((noinline)) void kpro_masks(const int16_t* pl, const uint64_t stride, const int nv, uint64_t* ovl,
                                                     uint64_t* eq, uint64_t* dpne) {
  VPlan a[RPEG_MAX_V];
#pragma unroll
  for (int v = 0; v < RPEG_MAX_V; ++v)
    if (v < nv) a[v] = kpro_vplan(pl, stride, v);
  const PlanMasks pm = plan_masks(a, nv);
  *ovl = pm.ovl;
  *eq = pm.eq;
  *dpne = pm.dpne;
}

__device__ __attribute__((noinline)) void kpro_vmem(const rpeg_problem_t& P, const int16_t* pl, const uint64_t stride,
                                                    const rpeg_struct_t& st, const int v, double* out, const uint64_t out_stride) {
  const rpeg_struct_t& su = ke_common(st);
  const int x = __builtin_amdgcn_readfirstlane(v);
  const bool coresident = struct_coresident(su);
  const VMem m = vertex_memory(ke_common(P), su.vertex[x], kpro_vplan(pl, stride, x), coresident);
  // (of shards of one model the largest is looked for, whose product is the largest product)
  const double w = (double)m.w_shard, served = (double)ke_common(P).model[su.vertex[x].model].sb * w;
  out[0 * out_stride] = coresident ? w : served;
  out[1 * out_stride] = coresident ? served : m.mem_w;
  out[2 * out_stride] = m.opt;
  out[3 * out_stride] = m.extra;
}

// Plan i of this lane, structure su (uniform), one row of the first launch's grid (uniform): the duration of one slot
// of the universe; or the pair relations of the plan; or the memory terms of one vertex.
__device__ inline void kpro_row(const PrologueLaunch& L, const uint64_t i, const int su, const int split, const int row) {
  const rpeg_problem_t& P = ke_common(*L.P);
  const rpeg_struct_t& st = P.st[su];
  const int16_t* pl = L.vert + i;
  if (row < (int)L.max_uni) {
    if (row >= (int)L.n_uni[su]) return;
    const SlotDesc sd = ke_common(L.uni[(size_t)su * RPEG_MAX_UNIVERSE + row]);   // uniform
    if (!slot_in_split(P, split, sd)) return;                          // this lane's split variant has no such phase
    L.dur[(uint64_t)row * L.dur_stride + i] = kpro_slot_duration(P, st, split, sd, pl, L.stride);
  } else if (row == (int)L.max_uni) {
    kpro_masks(pl, L.stride, st.n_vertex, L.aux_ovl + i, L.aux_eq + i, L.aux_dpne + i);
  } else {
    const int v = row - (int)L.max_uni - 1;
    if (v < st.n_vertex) kpro_vmem(P, pl, L.stride, st, v, L.vm + (uint64_t)(v * 4) * L.dur_stride + i, L.dur_stride);
  }
}

// plan_vorder (rpeg_class.h) from the pair relations instead of the plan fields: two allocations are disjoint exactly
// when they do not intersect.  Four bits a position.
__device__ inline uint32_t kpro_vorder(const rpeg_problem_t& P, const rpeg_struct_t& st, int split, uint64_t ovl) {
  const int nv = st.n_vertex, nph = split > 0 ? P.n_phase[split] : 0;
  unsigned gen_split = 0, moved = 0;
  uint32_t order = 0u, c = 0u;
  auto disjoint = [&](int u, int v) { return !((ovl >> (8 * u + v)) & 1ull); };
  if (nph > 0) {
    for (int e = 0; e < st.n_edge; ++e)
      if (st.edge[e].gen_inf && disjoint(st.edge[e].src, st.edge[e].dst)) gen_split |= 1u << st.edge[e].src;
    for (int e = 0; e < st.n_edge; ++e) {
      const int u = st.edge[e].src, v = st.edge[e].dst;
      if (((gen_split >> u) & 1u) && st.vertex[v].role == RPEG_ROLE_INF && disjoint(u, v)) moved |= 1u << v;
    }
  }
  for (int v = 0; v < nv; ++v)
    if (!((moved >> v) & 1u)) { order |= (uint32_t)v << c; c += 4u; }
  if (moved == 0u) return order;
  unsigned done = 0;   // the vertices taken out, in the order of the edges that split them
  for (int e = 0; e < st.n_edge; ++e) {
    const int u = st.edge[e].src, v = st.edge[e].dst;
    if (!((moved >> v) & 1u) || ((done >> v) & 1u)) continue;
    if (((gen_split >> u) & 1u) && st.vertex[v].role == RPEG_ROLE_INF && disjoint(u, v)) {
      done |= 1u << v;
      order |= (uint32_t)v << c;
      c += 4u;
    }
  }
  return order;
}

// The maximal cliques among the first NV vertices (clique_sets of rpeg_core.h).
template <int NV, int V, unsigned M>
__device__ inline void kpro_cliques(const unsigned (&row)[NV], const unsigned c, uint64_t& found) {
  if constexpr (V == NV) {
    if (M != 0u && c == M) found |= 1ull << M;
  } else {
    kpro_cliques<NV, V + 1, M>(row, c, found);
    kpro_cliques<NV, V + 1, (M | (1u << V))>(row, c & row[V], found);
  }
}

// device_peak_max of rpeg_core.h for the plan of this lane; no structure of the problem has more than NV vertices.  Everything lies in
// registers: the memory terms are fetched in the order in which the reference sums them, a plan's own (what column of the
// table a lane reads is its affair), and every loop runs over the compile-time bound.
// Bound: vector issue, and the scheduling kernels beside it, which leave it registers but hardly any LDS.  With terms and order in
// LDS, indexed at run time, its wavefronts waited for LDS to become free and then for their reads: 1,048,576 DPO plans, three
// vertices, 64 / now 35 us; 65,536 GRPO, four, 41 / 21; 262,144 AC-share, six, 563 / 172; 20,011 PPO 117 / 50.  (Both memory models in
// one loop: the terms that it shares out ahead of the loop took 60 registers more than there are.)
template <int NV, bool CORESIDENT>
__device__ inline double kpro_peak(const rpeg_problem_t& P, const rpeg_struct_t& st, const uint64_t ovl, const uint64_t eq,
                                                      const uint32_t order, const double* vm, const uint64_t stride) {
  const int nv = st.n_vertex;
  double x[NV][4];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    if (i >= nv) break;
    const double* const t = vm + (uint64_t)(((order >> (4 * i)) & 0xFu) * 4u) * stride;
#pragma unroll
    for (int f = 0; f < 4; ++f) x[i][f] = t[(uint64_t)f * stride];
  }
  // the structure's vertex sets (uniform): vertices of the same model, training, of trainable models
  uint64_t same_model = 0;
  unsigned train = 0, trainable = 0;
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    if (v >= nv) break;
    if (st.vertex[v].role == RPEG_ROLE_TRAIN) train |= 1u << v;
    if (st.mem_trainable[st.vertex[v].model]) trainable |= 1u << v;
#pragma unroll
    for (int w = 0; w < NV; ++w)
      if (w < nv && st.vertex[w].model == st.vertex[v].model) same_model |= 1ull << (8 * v + w);
  }
  // the same by position; where the order is that of the vertices (no vertex moved), position i is vertex i
  uint64_t key = eq & same_model, model = same_model;   // rows of 8 bits: of the position's worker key, of its model
  unsigned trained = train, learns = trainable;
  const bool moved = order != (0x76543210u & ((1u << (4 * nv)) - 1u));
  if (moved) {
    uint64_t key_at = 0, model_at = 0;
    trained = learns = 0u;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      if (i >= nv) break;
      const uint32_t v = (order >> (4 * i)) & 0xFu;
      const unsigned k = mask_row(key, (int)v), m = mask_row(model, (int)v);
      trained |= ((train >> v) & 1u) << i;
      learns |= ((trainable >> v) & 1u) << i;
#pragma unroll
      for (int j = 0; j < NV; ++j) {
        if (j >= nv) break;
        const uint32_t w = (order >> (4 * j)) & 0xFu;
        key_at |= (uint64_t)((k >> w) & 1u) << (8 * i + j);
        model_at |= (uint64_t)((m >> w) & 1u) << (8 * i + j);
      }
    }
    key = key_at;
    model = model_at;
  }
  unsigned row[NV];
#pragma unroll
  for (int v = 0; v < NV; ++v) row[v] = v < nv ? mask_row(ovl, v) & ((1u << nv) - 1u) : 0u;
  uint64_t found = 0;
  kpro_cliques<NV, 0, 0u>(row, (1u << nv) - 1u, found);
  double best = -1.0;
  while (found) {
    const unsigned set = (unsigned)__builtin_ctzll(found);
    found &= found - 1ull;
    unsigned M = set;
    if (moved) {
      M = 0u;
#pragma unroll
      for (int i = 0; i < NV; ++i)
        if (i < nv) M |= ((set >> ((order >> (4 * i)) & 0xFu)) & 1u) << i;
    }
    int groups = 0;
#pragma unroll
    for (int i = 0; i < NV; ++i) groups += ((M >> i) & 1u) && (mask_row(key, i) & M & ((1u << i) - 1u)) == 0u ? 1 : 0;
    double peak;
    if constexpr (CORESIDENT) {   // fields: parameters, their bytes, dp, transients
      double stat = 0.0, transient = 0.0;
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        if (!((M >> i) & 1u)) continue;
        transient = dmax(transient, x[i][3]);
        const unsigned same = M & mask_row(model, i);
        if (same & ((1u << i) - 1u)) continue;
        double wmax = 0.0, sbw = 0.0, dp = x[i][2];
#pragma unroll
        for (int j = i; j < NV; ++j) {
          if (!((same >> j) & 1u)) continue;
          wmax = dmax(wmax, x[j][0]);
          sbw = dmax(sbw, x[j][1]);
          if ((trained >> j) & 1u) dp = x[j][2];
        }
        double b = sbw;
        if (same & trained) b = (sbw + 12.0 * wmax / (P.optimizer_stage >= 1 ? dp : 1.0)) + sbw / (P.optimizer_stage >= 2 ? dp : 1.0);
        stat += b;
      }
      peak = ((double)groups * P.group_overhead + stat) + transient;
    } else {                      // fields: bytes of the parameters as served, weights, optimizer shard, role extras
      double persistent = 0.0;
#pragma unroll
      for (int i = 0; i < NV; ++i)   // optimizer shards of the training vertices
        if (((M & trained & learns) >> i) & 1u) persistent += x[i][2];
      unsigned serving = 0u;         // serving shards: one per worker key that is not a training worker
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        if (!(((M & learns & ~trained) >> i) & 1u)) continue;
        const unsigned mates = mask_row(key, i) & M;
        if (mates & trained) continue;
        if (!(mates & serving)) {
          double ws = 0.0;
#pragma unroll
          for (int j = 0; j < NV; ++j)
            if ((mates >> j) & 1u) ws = dmax(ws, x[j][0]);
          persistent += ws;
        }
        serving |= 1u << i;
      }
#pragma unroll
      for (int i = 0; i < NV; ++i) { // frozen weights: one entry per model, its largest shard
        if (!(((M & ~learns) >> i) & 1u)) continue;
        const unsigned same = M & mask_row(model, i);
        if (same & ((1u << i) - 1u)) continue;
        double wb = 0.0;
#pragma unroll
        for (int j = i; j < NV; ++j)
          if ((same >> j) & 1u) wb = dmax(wb, x[j][1]);
        persistent += wb;
      }
      double top = 0.0;
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        if (!((M >> i) & 1u)) continue;
        const bool resident = !((learns >> i) & 1u) || (mask_row(key, i) & serving) != 0u;
        top = dmax(top, resident ? x[i][3] : x[i][1] + x[i][3]);
      }
      peak = (double)groups * P.group_overhead + persistent + top;
    }
    if (P.max_groups > 0 && groups > P.max_groups) peak = __builtin_inf();
    if (peak > best) best = peak;
  }
  return best;
}

__device__ __attribute__((noinline)) double kpro_penalty(double peak, double cap) { return oom_penalty(peak, cap); }

// The second launch: largest device peak, penalty factor and gate bits of plan i of this lane, structure su (uniform),
// from the pair relations and the per-vertex memory terms the first launch left.
template <int NV>
__device__ inline void kpro_peaks(const PrologueLaunch& L, const uint64_t i, const int su, const PlanHead h) {
  const rpeg_problem_t& P = ke_common(*L.P);
  const rpeg_struct_t& st = P.st[su];
  const uint64_t ovl = L.aux_ovl[i], eq = L.aux_eq[i];
  const uint32_t order = kpro_vorder(P, st, h.split, ovl);
  const double peak = struct_coresident(st) ? kpro_peak<NV, true>(P, st, ovl, eq, order, L.vm + i, L.dur_stride)
                                            : kpro_peak<NV, false>(P, st, ovl, eq, order, L.vm + i, L.dur_stride);
  const bool stale_ok = stale_layout_ok(st, h, ovl);
  const bool mem_ok = !(peak > P.cap);
  L.aux_pen[i] = mem_ok ? 1.0 : kpro_penalty(peak, P.cap);
  L.aux_mask[i] = (uint8_t)(RPEG_MASK_VALID | (stale_ok ? RPEG_MASK_STALE_OK : 0) | (mem_ok ? RPEG_MASK_MEM_OK : 0));
  if (L.peak) L.peak[i] = peak;
}

#endif  // __HIPCC__

}  // namespace rpeg
#endif
