// rpeg_lower.h - host-side lowering of one class signature into a class blob.
//
// Follows RPEG/passes/unroll.py:85-152 and RPEG/passes/lower.py:330-851 statement by statement on
// vertex indices instead of objects, answering every plan predicate from the signature bits
// (rpeg_class.h).  Node order is the insertion order of the reference's `nodes` dict (with the
// pop-and-reappend of split inference vertices), edge order the append order of its `edges` list:
// both decide scheduler ties.  Also derives what schedule() derives from the graph alone:
// reserved allocations (RPEG/passes/transfer_resources.py:18-148), tie-break keys and chain
// groups (RPEG/schedule/scheduler.py:367-397).
#ifndef RPEG_LOWER_H
#define RPEG_LOWER_H

#include <algorithm>
#include <cstring>
#include <stdexcept>
#include <string>
#include <utility>
#include <vector>

#include "rpeg_class.h"

namespace rpeg {

// What lowering looks up in a problem's structures for every class, found once per problem: the slot universe
// (slot_universe) with every descriptor's place in it, and the relation pair of two vertices.
struct LowerTables {
  static constexpr uint8_t NONE = 0xFF;
  struct Struct {
    SlotDesc uni[RPEG_MAX_UNIVERSE];
    int n_uni;
    uint8_t at[5 * 16 * 8];                 // key() -> place in `uni`
    uint8_t rel[RPEG_MAX_V][RPEG_MAX_V];    // vertex pair -> index in rpeg_struct_t::rel
  } st[RPEG_MAX_STRUCT];
  static_assert(RPEG_MAX_E <= 16 && RPEG_MAX_V <= 16 && RPEG_MAX_PUB <= 16 && RPEG_MAX_PH <= 7 && RPEG_MAX_MODEL <= 7, "fields of a key");
  static unsigned key(unsigned type, unsigned a, unsigned b, unsigned q) { return (type * 16 + a) * 8 + (type == SLOT_RESHARD ? b : q == 0xFF ? 7u : q); }
  // (only: of that structure alone)
  explicit LowerTables(const rpeg_problem_t& P, int only = -1) {
    for (int s = 0; s < RPEG_MAX_STRUCT; ++s) {
      Struct& t = st[s];
      t.n_uni = 0;
      std::memset(t.at, NONE, sizeof t.at);
      std::memset(t.rel, NONE, sizeof t.rel);
      if (s >= P.n_struct || (only >= 0 && s != only)) continue;
      t.n_uni = slot_universe(P, P.st[s], t.uni);
      for (int u = 0; u < t.n_uni && u < RPEG_MAX_UNIVERSE; ++u) {
        const unsigned k = key(t.uni[u].type, t.uni[u].a, t.uni[u].b, t.uni[u].q);
        if (k < sizeof t.at) t.at[k] = (uint8_t)u;
      }
      for (int r = std::min<int>(P.st[s].n_rel, RPEG_MAX_REL) - 1; r >= 0; --r) {   // (of several entries for a pair the first)
        const rpeg_rel_t& x = P.st[s].rel[r];
        if ((unsigned)x.u < RPEG_MAX_V && (unsigned)x.v < RPEG_MAX_V) t.rel[x.u][x.v] = t.rel[x.v][x.u] = (uint8_t)r;
      }
    }
  }
};

struct SigView {
  const rpeg_struct_t* st;
  const LowerTables::Struct* tab;
  uint64_t sig;
  int structure() const { return (int)(sig & 3); }
  int split() const { return (int)((sig >> 2) & 7); }
  int tau(int slot) const { return slot < 0 ? 0 : (int)((sig >> (5 + 2 * slot)) & 3); }
  int rel_index(int u, int v) const {
    const uint8_t r = tab->rel[u][v];
    if (r == LowerTables::NONE) throw std::logic_error("lowering asked for a vertex pair outside the relation table");
    return r;
  }
  unsigned bits(int u, int v) const { return (unsigned)((sig >> (SIG_REL_SHIFT + 4 * rel_index(u, v))) & 15); }
  bool eq(int u, int v) const { return u == v || (bits(u, v) & 3) == 0; }
  bool disjoint(int u, int v) const {
    if (u == v) return false;
    if (!(st->rel[rel_index(u, v)].flags & RPEG_NEED_DISJ))
      throw std::logic_error("disjointness queried for a pair that does not record it");
    return (bits(u, v) & 3) == 2;
  }
  bool pi_eq(int u, int v) const {
    if (u == v) return true;
    if (!(st->rel[rel_index(u, v)].flags & RPEG_NEED_PI)) throw std::logic_error("pi equality not recorded");
    return (bits(u, v) & 4) != 0;  // recorded only when the allocations are equal
  }
};

struct LoweredNode {
  int kind;     // 0 OP, 1 COMM, 2 RESHARD
  int vertex;   // OP: template vertex
  int step;     // OP: unroll step k
  int sub;      // OP: -1 unsplit, else phase index
  int a0, a1;   // COMM/RESHARD: source / destination vertex (allocations)
  int weight;   // COMM/RESHARD: label starts with "W_"
  int model;    // RESHARD: model
  int slot;
  bool alive;
};

struct LoweredClass {
  std::vector<LoweredNode> nodes;          // alive nodes, reference order
  std::vector<std::pair<int, int>> edges;  // indices into nodes, reference order
  std::vector<uint8_t> blob;
};

// Whether the nodes of[beg[k]], ... of every chain k follow each other within their tie-break class, in that order and with no
// other node of the class between them, and each is a successor of the one before it.  k_quad gives all of them the rank of the
// first, which it finds by the place in the chain.
inline bool chains_in_sequence(const int* beg, size_t n_chains, const int* of, const int* adj_beg, const int* adj_to, const NodeRec* recs) {
  for (size_t k = 0; k < n_chains; ++k)
    for (int j = beg[k] + 1; j < beg[k + 1]; ++j) {
      const int u = of[j - 1], v = of[j];
      if (u > v || recs[u].ptkey != recs[v].ptkey) return false;
      for (int w = u + 1; w < v; ++w)
        if (recs[w].ptkey == recs[u].ptkey) return false;
      if (std::find(adj_to + adj_beg[u], adj_to + adj_beg[u + 1], v) == adj_to + adj_beg[u + 1]) return false;
    }
  return true;
}

// Lowers one class after the other; run() leaves the last one in `out`.  A class is lowered on the critical path of the
// first call that meets it, so the arrays live as long as the object and keep their memory, the slots are found through
// the problem's tables, an edge is looked for among its source's few successors, and the blob's records are written where
// they belong.  us per class (one core of a 2.7 GHz host; with arrays of its own for every class, slots and universe searched
// linearly and an open-addressing table of edges -> now): PPO, 84 nodes 11.4 -> 6.0; GRPO, 47 nodes 6.2 -> 3.2; AC-share,
// 150 nodes 16.0 -> 9.1; PPO of 4 steps, 91 nodes 11.2 -> 5.7.  With what k_quad keeps (few_lanes): 6.7, 3.4, 11.0 and 6.7.
class Lowering {
 public:
  LoweredClass out;

  Lowering(const rpeg_problem_t& problem, const LowerTables& tables) : P(problem), T(tables) {}

  // few_lanes: with what only k_quad reads of a class (QuadRec), a sixth to a fifth of the rest in time, a tenth in bytes.
  // The calls that give every plan a wavefront lower without it, on the calling thread (the first pass on 100 new PPO plans
  // 378 -> 340 us, on 41 AC-share plans 634 -> 561); a class that they have met first is lowered once more when it comes up in a
  // batch for k_quad.
  void run(uint64_t sig_bits, bool few_lanes = true) {
    const int s = (int)(sig_bits & 3);
    const SigView sg{&P.st[s], &T.st[s], sig_bits};
    if (T.st[s].n_uni > RPEG_MAX_UNIVERSE) throw std::runtime_error("slot universe too large");
    graph(sg);
    blob(sg, few_lanes);
  }

 private:
  const rpeg_problem_t& P;
  const LowerTables& T;
  // the graph under construction: per node its first and last outgoing edge, per edge the next one of its source
  std::vector<int> out_first, out_last, out_next;
  std::vector<SlotDesc> slots;
  std::vector<uint8_t> umap;                  // per slot: its place in the structure's slot universe
  uint8_t slot_at[RPEG_MAX_UNIVERSE];         // place in the universe -> slot
  std::vector<int> base, gfirst, ifirst;
  std::vector<std::pair<int, int>> pass1, pass2;
  std::vector<int> n_po, n_so, a_po, a_so, remap;
  struct Tr { int node, pred, succ; };
  std::vector<Tr> to_train, to_serving;
  // and what the blob needs of it
  std::vector<int> adj_beg, adj_to, indeg, deg, cur, topo, chain_beg, chain_of, level, place, chain_n, chain_i, lbeg;
  // and what k_quad keeps of it (few_lanes)
  std::vector<uint64_t> anc, row_pred;        // a bit each: per node its ancestors; per row the predecessors of the last node that has it
  std::vector<int> row_of;                    // per node: its ready-time row
  std::vector<uint16_t> types;
  std::vector<uint8_t> type_of;               // per node
  uint8_t type_at[RPEG_MAX_V * 8 + 1][1 << RPEG_MAX_V] = {};   // (cond, blocked) -> type + 1; all zero between classes
  int n_rows = 0, n_rank_rows = 0;
  std::vector<int> rank_row, by_place, freed_first, freed_next, free_rows;   // per node, by place, per level, per node, rows
  // Reservation types and ready-time rows (QuadRec); false where they outgrow its fields.  W: words of a set of nodes.
  template <int W>
  bool quad_rows(const NodeRec* recs, const uint16_t* pbeg, const uint16_t* pred, int n) {
    anc.resize((size_t)n * W);   // (in topological order a node's set is written before it is read)
    row_pred.resize((size_t)(QUAD_ROWS + 1) * W);
    row_of.assign(n, 0); type_of.resize(n);
    n_rows = 1;
    for (int v : topo) {
      uint8_t& type = type_at[recs[v].cond][recs[v].blocked];
      if (!type) {
        types.push_back((uint16_t)(recs[v].blocked | recs[v].cond << 8));
        type = (uint8_t)types.size();
      }
      type_of[v] = (uint8_t)(type - 1);
      if (recs[v].indeg > QUAD_INDEG || types.size() > QUAD_TYPES) return false;
      uint64_t* const a = &anc[(size_t)v * W];
      const uint16_t* const p = pred + pbeg[v];
      const int d = recs[v].indeg;
      if (d == 0) { for (int w = 0; w < W; ++w) a[w] = 0; continue; }
      uint64_t all[W], common[W], own[W] = {};   // ancestors that some predecessor has, and that all have; the predecessors
      for (int w = 0; w < W; ++w) all[w] = common[w] = anc[(size_t)p[0] * W + w];
      own[p[0] >> 6] |= 1ull << (p[0] & 63);
      for (int j = 1; j < d; ++j) {
        const uint64_t* const x = &anc[(size_t)p[j] * W];
        for (int w = 0; w < W; ++w) { all[w] |= x[w]; common[w] &= x[w]; }
        own[p[j] >> 6] |= 1ull << (p[j] & 63);
      }
      for (int w = 0; w < W; ++w) a[w] = all[w] | own[w];
      if (d < 2) continue;
      int r = 1;
      for (; r < n_rows; ++r) {
        uint64_t missing = 0;
        for (int w = 0; w < W; ++w) missing |= row_pred[(size_t)r * W + w] & ~common[w];
        if (!missing) break;
      }
      if (r > (int)QUAD_ROWS) return false;
      n_rows = std::max(n_rows, r + 1);
      for (int w = 0; w < W; ++w) row_pred[(size_t)r * W + w] = own[w];
      row_of[v] = r;
    }
    return true;
  }
  bool quad_rows(const NodeRec* recs, const uint16_t* pbeg, const uint16_t* pred, int n) {
    static_assert(QUAD_NODES < 8 * 64, "sets of up to eight words");
    types.clear();
    if (n > (int)QUAD_NODES || (int)topo.size() != n) return false;
    const auto f = [&] {
      switch ((n + 63) / 64) {
        case 0: case 1: return quad_rows<1>(recs, pbeg, pred, n);
        case 2: return quad_rows<2>(recs, pbeg, pred, n);
        case 3: return quad_rows<3>(recs, pbeg, pred, n);
        case 4: return quad_rows<4>(recs, pbeg, pred, n);
        default: return quad_rows<8>(recs, pbeg, pred, n);
      }
    };
    const bool fits = f();
    for (uint16_t t : types) type_at[t >> 8][t & 0xFFu] = 0;
    return fits;
  }

  // Rows of the rank pass (RankRec), level by level: a row is given on in the level behind the last one that reads it.  False
  // where there are too many.
  bool rank_rows(const uint16_t* pbeg, const uint16_t* pred, int n, int n_levels) {
    rank_row.resize(n); by_place.resize(n); freed_next.resize(n);
    freed_first.assign(n_levels, -1);   // per level: the nodes whose rows it reads last
    for (int v = 0; v < n; ++v) by_place[place[v]] = v;
    free_rows.clear();
    n_rank_rows = 2;
    for (int l = 0; l < n_levels; ++l) {
      if (l > 0)
        for (int v = freed_first[l - 1]; v >= 0; v = freed_next[v]) free_rows.push_back(rank_row[v]);
      for (int i = lbeg[l]; i < lbeg[l + 1]; ++i) {
        const int v = by_place[i];
        int last = -1;
        for (int j = pbeg[v]; j < pbeg[v + 1]; ++j) last = std::max(last, level[pred[j]]);
        rank_row[v] = 1;
        if (last < 0) continue;
        if (free_rows.empty()) {
          rank_row[v] = n_rank_rows++;
        } else {
          rank_row[v] = free_rows.back();
          free_rows.pop_back();
        }
        freed_next[v] = freed_first[last];
        freed_first[last] = v;
      }
    }
    return n_rank_rows <= (int)RANK_ROWS;
  }

  int slot(const SigView& sg, SlotType t, int a, int b, int q) {
    const uint8_t u = sg.tab->at[LowerTables::key(t, (unsigned)a, (unsigned)b, (unsigned)q)];
    if (u == LowerTables::NONE) throw std::logic_error("a duration slot outside the slot universe");
    if (slot_at[u] == LowerTables::NONE) {
      slot_at[u] = (uint8_t)slots.size();
      slots.push_back(sg.tab->uni[u]);
      umap.push_back(u);
    }
    return slot_at[u];
  }
  int add_node(const LoweredNode& n) {
    out.nodes.push_back(n);
    out_first.push_back(-1);
    out_last.push_back(-1);
    return (int)out.nodes.size() - 1;
  }
  void add_edge(int a, int b) {
    for (int e = out_first[a]; e >= 0; e = out_next[e])
      if (out.edges[e].second == b) return;
    const int e = (int)out.edges.size();
    out.edges.push_back({a, b});
    out_next.push_back(-1);
    (out_last[a] < 0 ? out_first[a] : out_next[out_last[a]]) = e;
    out_last[a] = e;
  }
  void graph(const SigView& sg) {
    const rpeg_struct_t& st = *sg.st;
    const int nv = st.n_vertex, K = P.K_eval, split = sg.split();
    const int nph = split > 0 ? P.n_phase[split] : 0;
    std::vector<LoweredNode>& nodes = out.nodes;
    std::vector<std::pair<int, int>>& edges = out.edges;
    nodes.clear(); edges.clear(); out_first.clear(); out_last.clear(); out_next.clear(); slots.clear(); umap.clear();
    std::memset(slot_at, LowerTables::NONE, sizeof slot_at);

    // per (vertex, step): the unsplit node; the first of the generation / inference sub-nodes (they are created one
    // after the other, so sub-node q of a vertex and step is first + q; -1: none)
    base.assign((size_t)nv * K, -1); gfirst.assign((size_t)nv * K, -1); ifirst.assign((size_t)nv * K, -1);
    auto at = [&](int v, int k) { return (size_t)v * K + k; };

    // which generation vertices split: quantile phases exist and some inference consumer is disjoint
    unsigned gen_split = 0;
    if (nph > 0)
      for (int e = 0; e < st.n_edge; ++e) {
        const rpeg_edge_t& ed = st.edge[e];
        if (st.vertex[ed.src].role == RPEG_ROLE_GEN && st.vertex[ed.dst].role == RPEG_ROLE_INF &&
            sg.disjoint(ed.src, ed.dst))
          gen_split |= 1u << ed.src;
      }

    // 1) operator nodes, step-major in template order (unroll.py:103-110, lower.py:433-474)
    for (int k = 0; k < K; ++k)
      for (int v = 0; v < nv; ++v) {
        if (nph > 0 && st.vertex[v].role == RPEG_ROLE_GEN && ((gen_split >> v) & 1u)) {
          for (int q = 0; q < nph; ++q) {
            const int id = add_node({0, v, k, q, v, v, 0, st.vertex[v].model, slot(sg, SLOT_OP_SUB, v, 0, q), true});
            if (q == 0) gfirst[at(v, k)] = id;
          }
          for (int q = 1; q < nph; ++q) add_edge(gfirst[at(v, k)] + q - 1, gfirst[at(v, k)] + q);
        } else {
          base[at(v, k)] = add_node({0, v, k, -1, v, v, 0, st.vertex[v].model, slot(sg, SLOT_OP_UNSPLIT, v, 0, 0), true});
        }
      }

    // 2) data edges, generation->inference edges of split generators first (lower.py:476-597)
    auto edge_or_comm = [&](int a, int b, int e, int q) {
      const int va = nodes[a].vertex, vb = nodes[b].vertex;
      if (sg.eq(va, vb)) { add_edge(a, b); return; }
      int c = add_node({1, -1, nodes[a].step, -1, va, vb, st.edge[e].is_weight, -1,
                        slot(sg, SLOT_COMM_DATA, e, 0, q < 0 ? 0xFF : q), true});
      add_edge(a, c);
      add_edge(c, b);
    };
    bool any_dead = false;
    pass1.clear(); pass2.clear();   // (step, edge)
    for (int k = 0; k < K; ++k)
      for (int e = 0; e < st.n_edge; ++e) {
        const rpeg_edge_t& ed = st.edge[e];
        if (gfirst[at(ed.src, k)] >= 0 && st.vertex[ed.dst].role == RPEG_ROLE_INF) pass1.push_back({k, e});
        else pass2.push_back({k, e});
      }
    pass1.insert(pass1.end(), pass2.begin(), pass2.end());
    for (auto& ke : pass1) {
      const int k = ke.first, e = ke.second;
      const rpeg_edge_t& ed = st.edge[e];
      const int u = ed.src, v = ed.dst;
      const int gu = gfirst[at(u, k)];
      const bool src_gen_split = gu >= 0;
      if (src_gen_split && st.vertex[v].role == RPEG_ROLE_INF) {
        if (sg.disjoint(u, v)) {
          if (ifirst[at(v, k)] < 0) {
            if (base[at(v, k)] >= 0) { nodes[base[at(v, k)]].alive = false; any_dead = true; base[at(v, k)] = -1; }
            for (int q = 0; q < nph; ++q) {
              const int id = add_node({0, v, k, q, v, v, 0, st.vertex[v].model, slot(sg, SLOT_OP_SUB, v, 0, q), true});
              if (q == 0) ifirst[at(v, k)] = id;
            }
            for (int q = 1; q < nph; ++q) add_edge(ifirst[at(v, k)] + q - 1, ifirst[at(v, k)] + q);
          }
          for (int q = 0; q < nph; ++q) edge_or_comm(gu + q, ifirst[at(v, k)] + q, e, q);
        } else {
          edge_or_comm(gu + nph - 1, base[at(v, k)], e, -1);
        }
      } else if (src_gen_split) {
        edge_or_comm(gu + nph - 1, base[at(v, k)], e, -1);
      } else if (ifirst[at(u, k)] >= 0) {
        if (base[at(v, k)] < 0) throw std::runtime_error("destination node of a split inference edge not found");
        edge_or_comm(ifirst[at(u, k)] + nph - 1, base[at(v, k)], e, -1);
      } else {
        if (base[at(u, k)] < 0 || base[at(v, k)] < 0) throw std::runtime_error("edge endpoint missing");
        edge_or_comm(base[at(u, k)], base[at(v, k)], e, -1);
      }
    }

    // 3) within-step weight reshards between consecutive vertices of one trainable model (lower.py:626-681)
    auto last_of = [&](int v, int k) {
      if (gfirst[at(v, k)] >= 0) return gfirst[at(v, k)] + nph - 1;
      if (ifirst[at(v, k)] >= 0) return ifirst[at(v, k)] + nph - 1;
      return base[at(v, k)];
    };
    auto first_of = [&](int v, int k) {
      if (gfirst[at(v, k)] >= 0) return gfirst[at(v, k)];
      if (ifirst[at(v, k)] >= 0) return ifirst[at(v, k)];
      return base[at(v, k)];
    };
    unsigned resharded = 0;
    bool any_reshard = false;
    auto make_reshard = [&](int a, int b, int model) {
      any_reshard = true;
      return add_node({2, -1, nodes[a].step, -1, nodes[a].vertex, nodes[b].vertex, 1, model,
                       slot(sg, SLOT_RESHARD, nodes[a].vertex, model, 0), true});
    };
    for (int p = 0; p < st.n_pair; ++p) {
      const rpeg_pair_t& pr = st.pair[p];
      if (sg.tau(pr.tau_slot) > 0 && sg.disjoint(pr.u, pr.v)) continue;  // shadow pair
      if (pr.reach && !sg.eq(pr.u, pr.v)) continue;
      for (int k = 0; k < K; ++k) {
        const int a = last_of(pr.u, k), b = first_of(pr.v, k);
        const bool same = sg.eq(pr.u, pr.v);
        if (same && sg.pi_eq(pr.u, pr.v)) continue;
        if (!same) { add_edge(a, b); continue; }
        int r = make_reshard(a, b, pr.model);
        add_edge(a, r);
        add_edge(r, b);
        resharded |= 1u << pr.v;
      }
    }

    // 4a) publication edges (unroll.py:121-135, lower.py:683-728)
    for (int k = 1; k < K; ++k)
      for (int p = 0; p < st.n_pub; ++p) {
        const rpeg_pub_t& pb = st.pub[p];
        const int t = sg.tau(pb.tau_slot);
        if (k <= t) continue;
        const int ks = k - (t + 1) > 0 ? k - (t + 1) : 0;
        const int a = base[at(pb.src, ks)];
        const int b = first_of(pb.dst, k);
        if (a < 0 || b < 0) throw std::runtime_error("publication endpoint missing");
        if ((resharded >> pb.dst) & 1u) continue;
        const bool same = sg.eq(pb.src, pb.dst);
        if (same && sg.pi_eq(pb.src, pb.dst)) { add_edge(a, b); continue; }
        int c;
        if (same) c = make_reshard(a, b, pb.model);
        else c = add_node({1, -1, nodes[a].step, -1, pb.src, pb.dst, 1, pb.model, slot(sg, SLOT_COMM_PUB, p, 0, 0), true});
        add_edge(a, c);
        add_edge(c, b);
      }

    // 4b) lifetime barriers between colocated trainable layouts (lower.py:730-793)
    if (any_reshard) {
      // operator predecessors / successors of the reshard nodes: how many, and one of them
      n_po.assign(nodes.size(), 0); n_so.assign(nodes.size(), 0); a_po.assign(nodes.size(), -1); a_so.assign(nodes.size(), -1);
      for (auto& ed : edges) {
        if (nodes[ed.second].kind == 2 && nodes[ed.first].kind == 0) { ++n_po[ed.second]; a_po[ed.second] = ed.first; }
        if (nodes[ed.first].kind == 2 && nodes[ed.second].kind == 0) { ++n_so[ed.first]; a_so[ed.first] = ed.second; }
      }
      to_train.clear(); to_serving.clear();
      for (int i = 0; i < (int)nodes.size(); ++i) {
        if (!nodes[i].alive || nodes[i].kind != 2) continue;
        if (n_po[i] != 1 || n_so[i] != 1) continue;
        const LoweredNode &pn = nodes[a_po[i]], &sn = nodes[a_so[i]];
        if (pn.model != sn.model || !st.trainable[pn.model]) continue;
        const int pr = st.vertex[pn.vertex].role, sr = st.vertex[sn.vertex].role;
        if (pr != RPEG_ROLE_TRAIN && sr == RPEG_ROLE_TRAIN) to_train.push_back({i, a_po[i], a_so[i]});
        else if (pr == RPEG_ROLE_TRAIN && sr != RPEG_ROLE_TRAIN) to_serving.push_back({i, a_po[i], a_so[i]});
      }
      for (auto& rt : to_train)
        for (auto& pb : to_serving) {
          const LoweredNode &producer = nodes[rt.pred], &consumer = nodes[pb.succ];
          if (producer.model == consumer.model || producer.step != consumer.step) continue;
          if (sg.disjoint(producer.vertex, consumer.vertex)) continue;
          if (!st.reach[producer.vertex][consumer.vertex]) continue;
          add_edge(rt.node, pb.node);
        }
    }

    // compact to alive nodes, keep order
    if (any_dead) {
      remap.assign(nodes.size(), -1);
      int n = 0;
      for (int i = 0; i < (int)nodes.size(); ++i)
        if (nodes[i].alive) {
          remap[i] = n;
          nodes[n] = nodes[i];
          out_first[n++] = out_first[i];
        }
      nodes.resize(n);
      for (auto& ed : edges) {
        if (remap[ed.first] < 0 || remap[ed.second] < 0) throw std::runtime_error("edge to a removed node");
        ed = {remap[ed.first], remap[ed.second]};
      }
    }
  }
  void blob(const SigView& sg, bool few_lanes) {
    const rpeg_struct_t& st = *sg.st;
    const int nv = st.n_vertex, K = P.K_eval, split = sg.split();
    const int nph = split > 0 ? P.n_phase[split] : 0;
    const std::vector<LoweredNode>& nodes = out.nodes;
    const std::vector<std::pair<int, int>>& edges = out.edges;
    const int n = (int)nodes.size(), ne = (int)edges.size();
    if (n > 65535) throw std::runtime_error("too many lowered nodes");

    // adjacency in edge order, in-degrees, Kahn order (scheduler.py:28-67)
    adj_beg.resize(n + 1); adj_to.resize(ne);   // (successors of a node in the order of its edges)
    indeg.assign(n, 0);
    int n_init = 0, used = 0;
    for (int i = 0; i < n; ++i) {
      adj_beg[i] = used;
      for (int e = out_first[i]; e >= 0; e = out_next[e]) { adj_to[used++] = edges[e].second; ++indeg[edges[e].second]; }
    }
    adj_beg[n] = used;
    topo.clear();
    deg = indeg;
    for (int i = 0; i < n; ++i) if (deg[i] == 0) topo.push_back(i);
    n_init = (int)topo.size();
    for (size_t h = 0; h < topo.size(); ++h)
      for (int j = adj_beg[topo[h]]; j < adj_beg[topo[h] + 1]; ++j) if (--deg[adj_to[j]] == 0) topo.push_back(adj_to[j]);
    const bool cycle = (int)topo.size() != n;

    // chain groups: quantile sub-nodes of one (vertex, step) (scheduler.py:369-378), the groups in the order of
    // (vertex, step), the members of a group in node order
    auto at = [&](int v, int k) { return (size_t)v * K + k; };
    chain_beg.assign((size_t)nv * K + 1, 0);
    for (int i = 0; i < n; ++i)
      if (nodes[i].kind == 0 && nodes[i].sub >= 0) ++chain_beg[at(nodes[i].vertex, nodes[i].step) + 1];
    int n_groups = 0;
    for (size_t k = 0; k < (size_t)nv * K; ++k) {
      n_groups += chain_beg[k + 1] != 0 ? 1 : 0;
      chain_beg[k + 1] += chain_beg[k];
    }
    const int n_gm = chain_beg.back();
    chain_of.resize(n_gm);
    cur.assign(chain_beg.begin(), chain_beg.end() - 1);
    for (int i = 0; n_gm && i < n; ++i)
      if (nodes[i].kind == 0 && nodes[i].sub >= 0) chain_of[cur[at(nodes[i].vertex, nodes[i].step)]++] = i;

    // vertex order of first appearance among operator nodes (dict orders of memory.py:763-808)
    uint8_t vorder[8] = {0, 1, 2, 3, 4, 5, 6, 7};
    {
      unsigned seen_v = 0;
      int c = 0;
      for (int i = 0; i < n && c < nv; ++i)
        if (nodes[i].kind == 0 && !((seen_v >> nodes[i].vertex) & 1u)) { seen_v |= 1u << nodes[i].vertex; vorder[c++] = (uint8_t)nodes[i].vertex; }
      if (c != nv) throw std::runtime_error("a template vertex has no lowered operator node");
      // The memory launch derives this order from the plan alone (plan_vorder): hold the two to each other here,
      // from the signature's predicates, for every class that is ever lowered.
      unsigned gs = 0, moved = 0;
      uint8_t want[RPEG_MAX_V], tail[RPEG_MAX_V];
      int n_want = 0, n_tail = 0;
      if (nph > 0) {
        for (int e = 0; e < st.n_edge; ++e)
          if (st.edge[e].gen_inf && sg.disjoint(st.edge[e].src, st.edge[e].dst)) gs |= 1u << st.edge[e].src;
        for (int e = 0; e < st.n_edge; ++e) {
          const int u = st.edge[e].src, v = st.edge[e].dst;
          if (!((gs >> u) & 1u) || st.vertex[v].role != RPEG_ROLE_INF || ((moved >> v) & 1u)) continue;
          if (sg.disjoint(u, v)) { moved |= 1u << v; tail[n_tail++] = (uint8_t)v; }
        }
      }
      for (int v = 0; v < nv; ++v)
        if (!((moved >> v) & 1u)) want[n_want++] = (uint8_t)v;
      for (int j = 0; j < n_tail; ++j) want[n_want++] = tail[j];
      for (int v = 0; v < nv; ++v)
        if (want[v] != vorder[v]) throw std::logic_error("vertex order of the lowered graph differs from the plan's own");
    }

    // levels (from the nodes without successors up) and places in their order
    level.assign(n, 0); place.resize(n);
    int n_levels = n ? 1 : 0;
    for (int h = (int)topo.size() - 1; h >= 0; --h) {
      const int v = topo[h];
      int l = 0;
      for (int j = adj_beg[v]; j < adj_beg[v + 1]; ++j) l = std::max(l, level[adj_to[j]] + 1);
      level[v] = l;
      n_levels = std::max(n_levels, l + 1);
    }
    lbeg.assign(n_levels + 1, 0);
    for (int v = 0; v < n; ++v) ++lbeg[level[v] + 1];
    for (int l = 0; l < n_levels; ++l) lbeg[l + 1] += lbeg[l];
    cur.assign(lbeg.begin(), lbeg.end() - 1);
    for (int v = 0; v < n; ++v) place[v] = cur[level[v]]++;

    // the blob
    auto align8 = [](size_t x) { return (x + 7) & ~size_t(7); };
    ClassHdr h{};
    h.n_nodes = n; h.n_slots = (uint32_t)slots.size(); h.n_succ = (uint32_t)used; h.n_init = (uint32_t)n_init;
    h.n_groups = (uint32_t)n_groups; h.n_gmembers = (uint32_t)n_gm;
    h.structure = sg.structure(); h.split = split; h.error = cycle ? 1u : 0u;
    std::memcpy(h.vorder, vorder, 8);
    size_t off = align8(sizeof(ClassHdr));
    h.off_node = (uint32_t)off; off = align8(off + (size_t)n * sizeof(NodeRec));
    h.off_succ = (uint32_t)off; off = align8(off + (size_t)used * 2);
    h.off_init = (uint32_t)off; off = align8(off + (size_t)n_init * 2);
    h.off_topo = (uint32_t)off; off = align8(off + (size_t)n * 2);
    h.off_slot = (uint32_t)off; off = align8(off + slots.size() * sizeof(SlotDesc));
    h.off_group = (uint32_t)off; off = align8(off + (size_t)n_groups * sizeof(GroupRec));
    h.off_gmember = (uint32_t)off; off = align8(off + (size_t)n_gm * 2);
    h.off_pbeg = (uint32_t)off; off = align8(off + ((size_t)n + 1) * 2);
    h.off_pred = (uint32_t)off; off = align8(off + (size_t)ne * 2);
    h.off_umap = (uint32_t)off; off = align8(off + umap.size());
    h.n_levels = (uint32_t)n_levels;
    h.off_lrec = (uint32_t)(off = (off + 15) & ~size_t(15)); off = align8(off + (size_t)n * sizeof(LevelRec));
    h.off_orec = (uint32_t)off; off = align8(off + (size_t)n * sizeof(OrderRec));
    h.off_lbeg = (uint32_t)off; off = align8(off + lbeg.size() * 2);
    h.off_place = (uint32_t)off; off = align8(off + (size_t)n * 2);
    h.off_glvl = (uint32_t)off; off = align8(off + (size_t)n_gm * 2);
    h.off_qrec = (uint32_t)off;
    if (few_lanes) off = align8(rank_rec_offset(h) + ((size_t)n + 2) * sizeof(RankRec));
    h.off_type = (uint32_t)off;   // (the last one: its length is known when the nodes are)
    off = (off + 15) & ~size_t(15);   // (blobs start on sixteen-byte boundaries of the pool)
    out.blob.assign(off + (few_lanes ? 2 * QUAD_TYPES : 0), 0);
    uint8_t* const B = out.blob.data();
    NodeRec* const recs = (NodeRec*)(B + h.off_node);
    uint16_t* const succ = (uint16_t*)(B + h.off_succ);
    for (int i = 0; i < n; ++i) {
      const LoweredNode& nd = nodes[i];
      NodeRec r{};
      r.succ_begin = (uint16_t)adj_beg[i];
      const int n_adj = adj_beg[i + 1] - adj_beg[i];
      if (n_adj > 255 || indeg[i] > 255 || adj_beg[i + 1] > 65535)
        throw std::runtime_error("node degree out of range");
      r.n_succ = (uint8_t)n_adj;
      for (int j = adj_beg[i]; j < adj_beg[i + 1]; ++j) succ[j] = (uint16_t)adj_to[j];
      r.slot = (uint8_t)nd.slot;
      r.indeg = (uint8_t)indeg[i];
      if (nd.kind == 0) {
        r.ptkey = (uint8_t)(8 + st.vertex[nd.vertex].topo_idx);
        r.blocked = (uint8_t)(1u << nd.vertex);
      } else {
        r.ptkey = (uint8_t)nv;  // comm_prio 0, topo_idx = number of template ids (scheduler.py:391-397)
        // transfer_resources.py:73-148.  "destination_only": weights reserve the destination, activations
        // also the source unless both adjacent operators use the same dp (a per-plan bit).
        // "both_endpoints" for the payload class: source and destination, whatever dp is.  A reshard's
        // two allocations are one and the same.
        const bool both = nd.kind == 1 && (P.transfer_both >> (nd.weight ? 0 : 1) & 1);
        r.blocked = (uint8_t)(1u << nd.a1 | (both ? 1u << nd.a0 : 0u));
        // (with both endpoints reserved the condition adds nothing to `blocked`; it is kept as the record of which
        // endpoint is the source: the utilisation lists a transfer's source devices before its destination's)
        r.cond = nd.weight && !both ? 0 : (uint8_t)(1 + nd.a0 * 8 + nd.a1);
      }
      recs[i] = r;
    }
    uint16_t* const init = (uint16_t*)(B + h.off_init);
    for (int i = 0; i < n_init; ++i) init[i] = (uint16_t)topo[i];   // (the Kahn order begins with the nodes without predecessors)
    uint16_t* const topo16 = (uint16_t*)(B + h.off_topo);
    for (size_t i = 0; i < topo.size(); ++i) topo16[i] = (uint16_t)topo[i];
    if (!slots.empty()) std::memcpy(B + h.off_slot, slots.data(), slots.size() * sizeof(SlotDesc));
    if (!umap.empty()) std::memcpy(B + h.off_umap, umap.data(), umap.size());
    GroupRec* group = (GroupRec*)(B + h.off_group);
    for (size_t k = 0; k < (size_t)nv * K; ++k)
      if (chain_beg[k + 1] != chain_beg[k]) *group++ = GroupRec{(uint16_t)chain_beg[k], (uint16_t)(chain_beg[k + 1] - chain_beg[k])};
    uint16_t *const gmember = (uint16_t*)(B + h.off_gmember), *const glvl = (uint16_t*)(B + h.off_glvl);
    for (int k = 0; k < n_gm; ++k) { gmember[k] = (uint16_t)chain_of[k]; glvl[k] = (uint16_t)place[chain_of[k]]; }
    // predecessors in edge order
    uint16_t *const pbeg = (uint16_t*)(B + h.off_pbeg), *const pred = (uint16_t*)(B + h.off_pred);
    cur.resize(n);
    for (int i = 0; i < n; ++i) { cur[i] = pbeg[i]; pbeg[i + 1] = (uint16_t)(pbeg[i] + indeg[i]); }
    for (auto& ed : edges) pred[cur[ed.second]++] = (uint16_t)ed.first;
    if (few_lanes) {
      if (chains_in_sequence(chain_beg.data(), (size_t)nv * K, chain_of.data(), adj_beg.data(), adj_to.data(), recs) && quad_rows(recs, pbeg, pred, n) && rank_rows(pbeg, pred, n, n_levels)) {
        h.n_rows = (uint32_t)n_rows;
        h.n_types = (uint32_t)types.size();
        std::memcpy(B + h.off_type, types.data(), types.size() * 2);
        uint32_t* const qrec = (uint32_t*)(B + h.off_qrec);
        for (int v = 0; v < n; ++v)
          qrec[place[v]] = std::min<uint32_t>(recs[v].n_succ, 7u) | (uint32_t)recs[v].indeg << 3 | (uint32_t)recs[v].slot << 10 | (uint32_t)type_of[v] << 18 | (uint32_t)row_of[v] << 24;
      }
      off = (h.off_type + (size_t)h.n_types * 2 + 15) & ~size_t(15);
      out.blob.resize(off);   // (never more: B stays)
    }
    h.bytes = (uint32_t)off;
    std::memcpy(B, &h, sizeof h);
    // the orders of the one-plan-per-wavefront kernel: by level, and by tie-break class
    LevelRec* const lrec = (LevelRec*)(B + h.off_lrec);
    uint16_t *const lbeg16 = (uint16_t*)(B + h.off_lbeg), *const place16 = (uint16_t*)(B + h.off_place);
    for (size_t l = 0; l < lbeg.size(); ++l) lbeg16[l] = (uint16_t)lbeg[l];
    for (int v = 0; v < n; ++v) {
      const NodeRec& nr = recs[v];
      LevelRec r;
      for (int j = 0; j < 4; ++j) r.succ[j] = (uint16_t)(j < nr.n_succ ? place[adj_to[adj_beg[v] + j]] : n);
      r.node = (uint16_t)v;
      r.slot = nr.slot; r.blocked = nr.blocked; r.cond = nr.cond; r.indeg = nr.indeg;
      r.n_succ = nr.n_succ; r.pad = 0;
      lrec[place[v]] = r;
      place16[v] = (uint16_t)place[v];
    }
    OrderRec* const orec = (OrderRec*)(B + h.off_orec);
    RankRec* const rrec = (RankRec*)(B + rank_rec_offset(h));   // (with rows)
    int first[257] = {}, next[256];
    for (int v = 0; v < n; ++v) ++first[recs[v].ptkey + 1];
    for (int k = 0; k < 256; ++k) { next[k] = first[k]; first[k + 1] += first[k]; }
    chain_n.assign(n, 1); chain_i.assign(n, 0);
    for (size_t k = 0; n_gm && k < (size_t)nv * K; ++k) {
      const int count = chain_beg[k + 1] - chain_beg[k];
      if (count > 255) throw std::runtime_error("chain group too long");
      for (int j = 0; j < count; ++j) { chain_n[chain_of[chain_beg[k] + j]] = count; chain_i[chain_of[chain_beg[k] + j]] = j; }
    }
    for (int v = 0; v < n; ++v) {
      const int k = recs[v].ptkey;
      if (h.n_rows) {
        RankRec r{};
        for (int j = 0; j < 4 && j < recs[v].n_succ; ++j) r.succ[j] = (uint8_t)rank_row[adj_to[adj_beg[v] + j]];
        r.row = (uint8_t)rank_row[v];
        r.slot = recs[v].slot;
        r.id = (uint16_t)((uint32_t)next[k] | (recs[v].n_succ > 4 ? RANK_MORE : 0u));
        rrec[place[v]] = r;
      }
      orec[next[k]++] = OrderRec{(uint16_t)place[v], (uint16_t)first[k], (uint16_t)first[k + 1], (uint8_t)chain_n[v], (uint8_t)chain_i[v]};
    }
    if (h.n_rows) {
      rrec[n] = RankRec{{0, 0, 0, 0}, 1, 0, (uint16_t)n};
      rrec[n + 1] = RankRec{{0, 0, 0, 0}, 1, 0, (uint16_t)n_rank_rows};
    }
  }
};

// one class of a problem (a caller with many keeps the tables and a Lowering)
inline LoweredClass lower_class(const rpeg_problem_t& P, uint64_t sig_bits, bool few_lanes = true) {
  const LowerTables tables(P, (int)(sig_bits & 3));
  Lowering l(P, tables);
  l.run(sig_bits, few_lanes);
  return std::move(l.out);
}

}  // namespace rpeg
#endif
