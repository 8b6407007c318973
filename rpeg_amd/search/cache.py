"""Evaluation cache and canonical configuration hash (mirror of RPEG/search/cache.py:22-185)."""

import hashlib
import json
from dataclasses import dataclass, field
from operator import itemgetter
from typing import Dict, Optional, Tuple


@dataclass
class EvalCache:
    _store: Dict[str, Tuple[float, object, bool]] = field(default_factory=dict)
    hits: int = 0
    misses: int = 0   # unique evaluations stored

    def get(self, key: str) -> Optional[Tuple[float, object, bool]]:
        if key in self._store:
            self.hits += 1
            return self._store[key]
        return None

    def put(self, key: str, score: float, trace, feasible: bool) -> None:
        self._store[key] = (score, trace, feasible)
        self.misses += 1

    def __contains__(self, key: str) -> bool:
        return key in self._store

    def size(self) -> int:
        return len(self._store)

    def stats(self) -> str:
        total = self.hits + self.misses
        rate = self.hits / total if total > 0 else 0.0
        return f"hits={self.hits}  misses={self.misses}  total={total}  hit_rate={rate:.1%}"


def _container(c) -> dict:
    return {"name": c.name, "count": c.count, "elem": c.elem_size_bytes}


def _vertex(v) -> dict:
    by_name = lambda x: x["name"]  # noqa: E731
    return {"id": v.id, "role": v.kind.role.value, "model": v.kind.model.value,
            "read": sorted((_container(c) for c in v.kind.read), key=by_name),
            "write": sorted((_container(c) for c in v.kind.write), key=by_name)}


def _edge(e) -> dict:
    return {"src": e.src.id, "dst": e.dst.id, "container": _container(e.container)}


_dumps = json.JSONEncoder(separators=(",", ":"), sort_keys=True).encode   # (json.dumps makes an encoder a call: 3 us)
_graph_text = {}   # id(rpeg) -> (rpeg, _KeyText of the template)


class _KeyText:
    """What of a key's text depends on the template only: the four entries of the template graph, and, for a plan that gives
    every template vertex whole numbers, the whole text as a format and the places of its numbers in the plan's row."""

    def __init__(self, rpeg):
        ends = lambda x: (x["src"], x["dst"])  # noqa: E731
        self.data_edges = _dumps(sorted((_edge(e) for e in rpeg.data_edges), key=ends))
        self.pub_edges = _dumps(sorted((_edge(e) for e in rpeg.pub_edges), key=ends))
        self.tau = _dumps({m.value: t for m, t in rpeg.tau.items()})
        self.vertices = _dumps(sorted((_vertex(v) for v in rpeg.vertices), key=lambda x: x["id"]))
        ids = [v.id for v in rpeg.vertices]
        # (of other names, or none, json makes the text)
        self.vertex_of = tuple(rpeg.vertices) if ids and len(set(ids)) == len(ids) and all(type(x) is str for x in ids) else None
        if self.vertex_of is None:
            return
        order = sorted(range(len(ids)), key=ids.__getitem__)
        name = [_dumps(x).replace("%", "%%") for x in ids]
        three = "[%d,%d,%d]"
        entries = (",".join(name[x] + ":%d" for x in order), ",".join(name[x] + ":" + three for x in order),
                   ",".join(f'{name[x]}:{{"extent":{three},"origin":{three}}}' for x in order))
        fixed = [x.replace("%", "%%") for x in (self.data_edges, self.pub_edges, self.tau, self.vertices)]
        self.format = ('{"data_edges":%s,"mb":{%s},"pi":{%s},"pub_edges":%s,"sigma":{%s},"tau":%s,"vertices":%s}' %
                       (fixed[0], entries[0], entries[1], fixed[1], entries[2], fixed[2], fixed[3]))
        row = 10     # of a vertex: three degrees, micro-batches, origin, extent
        self.places = itemgetter(*([row * x + 3 for x in order] + [row * x + f for x in order for f in (0, 1, 2)] +
                                   [row * x + f for x in order for f in (7, 8, 9, 4, 5, 6)]))

    def of_row(self, row) -> str:
        return hashlib.sha256((self.format % self.places(row)).encode("utf-8")).hexdigest()

    def row_of(self, plan):
        """The plan as a row of whole numbers; None where it is none, or covers other vertices than the template's."""
        verts, row = self.vertex_of, []
        parts = by_vertex(verts, plan) if verts is not None else None
        if parts is None:
            return None
        for a, p, m in parts:
            if not len(p) == len(a.origin) == len(a.extent) == 3:
                return None
            row += (*p, m, *a.origin, *a.extent)
        return row if set(map(type, row)) == {int} else None


def by_vertex(verts, plan):
    """(allocation, degrees, micro-batches) of each of the vertices `verts` (a tuple), for a plan of these and no others; else None.
    (Tables in the order of the vertices, as they mostly are, are read in that order: a look-up hashes the vertex.)"""
    sigma, pi, mb = plan.sigma, plan.pi, plan.mb
    if tuple(sigma) == verts and tuple(pi) == verts and tuple(mb) == verts:
        return zip(sigma.values(), pi.values(), mb.values())
    if not len(sigma) == len(pi) == len(mb) == len(verts) or any(v not in sigma or v not in pi or v not in mb for v in verts):
        return None
    return [(sigma[v], pi[v], mb[v]) for v in verts]


def key_text(rpeg) -> _KeyText:
    hit = _graph_text.get(id(rpeg))
    if hit is not None and hit[0] is rpeg:
        return hit[1]
    text = _KeyText(rpeg)
    if len(_graph_text) >= 64:
        _graph_text.clear()
    _graph_text[id(rpeg)] = (rpeg, text)
    return text


def config_hash(rpeg, plan) -> str:
    """sha256 of the canonical JSON of (template graph, plan); same payload and key order as the
    reference (RPEG/search/cache.py:160-185: keys sorted at every level, no blanks), so keys are
    interchangeable with caches it wrote.  The text is put together from its seven top-level entries in key
    order; what depends on the template alone is kept per template object, since a search hashes
    thousands of plans of a few templates."""
    text = key_text(rpeg)
    row = text.row_of(plan)
    if row is not None:
        return text.of_row(row)
    sigma = _dumps({v.id: {"origin": list(a.origin), "extent": list(a.extent)} for v, a in plan.sigma.items()})
    pi = _dumps({v.id: list(p) for v, p in plan.pi.items()})
    mb = _dumps({v.id: m for v, m in plan.mb.items()})
    whole = ('{"data_edges":' + text.data_edges + ',"mb":' + mb + ',"pi":' + pi + ',"pub_edges":' + text.pub_edges +
             ',"sigma":' + sigma + ',"tau":' + text.tau + ',"vertices":' + text.vertices + "}")
    return hashlib.sha256(whole.encode("utf-8")).hexdigest()


def _config_hash_plain(rpeg, plan) -> str:
    """The same key from one json.dumps of the whole payload, as the reference writes it; kept to check the
    assembled text against."""
    by_id = lambda kv: kv[0].id  # noqa: E731
    ends = lambda x: (x["src"], x["dst"])  # noqa: E731
    payload = {
        "vertices": sorted((_vertex(v) for v in rpeg.vertices), key=lambda x: x["id"]),
        "data_edges": sorted((_edge(e) for e in rpeg.data_edges), key=ends),
        "pub_edges": sorted((_edge(e) for e in rpeg.pub_edges), key=ends),
        "tau": {m.value: t for m, t in sorted(rpeg.tau.items(), key=lambda kv: kv[0].value)},
        "sigma": {v.id: {"origin": list(a.origin), "extent": list(a.extent)}
                  for v, a in sorted(plan.sigma.items(), key=by_id)},
        "pi": {v.id: list(p) for v, p in sorted(plan.pi.items(), key=by_id)},
        "mb": {v.id: m for v, m in sorted(plan.mb.items(), key=by_id)},
    }
    text = json.dumps(payload, separators=(",", ":"), sort_keys=True)
    return hashlib.sha256(text.encode("utf-8")).hexdigest()
