"""What a user of the framework has it do, as cases that can be timed.

A Graph500 program generates a graph on the device (or hands over an edge list of its own), builds
the CSR, searches it from many roots, validates the trees; a service keeps a graph and answers
batches of queries.  Each kind of case is one of those programs:

  search   `Bfs.run` from each of `roots` roots, then `Bfs.levels` of the last one
  checked  `Bfs.run` and `Bfs.validate` for each root: the benchmark's own loop
  batch    `MultiBfs.run` over all roots at once: uint8 levels on the device, traversed edges
  serve    `serve.Server` answering `roots` queries of `targets` vertices each
  build    `Graph.generate` + `construct`, an engine, one search and its levels (take "levels") or
           the CSR on the host (take "csr")
  list     `Graph.from_edges` of a host edge list + `construct`, then as `build`

Sizes are Graph500 SCALEs (2^scale vertices) and edge factors of this repository's tests and
benchmark (SCALE 12 to 26, edge factor 16) and what lies between them.  Every output is a whole
number: levels (a vertex's depth does not depend on which parent found it; parents do and are
covered by `checked`), counts, or the CSR.
"""
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if os.path.join(ROOT, "graph500-bfs_amd") not in sys.path:
    sys.path.insert(0, os.path.join(ROOT, "graph500-bfs_amd"))

import g500bfs as G  # noqa: E402
import serve  # noqa: E402


def case(kind, scale, roots, edgefactor=16, **more):
    return dict(kind=kind, scale=scale, edgefactor=edgefactor, roots=roots, corebfs=False, **more)


def listed():
    return [
        # one search of a toy graph: launches, hand-offs and the call itself
        dict(case("search", 12, 1, alpha=10.0, beta=14.0), name="search_s12"),
        # a graph whose bitmaps and queues stay in cache, sixteen roots in turn
        dict(case("search", 18, 16, alpha=10.0, beta=14.0), name="search_s18"),
        # the drop-in driver's SCALE-24 run, half its 64 search keys
        dict(case("search", 24, 32, alpha=10.0, beta=14.0), name="search_s24"),
        # the headline benchmark: SCALE 26, 64 search keys
        dict(case("search", 26, 64, alpha=10.0, beta=14.0), name="search_s26"),
        # the benchmark's loop with every tree validated (validation level 2)
        dict(case("checked", 24, 4), name="checked_s24"),
        # one lane word of roots on a graph that fits the last-level cache
        dict(case("batch", 20, 64), name="batch_s20_r64"),
        # a batch that fills its last lane word in part
        dict(case("batch", 24, 200), name="batch_s24_r200"),
        # the benchmark's batched form at its own scale
        dict(case("batch", 26, 128), name="batch_s26_r128"),
        # one burst of queries at a resident graph, more than one batch holds
        dict(case("serve", 23, 300, targets=4), name="serve_s23_q300"),
        # generation and construction up to the first search
        dict(case("build", 24, 1, take="levels"), name="build_s24"),
        # the same with the trees pruned first (the driver's -C)
        dict(case("build", 22, 1, take="levels") | {"corebfs": True}, name="build_core_s22"),
        # a program's own edge list, sizes of no power of two, its CSR read back
        dict(kind="list", vertices=300007, edges=3000001, symmetric=False, corebfs=False,
             take="csr", name="list_3m"),
    ]


def draw(rng):
    kind = rng.choice(("search", "search", "checked", "batch", "batch", "serve", "build", "list"))
    # edge factors below, at and above the benchmark's; the graph of the largest draw stays below
    # the largest listed one
    ef = rng.choice((5, 8, 11, 16, 16, 16, 23, 32))
    if kind == "search":
        scale = rng.randint(10, 25)
        alpha, beta = rng.choice(((10.0, 14.0), (10.0, 14.0), (25.5, 20.6), (4.0, 24.0)))
        c = case("search", scale, rng.randint(1, 48), ef, alpha=alpha, beta=beta)
        c["corebfs"] = scale <= 21 and rng.random() < 0.3
        return c
    if kind == "checked":
        c = case("checked", rng.randint(10, 24), rng.randint(1, 5), ef)
        c["corebfs"] = c["scale"] <= 21 and rng.random() < 0.3
        return c
    if kind == "batch":
        return case("batch", rng.randint(10, 24), rng.randint(1, 256), ef)
    if kind == "serve":
        return case("serve", rng.randint(12, 23), rng.randint(1, 500), ef,
                    targets=rng.randint(1, 9))
    if kind == "build":
        scale = rng.randint(10, 23)
        core = scale <= 21 and rng.random() < 0.3
        return case("build", scale, 1, ef,
                    take="csr" if scale <= 19 and rng.random() < 0.5 else "levels") | \
            {"corebfs": core}
    vertices = int(2 ** rng.uniform(9, 21)) | 1
    edges = int(2 ** rng.uniform(12, 23)) | 1
    return dict(kind="list", vertices=vertices, edges=edges, symmetric=rng.random() < 0.3,
                corebfs=rng.random() < 0.3, take=rng.choice(("csr", "levels")))


def kronecker(c, seed):
    g = G.Graph.generate(c["scale"], c["edgefactor"], 2 + seed, 3 + 7 * seed)
    return g.construct(corebfs=c["corebfs"])


def host_edges(c, seed):
    """A skewed edge list with self loops and repeated edges, both on the host as int64."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    ne, nv = c["edges"], c["vertices"]
    v = torch.zeros(2, ne, dtype=torch.int64, device="cuda")
    for _ in range(max(1, (nv - 1).bit_length())):  # one quadrant of the adjacency matrix a step
        r = torch.rand(ne, generator=gen, device="cuda")
        src = r >= 0.76
        v[0] = 2 * v[0] + src
        v[1] = 2 * v[1] + (((r >= 0.57) & ~src) | (r >= 0.95))
    label = torch.randperm(nv, generator=gen, device="cuda")
    v = label[v % nv]
    if c["symmetric"]:
        v = torch.cat([v, v.flip(0)], dim=1)
    v = v.cpu().numpy()
    return np.ascontiguousarray(v[0]), np.ascontiguousarray(v[1])


def prepare(c, seed):
    s = dict(c=c, seed=seed)
    if c["kind"] in ("list", "build") and c["take"] == "csr":  # room for any graph's columns
        ne = c["edges"] if c["kind"] == "list" else c["edgefactor"] << c["scale"]
        s["col"] = np.zeros(2 * ne, np.uint32)
    if c["kind"] == "list":
        s["v0"], s["v1"] = host_edges(c, seed)
        # the endpoint of an edge between two vertices: a root with something to reach
        s["root"] = int(s["v0"][np.argmax(s["v0"] != s["v1"])])
        return s
    if c["kind"] == "build":
        return s
    s["graph"] = g = kronecker(c, seed)
    roots = g.find_roots(min(c["roots"], 256), r1=seed % 100)
    s["roots"] = np.resize(roots, min(c["roots"], max(1, len(roots))))
    if c["kind"] in ("search", "checked"):
        s["bfs"] = G.Bfs(g)
    elif c["kind"] == "batch":
        s["batch"] = G.MultiBfs(g, max_roots=len(s["roots"]))
    else:
        rng = np.random.default_rng(seed)
        s["server"] = serve.Server([g], max_batch=256, hbm_budget=16 << 30, max_engines_per_graph=2)
        s["queries"] = [(int(roots[rng.integers(len(roots))]),
                         rng.integers(0, g.info.n, c["targets"])) for _ in range(c["roots"])]
    return s


class DeviceLevels:
    """The batch's level arrays where they lie on the device, one row a root."""

    def __init__(self, batch):
        self.batch = batch  # owns the memory
        ptr, stride = batch.device_levels()
        self.__cuda_array_interface__ = dict(shape=(batch.nroots, stride), typestr="|u1",
                                             data=(ptr, False), strides=None, version=2)


INFO = ("log_n", "n", "n_c", "m", "m_sym", "nedges_input", "max_used_vertex", "max_degree",
        "core_vertices", "tree_vertices", "removed_parents", "hd_root")


def taken(graph, s, root):
    """What a program reads of a new graph: its sizes, and its CSR or a first search's levels."""
    if s["c"]["take"] == "csr":
        out = graph.csr()
        col = s["col"]
        col[:len(out["col"])] = out["col"]
        col[len(out["col"]):] = 0
        out["col"] = col
    else:
        bfs = G.Bfs(graph)
        if root is None:
            root = int(graph.find_roots(1)[0])
        out = dict(at=bfs.run(root), levels=bfs.levels())
        bfs.destroy()
    info = graph.refresh().info  # the first engine of a CoreBFS graph completes it
    out["info"] = np.array([getattr(info, f) for f in INFO], np.int64)
    graph.free()
    return out


def run(s):
    c = s["c"]
    if c["kind"] == "search":
        bfs = s["bfs"]
        at = [bfs.run(int(r), c["edgefactor"], c["alpha"], c["beta"]) for r in s["roots"]]
        return dict(at=np.stack(at), levels=bfs.levels())
    if c["kind"] == "checked":
        bfs, at, said = s["bfs"], [], []
        for r in s["roots"]:
            at.append(bfs.run(int(r), c["edgefactor"]))
            ok, te, errs = bfs.validate(int(r))
            said.append([int(ok), te] + list(errs.values()))
        return dict(at=np.stack(at), said=np.array(said, np.int64), levels=bfs.levels())
    if c["kind"] == "batch":
        batch = s["batch"]
        batch.run(s["roots"])
        return dict(levels=torch.as_tensor(DeviceLevels(batch), device="cuda"), te=batch.te())
    if c["kind"] == "serve":
        srv = s["server"]
        queries = [serve.Query(i, 0, root, targets) for i, (root, targets) in enumerate(s["queries"])]
        for q in queries:
            srv.submit(q)
        srv.drain()
        srv.done.clear()
        return dict(te=np.array([q.te for q in queries], np.int64),
                    levels=np.stack([q.levels for q in queries]))
    if c["kind"] == "build":
        return taken(kronecker(c, s["seed"]), s, None)
    graph = G.Graph.from_edges(s["v0"], s["v1"])
    graph.construct(corebfs=c["corebfs"], symmetric_input=c["symmetric"])
    return taken(graph, s, s["root"])


def work(c):
    """Bytes that one pass cannot do without, each input read once and each output written once.

    A search reads one neighbour (4) of every vertex and writes its pred entry (8); levels read the
    entries (8) and write 2.  Validation reads every edge (8) and pred (8).  A batch writes a level
    byte per root and vertex and reads the CSR once.  A build writes and reads the edge list (8
    each) and writes both directions of every edge (4 each), row offsets (8), degrees and both
    vertex maps (4 each).
    """
    if c["kind"] == "list":
        n, ne = c["vertices"], c["edges"] * (2 if c["symmetric"] else 1)
        csr = 4 * ne * (1 if c["symmetric"] else 2) + 20 * n
        # the host's list (16 an edge) is read, and the CSR read back or a search done
        return dict(bytes=16 * ne + 8 * ne + csr + (csr if c["take"] == "csr" else 22 * n), flops=0)
    n = 1 << c["scale"]
    ne = n * c["edgefactor"]
    csr = 8 * ne + 20 * n
    if c["kind"] == "search":
        return dict(bytes=c["roots"] * 12 * n + 10 * n, flops=0)
    if c["kind"] == "checked":
        return dict(bytes=c["roots"] * (12 * n + 8 * ne + 8 * n) + 10 * n, flops=0)
    if c["kind"] == "batch":
        return dict(bytes=c["roots"] * n + csr, flops=0)
    if c["kind"] == "serve":
        batches = -(-c["roots"] // 256)
        return dict(bytes=batches * csr + c["roots"] * c["targets"] * 17, flops=0)
    return dict(bytes=16 * ne + csr + (csr if c["take"] == "csr" else 22 * n), flops=0)
