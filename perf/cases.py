"""The products and training passes whose speed is measured, through research_amd's public entry points.

A case is a dict with a "kind" and its sizes:

  laplacian  C = A*A of the 2D 5-point Laplacian on nx * ny points (ultra-sparse rows)
  rect       C = A*A^T of a short, wide, mostly scattered matrix (ultra-sparse rows, some outliers)
  er         C = A*A of an Erdos-Renyi matrix (uniform rows)
  banded     C = A*A of a banded matrix (products merge: the estimation workflow)
  rmat       C = A*A of an R-MAT graph, (a, b, c) = (.57, .19, .19) (skewed rows, hubs)
  panel      rows of an R-MAT graph's square, cut so that they make `products` products, as a
             program whose C does not fit the card computes it
  replay     a planned product recomputed from A's current values by its captured graph
  batch      many independent products C_i = A_i*A_i at once: "learned" runs them eagerly with the
             trained row-size predictor, "graph" launches the captured whole path
  train      one epoch of the row-size predictor's training

C comes back as (row offsets, column ids, values)."""
import functools
import math

import numpy as np
import torch

import research_amd as ra
from research_amd import ocean, predictor
from research_amd.workloads import batched_products

DEVICE = "cuda"
ABC = (0.57, 0.19, 0.19)


def listed():
    return [
        # the smallest call: a mesh of 4096 points, where launches and waits are all there is
        {"name": "laplacian-64", "kind": "laplacian", "nx": 64, "ny": 64, "f32": False},
        # bench.py's Laplacian
        {"name": "laplacian-256", "kind": "laplacian", "nx": 256, "ny": 256, "f32": False},
        # bench.py's rectangular product, two operands
        {"name": "rect-2^18", "kind": "rect", "rows": 1 << 18, "cols": 1 << 21, "mean": 8.0, "f32": True},
        # a small graph by itself, of the size that the batches are made of
        {"name": "rmat-2^13", "kind": "rmat", "log_n": 13, "degree": 16.0, "f32": True},
        # uniform sparsity, an odd size
        {"name": "er-100003", "kind": "er", "n": 100003, "degree": 24.0, "f32": False},
        # a banded operator, 33 entries a row
        {"name": "banded-131072", "kind": "banded", "n": 131072, "bandwidth": 33, "f32": True},
        # a graph whose square fits the card, with the default configuration
        {"name": "rmat-2^18", "kind": "rmat", "log_n": 18, "degree": 16.0, "f32": False},
        # a panel of bench.py's R-MAT 2^20, from the middle of its products
        {"name": "panel-2^20", "kind": "panel", "log_n": 20, "degree": 16.0, "at": 0.37, "products": 2.5e9, "f32": False},
        # the same sparsity again with new values, as an iteration over a fixed mesh or graph has it
        {"name": "replay-2^16", "kind": "replay", "log_n": 16, "degree": 12.0, "f32": False},
        # 128 mixed products at once: predicted capacities, and the captured whole path
        {"name": "batch-learned-128", "kind": "batch", "count": 128, "how": "learned"},
        {"name": "batch-graph-128", "kind": "batch", "count": 128, "how": "graph"},
        # the predictor's training, at its own batch size
        {"name": "train-2^18", "kind": "train", "rows": 1 << 18, "batch": 8192},
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _edges_products(log_n, degree):
    """About the products of an R-MAT square (duplicates merge, so fewer come out)."""
    return (degree * 2.0 ** log_n) ** 2 * 0.6352 ** log_n


def draw(rng):
    kind = rng.choice(["laplacian", "rect", "er", "banded", "rmat", "rmat", "panel", "replay", "batch", "train"])
    f32 = rng.random() < 0.5
    if kind == "laplacian":
        return {"kind": kind, "nx": int(_log(rng, 40, 700)), "ny": int(_log(rng, 40, 700)), "f32": f32}
    if kind == "rect":
        rows = int(_log(rng, 4000, 1 << 18))
        return {"kind": kind, "rows": rows, "cols": int(rows * rng.uniform(2.0, 8.0)), "mean": round(rng.uniform(3.0, 9.0), 2), "f32": f32}
    if kind == "er":
        return {"kind": kind, "n": int(_log(rng, 500, 150000)), "degree": float(rng.randint(2, 32)), "f32": f32}
    if kind == "banded":
        return {"kind": kind, "n": int(_log(rng, 500, 150000)), "bandwidth": 2 * rng.randint(1, 32) + 1, "f32": f32}
    if kind in ("rmat", "replay"):
        log_n = rng.randint(9, 18 if kind == "rmat" else 16)
        most = math.sqrt(_edges_products(18, 16.0) / _edges_products(log_n, 1.0))
        return {"kind": kind, "log_n": log_n, "degree": round(_log(rng, 4.0, min(most, 40.0)), 2), "f32": f32}
    if kind == "panel":
        return {"kind": kind, "log_n": rng.randint(18, 20), "degree": round(rng.uniform(8.0, 16.0), 2), "at": round(rng.uniform(0.0, 0.9), 3),
                "products": float(int(_log(rng, 1e8, 2.4e9))), "f32": f32}
    if kind == "batch":
        return {"kind": kind, "count": int(_log(rng, 8, 127)), "how": rng.choice(["learned", "graph"])}
    return {"kind": "train", "rows": int(_log(rng, 20000, 250000)), "batch": rng.choice([4096, 8192, 8192, 16384])}


# ------------------------------------------------------------------ inputs
class Matrix:
    """A CSR matrix on the GPU: torch tensors, and the library's view of them."""

    def __init__(self, rows, cols, offsets, col_ids, values):
        self.rows, self.cols, self.offsets, self.col_ids, self.values = rows, cols, offsets, col_ids, values
        self.first = int(offsets[0])
        self.nnz = int(offsets[-1]) - self.first
        d = ra.DeviceCSR()
        d.m.rows, d.m.cols, d.m.nnz = rows, cols, self.nnz
        d.m.vtype, d.m.off_bytes = (ocean.OC_F32 if values.dtype == torch.float32 else ocean.OC_F64), 4
        d.m.row_offsets, d.m.col_ids, d.m.values = offsets.data_ptr(), col_ids.data_ptr(), values.data_ptr()
        d.m.on_device, d.m.owned = 1, 0  # the tensors keep the memory
        self.dev = d

    @classmethod
    def of(cls, M):
        up = [torch.from_numpy(a).to(DEVICE) for a in (M.row_offsets.astype(np.uint32).view(np.int32), M.col_ids.view(np.int32), M.values)]
        return cls(M.rows, M.cols, *up)

    def lengths(self):
        return self.offsets.long().diff()

    def row_products(self, B):
        """Products of each row of self * B."""
        e = B.lengths()[self.col_ids[self.first:self.first + self.nnz].long()]
        cs = torch.cat([e.new_zeros(1), e.cumsum(0)])
        o = self.offsets.long() - self.first
        return cs[o[1:]] - cs[o[:-1]]


def _csr(rows, cols, row, col, values):
    """The entries (row, col, value) as a matrix with sorted rows."""
    key, order = ((row << 32) + col).sort()
    counts = torch.bincount(key >> 32, minlength=rows)
    offsets = torch.cat([counts.new_zeros(1), counts.cumsum(0)]).int()
    return Matrix(rows, cols, offsets, (key & 0xFFFFFFFF).int(), values[order])


def _values(n, f32, g):
    return torch.rand(n, generator=g, device=DEVICE, dtype=torch.float32 if f32 else torch.float64) * 2 - 1


# A case's sparsity has one size of C, whatever the seed: the seed renumbers the rows and columns
# in a way that keeps the matrix's character, and gives the values.
def _rmat(log_n, degree, f32, seed, bits=32):
    """R-MAT by the quadrants' probabilities, duplicates merged, values U[-1, 1). The seed flips
    bits of the vertices' numbers, which exchanges quadrants (the lowest `bits` of them only)."""
    g = torch.Generator(DEVICE).manual_seed(log_n)
    a, b, c = ABC
    n, edges = 1 << log_n, int(degree * 2 ** log_n)
    key = torch.zeros(edges, dtype=torch.int64, device=DEVICE)
    for _ in range(log_n):
        u = torch.rand(edges, generator=g, device=DEVICE)
        key = key * 2 + ((u >= a + b).long() << 32) + (((u >= a) & (u < a + b)) | (u >= a + b + c)).long()
    key = torch.unique(key)
    g.manual_seed(seed)
    flip = int(torch.randint(n, (1,), generator=g, device=DEVICE)) & ((1 << bits) - 1)
    return _csr(n, n, (key >> 32) ^ flip, (key & 0xFFFFFFFF) ^ flip, _values(key.numel(), f32, g))


def _moved(h, seed, row_reach, col_reach, normal=False):
    """A host matrix renumbered: each row moves by up to about row_reach places, each column by up
    to col_reach (a square matrix's rows and columns alike), with new values."""
    g = torch.Generator(DEVICE).manual_seed(seed)

    def numbers(n, reach):
        at = torch.arange(n, device=DEVICE) + torch.rand(n, generator=g, device=DEVICE, dtype=torch.float64) * reach
        return at.argsort().argsort()

    p = numbers(h.rows, row_reach)
    q = p if h.rows == h.cols else numbers(h.cols, col_reach)
    M = Matrix.of(h)
    row = torch.repeat_interleave(p, M.lengths())
    f32 = M.values.dtype == torch.float32
    v = torch.randn(M.nnz, generator=g, device=DEVICE, dtype=M.values.dtype) if normal else _values(M.nnz, f32, g)
    return _csr(h.rows, h.cols, row, q[M.col_ids.long()], v)


def _transposed(M):
    row = torch.repeat_interleave(torch.arange(M.rows, device=DEVICE), M.lengths())
    return _csr(M.cols, M.rows, M.col_ids.long(), row, M.values)


def _operands(case, seed):
    """(A, B) of a product; B is A where C = A*A."""
    kind = case["kind"]
    vt = ocean.OC_F32 if case["f32"] else ocean.OC_F64
    if kind in ("rmat", "replay"):
        A = _rmat(case["log_n"], case["degree"], case["f32"], seed)
    elif kind == "laplacian":
        A = Matrix.of(ra.CSR.laplacian2d(case["nx"], case["ny"], vtype=vt, seed=seed))
    elif kind == "banded":
        A = Matrix.of(ra.CSR.banded(case["n"], case["bandwidth"], vtype=vt, seed=seed))
    elif kind == "er":
        A = _moved(ra.CSR.erdos_renyi(case["n"], case["degree"], vtype=vt), seed, case["n"], case["n"])
    elif kind == "rect":
        stride = max(1, case["cols"] // case["rows"])
        h = ra.CSR.rect_band(case["rows"], case["cols"], case["mean"], 0.3, 4096, stride, vtype=vt, value_dist=1)
        A = _moved(h, seed, 64, 64 * stride, normal=True)
        return A, _transposed(A)
    else:
        # the rows from the share `at` of all products on, as many as make `products`, in whole
        # blocks of 1024, inside which the seed renumbers
        M = _rmat(case["log_n"], case["degree"], case["f32"], seed, 10)
        cum = M.row_products(M).cumsum(0)[1023::1024]
        first = case["at"] * float(cum[-1])
        r0, r1 = (1024 * int(x) for x in torch.searchsorted(cum.double(), torch.tensor([first, first + case["products"]], device=DEVICE, dtype=torch.float64)))
        r1 = max(r1, r0 + 1024)
        return Matrix(r1 - r0, M.cols, M.offsets[r0:r1 + 1], M.col_ids, M.values), M
    return A, A


@functools.lru_cache(1)
def _batch_patterns(count):
    return batched_products(ra, count)


def _batch(count, seed):
    """The mixed products, in an order of the seed's and with its values."""
    g = torch.Generator(DEVICE).manual_seed(seed)
    mats = _batch_patterns(count)
    out = []
    for i in torch.randperm(count, generator=g, device=DEVICE).tolist():
        M = Matrix.of(mats[i])
        M.values.copy_(_values(M.nnz, True, g))
        out.append(M)
    return out


class Array:
    """Device memory of the library as a tensor; `owner` lives as long as the tensor does."""

    def __init__(self, ptr, count, kind, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (count,), "typestr": kind, "data": (ptr if count else 0, False), "version": 2, "strides": None}


def _tensors(C):
    """C's row offsets, column ids and values, without a copy."""
    m = C.m
    return tuple(torch.as_tensor(Array(p, n, k, C), device=DEVICE) for p, n, k in
                 ((m.row_offsets, m.rows + 1, "<i8"), (m.col_ids, m.nnz, "<i4"), (m.values, m.nnz, "<f4" if m.vtype == ocean.OC_F32 else "<f8")))


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        mats = _batch(case["count"], seed)
        b = ra.Batch(ra.Config(numeric_expansion_coe=2.0))  # the autotuner's choice for batches
        b.set_inputs([M.dev for M in mats])
        s = {"kind": kind, "how": case["how"], "batch": b, "mats": mats}
        if case["how"] == "learned":
            s["model"] = ra.Mlp(0)
            s["model"].load(predictor.DEFAULT_MODEL)
            ocean._check(ocean.lib.oc_spgemm_set_model(ocean.lib.oc_batch_handle(b.h), s["model"].h, 0.99))
        else:
            b.plan()
            b.capture_full()
        return s
    if kind == "train":
        X, y = [], []
        n = case["rows"] // 3 + 1
        for M in (_rmat(max(10, round(math.log2(n))), 8.0, True, seed), Matrix.of(ra.CSR.erdos_renyi(n, 12.0, vtype=1, seed=seed)),
                  Matrix.of(ra.CSR.banded(n, 17, vtype=1, seed=seed))):
            X.append(ra.Mlp.features(M.dev, M.dev).to_array(np.float32, M.rows * ocean.MLP_FEATURES).reshape(M.rows, -1))
            y.append(ra.Mlp.labels(predictor.exact_counts(M.dev, M.dev), M.rows).to_array(np.uint8, M.rows))
        X, y = np.concatenate(X), np.concatenate(y)
        at = np.random.default_rng(seed).choice(len(y), case["rows"], replace=len(y) < case["rows"])
        return {"kind": kind, "mlp": ra.Mlp(seed), "x": ra.DeviceBuffer.from_array(X[at]), "y": ra.DeviceBuffer.from_array(y[at]),
                "rows": case["rows"], "batch": case["batch"]}
    A, B = _operands(case, seed)
    # bench.py runs its R-MAT 2^20 with the autotuner's symbolic expansion
    sp = ra.SpGEMM(ra.Config(symbolic_expansion_coe=3.0) if kind == "panel" else ra.Config())
    s = {"kind": kind, "A": A, "B": B, "sp": sp}
    if kind == "replay":
        s["C"] = sp.plan(A.dev, B.dev)
        sp.capture()
    return s


def run(state):
    kind = state["kind"]
    if kind == "batch":
        b = state["batch"]
        if state["how"] == "learned":
            b.run()
        else:
            b.launch_full()
        return _tensors(b.result()[0])
    if kind == "train":
        losses = state["mlp"].train(state["x"], state["y"], state["rows"], state["batch"], 1, 2e-3)
        return {"losses": losses, "weights": state["mlp"].params()}
    if kind == "replay":
        state["sp"].graph_launch()
        return _tensors(state["C"])
    return _tensors(state["sp"].run(state["A"].dev, state["B"].dev))


def work(case):
    """A and B read once, C written once; a multiplication and an addition for each product. C's
    size is that of one set of inputs."""
    if case["kind"] == "train":
        # features and labels in, weights and moments in and out; two products for the forward pass
        # over the 5768 weights, four for the backward
        return {"bytes": case["rows"] * (4 * ocean.MLP_FEATURES + 1) + 6 * 4 * ocean.MLP_NPARAM, "flops": 6.0 * case["rows"] * ocean.MLP_NPARAM}
    s = prepare(case, 1)
    pairs = [(M, M) for M in s["mats"]] if case["kind"] == "batch" else [(s["A"], s["B"])]
    products, read = 0, 0
    for A, B in pairs:
        products += int(A.row_products(B).sum())
        for M in {id(A): A, id(B): B}.values():
            read += 4 * (M.rows + 1) + (4 + M.values.element_size()) * M.nnz
    return {"bytes": read + sum(t.numel() * t.element_size() for t in run(s)), "flops": 2.0 * products}


# ------------------------------------------------------------------- exact
def _square_values(A, B, limit=1 << 26):
    """C's values in row and column order, in 64 bits: every product with its key, sorted and summed."""
    lens, starts = B.lengths(), B.offsets.long()
    cum = A.row_products(B).cumsum(0)
    o = A.offsets.long()
    got, r0, done = [], 0, 0
    while r0 < A.rows:
        r1 = int(torch.searchsorted(cum, done + limit, right=True))
        r1 = min(A.rows, max(r1, r0 + 1))
        e0, e1 = int(o[r0]), int(o[r1])
        k = A.col_ids[e0:e1].long()
        row = torch.repeat_interleave(torch.arange(r1 - r0, device=DEVICE), o[r0 + 1:r1 + 1] - o[r0:r1])
        n = lens[k]
        ends = n.cumsum(0)
        of = torch.repeat_interleave(torch.arange(e1 - e0, device=DEVICE), n)
        at = torch.arange(of.numel(), device=DEVICE) - (ends - n)[of] + starts[k][of]
        key, order = (row[of] * B.cols + B.col_ids[at].long()).sort()
        prod = (A.values[e0:e1].double()[of] * B.values[at].double())[order]
        _, inverse = torch.unique_consecutive(key, return_inverse=True)
        total = int(inverse[-1]) + 1 if inverse.numel() else 0
        got.append(torch.zeros(total, dtype=torch.float64, device=DEVICE).index_add_(0, inverse, prod))
        done, r0 = int(cum[r1 - 1]), r1
    return torch.cat(got) if got else torch.zeros(0, dtype=torch.float64, device=DEVICE)


def exact(case, seed):
    if case["kind"] == "train":
        return None
    if case["kind"] == "batch":
        return None, None, torch.cat([_square_values(M, M) for M in _batch(case["count"], seed)])
    return None, None, _square_values(*_operands(case, seed))
