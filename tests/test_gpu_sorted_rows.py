"""Numeric hash rows sorted by column without a table (num_sort_row) at the
edges of what it takes: 63 to 65 A entries, as many products as a lane keeps
(5 for each thread) and as the LDS of each table size holds, an eighth more
products than outputs, duplicates, empty B rows at the ends and in between, and
buckets one below, at and one above
the crowding limit.  The structure is bit-exact; each value is a sum of at
most 3 products, within 1e-12 (f64) and 1e-5 (f32) of the oracle's,
condition-normalised."""
import numpy as np
import pytest

from helpers import check_product, log

pytestmark = pytest.mark.gpu

COLS = 1 << 24


def _lengths(rng, entries, products):
    """B row lengths of one A row: about a quarter empty, the ends among them."""
    w = rng.random(entries) * (rng.random(entries) > 0.25)
    if entries > 2:
        w[0] = w[-1] = 0.0
    w[entries // 2] = 1.0
    n = np.floor(products * w / w.sum()).astype(np.int64)
    n[entries // 2] += products - n.sum()
    return n


def _deal(pool, lengths):
    """B rows of those lengths, from the pool again and again."""
    at, out = 0, []
    for n in lengths:
        out.append(np.sort(pool[(at + np.arange(n)) % len(pool)]))
        at += n
    return out


def _check(gpu, rows, vtype, name):
    """rows: the B rows of each A row, which belong to it alone."""
    rng = np.random.default_rng(len(rows))
    dt = np.float32 if vtype else np.float64
    b = [c for row in rows for c in row]
    bro = np.r_[0, np.cumsum([len(c) for c in b])].astype(np.uint32)
    aro = np.r_[0, np.cumsum([len(row) for row in rows])].astype(np.uint32)
    B = gpu.CSR(len(b), COLS, bro, np.concatenate(b).astype(np.uint32),
                rng.uniform(-1, 1, int(bro[-1])).astype(dt))
    A = gpu.CSR(len(rows), len(b), aro, np.arange(len(b), dtype=np.uint32),
                rng.uniform(-1, 1, len(b)).astype(dt))
    dA, dB = A.upload(), B.upload()
    for workflow in (0, 1):
        log(f"case: sorted rows {name} vtype {vtype} workflow {workflow}")
        sp = gpu.SpGEMM(gpu.Config(use_ultrasparse_workflow=0))
        sp.set_workflow(workflow)
        check_product(A, B, sp.run(dA, dB).download(), 1e-5 if vtype else 1e-12, name)


def _edges():
    """Products around each table's limits: its LDS after the counters, 12
    bytes a product, and 5 products for each of its threads."""
    out = [1, 2, 63, 64, 65]
    for slots, threads in ((200, 64), (488, 128), (1064, 256), (2216, 512)):
        most = 2 * slots // 3 + 1
        lds = -(-(1280 + 4 * slots + 8) // 8) * 8 + 8 * slots + 6 * most
        lds = -(-lds // 8) * 8 + threads // 64 * 512
        fit = (lds - (1280 + 16 * threads + 16)) // 12
        out += [fit - 1, fit, fit + 1, 5 * threads - 1, 5 * threads, 5 * threads + 1]
    return out


@pytest.mark.parametrize("vtype", [0, 1])
@pytest.mark.parametrize("entries", [1, 2, 63, 64, 65])
def test_limits(gpu, entries, vtype):
    rng = np.random.default_rng(entries)
    rows = []
    for p in _edges():
        # outputs: another table size, and about an eighth less than products
        eighth = -(-8 * p // 9)
        for outputs in {p, eighth - 1, eighth, eighth + 1, int(0.57 * p), p // 2}:
            outputs = min(p, max(1, outputs))
            lengths = _lengths(rng, entries, p)
            pool = rng.choice(COLS, max(outputs, int(lengths.max())), replace=False)
            rows.append(_deal(pool, lengths))
    _check(gpu, rows, vtype, f"limits, {entries} entries")


@pytest.mark.parametrize("vtype", [0, 1])
def test_crowding(gpu, vtype):
    """23, 24 and 25 products of one bucket: in columns of their own, all in
    one column, and in a few; the others spread."""
    rng = np.random.default_rng(5)
    rows = []
    for p in (60, 200, 500, 1200, 2500):
        for crowd in (23, 24, 25):
            for apart in (crowd, 1, 4):
                spread = rng.choice(COLS // 2, p - crowd, replace=False)
                near = COLS - 5000 + np.arange(crowd) % apart
                cols = np.r_[spread, near]
                rng.shuffle(cols)
                # each near column at most once in a B row
                b = [[] for _ in range(60)]
                for i, c in enumerate(cols):
                    b[i % 60].append(c)
                b = [np.sort(np.array(x, np.int64)) for x in b]
                if all(len(np.unique(x)) == len(x) for x in b):
                    rows.append(b)
                else:
                    b = [np.sort(x) for x in np.array_split(spread, 30)] + [np.array([c]) for c in near]
                    rows.append(b)
    _check(gpu, rows, vtype, "crowding")
