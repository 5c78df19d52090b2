"""Order of the numeric hash rows: keys grouped by column bucket, with the
radix sort for rows whose columns crowd into few buckets.  Rows at the edges
of every table size, with columns spread, crowded at both ends of a wide
span, crowded just below and above the crowding limit, and skewed."""
import numpy as np
import pytest

from helpers import check_product, log

pytestmark = pytest.mark.gpu

COLS = 1 << 24
# outputs of a row around each table's capacity with the numeric expansion
# of 1.5 (tables of 200, 488, 1064, 2216, 4776 and 9640 slots)
SIZES = [1, 2, 63, 133, 134, 325, 326, 709, 710, 1477, 1478, 3184, 3185, 6426]


def _columns(rng, n, kind):
    if kind == "spread":
        c = rng.choice(COLS, n, replace=False)
    elif kind == "ends":  # both ends of the span, nothing between
        c = np.r_[np.arange(n // 2), COLS - 1 - np.arange(n - n // 2)]
    elif kind.startswith("crowd"):  # that many in one place, the rest spread
        k = min(n, int(kind[5:]))
        c = np.r_[np.arange(k) + 5_000_000, 6_000_000 + rng.choice(COLS - 6_000_000, n - k, replace=False)]
    else:  # skewed towards 0, as an R-MAT row
        c = np.array([], np.int64)
        while len(c) < n:
            c = np.unique(np.r_[c, (COLS * rng.random(2 * n) ** 6).astype(np.int64)])
        c = rng.choice(c, n, replace=False)
    return np.sort(c)


def _csr(gpu, rows, cols, lists, rng, vtype):
    ro = np.r_[0, np.cumsum([len(x) for x in lists])].astype(np.uint32)
    ci = np.concatenate(lists).astype(np.uint32)
    return gpu.CSR(rows, cols, ro, ci, rng.uniform(-1, 1, len(ci)).astype(np.float32 if vtype else np.float64))


@pytest.mark.parametrize("kind", ["spread", "ends", "crowd191", "crowd193", "skewed"])
@pytest.mark.parametrize("vtype", [0, 1])
def test_row_order(gpu, kind, vtype):
    rng = np.random.default_rng(len(kind) + vtype)
    blists, alists = [], []
    for n in SIZES:
        c = _columns(rng, n, kind)
        k = len(blists)
        blists += [c, c[::2], c[n // 3:]]  # one row with them all, two with some
        alists += [np.array([k, k + 1, k + 2])] * 3
    A = _csr(gpu, len(alists), len(blists), alists, rng, vtype)
    B = _csr(gpu, len(blists), COLS, blists, rng, vtype)
    dA, dB = A.upload(), B.upload()
    for workflow in (0, 1):
        log(f"case: hash row order {kind} vtype {vtype} workflow {workflow}")
        sp = gpu.SpGEMM(gpu.Config(use_ultrasparse_workflow=0))
        sp.set_workflow(workflow)
        check_product(A, B, sp.run(dA, dB).download(), 1e-5 if vtype else 1e-12, kind)
