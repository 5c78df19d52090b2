"""Rows whose products are walked in blocks of 64 (for_products, flat_owner) at
the edges of that walk: A rows of 63 to 129 entries and more chunks than waves,
B rows that are empty in between and at both ends of a chunk, so short that a
block holds many starts, or so long that they are swept apart.  The same
structure in wide spans (hash rows) and narrow ones (dense rows), in both
workflows.  The structure is bit-exact and the values are within 1e-12 (f64)
and 1e-5 (f32) of the oracle's, condition-normalised."""
import numpy as np
import pytest

from helpers import check_product, log

pytestmark = pytest.mark.gpu


def _lengths(rng, entries, kind):
    if kind == "ones":  # 64 starts a block
        return np.ones(entries, np.int64)
    if kind == "dozen":  # 12 or 13 starts in many blocks
        return rng.integers(4, 7, entries)
    if kind == "gaps":  # empty between and at the ends of every chunk
        n = rng.integers(1, 30, entries) * (rng.random(entries) > 0.4)
        n[::64] = 0
        n[63::64] = 0
        n[-1] = 0
        n[entries // 2] = 7
        return n
    if kind == "last":  # only the last entry of a chunk has products
        n = np.zeros(entries, np.int64)
        n[63::64] = 70
        n[-1] = 129
        return n
    # "apart": a few B rows much longer than a chunk's share, the rest short
    n = rng.integers(1, 4, entries)
    n[[0, entries // 2, entries - 1]] = (600, 900, 1400)
    return n


KINDS = ["ones", "dozen", "gaps", "last", "apart"]
ENTRIES = [1, 2, 63, 64, 65, 127, 128, 129, 1023, 1025, 2100]


@pytest.mark.parametrize("cols", [1 << 22, 9000, 1500])
@pytest.mark.parametrize("vtype", [0, 1])
def test_walk(gpu, cols, vtype):
    rng = np.random.default_rng(cols)
    dt = np.float32 if vtype else np.float64
    alen, blen = [], []
    for kind in KINDS:
        for entries in ENTRIES:
            alen.append(entries)
            blen.append(_lengths(rng, entries, kind))
    blen = np.concatenate(blen)
    # strictly ascending columns in every B row
    bcols = [np.sort(rng.choice(cols, n, replace=False)) if n else np.empty(0, np.int64)
             for n in blen]
    bro = np.r_[0, np.cumsum(blen)].astype(np.uint32)
    B = gpu.CSR(len(blen), cols, bro, np.concatenate(bcols).astype(np.uint32),
                rng.uniform(-1, 1, int(bro[-1])).astype(dt))
    aro = np.r_[0, np.cumsum(alen)].astype(np.uint32)
    A = gpu.CSR(len(alen), len(blen), aro, np.arange(len(blen), dtype=np.uint32),
                rng.uniform(-1, 1, len(blen)).astype(dt))
    dA, dB = A.upload(), B.upload()
    for workflow in (0, 1):
        log(f"case: flat walk cols {cols} vtype {vtype} workflow {workflow}")
        sp = gpu.SpGEMM(gpu.Config(use_ultrasparse_workflow=0))
        sp.set_workflow(workflow)
        C = sp.run(dA, dB)
        check_product(A, B, C.download(), 1e-5 if vtype else 1e-12, f"flat walk {cols}")
        if workflow == 0:
            bins = np.diff(np.array(sp.get_stats()["binning_2"]))
            hashed, dense = int(bins[1:7].sum()), int(bins[7:13].sum())
            log(f"hash rows {hashed}, dense rows {dense}")
            assert (hashed if cols > 9952 else dense) > 0
