"""GPU parity of the tile-start table through the one-gather rank tiles
(the role of denseNumericIterKernel's column windows,
kernels/AccumulatorDense.cuh:610-806): tables of one tile (the row's two ends
and nothing between), of 64, 65 and 66 starts a row, row counts that leave a
part of the last workgroup, empty B rows, rows with entries in the first and
the last column, and blocks of a batch, whose tiles are counted from the
block's first column.  The structure is bit-exact and the FP64 values are
within 1e-12 of the oracle's, condition-normalised."""
import numpy as np
import pytest

from helpers import check_product, log

pytestmark = pytest.mark.gpu


def _operands(gpu, rows, cols, seed):
    """B with short rows and one of 9000 entries; a first row of A that takes
    every B row, whose outputs fit no hash table and whose span no dense one."""
    rng = np.random.default_rng(seed)
    blen = rng.integers(0, 60, rows)
    blen[::7] = 0
    blen[1] = min(cols, 9000)
    bcols = [np.sort(rng.choice(cols, int(L), replace=False)) for L in blen]
    bcols[2] = np.array([0, cols - 1])
    bcols[rows - 1] = np.array([0, cols - 1])
    brp = np.zeros(rows + 1, np.uint32)
    np.cumsum([len(c) for c in bcols], out=brp[1:])
    B = gpu.CSR(rows, cols, brp, np.concatenate(bcols).astype(np.uint32),
                rng.uniform(-1, 1, int(brp[-1])))
    acols = [np.arange(rows), np.arange(1, rows, 2), np.array([2, rows - 1])]
    arp = np.zeros(len(acols) + 1, np.uint32)
    np.cumsum([len(c) for c in acols], out=arp[1:])
    A = gpu.CSR(len(acols), rows, arp, np.concatenate(acols).astype(np.uint32),
                rng.uniform(-1, 1, int(arp[-1])))
    return A, B


def _long_rows(stats):
    """Rows of the bin whose numeric kernels read the table."""
    return int(np.diff(np.array(stats["binning_2"]))[13])


@pytest.mark.parametrize("cols,log_tile", [(1 << 15, 16), (1 << 16, 16), ((1 << 16) - (1 << 10), 10),
                                           ((1 << 16) - 1, 10), ((1 << 16) + 1, 10)])
@pytest.mark.parametrize("rows", [1023, 2049])
def test_tile_starts(gpu, rows, cols, log_tile):
    log(f"case: tile starts, B {rows} x {cols}, tiles 2^{log_tile}")
    A, B = _operands(gpu, rows, cols, rows + cols)
    sp = gpu.SpGEMM(gpu.Config(use_tiled_numeric=3, tile_log2_cols=log_tile))
    sp.set_workflow(0)
    C = sp.run(A.upload(), B.upload()).download()
    assert _long_rows(sp.get_stats()) >= 1
    check_product(A, B, C, 1e-12, f"tile starts {rows} x {cols}")


@pytest.mark.parametrize("log_tile", [10, 16])
def test_tile_starts_of_blocks(gpu, log_tile):
    """Blocks of unequal width: every base but the first is not zero, and the
    narrower blocks leave the table's last tiles empty."""
    log(f"case: tile starts of blocks, tiles 2^{log_tile}")
    pairs = [_operands(gpu, rows, cols, cols) for rows, cols in
             ((1023, 30_001), (300, 500), (2049, 64_512), (1025, 40_000))]
    up = [(A.upload(), B.upload()) for A, B in pairs]
    b = gpu.Batch(gpu.Config(use_tiled_numeric=3, tile_log2_cols=log_tile))
    b.set_inputs([a for a, _ in up], [c for _, c in up])
    b.run()
    assert _long_rows(b.get_stats()) >= 3
    for i, (A, B) in enumerate(pairs):
        check_product(A, B, b.extract(i).download(), 1e-12, f"block {i}")
