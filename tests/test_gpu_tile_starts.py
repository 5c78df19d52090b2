"""GPU parity of the tile-start table through the one-gather rank tiles
(the role of denseNumericIterKernel's column windows,
kernels/AccumulatorDense.cuh:610-806): tables of one tile, of 64, 65 and
66 starts a row, row counts that leave a part of the last workgroup, empty
B rows and rows with entries in the first and the last column.  The structure
is bit-exact and the FP64 values are within 1e-12 of the oracle's,
condition-normalised."""
import numpy as np
import pytest

from helpers import check_product, log

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cols", [1 << 10, (1 << 16) - (1 << 10), (1 << 16) - 1, (1 << 16) + 1])
@pytest.mark.parametrize("rows", [1023, 2049])
def test_tile_starts(gpu, rows, cols):
    log(f"case: tile starts, B {rows} x {cols}, tiles 2^10")
    rng = np.random.default_rng(rows + cols)
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
    sp = gpu.SpGEMM(gpu.Config(use_tiled_numeric=3, tile_log2_cols=10))
    sp.set_workflow(0)
    C = sp.run(A.upload(), B.upload()).download()
    check_product(A, B, C, 1e-12, f"tile starts {rows} x {cols}")
