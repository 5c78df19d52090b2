"""The scan's two-launch form and the bin scan's chunks at the edges of their
ranges, including arrays that are not 16-byte aligned."""
import numpy as np
import pytest

from helpers import log
from oracle import oracle as ora

pytestmark = pytest.mark.gpu


# one launch to 8192, two to 2^20, three beyond; tiles of 2048, 8 per thread
@pytest.mark.parametrize("n", [8192, 8193, 8200, 10239, 10240, 10241, (1 << 20) - 1, 1 << 20, (1 << 20) + 1])
@pytest.mark.parametrize("shift", [(0, 0), (1, 0), (0, 1)])
def test_scan_edges(gpu, n, shift):
    log(f"case: scan n={n} shifted by {shift}")
    x = np.random.default_rng(n).integers(0, 1 << 32, n, dtype=np.uint64).astype(np.uint32)
    si, so = shift
    dx = gpu.DeviceBuffer.from_array(np.r_[np.zeros(si, np.uint32), x])
    dy = gpu.DeviceBuffer.from_array(np.full(n + 3 + so, 7, np.uint64))
    gpu._check(gpu.lib.oc_scan_u32(dx.ptr + 4 * si, dy.ptr + 8 * so, n, None))
    got = dy.to_array(np.uint64, n + 3 + so)
    want = np.zeros(n + 1, np.uint64)
    np.cumsum(x.astype(np.uint64), out=want[1:])
    assert np.array_equal(got[so:so + n + 1], want)
    assert np.all(got[so + n + 1:] == 7) and np.all(got[:so] == 7)


# blocks of 256 rows, scanned 512 blocks at a time
@pytest.mark.parametrize("rows", [256 * 64, 256 * 511 + 1, 256 * 512, 256 * 512 + 1, 256 * 1024 + 255])
def test_bin_groups(gpu, rows):
    log(f"case: bins of {rows} rows")
    rng = np.random.default_rng(rows)
    t = gpu.tables(0)
    products = (2.0 ** rng.uniform(0, 20, rows)).astype(np.uint32)
    left = rng.integers(0, 1000, rows).astype(np.uint32)
    right = left + (2.0 ** rng.uniform(0, 21, rows)).astype(np.uint32)
    d = [gpu.DeviceBuffer.from_array(a) for a in (products, left, right)]
    bor, brows, boff = gpu.DeviceBuffer(rows), gpu.DeviceBuffer(4 * rows), gpu.DeviceBuffer(64)
    gpu._check(gpu.lib.oc_bin_symbolic(0, rows, d[0].ptr, d[1].ptr, d[2].ptr, 0, 1.25, 0.0,
                                       bor.ptr, brows.ptr, boff.ptr, None))
    want = ora.bin_symbolic(products, left, right, t["hash_sym"], t["dense_sym"],
                            t["max_dense_sym_bin"], 0, 1.25, 0.0)
    assert np.array_equal(bor.to_array(np.uint8, rows), want)
    assert np.array_equal(brows.to_array(np.uint32, rows), np.argsort(want, kind="stable"))
    offs = boff.to_array(np.uint32, 16)
    assert np.array_equal(offs, np.r_[0, np.cumsum(np.bincount(want, minlength=15))])
