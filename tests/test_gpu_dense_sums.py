"""The numeric dense rows tell set columns from their sums (-0.0 is "no
product"): values whose products or sums are zeros of either sign, underflow,
denormals, infinities and NaN have to keep their column, at spans around the
64-column chunks and in every workgroup size."""
import numpy as np
import pytest

from helpers import log
from oracle import oracle as ora

pytestmark = pytest.mark.gpu

SPECIAL = [0.0, -0.0, 1.0, -1.0, 1e-160, -1e-160, 5e-324, -5e-324, 1e300, -1e300]


def _operands(gpu, rows, inner, span, first, vtype, values):
    """A: rows x inner, full; B: inner x (first + span), every column of
    [first, first + span) in some B row and the outermost two in all."""
    rng = np.random.default_rng(span)
    bro, bci = [0], []
    for k in range(inner):
        cols = np.unique(np.r_[0, span - 1, np.arange(k, span, inner)]) + first
        bci.append(cols)
        bro.append(bro[-1] + len(cols))
    bci = np.concatenate(bci).astype(np.uint32)
    dt = np.float32 if vtype else np.float64
    A = gpu.CSR(rows, inner, (np.arange(rows + 1) * inner).astype(np.uint32),
                np.tile(np.arange(inner), rows).astype(np.uint32),
                rng.choice(values, rows * inner).astype(dt))
    B = gpu.CSR(inner, first + span, np.array(bro, np.uint32), bci,
                rng.choice(values, len(bci)).astype(dt))
    return A, B


# spans around a chunk, around each bin's widest (480, 1120, 2368, 4896, 9952)
@pytest.mark.parametrize("span", [33, 63, 64, 65, 127, 449, 480, 481, 1120, 2337, 4896, 9921])
@pytest.mark.parametrize("vtype", [0, 1])
def test_signed_zeros_and_underflow(gpu, span, vtype):
    log(f"case: dense sums span {span} vtype {vtype}")
    values = [v for v in SPECIAL if not vtype or abs(v) in (0.0, 1.0)] + ([1e-30, -1e-30] if vtype else [])
    A, B = _operands(gpu, 70, 40, span, 31, vtype, values)
    sp = gpu.SpGEMM(gpu.Config(use_ultrasparse_workflow=0))
    for workflow in (0, 1):
        sp.set_workflow(workflow)
        C = sp.run(A.upload(), B.upload()).download()
        # every sum is exact or within 40 roundings of its largest partial
        # sum; denormal sums within 40 of their spacing
        tol = 1e-5 if vtype else 40 * 2.0 ** -53
        rp, cols, vals, cond = ora.numeric(A, B, compensated=1)
        assert np.array_equal(C.row_offsets.astype(np.uint64), rp)
        assert np.array_equal(C.col_ids, cols)
        err = np.abs(C.values.astype(np.float64) - vals)
        fl = np.isfinite(cond)
        assert np.all(err[fl] <= tol * cond[fl] + 40 * 5e-324 + (1e-45 if vtype else 0.0))


def test_infinities_and_nan(gpu):
    log("case: dense sums, infinities and NaN")
    A, B = _operands(gpu, 5, 40, 200, 0, 0, [1.0, -1.0, np.inf, -np.inf, np.nan, 0.0])
    sp = gpu.SpGEMM(gpu.Config(use_ultrasparse_workflow=0))
    sp.set_workflow(0)
    C = sp.run(A.upload(), B.upload()).download()
    D = np.zeros((5, 200))
    a = A.values.reshape(5, 40)
    with np.errstate(invalid="ignore"):
        for k in range(40):
            s = slice(B.row_offsets[k], B.row_offsets[k + 1])
            D[:, B.col_ids[s]] += a[:, k:k + 1] * B.values[s][None, :]
    assert np.array_equal(C.row_offsets, np.arange(6) * 200)
    got = C.values.reshape(5, 200)
    assert np.array_equal(np.isnan(got), np.isnan(D))
    assert np.array_equal(got[np.isinf(D)], D[np.isinf(D)])
