"""What a value-only replay launches: one kernel for each numeric bin that has
rows, and the clearing of a row-claim counter only for bins that claim rows.
Counted as the nodes of a captured replay."""
import ctypes as C

import numpy as np
import pytest

from helpers import check_product, log

pytestmark = pytest.mark.gpu


def _captured_nodes(gpu, hip, sp):
    # the launches alone: the C entry waits for them, which a capture forbids
    replay_async = gpu.lib["_ZN2oc19spgemm_replay_asyncEP9oc_spgemmP12ihipStream_t"]
    replay_async.argtypes, replay_async.restype = [C.c_void_p, C.c_void_p], C.c_int
    stream, graph, n = C.c_void_p(), C.c_void_p(), C.c_size_t(0)
    assert hip.hipStreamCreate(C.byref(stream)) == 0
    assert hip.hipStreamBeginCapture(stream, 2) == 0  # relaxed: this thread allocates nothing
    rc = replay_async(sp.h, stream)
    assert hip.hipStreamEndCapture(stream, C.byref(graph)) == 0
    assert rc == 0
    assert hip.hipGraphGetNodes(graph, None, C.byref(n)) == 0
    assert hip.hipGraphDestroy(graph) == 0 and hip.hipStreamDestroy(stream) == 0
    return n.value


@pytest.mark.parametrize("name", ["er", "rmat12"])
def test_one_launch_a_bin(gpu, name):
    log(f"case: replay nodes {name}")
    hip = C.CDLL("libamdhip64.so")
    A = gpu.CSR.erdos_renyi(3000, 8.0, seed=3) if name == "er" else gpu.CSR.rmat(12, 8 << 12, seed=1)
    sp = gpu.SpGEMM(gpu.Config(use_ultrasparse_workflow=0))
    dA = A.upload()
    dC = sp.plan(dA, dA)
    bins = np.diff(np.array(sp.get_stats()["binning_2"]))
    assert bins[13] == 0  # no long rows
    assert _captured_nodes(gpu, hip, sp) == np.count_nonzero(bins[:13])
    sp.replay()
    check_product(A, A, dC.download(), 1e-12, name)
