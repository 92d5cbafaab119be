"""How large a graph the allocation-free entry point takes: what its scratch
array holds beside 1,024 wavefronts' regions (256 compute units) must not
grow."""
import numpy as np
import pytest

from rdmce_amd import _lib
from test_zz_no_alloc import HIST, Hip, lib

pytestmark = pytest.mark.gpu

# Counters 256 B, sizes 512 B, two u64 arrays of n + 1, one root, 1,024 deferred
# roots, per wavefront a 128-byte record, a user count and a work bit, and the
# 8 KB that idle counts once took: 4,096 B for each of a wavefront's two
# regions remain up to this many vertices.
LARGEST = 3_660_447


def test_largest_graph_still_fits():
    print("[gpu-case] noalloc largest graph", flush=True)
    hip = Hip()
    try:
        p = hip.put(np.zeros(16, dtype=np.uint64))  # (never read: there is no edge)
        out = hip.put(np.full(4 + HIST, 7, dtype=np.uint64))
        L = lib()
        assert L.mce_solve_device_csr_noalloc(0, LARGEST, 0, p, p, p, HIST, None, out) == _lib.MCE_OK
        assert not hip.get(out, 4 + HIST, np.uint64).any()
        assert L.mce_solve_device_csr_noalloc(0, LARGEST + 4096, 0, p, p, p, HIST, None, out) == _lib.MCE_ERR_UNSUPPORTED
    finally:
        hip.free()
