"""The benchmark's bytes as the kernels load them: the model per row, and the
committed traffic summaries of the kernel that reads row patterns."""
import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)

import bench  # noqa: E402


def test_loaded_bytes_per_row():
    # 27 values, one byte for the columns, x and y
    assert bench.spmv_loaded_bytes(1) == 27 * 8 + 1 + 16 == 233
    assert bench.spmv_loaded_bytes(1, vb=2) == 27 * 2 + 1 + 16 == 71


def test_committed_traffic_of_the_pattern_kernel():
    for n in (320, 512):
        t = bench.loaded_traffic((n, n, n))
        assert t is not None and 1.0 <= t / bench.spmv_loaded_bytes(n ** 3) <= 1.15, (n, t)
        assert t < bench.profiled_traffic((n, n, n))
    assert bench.loaded_traffic((48, 40, 32)) is None


@pytest.mark.gpu
@pytest.mark.parametrize("mode", [0, 1])
def test_batch_bytes(hip, mode):
    """A batch of one moves what its problem does alone, and 8 B a row more: its x
    update is not deferred."""
    B = hip.Batch([(32, 24, 16)], stores=hip.STORE_F64 if mode == 0 else hip.STORE_MIXED)
    P = B.problems[0]
    fast = B.stream_bytes(mode)
    assert fast == pytest.approx(P.stream_bytes(mode)[1] + 8 * P.m, rel=1e-12)
    assert fast < B.profile(iters=1, mode=mode)["iteration"][1]
    P.set_row_patterns(False)
    assert fast < B.stream_bytes(mode) == pytest.approx(P.stream_bytes(mode)[1] + 8 * P.m, rel=1e-12)
    B.close()
