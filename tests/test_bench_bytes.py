"""Host logic of bench.py (no GPU): the bytes that kernels sharing rows ask for."""
import bench
from angelo_amd.workloads import WORKLOADS


def test_forward_rows_of_shared_cells():
    spec = WORKLOADS["neuralangelo-fp32"]
    L = 16
    full = bench.algorithmic_bytes("geo_fwd", spec, 1, 0, 0)
    # no offset leaves its cell: two clusters' centres alone
    still = bench.requested_bytes("geo_fwd", spec, 1, 0, 0, offsets=[0.0] * L)
    assert full - still == (13 - 2) * 8 * L * 8
    # every offset crosses a face, or lies beyond the next cell
    assert bench.requested_bytes("geo_fwd", spec, 1, 0, 0, offsets=[1.0] * L) \
        == still + 12 * 4 * L * 8
    assert bench.requested_bytes("geo_fwd", spec, 1, 0, 0, offsets=[1.5] * L) \
        == still + 12 * 8 * L * 8
    # the analytic form gathers in full
    spec = WORKLOADS["neuralangelo-analytic"]
    assert bench.requested_bytes("geo_fwd", spec, 1, 0, 0, offsets=[0.5] * L) \
        == bench.algorithmic_bytes("geo_fwd", spec, 1, 0, 0)


def test_paged_reduction_bytes():
    spec = WORKLOADS["neuralangelo-fp32"]
    assert bench.requested_bytes("seg_reduce", spec, 0, 0, 1000, table_rows=10) == 16080
    assert bench.requested_bytes("seg_reduce", spec, 0, 0, 1000, mixed=True, table_rows=10) == 12080
    assert bench.requested_bytes("march_count", spec, 10, 2, 0) is None
