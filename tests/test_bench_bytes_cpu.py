"""The bytes that the benchmark counts for adjoint launches (no GPU)."""
import bench


def test_bytes_of_sweeps_side_by_side():
    S = 16 << 21
    one_by_one = bench.adjoint_bytes_per_launch(passes=2, sweeps=21, launches=42, state_bytes=S)
    together = bench.adjoint_bytes_per_launch(passes=2, sweeps=21, launches=2, state_bytes=S)
    assert one_by_one == 3.5 * S  # 3 states in the first pass of a sweep, 4 in the second
    assert together == 21 * one_by_one
    assert bench.adjoint_bytes_per_launch(passes=1, sweeps=3, launches=1, state_bytes=S) == 9 * S
