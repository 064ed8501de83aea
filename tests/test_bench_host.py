"""bench.py's key of a committed traffic figure: the sweep kernel that a run
launches, with the shape the library was built for."""
import bench


def test_traffic_belongs_to_the_kernel_that_runs():
    columns = bench.sweep_kernel_name(False, 2)
    assert columns.startswith("columnSweepKernel<float> ") and bench.measured_traffic(columns) > 0
    # another shape of it, or a kernel that no summary covers
    assert bench.measured_traffic("columnSweepKernel<float> 1x2x3") is None
    assert bench.measured_traffic(bench.sweep_kernel_name(False, 4)) is None
    names = {bench.sweep_kernel_name(f, s) for f in (False, True) for s in (2, 4, 5)}
    assert len(names) == 6
