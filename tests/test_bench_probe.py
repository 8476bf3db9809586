"""bench.py --gemm-phase builds an instrumented copy of the state kernel from the
current source: every place it stamps is still there."""
import bench


def test_probe_patches_fit_the_current_source():
    src = bench.probe_source()
    assert src.count('gp_time()') > 6 and 'vgdr_probe_read' in src
