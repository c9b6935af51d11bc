"""The roofline's `traffic` of bench.py comes from a counter summary in the tree."""
import bench


def test_traffic_is_measured():
    for which, per_cell in (("f32", 12), ("f64", 24)):
        t = bench.measured_traffic(which)
        # At least the algorithmic bytes of a launch at 256^3, and not some other kernel's.
        assert t is not None and 1.0 <= t / (per_cell * 256 ** 3) < 1.6
