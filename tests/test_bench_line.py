"""Figures of the bench line that are formed from the timers."""
import bench


def test_rhs_rate_counts_the_shell_launches():
    """the shell's points are among the updates, so its launches are part of the time"""
    one = bench.fmr_rhs_fp64({"z4_rhs": 250.0, "z4_rhs_edge": 0.0}, 1000)
    two = bench.fmr_rhs_fp64({"z4_rhs": 200.0, "z4_rhs_edge": 50.0}, 1000)
    assert one == two
    assert one["rhs_ms_per_coarse_step"] == 250.0
    assert abs(one["achieved"] * 1e12 * 0.25 - bench.FLOP_PER_POINT_RHS * 4000) <= 1e-9 * one["flop_per_coarse_step"]
    assert bench.fmr_rhs_fp64({"z4_rhs": 0.0, "z4_rhs_edge": 0.0}, 1000) is None
