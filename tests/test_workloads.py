"""The bytes that the BGK workload reports its bandwidth with."""
from frhip.workloads import bgk_call_bytes


def test_bgk_bytes_count_the_moments_pass_where_it_runs():
    large = 128 * 128 * 9 * 576  # 679 MB: the moments once per call, 64 B per value and step
    assert bgk_call_bytes(large, 3) == large * (3 * 64 + 8)
    small = 20 * 33 * 9 * 176  # 8 MB: moments in every stage, 29.3 B per value and stage
    assert bgk_call_bytes(small, 3) == small * 9 * (8 + 64 / 3)
