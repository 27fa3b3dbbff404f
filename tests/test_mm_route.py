"""The host rule that sends a MUL_MAT of several rows to the matvec or to the few-row kernels (csrc/mm_route.hpp), on
the CPU at measured shapes. No GPU calls."""


def test_few_rows_route(native):
    assert "calls" in native("few_rows_route_check")
