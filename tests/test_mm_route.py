"""csrc/mm_route.hpp on the CPU: the rule that sends a MUL_MAT of several rows to the matvec or to the few-row kernels,
at measured shapes, and the Q4_K prefill kernel's split of a row over its waves. No GPU calls."""


def test_few_rows_route(native):
    assert "calls" in native("few_rows_route_check")


def test_q4k_prefill_split(native):
    assert "row lengths" in native("mm_split_check")
