"""The host planner of FLASH_ATTN_EXT (csrc/fa_plan.hpp) on the CPU: the work lists and tile maps of the
matrix-core score route, for every number of KV heads. No GPU calls."""


def test_score_route_tile_map(native):
    """1 .. 64 KV heads: the cap on the chunk length (4 floor(9344 / (16 n_head_kv)) groups) is no multiple of a
    tile for most counts from 19 on; such rows of several chunks stay on the one-row score kernel."""
    assert "on the matrix cores" in native("fa_plan_check")
