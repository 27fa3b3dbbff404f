"""The runtime's host-side objects (csrc/runtime.hpp) on the CPU over a pretended device. No GPU calls."""


def test_pinned_slots_outlive_their_readers(native):
    """A pinned slot is written again, or given back, only after the copy or kernel that reads it has run, also
    when the event behind that reader cannot be recorded."""
    assert "no slot" in native("pinned_slots_check")
