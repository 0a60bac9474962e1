"""What bench.py prints beside its times, on the CPU."""
import math

import bench


def test_roofline_of_a_kernel_with_several_launches_per_step():
    """A step may launch a kernel several times (rectangles of a wide head, windows of a long sequence): flops, vector
    instructions and time are those of the step."""
    flops, entries = 4.0e12, 1.0e10
    kernels = {"chunk_bwd_local_kernel": {"avg_ms": 1.0, "launches": 40, "ms_per_step": 4.0}}
    roof = bench.mfma_roofline("c2", "chunk_bwd_local_kernel", kernels, flops, entries, "")
    assert math.isclose(roof["achieved"], flops / 4e-3 / 1e12) and math.isclose(roof["frac"], roof["achieved"] / 2500.0)
    ops = bench.counter("c2", "chunk_bwd_local_kernel", "valu_ops_per_entry")
    assert math.isclose(roof["valu"]["achieved"], ops * entries * 2 / 4e-3 / 1e12)


def test_kernel_times_per_step_come_from_all_launches(monkeypatch):
    from palimpsa_amd import _lib

    class Event:
        def __init__(self, **_):
            pass

        def record(self):
            pass

        def elapsed_time(self, _):
            return 1.0

    torch = type("torch", (), {"cuda": type("cuda", (), {"synchronize": staticmethod(lambda: None), "Event": Event})})
    monkeypatch.setattr(_lib, "profile_enable", lambda on: None)
    monkeypatch.setattr(_lib, "profile_read", lambda: {"k": (80.0, 40)})
    _, _, kernels = bench.timed_loop(torch, lambda: None, 10, 0)
    assert kernels["k"] == {"avg_ms": 2.0, "launches": 40, "ms_per_step": 8.0}
