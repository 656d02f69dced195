"""bench.py under a profiler: the live loop is left out before any GPU call."""
import importlib.util
import os
import sys

import pytest

BENCH = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "bench.py")


def _bench():
    spec = importlib.util.spec_from_file_location("bench_under_test", BENCH)
    module = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(module)
    return module


@pytest.mark.parametrize("environ,steps", [({}, 20), ({"ROCM_PATH": "/opt/rocm", "ROCR_VISIBLE_DEVICES": "0"}, 20),
                                           ({"ROCP_TOOL_LIBRARIES": "tool.so"}, 0), ({"ROCPROF_KERNEL_TRACE": "1"}, 0)])
def test_the_live_loop_is_skipped_under_a_profiler(monkeypatch, environ, steps):
    bench, seen = _bench(), []
    for k in list(os.environ):
        if k.startswith(("ROCP", "ROCM", "ROCR")):
            monkeypatch.delenv(k)
    for k, v in environ.items():
        monkeypatch.setenv(k, v)
    monkeypatch.setattr(sys, "argv", ["bench.py", "--workload", "config2"])
    monkeypatch.setattr(bench, "decode_workload", lambda args: seen.append(args.live_steps) or {})
    bench.main()
    assert seen == [steps]
