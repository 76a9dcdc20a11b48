"""The benchmark's roofline takes its durations and traffic from the launch it names: the pairing of a
profiled child's dispatches with the launch names, on synthetic traces. No GPU calls."""
import argparse
import os
import sys

import pytest

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import bench

# a profiled step: its launches' names and kernels (the parameter write of a forward has no name)
STEP = [("step_begin", "void fllm::k_step_begin<false>(int)", 1024), ("qkv_rope_kv", "void fllm::k_gemv_mfma<1>(int)", 256),
        ("ffn_gate_up", "void fllm::k_gemv_mfma<2>(int)", 448), ("argmax", "fllm::k_argmax_keys(int)", 1)]
NAMES = [n for n, _, _ in STEP] * 2
MB = 66.0
US = {"ffn_gate_up": 14}


def _children(extra=(), traffic=MB):
    """rocprof_child over two steps, each with the kernels of `extra` before it."""
    rows = [(None, k, 1) for k in extra]
    order = [(None, "fllm::k_pf_embed(int)", 8)] + 2 * (rows + STEP)

    def child(args, mode, tmp, child="--child-profile"):
        if mode == "trace":
            return [{"Kernel_Name": k, "Grid_Size": str(g), "Start_Timestamp": str(1000000 * i),
                     "End_Timestamp": str(1000000 * i + 1000 * US.get(n, 5))} for i, (n, k, g) in enumerate(order)]
        kib = {"ffn_gate_up": traffic * 1e6 / 1024 if mode == "FETCH_SIZE" else 0.0}
        out = [{"Counter_Name": c, "Dispatch_Id": str(i), "Kernel_Name": k, "Counter_Value": str(kib.get(n, 1.0))}
               for i, (n, k, _) in enumerate(order) for c in mode.split()]
        return out + [{"Counter_Name": c, "Dispatch_Id": "99", "Kernel_Name": "copyBuffer",
                       "Counter_Value": str(bench.COPY_BYTES / 1024.0)} for c in mode.split()]
    return child


def _roofline(monkeypatch, **kw):
    monkeypatch.setattr(bench, "rocprof_child", _children(**kw))
    return bench.profiler_roofline(argparse.Namespace(), MB * 1e6, "ffn_gate_up", NAMES)


@pytest.mark.parametrize("extra", [(), ("fllm::k_set_params(int)",)], ids=["named", "parameters"])
def test_roofline_is_the_named_launch(monkeypatch, extra):
    r = _roofline(monkeypatch, extra=extra)
    assert r["kernel_symbol"] == "void fllm::k_gemv_mfma<2>" and r["avg_launch_us"] == 14.0
    assert r["traffic"] == pytest.approx(MB * 1e6, rel=1e-6)


def test_roofline_refuses_shifted_launches(monkeypatch):
    """A launch without a name before each step shifts every position of the steps before the last."""
    with pytest.raises(RuntimeError, match="ffn_gate_up"):
        _roofline(monkeypatch, extra=("fllm::k_unnamed(int)",))


def test_roofline_refuses_traffic_below_the_weights(monkeypatch):
    with pytest.raises(RuntimeError, match="MB to read"):
        _roofline(monkeypatch, traffic=0.57 * MB)
