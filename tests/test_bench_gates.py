"""The parity gates of bench.py compare two different ways through a stack, whichever way a batch goes by itself, and the rows it
calls one launch are one launch.  (A recording stands for the library: which calls are made is what is looked at.)"""
from unittest import mock
import numpy as np
import pytest
import bench
from zerocool_amd import workload


def context(single_launch, persistent=True, outputs=None):
    """A recorded context.  A batch goes as a single launch by itself, or layer by layer; outputs: what each way leaves."""
    ctx = mock.MagicMock()
    ctx.stack_single_launch.return_value = single_launch
    ctx.stack_is_persistent.return_value = persistent
    ctx.ways = []

    def decode(stack, x, tokens, out, trace=None, layered=False, single=False):
        ctx.ways.append("layers" if layered or not (single or single_launch) else "launch")

    ctx.stack_decode.side_effect = decode
    ctx.timer_stop.return_value = 1.0
    out = mock.MagicMock()
    out.numpy.side_effect = lambda dtype: np.full(4, (outputs or {}).get(ctx.ways[-1], 0), dtype)
    return ctx, out


@pytest.mark.parametrize("single_launch", [False, True])
def test_a_gate_goes_both_ways(single_launch):
    ctx, out = context(single_launch)
    bench.check_ways(ctx, "stack", "x", 8, out, "trace")
    assert sorted(ctx.ways) == ["launch", "layers"]
    ctx, out = context(single_launch, outputs={"launch": 1, "layers": 2})
    with pytest.raises(SystemExit, match="disagree"):
        bench.check_ways(ctx, "stack", "x", 8, out, "trace")


def test_a_gate_with_one_way_only_is_refused():
    ctx, out = context(False, persistent=False)
    with pytest.raises(SystemExit, match="nothing to check"):
        bench.check_ways(ctx, "stack", "x", 8, out, "trace")


def test_one_launch_rows_are_one_launch(monkeypatch):
    ctx, out = context(False)
    ctx.alloc.return_value = out
    monkeypatch.setattr(workload, "LayerWeights", mock.MagicMock())
    monkeypatch.setattr(workload, "hidden_rows", mock.MagicMock())
    monkeypatch.setattr(workload, "layer_bytes", lambda *a: 1)
    monkeypatch.setattr("zerocool_amd.StackTrace", mock.MagicMock())
    row = bench.one_launch_layer(ctx, "S", 8, 3)
    assert set(ctx.ways) == {"launch"} and row["path"] == "persistent single-launch kernel"
