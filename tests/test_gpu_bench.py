"""The benchmark's timed steps run what a user's program runs."""
import json
import sys

import pytest

pytestmark = pytest.mark.gpu


def test_timed_steps_use_the_native_sequences(gpu_device, monkeypatch, capsys):
    import bench
    from fusionllm_amd import _kernels as K
    native, real = [], K.block_host
    monkeypatch.setattr(K, "block_host", lambda: native.append(real() is not None) or real())
    steps, warmup = 4, 2
    monkeypatch.setattr(sys, "argv", ["bench.py", "--steps", str(steps), "--warmup", str(warmup),
                                      "--no-cpu-baseline"])
    bench.main()
    line = json.loads(capsys.readouterr().out.strip().splitlines()[-1])
    assert line["steps"] == steps and line["value"] > 0 and line["roofline"]["launches_timed"] > 0
    # one call per forward and one per backward
    assert sum(native) >= 2 * (warmup + steps)
