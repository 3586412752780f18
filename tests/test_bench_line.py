"""The benchmark's one result line stays short enough to be read whole from a log's last 12,000 characters."""
from __future__ import annotations

import json
from types import SimpleNamespace

import bench


def _line():
    """A result of the default run's shape: 24 measurements of a dozen figures with their texts and breakdowns."""
    def one(i):
        return {"workload": "a workload described in a sentence of some length, " * 2, "ms_per_step": 3.4262788000006594 + i,
                "qps": 298866.5137232273, "phases_ms": {f"phase{j}": 0.123456789012345 for j in range(12)},
                "equals_fp32_scan": True,
                "roofline": {"kernel": "some_kernel<1, 2, 3> (what it does and on which operands, at length)", "frac": 0.6348207783582,
                             "achieved": 1010.695977569987, "measured_ceiling": {"instruction": "fp16", "rate": 1592.0965602}}}

    return {"metric": "m", "value": 298866.5137232273, "ms_per_step": 3.4262788000006594,
            "roofline": {"frac": 0.4042783910279948, "kernel": "k", "power_limited_ceiling": "x" * 300},
            "cpu_baseline": None, "extra": {f"case{i}": one(i) for i in range(24)}}


def test_line_is_short_and_keeps_the_figures(capsys, tmp_path):
    full = _line()
    assert len(json.dumps(full)) > 12_000
    bench.emit(SimpleNamespace(details=str(tmp_path / "all.json")), full)
    out = capsys.readouterr().out
    assert out.count("\n") == 1 and len(out) < 9_000
    got = json.loads(out)
    assert got["value"] == full["value"] and got["ms_per_step"] == full["ms_per_step"]
    assert got["roofline"] == {"frac": 0.4042783910279948, "kernel": "k"}
    assert got["extra"]["case3"] == {"ms_per_step": 6.4263, "qps": 298870.0, "equals_fp32_scan": True,
                                     "roofline": {"frac": 0.63482, "achieved": 1010.7, "measured_ceiling": {"rate": 1592.1}}}
    assert json.loads((tmp_path / "all.json").read_text())["extra"]["case3"]["phases_ms"]["phase0"] == 0.123456789012345


def test_details_are_optional(capsys):
    bench.emit(SimpleNamespace(details=None), {"metric": "m", "value": None, "extra": {}})
    assert json.loads(capsys.readouterr().out) == {"metric": "m", "value": None, "extra": {}}
