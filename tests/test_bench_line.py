"""The benchmark's output line: short enough to be read whole from the end of
its output, with every key of its contract and the sections' figures."""
import json

import bench

CONTRACT = {"metric": bench.METRIC, "value": 1.763456789012e11, "unit": "DOF-updates/s", "n_gpus": 1, "steps": 20,
            "warmup": 5, "ms_per_step": 0.1115, "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
            "dtype": "f32", "data": "synthetic", "config": {"workload": "w" * 300, "elements": 65536}}


def _section(n, depth=2):
    leg = {"ms_per_step": 0.123456789, "dof_updates_per_s": 1.23456789e11, "stage_ms": [0.1] * 3, "note": "n" * 200}
    return leg if depth == 0 else {f"leg{i}": _section(n, depth - 1) for i in range(n)}


def test_line_keeps_contract_and_figures():
    record = dict(CONTRACT, triangles={"workload": "x" * 500, "fp64": _section(1, 0)}, batched=None)
    line = json.loads(bench.output_line(record))
    assert {k: line[k] for k in CONTRACT} == CONTRACT
    assert line["triangles"] == {"fp64": {"ms_per_step": 0.12346, "dof_updates_per_s": 1.2346e11}}
    assert line["batched"] is None


def test_line_is_short():
    record = dict(CONTRACT, **{k: _section(6) for k in bench.DETAIL})
    assert len(json.dumps(record)) > 50000
    line = bench.output_line(record)
    assert len(line) <= bench.LINE_MAX and "\n" not in line
    assert {k: json.loads(line)[k] for k in CONTRACT} == CONTRACT
