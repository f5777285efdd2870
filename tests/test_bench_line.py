"""The benchmark's line on stdout: every contract field of the record, without
the threshold tables and texts that make it too long for a log's tail."""
import json
import os
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def test_headline_keeps_the_contract_and_drops_the_tables():
    import bench
    contract = {"metric": bench.METRIC, "value": 157929.16005784925, "unit": "Q(f) evals/s", "n_gpus": 1, "steps": 20,
                "warmup": 5, "ms_per_step": 25.935679, "higher_is_better": True, "scaling": "weak",
                "vs_baseline": None, "dtype": "f32", "data": "synthetic", "config": {"points": 4096}}
    table = {f"0.{i}/0": {"value": 1.0 / 3.0, "rel_l2_vs_fp64": 1e-3} for i in range(40)}
    blk = {"value": 2.0, "rel_l2_vs_fp64": 1e-3, "fallback_rate": 0.1, "by_threshold": table,
           "fastest_within_1e-3": {"value": 1.0 / 3.0}}
    record = dict(contract, roofline={"frac": 1.0 / 3.0, "note": "x" * 400},
                  surrogate=dict(blk, low_knudsen_field=dict(blk)))
    out = bench.headline(record)
    for k, v in contract.items():
        assert out[k] == (float(f"{v:.7g}") if isinstance(v, float) else v)
    assert out["roofline"] == {"frac": 0.3333333}
    for sec in (out["surrogate"], out["surrogate"]["low_knudsen_field"]):
        assert "by_threshold" not in sec and sec["value"] == 2.0 and sec["fastest_within_1e-3"]["value"] == 0.3333333
    assert "by_threshold" in record["surrogate"]
    assert len(json.dumps(out)) < 1500
