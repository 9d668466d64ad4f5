"""The bench's JSON line stays short enough to be read back from the end of its
output: no time series, floats rounded, every figure still there."""
import json

import numpy as np

import bench


def _result(points):
    rng = np.random.default_rng(1)
    names = ("omega", "impulse", "angular_impulse", "helicity", "ke")
    paths = {}
    for p in ("fp64", "fp32c", "learned", "quadrupole"):
        rec = {"dev": {k: rng.random(points).tolist() for k in names},
               "drift": {k: rng.random(points).tolist() for k in names},
               "e_u_maxnorm": rng.random(points).tolist(), "e_u_rms": rng.random(points).tolist()}
        rec["max_dev"] = {k: max(v) for k, v in rec["dev"].items()}
        rec["max_drift"] = {k: max(v) for k, v in rec["drift"].items()}
        rec["max_e_u_maxnorm"] = max(rec["e_u_maxnorm"])
        paths[p] = rec
    runs = [{"nu": nu, "particles": 65536, "t": np.linspace(0, 0.4, points).tolist(), "paths": paths, "seconds": 1.23456789}
            for nu in (1e-4, 0.0)]
    return {"metric": "steps/s", "value": 0.42343427194403133, "n_gpus": 1, "higher_is_better": True, "vs_baseline": None,
            "drift": {"workload": "leapfrog_64k", "steps": 200, "runs": runs}}


def test_line_without_series():
    r = _result(21)
    line = bench.result_line(r)
    assert "\n" not in line and len(line) < 3000
    back = json.loads(line)
    assert back["value"] == 0.4234343 and back["n_gpus"] == 1 and back["higher_is_better"] is True
    assert back["vs_baseline"] is None
    for run, ref in zip(back["drift"]["runs"], r["drift"]["runs"]):
        assert set(run) == {"nu", "particles", "paths", "seconds"}
        for p, rec in run["paths"].items():
            assert set(rec) == {"max_dev", "max_drift", "max_e_u_maxnorm"}
            for k, v in rec["max_dev"].items():
                assert abs(v - ref["paths"][p]["max_dev"][k]) <= 5e-3 * v
    assert "t" in r["drift"]["runs"][0] and "dev" in r["drift"]["runs"][0]["paths"]["fp64"]  # the result itself is kept


def test_line_with_series():
    back = json.loads(bench.result_line(_result(21), series=True))
    assert len(back["drift"]["runs"][1]["t"]) == 21 and len(back["drift"]["runs"][0]["paths"]["fp32c"]["dev"]["ke"]) == 21


def test_line_without_a_drift_leg():
    assert json.loads(bench.result_line({"value": 1.5, "steps": 3})) == {"value": 1.5, "steps": 3}
