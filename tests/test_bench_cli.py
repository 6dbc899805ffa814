"""bench.py's command line on the CPU: --gpus above 1 exits with a message before any GPU
or torch work (one GPU is the whole measurement)."""

import json
import subprocess
import sys
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]


def test_more_than_one_gpu_exits_with_a_message():
    for n in ("2", "8"):
        r = subprocess.run([sys.executable, str(ROOT / "bench.py"), "--gpus", n], capture_output=True, text=True,
                           timeout=60, cwd=ROOT)
        assert r.returncode == 2, r.stderr
        assert "one GPU only" in r.stderr and f"--gpus {n}" in r.stderr
        assert r.stdout == ""  # no JSON line


def _extra(rows):
    """Records of the shape and number that a default run measures, at full float length."""
    x = 12345678901.234567
    roof = {"bound": "hbm", "achieved": x, "peak": 8000.0, "unit": "GB/s", "frac": 0.16318375809232177, "traffic": None}
    step = {"n_envs": 65536, "steps": 1000, "env_steps_per_s": x, "us_per_launch": 3.3712229728698726, "roofline": roof,
            "cpu_baseline": {"value": x, "unit": "env-steps/s", "sample": "s" * 90}, "speedup_vs_cpu": 1766.4341861999876}
    sweeps = {str(s): dict(step, wall_s=0.029813063000005968, alive_after=[[32, 105973]] * 8) for s in (4, 8, 16)}
    return {"cartpole_sweep": {"rows": [{"n": 1 << i, "single": x, "sampled": x, "fused_array": x} for i in range(rows)],
                               "crossover_n": 1},
            "cartpole_copy_floor": [{"n_envs": 1 << 18, "copy_us_per_launch": 2.9276499524712563}] * 2,
            "legged4_es_rollout": {"by_sweeps": sweeps}, "legged2_es_rollout": {"by_sweeps": sweeps},
            "step_bodies": {f"body{i}": step for i in range(12)},
            "legged_step_sweeps": {f"c{c}_s{s}": step for c in (2, 4) for s in (1, 2, 4, 8, 16, 32)}}


def test_result_line_fits_a_log_tail():
    """The line is one short JSON object: every contract key, each workload's rates, and nothing of
    what only the full record holds; entries that do not fit leave it, the headline never does."""
    sys.path.insert(0, str(ROOT))
    import bench

    line = {"metric": bench.METRIC, "value": 60312345678.123456, "unit": "env-steps/s", "n_gpus": 1, "steps": 20,
            "warmup": 5, "ms_per_step": 0.004791637856415464, "higher_is_better": True, "scaling": "weak",
            "vs_baseline": None, "dtype": "fp32", "data": "synthetic", "config": {"workload": "w" * 200},
            "roofline": {"frac": 0.40412}, "cpu_baseline": {"value": 63232219.5}, "extra": _extra(23)}
    text = bench.result_line(line)
    got = json.loads(text)
    assert len(text) < bench.LINE_CHARS < 8000 and "\n" not in text
    assert got["extra"].keys() == line["extra"].keys()
    assert {k: v for k, v in got.items() if k != "extra"} == {k: v for k, v in line.items() if k != "extra"}
    assert got["extra"]["step_bodies"]["body0"] == {"env_steps_per_s": 1.235e10, "us_per_launch": 3.371, "frac": 0.1632,
                                                    "speedup_vs_cpu": 1766.0}
    assert got["extra"]["cartpole_sweep"]["rows"]["4"] == 1.235e10
    long = json.loads(bench.result_line(dict(line, extra=_extra(2000))))
    assert "cartpole_sweep" not in long["extra"] and "step_bodies" in long["extra"] and long["value"] == line["value"]
