"""bench.py's line on stdout: whole in the tail of a log, with the measurement as it is
(no GPU)."""
import json
import os
import sys

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import bench                                                   # noqa: E402


def report(entries):
    """A report of the shape that a full run makes, its lists of this length."""
    x = 1.0 / 3.0
    error = [dict(n=q, steps=q, rho=[x, x], eps=[x, x], vel=[x, x]) for q in range(entries)]
    solve = dict(wall_s=x, time_to_solution_s=dict(p50=x, p99=x, max=x), node_steps_per_s=x, max_members=1024)
    roofline = dict(kernel="k" * 90, traffic_source="profiles/" + "t" * 60, bound="valu", achieved=x, peak=x,
                    unit="TFLOP/s", frac=x, traffic=3558703446, flops_per_launch=dict(fp64=1 << 40), note="n" * 200,
                    hbm=dict(achieved=x, peak=8000.0, unit="GB/s", frac=x, algorithmic_bytes=1 << 31, traffic=1 << 31),
                    issue=dict(valu_wave_instructions=x, issue_ms=x, kernel_ms=x, busy_frac=x, note="n" * 130),
                    l2_hit_rate=x, gather=dict(loads_per_neighbour=6, floor_ms=x, kernel_ms=x, frac=x, note="n" * 250))
    stage = dict(ghosts=x, neighbors=x, cull=x, sum_density=x, derivatives=x, pack=x)
    parity = dict(csr_bitexact=True, directed_entries=255578960, fields_rel_linf_l2={f"f{q}": [x, x] for q in range(20)},
                  worst=x, bar=1e-12, within_bar=True, check_s=x, oracle="o" * 90)
    return dict(metric=bench.METRIC, value=17925876543.123456, unit="pair-interactions/s", n_gpus=1, steps=20, warmup=5,
                ms_per_step=7.3187654321, higher_is_better=True, scaling="weak", vs_baseline=None, dtype="f64",
                data="synthetic",
                config=dict(workload="w" * 150, nodes=2097152, ghost_nodes=301232, pairs=131196424, stage_ms=stage),
                roofline=roofline, density_gather=dict(frac=x, note="n" * 130), parity_vs_oracle=parity,
                mixed_pass=dict(value=x, ms_per_step=x, speedup_vs_fp64=x, stage_ms=stage, roofline=roofline,
                                parity_vs_oracle=parity),
                rk2=dict(steps=5, ms_per_step=x, dt=[x] * 5, step="s" * 120, pairs_per_s=x),
                copy_probe=dict(bytes_read=1 << 28, ms=x, GBps=x, kernel="k" * 40),
                ensemble=dict(solve, workload="w" * 200, error_vs_fp64=dict(per_member=error, note="n" * 300),
                              sequential_plain=dict(sample=error, speedup=x, method="m" * 200)),
                serving=dict(workload="w" * 200, batched=solve, one_at_a_time=solve, fp64_lane=solve,
                             error_vs_fp64=dict(rel_linf=dict(rho=x, eps=x, vel=x), within_bar=False, per_request=error)),
                periodic=dict(workload="w" * 200, fp64=dict(ms_per_step=x, drift=error),
                              mixed=dict(ms_per_step=x, drift=error)),
                autotune=dict(table_file="t" * 60, imported=20, decisions=error, variants="v" * 100),
                cpu_baseline=dict(value=48502689.87298658, unit="pair-interactions/s", cores=16, kind="port",
                                  sample="s" * 230, stage_ms=stage, cpu_model="AMD EPYC", host_cpus=16))


def test_line_is_short_and_complete():
    for entries in (8, 400):
        full = report(entries)
        text = bench.stdout_line(full)
        assert "\n" not in text and len(text) <= bench.LINE_LIMIT <= 4000
        line = json.loads(text)
        for k in ("metric", "value", "unit", "n_gpus", "steps", "warmup", "ms_per_step", "higher_is_better", "scaling",
                  "vs_baseline", "dtype", "data"):
            assert line[k] == full[k], k
        assert line["config"]["workload"] == full["config"]["workload"]
        for k in ("roofline", "cpu_baseline", "parity_vs_oracle", "ensemble", "serving", "mixed_pass"):
            assert k in line, k
        assert line["roofline"]["frac"] and line["ensemble"]["time_to_solution_s"]["p99"]


def test_report_holds_everything(tmp_path, capsys):
    full = report(8)
    path = str(tmp_path / "report.json")
    bench.emit(full, path)
    assert json.load(open(path)) == full
    assert capsys.readouterr().out.count("\n") == 1
