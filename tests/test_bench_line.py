"""bench.py's result line: one JSON object that a reader of the output's last
8,000 characters gets whole, with the contract's keys and the summaries."""
import json


def result():
    shape = {"waves": 1, "stage_words": 512, "grid": 0, "use_queue": 0, "mode": 4, "group_size": 16,
             "lds_bytes": 16384, "reserved": 0, "tok_group": 4, "tok_chains": 16}
    third = 1.0 / 3.0
    mesh = {"workload": "heightfield_1900_q16", "n_tris": 7212402, "n_verts_out": 4376519, "meshlets": 32098,
            "g_bits": [16, 16, 16], "stream_bytes": 13333333, "side_bytes": 5333333, "bpv": third, "tune": shape,
            "ms_wall": third, "ms_kernel": third, "gtris_s": third, "hbm_gb_s": third,
            "algorithmic_bytes": 155555555, "pred_n": [33, 32, -33] * 3, "pred_K": [5, 5, 5], "prep_s": third,
            "search_write_s": third, "hbm_frac": third, "tune_sweep_ms": [[4, 16, 16384, 4, 16, 0, 0, 0.1234]] * 34}
    enc = {"bytes": 161106, "search_s": third, "predictor_s": third, "coder_s": third,
           "pred_n": [32, 32, -32] * 3, "pred_K": [5, 5, 5]}
    row = {"mesh": "uv_sphere_185369_2000054", "n_tris": 185369, "exhaustive": enc, "learned": enc,
           "learned_fallback": enc, "decode_equal": True, "exhaustive_cpu": enc}
    agg = {k: third for k in ("exhaustive_search_s", "learned_search_s", "speedup", "regret", "fallback_search_s",
                              "fallback_speedup", "fallback_regret", "cpu_exhaustive_search_s",
                              "speedup_vs_cpu_exhaustive")}
    mode = {"ms_wall": third, "ms_gpu": third, "gtris_s": third, "hbm_gb_s": third}
    return {"metric": "m", "value": third, "unit": "Gtris/s", "n_gpus": 1, "steps": 20, "warmup": 5,
            "ms_per_step": third, "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
            "dtype": "int32+f64", "data": "synthetic", "config": mesh,
            "details": {"v5": dict(mesh, f32_chain=mesh), "q16": mesh, "ico": mesh,
                        "learned_encode": {"headline_mesh": agg, "heldout": agg, "all": agg, "per_mesh": [row] * 51},
                        "batched": dict(mesh, graph=mode, launch=mode, per_mesh=mode, per_mesh_python=mode)}}


def test_result_line_fits_and_keeps_its_keys():
    import bench
    out = result()
    assert len(json.dumps(out)) > 40000
    line = bench.result_line(out)
    assert "\n" not in line and len(line) < 7500
    got = json.loads(line)
    for k in ("metric", "value", "unit", "n_gpus", "steps", "warmup", "ms_per_step", "higher_is_better", "scaling",
              "vs_baseline", "dtype", "data", "config"):
        assert k in got
    assert got["value"] == got["ms_per_step"] == 0.333333 and got["config"]["n_tris"] == 7212402
    assert got["details"]["batched"]["per_mesh"]["ms_wall"] == 0.333333   # a mode's figures, not rows
    assert got["details"]["learned_encode"]["all"]["speedup"] == 0.333333
    assert "per_mesh" not in got["details"]["learned_encode"] and "tune_sweep_ms" not in line
