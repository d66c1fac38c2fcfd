"""bench.py's host-side contract, without a GPU: the multi-GPU refusal, the
variant table of the Barnes-Hut block and the roofline figures it reads from the
counter summaries in profiles/."""
import json
import sys
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]
sys.path.insert(0, str(ROOT))

import bench  # noqa: E402


def test_more_than_one_gpu_is_refused(capsys):
    assert bench.main(["--gpus", "2"]) == 2
    assert "one GPU" in capsys.readouterr().err


def test_variant_labels_unique_and_counter_keys_name_variants():
    labels = [v[0] for v in bench.bh_variants(True)]
    assert len(labels) == len(set(labels))
    for key, label in bench.BH_COUNTER_VARIANT.items():
        assert label in labels, (key, label)


def test_roofline_figures_follow_the_preferred_variant():
    n = 1 << 22
    morton = "morton tree: quadrupole theta=0.6, local far field, near 2"
    heap = "quadrupole theta=0.62, local far field, near 3"
    r = bench.bh_roofline_from_profile(n, morton)
    assert r["variant"] == morton and r["source"].endswith("bh_morton_two_level_walk_plummer_4194304.md")
    assert r["valu"] > 0 and r["traffic"] > 0
    r = bench.bh_roofline_from_profile(n, heap)
    assert r["variant"] == heap and r["source"].endswith("bh_two_level_walk_counters_plummer_4194304.md")
    # a variant without counters falls back to one that has them
    assert bench.bh_roofline_from_profile(n, "plain theta=0.5") is not None
    assert bench.bh_roofline_from_profile(1 << 10, morton) is None


def test_direct_traffic_figure_present():
    assert bench.traffic_from_profile(1 << 18) > 0


def test_roofline_falls_back_to_the_same_tree():
    n = 1 << 22
    r = bench.bh_roofline_from_profile(n, "morton tree: quadrupole theta=0.7, local far field, near 3")
    assert r["variant"].startswith("morton tree:")
    r = bench.bh_roofline_from_profile(n, "quadrupole theta=0.8, local far field, near 5")
    assert not r["variant"].startswith("morton tree:")


def _run(label):
    """A Barnes-Hut run as bh_bench leaves it, every number with all its digits."""
    x = 123.45678901234567
    err = {"rms": x, "p99": x, "max": x, "samples": 8192}
    return {"variant": label, "ratio": x, "theta": 0.6, "tree": "morton", "multipole": "quadrupole", "quad_near": 2.0,
            "far_field": "local", "steps_per_s": x, "ms_per_step": x, "tree_build_ms": x, "walk_ms": x,
            "group_walk_ms": x, "interactions_per_body": x, "node_visits_per_body": x, "node_GB_per_s": x,
            "spills_or_fallbacks": 0, "rk4_steps_per_s": x, "force_rel_err": err,
            "force_rel_err_by_seed": {"4": err, "5": err, "6": err}, "rms_max_over_seeds": x, "p99_max_over_seeds": x}


def test_line_is_short_and_whole():
    """The line of a full run fits where only the end of the output is kept, with the
    contract's keys, the value to its last digit and every variant."""
    x = 123.45678901234567
    labels = [v[0] for v in bench.bh_variants(True)]
    best = {"variant": labels[-2], "tree": "morton", "steps_per_s": x, "rms": x, "rms_max_over_seeds": x, "walk_ms": x,
            "tree_build_ms": x, "speedup_vs_plain_theta_0.5": x}
    equal = [{"plain": labels[k], "plain_rms": x, "plain_p99": x, "plain_rms_max_over_seeds": x, "plain_steps_per_s": x,
              "fastest": labels[-2], "rms": x, "p99": x, "rms_max_over_seeds": x, "steps_per_s": x, "speedup": x}
             for k in range(3)]
    text = "x" * 300
    base = {"value": x, "unit": "pair-interactions/s", "cores": 16, "kind": "port", "sample": text[:220]}
    roof = {f"figure_{k}": x for k in range(12)} | {"kernel": text[:80], "variant": labels[-2], "source": text[:60]}
    contract = {"metric": bench.METRIC, "value": 5113514432704.267, "unit": "pair-interactions/s", "n_gpus": 1,
                "steps": 20, "warmup": 5, "ms_per_step": 846.6441409999987, "higher_is_better": True, "scaling": "weak",
                "vs_baseline": None, "dtype": "fp32", "data": "synthetic"}
    out = contract | {
        "config": {"workload": text[:180], "n": 262144, "fcompute_per_step": 63.0, "parallelism": "single-gpu"},
        "roofline": roof, "force_error": {"rms_rel": x, "max_rel": x, "vs": text[:50]}, "cpu_baseline": base,
        "barnes_hut": {"workload": text, "n": 1 << 22, "error_seeds": [4, 5, 6], "runs": [_run(v) for v in labels],
                       "best_at_rms_1e-3": best, "roofline": roof,
                       "learned_gate": {"learned": labels[-1], "rms_by_seed": {"4": x, "5": x, "6": x},
                                        "without_network": {"variant": labels[-1], "steps_per_s": x, "rms_by_seed":
                                                            {"4": x, "5": x, "6": x}}} | {f"k{k}": x for k in range(7)},
                       "at_equal_error": equal, "cpu_baseline": base},
        "two_plummer": {"workload": text, "n": 1 << 20, "runs": [_run(v) for v in labels[:4]], "best_at_rms_1e-3": best},
        "vector_ops": {"n": 1 << 22, "runs": [{"op": "fmaddn_corr k=12", "bytes": x, "ms": x, "GB_per_s": x,
                                               "frac_of_8TBps": x}] * 4},
    }
    line = bench.bench_line(out)
    assert len(line.encode()) <= bench.LINE_BYTES and "\n" not in line
    back = json.loads(line)
    assert {k: back[k] for k in contract} == contract
    assert [r["variant"] for r in back["barnes_hut"]["runs"]] == labels
    assert back["barnes_hut"]["runs"][0]["steps_per_s"] == 123.46
    assert len(back["vector_ops"]["runs"]) == 4 and back["vector_ops"]["runs"][0]["ms"] == 123.46
