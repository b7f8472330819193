"""bench.py's printed line: short enough for a log that keeps the last 8 KB of a run, the contract's own
values as measured.  (The default run measures 16 points; its figures here are the longest floats there are.)"""
import json

import bench

X = 1234567.8901234567


def _result(tokens):
    return dict(
        tokens=tokens, ms_per_step=X, tokens_per_s=X, graph_replay_ms_per_step=None, active_experts=X,
        stage_ms={n: X for n in ("router", "permute", "expert_gate_up", "expert_down", "combine", "forward")},
        stage_launches={n: 1 for n in ("router", "permute", "expert_gate_up", "expert_down", "combine", "forward")},
        forward_gbs=X, forward_tflops=X, forward_hbm_frac=X, forward_mfma_frac=X, algorithmic_bytes=X,
        algorithmic_flops=X,
        roofline=dict(bound="mfma", kernel="expert_gate_up", achieved=X, peak=2500.0, unit="TFLOP/s", frac=X,
                      traffic=X, kernel_ms=X, algorithmic_flops=X, traffic_source=dict(
                          file="profiles/ffn_kernels_deepseek_bf16_hbm_counters.txt", kernels_sha="0" * 16,
                          this_build="0" * 16, current=True)))


def _line():
    parity = dict(routing_mismatched_tokens=0, tokens_routed=16384, max_rel_err_vs_cpu_path=X, bar=X,
                  within_bar=True, sample_tokens=64, min_routing_margin=X, at_token=11351,
                  median_routing_margin=X, max_abs_diff=X, mean_abs_diff=X, rmse=X, argmax_match_rows=64,
                  argmax_rows=64)
    head = _result(4096)
    line = dict(
        metric="Mixtral-shape MoE layer tok/s; decode HBM GB/s and prefill MFMA TFLOPS", value=X, unit="tokens/s",
        n_gpus=1, steps=20, warmup=5, ms_per_step=X, higher_is_better=True, scaling="weak", vs_baseline=None,
        dtype="bf16", data="synthetic", config=dict(workload="w" * 180, tokens_per_step=4096),
        roofline=head["roofline"], cpu_baseline=dict(value=X, unit="tokens/s", cores=16, kind="port", sample="s" * 120),
        prefill=head, decode=_result(1), decode16=_result(16),
        sweep=[dict(r, **bench.compact("mixtral_bf16", r)) for r in (_result(128), _result(512))],
        parity=parity, host_entry=dict(tokens=4096, forward_host_ms=X, forward_host_pinned_ms=X, tokens_per_s=X,
                                       host_bytes_moved=X, note="n" * 110), kernels_sha="0" * 16)
    line["configs"] = [bench.compact("deepseek_bf16", _result(16384)) for _ in range(17)]
    line["configs"][0]["numeric_policy"] = "strict"
    line["configs_parity"] = {n: parity for n in ("mixtral_bf16", "tiny_f32", "mixtral_int8", "qwen_bf16",
                                                  "deepseek_bf16")}
    return line


def test_the_printed_line_fits_a_short_log():
    line = _line()
    text = json.dumps(bench.short_line(line))
    assert len(text) < 7500 < len(json.dumps(line)), len(text)
    out = json.loads(text)
    assert set(out) == set(line)
    for k in ("metric", "value", "unit", "n_gpus", "steps", "warmup", "ms_per_step", "higher_is_better", "scaling",
              "vs_baseline", "dtype", "data", "config", "cpu_baseline"):
        want = dict(line[k], value=float(f"{X:.5g}")) if k == "cpu_baseline" else line[k]
        assert out[k] == want, k
    assert abs(out["roofline"]["frac"] / X - 1) < 1e-4 and len(out["configs"]) == 17
    assert out["configs"][0]["numeric_policy"] == "strict" and out["configs_parity"]["tiny_f32"]["within_bar"]


def test_a_line_without_the_list_of_configurations():
    line = _line()
    del line["configs"], line["configs_parity"]
    line["parity"] = line["decode"] = None
    assert set(bench.short_line(line)) == set(line)
