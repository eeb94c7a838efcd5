"""bench.py's command-line contract: one JSON line with the agreed keys on one GPU, a refusal for more."""
import json
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_more_than_one_gpu_is_refused():
    proc = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), "--gpus", "2"], cwd=ROOT,
                          stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True, timeout=120)
    assert proc.returncode != 0 and proc.stdout.strip() == ""
    assert "one GPU" in proc.stderr and "--gpus 2" in proc.stderr


@pytest.mark.parametrize("kernel,r,s,fragments", [
    ("inconv_mfma_kernel<7, 7, 4, 1, 1>", 7, 7, 12), ("inconv_mfma_kernel<7, 7, 2, 1, 1>", 7, 7, 12), ("inconv_mfma_kernel<3, 3, 1, 0, 1>", 3, 3, 3),
    ("inconv_mfma_kernel<3, 3, 2, 0, 1>", 3, 3, 4), ("inconv_mfma_kernel<11, 11, 4, 0, 2>", 11, 11, 27), ("inconv_mfma_kernel<7, 8, 7, 0, 1>", 7, 8, 11),
    ("inconv_mfma_ring_kernel", 11, 11, 33), ("inconv_tiled_kernel<8, true, false, true, false>", 7, 7, 0)])
def test_first_layer_products_that_are_multiplied(kernel, r, s, fragments):
    """Counted by the selected kernel's order of K (inconv_mfma.hip: sets_of, steps_of)."""
    import bench
    assert bench.first_layer_fragments(kernel, r, s) == fragments


def test_layers_that_go_together_are_one_launch():
    """A run's record: all its operations and every output, the activations in between not read from memory."""
    import bench
    from tcbnn_amd import nets
    spec = nets.SPECS["mnist_mlp"](batch=64)
    alone = [bench.layer_work(L, spec) for L in spec]
    run = bench.launch_work(spec, spec)
    assert run["bops"] == sum(w["bops"] for w in alone) > 0
    assert sum(w["bytes"] for w in alone) - run["bytes"] == sum(64 * L["inp"] / 8 for L in spec[1:])
    assert bench.launch_work(spec[1:2], spec) == alone[1]


@pytest.mark.gpu
def test_the_mlp_is_reported_as_it_is_launched(gpu):
    proc = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), "--net", "mnist_mlp", "--batch", "256", "--steps", "3", "--warmup", "1",
                           "--no-cpu"], cwd=ROOT, stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True, timeout=120)
    assert proc.returncode == 0, proc.stderr
    d = json.loads(proc.stdout)
    assert [(r["kernel"], r["launches_per_step"]) for r in d["roofline_all_kernels"]] == [("fc_chain_kernel", 1)]
    assert d["roofline_bit_layers"]["launches_per_step"] == 1


@pytest.mark.gpu
def test_one_json_line_with_the_contract_keys(gpu):
    proc = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), "--steps", "3", "--warmup", "1",
                           "--cpu-batch", "2"], cwd=ROOT, stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True,
                          timeout=280)
    assert proc.returncode == 0, proc.stderr
    lines = [ln for ln in proc.stdout.splitlines() if ln.strip()]
    assert len(lines) == 1
    d = json.loads(lines[0])
    for key in ("metric", "value", "unit", "n_gpus", "steps", "warmup", "ms_per_step", "higher_is_better", "scaling",
                "vs_baseline", "dtype", "data", "config", "roofline", "cpu_baseline"):
        assert key in d, key
    assert d["n_gpus"] == 1 and d["steps"] == 3 and d["warmup"] == 1 and d["higher_is_better"] is True
    assert d["unit"] == "images/s" and "workload" in d["config"] and "model" not in d["config"]
    assert abs(d["value"] - 256 / (d["ms_per_step"] * 1e-3)) <= 0.01 * d["value"]
    assert abs(d["vs_baseline"] - d["value"] / 5600.0) <= 0.01 * d["vs_baseline"]
    r = d["roofline"]
    for key in ("bound", "achieved", "peak", "unit", "frac", "traffic"):
        assert key in r, key
    assert r["bound"] in ("hbm", "mfma") and abs(r["frac"] - r["achieved"] / r["peak"]) < 1e-3
    # the first layer's record says what its kernel executes: products on the matrix cores, not additions on the VALU
    assert "inconv_mfma" in r["kernel"] and "valu_fp32" not in r and "valu" not in r["binding"]
    m = r["matrix_fp16"]
    # (7x7/4: two rows' sums under way, six fragments for the twelve pairs of a row and a channel; not the fourteen of four taps each)
    assert m["flops_per_launch"] == 256 * 56 * 56 * 64 * 2 * 2 * 16 * 12 and 0 < m["frac"] < 1
    assert abs(m["achieved"] - m["flops_per_launch"] / r["avg_launch_ms"] / 1e9) <= 0.02 * m["achieved"]
    c = d["cpu_baseline"]
    for key in ("value", "unit", "cores", "kind", "sample"):
        assert key in c, key
    assert c["kind"] in ("port", "reference") and c["cores"] >= 1
    # the untimed clock-settling passes are reported, and the several-batches-in-flight figure stays out of `value`
    assert d["preheat"]["steps"] >= 8 and d["preheat"]["ms"] > 0
    a = d["as_launched"]
    assert a["unit"] == "images/s" and abs(a["value"] - 256 / (a["ms_per_step"] * 1e-3)) <= 0.01 * a["value"]
    f = d["batches_in_flight"]
    assert f["batches_in_flight"] == 2 and f["unit"] == "images/s" and f["steps"] >= 100
    assert abs(f["value"] - 256 / (f["ms_per_step"] * 1e-3)) <= 0.01 * f["value"]
    assert r["traffic"] is None or r["traffic"] > 0
    assert r["traffic_stale"] == (r["traffic"] is None)
    # the packed first-layer input is a request: its figures stay beside `value`, with the cost of the extra pass
    u = d["packed_input"]
    assert "direct" in u["kernel"] and "direct" not in r["kernel"]
    assert u["pack_ms"] > 0 and u["value_with_pack_in_every_step"] < u["value"]
    assert abs(u["value_with_pack_in_every_step"] - 256e3 / (u["ms_per_step"] + u["pack_ms"])) <= 0.01 * u["value"]
