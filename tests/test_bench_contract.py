"""The bench.py output contract: one JSON line with the metric, its roofline and CPU baseline
blocks (GPU), and a clear refusal of more than one GPU (CPU)."""
import json
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_more_than_one_gpu_is_refused():
    r = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), "--gpus", "2"], capture_output=True,
                       text=True, timeout=120, cwd=ROOT)
    assert r.returncode != 0
    assert "one GPU" in r.stdout + r.stderr


@pytest.mark.gpu
def test_default_line_contract():
    # a short default run (few steps, no extra blocks): every field the line promises, with values
    # that are consistent with each other
    r = subprocess.run([sys.executable, "-u", os.path.join(ROOT, "bench.py"), "--steps", "5", "--warmup", "2",
                        "--no-blocks"], capture_output=True, text=True, timeout=300, cwd=ROOT)
    assert r.returncode == 0, r.stderr[-2000:]
    lines = [ln for ln in r.stdout.splitlines() if ln.strip().startswith("{")]
    assert len(lines) == 1
    d = json.loads(lines[0])
    for k in ("metric", "value", "unit", "n_gpus", "steps", "warmup", "ms_per_step", "higher_is_better", "scaling",
              "vs_baseline", "dtype", "data", "config", "roofline", "cpu_baseline"):
        assert k in d, k
    assert d["n_gpus"] == 1 and d["steps"] == 5 and d["warmup"] == 2 and d["higher_is_better"] is True
    assert "workload" in d["config"]
    ro = d["roofline"]
    for k in ("bound", "achieved", "peak", "unit", "frac", "traffic"):
        assert k in ro, k
    assert ro["bound"] == "hbm" and ro["unit"] == "GB/s" and ro["peak"] == 8000.0
    assert abs(ro["frac"] - ro["achieved"] / ro["peak"]) < 1e-9 and 0.0 < ro["frac"] < 1.0
    cb = d["cpu_baseline"]
    for k in ("value", "unit", "cores", "kind", "sample"):
        assert k in cb, k
    assert cb["kind"] in ("port", "reference") and cb["cores"] >= 1 and cb["value"] > 0
    # DOF-updates per second of the timed steps: value = ndof * steps / wall time
    ndof = d["config"].get("ndof")
    if ndof:
        assert abs(d["value"] * d["ms_per_step"] * 1e-3 / ndof - 1.0) < 0.05


@pytest.mark.gpu
@pytest.mark.parametrize("kind,n,geometry", [("quad4", 700, (64, 64, 64, 64)), ("hex8", 48, (192, 192, 768, 800))])
def test_quadrature_rows_count_the_bytes_they_move(kind, n, geometry):
    # geometry + elemvec + qtensor per element: what the kernels move, not the stored geometry they no longer read
    import bench

    blk = bench.api_kernels(kind, n)
    vec, ten = (64, 288) if kind == "quad4" else (192, 576)
    for nm, scale, geo in (("f64", 1.0, geometry[:2]), ("f32", 0.5, geometry[2:])):
        for key, g in (("SymGradN_vector", geo[0]), ("GradN_vector", geo[0]), ("Int_gradN_dot_tensor2_dV", geo[1])):
            row = blk[nm][key]
            assert row["bytes_per_element"] == g + scale * (vec + ten)
            gbs = row["bytes_per_element"] * blk["nelem"] / row["us"] * 1e-3
            assert abs(row["achieved_GBs"] / gbs - 1.0) < 1e-9 and abs(row["frac"] * bench.HBM_PEAK_GBS / gbs - 1.0) < 1e-9
