"""Two-table mode of the profile summary: passes of a sample are found by their order, whether or not a step has a norm pass
of its own (norms folded into the write before, or none needed).  Synthetic traces; no device calls."""
import csv

import pytest

from _pkg import PKG_DIR  # noqa: F401
import importlib.util
import os

spec = importlib.util.spec_from_file_location("rocprof_summary", os.path.join(PKG_DIR, "rocprof_summary.py"))
rs = importlib.util.module_from_spec(spec)
spec.loader.exec_module(rs)

V = "HIP_vector_type<float, 2u>"                          # as traces spell float2
NORM, WRITE = f"void gs::gather_kernel<{V}, 1, 2>(x)", f"void gs::gather_kernel<{V}, 2, 2>(x)"
FOLD = f"void gs::gather_fold_kernel<{V}, 4, 2, true, false>(x)"
SAMPLES = {"every step": [NORM, WRITE, NORM, WRITE, NORM, WRITE], "none needed": [WRITE, NORM, WRITE, WRITE],
           "folded": [NORM, WRITE, NORM, FOLD, WRITE]}


@pytest.mark.parametrize("sample", SAMPLES.values(), ids=SAMPLES.keys())
def test_gather_finds_passes_of_any_kind(sample, tmp_path):
    other = "void gs::sweep_reduce_kernel<2>(x)"
    (tmp_path / "plan.txt").write_text("3 3 20\n" + "0 20 20 0 0 0 1 0 0 0 0 0 1 0\n" * 3)
    for name, counter in (("trace", None), ("fetch", "FETCH_SIZE"), ("write", "WRITE_SIZE")):
        (tmp_path / name).mkdir()
        rows, t, n = [], 0, 0
        for kern in [*([] if name == "trace" else ["copy_probe_kernel"]), *3 * [k for s in sample for k in (s, other)], NORM]:
            us = 1000 if kern == NORM else 2000
            rows.append(dict(Kernel_Name=kern, Dispatch_Id=n, Start_Timestamp=t, End_Timestamp=t + 1000 * us,
                             Counter_Name=counter, Counter_Value=1024.0))
            t, n = t + 1000 * us + 10, n + 1
        file = "run_kernel_trace.csv" if name == "trace" else "run_counter_collection.csv"
        with open(tmp_path / name / file, "w", newline="") as f:
            w = csv.DictWriter(f, rows[0].keys())
            w.writeheader()
            w.writerows(rows)
    out = rs.gather(str(tmp_path / "trace"), str(tmp_path / "fetch"), str(tmp_path / "write"), str(tmp_path / "plan.txt"), 1, 3)
    norms, writes = sample.count(NORM), 3
    assert out.count("| norm |") == norms and out.count("| write |") == writes
    assert f"gather kernels {norms + 2.0 * writes:.1f} ms" in out
