"""tools/pmc_traffic.py on a synthetic counter file: every projection of a batched step is told apart by its place in the step."""
from __future__ import annotations

import csv
import json
import os
import subprocess
import sys

import pytest

from conftest import ROOT


@pytest.mark.parametrize("kernels", [("gemm_block_kernel", "gemm_block_kernel", "gemm_block_kernel", "gemm_wide_kernel", "gemm_wide_kernel"),
                                     ("gemm_few_kernel", "gemm_few_kernel", "gemm_few_kernel", "gemm_wide_kernel", "gemm_wide_kernel")])
def test_classes_by_step_position(tmp_path, kernels):
    names = ["qkv", "o", "gate_up", "down", "lm_head"]
    kib = dict(zip(names, (3000, 2000, 9000, 5000, 40000)))
    rows = []
    for _ in range(2):
        step = ["step_begin_kernel"] + [n for _ in range(22) for n in ("qkv", "attn_spread_kernel", "o", "gate_up", "down")] + ["lm_head"]
        for n in step:
            k = kernels[names.index(n)] if n in names else n
            rows.append(dict(Dispatch_Id=len(rows) + 1, Kernel_Name="void ti::%s<4, 4>(ti::GemvArgs)" % k, Counter_Name="FETCH_SIZE", Counter_Value=kib.get(n, 7)))
    src, dst = tmp_path / "c.csv", tmp_path / "o.json"
    with open(src, "w", newline="") as f:
        w = csv.DictWriter(f, rows[0])
        w.writeheader()
        w.writerows(rows)
    subprocess.run([sys.executable, os.path.join(ROOT, "tools", "pmc_traffic.py"), str(src), str(dst), "--model", "tinyllama-1.1b", "--batch", "64"],
                   check=True, capture_output=True)
    out = json.load(open(dst))
    assert out["class_labels"] == "step position"
    fam = out["kernels"]["gemm_family"]
    assert fam["dispatches"] == 2 * (4 * 22 + 1)
    assert {n: c["traffic_bytes"] for n, c in fam["classes"].items()} == {n: v * 2048 for n, v in kib.items()}
