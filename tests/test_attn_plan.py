"""Which kernel prompt attention of the layer-stack models takes (attn_plan.hpp, plain C++ on the CPU): calls whose measured times (us, beside each, with keys
that are new to the caches: waves on their own / 16 / 32 rows a wave) the rules have to tell apart."""
from __future__ import annotations

import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

GQA = [   # dim, rows, position, heads, kv-heads, kernel
    (128, 40, 0, 16, 4, 16),        # 8.8 / 7.5
    (128, 300, 0, 8, 2, 16),        # 12.4 / 11.2
    (128, 64, 1000, 20, 5, 16),     # a prompt 634 / 605
    (128, 500, 0, 16, 4, 16),       # 13.5 / 13.2
    (128, 400, 0, 32, 8, 16),       # 18.1 / 13.3
    (128, 600, 0, 4, 1, 16),        # a prompt 354 / 341
    (128, 1000, 0, 16, 4, 16),      # 27.1 / 21.2 / 28.6
    (128, 1300, 0, 16, 4, 32),      # 37.3 / 40.7 / 35.2
    (128, 2048, 0, 16, 4, 32),      # 59.0 / 59.3 / 46.9
    (64, 300, 0, 16, 4, 16),        # 8.1 / 7.7
    (64, 500, 0, 16, 4, 0),         # 8.7 / 9.3
    (64, 2048, 0, 4, 1, 0),         # 19.8 / 23.2
    (64, 30, 1800, 12, 3, 0),       # a prompt 288 / 306
    (64, 256, 0, 48, 12, 16),       # 8.5 / 7.0
    (64, 500, 0, 32, 8, 16),        # 12.2 / 9.5
    (64, 2048, 0, 16, 4, 16),       # 36.1 / 29.2 / 35.6
    (64, 1300, 0, 32, 8, 16),       # 38.8 / 30.6 / 33.5
    (64, 2048, 0, 32, 8, 32),       # 64.8 / 51.2 / 47.7
]
LATENT = [   # dim, rot, rows, heads, kernel
    (128, 64, 40, 4, 16),       # 11.0 / 6.5
    (128, 64, 640, 4, 16),      # 22.5 / 16.2
    (128, 64, 1000, 16, 16),    # 34.1 / 22.8 / 31.1
    (128, 64, 1300, 16, 32),    # 46.0 / 46.3 / 39.2
    (128, 64, 2048, 16, 32),    # 67.7 / 69.7 / 55.0
    (128, 64, 1300, 24, 0),     # 54.7 / 56.7 / 63.1
    (128, 64, 1300, 40, 32),    # 79.1 / 91.1 / 71.3
    (128, 64, 3000, 12, 0),     # 105 / 150 / 134
    (128, 32, 1300, 12, 16),    # 40.7 / 26.4 / 37.9
    (128, 32, 2048, 16, 32),    # 67.7 / 67.4 / 57.7
    (128, 32, 3000, 12, 0),     # 101 / 136 / 130
    (64, 64, 1000, 16, 16),     # 24.5 / 16.4 / 21.4
    (64, 64, 1300, 16, 32),     # 32.0 / 31.6 / 27.0
    (64, 64, 1300, 24, 0),      # 35.4 / 36.4 / 40.2
    (64, 32, 2048, 2, 16),      # 32.3 / 25.8 / 35.5
    (64, 32, 2048, 16, 16),     # 46.9 / 32.4 / 36.1
    (64, 32, 2048, 40, 16),     # 107 / 80 / 97
]


def test_kernels(tmp_path):
    lines = ["gqa_rows_a_wave(%d, %d, %d, %d, %d)" % c[:5] for c in GQA] + ["latent_rows_a_wave(%d, %d, %d, %d)" % c[:4] for c in LATENT]
    (tmp_path / "plan.cpp").write_text('#include <stdio.h>\n#include "attn_plan.hpp"\nint main() {\n' +
                                       "".join('  printf("%%d\\n", ti::%s);\n' % s for s in lines) + "}\n")
    exe = str(tmp_path / "plan")
    subprocess.run(["g++", "-std=c++20", "-O1", "-I" + os.path.join(ROOT, "turboinfer_amd", "csrc", "kernels"), str(tmp_path / "plan.cpp"), "-o", exe], check=True)
    got = [int(v) for v in subprocess.run([exe], capture_output=True, text=True, check=True).stdout.split()]
    for call, want, have in zip(lines, [c[-1] for c in GQA + LATENT], got, strict=True):
        assert have == want, call
