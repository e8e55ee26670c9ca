"""Which kernel prompt attention of the layer-stack models takes (attn_plan.hpp, plain C++ on the CPU): calls whose measured times (us, beside each:
waves on their own / 16 / 32 rows a wave) the rules have to tell apart."""
from __future__ import annotations

import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

GQA = [   # dim, rows, position, heads, kv-heads, kernel
    (128, 40, 0, 16, 4, 16),        # 7.0 / 7.0
    (128, 200, 0, 8, 2, 0),         # 7.3 / 8.5
    (128, 500, 0, 8, 2, 0),         # 9.6 / 11.5
    (128, 1000, 0, 4, 1, 0),        # 13.3 / 17.0
    (128, 64, 1000, 16, 4, 0),      # 14.1 / 19.1
    (128, 20, 3000, 16, 4, 0),      # 26.4 / 41.9
    (128, 256, 0, 32, 8, 16),       # 9.3 / 8.9
    (128, 1000, 0, 16, 4, 16),      # 23.5 / 18.5 / 25.6
    (128, 1000, 3000, 16, 4, 16),   # 103 / 61 / 82
    (128, 1500, 0, 16, 4, 32),      # 47.0 / 44.9 / 38.4
    (128, 2048, 0, 16, 4, 32),      # 50.9 / 54.2 / 44.1
    (64, 500, 0, 16, 4, 0),         # 7.1 / 8.1
    (64, 2000, 0, 4, 1, 0),         # 14.5 / 19.4
    (64, 256, 0, 48, 12, 16),       # 7.8 / 6.6
    (64, 2048, 0, 16, 4, 16),       # 32.0 / 28.1 / 33.0
    (64, 800, 0, 48, 12, 16),       # 29.9 / 21.5 / 25.2
    (64, 2048, 0, 32, 8, 32),       # 59.2 / 48.7 / 46.6
]
LATENT = [   # dim, rot, rows, position, heads, kernel
    (128, 64, 100, 0, 4, 16),       # 7.2 / 6.9
    (128, 64, 700, 0, 4, 0),        # 14.0 / 16.8
    (128, 64, 700, 0, 8, 0),        # 15.4 / 17.1
    (128, 64, 300, 0, 20, 16),      # 12.1 / 11.1
    (128, 64, 64, 1000, 16, 0),     # 20.3 / 24.0
    (128, 64, 500, 1000, 8, 0),     # 25.4 / 30.9
    (128, 64, 1000, 3000, 4, 16),   # 100 / 71 / 104
    (128, 64, 64, 3000, 24, 16),    # 75.8 / 58.4 / 65.2
    (128, 64, 1024, 0, 16, 16),     # 28.3 / 22.2 / 30.5
    (128, 64, 2048, 0, 16, 32),     # 64.8 / 68.3 / 53.1
    (128, 64, 1300, 0, 24, 0),      # 48.1 / 51.4 / 57.5
    (128, 64, 3000, 0, 12, 0),      # 103 / 142 / 127
    (128, 32, 1300, 0, 12, 16),     # 35.5 / 25.9 / 37.1
    (128, 32, 2048, 0, 16, 32),     # 62.4 / 62.3 / 52.1
    (128, 32, 3000, 0, 12, 0),      # 97.8 / 129 / 124
    (64, 64, 300, 0, 8, 16),        # 8.2 / 7.7
    (64, 64, 1024, 0, 16, 16),      # 21.0 / 14.3
    (64, 64, 1300, 0, 24, 0),       # 33.6 / 33.6 / 38.6
    (64, 32, 300, 0, 8, 16),        # 7.8 / 7.3
    (64, 32, 2048, 0, 2, 0),        # 21.7 / 23.0
    (64, 32, 2048, 0, 24, 16),      # 60.8 / 49.9 / 62.0
]


def test_kernels(tmp_path):
    lines = ["gqa_rows_a_wave(%d, %d, %d, %d, %d)" % c[:5] for c in GQA] + ["latent_rows_a_wave(%d, %d, %d, %d, %d)" % c[:5] for c in LATENT]
    (tmp_path / "plan.cpp").write_text('#include <stdio.h>\n#include "attn_plan.hpp"\nint main() {\n' +
                                       "".join('  printf("%%d\\n", ti::%s);\n' % s for s in lines) + "}\n")
    exe = str(tmp_path / "plan")
    subprocess.run(["g++", "-std=c++20", "-O1", "-I" + os.path.join(ROOT, "turboinfer_amd", "csrc", "kernels"), str(tmp_path / "plan.cpp"), "-o", exe], check=True)
    got = [int(v) for v in subprocess.run([exe], capture_output=True, text=True, check=True).stdout.split()]
    for call, want, have in zip(lines, [c[5] for c in GQA + LATENT], got, strict=True):
        assert have == want, call
