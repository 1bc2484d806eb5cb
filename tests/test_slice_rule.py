"""Where the sampler cuts a batch's rows over the GPU (csrc/slice_rule.h): sizes that were timed
slower cut keep one workgroup per row, sizes that were timed faster are cut."""

import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]


def _ask(tmp_path, call):
    src = tmp_path / "rule.cpp"
    src.write_text('#include <stdio.h>\n#include "slice_rule.h"\nint main() { puts(dsv41::%s ? "cut" : "whole"); }\n' % call)
    exe = tmp_path / "rule"
    subprocess.run(["g++", "-std=c++17", "-I", str(ROOT / "tiny-dsv41_amd" / "csrc"), "-o", str(exe), str(src)], check=True)
    return subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout.strip()


# min-p, rows, slices, vocabulary, bytes a logit, history, depth (min-p); cut / whole as timed
SLICES = [
    ("true, 128, 12, 129280, 2, 0, 2.4", "cut"),      # 0.72
    ("true, 128, 12, 129280, 2, 2048, 2.4", "cut"),   # 0.92
    ("true, 128, 12, 129280, 2, 4096, 2.4", "whole"),  # 1.27
    ("true, 64, 22, 129280, 2, 8192, 2.4", "whole"),  # 1.50
    ("true, 1, 64, 129280, 4, 8192, 2.4", "cut"),     # 0.92
    ("true, 1, 64, 129280, 4, 16384, 2.4", "whole"),  # 1.17
    ("true, 256, 6, 64000, 4, 8192, 2.4", "whole"),   # 2.84
    ("true, 256, 6, 129280, 2, 64, 2.4", "cut"),      # 0.99
    ("true, 256, 6, 129280, 4, 0, 2.4", "whole"),     # 1.07
    ("true, 200, 7, 129280, 4, 0, 2.4", "cut"),       # 0.99
    ("true, 1, 6, 12000, 4, 16384, 2.4", "whole"),    # 1.57
    ("false, 128, 6, 32000, 2, 4096, 2.4", "whole"),  # 1.38
    ("false, 128, 6, 129280, 2, 2048, 2.4", "cut"),   # 0.83
    ("false, 4, 75, 151936, 4, 8192, 2.4", "cut"),    # 0.61
    ("false, 1, 16, 32000, 2, 8192, 2.4", "whole"),   # 1.17
    ("false, 1, 9, 17000, 2, 4096, 2.4", "whole"),    # 1.10
    ("false, 64, 12, 151936, 4, 4096, 2.4", "cut"),   # 0.81
    ("false, 64, 11, 32000, 2, 4096, 2.4", "whole"),  # 1.18
    ("true, 32, 43, 129280, 4, 4096, 2.4", "cut"),    # 0.86
    ("true, 64, 22, 151936, 2, 4096, 2.4", "whole"),  # 1.12
    ("true, 256, 6, 151936, 2, 0, 0.41", "whole"),  # 1.13
    ("true, 256, 6, 151936, 2, 0, 1.8", "whole"),  # 1.00, with 300 history ids 1.16
    ("true, 200, 7, 129280, 4, 300, 0.97", "whole"),  # 1.17
    ("true, 160, 9, 129280, 2, 0, 0.97", "cut"),  # 0.91
    ("true, 128, 12, 129280, 4, 0, 1.8", "cut"),  # 0.87
    ("true, 256, 6, 129280, 2, 0, 4.7", "cut"),  # 0.84
]


@pytest.mark.parametrize("args,way", SLICES)
def test_top_p_and_min_p(tmp_path, args, way):
    assert _ask(tmp_path, f"slices_pay({args})") == way


# replay, rows, vocabulary, history
SPREAD = [
    ("false, 128, 9000, 16384", "cut"),    # (draws of at most 128 rows always were)
    ("true, 1, 151936, 0", "cut"),         # 0.68
    ("true, 1, 151936, 16384", "cut"),     # (8192: 0.74)
    ("true, 1, 9000, 0", "whole"),         # 1.10
    ("true, 128, 129280, 1024", "cut"),    # 0.95
    ("true, 128, 129280, 4096", "whole"),  # 1.11
    ("true, 128, 32000, 2048", "whole"),   # 1.08
    ("true, 64, 64000, 8192", "whole"),    # 1.13
    ("false, 300, 2600, 0", "cut"),
    ("false, 300, 129280, 0", "cut"),      # 0.85
    ("false, 300, 9000, 1024", "cut"),     # 0.92
    ("false, 300, 151936, 2048", "cut"),   # 0.91
    ("false, 400, 151936, 4096", "whole"),  # 1.08
    ("false, 448, 32000, 2048", "whole"),  # 1.16
    ("false, 300, 9000, 8192", "whole"),   # 1.16
    ("true, 448, 151936, 0", "cut"),       # 0.99
    ("true, 300, 32000, 4096", "whole"),   # 1.15
]


@pytest.mark.parametrize("args,way", SPREAD)
def test_full_vocabulary(tmp_path, args, way):
    assert _ask(tmp_path, f"spread_pays({args})") == way
