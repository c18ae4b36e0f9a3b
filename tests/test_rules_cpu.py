"""The dispatch rules of csrc/rules.h at sizes where both sides were timed on the card:
the quicker side is taken (sizes within 5 % of each other are left to the rule).
"""
import os
import subprocess

from helpers import ROOT

APG = [  # n, t, oc, channels per workgroup, us by sample, us by channels
    (1, 6000, 64, 2, 482.1, 38.8), (2, 6000, 64, 2, 502.1, 41.0), (4, 1500, 64, 2, 113.9, 14.1), (4, 375, 64, 2, 22.0, 5.9),
    (1, 100, 64, 2, 7.7, 4.3), (1, 12, 64, 2, 3.3, 4.2), (8, 4, 64, 2, 3.1, 4.6), (32, 100, 64, 2, 8.4, 14.5),
    (32, 750, 64, 2, 63.5, 36.5), (128, 375, 64, 2, 39.1, 87.2), (128, 750, 64, 2, 76.9, 130.9), (64, 6000, 64, 2, 641.7, 405.4),
    (256, 6000, 64, 2, 902.6, 1662.4), (512, 25, 64, 2, 7.2, 196.9), (512, 1500, 64, 2, 396.3, 868.9),
    (256, 750, 8, 2, 17.4, 39.9), (64, 12, 8, 2, 6.4, 4.7), (1, 750, 8, 2, 10.2, 5.0),
    (256, 750, 7, 1, 16.8, 52.1), (256, 3000, 7, 1, 47.3, 170.9), (8, 200, 7, 1, 8.1, 3.9), (256, 3000, 1, 1, 39.2, 9.0),
    (1, 750, 1024, 2, 964.0, 18.2), (16, 750, 1024, 2, 1050.0, 265.1), (8, 12, 1024, 2, 12.8, 50.5), (256, 25, 1024, 2, 53.7, 1551.7),
]

ONE_ROW = [  # key blocks, groups of 64 weight rows, us in three launches, us in one (norm prologue)
    (32, 16, 7.2, 5.3), (32, 64, 8.0, 5.6), (32, 96, 8.3, 5.7), (32, 204, 10.0, 7.3), (32, 256, 7.4, 6.5), (32, 320, 8.8, 8.3),
    (32, 512, 10.0, 9.3), (64, 192, 13.4, 9.6), (64, 256, 11.0, 9.7), (64, 320, 13.1, 12.1), (64, 512, 16.1, 14.4),
    (33, 128, 9.3, 6.7), (33, 288, 9.4, 9.9), (40, 320, 9.5, 10.3), (8, 288, 5.4, 6.2), (8, 512, 5.9, 6.6), (16, 288, 6.4, 6.8),
    (192, 32, 12.0, 14.2), (32, 2370, 29.8, 35.0),
]

TILES = [  # 64 x 64 tiles, resident workgroups, key splits of the 128 x 128 tiles, key blocks, us 128 x 128, us 64 x 64 (or per cent)
    (1, 512, 4, 64, 27.5, 13.2), (288, 512, 4, 64, 54.8, 49.3), (512, 512, 2, 64, 31.9, 21.4), (512, 512, 4, 304, 100.0, 90.0),
    (1152, 512, 1, 64, 54.8, 49.3), (1600, 512, 1, 64, 64.0, 70.0), (640, 512, 3, 128, 56.0, 60.0),
    (672, 512, 2, 192, 100.0, 89.0), (770, 512, 2, 192, 93.5, 84.7), (1024, 512, 2, 192, 100.0, 94.0), (1088, 512, 1, 20, 100.0, 94.0), (960, 512, 1, 12, 100.0, 93.0),
    (640, 512, 1, 8, 100.0, 92.0), (768, 512, 1, 8, 100.0, 92.0), (768, 512, 1, 5, 100.0, 104.0), (1088, 512, 1, 8, 100.0, 107.0), (1078, 512, 1, 5, 100.0, 122.0), (544, 512, 1, 1, 100.0, 110.0),
    (912, 512, 1, 4, 14.4, 15.2), (1088, 512, 1, 1, 100.0, 131.0),
]


def _run(tmp_path, expr, rows):
    src = tmp_path / "r.cpp"
    body = "".join(f"    printf(\"%d\\n\", (int) ({expr(r)}));\n" for r in rows)
    src.write_text('#include "rules.h"\n#include <cstdio>\nusing namespace mi;\nint main() {\n' + body + "}\n")
    exe = tmp_path / "r"
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "hbd-acestep.cpp_amd", "csrc"), str(src), "-o", str(exe)],
                   check=True)
    return [int(v) for v in subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout.split()]


def test_apg_takes_the_quicker_split(tmp_path):
    got = _run(tmp_path, lambda r: f"apg_by_sample({r[0]}, {r[1]}, {r[2]}, {r[3]})", APG)
    bad = [r for r, g in zip(APG, got) if g != (r[4] < r[5])]
    assert not bad, bad


def test_one_row_takes_the_quicker_route(tmp_path):
    got = _run(tmp_path, lambda r: f"mmv_one_launch({r[0]}, {r[1]})", ONE_ROW)
    bad = [r for r, g in zip(ONE_ROW, got) if g != (r[3] < r[2])]
    assert not bad, bad


def test_products_take_the_quicker_tiles(tmp_path):
    got = _run(tmp_path, lambda r: f"mmq_small_tiles({r[0]}, {r[1]}, {r[2]}, {r[3]})", TILES)
    bad = [r for r, g in zip(TILES, got) if g != (r[5] < r[4])]
    assert not bad, bad
