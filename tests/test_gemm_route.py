"""The rules that choose a form for an M > 1 product (llm-kv260_amd/csrc/gemm_route.h),
held on the CPU against times measured on an MI355X (256 CUs, weights rotated through
400 MB): a rule may cost at most 6% of the best form at any measured size. Two simpler
rules miss that at a tenth of the sizes, and are checked to: 32-token items whenever
there are 160 of them, and a line in rows x m for the whole-prompt kernel."""

from __future__ import annotations

import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CUS = 256

# m, rows, k, then microseconds: class-split kernel with 16-token and 32-token items,
# whole-prompt kernel.
TIMES = (
    (130, 64, 256, 4.5, 4.2, 3.5), (130, 700, 256, 6.3, 4.4, 3.5), (130, 1024, 256, 8.8, 5.6, 3.5),
    (130, 1400, 256, 10.7, 5.8, 3.6), (12, 5000, 256, 5.0, 5.0, 4.0), (112, 1280, 512, 8.5, 5.9, 4.4),
    (72, 1536, 512, 5.9, 5.7, 4.5), (160, 1536, 512, 9.2, 6.2, 4.6), (160, 2048, 512, 8.8, 6.5, 4.6),
    (100, 2304, 512, 8.4, 6.3, 4.7), (160, 2304, 512, 9.0, 6.5, 4.8), (130, 1024, 768, 9.6, 6.9, 5.1),
    (72, 1536, 768, 6.7, 6.7, 5.3), (16, 3072, 768, 4.7, 5.2, 5.3), (24, 3072, 768, 6.4, 5.3, 5.5),
    (64, 3333, 768, 11.5, 7.2, 5.5), (12, 10240, 768, 8.8, 7.4, 5.5), (12, 16384, 768, 11.2, 9.1, 5.9),
    (17, 2304, 1024, 6.0, 4.8, 6.0), (80, 3333, 1024, 8.6, 8.0, 6.1), (100, 3333, 1024, 10.7, 10.2, 6.2),
    (128, 3333, 1024, 11.3, 10.5, 6.2), (33, 5000, 1024, 7.5, 7.6, 6.1), (130, 1024, 1280, 11.5, 8.4, 6.7),
    (130, 1400, 1280, 14.5, 8.7, 6.8), (160, 768, 1536, 7.6, 6.4, 7.5), (128, 3072, 1536, 14.2, 10.3, 7.6),
    (64, 3333, 1536, 12.8, 9.2, 7.7), (72, 3333, 1536, 13.4, 10.5, 7.5), (100, 3333, 1536, 14.5, 12.9, 7.6),
    (128, 3333, 1536, 18.3, 13.2, 7.7), (48, 4096, 1536, 10.3, 8.8, 7.4), (48, 5000, 1536, 12.9, 10.2, 7.5),
    (33, 2048, 2048, 7.0, 6.6, 8.8), (24, 3072, 2048, 7.0, 6.7, 8.8), (64, 3072, 2048, 8.3, 9.4, 8.8),
    (96, 4096, 2048, 13.4, 11.5, 8.9), (48, 5120, 2048, 10.3, 11.3, 8.9), (17, 7168, 2048, 10.2, 9.0, 9.3),
    (48, 1024, 2304, 7.8, 8.8, 9.4), (130, 1400, 2304, 20.2, 12.1, 9.5), (72, 1536, 2304, 11.1, 11.6, 9.4),
    (24, 2048, 2304, 7.9, 8.7, 9.6), (100, 2304, 2304, 20.1, 14.7, 9.5), (48, 3333, 2304, 16.2, 12.1, 9.6),
    (16, 10240, 2304, 16.0, 14.5, 10.4), (16, 16384, 2304, 20.1, 19.1, 10.9),
    (128, 900, 2560, 10.1, 8.6, 10.1), (80, 3072, 2560, 17.0, 13.0, 10.2),
    (128, 3333, 2560, 24.9, 18.3, 10.4), (128, 4096, 2560, 23.9, 17.5, 10.6),
    (100, 2304, 3072, 13.1, 14.6, 11.5), (100, 3072, 3072, 17.9, 14.8, 11.6),
    (160, 3072, 3072, 21.4, 19.5, 11.8), (32, 3333, 3072, 9.9, 8.5, 11.8),
    (72, 3333, 3072, 15.4, 15.4, 11.7), (100, 3333, 3072, 19.2, 20.2, 11.7),
    (25, 7168, 3072, 13.5, 11.8, 12.3), (25, 256, 3584, 7.5, 9.1, 12.6), (128, 900, 3584, 11.9, 10.1, 12.8),
    (72, 1536, 3840, 15.7, 16.5, 13.6), (100, 2304, 3840, 28.8, 21.9, 13.8),
    (160, 2304, 3840, 39.3, 22.3, 14.1), (16, 3072, 3840, 11.1, 12.4, 14.2),
    (32, 3072, 3840, 15.7, 12.4, 16.5), (100, 2304, 4096, 15.7, 17.9, 14.3),
    (128, 900, 5120, 14.1, 12.0, 16.8), (128, 3333, 5120, 30.3, 30.5, 17.9),
    (25, 256, 5632, 9.9, 12.3, 18.5), (128, 900, 5632, 15.5, 13.2, 18.5), (12, 5000, 5632, 14.0, 17.5, 19.6),
    (100, 2304, 5888, 40.5, 31.7, 19.9), (32, 3072, 5888, 21.8, 17.2, 23.8),
    (130, 3072, 5888, 61.4, 42.5, 20.2), (160, 3072, 5888, 73.0, 42.7, 21.1),
    (72, 3333, 5888, 47.9, 32.3, 20.1), (100, 3333, 5888, 58.6, 43.5, 20.3),
    (16, 10240, 5888, 32.7, 31.6, 21.2), (16, 16384, 5888, 40.8, 41.8, 22.4),
    (25, 256, 6144, 8.3, 12.7, 19.5), (17, 3333, 6144, 13.2, 13.0, 20.9), (12, 6144, 6144, 13.1, 18.2, 21.3),
    (17, 7680, 6144, 21.9, 18.6, 21.5), (128, 1536, 7168, 18.2, 21.2, 22.6),
    (32, 4096, 7168, 15.9, 15.2, 25.5), (32, 256, 7680, 12.4, 15.6, 25.1),
    (48, 2560, 7680, 17.7, 22.3, 25.1), (64, 2560, 7680, 26.6, 23.1, 26.8),
    (32, 7680, 7680, 33.5, 25.0, 29.6), (24, 512, 8192, 10.3, 16.1, 25.5),
    (24, 2048, 8192, 10.7, 16.3, 26.9), (64, 2048, 8192, 16.2, 16.6, 27.3),
    (33, 2304, 8192, 15.6, 22.2, 26.4), (33, 2560, 8192, 16.0, 22.6, 26.5),
    (32, 4608, 8192, 20.8, 24.3, 28.2), (17, 7168, 8192, 27.4, 23.2, 27.5),
    (25, 256, 10240, 11.7, 19.1, 30.7), (80, 1536, 10240, 18.6, 27.0, 32.0),
    (64, 3072, 10240, 25.0, 29.2, 32.9), (128, 4096, 10240, 60.9, 54.4, 32.7),
    (17, 7680, 10240, 33.1, 27.7, 33.4), (25, 256, 11776, 17.4, 21.9, 34.6),
    (48, 2560, 11776, 24.7, 31.6, 36.2), (128, 4096, 11776, 85.5, 62.0, 37.7),
    (17, 5000, 11776, 37.8, 31.3, 37.1), (48, 5000, 11776, 50.2, 46.7, 37.0),
    (32, 7680, 11776, 47.1, 35.0, 43.4), (48, 7680, 11776, 68.3, 61.1, 37.9),
    (64, 1024, 16128, 37.3, 40.6, 54.1), (64, 1536, 16128, 53.2, 41.1, 55.0),
    (130, 2048, 16128, 119.3, 80.4, 48.8), (100, 2304, 16128, 98.7, 80.2, 48.9),
    (100, 3072, 16128, 142.9, 81.5, 49.4), (130, 3072, 16128, 156.5, 108.6, 49.4),
    (160, 3072, 16128, 188.7, 109.8, 52.0), (100, 3333, 16128, 147.6, 110.3, 49.7),
    (25, 768, 16384, 17.2, 28.7, 51.0), (33, 1536, 16384, 26.1, 29.3, 49.4),
    (72, 1536, 16384, 26.5, 40.3, 49.3), (64, 3072, 16384, 36.9, 43.4, 53.0),
    (17, 7168, 16384, 49.6, 41.6, 52.2),
)

# m, rows, k, then microseconds: 8-row and 16-row items of the class-split kernel.
ROW_TIMES = (
    (16, 2048, 8192, 10.1, 10.4), (16, 2064, 8192, 15.4, 10.3), (16, 2064, 8448, 39.7, 20.7),
    (16, 2304, 16384, 27.6, 17.4), (16, 3072, 8192, 16.1, 10.5), (16, 4000, 11776, 34.1, 18.3),
    (16, 4096, 8192, 16.2, 10.7),
)

# m, rows, k, then microseconds: row-split and whole-prompt kernel, matrices of many rows.
MANY_ROWS_TIMES = (
    (16, 8200, 2048, 7.1, 9.3), (17, 8200, 2048, 9.6, 9.4), (24, 16384, 2048, 10.3, 10.1), (16, 32000, 2048, 13.6, 14.4),
    (17, 32000, 2048, 18.6, 14.4), (17, 128256, 2048, 73.4, 51.5), (32, 8192, 8192, 27.2, 29.1), (32, 9216, 4096, 15.7, 16.6), (28, 12288, 8192, 27.8, 29.4),
    (17, 16384, 8192, 28.5, 30.5), (32, 16384, 4096, 16.6, 17.5), (32, 16384, 16384, 52.4, 59.0),
    (32, 28672, 8192, 53.8, 41.8), (17, 28672, 4096, 30.3, 24.7), (33, 16384, 8192, 41.8, 39.3),
)


def _covers(m, rows, tokens):
    return -(-(-(-rows // 16) * -(-m // tokens)) // CUS)


# Where the choice of items matters: more than 16 tokens, and not so many, or rows so
# short, that the whole-prompt kernel is far ahead of both.
SPLIT_TIMES = [t for t in TIMES if t[0] > 16 and t[2] > 256 and _covers(t[0], t[1], 32) <= 2]


@pytest.fixture(scope="module")
def routes(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("gemm_route") / "gemm_route_sim")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Wextra", "-Werror",
                    "-I", os.path.join(ROOT, "llm-kv260_amd", "csrc"),
                    os.path.join(ROOT, "tests", "gemm_route_sim.cpp"), "-o", exe], check=True)

    def run(sizes):
        text = "".join(f"{m} {rows} {k} {CUS}\n" for m, rows, k in sizes)
        out = subprocess.run([exe], input=text, capture_output=True, text=True, check=True, timeout=60).stdout
        # Per size: the class-split kernel's tokens and rows per item, and the form taken.
        return [(int(t[5:]), int(r[4:]), f) for t, r, f in (line.split() for line in out.splitlines())]
    return run


def _slow(times, chosen, forms=3):
    """The sizes at which the chosen form (an index into a row's times) is over 6% off the best of the first `forms`."""
    return [(t[:3], c) for t, c in zip(times, chosen) if t[3 + c] > 1.06 * min(t[3:3 + forms])]


def _index(tokens, form="split"):
    return 2 if form == "tiles" else int(tokens == 32)


def test_items_of_the_class_split_kernel(routes):
    got = routes([t[:3] for t in SPLIT_TIMES])
    assert not _slow(SPLIT_TIMES, [_index(tokens) for tokens, _, _ in got], 2)


def test_form_taken(routes):
    got = routes([t[:3] for t in TIMES])
    assert not _slow(TIMES, [_index(tokens, form) for tokens, _, form in got])


def test_line_in_rows_times_tokens_is_caught(routes):
    got = routes([t[:3] for t in TIMES])
    line = [2 if t[0] * t[1] >= (45000 if t[2] % 512 else 220000 - 42600000 // t[2]) else _index(tokens)
            for t, (tokens, _, _) in zip(TIMES, got)]
    assert len(_slow(TIMES, line)) > len(TIMES) // 10


def test_items_by_their_number_alone_are_caught():
    by_number = [int(-(-t[1] // 16) * -(-t[0] // 32) >= 160) for t in SPLIT_TIMES]
    assert len(_slow(SPLIT_TIMES, by_number, 2)) > len(SPLIT_TIMES) // 10


def test_rows_of_an_item(routes):
    got = routes([t[:3] for t in ROW_TIMES])
    assert [rows for _, rows, _ in got] == [8 if t[3] < t[4] else 16 for t in ROW_TIMES]


def test_many_rows(routes):
    got = routes([t[:3] for t in MANY_ROWS_TIMES])
    assert [form for _, _, form in got] == ["rows" if t[3] < t[4] else "tiles" for t in MANY_ROWS_TIMES]
