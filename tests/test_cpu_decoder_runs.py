"""The run lengths of the recurrences (csrc/runs.h), which are host code without HIP: compiled here and asked for steps whose
best lengths were measured."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "multimodal-financial-analysis-tool-using-paligemma_amd", "csrc")
ASK = r"""
#include <cstdio>
#include <cstdlib>
#include <vector>
#include "runs.h"
int main(int n, char** v) {  // channels, states, lengths
    std::vector<int32_t> lens;
    for (int i = 3; i < n; ++i) lens.push_back(atoi(v[i]));
    const int C = atoi(v[1]), N = atoi(v[2]);
    std::printf("%d %d\n", pgmi::scan_run_rows(lens.data(), (int)lens.size(), pgmi::scan_columns(C, N), pgmi::scan_workgroups(C, N)),
                pgmi::gru_run_rows(lens.data(), (int)lens.size(), pgmi::gru_columns(C)));
}
"""


def compiled(tmp_path_factory, name, source):
    """The program, as a function of its arguments: the whole numbers of each line that it prints."""
    at = tmp_path_factory.mktemp(name)
    (at / "ask.cpp").write_text(source)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, str(at / "ask.cpp"), "-o", str(at / "ask")], check=True)
    return lambda *a: [[int(x) for x in line.split()] for line in subprocess.run([str(at / "ask"), *map(str, a)], check=True, capture_output=True,
                                                                                 text=True).stdout.splitlines()]


@pytest.fixture(scope="module")
def ask(tmp_path_factory):
    run = compiled(tmp_path_factory, "runs", ASK)
    return lambda *a: run(*a)[0]


# channels, states, lengths; the shortest and longest run length of those within 4 % of the best measured
@pytest.mark.parametrize("C,N,lens,least,most", [
    (2048, 16, [200], 16, 16), (2048, 16, [500], 16, 16), (2048, 16, [1000], 16, 32), (2048, 16, [4000], 32, 64),
    (4096, 16, [1024, 387, 129], 48, 64), (2048, 32, [500], 16, 16), (2048, 32, [1000], 16, 32), (2048, 32, [4000], 32, 64),
    (2048, 64, [500], 16, 32), (2048, 64, [1000], 16, 64), (2048, 64, [4000], 32, 64), (4096, 64, [1540], 32, 64),
    (2048, 128, [200], 16, 24), (2048, 128, [500], 16, 64), (2048, 128, [1540], 48, 64), (2048, 128, [4000], 32, 64),
    (2048, 256, [500], 60, 64), (2048, 256, [1000], 48, 64), (2048, 256, [1540], 48, 64), (2048, 256, [4000], 48, 64),
    (2048, 256, [500, 300, 100, 60], 56, 64),
    # sequences that are walked whole, and just no more
    (2048, 16, [17], 17, 64), (2048, 16, [32], 32, 64), (2048, 16, [40], 16, 64), (2048, 16, [48], 16, 16), (512, 16, [64] * 8, 16, 16),
    (4096, 16, [64] * 8, 64, 64), (2048, 64, [64] * 8, 64, 64), (2048, 64, [20] * 8, 20, 64), (4096, 16, [40] * 32, 40, 64), (2048, 16, [1], 1, 64)])
def test_scan(ask, C, N, lens, least, most):
    assert least <= ask(C, N, *lens)[0] <= most


@pytest.mark.parametrize("C,lens,rows", [(2048, [1024], 32), (2048, [500], 32), (2048, [370], 24), (2048, [300], 16), (2048, [100], 8), (2048, [41], 8), (2048, [40], 40), (1024, [40] * 32, 40), (300, [17, 3], 17), (128, [9000], 32),
                                         (128, [7000], 32), (64, [2000], 24), (64, [700], 16),
                                         (64, [300], 8), (128, [100, 3], 8)])
def test_gru(ask, C, lens, rows):
    assert ask(C, 16, *lens)[1] == rows


# the steps of test_gpu_decoder_runs.py, whose layers are all a workgroup wide
@pytest.mark.parametrize("n,length,scan,gru", [(36, 450, 32, 32), (30, 400, 50, 32), (20, 450, 36, 32), (3, 97, 16, 8), (36, 448, 64, 32),
                                               (16, 450, 30, 24), (12, 450, 22, 16), (10, 450, 18, 16)])
@pytest.mark.parametrize("C,N", [(72, 12), (40, 9), (128, 16)])
def test_steps_of_many_sequences(ask, C, N, n, length, scan, gru):
    assert ask(C, N, *(length - 7 * (r % 5) for r in range(n))) == [scan, gru]


WALKS = r"""
#include <cstdio>
#include <cstdlib>
#include <vector>
#include "runs.h"
int main(int n, char** v) {  // channels, states, lengths
    std::vector<int32_t> lens;
    for (int i = 3; i < n; ++i) lens.push_back(atoi(v[i]));
    const int C = atoi(v[1]), N = atoi(v[2]), k = (int)lens.size();
    const int run = pgmi::scan_run_rows(lens.data(), k, pgmi::scan_columns(C, N), pgmi::scan_workgroups(C, N));
    const pgmi::ScanStep s = pgmi::scan_step_of(lens.data(), k, run);
    std::printf("%d %d\n", (int)pgmi::scan_walks(s, C, N, false), (int)pgmi::scan_walks(s, C, N, true));
}
"""


@pytest.fixture(scope="module")
def walks(tmp_path_factory):
    run = compiled(tmp_path_factory, "walks", WALKS)
    return lambda *a: run(*a)[0]


# whole sequences with a lane per state (bf16, fp32) where that was the faster form by more than the rule's error
@pytest.mark.parametrize("C,N,lens,bf16,f32", [
    (4096, 16, [1024, 387, 129], 1, 1), (4096, 16, [1540], 1, 1), (4096, 16, [512] * 8, 1, 1), (4096, 16, [4096], 1, 1),
    (2048, 16, [500], 1, 1), (2048, 16, [1000], 1, 1), (2048, 16, [4096], 0, 0), (1024, 16, [3000], 0, 0), (512, 16, [700], 1, 1),
    (64, 16, [1500], 0, 0), (64, 16, [300], 1, 1), (4096, 16, [33] * 64, 0, 0), (8192, 16, [64] * 32, 0, 0), (1024, 16, [64] * 32, 1, 1),
    (1000, 12, [1000], 0, 0), (520, 10, [1000], 0, 0), (264, 16, [1000] * 2, 0, 0), (1000, 12, [300], 1, 1), (4096, 9, [1000], 1, 1),
    (72, 12, [70, 33, 5], 1, 1), (72, 8, [70, 33, 5], 0, 0), (72, 17, [70, 33, 5], 0, 0), (2048, 64, [500], 0, 0), (64, 9, [1], 1, 1)])
def test_scan_walks(walks, C, N, lens, bf16, f32):
    assert walks(C, N, *lens) == [bf16, f32]


GRU_WALKS = r"""
#include <cstdio>
#include <cstdlib>
#include <vector>
#include "runs.h"
int main(int n, char** v) {  // channels, lengths
    std::vector<int32_t> lens;
    for (int i = 2; i < n; ++i) lens.push_back(atoi(v[i]));
    const int C = atoi(v[1]), k = (int)lens.size();
    const pgmi::ScanStep s = pgmi::scan_step_of(lens.data(), k, pgmi::gru_run_rows(lens.data(), k, (C + 127) / 128));
    std::printf("%d %d\n", (int)pgmi::gru_walks(s, C, false), (int)pgmi::gru_walks(s, C, true));
}
"""


@pytest.fixture(scope="module")
def gru_walks(tmp_path_factory):
    run = compiled(tmp_path_factory, "gru_walks", GRU_WALKS)
    return lambda *a: run(*a)[0]


# minGRU's sequences walked whole (bf16, fp32) where that was the faster form by more than the rule's error
@pytest.mark.parametrize("C,lens,bf16,f32", [
    (2048, [1024, 387, 129], 1, 1), (1024, [500], 1, 1), (2048, [60], 1, 1), (4096, [1000], 1, 1), (2048, [1000] * 4, 1, 1),
    (1024, [512] * 8, 1, 1), (256, [64] * 32, 1, 1), (44, [300], 1, 1), (1024, [33] * 64, 0, 0), (4096, [33] * 64, 0, 0),
    (4096, [64] * 32, 0, 0), (300, [2000], 0, 0), (4088, [1000], 1, 1), (64, [4096], 0, 0), (256, [4096], 0, 0), (44, [2000], 0, 0)])
def test_gru_walks(gru_walks, C, lens, bf16, f32):
    assert gru_walks(C, *lens) == [bf16, f32]


TILES = r"""
#include <cstdio>
#include <cstdlib>
#include "runs.h"
int main(int n, char** v) {  // heads per key/value head, starts and lengths in turn
    std::vector<int32_t> starts, lens;
    for (int i = 2; i < n; i += 2) {
        starts.push_back(atoi(v[i]));
        lens.push_back(atoi(v[i + 1]));
    }
    for (const pgmi::AttnTile& t : pgmi::attn_tiles(starts.data(), lens.data(), (int)lens.size(), atoi(v[1]), 64)) std::printf("%d %d\n", t.seq, t.first);
}
"""


@pytest.fixture(scope="module")
def attn_tiles(tmp_path_factory):
    run = compiled(tmp_path_factory, "attn_tiles", TILES)
    return lambda *a: [tuple(line) for line in run(*a)]


@pytest.mark.parametrize("R", [1, 3, 8])
@pytest.mark.parametrize("seqs", [[(0, 500)], [(7, 1)], [(0, 1024), (0, 387), (0, 129)], [(900, 63), (0, 64), (64, 65), (63, 1), (5, 900)],
                                  [(2147480000, 640), (0, 640)]])
def test_attn_tiles(attn_tiles, R, seqs):
    """Every tile once, in the order of the 64 keys its last position falls in."""
    got = attn_tiles(R, *(x for s in seqs for x in s))
    assert sorted(got) == [(r, f) for r, (_, n) in enumerate(seqs) for f in range(0, n * R, 64)]
    end = [(seqs[r][0] + (min(f + 64, seqs[r][1] * R) - 1) // R) // 64 for r, f in got]
    assert end == sorted(end)


TEAMS = r"""
#include <cstdio>
#include <cstdlib>
#include "runs.h"
int main(int n, char** v) {  // heads, key/value heads, width, window, kept, starts and lengths in turn
    std::vector<int32_t> starts, lens;
    for (int i = 6; i < n; i += 2) {
        starts.push_back(atoi(v[i]));
        lens.push_back(atoi(v[i + 1]));
    }
    std::printf("%d\n", (int)pgmi::wattn_teams(starts.data(), lens.data(), (int)lens.size(), atoi(v[1]), atoi(v[2]), atoi(v[3]), atoi(v[3]), atoi(v[4]),
                                               atoi(v[5])));
}
"""


@pytest.fixture(scope="module")
def teams(tmp_path_factory):
    return compiled(tmp_path_factory, "teams", TEAMS)


# steps whose better form was measured to be so by more than the rule's error
@pytest.mark.parametrize("H,G,d,window,keep,lens,two", [
    (16, 2, 128, 1024, 0, [1024, 387, 129], 1), (16, 2, 128, 1024, 0, [500], 1), (16, 2, 128, 1024, 16, [600, 500], 1),
    (8, 2, 128, 1024, 0, [2048], 1), (16, 2, 64, 1024, 0, [1000] * 2, 1), (16, 2, 256, 1024, 0, [500], 1), (8, 8, 256, 1024, 0, [400] * 3, 1),
    (8, 2, 128, 1024, 0, [1411, 700, 510, 256, 90], 1),
    (16, 2, 128, 1024, 0, [300] * 4, 0), (32, 8, 128, 1024, 0, [130] * 4, 0), (16, 2, 128, 256, 0, [600, 500], 0), (16, 2, 128, 1024, 0, [512] * 8, 0),
    (16, 2, 128, 1024, 0, [4096], 0), (16, 2, 256, 1024, 0, [300] * 4, 0), (16, 2, 128, 256, 0, [1540], 0), (32, 8, 128, 1024, 0, [1024, 387, 129], 0),
    (16, 2, 64, 1024, 0, [512] * 8, 0), (16, 2, 128, 1024, 0, [60], 0)])
def test_teams(teams, H, G, d, window, keep, lens, two):
    assert teams(H, G, d, window, keep, *(x for n in lens for x in (0, n))) == [[two]]


def test_teams_of_huge_steps(teams):
    assert teams(8, 1, 128, 2147483647, 2147483647, 2147480000, 640) in ([[0]], [[1]])
