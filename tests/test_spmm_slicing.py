"""How products deal their feature columns out over work-groups, compiled by the host compiler: every column has its lane group, the launch
stays within the 2^32 work-items of a dimension, and fewer slices are taken only where it would not."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PROGRAM = r"""
#include <cstdio>
#include "spmm_slices.h"
int main()
{
    long long waves;
    int K, n_cols, lines;
    while (scanf("%d %d %d %lld", &K, &n_cols, &lines, &waves) == 4) {
        const drone::Slicing s = drone::slicing(K, n_cols, lines, waves, (waves + 3) / 4, 256);
        printf("%d %d\n", s.lanes, s.bits);
    }
}
"""


@pytest.fixture(scope="module")
def slicing(tmp_path_factory):
    where = tmp_path_factory.mktemp("slicing")
    (where / "slicing.cpp").write_text(PROGRAM)
    subprocess.check_call(["g++", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "drone_amd", "csrc"), "slicing.cpp", "-o", "slicing"], cwd=where)

    def call(cases):
        text = "".join("%d %d %d %d\n" % c for c in cases)
        out = subprocess.run([str(where / "slicing")], input=text, capture_output=True, text=True, check=True).stdout
        return [tuple(map(int, line.split())) for line in out.splitlines()]

    return call


def _items(waves, bits):
    return (waves + 3) // 4 * 256 << bits


def test_launches_stay_within_a_dimension(slicing):
    # waves: 17 M vertices of some 40 entries (a chunk each), the limits of two and four slices, the most chunks of 2^31 entries
    waves = [1, 4096, 8193, 3_000_000, 16_777_212, 16_777_213, 17_000_000, 33_554_428, 33_554_429, 66_076_419]
    cases = [(K, n_cols, lines, w) for K in (4, 16, 112, 127, 128, 239, 240, 256, 300) for n_cols in (1000, 90_001, 17_000_000)
             for lines in (0, 1) for w in waves]
    for (K, n_cols, lines, w), (lanes, bits) in zip(cases, slicing(cases)):
        assert _items(w, bits) < 2 ** 32, (K, n_cols, lines, w, lanes, bits)
        assert lanes in (4, 8, 16, 32, 64) and 1 <= 1 << bits <= 16
        assert (lanes * 4 << bits) >= min(K, 256)  # (wider products go round)


@pytest.mark.parametrize("K,most", [(112, 1), (128, 1), (240, 2), (256, 2)])
def test_fewer_slices_only_where_they_do_not_fit(slicing, K, most):
    waves = [100_000, 16_000_000, 16_777_212, 16_777_213, 33_554_428, 33_554_429, 60_000_000]
    for w, (lanes, bits) in zip(waves, slicing([(K, 17_000_000, 1, w) for w in waves])):
        assert bits == max(b for b in range(most + 1) if _items(w, b) < 2 ** 32)
        assert lanes == 16 << (most - bits)


def test_small_products(slicing):
    assert slicing([(128, 2708, 1, 1000), (128, 2708, 1, 4096), (128, 2708, 1, 4097), (7, 2708, 1, 10), (300, 401, 0, 301)]) == \
        [(4, 3), (16, 1), (32, 0), (4, 0), (4, 4)]
