"""Host half of the locality ordering (csrc/locality_chain.h), compiled by itself with the address sanitizer: whatever
the pivots' rows hold, every pivot gets a place of its own and every point a number of its own."""
import os
import shutil
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include "locality_chain.h"

// chain M D N < rows (M x D floats), labels (N ints) > places (M ints), order (N ints)
int main(int, char **argv) {
    const int M = std::atoi(argv[1]), D = std::atoi(argv[2]), N = std::atoi(argv[3]);
    std::vector<float> rows((size_t)M * D);
    std::vector<int> labels(N), order(N);
    if (std::fread(rows.data(), sizeof(float), rows.size(), stdin) != rows.size()) return 2;
    if (std::fread(labels.data(), sizeof(int), labels.size(), stdin) != labels.size()) return 2;
    const std::vector<int> place = tsnehip::chain_pivots(rows.data(), M, D);
    const bool all_near = tsnehip::order_by_place(labels.data(), N, place, order.data());
    if (all_near != (*std::min_element(labels.begin(), labels.end()) >= 0)) return 3;
    std::fwrite(place.data(), sizeof(int), place.size(), stdout);
    std::fwrite(order.data(), sizeof(int), order.size(), stdout);
    return 0;
}
"""


@pytest.fixture(scope="module")
def chain(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("no host compiler")
    folder = tmp_path_factory.mktemp("chain")
    source, program = folder / "chain.cpp", folder / "chain"
    source.write_text("#include <algorithm>\n#include <cstdlib>\n" + PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=address", "-static-libasan", "-D_GLIBCXX_ASSERTIONS", "-I",
                    os.path.join(ROOT, "tsne-cuda_amd", "csrc"), str(source), "-o", str(program)], check=True)

    def run(rows, labels):
        m, d = rows.shape
        env = {k: v for k, v in os.environ.items() if k != "LD_PRELOAD"}
        done = subprocess.run([str(program), str(m), str(d), str(len(labels))], env=env, capture_output=True,
                              input=rows.astype(np.float32).tobytes() + labels.astype(np.int32).tobytes())
        assert done.returncode == 0, done.stderr.decode()[-2000:]
        out = np.frombuffer(done.stdout, np.int32)
        return out[:m], out[m:]

    return run


def greedy(rows):
    """The chain in numpy: nearest pivot not yet placed, the first of them where no distance is finite."""
    m = len(rows)
    place = np.full(m, -1)
    cur = 0
    with np.errstate(all="ignore"):
        for pos in range(m):
            place[cur] = pos
            left = np.flatnonzero(place < 0)
            if left.size == 0:
                break
            d2 = ((rows[left].astype(np.float64) - rows[cur].astype(np.float64)) ** 2).sum(1)
            finite = np.isfinite(d2)
            cur = left[np.argmin(np.where(finite, d2, np.inf))] if finite.any() else left[0]
    return place


@pytest.mark.parametrize("bad", [[], [0], [63], [0, 1, 5], list(range(64))])
@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf])
def test_every_pivot_and_every_point_has_a_place(chain, bad, value):
    rng = np.random.default_rng(len(bad))
    rows = rng.standard_normal((64, 5)).astype(np.float32)
    rows[bad, 2] = value
    labels = rng.integers(0, 64, size=1000)
    place, order = chain(rows, labels)
    assert np.array_equal(place, greedy(rows))
    assert np.array_equal(np.sort(place), np.arange(64))
    assert np.array_equal(order, np.argsort(place[labels], kind="stable"))
    labels[[17, 999]] = -1  # points at no finite distance from a pivot go with pivot 0
    place, order = chain(rows, labels)
    assert np.array_equal(order, np.argsort(place[np.maximum(labels, 0)], kind="stable"))
