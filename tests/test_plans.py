"""Sizes the library's host code plans with, at the ends of their ranges (CPU:
tests/plan_host.cpp calls the planning functions, nothing runs on a GPU)."""
import os
import random
import shutil
import subprocess

import pytest

import lpma_amd as L

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "lpma_amd", "csrc")


@pytest.fixture(scope="module")
def plans(tmp_path_factory):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    L.lib()
    exe = str(tmp_path_factory.mktemp("plans") / "plan_host")
    r = subprocess.run([hipcc, "-x", "hip", "--offload-arch=gfx950", "-std=c++17", "-I" + CSRC, "-c",
                        os.path.join(HERE, "plan_host.cpp"), "-o", exe + ".o"], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([hipcc, "--offload-arch=gfx950", exe + ".o", L.LIB_PATH, "-o", exe,
                        "-Wl,-rpath," + os.path.dirname(L.LIB_PATH)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr

    def ask(lines):
        r = subprocess.run([exe], input="\n".join(lines) + "\n", capture_output=True, text=True)
        assert r.returncode == 0, r.stderr
        return [[int(x) for x in line.split()] for line in r.stdout.splitlines()]

    return ask


def pagerank_sizes():
    """(V, log2 of the segment's slots, height, edges): the largest graphs, the sparsest and random ones."""
    top = 1 << 32
    out = [(1 << 27, 5, 27, int(e)) for e in (1.7e9, 2.4e9, 3.35e9, 3.5e9, top - (1 << 27))]
    out += [(1 << 24, 5, 27, top - (1 << 24)), ((1 << 24) + 1, 5, 27, top - (1 << 24) - 1), (1 << 16, 5, 27, top - (1 << 16)),
            (1 << 22, 10, 22, top - (1 << 22)), (1 << 27, 5, 23, 0), (1 << 27, 5, 23, 1), (1, 1, 0, 0)]
    rng = random.Random(5)
    for _ in range(300):
        V, log2S = int(2 ** rng.uniform(0, 27)), rng.randint(1, 10)
        E = int(2 ** rng.uniform(0, 31.9))
        H = 0
        while H < 31 and (1 << (H + log2S)) < E + V:
            H += 1
        if E + V <= 1 << (H + log2S) <= top:
            out.append((V, log2S, H, E))
    return out


def test_pagerank_edge_words_stay_within_32_bits(plans):
    """Offsets of edge words are 32-bit sums on the device."""
    sizes = pagerank_sizes()
    for size, (words, room, bins, parts) in zip(sizes, plans(["pagerank %d %d %d %d" % s for s in sizes])):
        assert words < 1 << 32, (size, words, bins, parts)
        assert words >= size[3], (size, words)


def test_pagerank_edge_words_memory(plans):
    """An edge takes at most two words, itself and its share of the rows (8 B),
    and a ranking a group of words beyond that."""
    sizes = pagerank_sizes()
    for size, (words, room, bins, parts) in zip(sizes, plans(["pagerank %d %d %d %d" % s for s in sizes])):
        assert room <= 2 * size[3] + 64, (size, room, bins, parts)


def test_sort_scratch_grows_with_the_batch(plans):
    """lpma_reserve(n) sizes the scratch of every batch of up to n keys."""
    rng = random.Random(6)
    edges = [1 << 10, 1 << 12, 1 << 16, 1 << 17, 1 << 18, 1 << 19, 1 << 20, 1 << 22]
    ns = sorted({1, 2, 300} | {e + d for e in edges for d in (-1, 0, 1)} | {int(2 ** rng.uniform(0, 31)) for _ in range(500)})
    got = [w for w, in plans(["sort %d" % n for n in ns])]
    for (n, w), (n2, w2) in zip(zip(ns, got), list(zip(ns, got))[1:]):
        assert w <= w2, (n, w, n2, w2)
