"""The memory ranges that the matrix products' loads may touch (csrc/gemm_tiles.h, the arithmetic that
the kernel itself runs), walked tile by tile on the CPU: none leaves its operand, whatever edge a tile or
a quarter of one lies past and however few rows a last stage of K holds."""

import random
import shutil
import subprocess
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent


@pytest.fixture(scope="module")
def walker(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("needs a host C++ compiler")
    exe = tmp_path_factory.mktemp("gemm") / "gemm_ranges"
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", str(HERE / "gemm_ranges.cpp"), "-o", str(exe)], check=True)
    return exe


def _cases():
    # The d logits under d weight at one token past a stage, hidden sizes as its columns, and Muon's shapes.
    for vocab in (50257, 32003, 32000, 50304):
        for k in (1025, 65, 1, 1531):
            yield 1, vocab, 1024, k, ((vocab + 127) // 128 | 1) * 128
    for width in (576, 1600, 640, 768):
        for k in (1025, 64, 129):
            yield 1, width, 50257, k, width
    rng = random.Random(0)
    for _ in range(400):
        tr, mn, other = rng.randrange(2), rng.choice([1, 7, 8, 63, 65, 127, 129, 255, 257, 300, 513, 769]), rng.choice([8, 257, 600])
        k = rng.choice([0, 1, 2, 15, 16, 17, 63, 64, 65, 127, 129, 193, 257])
        cols = (mn if tr else k) + 7 & ~7
        yield tr, mn, other, k, max(cols, 8) + rng.choice([0, 0, 8, 64, 120])


def test_no_load_leaves_its_operand(walker):
    lines = "\n".join(" ".join(map(str, c)) for c in _cases())
    r = subprocess.run([str(walker)], input=lines, capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
    assert int(r.stdout.split()[0]) > 100000
