"""The march length of HLLD's accumulating passes (csrc/march.hpp, compiled
here for the host): the same choice as trying every number of chunks, at a
cost that does not grow with the line."""
import ctypes
import os
import random
import subprocess
import time

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def march(tmp_path_factory):
    d = tmp_path_factory.mktemp("march")
    src, lib = d / "march.cpp", d / "march.so"
    src.write_text('#include "march.hpp"\nextern "C" int cells(unsigned b, int nd, int r, int m)\n'
                   '{ return pamhd_dev::march_cells(b, nd, r, m); }\n')
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-I",
                    os.path.join(ROOT, "pamhd_amd", "csrc"), "-o", str(lib), str(src)], check=True)
    f = ctypes.CDLL(str(lib)).cells
    f.argtypes = [ctypes.c_uint, ctypes.c_int, ctypes.c_int, ctypes.c_int]
    return f


def _exhaustive(blocks, nd, resident, most):
    best, best_cost = 1, 1e300
    for chunks in range(1, nd + 1):
        km = -(-nd // chunks)
        if km > most:
            continue
        cost = float(-(-blocks * chunks // (256 * resident))) * (km + 1.5)
        if cost < best_cost:
            best, best_cost = km, cost
    return best


def test_choice_of_every_chunk_count(march):
    rng = random.Random(4)
    for _ in range(400):
        args = (int(2 ** rng.uniform(0, 20)), int(2 ** rng.uniform(0, 11)), rng.choice((2, 3)),
                rng.choice((1, 2, 8, 31, 32)))
        assert march(*args) == _exhaustive(*args), args


def test_cost_on_long_lines(march):
    """a loop over the chunk counts takes 0.05 s a call on a line of 2^24 cells"""
    t = time.perf_counter()
    for k in range(100):
        assert 1 <= march(8 + k, 1 << 24, 3, 32) <= 32
    assert time.perf_counter() - t < 0.5
