"""The strip kernel's band count (csrc/strip_bands.hpp), compiled for the
host: the count that trying every one finds, block sums within the partial
buffer, and no search whose length grows with the mesh (it runs on every
launch)."""
import ctypes
import os
import random
import shutil
import subprocess
import time

import pytest

from conftest import PKG

MAX_SUMS = 4096


@pytest.fixture(scope="module")
def bands(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("no host compiler")
    d = tmp_path_factory.mktemp("bands")
    src, so = d / "b.cpp", d / "b.so"
    src.write_text('#include "strip_bands.hpp"\n'
                   'extern "C" int bands(long s, int y, long r, long m) { return sipg_internal::strip_bands(s, y, r, m); }\n')
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I" + os.path.join(PKG, "csrc"), "-o", str(so),
                    str(src)], check=True)
    f = ctypes.CDLL(str(so)).bands
    f.argtypes = [ctypes.c_long, ctypes.c_int, ctypes.c_long, ctypes.c_long]
    return f


def _every(nstrip, dimy, res):
    best, cost = 1, None
    for nb in range(1, (dimy + 3) // 4 + 1):
        if nb > 1 and nstrip * nb > MAX_SUMS:
            break
        rows = (-(-dimy // nb) + 3) // 4
        c = -(-nstrip * nb // res) * (4 * rows + 5)
        if cost is None or c < cost:
            best, cost = nb, c
    return best


def test_equals_trying_every_count(bands):
    rng = random.Random(5)
    cases = [(1, 1, 256), (1, 4096, 2048), (119, 5145, 1280), (4097, 9, 512), (5000, 100, 256), (4096, 8, 256),
             (2048, 64, 1024)]
    cases += [(int(4500 ** rng.random()), int(9000 ** rng.random()), 256 * rng.randint(1, 8)) for _ in range(2000)]
    bad = [c for c in cases if bands(*c, MAX_SUMS) != _every(*c)]
    assert not bad, (len(bad), bad[:5])


def test_block_sums_stay_within_the_partial_buffer(bands):
    # 355 x 5145 elements in strips of three, 1280 resident workgroups: 43
    # bands would be 5,117 block sums, which the solvers fold in an extra launch
    rng = random.Random(6)
    for nstrip, dimy, res in [(119, 5145, 1280)] + [(int(4500 ** rng.random()), int(70000 ** rng.random()),
                                                     256 * rng.randint(1, 8)) for _ in range(2000)]:
        nb = bands(nstrip, dimy, res, MAX_SUMS)
        assert 1 <= nb <= max(1, (dimy + 3) // 4)
        assert nb == 1 or nstrip * nb <= MAX_SUMS, (nstrip, dimy, res)


def test_the_search_does_not_grow_with_the_mesh(bands):
    # trying every count: 16,384 of them; a call through ctypes takes about 1 us
    best = 1e9
    for _ in range(20):
        t = time.perf_counter()
        for _ in range(50):
            bands(1, 65536, 1024, MAX_SUMS)
        best = min(best, (time.perf_counter() - t) / 50)
    assert best < 6e-6, best
