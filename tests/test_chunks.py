"""The chunks of the k-marching launches (tosca_amd/csrc/chunks.h, host code): the choice is the one of the rule
written out over every chunk count, and finding it does not take a time that grows with the planes (a caller
waits for it several times a step).  RULES and plane_chunk here tell the GPU tests which chunks a grid gets."""
import ctypes
import math
import re
import shutil
import subprocess
import time
from pathlib import Path

import numpy as np
import pytest

HEADER = Path(__file__).resolve().parents[1] / "tosca_amd" / "csrc" / "chunks.h"
NUM_CU = 256
RULES = {n: (int(a), int(b), float(d)) for n, a, b, d in
         re.findall(r"constexpr ChunkRule CHUNK_(\w+)\{(\d+), (\d+), ([\d.e]+)\};", HEADER.read_text())}


def plane_chunk(nk, tiles, rule):
    """planes per chunk of nk planes over `tiles` column tiles, every chunk count tried"""
    per_cu, over, drift = RULES[rule]
    c = np.arange(1, nk + 1)
    k = (nk + c - 1) // c
    n = (nk + k - 1) // k
    slots = per_cu * NUM_CU
    cost = ((tiles * n + slots - 1) // slots).astype(float) * (k + over) * (1.0 + k / drift)
    return int(k[np.argmin(cost)])                         # the first of the least


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    if not shutil.which("g++"):
        pytest.skip("g++ not available")
    d = tmp_path_factory.mktemp("chunks")
    (d / "c.cpp").write_text(f'#include "{HEADER}"\nextern "C" int pc(int nk, int tiles, int p, int o, double d) '
                             "{ return tosca::plane_chunk(nk, tiles, tosca::ChunkRule{p, o, d}); }\n")
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", str(d / "c.cpp"), "-o", str(d / "c.so")], check=True)
    so = ctypes.CDLL(str(d / "c.so"))
    so.pc.argtypes = [ctypes.c_int] * 4 + [ctypes.c_double]
    return so


def test_choice(lib):
    assert len(RULES) == 10
    for rule, (p, o, d) in RULES.items():
        for nk in [*range(1, 80), 95, 96, 97, 128, 191, 192, 193, 500, 513, 2000, 4001]:
            for tiles in (1, 2, 3, 4, 7, 12, 35, 63, 64, 65, 128, 255, 256, 257, 700, 1500):
                assert lib.pc(nk, tiles, p, o, d) == plane_chunk(nk, tiles, rule), (rule, nk, tiles)


def test_host_time(lib):
    """200000 planes: 1.3 ms a launch where every count is tried, about 0.01 ms over the distinct lengths."""
    p, o, d = RULES["FORMU"]
    best = math.inf
    for _ in range(20):
        t = time.perf_counter()
        lib.pc(200000, 1, p, o, d)
        best = min(best, time.perf_counter() - t)
    assert best < 2e-4, f"{best * 1e6:.0f} us"
