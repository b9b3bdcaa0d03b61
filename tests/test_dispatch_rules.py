"""The rules on sizes that choose a launch (csahca_amd/csrc/dispatch.hpp), built
alone with the host compiler."""
import ctypes
import re
import subprocess
from pathlib import Path

import numpy as np
import pytest

CSRC = Path(__file__).resolve().parents[1] / "csahca_amd" / "csrc"
SHIM = r"""
#include "dispatch.hpp"
extern "C" {
int64_t split_tile(int64_t tile, int64_t total, int64_t bh, int64_t D, int64_t esz, int vec) {
  return csahca::csa_split_tile(tile, total, bh, D, esz, vec != 0);
}
int hybrid_one_read(int64_t esz, int64_t D, int64_t chunk, int64_t hca_chunk, int64_t items) {
  return csahca::csa_hybrid_one_read(esz, D, chunk, hca_chunk, items);
}
int select_topk_regs(int64_t C, int64_t k) { return csahca::csa_select_topk_regs(C, k); }
int step_topk_regs(int64_t C, int64_t k, int64_t bh, int fine) {
  return csahca::csa_step_topk_regs(C, k, bh, fine != 0);
}
}
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    (d / "shim.cpp").write_text(SHIM)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-O1", "-shared", "-fPIC", f"-I{CSRC}", "-o",
                    str(d / "rules.so"), str(d / "shim.cpp")], check=True)
    lib = ctypes.CDLL(str(d / "rules.so"))
    lib.split_tile.restype = ctypes.c_int64
    lib.split_tile.argtypes = [ctypes.c_int64] * 5 + [ctypes.c_int]
    lib.step_topk_regs.argtypes = [ctypes.c_int64] * 3 + [ctypes.c_int]
    lib.select_topk_regs.argtypes = [ctypes.c_int64] * 2
    lib.hybrid_one_read.argtypes = [ctypes.c_int64] * 5
    return lib


@pytest.mark.parametrize("tile,total,bh,D,esz,want", [
    (16, 3200, 8, 40, 2, 16),     # tiles of 64 took 1.43 times as long
    (32, 3200, 8, 96, 2, 32),     # 1.24
    (32, 3200, 256, 40, 2, 32),   # 1.16
    (64, 3200, 256, 96, 2, 64),   # 1.15
    (16, 800, 256, 96, 2, 16),    # 1.08
    (8, 1600, 8, 96, 2, 16),
    (8, 800, 8, 96, 2, 16),
    (4, 400, 32, 96, 2, 8),
    (4, 200, 8, 96, 2, 4),
    (1, 64, 1, 96, 2, 4),
    (3, 64, 1, 96, 2, 4),
    (5, 3200, 8, 96, 2, 16),
    (12, 3200, 8, 96, 2, 16),
    (8, 3200, 256, 96, 2, 32),    # 300 MiB of rows of 192 bytes
    (16, 800, 256, 192, 2, 16),
    (4, 256, 256, 192, 2, 8),
    (4, 3200, 256, 192, 2, 64),   # 600 MiB of rows of 384: no limit
    (4, 3200, 256, 320, 4, 100),  # rows of 1280
    (4, 6400, 32, 320, 4, 100),
    (64, 3200, 256, 192, 2, 64),
])
def test_generic_split_keeps_its_chain_short(rules, tile, total, bh, D, esz, want):
    assert rules.split_tile(tile, total, bh, D, esz, 0) == want


@pytest.mark.parametrize("tile,total,bh,D,esz,want", [
    (8, 512, 8, 128, 2, 16),      # a batch of row loads
    (8, 480, 48, 64, 2, 32),
    (8, 512, 16, 256, 4, 8),
    (8, 2048, 8, 128, 2, 32),     # 64 tiles a head
    (8, 1024, 64, 128, 2, 16),
    (5, 192, 6, 128, 2, 16),
    (64, 4352, 12, 128, 4, 72),   # a tile just below the line: twice it was 1.22 times as slow
    (80, 6000, 8, 64, 4, 96),     # 1.09
    (72, 4352, 12, 128, 4, 72),
    (200, 4352, 12, 128, 4, 200),
    (1, 16384, 1, 128, 2, 128),
    (8, 2048, 256, 128, 2, 64),   # 8192 wavefronts
])
def test_vectorised_split(rules, tile, total, bh, D, esz, want):
    assert rules.split_tile(tile, total, bh, D, esz, 1) == want


@pytest.mark.parametrize("vec", [0, 1])
def test_split_fits_the_callers_workspace(rules, vec):
    """Never more tiles than the caller's own tile makes, never an empty tile."""
    for tile in (1, 3, 5, 7, 8, 16, 33, 64, 128, 1000, 1 << 31):
        for total in (0, 1, 4, 17, 64, 100, 3200, 16384, 2**31 - 16384, 2**31 - 1):
            for bh in (1, 8, 256, 100000):
                for D, esz in ((64, 2), (128, 2), (256, 4)):
                    t = rules.split_tile(tile, total, bh, D, esz, vec)
                    assert 1 <= t <= max(total, 1)
                    assert t >= min(tile, max(total, 1))
                    assert -(-total // t) <= max(1, -(-total // tile))


@pytest.mark.parametrize("C,k,bh,fine,want", [
    (1, 1, 1, 1, 2), (64, 64, 8, 1, 2), (64, 64, 8, 0, 8), (64, 65, 1, 1, 0),
    (65, 63, 256, 1, 2), (65, 64, 8, 1, 0), (84, 44, 256, 1, 2), (84, 45, 8, 1, 0),
    (96, 43, 256, 0, 8), (96, 45, 16, 1, 2), (96, 44, 17, 1, 0), (128, 41, 256, 1, 2), (128, 44, 8, 1, 0),
    (132, 37, 48, 0, 8), (144, 39, 256, 1, 8), (144, 42, 8, 1, 0), (192, 37, 17, 1, 8), (192, 38, 17, 1, 0),
    (193, 36, 256, 1, 8), (193, 37, 17, 1, 0), (256, 38, 16, 1, 8), (256, 39, 8, 1, 0),
    (257, 34, 256, 1, 8), (512, 35, 17, 1, 0), (512, 36, 16, 0, 8), (512, 37, 8, 1, 0),
    (513, 32, 256, 1, 16), (513, 32, 256, 0, 32), (1024, 33, 17, 1, 0), (1024, 34, 16, 1, 16), (1024, 35, 8, 1, 0),
    (1025, 32, 256, 1, 32), (2048, 34, 8, 1, 32), (2048, 35, 8, 1, 0), (2049, 1, 1, 1, 0), (512, 100, 1, 1, 0),
])
def test_step_selection_takes_registers_where_they_rarely_fail(rules, C, k, bh, fine, want):
    """33-38 of more than 128 chunks, and 41-63 of up to 128 that cannot or hardly
    fail, went to all wavefronts, 5-10% slower a step than one wavefront's
    registers."""
    assert rules.step_topk_regs(C, k, bh, fine) == want


def test_step_selection_registers_cannot_fail_up_to_84_chunks(rules):
    """Lane L of 64 holds keys L, L + 64 (rotated); the threshold is the k-th
    largest lane maximum; 64 candidates fit."""
    rng = np.random.default_rng(0)
    for C in range(65, 85):
        k = max(k for k in range(1, 65) if rules.step_topk_regs(C, k, 256, 1))
        assert k == 128 - C
        keys = np.full((200, 128), -1)
        keys[:, :C] = rng.random((200, C)).argsort(-1)
        keys[:20, :C] = np.arange(C)         # the second row holds the largest
        keys[20:40, :C] = np.arange(C)[::-1]
        lanes = keys.reshape(200, 2, 64).max(1)
        t = np.sort(lanes, -1)[:, 64 - k]
        assert (keys >= t[:, None]).sum(-1).max() <= 64


def test_step_selection_registers_hold_every_key(rules):
    for C in range(1, 2049):
        for fine in (0, 1):
            m = rules.step_topk_regs(C, 8, 8, fine)
            assert m in ((2, 8, 16, 32) if fine else (8, 32)) and 64 * m >= C


@pytest.mark.parametrize("C,k,want", [
    (1, 1, 2), (64, 64, 2), (64, 65, 0), (65, 63, 2), (65, 64, 0), (84, 44, 2), (84, 45, 0), (96, 43, 2), (96, 44, 0),
    (128, 41, 2), (128, 42, 0), (129, 1, 4), (129, 39, 4), (192, 37, 4), (192, 38, 0), (193, 1, 0),
])
def test_selection_op_takes_registers_up_to_192_chunks(rules, C, k, want):
    """129-192 chunks, and 41-63 of 65-84, went to the workgroup's top-k, 2-7%
    slower a call."""
    assert rules.select_topk_regs(C, k) == want


@pytest.mark.parametrize("esz,D,chunk,hca_chunk,items,want", [
    (2, 64, 32, 128, 1, 1),         # 16 KiB an item
    (2, 64, 32, 256, 255, 0),       # 32 KiB, CSA chunks of one row group: 2-6% slower
    (2, 64, 32, 256, 256, 1),
    (2, 64, 64, 256, 1, 1),
    (2, 64, 32, 512, 511, 0),       # 64 KiB: 4-27% slower
    (2, 64, 64, 512, 127, 0),       # 7-9%
    (2, 64, 64, 512, 128, 1),
    (2, 64, 32, 1024, 511, 0),      # 128 KiB: 15-65%
    (2, 64, 64, 1024, 255, 0),
    (2, 64, 64, 1024, 256, 1),
    (2, 256, 16, 64, 1, 1),
    (2, 256, 32, 128, 255, 0),      # 1-10%
    (2, 256, 32, 128, 256, 1),
    (2, 256, 64, 128, 127, 0),
    (2, 256, 64, 128, 128, 1),
    (2, 256, 64, 256, 191, 0),
    (2, 256, 64, 256, 192, 1),
    (4, 64, 16, 128, 1, 1),
    (4, 64, 16, 256, 191, 0),       # 4-9%
    (4, 64, 32, 256, 1, 1),
    (4, 64, 32, 512, 127, 0),       # 12%
    (4, 64, 32, 512, 128, 1),
    (4, 64, 16, 512, 255, 0),
    (4, 128, 16, 128, 1, 1),
    (4, 256, 16, 64, 127, 0),
    (4, 256, 16, 64, 128, 1),
    (4, 256, 64, 256, 511, 0),      # more than 128 KiB
    (4, 256, 64, 256, 512, 1),
    (2, 128, 64, 64, 3071, 0),      # 16-bit head_dim 128, 16 KiB: from 48 MiB of K
    (2, 128, 64, 64, 3072, 1),
    (2, 128, 64, 256, 1023, 0),     # 64 KiB: from 64 MiB (3% slower at 48)
    (2, 128, 64, 256, 1024, 1),
    (2, 128, 16, 512, 639, 0),      # 128 KiB, one row group: 6% slower at 64
    (2, 128, 16, 512, 640, 1),
    (2, 128, 64, 2048, 511, 0),
])
def test_hybrid_reads_k_once_where_wavefronts_are_many(rules, esz, D, chunk, hca_chunk, items, want):
    assert rules.hybrid_one_read(esz, D, chunk, hca_chunk, items) == want


def test_the_step_kernels_traffic_record_covers_every_source():
    """bench.py reports profiles/traffic.json only for the sources it names; the
    rules' header picks the step's instantiation and was not among them."""
    bench = (CSRC.parents[1] / "bench.py").read_text()
    named = set(re.findall(r'"([^"]+)"', re.search(r"STEP_KERNEL_SOURCES = \(([^)]*)\)", bench).group(1)))
    seen, todo = set(), ["csa_step.hip"]
    while todo:
        name = todo.pop()
        if name not in seen and (CSRC / name).exists():
            seen.add(name)
            todo += re.findall(r'#include "([^"]+)"', (CSRC / name).read_text())
    assert named == seen
