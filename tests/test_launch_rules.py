"""CPU checks of the launch rules in csrc/launch_rules.hpp, compiled for the host: the kernels'
index arithmetic walked over sizes that no test allocates."""
import ctypes
import math
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = """
#include "launch_rules.hpp"
extern "C" uint32_t chain_grid(uint64_t chunks, uint64_t C, int vec, int* lane_cols) {
    const icx::ChainGrid g = icx::chain_grid(chunks, C, vec);
    *lane_cols = g.lane_cols;
    return g.blocks;
}
extern "C" int layer_norm_rows(uint64_t rows, uint64_t cols, uint64_t cus) { return icx::layer_norm_rows(rows, cols, cus); }
extern "C" uint32_t chain_in_flight(int vec) { return icx::chain_in_flight(vec); }
"""
THREADS = 256


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    (d / "rules.cpp").write_text(SOURCE)
    so = str(d / "rules.so")
    subprocess.check_call(["g++", "-std=c++17", "-shared", "-fPIC", "-Wall", "-Werror",
                           "-I", os.path.join(ROOT, "iconnx_amd", "csrc"), str(d / "rules.cpp"), "-o", so])
    lib = ctypes.CDLL(so)
    lib.chain_grid.argtypes = [ctypes.c_uint64, ctypes.c_uint64, ctypes.c_int, ctypes.c_void_p]
    lib.chain_grid.restype = lib.chain_in_flight.restype = ctypes.c_uint32
    lib.layer_norm_rows.argtypes = [ctypes.c_uint64] * 3
    return lib


def chain_grid(rules, chunks, C, vec=1):
    lane = ctypes.c_int()
    blocks = rules.chain_grid(chunks, C, vec, ctypes.byref(lane))
    return blocks, bool(lane.value)


# widths about the factors of the block size, past 2^21, 2^23 and 2^24 (where a grid of whole
# rows wraps the index or passes the threads of a launch) and 2^29
WIDTHS = [1, 2, 3, 64, 205, 256, 1023, 1024, 1025, 2047, 2049, 4095, 16383, 16385, 30522, 99999, 262144, 1000003, 2096131, 2097151,
          2097152, 2097153, 2097155, 8388609, 16777215, 16777217, 1 << 29, (1 << 31) - 1]


@pytest.mark.parametrize("C", WIDTHS)
def test_chain_grid_index_does_not_wrap(rules, C):
    for vec in (1, 4):
        most = ((1 << 31) - 1) // (vec * C)  # rows of 32-bit indices
        for rows in {r for r in (1, 3, 20, 1000, 70000, most) if 0 < r <= most}:
            chunks = rows * C
            blocks, lane_cols = chain_grid(rules, chunks, C, vec)
            stride = blocks * THREADS
            step = rules.chain_in_flight(vec) * stride
            assert 1 <= blocks <= -(-chunks // THREADS)  # no block without a chunk
            assert chunks - 1 + step < 1 << 32  # b += step, computed in 32 bits, passes the end
            if lane_cols:  # every chunk of a lane has the lane's first column
                assert stride >= chunks or stride % C == 0


@pytest.mark.parametrize("chunks,C", [(300 * 1025, 1025), (150 * 2047, 2047), (900 * 2049, 2049), (5 * 99999, 99999),
                                      (3000 * 456, 456), (1000003, 1000003)])
def test_chain_grid_covers_every_chunk_once(rules, chunks, C):
    blocks, lane_cols = chain_grid(rules, chunks, C)
    U = rules.chain_in_flight(1)
    lanes = np.arange(blocks * THREADS, dtype=np.uint32)
    seen = np.zeros(chunks, np.int64)
    b = lanes[lanes < chunks]
    for _ in range(math.ceil(chunks / (U * len(lanes))) + 1):
        for u in range(U):
            j = b.astype(np.int64) + u * len(lanes)
            j, first = j[j < chunks], (b % C)[j < chunks]
            seen[j] += 1
            if lane_cols:
                assert np.array_equal(j % C, first)
        b = b + np.uint32(U * len(lanes))
        b = b[b < chunks]
    assert len(b) == 0 and (seen == 1).all()


# up to the rows that fill 288 GB in place, and to those that 32 rows a block can launch
@pytest.mark.parametrize("cols", [1, 4, 100, 128, 129, 384, 1023, 1025, 2048, 2049, 4096, 12288, 12289, 100000])
def test_layer_norm_blocks_fit_a_launch(rules, cols):
    for rows in (1, 2, 511, 512, 513, 100000, (1 << 24) - 1, 1 << 24, (1 << 24) + 1, 1 << 26, (72 << 30) // cols):
        rows = min(rows, 32 * ((1 << 24) - 1))
        rpb = rules.layer_norm_rows(rows, cols, 256)
        blocks = -(-rows // (rpb or 32))
        assert blocks * 256 < 1 << 32
        if rpb:
            assert rpb in (1, 2, 4, 8, 16, 32) and rpb * (-(-cols // 16) * 16 + 8 + 2) * 4 <= 65536  # LDS
        else:  # only where the staging kernel cannot
            assert cols > 12288 or -(-rows // (rpb or max(1, 4096 // cols))) >= 1 << 24
