"""Every output tile belongs to exactly one workgroup of the grid, and no XCD (workgroup id modulo 8) has much more than its share:
the numbering shared by the prefill kernels, compiled for the host."""
import ctypes
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#define __device__
#define __forceinline__ inline
#include <algorithm>
using std::min;
#include "abq_tile_numbering.h"
extern "C" int tile(int id, int m_blocks, int n_blocks, int *mb, int *nb) { return abq::tile_of_workgroup(id, m_blocks, abq::tile_columns(m_blocks, n_blocks), mb, nb) && *nb < n_blocks; }
extern "C" unsigned grid(int m_blocks, int n_blocks) { return abq::tile_grid(m_blocks, n_blocks); }
"""


@pytest.fixture(scope="module")
def numbering(tmp_path_factory):
    d = tmp_path_factory.mktemp("numbering")
    src, lib = d / "numbering.cpp", d / "numbering.so"
    src.write_text(SOURCE)
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-I", os.path.join(ROOT, "abq-llm_amd", "csrc"), "-o", str(lib), str(src)])
    return ctypes.CDLL(str(lib))


@pytest.mark.parametrize("m_blocks", [1, 2, 3, 4, 5, 7, 8, 13, 128, 203])
@pytest.mark.parametrize("n_blocks", [1, 2, 7, 8, 9, 15, 16, 33, 86, 172])
def test_every_tile_once_and_evenly(numbering, m_blocks, n_blocks):
    seen, per_xcd = set(), [0] * 8
    for i in range(numbering.grid(m_blocks, n_blocks)):
        mb, nb = ctypes.c_int(), ctypes.c_int()
        if numbering.tile(i, m_blocks, n_blocks, ctypes.byref(mb), ctypes.byref(nb)):
            assert 0 <= mb.value < m_blocks and 0 <= nb.value < n_blocks
            assert (mb.value, nb.value) not in seen
            seen.add((mb.value, nb.value))
            per_xcd[i % 8] += 1
    assert len(seen) == m_blocks * n_blocks
    # no XCD has a round of its 32 compute units and an eighth more than an even share
    assert 8 * max(per_xcd) <= len(seen) + 256 or 64 * max(per_xcd) <= 9 * len(seen)
