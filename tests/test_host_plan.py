"""Launch plans of the one-launch layer kernels as the library reports them (no GPU needed)."""
import ctypes
import os
import subprocess
import sys

import pytest

from conftest import ROOT


def _plan(lib, rows, n_in, n_out, k):
    out = [ctypes.c_int() for _ in range(4)]
    assert lib.exl3_linear_plan(rows, n_in // 16, n_out // 16, k, *[ctypes.byref(v) for v in out]) == 0
    n_splits, tile_rows, waves, atomic = (v.value for v in out)
    return -(-n_splits // waves), tile_rows, waves, bool(atomic)


@pytest.fixture(scope="module")
def lib():
    from ponyexl3_amd import _lib

    return _lib.load()


@pytest.mark.parametrize("rows", range(2, 9))
def test_large_launches_reduce_in_fp32_or_in_words_as_good(lib, rows):
    """A launch of more atomics than the whole-block kernel sends through its accumulators (300 k, 800 k at
    two rows) takes fp32 partial rows, or words of at least 30 fraction bits: up to 31 partial rows."""
    limit = 800000 if rows == 2 else 300000
    seen = 0
    for n_in in (1664, 2560, 5120, 6144, 8192, 14336, 15872, 16000, 16384, 17408):
        for n_out in (1024, 2560, 5120, 5888, 10240, 12288, 34816):
            for k in range(1, 9):
                partials, tile_rows, waves, atomic = _plan(lib, rows, n_in, n_out, k)
                # per column group: the same splits in partial rows of eight waves of half blocks
                whole = n_out * rows * (-(-n_in // 512) if tile_rows == 4 else partials)
                if atomic and whole > limit:
                    seen += 1
                    assert partials <= 31, (n_in, n_out, k)
    assert seen or rows in (2, 7, 8)


def _whole_block_contributors(n_in, n_out, k):
    """Contributors per sum of one row's launch in whole blocks (0: fp32 partial rows): up to twelve waves per
    SIMD, two blocks to a wave from K = 5 on where that leaves two, and workgroups of eight waves where those of four would
    issue more than 300 k atomics."""
    blocks, groups = n_in // 128, n_out // 128
    splits = min(max(12288 // groups, 1), blocks)
    per = -(-blocks // splits)
    if k >= 5 and per == 1 and blocks >= 2 and groups * ((blocks + 1) // 2) >= 2048:
        per = 2
    splits = -(-blocks // per)
    for waves in (4, 8):
        n = -(-splits // waves)
        if n <= 255 and groups * n * 128 <= 300000:
            return n
    return 0


def test_one_row_of_a_full_chip_keeps_the_fraction_bits_of_whole_blocks(lib):
    """Where 4096 waves of whole blocks and more would run, one row takes half blocks only if its sums stay as fine:
    accumulators where whole blocks have them, in words of no fewer fraction bits (33 up to 15 contributors, 30 up
    to 31, ...); else the plan of whole blocks."""
    halves = 0
    for n_in in range(1024, 17409, 128):
        for n_out in list(range(1024, 65537, 1664)) + [34816, 151936, 303872]:
            if n_in // 128 * (n_out // 128) < 4096:
                continue
            for k in range(1, 9):
                n, tile_rows, waves, atomic = _plan(lib, 1, n_in, n_out, k)
                whole = _whole_block_contributors(n_in, n_out, k)
                if tile_rows == 4:
                    halves += 1
                    assert whole and atomic and max(n.bit_length(), 4) <= max(whole.bit_length(), 4), (n_in, n_out, k)
                else:
                    assert atomic == (whole > 0) and (not whole or n == whole), (n_in, n_out, k)
    assert halves > 1000


# none left over by workgroups of four; one and two; the same in as many rounds; three; whole blocks eight to a workgroup: none left over by
# the fours in as many rounds and in fewer, one, three in as many and in fewer; K = 3 on both sides, K = 4
@pytest.mark.parametrize("k,n_in,n_out,half", [
    (2, 2048, 65536, False), (1, 2048, 65536, False), (2, 3072, 31104, False), (1, 9728, 13824, False),
    (2, 3200, 31360, True), (2, 2816, 51840, True), (2, 1280, 52480, True), (2, 4864, 15232, True),
    (2, 4736, 19328, False), (1, 9472, 8320, False), (2, 1408, 61952, False),
    (1, 2560, 63104, False), (2, 6144, 30336, False), (2, 4608, 34176, True), (2, 6656, 27392, True), (2, 2688, 56064, True),
    (2, 3456, 47232, False), (1, 2944, 55296, True), (3, 2048, 65536, False), (3, 3840, 33792, True), (4, 2048, 65536, True), (4, 9728, 13824, True)])
def test_one_row_of_light_layers_takes_half_blocks_where_they_balance(lib, k, n_in, n_out, half):
    """Up to K = 3 half blocks come in workgroups of eight only where they fill the chip in fewer rounds than the whole ones."""
    _, tile_rows, _, _ = _plan(lib, 1, n_in, n_out, k)
    assert (tile_rows == 4) == half


_PLANS = """
import ctypes, sys
sys.path.insert(0, sys.argv[1])
from ponyexl3_amd import _lib
lib = _lib.load()
for rows in range(1, 9):
    for n_in, n_out in ((128, 128), (1664, 2560), (5120, 1024), (5120, 5120), (5120, 10240), (17408, 5120), (5120, 34816)):
        for k in (2, 4, 6, 8):
            out = [ctypes.c_int() for _ in range(4)]
            assert lib.exl3_linear_plan(rows, n_in // 16, n_out // 16, k, *[ctypes.byref(v) for v in out]) == 0
            n_splits, _, waves, atomic = (v.value for v in out)
            partials = -(-n_splits // waves)
            print(partials, partials * n_out * rows * 3 // (8 if rows == 2 else 3), atomic)
"""


@pytest.mark.parametrize("limit", [0, 50000, 300000, 1 << 30])
def test_the_atomics_switch_reaches_every_one_launch_kernel(limit):
    """EXL3_LINEAR_MAX_ATOMICS (read once per process): launches of more atomics reduce through partial rows,
    launches of as many or fewer through accumulators, whether waves take whole or half blocks."""
    env = dict(os.environ, EXL3_LINEAR_MAX_ATOMICS=str(limit))
    run = subprocess.run([sys.executable, "-c", _PLANS, ROOT], env=env, capture_output=True, text=True, check=True)
    rows = [tuple(map(int, line.split())) for line in run.stdout.splitlines()]
    assert len(rows) == 8 * 7 * 4
    for partials, atomics, atomic in rows:
        assert atomic == (partials <= 255 and atomics <= limit)
