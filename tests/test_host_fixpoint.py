"""The 64-bit accumulator words of the atomic split reductions (count << 56 | fixed-point
sum), compiled for the host: counts up to 255 contributors, negative sums, the clamp and
non-finite partial sums."""
import ctypes
import math
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
MASK = (1 << 64) - 1


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("fixpoint") / "fixpoint_shim.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", os.path.join(HERE, "fixpoint_shim.cpp"),
                    "-o", so], check=True)
    lib = ctypes.CDLL(so)
    lib.shim_fix_word.restype = ctypes.c_uint64
    lib.shim_fix_word.argtypes = [ctypes.c_float]
    lib.shim_fix_count.restype = ctypes.c_int
    lib.shim_fix_count.argtypes = [ctypes.c_uint64]
    lib.shim_fix_value.restype = ctypes.c_float
    lib.shim_fix_value.argtypes = [ctypes.c_uint64]
    return lib


def _accumulate(lib, values):
    w = 0
    for v in values:
        w = (w + lib.shim_fix_word(float(v))) & MASK  # what the 64-bit atomic add does
    return w


@pytest.mark.parametrize("n", [1, 2, 127, 128, 129, 200, 255])
@pytest.mark.parametrize("sign", [1.0, -1.0])
def test_count_and_sum_survive_up_to_255_contributors(shim, n, sign):
    rng = np.random.default_rng(n)
    vals = (sign * np.abs(rng.standard_normal(n)) * 300.0).astype(np.float32)
    w = _accumulate(shim, vals)
    assert shim.shim_fix_count(w) == n
    total = float(np.sum(vals.astype(np.float64)))
    assert abs(shim.shim_fix_value(w) - total) <= n * 2.0 ** -20 + abs(total) * 2.0 ** -23


def test_mixed_signs_cancel_exactly_on_grid_values(shim):
    vals = [1.5, -1.5, 1024.25, -1024.25, -0.125]
    w = _accumulate(shim, vals)
    assert shim.shim_fix_count(w) == 5 and shim.shim_fix_value(w) == -0.125
    # every intermediate count is visible to a lane that reads the word back
    w = 0
    for i, v in enumerate(vals):
        w = (w + shim.shim_fix_word(v)) & MASK
        assert shim.shim_fix_count(w) == i + 1


def test_order_independence(shim):
    rng = np.random.default_rng(3)
    vals = (rng.standard_normal(40) * 100).astype(np.float32)
    a = _accumulate(shim, vals)
    b = _accumulate(shim, vals[::-1])
    c = _accumulate(shim, rng.permutation(vals))
    assert a == b == c


def test_clamp_rounds_to_infinity_in_fp16(shim):
    w = _accumulate(shim, [1e9, 3.0])
    assert shim.shim_fix_count(w) == 2
    with np.errstate(over="ignore"):
        assert np.isinf(np.float16(shim.shim_fix_value(w)))
    w = _accumulate(shim, [-1e9] * 255)
    assert shim.shim_fix_count(w) == 255
    with np.errstate(over="ignore"):
        assert np.float16(shim.shim_fix_value(w)) == -np.inf


@pytest.mark.parametrize("bad", [math.nan, math.inf, -math.inf])
@pytest.mark.parametrize("n_bad,n_ok", [(1, 0), (1, 254), (255, 0), (3, 100)])
def test_non_finite_partial_sums_poison_the_total(shim, bad, n_bad, n_ok):
    vals = [bad] * n_bad + [-262144.0] * n_ok  # the most negative legitimate partial sums
    w = _accumulate(shim, vals)
    assert shim.shim_fix_count(w) == n_bad + n_ok
    assert math.isnan(shim.shim_fix_value(w))


def test_preseeded_count_never_completes(shim):
    """A word that starts with count 255 ends one short of the number of contributors:
    what the GPU test of the bounded wait relies on."""
    w = 0xFF << 56
    for _ in range(5):
        w = (w + shim.shim_fix_word(1.0)) & MASK
    assert shim.shim_fix_count(w) == 4


def _reduce(lib, partial):
    partial = np.ascontiguousarray(partial, np.float32)
    c, n = partial.shape
    total, count = np.empty(n, np.float32), np.empty(n, np.int32)
    as_p = lambda a: a.ctypes.data_as(ctypes.c_void_p)
    lib.shim_fix_reduce(as_p(partial), c, n, as_p(total), as_p(count))
    return total, count


@pytest.mark.parametrize("contributors", [1, 2, 10, 15, 16, 20, 31])
@pytest.mark.parametrize("scale", [30.0, 1.0, 1e-3, 1e-4, 1e-5, 1e-6])
def test_words_of_few_contributors_lose_nothing_against_fp32_partial_rows(shim, contributors, scale):
    """Totals of partial sums of 512 products at activations of `scale`, after the fp16 cast that
    follows: as far from 64 bits as an fp32 sum in index order. Up to 31 contributors the words
    have 30 fraction bits or more; their roundings (31 of 2^-30/sqrt(12) rms) are at most 1/11 of the
    rms of the cast on fp16's finest grid, 2^-24/sqrt(12): 0.4 % of its error, tolerance 1 %."""
    rng = np.random.default_rng(contributors)
    partial = (rng.standard_normal((contributors, 1 << 15)) * (scale * 512 ** 0.5 * 1.24)).astype(np.float32)
    exact = partial.astype(np.float64).sum(axis=0)
    rows = partial[0].copy()
    for p in partial[1:]:
        rows += p
    total, count = _reduce(shim, partial)
    assert (count == contributors).all()
    err = lambda v: float(np.linalg.norm(v.astype(np.float16).astype(np.float64) - exact))
    assert np.isfinite(total).all()
    assert err(total) <= 1.01 * err(rows) + 1e-12


@pytest.mark.parametrize("contributors", [1, 15, 16, 31, 32, 63, 64, 127, 128, 255])
def test_words_at_both_ends_of_every_count_width(shim, contributors):
    """Extremes of the clamp, a single non-finite contributor and nothing but non-finite ones, at the
    smallest and the largest number of contributors of each width of the count."""
    c, big = contributors, 262144.0
    cols = np.full((c, 6), big, np.float32)
    cols[:, 1] = -big
    cols[:, 2] = np.inf
    cols[0, 3] = np.nan
    cols[0, 4] = -np.inf
    cols[:, 4][1:] = -big
    cols[:, 5] = np.where(np.arange(c) % 2, -3.5, 3.5)
    total, count = _reduce(shim, cols)
    assert (count == c).all()
    assert total[0] == c * big and total[1] == -c * big
    assert np.isnan(total[2:5]).all()
    assert total[5] == (3.5 if c % 2 else 0.0)
    # a word that starts with the count's field full never reads as complete
    lib, b = shim, shim.shim_fix_count_bits(c)
    lib.shim_fix_word_bits.restype = ctypes.c_uint64
    lib.shim_fix_word_bits.argtypes = [ctypes.c_float, ctypes.c_int]
    lib.shim_fix_count_of.argtypes = [ctypes.c_uint64, ctypes.c_int]
    w = 0xFF << 56
    for _ in range(c):
        w = (w + lib.shim_fix_word_bits(big, b)) & MASK
    assert lib.shim_fix_count_of(w, b) == c - 1
