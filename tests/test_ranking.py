"""The order by which singular values and column norms are ranked (csrc/ranking.h), compiled for the host: the ranks of
any values are a permutation, NaN and infinities included, and finite values are in descending order, ties by index."""
import ctypes
import itertools
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = r"""
#define __host__
#define __device__
#include "ranking.h"
extern "C" void ranks(const double* x, int64_t n, int64_t* out) {
  for (int64_t j = 0; j < n; ++j) {
    out[j] = 0;
    for (int64_t i = 0; i < n; ++i) out[j] += ranks_before(x[i], i, x[j], j);
  }
}
"""


@pytest.fixture(scope='module')
def ranks(tmp_path_factory):
    d = tmp_path_factory.mktemp('ranking')
    (d / 'ranking.cpp').write_text(SOURCE)
    subprocess.run(['g++', '-O2', '-shared', '-fPIC', '-I', os.path.join(ROOT, 'yastn_amd', 'csrc'),
                    str(d / 'ranking.cpp'), '-o', str(d / 'ranking.so')], check=True)
    fn = ctypes.CDLL(str(d / 'ranking.so')).ranks

    def run(x):
        x, out = np.ascontiguousarray(x, dtype=np.float64), np.empty(len(x), dtype=np.int64)
        fn(x.ctypes.data_as(ctypes.c_void_p), ctypes.c_int64(len(x)), out.ctypes.data_as(ctypes.c_void_p))
        return out
    return run


def test_ranks_are_a_permutation(ranks):
    values = (np.nan, -np.nan, np.inf, 0.0, 1e-320, 2.0, 1e300)
    for n in range(1, 6):
        for x in itertools.product(values, repeat=n):
            assert sorted(ranks(x)) == list(range(n)), x


def test_finite_values_descend_with_ties_by_index(ranks):
    rng = np.random.default_rng(3)
    for n in (1, 7, 130):
        x = rng.integers(0, 20, n).astype(np.float64)
        order = np.empty(n, dtype=np.int64)
        order[ranks(x)] = np.arange(n)
        assert np.array_equal(order, np.argsort(-x, kind='stable'))
