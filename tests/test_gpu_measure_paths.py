"""Spin sums on the device (alps_ed_vector_spin_moments, _flip_pairs) against
plain FP64 sums over the rows, where their kernels can go wrong: no high bits,
few, more than 12 and more than 16 (tiles of the matrix products), sectors at
both ends of n_up, segments of one row up to the longest class, pair lists on
both sides of the line between the pair kernel and the matrix of all pairs,
and a vector with an element that is not finite.

Tolerance: FP64 sums of at most 10^6 terms of mixed sign in any order stay
within 1e-12 of the sum of squares, as in the oracle comparison."""
import numpy as np
import pytest

import alps_amd as A
import oracle_lib as O
from test_gpu_parity import say, to_product

pytestmark = pytest.mark.gpu

SECTORS = [(2, 1), (5, 0), (5, 5), (8, 3), (12, 6), (12, 1), (12, 12), (13, 6), (13, 13), (14, 1), (17, 8), (21, 10),
           (22, 5), (22, 19), (24, 4), (25, 3), (27, 25), (28, 4), (29, 3), (32, 3), (32, 30), (32, 1)]


def flips(op, states, x, i, j, N):
    bi, bj = np.uint32(1 << (N - 1 - i)), np.uint32(1 << (N - 1 - j))
    rows = np.nonzero((states & bj != 0) & (states & bi == 0))[0]
    if not len(rows):
        return 0.0
    return float(x[rows] @ x[op.index(states[rows] ^ bi ^ bj).astype(np.int64)])


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("N,k", SECTORS)
def test_spin_sums_vs_rows(N, k, dtype):
    say("spin sums", N, k, dtype)
    op = A.Operator(to_product(O.lattice_model("chain lattice", N), k))
    v = A.Vector.from_numpy(np.random.default_rng(N + k).uniform(-1, 1, op.dim), dtype)
    x = v.numpy().astype(np.float64)
    states = op.states().astype(np.uint32)
    s = np.array([((states >> np.uint32(N - 1 - i)) & 1) - 0.5 for i in range(N)], dtype=np.float64)
    n2, sz, szsz = op.spin_moments(v)
    scale = 1e-12 * float(x @ x)
    assert abs(n2 - x @ x) <= scale
    assert np.abs(sz - s @ (x * x)).max() <= scale
    assert np.abs(szsz - (s * (x * x)) @ s.T).max() <= scale
    i, j = np.triu_indices(N, 1)
    got = op.flip_pairs(v, j, i)  # all pairs
    few = op.flip_pairs(v, i[-9:], j[-9:])
    want = np.array([flips(op, states, x, a, b, N) for a, b in zip(i, j)])
    assert np.abs(got - want).max() <= scale
    assert np.abs(few - want[-9:]).max() <= scale


def test_flip_pairs_of_a_vector_that_is_not_finite():
    op = A.Operator(to_product(O.lattice_model("chain lattice", 14), 7))
    x = np.random.default_rng(1).uniform(-1, 1, op.dim)
    x[1000] = np.inf
    v = A.Vector.from_numpy(x, "f64")
    i, j = np.triu_indices(14, 1)
    got = op.flip_pairs(v, i, j)
    want = np.concatenate([op.flip_pairs(v, i[a : a + 8], j[a : a + 8]) for a in range(0, len(i), 8)])
    assert np.array_equal(got, want, equal_nan=True)
    assert np.isfinite(got).any() and not np.isfinite(got).all()
