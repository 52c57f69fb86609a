"""H.v at the edges of its kernel paths, against the CPU oracle: staged and
gathered cross bonds on both sides of the rule that picks one (stage_cross,
ed_layout.hpp), the 512-thread workgroups of layouts with few segments and the
256-thread ones above them, segments from one row to the longest class (at
most 64 rows: one wave), sectors on both sides of ranked_rows (the rows per
segment from which on the xor page is used), low words shorter than 12 bits.

Tolerances: a row adds at most 64 terms |t x| <= 1 (and its diagonal, at most
64 terms) in FP64: at most 64 u * 64 = 4.5e-13 against entries whose norm is
at least sqrt(D); relative to the norm that stays below 1e-13 for the rms
error.  FP32 vectors add the rounding of y (6e-8) only: 2e-6 as elsewhere."""
import numpy as np
import pytest

import alps_amd as A
import oracle_lib as O
from test_gpu_parity import say, to_product

pytestmark = pytest.mark.gpu


def random_bonds(N, n_cross, n_groups, seed):
    """Random couplings on a ring's low and high bonds plus n_cross bonds
    between n_groups high bits and distinct low ones (site i is bit N-1-i;
    12 low bits)."""
    rng = np.random.default_rng(seed)
    high, low = N - 12, 12
    s = [i for i in range(N - 1) if i != high - 1]
    t = [i + 1 for i in s]
    for c in range(n_cross):
        s.append(c % n_groups)
        t.append(high + (5 * c + c // n_groups) % low)
    nb = len(s)
    return O.Model(N, np.array(s), np.array(t), rng.uniform(-1, 1, nb), rng.uniform(-1, 1, nb),
                   h=rng.uniform(-0.5, 0.5, N))


def lattice(L, W, seed):
    m = O.lattice_model("frustrated square lattice", L, W, by_type={1: (0.5, 0.5)})
    rng = np.random.default_rng(seed)
    m.jz = rng.uniform(-1, 1, m.n_bonds)
    m.jxy = rng.uniform(-1, 1, m.n_bonds)
    return m


CASES = {
    "gathered_7x4": (lambda: random_bonds(22, 7, 4, 1), [11, 1]),
    "staged_8x4": (lambda: random_bonds(22, 8, 4, 2), [11, 7, 16]),
    "gathered_9x5": (lambda: random_bonds(22, 9, 5, 9), [11]),
    "staged_12x1": (lambda: random_bonds(22, 12, 1, 3), [10]),
    "few_segments_8x4": (lambda: random_bonds(21, 8, 4, 4), [10]),
    "one_high_bit": (lambda: random_bonds(13, 12, 1, 5), [6, 0, 1, 12, 13]),
    "ring20": (lambda: O.lattice_model("chain lattice", 20), [10, 2, 18]),
    "ring21": (lambda: O.lattice_model("chain lattice", 21), [10]),
    "short_segments_25": (lambda: random_bonds(25, 9, 9, 10), [4, 5, 22]),
    "short_staged_25": (lambda: random_bonds(25, 24, 8, 11), [4, 21]),
    "ring22": (lambda: O.lattice_model("chain lattice", 22), [11, 3]),
    "lattice_4x3": (lambda: lattice(4, 3, 6), [6, 3]),
    "lattice_7x3": (lambda: lattice(7, 3, 7), [10, 20]),
    "lattice_11x2": (lambda: lattice(11, 2, 8), [11, 4]),
}


@pytest.mark.parametrize("name,k", [(n, k) for n, (_, ks) in CASES.items() for k in ks])
def test_hv_paths_vs_oracle(name, k):
    say("case", name, k)
    m = CASES[name][0]()
    op = A.Operator(to_product(m, k))
    # values that FP32 holds, so that one product of the oracle serves both
    x = np.random.default_rng(k).uniform(-1, 1, op.dim).astype(np.float32).astype(np.float64)
    want = O.spmv(m, k, x)
    for dtype, tol in (("f64", 1e-13), ("f32", 2e-6)):
        got = op.matvec(A.Vector.from_numpy(x, dtype), A.Vector(op.dim, dtype)).numpy()
        assert np.linalg.norm(got - want) <= tol * max(np.linalg.norm(want), 1e-300)
