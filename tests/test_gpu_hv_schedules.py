"""The FP32 schedules of H.v give identical results (the autotuner picks among
them by time): y and the coefficients of a recurrence, whose alpha partials
come from the same launches, to the bit.  Sectors past the line below which a
layout has one schedule (512 segments, one per high word), on every kernel
that has schedules: the page kernel with gathered and with staged cross bonds,
and the kernel with low-low target tables (short segments)."""
from math import comb

import numpy as np
import pytest

import alps_amd as A
import oracle_lib as O
from test_gpu_hv_paths import lattice, random_bonds
from test_gpu_parity import say, to_product

pytestmark = pytest.mark.gpu

CASES = {
    "gathered_ring22": (lambda: O.lattice_model("chain lattice", 22), 11, False),
    "staged_11x2": (lambda: lattice(11, 2, 8), 11, False),
    "tables_ring23": (lambda: O.lattice_model("chain lattice", 23), 8, True),
    "tables_odd_bonds": (lambda: random_bonds(23, 9, 5, 12), 8, True),
    "tables_8x3": (lambda: lattice(8, 3, 10), 8, True),
}


def segments(N, k):
    return sum(comb(N - 12, p) for p in range(N - 11) if 0 <= k - p <= 12)


@pytest.mark.parametrize("name", list(CASES))
def test_schedules_give_identical_results(name):
    mk, k, tables = CASES[name]
    m = mk()
    n_seg = segments(m.n_sites, k)
    rows = comb(m.n_sites, k) / n_seg
    assert n_seg > 512 and (rows < (500 if n_seg <= 1024 else 330)) == tables  # the line of the short segments
    op = A.Operator(to_product(m, k))
    say(name, op.dim, op.schedule())
    x = A.Vector(op.dim, "f32")
    x.fill_random(3)
    ys, runs = [], []
    for s in range(A.Operator.HV_SCHEDULES):
        op.set_schedule(s)
        ys.append(op.matvec(x, A.Vector(op.dim, "f32")).numpy())
        lz = A.Lanczos(op, "f32", max_steps=12)
        lz.start(seed=7)
        lz.steps(11)
        runs.append(lz.coefficients())
    for y in ys[1:]:
        assert np.array_equal(y.view(np.int32), ys[0].view(np.int32))
    for a, b in runs[1:]:
        assert np.array_equal(a.view(np.int64), runs[0][0].view(np.int64))
        assert np.array_equal(b.view(np.int64), runs[0][1].view(np.int64))
    want = O.spmv(m, k, x.numpy())
    np.testing.assert_allclose(ys[0], want, rtol=2e-6, atol=2e-6 * np.abs(want).max())


def test_one_schedule_is_not_timed():
    # 21 sites, 10 up: 352716 states in 512 segments, whose workgroups have
    # one form; 22 sites, 11 up: 1024 segments
    op = A.Operator(to_product(O.lattice_model("chain lattice", 21), 10))
    assert op.schedule() == (0, None)
    chosen, sec = A.Operator(to_product(O.lattice_model("chain lattice", 22), 11)).schedule()
    assert np.all(sec > 0) and sec[chosen] == sec.min()
