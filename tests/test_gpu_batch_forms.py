"""Batched solves on every form of the H.v launches (BatchHv, ed_batch.hpp):
problems that gather their cross bonds, ones that stage them (several bonds
per high bit) and ones with low-low target tables (short segments), alone and
next to each other, with momentum sectors, in both precisions.

A problem's numbers do not depend on the others in the batch, so a mix equals
the same problems alone to the bit; against the oracle the solves' accuracy of
1e-10 relative holds."""
import numpy as np
import pytest

import alps_amd as A
import oracle_lib as O
from test_gpu_hv_paths import lattice, random_bonds
from test_gpu_parity import random_xxz, say, to_product

pytestmark = pytest.mark.gpu

# name: model, n_up, nev (D < 1000 or nev > 2: FP64)
PROBLEMS = {
    "staged_4x4": (lambda: lattice(4, 4, 1), 8, 1),
    "staged_5x3": (lambda: lattice(5, 3, 2), 7, 2),
    "staged_6x3": (lambda: lattice(6, 3, 3), 9, 1),
    "staged_6x3_few_up": (lambda: lattice(6, 3, 4), 3, 1),
    "staged_4x4_f64": (lambda: lattice(4, 4, 5), 6, 3),
    "staged_random": (lambda: random_bonds(17, 20, 4, 6), 8, 1),
    "gathered_chain": (lambda: random_xxz(16, True, 7), 8, 1),
    "gathered_chain_f64": (lambda: random_xxz(10, True, 8), 5, 2),
    "tables_chain22": (lambda: random_xxz(22, True, 9), 5, 1),
    "tables_chain22_f64": (lambda: random_xxz(22, True, 10), 17, 3),
    "tables_lattice": (lambda: lattice(11, 2, 11), 17, 1),
}
MIXES = {
    "staged": ["staged_4x4", "staged_5x3", "staged_6x3", "staged_6x3_few_up", "staged_4x4_f64", "staged_random"],
    "tables": ["tables_chain22", "tables_chain22_f64", "tables_lattice"],
    "all": list(PROBLEMS),
}


def solve(names, steps=0, graphs=False, dtype="f32"):
    b = A.Batch(dtype, steps_per_round=steps, graphs=graphs, hbm_bytes=8 << 30)
    t = []
    for n in names:
        mk, k, nev = PROBLEMS[n]
        t.append(b.submit(to_product(mk(), k), nev=nev, seed=3))
    b.run()
    out = [np.array(b.result(x)["ev"]) for x in t]
    b.close()
    return out


@pytest.mark.parametrize("dtype", ["f32", "f64"])
@pytest.mark.parametrize("name", list(PROBLEMS))
def test_eigenvalues_vs_oracle(name, dtype):
    say("problem", name, dtype)
    mk, k, nev = PROBLEMS[name]
    (ev,) = solve([name], dtype=dtype)
    want = O.sparsediag(mk(), k, nev=nev, seed=3)["ev"]
    np.testing.assert_allclose(ev[:1], want[:1], rtol=1e-10)


@pytest.mark.parametrize("steps,graphs", [(3, False), (8, True)])
@pytest.mark.parametrize("mix", list(MIXES))
def test_a_mix_equals_its_problems_alone(mix, steps, graphs):
    say("mix", mix, steps, graphs)
    together = solve(MIXES[mix], steps, graphs)
    for name, ev in zip(MIXES[mix], together):
        assert np.array_equal(ev, solve([name], steps, graphs)[0]), name
