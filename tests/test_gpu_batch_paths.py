"""Batched solves at the edges of the step's paths: FP32 and FP64 problems side
by side, problems whose update forms the step's scalars and ones with
reduction launches (kBatchFuse, ed_batch.hpp: at most 4096 partials), groups
of one step up to many, one and two Ritz vectors, lengths that are not
multiples of four.

A problem's numbers do not depend on the others in the batch, so a mix equals
the same problems alone to the bit; small ones meet the oracle's eigenvalues
to 1e-10 relative, the accuracy of the solves."""
import numpy as np
import pytest

import alps_amd as A
import oracle_lib as O
from test_gpu_parity import random_xxz, say, to_product

pytestmark = pytest.mark.gpu

# sites, n_up, nev (D < 1000 or nev > 2: FP64)
MIXES = {
    "fp32_and_fp64": [(16, 8, 1), (10, 5, 1), (15, 6, 2), (11, 5, 3), (14, 7, 2), (13, 5, 1), (9, 1, 1)],
    "both_sides_of_the_line": [(23, 11, 1), (24, 12, 1), (14, 7, 1), (10, 4, 2)],
    "fp64_only": [(10, 5, 2), (12, 6, 4), (8, 2, 1)],
}


@pytest.mark.parametrize("steps,graphs", [(1, False), (3, False), (8, True), (0, False)])
@pytest.mark.parametrize("name", list(MIXES))
def test_a_mix_equals_its_problems_alone(name, steps, graphs):
    if name == "both_sides_of_the_line" and steps == 1:
        steps = 2
    say("mix", name, steps, graphs)

    def solve(problems):
        b = A.Batch("f32", steps_per_round=steps, graphs=graphs, hbm_bytes=16 << 30)
        t = [b.submit(to_product(random_xxz(n, True, n), k), nev=nev, seed=n) for n, k, nev in problems]
        b.run()
        return [np.array(b.result(x)["ev"]) for x in t]

    mix = MIXES[name]
    together = solve(mix)
    for (n, k, nev), ev in zip(mix, together):
        assert np.array_equal(ev, solve([(n, k, nev)])[0]), (n, k, nev)
        if n <= 16:
            want = O.sparsediag(random_xxz(n, True, n), k, nev=nev, seed=n)["ev"]
            np.testing.assert_allclose(ev[:1], want[:1], rtol=1e-10)
