"""Batches whose groups run on several streams: more groups than streams, with
and without instances of the persistent launch, groups of one and of many
instances (whose row launch is shaped for many), one group alone, odd and
unequal spaces around the group threshold, eager and replayed from a graph
with eager work between the replays.

Tolerance: 1e-10 against the single-instance engine calls, the bound of the
other batch tests.
"""

from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SPACES = {
    "groups only": [(8, 4, 4, 1), (8, 4, 4, 2), (8, 4, 4, 3), (9, 4, 5, 1), (9, 3, 5, 2), (10, 5, 5, 1)],
    "beside the persistent launch": [(4, 2, 2, 2), (7, 3, 4, 1), (8, 4, 4, 1), (8, 5, 4, 2), (10, 4, 3, 1)],
    "one group": [(8, 4, 4, 2)],
    "many of one group": [(9, 5, 4, 1)] * 9 + [(8, 4, 4, 1)] * 17,
}


@pytest.mark.parametrize("name", list(SPACES))
def test_batch_lanes(name):
    from slowquant_amd import engine as E
    from slowquant_amd.batch import InstanceSpec, build_instances, loop_energy_grad

    specs = [InstanceSpec(n, na, nb, layers, 100 + k) for k, (n, na, nb, layers) in enumerate(SPACES[name])]
    inst, thetas = build_instances(specs)
    b = E.Batch(inst)
    for rep in range(3):
        th = [t * (1.0 + 0.3 * rep) for t in thetas]
        e_ref, g_ref = loop_energy_grad(inst, th)
        for graph in (False, True):
            e, g = b.run(th, graph=graph)
            assert np.abs(np.asarray(e) - np.asarray(e_ref)).max() < 1e-10
            for x, y in zip(g, g_ref):
                assert np.abs(x - y).max() < 1e-10
