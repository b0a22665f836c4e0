"""Groups of eight and more instances (whose row launch takes more rows per
block) at 12 and 13 orbitals, where those rows leave least room for two blocks
on a CU, against the single-instance calls.

Tolerance: 1e-10, the bound of the other batch tests.
"""

from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,na,nb,count", [(12, 6, 6, 7), (12, 6, 6, 9), (12, 3, 6, 8), (13, 4, 3, 8), (13, 2, 10, 9)])
def test_many_instances_of_one_space(n, na, nb, count):
    from slowquant_amd import engine as E
    from slowquant_amd.batch import InstanceSpec, build_instances, loop_energy_grad

    inst, thetas = build_instances([InstanceSpec(n, na, nb, 1, 300 + k) for k in range(count)])
    b = E.Batch(inst)
    e_ref, g_ref = loop_energy_grad(inst, thetas)
    for graph in (False, True, True):
        e, g = b.run(thetas, graph=graph)
        assert np.abs(np.asarray(e) - np.asarray(e_ref)).max() < 1e-10
        for x, y in zip(g, g_ref):
            assert np.abs(x - y).max() < 1e-10
