"""The sweeps of the persistent batch launch: programs of a few and of more
rotations than are staged at a time, state vectors in LDS and beyond it,
several instances per workgroup, vanishing angles, every kernel shape.

Tolerance: 1e-10 against the single-instance engine calls, the bound of the
other batch tests.
"""

from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (orbitals, alpha, beta), workgroups
CASES = {
    "few": ([(2, 1, 1), (4, 2, 2), (5, 3, 2)], 0),
    "more than one chunk of rotations": ([(6, 3, 3), (8, 4, 4), (5, 2, 2), (6, 3, 3)], 2),
    "largest state in LDS and smaller": ([(8, 4, 4), (9, 3, 3), (4, 2, 2)], 0),
    "states beyond LDS": ([(9, 4, 5), (4, 2, 2), (9, 3, 4)], 2),
}


@pytest.mark.parametrize("name", list(CASES))
def test_persistent_sweeps(name):
    from slowquant_amd import engine as E
    from slowquant_amd.batch import loop_energy_grad
    from slowquant_amd.synthetic import synthetic_hamiltonian
    from slowquant_amd.util import UpsStructure

    spaces, nwg = CASES[name]
    inst, thetas = [], []
    for k, (n, na, nb) in enumerate(spaces):
        occ_spin = sorted([2 * p for p in range(na)] + [2 * p + 1 for p in range(nb)])
        unocc_spin = [s for s in range(2 * n) if s not in occ_spin]
        occ = list(range(min(na, nb)))
        lay = UpsStructure()
        lay.create_fUCC(occ, [p for p in range(n) if p not in occ], occ_spin, unocc_spin, n,
                        {"n_layers": 1, "S": True, "D": True})
        rng = np.random.default_rng(50 + k)
        h, g = synthetic_hamiltonian(n, 2 * n, rng)
        sp = E.Space(n, na, nb)
        inst.append((sp, E.Program(sp, lay.excitation_operator_type, lay.excitation_indices), E.Hamiltonian(sp, h, g, 0.3)))
        th = rng.normal(0.0, 0.3, lay.n_params)
        th[::5] = 0.0
        thetas.append(th)
    b = E.Batch(inst, nwg)
    e_ref, g_ref = loop_energy_grad(inst, thetas)
    for shape in ((1, 1), (2, 2), (4, 1)):
        b.configure(*shape)
        for graph in (False, True):
            e, g = b.run(thetas, graph=graph)
            assert np.abs(np.asarray(e) - np.asarray(e_ref)).max() < 1e-10
            for x, y in zip(g, g_ref):
                assert np.abs(x - y).max() < 1e-10
