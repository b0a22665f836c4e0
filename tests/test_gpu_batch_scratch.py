"""Scratch memory of the persistent launch: one slot per workgroup holds psi,
lambda and the largest G of one instance, also where the space with the most
orbital pairs is not the one with the most determinants; with the vectors in
LDS it holds G alone.
"""

from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _instance(E, n, na, nb, types, idx):
    from slowquant_amd.synthetic import synthetic_hamiltonian

    sp = E.Space(n, na, nb)
    return sp, E.Program(sp, types, idx), E.Hamiltonian(sp, *synthetic_hamiltonian(n, 2 * n, np.random.default_rng(n)))


@pytest.mark.parametrize("big,doubles", [((10, 5, 5), 57 * 63504), ((8, 4, 4), 36 * 4900)])
def test_slot_size(big, doubles):
    import torch

    from slowquant_amd import engine as E

    count = 60 if big[0] == 10 else 256
    many = _instance(E, *big, ["single"], [(0, 2 * big[0] - 2)])  # not a gate of neighbouring orbitals
    inst = [many] * (count - 1) + [_instance(E, 12, 1, 1, ["single"], [(0, 4)])]
    b = E.Batch(inst[-1:])  # what a first batch of the process allocates besides
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    b = E.Batch(inst)
    used = free - torch.cuda.mem_get_info()[0]
    assert used < 8 * count * doubles + (1 << 26)
    th = [np.array([0.1])] * count
    e, g = b.run(th)
    for k in (0, count - 1):
        e_ref, g_ref = inst[k][1].energy_grad(inst[k][2], th[k], E.hf_state(inst[k][0]))
        assert abs(e[k] - e_ref) < 1e-10 and np.abs(g[k] - g_ref).max() < 1e-10
