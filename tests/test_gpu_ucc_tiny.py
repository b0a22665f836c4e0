"""Unfactorised UCC at amplitudes around and below the smallest normal number,
where the reciprocal of T's row sums overflows: states, energies and gradients
are those of T = 0 (the difference is of the order of the amplitudes).
"""

from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [1e-290, 1e-300, 1e-307, 1e-309, 5e-324])
def test_tiny_amplitudes(size):
    import torch

    from slowquant_amd import engine as E
    from slowquant_amd.synthetic import synthetic_hamiltonian
    from slowquant_amd.util import UccStructure

    lay = UccStructure()
    lay.add_sa_singles([0, 1], [2, 3])
    lay.add_sa_doubles([0, 1], [2, 3])
    types = ["sa_single_ucc" if t == "sa_single" else t for t in lay.excitation_operator_type]
    sp = E.Space(4, 2, 2)
    prog = E.Program(sp, types, lay.excitation_indices)
    H = E.Hamiltonian(sp, *synthetic_hamiltonian(4, 8, np.random.default_rng(2)))
    psi0 = E.hf_state(sp)
    e0, g0 = E.ucc_energy_grad(prog, H, np.zeros(prog.n_gates), psi0)
    theta = size * (-1.0) ** np.arange(prog.n_gates)
    assert torch.allclose(E.ucc_expm(prog, theta, psi0), psi0, rtol=0.0, atol=1e-200)
    e, g = E.ucc_energy_grad(prog, H, theta, psi0)
    assert abs(e - e0) < 1e-12 and np.abs(g - g0).max() < 1e-12
