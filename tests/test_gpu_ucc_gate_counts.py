"""The gate dots of unfactorised UCC around the gate counts where their sums
change form (a copy per wave, one per block, global memory; slices where a
fixed order is asked for): a program that repeats its gates has, for every copy
of a gate, the gradient of the plain program at the summed amplitudes.  With
fixed-order sums in sigma, repeated calls give the same bits.

Tolerance: 1e-10, the bound of the other UCC gradient tests.
"""

from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _gates(n, na):
    from slowquant_amd.util import UccStructure

    lay = UccStructure()
    lay.add_sa_singles(list(range(na)), list(range(na, n)))
    lay.add_sa_doubles(list(range(na)), list(range(na, n)))
    types = ["sa_single_ucc" if t == "sa_single" else t for t in lay.excitation_operator_type]
    return types, list(lay.excitation_indices)


@pytest.mark.parametrize("det", [-1, 1])
@pytest.mark.parametrize("times", [1, 146, 147, 292, 293])  # 14 gates; 2048 and 4096 lie between
def test_repeated_gates(times, det):
    from slowquant_amd import engine as E
    from slowquant_amd.synthetic import synthetic_hamiltonian

    types, idx = _gates(4, 2)
    sp = E.Space(4, 2, 2)
    sp.configure_sigma(0, 0, det)
    H = E.Hamiltonian(sp, *synthetic_hamiltonian(4, 8, np.random.default_rng(1)))
    psi0 = E.hf_state(sp)
    theta = np.random.default_rng(2).normal(0.0, 0.3, len(types))
    e_ref, g_ref = E.ucc_energy_grad(E.Program(sp, types, idx), H, theta, psi0)
    many = E.Program(sp, types * times, idx * times)
    e, g = E.ucc_energy_grad(many, H, np.tile(theta / times, times), psi0)
    assert abs(e - e_ref) < 1e-10
    assert np.abs(g.reshape(times, -1) - g_ref).max() < 1e-10
    if det == 1:
        for _ in range(5):
            e1, g1 = E.ucc_energy_grad(many, H, np.tile(theta / times, times), psi0)
            assert e1 == e and np.array_equal(g1, g)


@pytest.mark.parametrize("n,na", [(6, 3), (8, 4)])
def test_fixed_order_gives_the_same_bits(n, na):
    from slowquant_amd import engine as E
    from slowquant_amd.synthetic import synthetic_hamiltonian

    types, idx = _gates(n, na)
    sp = E.Space(n, na, na)
    sp.configure_sigma(0, 0, 1)
    H = E.Hamiltonian(sp, *synthetic_hamiltonian(n, 2 * n, np.random.default_rng(1)))
    psi0 = E.hf_state(sp)
    prog = E.Program(sp, types, idx)
    theta = np.random.default_rng(2).normal(0.0, 0.1, len(types))
    e, g = E.ucc_energy_grad(prog, H, theta, psi0)
    for _ in range(20):
        e1, g1 = E.ucc_energy_grad(prog, H, theta, psi0)
        assert e1 == e and np.array_equal(g1, g)
