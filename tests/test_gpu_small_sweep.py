"""The one-block sweep of small spaces (sq_small.hip): states and adjoint
gradients against the oracle, and against the per-gate kernels at the sizes
the oracle is slow for.

Tolerances are those of the engine's other parity tests: states 1e-12,
gradients 1e-10 (a sweep of N gates adds about N rounding errors of 1e-16 per
amplitude, N < 1000 here).
"""

from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _layout(n, na, nb, options):
    from slowquant_amd.util import UpsStructure

    occ_spin = sorted([2 * p for p in range(na)] + [2 * p + 1 for p in range(nb)])
    unocc_spin = [s for s in range(2 * n) if s not in occ_spin]
    occ = list(range(min(na, nb)))
    lay = UpsStructure()
    lay.create_fUCC(occ, [p for p in range(n) if p not in occ], occ_spin, unocc_spin, n, dict(options))
    return lay


def _theta(n, seed):
    th = np.random.default_rng(seed).normal(0.0, 0.4, n)
    th[n // 2] = 0.0
    return th


def _start(sp, seed):
    import torch

    v = np.random.default_rng(seed).normal(size=sp.dim)
    return torch.tensor(v / np.linalg.norm(v), device="cuda")


ORACLE = [
    (2, 1, 1, {"n_layers": 1, "S": True, "D": True}),  # 4 determinants
    (4, 2, 2, {"n_layers": 1, "SAS": True, "SAD": True, "T": True, "Q": True}),
    (5, 3, 2, {"n_layers": 1, "SAS": True, "SAD": True}),  # odd, unequal spins
    (6, 3, 3, {"n_layers": 1, "SAS": True, "SAD": True}),
    (5, 2, 1, {"n_layers": 1, "SAGS": True, "GpD": True}),
]


@pytest.mark.parametrize("n,na,nb,options", ORACLE)
def test_against_oracle(n, na, nb, options):
    from oracle.ci import get_indexing
    from oracle.fermion import hamiltonian_active_fast
    from oracle.ups import construct_ups_state, gradient_adjoint
    from slowquant_amd import engine as E
    from slowquant_amd.synthetic import synthetic_hamiltonian

    lay = _layout(n, na, nb, options)
    th = _theta(lay.n_params, n)
    h, g = synthetic_hamiltonian(n, 2 * n, np.random.default_rng(1))
    sp = E.Space(n, na, nb)
    prog = E.Program(sp, lay.excitation_operator_type, lay.excitation_indices)
    x = _start(sp, 3)
    ref = sp.to_reference_numpy(x)
    ci = get_indexing(0, n, 0, na, nb)
    for dagger in (False, True):
        out = sp.to_reference_numpy(prog.state_prep(th, x, dagger=dagger))
        expect = construct_ups_state(ref, ci, th, lay, dagger=dagger)
        assert np.abs(out - expect).max() < 1e-12
    e, grad = prog.energy_grad(E.Hamiltonian(sp, h, g), th, x)
    e_ref, g_ref = gradient_adjoint(hamiltonian_active_fast(h, g, n), ref, ci, th, lay)
    assert abs(e - e_ref) < 1e-10
    assert np.abs(grad - g_ref).max() < 1e-10


PER_GATE = [
    (6, 3, 3, {"n_layers": 3, "S": True, "D": True}),  # more gates than one staged chunk of steps
    (8, 4, 4, {"n_layers": 1, "SAS": True, "SAD": True}),
    (9, 3, 3, {"n_layers": 1, "SAGS": True, "GpD": True}),  # more pairs per gate than threads
    (13, 2, 2, {"n_layers": 1, "SAS": True, "pD": True}),  # close to the largest space taken
    (13, 2, 3, {"n_layers": 1, "pD": True}),  # above it: both sides run per gate
]


@pytest.mark.parametrize("n,na,nb,options", PER_GATE)
def test_against_per_gate_kernels(n, na, nb, options, monkeypatch):
    from slowquant_amd import engine as E
    from slowquant_amd.synthetic import synthetic_hamiltonian

    lay = _layout(n, na, nb, options)
    th = _theta(lay.n_params, n)
    h, g = synthetic_hamiltonian(n, 2 * n, np.random.default_rng(2))
    sp = E.Space(n, na, nb)
    H = E.Hamiltonian(sp, h, g)
    x = _start(sp, 4)
    prog = E.Program(sp, lay.excitation_operator_type, lay.excitation_indices)
    psi, (e, grad) = prog.state_prep(th, x), prog.energy_grad(H, th, x)
    assert np.abs((prog.state_prep(th, psi, dagger=True) - x).cpu().numpy()).max() < 1e-12
    monkeypatch.setenv("SQ_SMALL_SWEEP", "0")
    old = E.Program(sp, lay.excitation_operator_type, lay.excitation_indices)
    assert float((old.state_prep(th, x) - psi).abs().max()) < 1e-12
    e_old, g_old = old.energy_grad(H, th, x)
    assert abs(e - e_old) < 1e-10
    assert np.abs(grad - g_old).max() < 1e-10
