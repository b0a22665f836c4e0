"""The windowed brick-wall sweeps (sq_tiles.hip) against the per-gate kernels:
window widths from 2 to 8 orbitals (by the tile target), windows that cover
the whole space, one tile and more tiles than blocks, electron counts at the
edges (empty and full strings, single-string spins), both layouts, unequal
spins, every thread count, U^+, the adjoint and the plain gradient.

Tolerances: states 1e-12, gradients 1e-10, as the engine's other parity tests.
"""

from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [
    # n, na, nb, layers, layout, tile target, threads
    (2, 1, 1, 2, "tups", 0, 0),
    (3, 1, 2, 2, "qnp", 0, 0),
    (5, 5, 2, 1, "tups", 0, 256),  # a full spin: one alpha string
    (6, 0, 3, 2, "tups", 0, 0),  # an empty spin
    (6, 3, 3, 3, "tups", 16, 0),  # narrow windows, many stages
    (7, 4, 3, 2, "qnp", 64, 512),
    (8, 4, 4, 3, "tups", 4096, 256),  # one tile of 70 x 70
    (8, 4, 4, 3, "tups", 0, 0),
    (9, 1, 8, 2, "tups", 0, 0),
    (9, 4, 5, 2, "tups", 4096, 512),
    (10, 5, 5, 2, "tups", 256, 0),
    (11, 6, 5, 2, "qnp", 0, 0),
    (12, 2, 3, 2, "tups", 0, 0),
    (14, 3, 3, 2, "tups", 0, 0),  # more tiles than blocks of the reverse sweep
]


@pytest.mark.parametrize("n,na,nb,layers,kind,target,threads", CASES)
def test_windows_against_per_gate_kernels(n, na, nb, layers, kind, target, threads, monkeypatch):
    import torch

    from slowquant_amd import engine as E
    from slowquant_amd.synthetic import synthetic_hamiltonian
    from slowquant_amd.util import UpsStructure

    lay = UpsStructure()
    lay.create_tiled(n, {"n_layers": layers, "do_" + kind: True})
    rng = np.random.default_rng(n)
    th = rng.normal(0.0, 0.4, lay.n_params)
    th[lay.n_params // 3] = 0.0
    h, g = synthetic_hamiltonian(n, 2 * n, rng)
    sp = E.Space(n, na, nb)
    H = E.Hamiltonian(sp, h, g)
    v = rng.normal(size=sp.dim)
    x = torch.tensor(v / np.linalg.norm(v), device="cuda")
    prog = E.Program(sp, lay.excitation_operator_type, lay.excitation_indices)
    prog.set_tile_shape(target, threads)
    monkeypatch.setenv("SQ_TILES", "0")
    monkeypatch.setenv("SQ_SMALL_SWEEP", "0")
    ref = E.Program(sp, lay.excitation_operator_type, lay.excitation_indices)
    want = [ref.state_prep(th, x), ref.state_prep(th, x, dagger=True)]
    e_ref, g_ref = ref.energy_grad(H, th, x)
    monkeypatch.delenv("SQ_TILES")
    for dagger in (False, True):
        assert float((prog.state_prep(th, x, dagger=dagger) - want[dagger]).abs().max()) < 1e-12
    e, grad = prog.energy_grad(H, th, x)
    assert abs(e - e_ref) < 1e-10
    assert np.abs(grad - g_ref).max() < 1e-10
    if sp.dim <= 2000:
        _, plain = prog.energy_grad(H, th, x, "plain")
        assert np.abs(plain - g_ref).max() < 1e-10
