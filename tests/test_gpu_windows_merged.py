"""Window tiles of several groups (few electrons in many orbitals, where one
group holds few strings) against the per-gate kernels: sides of one and of two
group counts, one tile, long rows and long columns, odd tile targets, empty
strings, every thread count, U^+ and the gradient.  And the sweep they are for
takes less time than one launch per rotation.

Tolerances: states 1e-12, gradients 1e-10, as the other window tests.
"""

from __future__ import annotations

import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [
    # n, na, nb, layers, layout, tile target, threads
    (9, 1, 1, 2, "tups", 0, 0),  # one tile
    (10, 0, 2, 2, "qnp", 0, 0),  # an empty spin
    (11, 2, 3, 2, "tups", 300, 256),
    (12, 10, 2, 2, "tups", 700, 512),
    (13, 3, 3, 2, "tups", 0, 0),
    (13, 1, 6, 1, "qnp", 4900, 256),  # long rows
    (14, 6, 1, 1, "tups", 2500, 0),  # long columns
    (14, 2, 7, 1, "tups", 0, 512),
    (15, 3, 2, 2, "tups", 0, 0),
    (16, 2, 2, 2, "tups", 100, 0),
    (16, 2, 3, 2, "qnp", 0, 0),
]


def _programs(n, na, nb, layers, kind, monkeypatch):
    from slowquant_amd import engine as E
    from slowquant_amd.util import UpsStructure

    lay = UpsStructure()
    lay.create_tiled(n, {"n_layers": layers, "do_" + kind: True})
    sp = E.Space(n, na, nb)
    prog, ref = (E.Program(sp, lay.excitation_operator_type, lay.excitation_indices) for _ in range(2))
    monkeypatch.setenv("SQ_TILES", "0")
    monkeypatch.setenv("SQ_SMALL_SWEEP", "0")
    ref.state_prep(np.zeros(lay.n_params), E.hf_state(sp))  # its plan is fixed here
    monkeypatch.delenv("SQ_TILES")
    return sp, prog, ref, lay.n_params


@pytest.mark.parametrize("n,na,nb,layers,kind,target,threads", CASES)
def test_merged_tiles_against_per_gate_kernels(n, na, nb, layers, kind, target, threads, monkeypatch):
    import torch

    from slowquant_amd import engine as E
    from slowquant_amd.synthetic import synthetic_hamiltonian

    sp, prog, ref, ng = _programs(n, na, nb, layers, kind, monkeypatch)
    rng = np.random.default_rng(n)
    th = rng.normal(0.0, 0.4, ng)
    H = E.Hamiltonian(sp, *synthetic_hamiltonian(n, 2 * n, rng))
    v = rng.normal(size=sp.dim)
    x = torch.tensor(v / np.linalg.norm(v), device="cuda")
    prog.set_tile_shape(target, threads)
    for dagger in (False, True):
        d = prog.state_prep(th, x, dagger=dagger) - ref.state_prep(th, x, dagger=dagger)
        assert float(d.abs().max()) < 1e-12
    e, g = prog.energy_grad(H, th, x)
    e_ref, g_ref = ref.energy_grad(H, th, x)
    assert abs(e - e_ref) < 1e-10 and np.abs(g - g_ref).max() < 1e-10
    if sp.dim <= 2000:
        _, plain = prog.energy_grad(H, th, x, "plain")
        assert np.abs(plain - g_ref).max() < 1e-10


def test_few_electrons_take_less_than_a_launch_per_rotation(monkeypatch):
    import torch

    from slowquant_amd import engine as E

    sp, prog, ref, ng = _programs(16, 3, 3, 2, "tups", monkeypatch)
    th = torch.full((ng,), 0.1, dtype=torch.float64, device="cuda")
    psi0 = E.hf_state(sp)
    out = torch.empty_like(psi0)

    def best(p):
        t = []
        for _ in range(8):
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            p.state_prep(th, psi0, out=out)
            torch.cuda.synchronize()
            t.append(time.perf_counter() - t0)
        return min(t)

    assert best(prog) < 0.5 * best(ref)
