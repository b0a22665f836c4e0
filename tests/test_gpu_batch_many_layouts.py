"""Batches whose instances of 4096 to 16383 determinants have many gate layouts:
results against the single-instance calls (1e-10, the bound of the other batch
tests), whichever route an instance takes, with 13-orbital instances among
them (which only groups serve); and a batch of sixty layouts takes no longer
than the persistent launch alone, within a third.
"""

from __future__ import annotations

import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _instances(cuts, spaces):
    from slowquant_amd import engine as E
    from slowquant_amd.synthetic import synthetic_hamiltonian
    from slowquant_amd.util import UpsStructure

    rng = np.random.default_rng(7)
    inst, thetas = [], []
    for n, na, nb in spaces:
        lay = UpsStructure()
        lay.create_tiled(n, {"n_layers": 3, "do_tups": True})
        sp = E.space_for(n, na, nb)
        for cut in cuts:
            m = lay.n_params - cut
            inst.append((sp, E.Program(sp, lay.excitation_operator_type[:m], lay.excitation_indices[:m]),
                         E.Hamiltonian(sp, *synthetic_hamiltonian(n, 2 * n, rng))))
            thetas.append(rng.normal(0.0, 0.1, m))
    return E, inst, thetas


@pytest.mark.parametrize("cuts,spaces", [
    (range(12), [(8, 4, 4)]),
    (range(5), [(8, 4, 4), (9, 4, 3), (13, 2, 2), (10, 5, 5), (6, 3, 3)]),
])
def test_many_layouts(cuts, spaces):
    from slowquant_amd.batch import loop_energy_grad

    E, inst, thetas = _instances(cuts, spaces)
    b = E.Batch(inst)
    e_ref, g_ref = loop_energy_grad(inst, thetas)
    for graph in (False, True, True):
        e, g = b.run(thetas, graph=graph)
        assert np.abs(np.asarray(e) - np.asarray(e_ref)).max() < 1e-10
        for x, y in zip(g, g_ref):
            assert np.abs(x - y).max() < 1e-10


def test_sixty_layouts_take_no_longer_than_the_persistent_launch(monkeypatch):
    import torch

    E, inst, thetas = _instances(range(60), [(8, 4, 4)])
    b = E.Batch(inst)
    monkeypatch.setenv("SQ_BATCH_GROUPS", "0")
    alone = E.Batch(inst)

    def best(x):
        t = []
        for _ in range(6):
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            x.run(thetas, graph=True)
            t.append(time.perf_counter() - t0)
        return min(t)

    assert best(b) < best(alone) * 4 / 3
