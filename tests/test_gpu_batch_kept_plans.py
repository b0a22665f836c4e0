"""Batched instances of fewer than 16384 determinants that run in groups: a later
change of their programs' tile shape or their space's sigma shape, and the end
of the programs, leave the batch's results alone, eager and replayed (the
persistent launch, which serves such instances too, depends on neither).

Tolerance: 1e-10, the bound of the other batch tests.
"""

from __future__ import annotations

import gc

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _batch():
    from slowquant_amd import engine as E
    from slowquant_amd.batch import InstanceSpec, build_instances, loop_energy_grad

    specs = [InstanceSpec(n, na, nb, layers, 500 + k)
             for k, (n, na, nb, layers) in enumerate([(8, 4, 4, 1), (9, 5, 4, 2), (8, 4, 4, 1), (8, 4, 4, 2)])]
    inst, thetas = build_instances(specs)
    return E.Batch(inst), inst, thetas, loop_energy_grad(inst, thetas)


def _check(b, thetas, ref, graph):
    e, g = b.run(thetas, graph=graph)
    assert np.abs(np.asarray(e) - np.asarray(ref[0])).max() < 1e-10
    for x, y in zip(g, ref[1]):
        assert np.abs(x - y).max() < 1e-10


@pytest.mark.parametrize("first", [False, True])
def test_shape_changes(first):
    b, inst, thetas, ref = _batch()
    if first:  # with a captured graph
        _check(b, thetas, ref, True)
    spaces = {id(s): s for s, _, _ in inst}.values()
    try:
        for _, p, _ in inst:
            p.set_tile_shape(512, 256)
        for rows, nsplit, det in ((4, 1, 0), (1, 3, 1), (0, 0, -1)):
            for s in spaces:
                s.configure_sigma(rows, nsplit, det)
            for graph in (True, False, True):
                _check(b, thetas, ref, graph)
    finally:
        for s in spaces:
            s.configure_sigma(0, 0, -1)


def test_programs_end():
    import torch

    b, inst, thetas, ref = _batch()
    _check(b, thetas, ref, True)
    b.instances = [(s, None, None) for s, _, _ in inst]
    del inst
    gc.collect()
    keep = [torch.full((1 << k,), float("nan"), dtype=torch.float64, device="cuda") for k in range(8, 20)]
    for graph in (True, False, True):
        _check(b, thetas, ref, graph)
    del keep
