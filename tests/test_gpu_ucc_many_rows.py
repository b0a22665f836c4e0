"""Unfactorised UCC above 2^24 determinants: the exponential of one alpha single
excitation on a random state against the rotation kernel of the same gate.

Tolerance: 1e-13 relative to the largest amplitude (about twenty terms).
"""

from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_one_excitation_of_many_determinants():
    import torch

    from slowquant_amd import engine as E

    sp = E.Space(16, 5, 5)
    assert sp.dim > 1 << 24
    prog = E.Program(sp, ["single"], [(8, 10)])  # alpha of orbital 4 to alpha of orbital 5
    v = torch.randn(sp.dim, dtype=torch.float64, device="cuda", generator=torch.Generator("cuda").manual_seed(1))
    for theta in (0.3, -1.2):
        got = E.ucc_expm(prog, np.array([theta]), v)
        expect = prog.state_prep(np.array([theta]), v)
        assert float((expect - v).abs().max()) > 0.1
        assert float((got - expect).abs().max()) < 1e-13 * float(v.abs().max())
