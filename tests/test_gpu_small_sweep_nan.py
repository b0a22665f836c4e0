"""An amplitude that is not a number or infinite makes the energy and gradient of
the one-block sweep NaN, as the per-gate kernels do, for rotations (fUCCSD) and
polynomial gates (spin-adapted doubles), from host and from device amplitudes.
"""

from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sweep", ["0", "1"])
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
@pytest.mark.parametrize("types,idx", [
    (["single", "double", "single"], [(0, 4), (0, 1, 4, 5), (1, 7)]),
    (["sa_single", "sa_double_1", "sa_double_4"], [(0, 2), (0, 0, 2, 2), (0, 1, 2, 3)]),
])
def test_nan_amplitude(sweep, bad, types, idx, monkeypatch):
    import torch

    from slowquant_amd import engine as E
    from slowquant_amd.synthetic import synthetic_hamiltonian

    monkeypatch.setenv("SQ_SMALL_SWEEP", sweep)
    sp = E.Space(4, 2, 2)
    prog = E.Program(sp, types, idx)
    H = E.Hamiltonian(sp, *synthetic_hamiltonian(4, 8, np.random.default_rng(1)))
    psi0 = E.hf_state(sp)
    for k in range(len(types)):
        theta = np.array([0.1, -0.2, 0.3])
        theta[k] = bad
        for th in (theta, torch.tensor(theta, device="cuda")):
            e, g = prog.energy_grad(H, th, psi0)
            assert np.isnan(e) and np.isnan(g).any(), (k, e, g)
        assert torch.isnan(prog.state_prep(theta, psi0)).any()
