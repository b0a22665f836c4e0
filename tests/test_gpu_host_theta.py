"""Energy and gradient from host parameters (sq_energy_grad_adjoint_host: theta
read from and results written to pinned memory, sigma zeroed and the energy
summed inside the first and last launch) against the device-parameter entry
point and the separate state, sigma and reverse calls, on every route of the
adjoint: brick-wall programs whose sigma adds into a zeroed vector or writes
it, the one-block sweep, brick walls with a gate no window holds, programs of
such gates only, and no gate at all.  Other parameters on the same program
follow, and two threads with a program and a stream each.

Tolerance: 1e-12 (energy) and 1e-10 (gradient), the engine's parity bounds.
"""

from __future__ import annotations

import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [
    (4, 2, 2, "tups"),
    (8, 4, 4, "tups"),
    (9, 4, 5, "tups"),
    (14, 4, 3, "tups"),  # sigma written, not added
    (5, 2, 3, "lone"),  # one-block sweep
    (9, 4, 5, "mixed"),
    (9, 4, 5, "lone"),
    (4, 2, 2, "empty"),
]


def _problem(n, na, nb, kind):
    from slowquant_amd import engine as E
    from slowquant_amd.synthetic import synthetic_hamiltonian
    from slowquant_amd.util import UpsStructure

    types, idx = [], []
    if kind in ("tups", "mixed"):
        lay = UpsStructure()
        lay.create_tiled(n, {"n_layers": 2, "do_tups": True})
        types, idx = list(lay.excitation_operator_type), list(lay.excitation_indices)
    if kind in ("lone", "mixed"):
        types += ["single", "double"]
        idx += [(0, 2 * (n - 1)), (0, 1, 2 * (n - 1), 2 * n - 1)]
    rng = np.random.default_rng(10 * n + na)
    h, g = synthetic_hamiltonian(n, 2 * n, rng)
    sp = E.Space(n, na, nb)
    return sp, E.Program(sp, types, idx), E.Hamiltonian(sp, h, g, e_core=0.5), rng


def _check(sp, prog, H, th):
    import torch

    from slowquant_amd import engine as E

    psi0 = E.hf_state(sp)
    dev = torch.tensor(th, dtype=torch.float64, device="cuda")
    e, g = prog.energy_grad(H, th, psi0)
    e_dev, g_dev = prog.energy_grad(H, dev, psi0)
    psi = prog.state_prep(dev, psi0)
    lam, e_sig = H.sigma(psi)
    g_rev = prog.adjoint_reverse(dev, psi, lam)
    assert abs(e - e_dev) < 1e-12 * max(1.0, abs(e)) and abs(e - e_sig) < 1e-12 * max(1.0, abs(e))
    assert g.shape == g_dev.shape == (len(th),)
    if len(th):
        assert np.abs(g - g_dev).max() < 1e-10
        assert np.abs(g - g_rev).max() < 1e-10


@pytest.mark.parametrize("n,na,nb,kind", CASES)
def test_host_parameters(n, na, nb, kind):
    sp, prog, H, rng = _problem(n, na, nb, kind)
    for _ in range(3):
        _check(sp, prog, H, rng.normal(0.0, 0.4, prog.n_gates))
    with pytest.raises(ValueError):
        from slowquant_amd import engine as E

        prog.energy_grad(H, np.zeros(prog.n_gates + 1), E.hf_state(sp))


def test_host_parameters_two_threads():
    import torch

    problems = [_problem(8, 4, 4, "tups"), _problem(8, 4, 4, "tups")]
    errors = []

    def work(k):
        try:
            sp, prog, H, _ = problems[k]
            rng = np.random.default_rng(k)
            with torch.cuda.stream(torch.cuda.Stream()):
                for _ in range(10):
                    _check(sp, prog, H, rng.normal(0.0, 0.4, prog.n_gates))
        except Exception as exc:  # noqa: BLE001 (reported by the main thread)
            errors.append(exc)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
