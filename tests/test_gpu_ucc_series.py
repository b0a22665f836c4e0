"""The merged sparsity pattern and the series over it (sq_ucc.hip) against the
kernels that rescan the terms (SQ_UCC_CSR=0), where rows are empty, short or
longer than a wave, where the exponential takes one Taylor series, one
Chebyshev series with 8, 12 or 16 nodes, or several intervals, and at theta = 0.

Tolerances: both sides sum the same series with rounding errors of about
nu * 1e-16 per amplitude (nu up to 40 here): 1e-12 on states; gradients are
quadratures bounded to 1e-13 relative on either side: 1e-10.
"""

from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [
    # n, na, nb, excitations, width of theta
    (2, 1, 1, "SD", 0.1),
    (4, 2, 2, "SD", 0.0),  # T = 0
    (4, 1, 1, "S", 0.3),
    (5, 2, 2, "SDTQ", 0.05),
    (6, 3, 3, "SD", 0.02),  # one Taylor series
    (6, 3, 3, "SD", 0.15),
    (6, 3, 3, "SD", 0.4),
    (6, 3, 3, "SDTQ56", 0.1),
    (6, 2, 2, "SD", 2.0),  # several intervals
    (7, 3, 3, "SD", 0.08),
    (8, 4, 4, "SDT", 0.02),
]


def _program(E, sp, n, na, exc):
    from slowquant_amd.util import UccStructure

    lay = UccStructure()
    occ, unocc = list(range(na)), list(range(na, n))
    occ_s, unocc_s = list(range(2 * na)), list(range(2 * na, 2 * n))
    for c in exc:
        if c == "S":
            lay.add_sa_singles(occ, unocc)
        elif c == "D":
            lay.add_sa_doubles(occ, unocc)
        else:
            {"T": lay.add_triples, "Q": lay.add_quadruples, "5": lay.add_quintuples,
             "6": lay.add_sextuples}[c](occ_s, unocc_s)
    types = ["sa_single_ucc" if t == "sa_single" else t for t in lay.excitation_operator_type]
    return E.Program(sp, types, lay.excitation_indices), lay.n_params


@pytest.mark.parametrize("n,na,nb,exc,width", CASES)
def test_series_against_term_scan(n, na, nb, exc, width, monkeypatch):
    import torch

    from slowquant_amd import engine as E
    from slowquant_amd.synthetic import synthetic_hamiltonian

    rng = np.random.default_rng(n)
    h, g = synthetic_hamiltonian(n, 2 * n, rng)
    sp = E.Space(n, na, nb)
    H = E.Hamiltonian(sp, h, g)
    v = rng.normal(size=sp.dim)
    x = torch.tensor(v / np.linalg.norm(v), device="cuda")
    got = []
    for flag in ("1", "0"):
        monkeypatch.setenv("SQ_UCC_CSR", flag)
        prog, n_theta = _program(E, sp, n, na, exc)
        th = np.random.default_rng(7).normal(0.0, width, n_theta)
        states = [E.ucc_expm(prog, th, x, t) for t in (1.0, -0.7)]
        e, grad = E.ucc_energy_grad(prog, H, th, x)
        e_only, none = E.ucc_energy_grad(prog, H, th, x, want_grad=False)
        assert none is None and abs(e - e_only) < 1e-11
        got.append((states, e, grad))
    for a, b in zip(got[0][0], got[1][0]):
        assert float((a - b).abs().max()) < 1e-12
    assert abs(got[0][1] - got[1][1]) < 1e-10
    assert np.abs(got[0][2] - got[1][2]).max() < 1e-10
