"""sigma of the largest spaces that the row path takes (15 orbitals with 5005 and
6435 beta strings, 16 with 8008) against the space with its spins exchanged:
the matrix of sigma transposed, from the matrix of psi transposed (the constant
sign of the exchange drops out).  The two take the excitation lists and the
partner tables of each other's spin, and other tiles.  sigma also keeps the
eigenvalues of a diagonal Hamiltonian.

Tolerance: 1e-12 relative to sigma's largest element (sums of some 1e4 terms).
"""

from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _problem(n, diagonal):
    from slowquant_amd.synthetic import synthetic_hamiltonian

    h, g = synthetic_hamiltonian(n, 2 * n, np.random.default_rng(n))
    if diagonal:
        p = np.arange(n)
        d = np.zeros_like(g)
        d[p[:, None], p[:, None], p, p] = g[p[:, None], p[:, None], p, p]
        h, g = np.diag(np.diag(h)), d
    return h, g


@pytest.mark.parametrize("n,na,nb", [(15, 5, 7), (15, 6, 8), (15, 7, 7), (16, 10, 6)])
def test_spin_exchange(n, na, nb):
    import torch

    from slowquant_amd import engine as E

    h, g = _problem(n, False)
    one, two = E.Space(n, na, nb), E.Space(n, nb, na)
    v = torch.randn(one.dim, dtype=torch.float64, device="cuda", generator=torch.Generator("cuda").manual_seed(n))
    shape = (one.n_alpha_strings, one.n_beta_strings)
    s, e = E.Hamiltonian(one, h, g, 0.7).sigma(v)
    one.__dict__["_work"].clear()
    t, f = E.Hamiltonian(two, h, g, 0.7).sigma(v.reshape(shape).T.contiguous().reshape(-1))
    scale = float(s.abs().max())
    d = s.reshape(shape) - t.reshape(shape[::-1]).T
    assert float(d.abs().max()) < 1e-12 * scale
    assert abs(e - f) < 1e-12 * abs(e) * 100 and abs(e - float((v * s).sum())) < 1e-10 * abs(e)


@pytest.mark.parametrize("n,na,nb", [(15, 5, 7), (16, 6, 6)])
def test_diagonal_hamiltonian(n, na, nb):
    import torch

    from slowquant_amd import engine as E

    h, g = _problem(n, True)
    sp = E.Space(n, na, nb)
    a, b = (torch.as_tensor(np.asarray(x).astype(np.int64), device="cuda") for x in sp.strings())
    occ_a, occ_b = (((x[:, None] >> torch.arange(n, device="cuda")) & 1).double() for x in (a, b))
    hd = torch.as_tensor(np.diag(h).copy(), device="cuda")
    gd = torch.as_tensor(np.einsum("ppqq->pq", g).copy(), device="cuda")
    # sum_p h_pp n_p + 1/2 sum_pq g_ppqq (n_p n_q - delta_pq n_p), n = n_alpha + n_beta
    one = hd - 0.5 * torch.diag(gd)
    diag = (occ_a @ one + 0.5 * ((occ_a @ gd) * occ_a).sum(1))[:, None] + (
        occ_b @ one + 0.5 * ((occ_b @ gd) * occ_b).sum(1))[None] + occ_a @ gd @ occ_b.T
    v = torch.randn(sp.dim, dtype=torch.float64, device="cuda", generator=torch.Generator("cuda").manual_seed(n))
    s, _ = E.Hamiltonian(sp, h, g).sigma(v)
    expect = diag.reshape(-1) * v
    assert float((s - expect).abs().max()) < 1e-12 * float(expect.abs().max())
