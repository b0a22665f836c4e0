"""RDMs from their spin parts (sq_rdm.hip) against the Gram matrix of the rows
E_pq psi formed with index arithmetic in torch: orbital counts around the
16-row tiles of the excitation lists and pairs, one and several groups of pair
tiles, empty, full and single-string spins, rows shorter than one column block
and with every remainder class, the longest row (3432 strings), rows in whole
rounds of blocks, fewer rows than blocks and rows cut into ranges; a second
call gives the same bits.

Tolerance: 1e-12 (elements of order 1 to 10, sums of at most 1e6 products of a
unit vector's amplitudes: 1e-14 in the mean square).
"""

from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [
    (1, 1, 0),
    (1, 1, 1),
    (2, 1, 1),
    (3, 0, 2),
    (4, 4, 2),
    (5, 2, 3),
    (6, 3, 0),
    (6, 3, 3),
    (7, 3, 4),
    (8, 4, 4),
    (9, 2, 6),
    (10, 5, 5),  # 252 rows on 252 blocks
    (11, 6, 3),  # 462 rows, the last 206 in ranges
    (12, 10, 2),
    (12, 6, 1),
    (13, 7, 2),  # four tiles of listed excitations, two groups of pair tiles
    (14, 2, 7),
    (14, 7, 1),
    (14, 3, 3),
]


def _images(n, strings):
    """E_pq on every string: target index (-1: none) and sign, [p][q][s]."""
    index = {int(s): i for i, s in enumerate(strings)}
    tgt = -np.ones((n, n, len(strings)), dtype=np.int64)
    sgn = np.zeros((n, n, len(strings)))
    for i, s in enumerate(int(x) for x in strings):
        for q in range(n):
            if not s >> q & 1:
                continue
            m = s & ~(1 << q)
            for p in range(n):
                if m >> p & 1:
                    continue
                between = m & ((1 << max(p, q)) - 1) & ~((1 << (min(p, q) + 1)) - 1)
                tgt[p, q, i] = index[m | 1 << p]
                sgn[p, q, i] = -1.0 if bin(between).count("1") & 1 else 1.0
    return tgt, sgn


@pytest.mark.parametrize("n,na,nb", CASES)
def test_rdms_against_gram_matrix(n, na, nb):
    import torch

    from slowquant_amd import engine as E

    sp = E.Space(n, na, nb)
    a, b = (np.asarray(x) for x in sp.strings())
    psi = torch.tensor(np.random.default_rng(20 * n + na).normal(size=sp.dim), device="cuda")
    psi /= torch.linalg.norm(psi)
    C = psi.reshape(len(a), len(b))
    (ta, sa), (tb, sb) = _images(n, a), _images(n, b)
    D = torch.zeros(n * n, len(a), len(b), dtype=torch.float64, device="cuda")
    for p in range(n):
        for q in range(n):
            for t, s, axis in ((ta[p, q], sa[p, q], 0), (tb[p, q], sb[p, q], 1)):
                src = np.flatnonzero(t >= 0)
                if len(src) == 0:
                    continue
                shape = (-1, 1) if axis == 0 else (1, -1)
                w = torch.tensor(s[src], device="cuda").reshape(shape)
                i = torch.tensor(src, device="cuda")
                j = torch.tensor(t[src], device="cuda")
                D[p * n + q].index_add_(axis, j, C.index_select(axis, i) * w)
    D = D.reshape(n * n, -1)
    M = (D @ D.T).reshape(n, n, n, n).cpu().numpy()
    r1 = (D @ psi).reshape(n, n).cpu().numpy()
    r2 = np.einsum("qprs->pqrs", M) - np.einsum("qr,ps->pqrs", np.eye(n), r1)
    g1, g2 = E.rdm12(sp, psi)
    assert np.abs(g1 - r1).max() < 1e-12
    assert np.abs(g2 - r2).max() < 1e-12
    h1, h2 = E.rdm12(sp, psi)
    assert np.array_equal(g1, h1) and np.array_equal(g2, h2)
