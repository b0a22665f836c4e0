"""The orbital gradient (k_kappa_grad, sq_orbital.hip) against numpy.einsum over
the full-space Gamma at sizes the loop restatement is slow for: fewer index
triples than a block has threads, one more than a multiple, many rounds of
triples, no inactive and no virtual orbitals, one kappa element and thousands.

Tolerance: 1e-12 relative to the largest element (sums of at most 4e4 terms).
"""

from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _full_gamma(ni, na, r1, r2):
    o = ni + na
    i, a = np.arange(ni), np.arange(ni, o)
    g1 = np.zeros((o, o))
    g1[i, i] = 2.0
    g1[ni:, ni:] = r1
    g2 = np.zeros((o,) * 4)
    g2[ni:, ni:, ni:, ni:] = r2
    for x in i:
        for y in i:
            g2[x, x, y, y] += 4.0
            g2[x, y, y, x] -= 2.0
        g2[np.ix_(a, a, [x], [x])] += 2.0 * r1[:, :, None, None]
        g2[np.ix_([x], [x], a, a)] += 2.0 * r1[None, None]
        g2[np.ix_([x], a, a, [x])] -= r1[None, :, :, None]
        g2[np.ix_(a, [x], [x], a)] -= r1[:, None, None, :]
    return g1, g2


@pytest.mark.parametrize("ni,na,nv,one", [(0, 2, 1, False), (3, 4, 2, True), (2, 6, 30, False), (10, 6, 4, False),
                                          (4, 12, 8, False), (0, 17, 0, False), (20, 12, 20, False)])
def test_orbital_gradient_against_einsum(ni, na, nv, one):
    from slowquant_amd import orbitals

    o, n = ni + na, ni + na + nv
    rng = np.random.default_rng(200 + n)
    h = rng.normal(size=(n, n))
    g = rng.normal(size=(n,) * 4)
    r1 = rng.normal(size=(na, na))
    r2 = rng.normal(size=(na,) * 4)
    idx = [(p, q) for p in range(n) for q in range(p + 1, n)]
    if one:
        idx = idx[-1:]
    G1, G2 = _full_gamma(ni, na, r1, r2)
    Y, V, Z, W = (np.zeros((n, n)) for _ in range(4))
    Y[:, :o] = h[:, :o] @ G1.T
    V[:, :o] = h[:o].T @ G1
    Z[:, :o] = g[:, :o, :o, :o].reshape(n, -1) @ G2.reshape(o, -1).T
    W[:, :o] = g[:o, :, :o, :o].transpose(1, 0, 2, 3).reshape(n, -1) @ G2.transpose(1, 0, 2, 3).reshape(o, -1).T
    m, k = np.asarray(idx).T
    expect = 2 * Y[k, m] - 2 * V[m, k] + Z[k, m] - W[m, k] - Z[m, k] + W[k, m]
    got = orbitals.orbital_gradient(h, g, idx, ni, na, r1, r2)
    assert np.abs(got - expect).max() < 1e-12 * max(1.0, np.abs(expect).max())
