"""The one-electron terms of the orbital gradient with as many and more occupied
orbitals than a block of k_kappa_grad has threads (256): g vanishes, so the
gradient is 2 (h G1^T)[n][m] - 2 (h^T G1)[m][n] with the full-space Gamma1.

Tolerance: 1e-12 relative to the largest element (sums of at most 300 terms).
"""

from __future__ import annotations

import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ni,na", [(254, 2), (255, 2), (270, 3)])
def test_orbital_gradient_one_electron_terms(ni, na):
    import torch

    from slowquant_amd import _native as N

    o, n = ni + na, ni + na + 1
    if torch.cuda.mem_get_info()[0] < 10 * n**4:
        pytest.skip("the integrals do not fit the card")
    rng = np.random.default_rng(ni)
    h, r1 = rng.normal(size=(n, n)), rng.normal(size=(na, na))
    idx = np.array([(0, n - 1), (ni - 1, ni), (1, o - 1), (o - 1, n - 1), (n - 1, o - 1)], dtype=np.int32)
    G1 = np.zeros((n, n))
    G1[np.arange(ni), np.arange(ni)] = 2.0
    G1[ni:o, ni:o] = r1
    m, k = idx.T
    expect = 2.0 * (h @ G1.T)[k, m] - 2.0 * (h.T @ G1)[m, k]
    dev = [torch.as_tensor(x, device="cuda") for x in (h, r1, np.zeros((na,) * 4))]
    g = torch.zeros(n**4, dtype=torch.float64, device="cuda")
    work = torch.empty(2 * len(idx), dtype=torch.float64, device="cuda")
    got = np.zeros(len(idx))
    ptr = [ctypes.c_void_p(x.data_ptr()) for x in (dev[0], g, dev[1], dev[2])]
    N.check(N.lib().sq_orbital_gradient(n, ni, na, *ptr, len(idx), idx.ctypes.data, got.ctypes.data,
                                        ctypes.c_void_p(work.data_ptr()), torch.cuda.current_stream().cuda_stream))
    del g
    torch.cuda.empty_cache()
    assert np.abs(got - expect).max() < 1e-12 * np.abs(expect).max()
