"""sigma = H psi over the nonvanishing alpha excitations (k_sigma_rows_list and
k_string_gemm, sq_rowsigma.hip) against the fixed-order full contraction
(k_sigma_rows) of the same space: orbital counts around the 16-row tiles of
the pair index, empty, full and single-string spins (lists of no and of one
k-step), more and fewer beta strings than a wave's tiles, products in the row
launch and as a launch of their own, both with remainders, a core energy, and
groups of instances with unequal spins.

Tolerance: 1e-12 of max|sigma| (sums of at most 1e4 terms, each 1.1e-16 of the
largest, add to 1e-14 in the mean square), energies 1e-10.
"""

from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [
    (1, 1, 0),
    (2, 1, 1),
    (3, 0, 2),  # no alpha excitation at all
    (4, 4, 2),  # only diagonal ones
    (5, 2, 3),
    (6, 3, 0),
    (7, 3, 4),
    (8, 4, 4),
    (9, 2, 6),
    (10, 5, 5),
    (10, 9, 1),
    (11, 5, 6),
    (12, 6, 5),
    (13, 2, 4),  # six tiles of the pair index, products in the row launch
    (13, 4, 5),  # and as a launch of their own
    (14, 3, 4),
    (14, 6, 3),
    (16, 3, 2),  # two slices of A per block
]


@pytest.mark.parametrize("n,na,nb", CASES)
def test_list_form_against_fixed_order_form(n, na, nb):
    import torch

    from slowquant_amd import _native as N
    from slowquant_amd import engine as E
    from slowquant_amd.synthetic import synthetic_hamiltonian

    rng = np.random.default_rng(16 * n + na)
    h, g = synthetic_hamiltonian(n, 2 * n, rng)
    sp = E.Space(n, na, nb)
    H = E.Hamiltonian(sp, h, g, e_core=-0.75)
    psi = torch.tensor(rng.normal(size=sp.dim), dtype=torch.float64, device="cuda")
    psi /= torch.linalg.norm(psi)
    got = {}
    for det in (0, 1):
        N.check(N.lib().sq_sigma_configure(sp.handle, 0, 0, det))
        got[det] = H.sigma(psi)
    for rows, split in ((1, 1), (3, 3)):
        N.check(N.lib().sq_sigma_configure(sp.handle, rows, split, 0))
        got[rows, split] = H.sigma(psi)
    ref, e_ref = got.pop(1)
    scale = max(1.0, float(ref.abs().max()))
    for key, (sig, e) in got.items():
        assert float((sig - ref).abs().max()) < 1e-12 * scale, key
        assert abs(e - e_ref) < 1e-10, key


def test_grouped_instances_of_unequal_spins():
    from slowquant_amd import engine as E
    from slowquant_amd.batch import InstanceSpec, build_instances, loop_energy_grad

    specs = [InstanceSpec(10, 5, 4, 2, 40 + i) for i in range(3)]
    inst, thetas = build_instances(specs)
    e_ref, g_ref = loop_energy_grad(inst, thetas)
    e, g = E.Batch(inst).run(thetas)
    assert np.abs(np.asarray(e) - np.asarray(e_ref)).max() < 1e-10
    for a, b in zip(g, g_ref):
        assert np.abs(a - b).max() < 1e-10
