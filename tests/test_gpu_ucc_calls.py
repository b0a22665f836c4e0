"""Calls of the UCC routines in sequence on one program: the block counters and
the pinned result block of the pattern (sq_ucc.hip) serve every next call, the
sigma that writes into the series' first vector alternates with the one that
does not, energies without gradients and plain exponentials come between.  Each
result against a fresh program's; two threads share one program.

Tolerance: 1e-12 (energy), 1e-10 (gradient): the same sums in the same order
but for the gate sums' atomic adds.
"""

from __future__ import annotations

import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _problem(n, na):
    from slowquant_amd import engine as E
    from slowquant_amd.synthetic import synthetic_hamiltonian
    from slowquant_amd.util import UccStructure

    lay = UccStructure()
    occ, unocc = list(range(na)), list(range(na, n))
    lay.add_sa_singles(occ, unocc)
    lay.add_sa_doubles(occ, unocc)
    types = ["sa_single_ucc" if t == "sa_single" else t for t in lay.excitation_operator_type]
    h, g = synthetic_hamiltonian(n, 2 * n, np.random.default_rng(n))
    sp = E.Space(n, na, na)
    return E, sp, lambda: E.Program(sp, types, lay.excitation_indices), E.Hamiltonian(sp, h, g, e_core=0.25)


# one element per row at most, short rows (16 lanes), longer ones (32 lanes)
@pytest.mark.parametrize("n,na", [(2, 1), (4, 2), (8, 4)])
def test_sequence_of_calls(n, na):
    E, sp, program, H = _problem(n, na)
    prog = program()
    psi0 = E.hf_state(sp)
    rng = np.random.default_rng(3)
    for width in (0.05, 2.5, 0.0, 0.4, 0.05):  # Taylor, several intervals, T = 0, Chebyshev
        th = rng.normal(0.0, width, prog.n_gates)
        e, g = E.ucc_energy_grad(prog, H, th, psi0)
        e1, none = E.ucc_energy_grad(prog, H, th, psi0, want_grad=False)
        psi = E.ucc_expm(prog, th, psi0)
        e2, g2 = E.ucc_energy_grad(prog, H, th, psi0)
        e_ref, g_ref = E.ucc_energy_grad(program(), H, th, psi0)
        _, e_sig = H.sigma(psi)
        assert none is None
        for x in (e, e1, e2, e_sig):
            assert abs(x - e_ref) < 1e-12 * max(1.0, abs(e_ref))
        assert np.abs(g - g_ref).max() < 1e-10 and np.abs(g2 - g_ref).max() < 1e-10


def test_two_threads_share_a_program():
    import torch

    E, sp, program, H = _problem(6, 3)
    prog = program()
    psi0 = E.hf_state(sp)
    thetas = np.random.default_rng(5).normal(0.0, 0.1, (2, prog.n_gates))
    refs = [E.ucc_energy_grad(program(), H, th, psi0) for th in thetas]
    devs = [torch.tensor(th, device="cuda") for th in thetas]
    torch.cuda.synchronize()
    errors = []

    def work(k):
        try:
            import ctypes

            from slowquant_amd import _native as N

            buf = torch.empty(int(N.lib().sq_ucc_work_bytes(sp.handle, prog.handle)) // 8, dtype=torch.float64,
                              device="cuda")
            s = torch.cuda.Stream()
            e, g = ctypes.c_double(), np.zeros(prog.n_gates)
            torch.cuda.synchronize()
            for _ in range(20):
                N.check(N.lib().sq_ucc_energy_grad(sp.handle, prog.handle, H.handle, devs[k].data_ptr(),
                                                   psi0.data_ptr(), ctypes.byref(e), g.ctypes.data, buf.data_ptr(),
                                                   s.cuda_stream))
                assert abs(e.value - refs[k][0]) < 1e-12 and np.abs(g - refs[k][1]).max() < 1e-10
        except Exception as exc:  # noqa: BLE001 (reported by the main thread)
            errors.append(exc)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
