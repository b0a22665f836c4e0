"""The first calls of two threads on one program take the same route: both
states equal a later call's bit for bit (the one-block sweep and the per-gate
kernels differ in rounding).
"""

from __future__ import annotations

import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_first_calls_of_two_threads():
    import torch

    from slowquant_amd import engine as E
    from slowquant_amd.util import UpsStructure

    lay = UpsStructure()
    occ = sorted(2 * p + s for p in range(4) for s in (0, 1))
    lay.create_fUCC(list(range(4)), list(range(4, 8)), occ, [s for s in range(16) if s not in occ], 8,
                    {"n_layers": 1, "S": True, "D": True})
    sp = E.Space(8, 4, 4)
    theta = torch.tensor(np.random.default_rng(0).normal(0.0, 0.3, lay.n_params), device="cuda")
    psi0 = E.hf_state(sp)
    sp.work(0)
    for _ in range(5):
        prog = E.Program(sp, lay.excitation_operator_type, lay.excitation_indices)
        out = [torch.empty_like(psi0) for _ in range(2)]
        torch.cuda.synchronize()
        gate = threading.Barrier(2)

        def call(k):
            gate.wait()
            prog.state_prep(theta, psi0, out=out[k])

        threads = [threading.Thread(target=call, args=(k,)) for k in range(2)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        torch.cuda.synchronize()
        later = prog.state_prep(theta, psi0)
        assert torch.equal(out[0], later) and torch.equal(out[1], later)
