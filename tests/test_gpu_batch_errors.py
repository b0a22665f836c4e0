"""Arguments a batch refuses on the host, before any launch."""

from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_batch_errors():
    from slowquant_amd import engine as E
    from slowquant_amd.batch import InstanceSpec, build_instances

    inst, _ = build_instances([InstanceSpec(4, 2, 2, 1, 11)])
    b = E.Batch(inst, 1)
    with pytest.raises(ValueError):
        b.set_theta(np.zeros(b.n_params + 1))
    sp, _, H = inst[0]
    # polynomial (sa_double_2) gates are not rotations
    with pytest.raises(ValueError):
        E.Batch([(sp, E.Program(sp, ["sa_double_2"], [(0, 1, 2, 3)]), H)], 1)
