"""The autotuner can keep the automatic shapes: with every other shape slower, or
a sigma that is faster alone but makes whole evaluations slower, it chooses
them, and a shape that is faster in whole evaluations replaces them.  The
engine's calls are stood in for by their times.
"""

from __future__ import annotations

import types

import pytest


class _Engine:
    """Times of an evaluation and of sigma alone by (target, threads, rows, split)."""

    def __init__(self, evaluation, sigma):
        self.shape = [0, 0, 0, 0]
        self.times = {"evaluation": evaluation, "sigma": sigma}
        self.last = None
        self.types, self.indices = ["sa_single"], [(0, 1)]
        self.n_orb = self.n_alpha = self.n_beta = 2

    def set_tile_shape(self, target=0, threads=0):
        self.shape[:2] = target, threads

    def configure_sigma(self, rows=0, nsplit=0, deterministic=-1):
        self.shape[2:] = rows, nsplit

    def energy_grad(self, *args):
        self.last = self.times["evaluation"](*self.shape)

    def sigma(self, *args, **kw):
        self.last = self.times["sigma"](*self.shape)

    def state_prep(self, *args):
        return None


CASES = [
    # whole evaluation, sigma alone, choice
    (lambda t, n, r, s: 1.0 + (t > 0) + (n > 0) + (r > 0) + (s > 0), lambda t, n, r, s: 1.0 + (r > 0) + (s > 0), (0, 0, 0, 0)),
    (lambda t, n, r, s: 1.0 + (n > 0) + (s == 4), lambda t, n, r, s: 1.0 - 0.5 * (s == 4), (0, 0, 0, 0)),
    (lambda t, n, r, s: 1.0 - 0.1 * (t == 2048) - 0.1 * (n == 256) - 0.1 * (r == 3), lambda t, n, r, s: 1.0 - 0.1 * (r == 3),
     (2048, 256, 3, 0)),
]


@pytest.mark.parametrize("evaluation,sigma,expect", CASES)
def test_default_shapes_are_candidates(evaluation, sigma, expect, monkeypatch):
    from slowquant_amd import autotune

    eng = _Engine(evaluation, sigma)

    def timed(fn, reps):
        fn()
        return eng.last

    monkeypatch.setattr(autotune, "_time", timed)
    monkeypatch.setattr(autotune, "program_key", lambda space, prog: "key")
    choice = autotune.tune(eng, eng, types.SimpleNamespace(sigma=eng.sigma), [0.1], None, use_cache=False)
    got = tuple(choice[k] for k in ("tile_target", "tile_threads", "rows_per_block", "nsplit"))
    assert got == expect and tuple(eng.shape) == expect
