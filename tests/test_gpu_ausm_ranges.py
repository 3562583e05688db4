"""The AUSM step at the ends of what it accepts, against the oracle within the
step's parity bar, 1e-11: time steps of zero (a batch member's, from the prep at
the end of the run) and far below a second; a species, or all of them, in
densities whose masses, products or reciprocals come near the ends of the double
range."""
from __future__ import annotations

import dataclasses
import os

import numpy as np
import pytest

from gitm_amd import synth
from oracle import cpu
from tests.helpers import assert_parity, subset

pytestmark = pytest.mark.gpu

THREADS = min(16, os.cpu_count() or 1)


def columns(n_alts, seed, ions=False):
    return subset(synth.make_columns(synth.GridSpec(1, 1, n_alts), seed=seed, ions=ions),
                  list(range(0, 81, 16)))


@pytest.mark.parametrize("ions", [False, True])
def test_steps_of_zero(solver, ions):
    import torch
    from gitm_amd import vertical
    dts = [2.0, 0.0, 5e-310, 1e-305, 1e-90, 0.5]
    cols = [columns((50, 61)[i % 2], 30 + i, ions) for i in range(len(dts))]
    p = synth.StepParams(use_ion_advection=ions)
    dev = [vertical.to_device(c) for c in cols]
    b = vertical.VerticalBatch(solver, dev, ions=ions)
    print(f"batch, steps {dts}, ions {ions}", flush=True)
    b.advance(p, "ausm", 1, dt=torch.tensor(dts, dtype=torch.float64, device="cuda"))
    for d, c, dt in zip(dev, cols, dts):
        ref = cpu.advance(c, dataclasses.replace(p, dt=dt), solver=1, threads=THREADS)
        assert_parity(vertical.to_host(d), ref, 1e-11, what=f"dt {dt}")
    b.close()


@pytest.mark.parametrize("dt", [5e-310, 1e-300, 1e-12])
def test_short_steps(solver, dt):
    from gitm_amd import vertical
    cols = columns(50, 41)
    p = synth.StepParams(dt=dt)
    d = vertical.to_device(cols)
    print(f"dt {dt}", flush=True)
    solver.advance(d, p, "ausm", 1)
    assert_parity(vertical.to_host(d), cpu.advance(cols, p, solver=1, threads=THREADS), 1e-11,
                  what=f"dt {dt}")


@pytest.mark.parametrize("species,factor", [(0, 1e-250), (0, 1e-290), (0, 1e-300), (5, 1e-300),
                                            (None, 1e-290), (None, 1e-200), (None, 1e100),
                                            (None, 1e140), (None, 1e200), (None, 1e250)])
def test_densities_far_from_one(solver, species, factor):
    """1e-300 of a species leaves mass densities of 1e-309; 1e140 of all gives
    products of two densities beyond 1e308."""
    from gitm_amd import vertical
    cols = columns(50, 42)
    odd = np.arange(cols["temp"].shape[0]) % 2 == 1
    if species is None:
        cols["nds"][odd] *= factor
        cols["rho"][odd] *= factor
    else:
        cols["nds"][odd, species] *= factor
    p = synth.StepParams()
    with np.errstate(all="ignore"):
        ref = cpu.advance(cols, p, solver=1, threads=THREADS)
    d = vertical.to_device(cols)
    print(f"species {species} x {factor}", flush=True)
    solver.advance(d, p, "ausm", 1)
    assert_parity(vertical.to_host(d), ref, 1e-11, what=f"species {species} x {factor}")
