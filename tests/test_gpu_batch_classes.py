"""The launches of a batch's AUSM step: one per class of column heights, with the
bits that each member has alone; members whose columns have ions and are
too tall for the kernel that splits a level over the species take one launch
together, not one each."""
from __future__ import annotations

import numpy as np
import pytest

from gitm_amd import synth
from tests.helpers import subset

pytestmark = pytest.mark.gpu

STATE = ("nds", "vvel", "vel", "temp", "rho", "ions")


def members(heights, columns, ions):
    return [subset(synth.make_columns(synth.GridSpec(1, 1, na), seed=80 + i, ions=ions),
                   list(range(columns))) for i, na in enumerate(heights)]


def same_as_alone(solver, cols, dev, params, dts=None):
    import dataclasses
    from gitm_amd import vertical
    for i, c in enumerate(cols):
        d = vertical.to_device(c)
        p = params if dts is None else dataclasses.replace(params, dt=dts[i])
        solver.advance(d, p, "ausm", 1)
        a, r = vertical.to_host(dev[i]), vertical.to_host(d)
        for k in STATE:
            if k in r:
                assert np.array_equal(a[k], r[k]), f"member {i}: {k}"


def test_tall_ion_members(solver):
    import torch
    from gitm_amd import vertical
    heights = [227, 50, 252, 240, 61, 252, 231, 250]
    dts = [2.0, 1.0, 0.5, 1.5, 2.0, 1.0, 0.25, 2.0]
    cols = members(heights, 5, True)
    dev = [vertical.to_device(c) for c in cols]
    p = synth.StepParams(use_ion_advection=True)
    b = vertical.VerticalBatch(solver, dev, ions=True)
    dt = torch.tensor(dts, dtype=torch.float64, device="cuda")
    for tile in (None, (4, 4, 0, 0), (4, 1, 2, 0)):  # each lays the carries out anew
        b.set_tile(tile)
        for d, c in zip(dev, cols):
            for k in STATE:
                d[k].copy_(torch.from_numpy(c[k]))
        print("tile", tile, flush=True)
        b.advance(p, "ausm", 1, dt=dt)
        same_as_alone(solver, cols, dev, p, dts)
    b.close()


def test_tall_ion_members_run_side_by_side(solver):
    """Sixteen members of nine columns leave 112 CUs idle: together they take
    about as long as one of them, not sixteen times as long (the bar: four)."""
    import torch
    from gitm_amd import vertical
    cols = members([252] * 16, 9, True)
    p = synth.StepParams(use_ion_advection=True)

    def ms(which):
        dev = [vertical.to_device(c) for c in which]
        b = vertical.VerticalBatch(solver, dev, ions=True)
        times = []
        for _ in range(7):
            e0, e1 = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            e0.record()
            b.advance(p, "ausm", 1, check=False)
            e1.record()
            torch.cuda.synchronize()
            times.append(e0.elapsed_time(e1))
        b.check()
        b.close()
        return sorted(times)[3]

    one, all_ = ms(cols[:1]), ms(cols)
    print(f"one member {one:.3f} ms, sixteen {all_:.3f} ms", flush=True)
    assert all_ < 4.0 * one


@pytest.mark.parametrize("ions", [False, True])
def test_height_classes(solver, ions):
    """Enough columns of 150 and of 100 levels to fill the chip twice: they and
    the 50-level members are launches of their own, the second with a member of
    fewer wavefronts than its workgroups hold; each member with its own step."""
    import torch
    from gitm_amd import vertical
    n_cu = torch.cuda.get_device_properties(0).multi_processor_count
    tall = -(-2 * n_cu // 81) + 1  # members' blocks of 81 columns
    layout = [(50, 1), (150, tall), (61, 1), (100, 2 * tall), (20, 1), (12, 1)]
    cols = [synth.make_columns(synth.GridSpec(nb, 1, na), seed=90 + i, ions=ions)
            for i, (na, nb) in enumerate(layout)]
    dts = [2.0, 1.5, 0.5, 1.0, 2.0, 0.25]
    dev = [vertical.to_device(c) for c in cols]
    b = vertical.VerticalBatch(solver, dev, ions=ions)
    p = synth.StepParams(use_ion_advection=ions)
    print(f"classes, ions {ions}", flush=True)
    b.advance(p, "ausm", 1, dt=torch.tensor(dts, dtype=torch.float64, device="cuda"))
    same_as_alone(solver, cols, dev, p, dts)
    b.close()
