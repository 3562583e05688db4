"""The tiles of a batch's Rusanov step, and what the tile search does for the
AUSM step, which is the same under each of them."""
from __future__ import annotations

import pytest

from gitm_amd import synth
from tests.test_gpu_batch import members

pytestmark = pytest.mark.gpu


def test_autotune_leaves_the_automatic_tile_for_ausm(solver):
    from gitm_amd import vertical
    b = vertical.VerticalBatch(solver, [vertical.to_device(c) for c in members()])
    automatic = b.tile()
    b.set_tile((4, 4, 0, 0))
    times = b.autotune(synth.StepParams(), "ausm", probe_columns=300)
    assert b.tile() == automatic
    assert len(times) == 32 and len(set(times.values())) == 1
    times = b.autotune(synth.StepParams(), "rusanov", probe_columns=300)
    assert len(times) == 32 and len(set(times.values())) > 1
    assert b.tile() == min(times, key=times.get)
    b.close()
