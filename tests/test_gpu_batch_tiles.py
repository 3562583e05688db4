"""The tiles of a batch's Rusanov step, and what the tile search does for the
AUSM step, which is the same under each of them."""
from __future__ import annotations

import pytest

from gitm_amd import synth
from tests.test_gpu_batch import members, run_tiles

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


@pytest.mark.parametrize("ions", [False, True])
def test_every_tile_of_the_rusanov_step(solver, ions):
    """Workgroups of 2, 3 or 4 wavefronts, 1..4 short columns per workgroup,
    carries in LDS or in device memory, one workgroup per task or a persistent
    grid: each tile gives the single grids' bits."""
    from gitm_amd import vertical
    cols = members(ions)
    p = synth.StepParams(use_ion_advection=ions)
    b = vertical.VerticalBatch(solver, [vertical.to_device(c) for c in cols], ions=ions)
    tiles = b.candidate_tiles()
    b.close()
    ran = run_tiles(solver, cols, p, "rusanov", tiles)
    if not ions:
        assert len(ran) == 32
    assert {t[0] for t in ran} == {2, 3, 4} and {t[2] for t in ran} == {0, 1, 2}
    assert any(t[3] == 1 for t in ran)


@pytest.mark.parametrize("ions", [False, True])
def test_mixed_wavefront_counts_of_the_rusanov_step(solver, ions):
    """Tall members needing 2 and 3 wavefronts in one launch: the 2-wave columns
    leave a 3-wave workgroup's last wavefront empty (it ends at once), so only a
    grid of one workgroup per task is accepted."""
    ms = [synth.Member(synth.GridSpec(1, 1, na), tinf, 700 + i)
          for i, (na, tinf) in enumerate(((150, 900.0), (70, 1200.0), (50, 800.0),
                                          (188, 1000.0)))]
    cols = [synth.member_columns(m, ions=ions) for m in ms]
    ran = run_tiles(solver, cols, synth.StepParams(use_ion_advection=ions), "rusanov",
                    [(3, 3, 1, 0), (3, 1, 0, 0), (3, 3, 0, 1), (4, 4, 0, 0), (3, 3, 2, 0)])
    assert ran == [(3, 3, 1, 0), (3, 1, 0, 0), (4, 4, 0, 0), (3, 3, 2, 0)]
