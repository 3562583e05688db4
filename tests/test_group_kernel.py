"""The AUSM step split over the species (gitm_amd/csrc/vert_group.h).

Its host build against the oracle within the step's parity bar (1e-11 per
step, the bar of the other parity tests) at the heights where it can go wrong:
the shortest and tallest columns, one, two, three and four wavefronts per
group, full and nearly empty last ones, segments of the hydrostatic product
with a short or missing tail; with ions, boundary options and without
friction.  On the GPU: ions at the tallest column that its LDS holds and one
level above it, alone and in a batch."""
from __future__ import annotations

import ctypes
import os
import subprocess

import numpy as np
import pytest

from gitm_amd import _abi, synth
from oracle import cpu
from tests.emu import emu
from tests.helpers import assert_parity, subset

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
MAX_IONS = 226


@pytest.fixture(scope="module")
def group(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("emu") / "libgv_emu_group.so")
    subprocess.run(["g++", "-std=c++20", "-O2", "-fPIC", "-shared", "-ffp-contract=off",
                    "-pthread", "-I" + os.path.join(ROOT, "include"),
                    "-I" + os.path.join(ROOT, "gitm_amd", "csrc"),
                    os.path.join(HERE, "emu", "emu_group.cpp"), "-o", so], check=True)
    return ctypes.CDLL(so)


def advance(lib, cols, sp, n_steps=1):
    nc, L = cols["temp"].shape
    keep = {k: np.array(v, dtype=np.float64, order="C") for k, v in cols.items()
            if k in _abi.COLUMN_KEYS}
    keep["logns"], keep["nden"] = np.zeros_like(keep["nds"]), np.zeros_like(keep["temp"])
    c = _abi.columns_struct({k: v.ctypes.data for k, v in keep.items()}, nc, L - 4)
    e = _abi.Error()
    rc = lib.gv_emu_group(ctypes.byref(emu.params_from(sp)), ctypes.byref(c), n_steps, nc,
                          ctypes.byref(e))
    return keep, (rc, e.column, e.level)


CASES = [(10, {}), (14, {}), (44, {}), (45, {}), (50, {}), (60, {}), (61, {}),
         (124, {}), (125, {"use_neutral_friction": False}), (188, {}), (189, {}), (252, {}),
         (18, {"use_ion_advection": True}),
         (61, {"use_ion_advection": True, "use_improved_ion_advection": False}),
         (50, {"use_msis": True}), (50, {"use_gswm_tides": True}),
         (50, {"use_waccm_tides": True}), (50, {"use_msis": True, "use_gswm_tides": True}),
         (50, {"use_coriolis": False})]


@pytest.mark.parametrize("n_alts,flags", CASES, ids=[f"{n}-{'-'.join(f) or 'plain'}"
                                                     for n, f in CASES])
def test_host_build_against_oracle(group, n_alts, flags):
    ions = bool(flags.get("use_ion_advection"))
    cols = subset(synth.make_columns(synth.GridSpec(1, 1, n_alts, stretched=n_alts == 124),
                                     seed=n_alts, ions=ions), [0, 40])
    if flags.get("use_msis"):
        cols["msis"] = synth.msis_bc_values(cols, seed=3)
    if flags.get("use_gswm_tides") or flags.get("use_waccm_tides"):
        cols["tides"] = synth.tides_values(cols, seed=3,
                                           absolute=bool(flags.get("use_waccm_tides")))
    sp = synth.StepParams(**flags)
    out, err = advance(group, cols, sp)
    assert err[0] == 0
    assert_parity(out, cpu.advance(cols, sp, solver=1, n_steps=1), 1e-11, what=f"nAlts {n_alts}")


@pytest.mark.parametrize("field,level", [("temp", 2), ("temp", 20), ("temp", 31), ("nds", 15)])
def test_errors_as_one_lane_per_level(group, field, level):
    """What stops the step stops it here too, at the same column and level: a
    NaN temperature makes the friction matrix singular, a density of zero is
    refused on entry and leaves the column as it was."""
    cols = subset(synth.make_columns(synth.GridSpec(1, 1, 30), seed=8), [0, 1, 2])
    if field == "temp":
        cols["temp"][1, level] = np.nan
    else:
        cols["nds"][1, 4, level] = 0.0
    out, (rc, column, lev) = advance(group, cols, synth.StepParams())
    with pytest.raises(RuntimeError, match=rf"column {column}, level {lev}\)"):
        emu.advance(cols, synth.StepParams(), solver=1, device_math=True)
    assert column == 1 and rc == (2 if field == "temp" else 1)
    if field == "nds":
        assert np.array_equal(out["temp"][1], cols["temp"][1])


def test_tallest_column_with_ions(group):
    assert group.gv_emu_group_max_alts(1) == MAX_IONS
    assert group.gv_emu_group_max_alts(0) == 252


@pytest.mark.gpu
@pytest.mark.parametrize("n_alts", [MAX_IONS, MAX_IONS + 1, 252])
def test_tall_columns_with_ions(solver, n_alts):
    from gitm_amd import vertical
    p = synth.StepParams(use_ion_advection=True)
    sets = [subset(synth.make_columns(synth.GridSpec(1, 1, na), seed=na, ions=True),
                   list(range(0, 81, 9))) for na in (n_alts, 50)]
    dev = [vertical.to_device(c) for c in sets]
    for d, c in zip(dev, sets):
        solver.advance(d, p, "ausm", 1)
        assert_parity(vertical.to_host(d), cpu.advance(c, p, solver=1, n_steps=1), 1e-11,
                      what=f"nAlts {n_alts}")
    members = [vertical.to_device(c) for c in sets]
    b = vertical.VerticalBatch(solver, members, ions=True)
    b.advance(p, "ausm", 1)
    for m, d in zip(members, dev):
        a, r = vertical.to_host(m), vertical.to_host(d)
        for k in ("nds", "vvel", "vel", "temp", "rho", "ions"):
            assert np.array_equal(a[k], r[k]), k
    b.close()
