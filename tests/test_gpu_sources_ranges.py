"""The sources step's quick divisions, bit for bit (signs of zeros included)
against the oracle's plain ones: the level counts at which the chains' blocks,
their remainders and the wavefronts end, and columns at and beyond the ranges
within which the quick forms hold, next to ordinary ones."""
from __future__ import annotations

import numpy as np
import pytest

from gitm_amd import synth
from oracle import cpu
from tests.test_gpu_sources import INC, STATE, gpu_sources

pytestmark = pytest.mark.gpu


def same_bits(a, b):
    a, b = np.ascontiguousarray(a), np.ascontiguousarray(b)
    return np.all((a.view(np.int64) == b.view(np.int64)) | (np.isnan(a) & np.isnan(b)))


def check(solver, cols, src):
    with np.errstate(all="ignore"):
        ref = cpu.sources(dict(cols, **src), 2.0, synth.species_masses(),
                          use_turbulent_cond=True, apply=True)
    out = gpu_sources(solver, cols, src, 2.0, True, True)
    L = cols["temp"].shape[1]
    for k in STATE:
        assert same_bits(out[k], ref[k]), k
    for k in INC:
        assert same_bits(out[k][..., 1:L - 1], ref[k][..., 1:L - 1]), k


@pytest.mark.parametrize("nalts", [10, 11, 12, 13, 14, 15, 16, 17, 18, 60, 61, 62, 124, 125,
                                   188, 189, 251, 252])
def test_level_counts(solver, nalts):
    print(f"sources, {nalts} levels", flush=True)
    cols = synth.make_columns(synth.GridSpec(1, 1, nalts, nlons=3, nlats=2), seed=61)
    check(solver, cols, synth.source_fields(cols, seed=61))


def zero(c, f, odd):
    c["vel"][odd], c["vvel"][odd] = 0.0, -0.0


def half_zero(c, f, odd):
    c["vel"][odd, :, :30], c["vvel"][odd, :, 30:] = 0.0, 0.0


def tiny(c, f, odd):
    c["vvel"][odd] *= 1e-70


def tinier(c, f, odd):
    c["vel"][odd] *= 1e-200


def large(c, f, odd):
    c["temp"][odd] *= 1e80


def stiff(c, f, odd):
    f["visc_coef"][odd] *= 1e70


def inviscid(c, f, odd):
    f["visc_coef"][odd], f["visc_coef_s"][odd], c["eddy"][odd] = 0.0, 0.0, 0.0


def antidiffusive(c, f, odd):
    f["kappa_temp"][odd] *= -1e3


def not_a_number(c, f, odd):
    c["temp"][odd, 20] = np.nan


def infinite(c, f, odd):
    c["vvel"][odd, 2, 25] = np.inf


@pytest.mark.parametrize("change", [zero, half_zero, tiny, tinier, large, stiff, inviscid,
                                    antidiffusive, not_a_number, infinite])
def test_ranges(solver, change):
    print(f"sources, {change.__name__}", flush=True)
    cols = synth.make_columns(synth.GridSpec(1, 1, 50, nlons=4, nlats=2), seed=62)
    src = synth.source_fields(cols, seed=62)
    change(cols, src, np.arange(cols["temp"].shape[0]) % 2 == 1)
    check(solver, cols, src)
