"""The sources step's quick divisions on columns with zeros: after a vertical
step the east and north winds of level 0 are exactly zero, and every column's
solves start from one.

On the CPU: the forward sweeps of gitm_amd/csrc/vert_sources_chain.h, quick and
plain, over random columns of one quantity whose right side is zero at level 0,
at the bottom levels, at some levels or everywhere: the quick sweep accepts the
column and gives the plain sweep's bits.  A value that is not zero but too small
for the quick divisions is refused.  On the GPU: stepped columns, bit for bit
the oracle's."""
from __future__ import annotations

import os
import subprocess

import numpy as np
import pytest

from gitm_amd import synth
from tests.test_gpu_sources_ranges import check

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <math.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <vector>
#define GV_HOST_EMULATION 1
#include "vert_sources_chain.h"
using namespace gv::chain;

static double uni(double lo, double hi) { return lo + (hi - lo) * drand48(); }

// A row of nA + 4 levels and what the rings read past it; level 1 is aligned.
struct Row {
  std::vector<double> v;
  double *p;
  explicit Row(int n) : v(n + 64, 1.0) {
    p = v.data() + 32;
    if ((size_t)(p + 1) % 16) p++;
  }
};

static long differ(const double *a, const double *b, int n) {
  long d = 0;
  for (int i = 0; i < n; i++) d += memcmp(a + i, b + i, sizeof(double)) != 0;
  return d;
}

int main() {
  srand48(5);
  const char *names[] = {"level 0", "bottom levels", "some levels", "everywhere", "tiny"};
  int rc = 0;
  for (int kind = 0; kind < 5; kind++) {
    long refused = 0, bits = 0, n = 0;
    for (int trial = 0; trial < 400; trial++) {
      const int nA = 10 + (int)(drand48() * 60), zeros = 1 + (int)(drand48() * (nA - 2));
      Row a(nA), c(nA), b(nA), d(nA);
      for (int k = 0; k <= nA + 1; k++) {
        const double m = exp(uni(-12.0, 6.0)), x = exp(uni(-3.0, 3.0)), y = 0.2 * x * uni(-1.0, 1.0);
        a.p[k] = k < 1 ? 0.0 : x - y;
        c.p[k] = k < 1 ? 0.0 : x + y;
        b.p[k] = k < 1 ? -1.0 : -1.0 / m - 2.0 * x;
        d.p[k] = -uni(-80.0, 80.0) / m;
        const bool zero = kind == 0   ? k == 0
                          : kind == 1 ? k < zeros
                          : kind == 2 ? drand48() < 0.3
                                      : kind == 3;
        if (zero) d.p[k] = drand48() < 0.5 ? 0.0 : -0.0;
        if (kind == 4) d.p[k] *= 1e-190;
      }
      for (int which = 0; which < 2; which++) {  // sweep, sweep2
        double out[2][2][300];
        bool ok[2];
        for (int fast = 0; fast < 2; fast++) {
          Row bb = b, w = d;
          bb.p = bb.v.data() + (b.p - b.v.data());
          w.p = w.v.data() + (d.p - d.v.data());
          Row rr(nA), den(nA);
          double cp = 0.0 / -1.0, dp = d.p[0] / -1.0;
          bb.p[0] = cp;
          if (which == 0) {
            w.p[0] = dp;
            ok[fast] = fast ? sweep<true>(a.p, c.p, bb.p, d.p, w.p, 2.0, nA, cp, dp)
                            : sweep<false>(a.p, c.p, bb.p, d.p, w.p, 2.0, nA, cp, dp);
          } else {
            // the pivots of the first sweep
            for (int k = 1; k <= nA; k++) {
              den.p[k] = b.p[k] - cp * a.p[k];
              rr.p[k] = div_recip(den.p[k]);
              cp = c.p[k] / den.p[k];
            }
            w.p[0] = dp;
            ok[fast] = fast ? sweep2<true>(a.p, w.p, den.p, rr.p, nA, dp)
                            : sweep2<false>(a.p, w.p, den.p, rr.p, nA, dp);
          }
          memcpy(out[fast][0], w.p, (nA + 1) * sizeof(double));
          memcpy(out[fast][1], bb.p, (nA + 1) * sizeof(double));
        }
        n++;
        refused += !ok[1];
        if (ok[1]) bits += differ(out[0][0], out[1][0], nA + 1) + differ(out[0][1], out[1][1], nA + 1);
      }
    }
    printf("%s: %ld sweeps, %ld refused, %ld values differ\n", names[kind], n, refused, bits);
    if (bits || refused != (kind == 4 ? n : 0)) rc = 1;
  }
  return rc;
}
"""


def test_quick_sweeps_take_zeros(tmp_path):
    src, exe = tmp_path / "chain.cpp", tmp_path / "chain"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off",
                    "-I" + os.path.join(ROOT, "include"),
                    "-I" + os.path.join(ROOT, "gitm_amd", "csrc"), str(src), "-o", str(exe),
                    "-lm"], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("nalts", [10, 37, 50, 100, 189])
def test_stepped_columns(solver, nalts):
    from gitm_amd import vertical
    cols = synth.make_columns(synth.GridSpec(1, 1, nalts, nlons=3, nlats=3), seed=63)
    src = synth.source_fields(cols, seed=63)
    d = vertical.to_device(cols)
    print(f"sources after a vertical step, {nalts} levels", flush=True)
    solver.advance(d, synth.StepParams(), "ausm", 1)
    cols.update({k: v for k, v in vertical.to_host(d).items() if k in cols})
    assert np.all(cols["vel"][:, :2, 1] == 0.0) and np.any(cols["vel"][:, :2, 2] != 0.0)
    check(solver, cols, src)
