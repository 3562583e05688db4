"""The AUSM step split over the species under the host sanitizers (CPU only):
its slots are written and read by different groups and phases, ordered by the
workgroup's barriers, and its boundary conditions by wavefronts alone
(tests/emu/sanitize_group.cpp).  Short and tall columns, one to three
wavefronts per group, ions, and the values of level 0 from MSIS and the tides."""
from __future__ import annotations

import os
import subprocess
from concurrent.futures import ThreadPoolExecutor

import pytest

from gitm_amd import synth
from tests.helpers import subset
from tests.test_emu_sanitizers import EMU, ROOT, run, write_case

FLAGS = {"thread": ["-fsanitize=thread"],
         "address": ["-fsanitize=address", "-fno-omit-frame-pointer"]}


def build(kind: str, out_dir: str) -> str:
    exe = os.path.join(out_dir, f"sanitize_group_{kind}")
    subprocess.run(["g++", "-std=c++20", "-g", "-O1", "-ffp-contract=off", "-pthread",
                    *FLAGS[kind], "-I" + os.path.join(ROOT, "include"),
                    "-I" + os.path.join(ROOT, "gitm_amd", "csrc"),
                    os.path.join(EMU, "sanitize_group.cpp"), "-o", exe], check=True)
    return exe


@pytest.fixture(scope="module")
def exes(tmp_path_factory):
    d = str(tmp_path_factory.mktemp("sanitize_group"))
    with ThreadPoolExecutor(2) as ex:
        return dict(zip(FLAGS, ex.map(lambda k: build(k, d), FLAGS)))


CASES = [("10", 10, 2, {}), ("50", 50, 1, {}), ("61", 61, 1, {}), ("130", 130, 1, {}),
         ("ions_18", 18, 2, {"ions": True}), ("ions_62", 62, 1, {"ions": True}),
         ("msis_gswm_30", 30, 2, {"msis": True, "gswm": True}), ("waccm_30", 30, 1, {"waccm": True})]


@pytest.mark.parametrize("kind", list(FLAGS))
@pytest.mark.parametrize("name,na,steps,opt", CASES, ids=[c[0] for c in CASES])
def test_group_kernel_under_sanitizer(exes, tmp_path, kind, name, na, steps, opt):
    cols = subset(synth.make_columns(synth.GridSpec(1, 1, na), seed=na, ions=opt.get("ions", False)),
                  [0, 40])
    if opt.get("msis"):
        cols["msis"] = synth.msis_bc_values(cols, seed=3)
    if opt.get("gswm") or opt.get("waccm"):
        cols["tides"] = synth.tides_values(cols, seed=3, absolute=opt.get("waccm", False))
    path = str(tmp_path / f"{name}.bin")
    write_case(path, cols, 1, steps, 0, **opt)
    run(exes[kind], path, kind)
