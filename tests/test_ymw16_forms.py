"""CPU comparison of the two forms of the YMW16 density that a pass may take: the
short one of the marches for every parameter set that is sent to it (the
template's with one parameter at a time across its range) against the literal
one, at 14000 points from the nebulae to the rim, within 1e-9 (rounding, most of
it in the Gum shell's angles) and finite in the same places."""
import os
import shutil
import subprocess

import numpy as np

from hammurabix_amd import Param, configs

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "hammurabix_amd", "csrc")


def test_short_form_where_it_is_taken(tmp_path):
    # the helpers that need the device are restated by the program
    for f in ("hamx_ymw16.h", "hamx_models.h", "hamx_cgs.h"):
        shutil.copy(os.path.join(CSRC, f), tmp_path)
    (tmp_path / "hamx_math.h").write_text("#pragma once\n")
    np.array(list(Param(text=configs.plain_forward(tereg="ymw16")).tereg_ymw16)).tofile(
        tmp_path / "p.bin")
    exe = str(tmp_path / "forms")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-I", str(tmp_path),
                    os.path.join(HERE, "ymw16_forms.cc"), "-o", exe], check=True)
    r = subprocess.run([exe, str(tmp_path / "p.bin")], capture_output=True, text=True, timeout=300)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
