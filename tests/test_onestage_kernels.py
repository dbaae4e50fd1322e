"""The bare right-hand side is compiled for every tile shape, storage and metric form.

cgfd_set_tile reaches cgfd_el_iso_onestage as it reaches a run; a shape whose
kernels are missing would silently run another one.  The library's own symbol
table lists the kernels (k_march<DX, DY, DZ, storage, arithmetic, TX, TY, waves,
metric form, PML, RK mode, surface rows>; mode 0 is the bare right-hand side).
"""
import re
import shutil
import subprocess

import pytest

import cgfd


@pytest.mark.skipif(shutil.which("nm") is None, reason="no nm")
@pytest.mark.parametrize("tile", ["64, 4", "32, 8", "64, 8", "32, 16"])
def test_every_shape_has_the_bare_right_hand_side(tile):
    out = subprocess.run(["nm", "-C", "--defined-only", cgfd.LIB_PATH], capture_output=True, text=True, check=True).stdout
    pat = re.compile(r"k_march<0, 0, 0, (\S+), (?:float|double), %s, \d+, (\d), (true|false), (\d), (true|false)>" % tile)
    have = {(m[1], int(m[2]), m[3] == "true", int(m[4])) for m in pat.finditer(out)}
    for storage in ("float", "double", "__half", "__hip_bfloat16"):
        forms = {met for s, met, _, mode in have if s == storage and mode == 1 and met != 3}
        assert {0, 1} <= forms
        for met in forms:
            for pml in (False, True):
                assert (storage, met, pml, 0) in have, (storage, met, pml)
