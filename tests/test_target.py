"""The target that the library is built for: SRAM-ECC on, which gathers into the registers of their own addresses rely on
(csrc/rank_whole.hpp); a code object without the mark would be taken by a device without it and give wrong numbers there."""
import re

from mustafar_amd import build


def test_every_code_object_asks_for_sram_ecc():
    with open(build.LIB, "rb") as f:
        targets = set(re.findall(rb"amdgcn-amd-amdhsa-+(gfx[0-9a-z]+(?::[a-z+-]+)*)", f.read()))
    assert targets == {b"gfx950:sramecc+"}
