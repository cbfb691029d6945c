"""What the batch's tuner times (autotune.trials), on the CPU: no candidate of a width that a scheme's faces do
not read."""

import pytest

from peregrine_amd import autotune, native
from peregrine_amd.simulator import EOS, RECON


@pytest.mark.parametrize("recon", ["constant", "muscl"])
@pytest.mark.parametrize("eos", sorted(EOS))
def test_only_a_choice_the_faces_read_is_timed(recon, eos):
    desc = native.CaseDesc()
    desc.recon, desc.eos = RECON[recon], EOS[eos]
    kinds = dict(autotune.trials(desc))
    assert kinds["stage"] == autotune.STAGE_TILES
    staged = recon == "muscl" and eos in ("cpg", "tpg")
    assert kinds.get("fluxk") == (None if staged else autotune.FLUXK_TILES)
