"""The autotuner times only what changes the launches: knobs of a form that
does not run keep the value they were given, whatever the timing noise."""
import pytest

from regcm_amd import synth
from regcm_amd.moloch import (MLC_FP64, MLC_MIXED, MLC_VAR_MIXED_MERGE, MLC_VAR_WAF_GROUP,
                              MLC_VAR_WAF_H, MLC_VAR_WAF_HGROUP, MLC_VAR_WAF_ROWS,
                              MLC_VAR_WAF_TILE, Moloch)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [MLC_FP64, MLC_MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("tile", [4, 8])
def test_knobs_of_the_other_form_stay(precision, tile):
    print(f"[tune] inert knobs, precision {precision}, tile {tile}", flush=True)
    given = {MLC_VAR_WAF_ROWS: 17, MLC_VAR_WAF_GROUP: 2, MLC_VAR_WAF_TILE: tile,
             MLC_VAR_WAF_HGROUP: 3, MLC_VAR_MIXED_MERGE: 6}
    g, f, _ = synth.config("small", nadv=1, nsound=1)
    with Moloch(g, precision) as m:
        m.load(f)
        m.init_moloch()
        for stage, value in given.items():
            m.set_variant(stage, value)
        m.autotune(1)
        got = {stage: m.get_variant(stage) for stage in given}
        if m.get_variant(MLC_VAR_WAF_H) == 0:
            kept = [MLC_VAR_WAF_TILE, MLC_VAR_WAF_HGROUP]
        else:
            kept = [MLC_VAR_WAF_ROWS, MLC_VAR_WAF_GROUP]
        if precision == MLC_FP64:
            kept.append(MLC_VAR_MIXED_MERGE)
    for stage in kept:
        assert got[stage] == given[stage], stage
