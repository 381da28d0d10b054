"""The curvature terms inside the row-streaming horizontal WAF.

The wave that holds ux and vx applies them; a launch of their own is left only
where no wave holds both.  Bar: no curvature launch for any field count and
group size, and the oracle's bits."""
import numpy as np
import pytest

import oracle_api as O
from regcm_amd import synth
from regcm_amd.moloch import MLC_FP64, MLC_MIXED, MLC_VAR_WAF_GROUP, Moloch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("group", [2, 4])
@pytest.mark.parametrize("over", [
    dict(nqx=2, ipptls=0), dict(nqx=2, ipptls=1), dict(nqx=2, ipptls=1, ntr=2),
    dict(nqx=2, ipptls=1, lrotllr=1), dict(nqx=2, ipptls=1, crm=1), dict(ntr=7), dict(ntr=9)],
    ids=["6", "7", "9", "7-rotllr", "7-periodic", "17", "19"])
def test_no_curvature_launch(over, group):
    print(f"[curvature] {over} group {group}", flush=True)
    g, f, _ = synth.config("crm-small" if over.get("crm") else "small", nadv=2, nsound=2, **over)
    ref = O.copy_fields(f)
    O.moloch_steps(g, ref, 1)
    for precision in (MLC_FP64, MLC_MIXED):
        with Moloch(g, precision) as m:
            m.load(f)
            m.init_moloch()
            m.set_variant(MLC_VAR_WAF_GROUP, group)
            m.profile(True)
            m.moloch(1)
            m.synchronize()
            assert "adv_curvature" not in m.kernel_stats(), precision
            if precision == MLC_FP64:
                jn = g.jx if g.crm else g.jx - 1
                im = g.iy if g.crm else g.iy - 1
                for n in ("ux", "vx"):
                    assert np.array_equal(ref[n][..., :im, :jn], m.get(n)[..., :im, :jn]), n
