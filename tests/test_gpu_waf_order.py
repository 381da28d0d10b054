"""The order of the vertical WAF's field groups follows the groups a call
launches: a knob or the tuner that changes their number changes the order with
it.  Bar: the oracle's bits on both sides of the switch, for group sizes set
after the domain's own choice, alone and in a batch whose members differ."""
import numpy as np
import pytest

import oracle_api as O
from regcm_amd import synth
from regcm_amd.moloch import MLC_FP64, MLC_MIXED, MLC_VAR_WAFV_GROUP, Moloch, MolochBatch

pytestmark = pytest.mark.gpu

FIELDS = ("u", "v", "w", "pai", "tetav", "qx", "trac")


def test_group_sizes_across_the_switch():
    """456 waves per field group, 16 fields in the first launch: one field per
    wave past the switch, two and four before it."""
    print("[waf order] 190x150x5", flush=True)
    g, f, _ = synth.config("small", jx=190, iy=150, kz=5, ntr=9, nadv=1, nsound=1)
    ref = O.copy_fields(f)
    O.moloch_steps(g, ref, 4)
    with Moloch(g) as m:
        m.load(f)
        m.init_moloch()
        for group in (4, 1, 2, 1):
            m.set_variant(MLC_VAR_WAFV_GROUP, group)
            m.moloch(1)
        m.synchronize()
        for n in FIELDS:
            jn = g.jx if n == "u" else g.jx - 1
            im = g.iy if n == "v" else g.iy - 1
            assert np.array_equal(ref[n][..., :im, :jn], m.get(n)[..., :im, :jn]), n


@pytest.mark.parametrize("precision", [MLC_FP64, MLC_MIXED], ids=["fp64", "mixed"])
def test_batch_members_on_both_sides(precision):
    print(f"[waf order] batch, precision {precision}", flush=True)
    doms = [synth.config("small", jx=jx, iy=100, kz=5, ntr=9, nadv=1, nsound=1)[:2]
            for jx in (190, 130, 70)]
    alone = []
    for g, f in doms:
        with Moloch(g, precision) as m:
            m.load(f)
            m.init_moloch()
            m.moloch(3)
            alone.append({n: m.get(n) for n in FIELDS})
    with MolochBatch([g for g, _ in doms], precision) as b:
        for i, (g, f) in enumerate(doms):
            b.member(i).load(f)
            b.member(i).init_moloch()
        for groups in ((4, 4, 4), (1, 4, 2), (1, 1, 1)):
            for i, v in enumerate(groups):
                b.member(i).set_variant(MLC_VAR_WAFV_GROUP, v)
            b.step(1)
        b.synchronize()
        for i in range(3):
            for n in FIELDS:
                assert np.array_equal(b.member(i).get(n), alone[i][n]), (i, n)
