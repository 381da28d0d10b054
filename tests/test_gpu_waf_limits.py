"""The WAF limiter at the upper end of the stored type's range.

Advection is homogeneous: every flux is linear in the field but for the
limiter, which takes ratios of its differences.  A tracer times a power of two
must therefore come out as the result times that power, bit for bit, as long
as nothing overflows.  Here the scaled tracer's neighbour differences lie in
the type's top binades, where a reciprocal of the difference is below the
smallest normal number.  The winds are slow, so that no flux overflows."""
import numpy as np
import pytest

from regcm_amd import synth
from regcm_amd.moloch import (MLC_FP64, MLC_MIXED, MLC_VAR_WAF_GROUP, MLC_VAR_WAF_H,
                              MLC_VAR_WAFV_GROUP, Moloch)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("variants", [
    {}, {MLC_VAR_WAF_H: 1}, {MLC_VAR_WAFV_GROUP: 2, MLC_VAR_WAF_GROUP: 2}],
    ids=["default", "tile", "two-fields"])
@pytest.mark.parametrize("precision,top", [(MLC_FP64, 1022), (MLC_MIXED, 126)],
                         ids=["fp64", "mixed"])
@pytest.mark.parametrize("crm", [0, 1], ids=["bounded", "periodic"])
def test_huge_differences_scale_exactly(precision, top, variants, crm):
    print(f"[waf limits] precision={precision} 2^{top} crm={crm} {variants}", flush=True)
    g, f, _ = synth.config("crm-small" if crm else "small", ntr=2, nadv=1, nsound=1, dtsec=1.0)
    for n in ("u", "v", "w"):
        f[n] *= 0.01
    rng = np.random.default_rng(5)
    shape = f["trac"][0].shape
    x = rng.choice([-1.0, 1.0], shape) * rng.uniform(0.5, 1.0, shape)
    x = x.astype(np.float32).astype(np.float64)      # exact in either type
    f["trac"][0], f["trac"][1] = x, x * 2.0 ** top
    with Moloch(g, precision) as m:
        m.load(f)
        m.init_moloch()
        for stage, value in variants.items():
            m.set_variant(stage, value)
        m.moloch(1)
        t = m.get("trac")
    assert np.all(np.isfinite(t))
    assert np.count_nonzero(t[0] - x) > t[0].size // 4      # the field has moved
    bad = t[0] * 2.0 ** top != t[1]
    assert not bad.any(), f"{np.count_nonzero(bad)} of {bad.size} values differ"
