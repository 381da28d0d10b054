"""The WAF passes against the oracle at the edges of their launch shapes:
every field count of a vertical group, columns as short as the register
windows, domains narrower than a wavefront and one point past it."""
import numpy as np
import pytest

import oracle_api as O
from regcm_amd import synth
from regcm_amd.moloch import MLC_VAR_WAFV_GROUP, Moloch

pytestmark = pytest.mark.gpu


def owned(name, a):
    j = a.shape[-1] if name == "u" else a.shape[-1] - 1
    i = a.shape[-2] if name == "v" else a.shape[-2] - 1
    return a[..., :i, :j]


def check(g, f, variants, label):
    """Two steps, bit for bit (the WAF uses only IEEE operations)."""
    print(f"[waf] {label}", flush=True)
    ref = O.copy_fields(f)
    O.moloch_steps(g, ref, 2)
    names = ("u", "v", "w", "pai", "tetav", "qx", "ux", "vx") + (("trac",) if g.ntr else ())
    with Moloch(g) as m:
        m.load(f)
        m.init_moloch()
        for stage, value in variants.items():
            m.set_variant(stage, value)
        m.moloch(2)
        m.synchronize()
        for n in names:
            a, b = owned(n, ref[n]), owned(n, m.get(n))
            assert np.array_equal(a, b), f"{label}: {n}: {np.count_nonzero(a != b)} differ"


@pytest.mark.parametrize("kz", [4, 5, 6, 17])
@pytest.mark.parametrize("group", [1, 2, 4])
@pytest.mark.parametrize("ntr", [0, 1, 2, 3])
def test_vertical_groups(kz, group, ntr):
    """6..9 fields: groups of 1 to 4 fields, full and one short."""
    g, f, _ = synth.config("small", kz=kz, jx=66, iy=11, nqx=2, ipptls=0, ntr=ntr)
    check(g, f, {MLC_VAR_WAFV_GROUP: group}, f"kz {kz} group {group} fields {6 + ntr}")


def test_extreme_values():
    """Tracers with huge, tiny, signed-zero and non-finite values: the limiter
    ratio overflows, underflows and divides by and into infinities."""
    print("[waf] extreme values", flush=True)
    g, f, _ = synth.config("small", nqx=2, ipptls=0, ntr=2)
    t = f["trac"]
    rng = np.random.default_rng(3)
    scale = rng.choice([1e300, -1e300, 1e-310, -0.0, 1e-31, 1e-29, 1e150, 1.0], t[0].shape)
    t[0] = scale * rng.uniform(0.5, 1.0, t[0].shape)
    t[1, 2, 5, 5] = np.inf
    t[1, 4, 9, 14] = -np.inf
    t[1, 6, 14, 8] = np.nan
    ref = O.copy_fields(f)
    O.moloch_steps(g, ref, 1)
    with Moloch(g) as m:
        m.load(f)
        m.init_moloch()
        m.moloch(1)
        a, b = owned("trac", ref["trac"]), owned("trac", m.get("trac"))
        for n in range(2):
            assert np.array_equal(a[n], b[n], equal_nan=True), \
                f"tracer {n}: {np.count_nonzero(~((a[n] == b[n]) | (np.isnan(a[n]) & np.isnan(b[n]))))}"
