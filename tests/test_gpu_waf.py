"""The WAF passes against the oracle at the edges of their launch shapes:
every field count of a vertical group, columns as short as the register
windows, domains narrower than a wavefront and one point past it."""
import numpy as np
import pytest

import oracle_api as O
from regcm_amd import synth
from regcm_amd.moloch import (MLC_MIXED, MLC_VAR_WAF_GROUP, MLC_VAR_WAF_H, MLC_VAR_WAF_ROWS,
                              MLC_VAR_WAFV_GROUP, Moloch, relative_l2)

pytestmark = pytest.mark.gpu


def owned(g, name, a):
    if g.crm:
        return a
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
            a, b = owned(g, n, ref[n]), owned(g, n, m.get(n))
            assert np.array_equal(a, b), f"{label}: {n}: {np.count_nonzero(a != b)} differ"


@pytest.mark.parametrize("kz", [4, 5, 6, 17])
@pytest.mark.parametrize("group", [1, 2, 4])
@pytest.mark.parametrize("ntr", [0, 1, 2, 3])
def test_vertical_groups(kz, group, ntr):
    """6..9 fields: groups of 1 to 4 fields, full and one short."""
    g, f, _ = synth.config("small", kz=kz, jx=66, iy=11, nqx=2, ipptls=0, ntr=ntr)
    check(g, f, {MLC_VAR_WAFV_GROUP: group}, f"kz {kz} group {group} fields {6 + ntr}")


# wave tiles: one wave holds 64 columns of a bounded domain, each further one
# 60; a periodic domain takes 60 per wave.  Rows: chunks that end on, before
# and past the last row
EDGES = [("bounded", jx, iy, {}) for jx, iy in ((64, 9), (65, 10), (66, 11), (125, 12), (126, 13))] \
    + [("rotllr", 65, 10, dict(lrotllr=1)), ("rotllr", 126, 13, dict(lrotllr=1))] \
    + [("periodic", jx, iy, dict(crm=1)) for jx, iy in ((24, 8), (60, 9), (61, 11), (122, 13))]


@pytest.mark.parametrize("kind,jx,iy,over", EDGES, ids=[f"{k}-{j}x{i}" for k, j, i, _ in EDGES])
@pytest.mark.parametrize("rows,group", [(4, 2), (5, 4), (256, 4)])
def test_row_streaming_edges(kind, jx, iy, over, rows, group):
    g, f, _ = synth.config("crm-small" if over.get("crm") else "small", jx=jx, iy=iy, kz=5,
                           ntr=1, **over)
    check(g, f, {MLC_VAR_WAF_H: 0, MLC_VAR_WAF_ROWS: rows, MLC_VAR_WAF_GROUP: group},
          f"{kind} {jx}x{iy} rows {rows} fields per wave {group}")


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
        a, b = owned(g, "trac", ref["trac"]), owned(g, "trac", m.get("trac"))
        for n in range(2):
            assert np.array_equal(a[n], b[n], equal_nan=True), \
                f"tracer {n}: {np.count_nonzero(~((a[n] == b[n]) | (np.isnan(a[n]) & np.isnan(b[n]))))}"


@pytest.mark.parametrize("group", [1, 2, 4])
def test_groups_of_a_tile_next_to_each_other(group):
    """More waves than one round of the chip: the vertical pass counts a tile's
    field groups first (25 fields, so that the domain stays small)."""
    g, f, _ = synth.config("small", jx=201, iy=190, kz=5, ntr=15, nadv=1, nsound=1)
    check(g, f, {MLC_VAR_WAFV_GROUP: group}, f"groups first, {group} per thread")


def test_groups_of_a_tile_next_to_each_other_mixed():
    """The same with the float and the double batch in one launch, against the
    oracle within the mixed form's error (one float rounding per operation)."""
    print("[waf] groups first, mixed", flush=True)
    g, f, _ = synth.config("small", jx=201, iy=190, kz=5, ntr=15, nadv=1, nsound=1)
    ref = O.copy_fields(f)
    O.moloch_steps(g, ref, 1)
    with Moloch(g, MLC_MIXED) as m:
        m.load(f)
        m.init_moloch()
        m.moloch(1)
        m.synchronize()
        for n, tol in (("u", 1e-5), ("tetav", 1e-6), ("pai", 1e-7), ("qx", 1e-5), ("trac", 1e-5)):
            assert relative_l2(owned(g, n, ref[n]), owned(g, n, m.get(n))) < tol, n
