"""The LDS-tile form of the horizontal WAF (MLC_VAR_WAF_H 1), which the
row-streaming default leaves to those who ask for it: tile heights, field
groups, the mixed form's merged launches, metrics formed from the orography,
and batches whose members record different numbers of launches.  Every test
sets the form, and every knob that changes the number of launches is checked
to change it, so that no test passes by running another form."""
import numpy as np
import pytest

import oracle_api as O
from regcm_amd import synth
from regcm_amd.moloch import (MLC_FP64, MLC_MIXED, MLC_VAR_LEVEL_CHUNK, MLC_VAR_MIXED_MERGE,
                              MLC_VAR_STAGGER_CHUNK, MLC_VAR_TERRAIN, MLC_VAR_WAF_H,
                              MLC_VAR_WAF_HGROUP, MLC_VAR_WAF_TILE, MLC_VAR_XCD_MAP, Moloch,
                              MolochBatch)

pytestmark = pytest.mark.gpu

FIELDS = ("u", "v", "w", "pai", "tetav", "qx", "ux", "vx")


def owned(g, name, a):
    if g.crm:
        return a
    j = a.shape[-1] if name == "u" else a.shape[-1] - 1
    i = a.shape[-2] if name == "v" else a.shape[-2] - 1
    return a[..., :i, :j]


def run(g, f, precision, variants, nsteps=2):
    """The fields after nsteps in the tile form, and the horizontal WAF's and
    the curvature's launches per advection."""
    with Moloch(g, precision) as m:
        m.load(f)
        m.init_moloch()
        m.set_variant(MLC_VAR_WAF_H, 1)
        for stage, value in variants.items():
            m.set_variant(stage, value)
        m.profile(True)
        m.moloch(nsteps)
        m.synchronize()
        s = m.kernel_stats()
        per = nsteps * g.nadv
        count = tuple(s.get(n, (0, 0.0))[0] // per for n in ("waf_horizontal", "adv_curvature"))
        return {n: m.get(n) for n in FIELDS + (("trac",) if g.ntr else ())}, count


SHAPES = [("small", {}), ("small", dict(jx=70, iy=9, kz=7)), ("small", dict(lrotllr=1, ntr=1)),
          ("crm-small", {}), ("crm-small", dict(jx=70, iy=9, kz=7, ntr=1))]


@pytest.mark.parametrize("name,over", SHAPES, ids=["bounded", "bounded-odd", "rotllr", "periodic",
                                                   "periodic-odd"])
@pytest.mark.parametrize("variants", [
    {MLC_VAR_WAF_TILE: 4}, {MLC_VAR_WAF_TILE: 8}, {MLC_VAR_WAF_TILE: 4, MLC_VAR_XCD_MAP: 0},
    {MLC_VAR_WAF_TILE: 8, MLC_VAR_XCD_MAP: 0}, {MLC_VAR_WAF_HGROUP: 1, MLC_VAR_LEVEL_CHUNK: 3},
    {MLC_VAR_WAF_HGROUP: 3, MLC_VAR_XCD_MAP: 0}, {MLC_VAR_WAF_HGROUP: 4, MLC_VAR_WAF_TILE: 8},
    {MLC_VAR_STAGGER_CHUNK: 7, MLC_VAR_WAF_TILE: 8},
    {MLC_VAR_TERRAIN: 8, MLC_VAR_WAF_TILE: 4}, {MLC_VAR_TERRAIN: 15, MLC_VAR_WAF_TILE: 8},
    {MLC_VAR_TERRAIN: 0, MLC_VAR_WAF_TILE: 8}],
    ids=["tile4", "tile8", "tile4-plain-order", "tile8-plain-order", "hgroup1", "hgroup3",
         "hgroup4-tile8", "stagger7-tile8", "formed-tile4", "all-formed-tile8", "streamed-tile8"])
def test_tile_form_matches_the_oracle(name, over, variants):
    print(f"[tile] {name} {over} {variants}", flush=True)
    g, f, _ = synth.config(name, nadv=2, nsound=2, **over)
    ref = O.copy_fields(f)
    O.moloch_steps(g, ref, 2)
    got, count = run(g, f, MLC_FP64, variants)
    # one or three fields per block leave ux and vx (third and fourth) in
    # different blocks
    assert count == (1, 1 if variants.get(MLC_VAR_WAF_HGROUP) in (1, 3) else 0)
    for n in got:
        a, b = owned(g, n, ref[n]), owned(g, n, got[n])
        assert np.array_equal(a, b), f"{n}: {np.count_nonzero(a != b)} differ"


@pytest.mark.parametrize("name,over", SHAPES, ids=["bounded", "bounded-odd", "rotllr", "periodic",
                                                   "periodic-odd"])
@pytest.mark.parametrize("terrain", [6, 14])
@pytest.mark.parametrize("tile", [4, 8])
def test_mixed_merges_give_the_same_bits(name, over, tile, terrain):
    """MLC_VAR_MIXED_MERGE: two launches per advection, or one by bit 1 (two
    block ranges) or by bit 2 (the same blocks).  A mixed step in the tile
    form also gives the row-streaming form's bits."""
    print(f"[tile] mixed {name} {over} tile {tile} terrain {terrain}", flush=True)
    g, f, _ = synth.config(name, nadv=2, nsound=2, **over)
    out = []
    for merge, hgroup, launches in ((0, 0, 2), (1, 0, 2), (2, 0, 1), (3, 2, 1), (4, 0, 1), (5, 0, 1)):
        got, count = run(g, f, MLC_MIXED, {MLC_VAR_MIXED_MERGE: merge, MLC_VAR_WAF_TILE: tile,
                                           MLC_VAR_WAF_HGROUP: hgroup, MLC_VAR_TERRAIN: terrain})
        assert count[0] == launches, merge
        out.append(got)
    with Moloch(g, MLC_MIXED) as m:
        m.load(f)
        m.init_moloch()
        m.moloch(2)
        out.append({n: m.get(n) for n in out[0]})
    for k, o in enumerate(out[1:]):
        for n in o:
            assert np.array_equal(owned(g, n, out[0][n]), owned(g, n, o[n])), (k, n)


def test_mixed_batch_of_members_on_different_launch_counts():
    """Members in the tile form whose steps record one or two horizontal WAF
    launches, before the batch's tuner makes them agree and after it."""
    print("[tile] mixed batch, members on different launch counts", flush=True)
    doms = [synth.config("small", **o)[:2] for o in (dict(), dict(jx=30, iy=26),
                                                     dict(jx=70, iy=22, kz=12))]
    knobs = [{MLC_VAR_MIXED_MERGE: 4}, {MLC_VAR_MIXED_MERGE: 1, MLC_VAR_WAF_HGROUP: 2},
             {MLC_VAR_MIXED_MERGE: 0, MLC_VAR_WAF_HGROUP: 1}]
    alone = []
    for (g, f), kn in zip(doms, knobs):
        with Moloch(g, MLC_MIXED) as m:
            m.load(f)
            m.init_moloch()
            m.moloch(4)
            alone.append({n: m.get(n) for n in FIELDS})
    counts = [run(g, f, MLC_MIXED, kn)[1] for (g, f), kn in zip(doms, knobs)]
    assert len(set(counts)) == 3, counts
    with MolochBatch([g for g, _ in doms], MLC_MIXED) as b:
        for i, (g, f) in enumerate(doms):
            b.member(i).load(f)
            b.member(i).init_moloch()
            b.member(i).set_variant(MLC_VAR_WAF_H, 1)
            for stage, value in knobs[i].items():
                b.member(i).set_variant(stage, value)
        b.step(2)
        b.autotune(1)
        for knob in (MLC_VAR_WAF_H, MLC_VAR_WAF_HGROUP, MLC_VAR_MIXED_MERGE):
            assert len({b.member(i).get_variant(knob) for i in range(3)}) == 1
        b.step(2)
        b.synchronize()
        for i in range(3):
            for n in FIELDS:
                assert np.array_equal(b.member(i).get(n), alone[i][n]), (i, n)
