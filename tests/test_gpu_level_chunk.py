"""The default level chunks of the divergence and the momentum update follow
one rule: domains that differ by a few columns take the same ones, and what is
chosen divides the column as the rule's cost says.  Bar: the oracle's bits at
the chosen chunks on both sides of one block per CU."""
import numpy as np
import pytest

import oracle_api as O
from regcm_amd import synth
from regcm_amd.moloch import (MLC_FP64, MLC_MIXED, MLC_VAR_LEVEL_CHUNK, MLC_VAR_MOM_CHUNK, Moloch)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [MLC_FP64, MLC_MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("kz", [23, 41])
def test_no_edge_at_a_full_chip(kz, precision):
    """252 x 252 makes 252 blocks of 64 x 4 columns, 256 x 256 makes 256: one
    per CU or four fewer."""
    print(f"[level chunk] kz {kz} precision {precision}", flush=True)
    got = []
    for n in (252, 256):
        with Moloch(synth.Grid(n, n, kz, 5000.0, 15.0), precision) as m:
            got.append([m.get_variant(v) for v in (MLC_VAR_LEVEL_CHUNK, MLC_VAR_MOM_CHUNK)])
    assert got[0] == got[1], got


@pytest.mark.parametrize("jx,iy,kz", [(252, 252, 5), (258, 260, 5), (24, 20, 23)])
def test_chosen_chunks_match_the_oracle(jx, iy, kz):
    print(f"[level chunk] {jx}x{iy}x{kz}", flush=True)
    g, f, _ = synth.config("small", jx=jx, iy=iy, kz=kz, nqx=2, ipptls=0, nadv=1, nsound=2)
    ref = O.copy_fields(f)
    O.moloch_steps(g, ref, 1)
    with Moloch(g) as m:
        m.load(f)
        m.init_moloch()
        m.moloch(1)
        for n in ("u", "v", "w", "pai"):
            jn = g.jx if n == "u" else g.jx - 1
            im = g.iy if n == "v" else g.iy - 1
            assert np.array_equal(ref[n][..., :im, :jn], m.get(n)[..., :im, :jn]), n
