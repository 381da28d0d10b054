"""The chunked column solve (SoundColumnChunk) at the edges of its level chunks.

A thread owns ceil(kz / threads) levels of its column, its last thread fewer,
and passes the values its upper neighbour needs through LDS.  Bar: w, pai and
u after two steps equal the oracle's bit for bit, for column heights on both
sides of every chunk's edge, both kinds of metrics and with the divergence
filter on and off."""
import numpy as np
import pytest

import oracle_api as O
from regcm_amd import synth
from regcm_amd.moloch import MLC_FP64, MLC_VAR_COLUMN_J, MLC_VAR_TERRAIN, Moloch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kz,cj,filt", [
    (4, 16, 1), (9, 32, 1), (16, 16, 1), (17, 16, 0), (33, 32, 1), (42, 64, 1), (48, 16, 0),
    (48, 32, 1), (49, 16, 1), (49, 32, 0), (64, 32, 1), (65, 16, 1), (128, 16, 1)])
def test_column_heights_match_the_oracle(kz, cj, filt):
    print(f"[column] kz={kz} column_j={cj} divfilter={filt}", flush=True)
    g, f, _ = synth.config("small", nadv=1, nsound=3, kz=kz, do_divfilter=filt)
    ref = O.copy_fields(f)
    O.moloch_steps(g, ref, 2)
    own = (Ellipsis, slice(0, g.iy - 1), slice(0, g.jx - 1))
    for terrain in (2, 0):
        with Moloch(g, MLC_FP64) as m:
            m.set_variant(MLC_VAR_COLUMN_J, cj)
            m.load(f)
            m.init_moloch()
            m.set_variant(MLC_VAR_TERRAIN, terrain)
            m.moloch(2)
            m.synchronize()
            for n in ("w", "pai", "u"):
                assert np.array_equal(ref[n][own], m.get(n)[own]), (n, terrain)
