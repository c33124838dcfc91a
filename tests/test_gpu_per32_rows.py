"""The per32 layer's bank row kernels (xl_per32_rows.hip) at the edges of what
they take: partly filled passes of 32 sub-blocks per half wave (256, 768, 2,304
values), five full passes (5,120), hidden rows that do not fit LDS (6 x 5,120 and
16 x 2,048 values: the general row kernel), one and 16 picks, layers of one type
and of several.

Bars: each pick's output against the oracle's chain within 1e-3 (the SwiGLU's exp
may move one hidden quant), the combine bit-exact over the device's own rows, and
the down rows of picks whose hidden rows do not fit LDS (general kernel) equal to
the same picks' rows in smaller calls, bit for bit.
"""
from __future__ import annotations

import numpy as np
import pytest

import crosslane_amd as xl
from tests.conftest import max_rel

pytestmark = pytest.mark.gpu

XXS, XS, IQ1 = 16, 17, 29
KINDS = {"iq2": [(XXS, XXS, XS)], "iq1": [(IQ1,) * 3], "xs": [(XS, XS, XXS)], "mixed": [(XXS, XXS, IQ1), (IQ1, IQ1, XS), (XS, XS, XXS)]}
SEED = 0x32B


@pytest.mark.parametrize("dim,ff,k", [(256, 256, 1), (768, 2304, 5), (5120, 256, 3), (256, 5120, 4), (512, 5120, 6),
                                      (1024, 2048, 16)])
@pytest.mark.parametrize("kind", sorted(KINDS))
def test_layer_rows(orc, kind, dim, ff, k):
    E = 16
    types = np.array([[KINDS[kind][e % len(KINDS[kind])] for e in range(E)]], np.int32)
    rng = np.random.default_rng(dim + ff + k)
    x = rng.standard_normal(dim).astype(np.float32)
    shared = rng.standard_normal(dim).astype(np.float32)
    w = rng.random(k).astype(np.float32)
    ids = rng.choice(E, k, replace=False).astype(np.int32)
    print(f"[gpu-step] per32 rows {kind} {dim}x{ff} ids={ids.tolist()}", flush=True)
    with xl.Lane(dim, ff, 1, E, types, max_picks=16) as lane:
        lane.generate(seed=SEED)
        y, out = lane.layer_forward_per32(0, ids, x, w, shared)
        parts = [lane.layer_forward_per32(0, ids[i:i + 4], x)[0] for i in range(0, k, 4)]
    assert np.array_equal(np.concatenate(parts).view(np.uint32), y.view(np.uint32))
    for i, e in enumerate(ids):
        t = tuple(int(v) for v in types[0, e])
        want = orc.expert32(t, *orc.gen_expert(t, SEED, 0, int(e), dim, ff), dim, ff, x)
        assert max_rel(y[i], want) < 1e-3, f"pick {i}"
    assert np.array_equal(out.view(np.uint32), orc.combine(ids, w, y, shared).view(np.uint32))
