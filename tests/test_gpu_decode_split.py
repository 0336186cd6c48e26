"""bf16 MFMA decodes whose 16-key tiles do not divide over the launch's waves:
fewer tiles than waves, one left over, one short of another round, a partial
last tile, and fused appends that move from one to the next."""
import math

import numpy as np
import pytest
import torch

from oracle import kv_oracle as O

pytestmark = pytest.mark.gpu

# Outputs are bf16 averages of N(0, 1) values under nearly flat weights (|o|
# well below 1): half a bf16 step there is 2^-9, and P's two bf16 terms and the
# fp32 sums add less than 2^-14.
ATOL = 2.0 ** -8


def _np(t):
    return t.float().cpu().numpy()


@pytest.mark.parametrize("layout,d,hq,qn", [("contig", 128, 2, 1), ("contig", 256, 8, 1), ("ring", 128, 4, 2),
                                            ("paged", 64, 8, 1), ("contig", 512, 8, 2), ("paged", 512, 8, 1)])
@pytest.mark.parametrize("wgs", [1, 3])
def test_tiles_left_over(layout, d, hq, qn, wgs):
    from kvrt import KVRuntime, LayerSpec

    waves = 4 * wgs
    # before the first of three fused steps; tiles of 16 keys
    lens = [1 + qn, 16 * (waves - 1) - 1, 16 * waves - qn - 1, 16 * (5 * waves) - 1, 16 * (5 * waves + 1) - qn,
            16 * (6 * waves - 1) + 3]
    gen = torch.Generator().manual_seed(d + hq + qn + wgs)
    for n in lens:
        # (a ring of its own per length: the window takes every key but the oldest)
        kw = dict(window=max(qn, n), ring_rows=max(qn, n) + qn - 1) if layout == "ring" else {}
        rt = KVRuntime([LayerSpec(kv_heads=1, head_dim=d, layout=layout, **kw)], 1, n + 3 * qn, max_q=qn,
                       decode_wgs=wgs, decode_kernel="mfma", device="cuda",
                       pool_pages=(n + 3 * qn) // 16 + 2 if layout == "paged" else 0)
        orc = O.OracleCache([O.OracleLayer(1, d, kw.get("window", 0))], 1)
        bf = lambda shape: torch.randn(shape, generator=gen).to(torch.bfloat16)
        k, v = bf((1, 1, n, d)), bf((1, 1, n, d))
        rt.import_(0, 0, k.cuda(), v.cuda())
        orc.append(0, 0, _np(k[0]), _np(v[0]))
        for _ in range(3):
            q, k, v = bf((1, hq, qn, d)), bf((1, 1, qn, d)), bf((1, 1, qn, d))
            out = rt.append_attend(0, q.cuda(), k.cuda(), v.cuda(), [0], 0.25 / math.sqrt(d))
            orc.append(0, 0, _np(k[0]), _np(v[0]))
            ref = orc.attend(0, 0, _np(q[0]), 0.25 / math.sqrt(d))
            np.testing.assert_allclose(_np(out[0]), ref, rtol=2.0 ** -8, atol=ATOL, err_msg=f"{n} keys")
        assert rt.health() == 0
        assert rt.counters()["mfma_decodes"] == 3


@pytest.mark.parametrize("d,hq,qn,streams,mfma", [(256, 8, 1, 1, True), (256, 5, 1, 1, True), (64, 4, 2, 1, True),
                                                  (128, 4, 1, 1, True), (128, 3, 1, 1, True), (256, 4, 1, 1, False),
                                                  (128, 2, 1, 1, False), (256, 8, 1, 2, False)])
@pytest.mark.parametrize("keys", [1, 33, 513])
def test_short_decodes_by_stream_count(d, hq, qn, streams, mfma, keys):
    """Under 2048 keys a single stream's 8 rows, and 4 rows to head_dim 128, run
    on MFMA tiles; fewer rows and batches do not."""
    from kvrt import KVRuntime, LayerSpec

    gen = torch.Generator().manual_seed(d + hq + keys)
    bf = lambda shape: torch.randn(shape, generator=gen).to(torch.bfloat16)
    rt = KVRuntime([LayerSpec(kv_heads=1, head_dim=d)], streams, keys + 4, max_q=qn, device="cuda")
    orc = O.OracleCache([O.OracleLayer(1, d, 0)], streams)
    for s in range(streams):
        k, v = bf((1, 1, keys, d)), bf((1, 1, keys, d))
        rt.import_(s, 0, k.cuda(), v.cuda())
        orc.append(s, 0, _np(k[0]), _np(v[0]))
    q, k, v = bf((streams, hq, qn, d)), bf((streams, 1, qn, d)), bf((streams, 1, qn, d))
    out = rt.append_attend(0, q.cuda(), k.cuda(), v.cuda(), list(range(streams)), 0.25 / math.sqrt(d))
    for s in range(streams):
        orc.append(s, 0, _np(k[s]), _np(v[s]))
        np.testing.assert_allclose(_np(out[s]), orc.attend(s, 0, _np(q[s]), 0.25 / math.sqrt(d)), rtol=2.0 ** -8,
                                   atol=ATOL)
    assert rt.counters()["mfma_decodes"] == int(mfma) and rt.health() == 0
