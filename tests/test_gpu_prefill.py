"""GPU parity of the chunked-prefill MFMA attention (kvrt_attend_prefill_async)
against the fp64 oracle: Gemma sliding layers at the reference's canonical
prefill length (Q = 291 with a 512 window, ring of 802 rows), Gemma full
layers (D = 512), talker prefill (16 q / 8 kv heads), Q3..Q8 text appends, paged
storage and ragged streams. Tolerance max-abs 1e-2 on bf16 outputs."""
from __future__ import annotations

import math

import numpy as np
import pytest
import torch

from oracle import kv_oracle as O
from tests.helpers import randn_bf16, to_np

pytestmark = pytest.mark.gpu
ATOL = 1e-2


def _setup(hq, hkv, d, window, layout, prefix_lens, qn, seed):
    from kvrt import KVRuntime, LayerSpec

    gen = torch.Generator().manual_seed(seed)
    kw = {}
    if layout == "ring":
        spec = LayerSpec(kv_heads=hkv, head_dim=d, layout="ring", window=window, ring_rows=window + qn - 1)
    elif layout == "paged":
        spec = LayerSpec(kv_heads=hkv, head_dim=d, layout="paged", window=window)
        kw = dict(block_size=16, pool_pages=512)
    else:
        spec = LayerSpec(kv_heads=hkv, head_dim=d, window=window)
    n = len(prefix_lens)
    rt = KVRuntime([spec], n, max(prefix_lens) + qn + 8, max_q=qn, device="cuda", **kw)
    orc = O.OracleCache([O.OracleLayer(hkv, d, window)], n)
    for s, p in enumerate(prefix_lens):
        if p:
            k, v = randn_bf16(gen, (1, hkv, p, d)), randn_bf16(gen, (1, hkv, p, d))
            rt.import_(s, 0, k.cuda(), v.cuda())
            orc.append(s, 0, to_np(k[0]), to_np(v[0]))
    # the chunk's own K/V rows go in first (prefill-length append), then attention
    k, v = randn_bf16(gen, (n, hkv, qn, d)), randn_bf16(gen, (n, hkv, qn, d))
    rt.append(0, k.cuda(), v.cuda(), list(range(n)))
    for s in range(n):
        orc.append(s, 0, to_np(k[s]), to_np(v[s]))
    q = randn_bf16(gen, (n, hq, qn, d), 0.5)
    return rt, orc, q


def _check(rt, orc, q, scale, prefill=True):
    n = q.shape[0]
    fn = rt.attend_prefill if prefill else rt.attend
    out = fn(0, q.cuda(), list(range(n)), scale)
    torch.cuda.synchronize()
    assert rt.health() == 0
    worst = 0.0
    for s in range(n):
        ref = orc.attend(s, 0, to_np(q[s]), scale)
        worst = max(worst, float(np.abs(to_np(out[s]) - ref).max()))
    assert worst <= ATOL, worst
    return out


@pytest.mark.parametrize(
    "hq,hkv,d,window,layout,prefix,qn",
    [
        (8, 1, 256, 512, "ring", [0], 291),          # Gemma sliding, canonical prefill target
        (8, 1, 256, 512, "ring", [700], 291),        # ... over a ring that has wrapped
        (8, 1, 512, 0, "contig", [0, 130], 291),     # Gemma full layers, D = 512
        (16, 8, 128, 0, "contig", [37, 0, 400], 100),  # talker prefill, ragged prefixes
        (8, 1, 256, 512, "ring", [1500, 20], 8),     # Q8 text append (64 rows per kv head)
        (8, 1, 256, 0, "contig", [300], 3),          # Q3 text append
        (4, 4, 64, 0, "paged", [45, 300], 37),       # paged pool
        (4, 2, 128, 24, "paged", [200], 50),         # paged + window
        # few query blocks over many keys: the keys of a block are split over
        # workgroups and the partials merged (8 and 2 key ranges)
        (8, 1, 512, 0, "contig", [2000, 900], 64),
        (4, 2, 128, 600, "paged", [1500], 40),
        # the talker's whole-response prefill: two row blocks x two key parts
        (16, 8, 128, 0, "contig", [0, 0, 0, 0], 512),
        # a wrapped ring layout, GQA groups of 4
        (8, 2, 128, 200, "ring", [900, 64], 77),
        # talker-sized grids: an odd block count over ragged prefixes, and a
        # windowed ring layout
        (16, 8, 128, 0, "contig", [0, 37, 300, 5], 481),
        (16, 8, 128, 200, "ring", [0, 900, 64, 10], 300),
        # GQA groups of 6 and 3 (index splits by a divisor that is not a power
        # of two)
        (6, 1, 128, 0, "contig", [100, 37], 50),
        (12, 2, 256, 512, "ring", [300], 40),
        (3, 1, 64, 0, "paged", [70], 33),
        # a key split (one long stream) leaves the short streams' later key
        # ranges empty: their clamped fetches must stay on mapped pages (the
        # health check below would report the device flag otherwise)
        (12, 4, 128, 0, "paged", [31, 839, 241], 1),
        (8, 2, 64, 0, "paged", [5, 1500], 3),
    ],
)
def test_prefill_matches_oracle(hq, hkv, d, window, layout, prefix, qn):
    rt, orc, q = _setup(hq, hkv, d, window, layout, prefix, qn, seed=hq * 7 + d + qn)
    _check(rt, orc, q, 1.0 / math.sqrt(d))


@pytest.mark.parametrize("d", [64, 128, 256, 512])
@pytest.mark.parametrize(
    "hq,hkv,window,layout,prefix,qn,scale,grow",
    [
        # last row of a 32-row block, one past it, one short of it
        (8, 1, 0, "contig", [0], 4, 1.0, 0.0),
        (8, 1, 0, "contig", [29, 31, 32, 33], 5, 1.0, 0.0),
        (5, 1, 0, "contig", [64], 13, 1.0, 0.0),
        (1, 1, 0, "contig", [0, 95], 33, 1.0, 0.0),
        # more row blocks than one workgroup's, keys split over workgroups
        (12, 2, 0, "contig", [1100, 3], 23, 1.0, 0.0),
        (8, 1, 90, "ring", [700, 40], 37, 1.0, 0.0),
        (8, 2, 0, "paged", [513], 31, 1.0, 0.0),
        # scores that rise along the keys move the running max again and again
        (8, 1, 0, "contig", [600], 9, 1.0, 12.0),
        (8, 1, 0, "contig", [300], 20, -1.0, 12.0),
        (8, 1, 200, "ring", [90], 64, 0.0, 0.0),
    ],
)
def test_prefill_row_blocks_and_key_blocks_at_their_edges(d, hq, hkv, window, layout, prefix, qn, scale, grow):
    """Rows (q heads x queries) in blocks of 32, keys in blocks of 32 over 1, 2
    or 4 parts and over workgroups; scales of either sign and zero. With
    ``grow`` the keys' lengths rise along the positions (scores of up to about
    grow * 8 log2 units), so that the accumulators are rescaled; outputs are
    then single values of N(0,1) rather than averages. Bound: an output's
    rounding to bf16 is at most 2^-8 of it, and 2e-3 covers the rest: |v| < 5
    times the weights' error, 2^-17 from their two bf16 terms and 100 * 2^-20
    from scores of up to 100 summed and scaled in fp32."""
    rt, orc, q = _setup(hq, hkv, d, window, layout, prefix, qn, seed=d + hq + qn)
    if grow:
        L = prefix[0] + qn
        k, v, _, _ = rt.storage(0)
        ramp = torch.linspace(0.05, grow, L).to(torch.bfloat16).float()
        kk = (k[0, :, :L].float().cpu() * ramp[None, :, None]).to(torch.bfloat16)
        vv = v[0, :, :L].clone()
        k[0, :, :L] = kk.cuda()
        orc = O.OracleCache([O.OracleLayer(hkv, d, window)], 1)
        orc.append(0, 0, to_np(kk), to_np(vv))
        q = q * 2
    n = q.shape[0]
    out = rt.attend_prefill(0, q.cuda(), list(range(n)), scale / math.sqrt(d))
    assert rt.health() == 0
    for i in range(n):
        ref = orc.attend(i, 0, to_np(q[i]), scale / math.sqrt(d))
        assert (np.abs(to_np(out[i]) - ref) <= 2.0 ** -8 * np.abs(ref) + 2e-3).all()


def test_prefill_single_query_and_decode_dispatch():
    """Q = 1 through the MFMA kernel; g * Q above 16 rows dispatches to it from attend()."""
    rt, orc, q = _setup(2, 1, 128, 0, "contig", [77], 1, seed=5)
    _check(rt, orc, q, 0.1)
    rt, orc, q = _setup(8, 1, 256, 512, "ring", [900], 4, seed=6)  # 32 rows per kv head
    _check(rt, orc, q, 1.0 / 16, prefill=False)


def test_prefill_and_decode_agree_where_both_apply():
    rt, orc, q = _setup(4, 2, 128, 0, "contig", [500, 123], 4, seed=7)
    a = rt.attend_prefill(0, q.cuda(), [0, 1], 0.09)
    b = rt.attend(0, q.cuda(), [0, 1], 0.09)  # 8 rows per kv head: decode kernel
    torch.cuda.synchronize()
    assert float((a.float() - b.float()).abs().max()) <= ATOL


def test_prefill_rejects_what_it_cannot_see():
    from kvrt import KVRTError, KVRuntime, LayerSpec

    rt = KVRuntime([LayerSpec(kv_heads=1, head_dim=256, layout="ring", window=64, ring_rows=64 + 8 - 1)], 1, 4096,
                   max_q=8, device="cuda")
    x = torch.zeros((1, 1, 1000, 256), dtype=torch.bfloat16, device="cuda")
    rt.import_(0, 0, x, x)
    q = torch.zeros((1, 8, 16, 256), dtype=torch.bfloat16, device="cuda")
    with pytest.raises(KVRTError) as e:  # 16 queries need 16 + 63 resident rows, the ring keeps 71
        rt.attend_prefill(0, q, [0], 0.1)
    assert e.value.code == -2
    q = torch.zeros((1, 8, 1001, 256), dtype=torch.bfloat16, device="cuda")
    with pytest.raises(KVRTError):  # more queries than positions
        rt.attend_prefill(0, q, [0], 0.1)
    assert rt.health() == 0


@pytest.mark.parametrize("logical_q", [3, 5, 7])
def test_even_physical_q_with_pad_row_truncation_equals_the_logical_q(logical_q):
    """The reference's variable-Q text step runs an even physical Q (logical
    + 1 pad row for odd logical Q), then truncates the cursor to the logical
    end (gemma4_listener_microbatch_impl.inc:3476-3586,
    native_listener_microbatch.py:1640-1655). kvrt takes any Q directly; both
    routes must give the same logical rows, cache and next decode."""
    from kvrt import KVRuntime, LayerSpec

    gen = torch.Generator().manual_seed(logical_q)
    hq, hkv, d = 8, 1, 256
    prefix = randn_bf16(gen, (1, hkv, 300, d))
    k = randn_bf16(gen, (1, hkv, logical_q + 1, d))
    v = randn_bf16(gen, (1, hkv, logical_q + 1, d))
    q = randn_bf16(gen, (1, hq, logical_q + 1, d), 0.5)
    outs, rts = [], []
    for physical in (logical_q, logical_q + 1):
        rt = KVRuntime([LayerSpec(kv_heads=hkv, head_dim=d, window=512)], 1, 512, max_q=8, device="cuda")
        rt.import_(0, 0, prefix.cuda(), prefix.cuda())
        rt.append(0, k[:, :, :physical].contiguous().cuda(), v[:, :, :physical].contiguous().cuda(), [0])
        outs.append(rt.attend_prefill(0, q[:, :, :physical].contiguous().cuda(), [0], 1 / 16))
        rt.truncate(0, 300 + logical_q)
        rts.append(rt)
    torch.cuda.synchronize()
    direct, padded = outs
    assert float((direct.float() - padded[:, :, :logical_q].float()).abs().max()) <= 1e-6
    assert rts[0].seq_length(0) == rts[1].seq_length(0) == 300 + logical_q
    qd = randn_bf16(gen, (1, hq, 1, d), 0.5).cuda()
    kd = randn_bf16(gen, (1, hkv, 1, d)).cuda()
    a = rts[0].append_attend(0, qd, kd, kd, [0], 1 / 16)
    b = rts[1].append_attend(0, qd, kd, kd, [0], 1 / 16)
    torch.cuda.synchronize()
    assert torch.equal(a, b)
    assert rts[0].health() == 0 and rts[1].health() == 0


# the prefill benchmark's cases: name, streams, Hq, Hkv, D, Q, prefix, window
BENCH_SHAPES = [
    ("thinker_sliding_q291", 4, 8, 1, 256, 291, 2048, 512),
    ("thinker_full_d512_q291", 4, 8, 1, 512, 291, 2048, 0),
    ("talker_prefill_q512", 4, 16, 8, 128, 512, 0, 0),
    ("thinker_prefill_q2048", 1, 8, 1, 256, 2048, 0, 0),
    ("thinker_full_d512_q2048", 4, 8, 1, 512, 2048, 2048, 0),
]


@pytest.mark.parametrize("name,n,hq,hkv,d,qn,prefix,window", BENCH_SHAPES, ids=[c[0] for c in BENCH_SHAPES])
def test_prefill_at_the_benchmark_shapes_on_sampled_rows(name, n, hq, hkv, d, qn, prefix, window):
    """The full-size chunks the prefill benchmark times (key-split grids,
    query-block pairs, the D 512 path, a wrapped ring): every q head of 12
    query rows per stream (the first, the last and 10 seeded others) against
    the oracle, which attends those rows only."""
    import random

    from kvrt import KVRuntime, LayerSpec

    gen = torch.Generator().manual_seed(qn + d + prefix)
    layout = "ring" if window else "contig"
    spec = LayerSpec(kv_heads=hkv, head_dim=d, layout=layout, window=window,
                     ring_rows=window + qn - 1 if window else 0)
    L = prefix + qn
    rt = KVRuntime([spec], n, L + 8, max_q=qn, device="cuda")
    ks, vs = [], []
    for s in range(n):
        k, v = randn_bf16(gen, (1, hkv, L, d)), randn_bf16(gen, (1, hkv, L, d))
        rt.import_(s, 0, k.cuda(), v.cuda())
        ks.append(to_np(k[0]))
        vs.append(to_np(v[0]))
    q = randn_bf16(gen, (n, hq, qn, d), 0.5)
    scale = 1.0 / math.sqrt(d)
    out = rt.attend_prefill(0, q.cuda(), list(range(n)), scale)
    torch.cuda.synchronize()
    assert rt.health() == 0
    r = random.Random(qn * 7 + d)
    worst = 0.0
    for s in range(n):
        rows = sorted({0, qn - 1, *r.sample(range(qn), min(qn, 10))})
        ref = O.attend(to_np(q[s])[:, rows], ks[s], vs[s], np.array([L - qn + i for i in rows]), scale, window)
        worst = max(worst, float(np.abs(to_np(out[s])[:, rows] - ref).max()))
    assert worst <= ATOL, worst


@pytest.mark.parametrize("hq,hkv,d,window,layout,prefix", [
    (8, 2, 64, 0, "paged", 1500), (16, 8, 128, 0, "paged", 60), (8, 1, 512, 0, "paged", 700), (8, 1, 256, 90, "paged", 200),
    (16, 8, 128, 0, "contig", 900), (8, 1, 256, 512, "ring", 300)])
def test_captured_prefill_replayed_below_its_query_count(hq, hkv, d, window, layout, prefix):
    """A captured chunk replayed after a rollback to fewer rows than queries:
    query i sits at position length - Q + i, and those before position 0 see no
    keys (zeros), whatever the other slots hold. The page arithmetic itself is
    tests/test_prefill_range.py's."""
    qn, left = 70, (7, 33)
    rt, orc, q = _setup(hq, hkv, d, window, layout, [prefix, prefix], qn, seed=d + hq)
    scale = 1.0 / math.sqrt(d)
    q, out = q.cuda(), torch.empty(q.shape, dtype=torch.bfloat16, device="cuda")
    rt.attend_prefill(0, q, [0, 1], scale, out=out)
    rt.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        rt.attend_prefill(0, q, [0, 1], scale, out=out)
    rt.sync_lengths()
    if layout == "ring":  # the rows of [0, left) are no longer stored: only an empty slot can be rolled back to
        left = (0, 0)
    for s, n in enumerate(left):
        rt.truncate(s, n)
        orc.truncate(s, 0, n)
    rt.synchronize()
    for _ in range(3):
        out.fill_(7.0)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        for s, n in enumerate(left):
            assert not out[s, :, :qn - n].any()
            if n:
                ref = orc.attend(s, 0, to_np(q[s])[:, qn - n:], scale)
                assert float(np.abs(to_np(out[s])[:, qn - n:] - ref).max()) <= ATOL
    assert rt.health() == 0


@pytest.mark.parametrize("d,hq,hkv,prefix,qn,window,split", [
    (512, 8, 1, 236, 64, 0, True), (512, 8, 1, 20, 64, 0, False), (256, 8, 1, 1500, 30, 0, True),
    (256, 8, 1, 100, 200, 512, False), (128, 16, 8, 2000, 20, 0, True), (128, 16, 8, 100, 60, 0, False)])
@pytest.mark.parametrize("where", ["k", "q"])
def test_nan_stays_nan_with_and_without_a_key_split(d, hq, hkv, prefix, qn, window, split, where):
    """A NaN in a key that every query sees makes their rows NaN, one in a query
    its own row, whichever launch shape the chunk takes."""
    rt, _, q = _setup(hq, hkv, d, window, "contig", [prefix], qn, seed=3)
    want = torch.zeros((1, hq, qn, d), dtype=torch.bool)
    if where == "k":
        rt.storage(0)[0][0, 0, prefix - 5, 3] = float("nan")  # kv head 0, seen by all queries
        want[:, :hq // hkv] = True
    else:
        q[0, 1, qn // 2, 7] = float("nan")
        want[0, 1, qn // 2] = True
    launches = rt.counters()["launches"]
    out = rt.attend_prefill(0, q.cuda(), [0], 1.0 / math.sqrt(d))
    assert rt.counters()["launches"] == launches + (2 if split else 1)
    assert torch.equal(out.isnan().cpu(), want)


def _sampled(hq, hkv, d, window, layout, lens, qn, mask=0):
    """A chunk of qn queries over sessions of lens rows against the oracle: every
    q head of the first, the last and 8 other query rows of each."""
    import random

    from kvrt import KVRuntime, LayerSpec

    gen = torch.Generator().manual_seed(qn + d + lens[0])
    r = random.Random(qn * 7 + d)
    ring = dict(ring_rows=window + qn - 1) if layout == "ring" else {}
    rt = KVRuntime([LayerSpec(kv_heads=hkv, head_dim=d, layout=layout, window=window, **ring)], len(lens),
                   max(lens) + 8, max_q=qn, device="cuda", pool_seed=3,
                   pool_pages=sum(n // 16 + 2 for n in lens) if layout == "paged" else 0)
    ks, vs, hide = [], [], None
    for s, n in enumerate(lens):
        k, v = randn_bf16(gen, (1, hkv, n, d)), randn_bf16(gen, (1, hkv, n, d))
        rt.import_(s, 0, k.cuda(), v.cuda())
        ks.append(to_np(k[0]))
        vs.append(to_np(v[0]))
    if mask:
        hide = (torch.rand(mask, generator=gen) < 0.5).to(torch.int64)
        hide[0] = 1  # every query sees a key
        for s in range(len(lens)):
            rt.set_prefix_attention(s, hide)
    q = randn_bf16(gen, (len(lens), hq, qn, d), 0.5)
    out = rt.attend_prefill(0, q.cuda(), list(range(len(lens))), 1.0 / math.sqrt(d))
    torch.cuda.synchronize()
    assert rt.health() == 0
    for s, n in enumerate(lens):
        rows = sorted({0, qn - 1, *r.sample(range(qn), min(qn, 8))})
        for i in rows:
            pos = n - qn + i
            seen = np.arange(max(0, pos - window + 1) if window else 0, pos + 1)
            if hide is not None:
                seen = seen[(seen >= mask) | (hide.numpy()[np.minimum(seen, mask - 1)] != 0)]
            ref = O.attend(to_np(q[s])[:, i:i + 1], ks[s][:, seen], vs[s][:, seen], np.array([len(seen) - 1]),
                           1.0 / math.sqrt(d), 0)
            assert float(np.abs(to_np(out[s])[:, i:i + 1] - ref).max()) <= ATOL, (s, i)


@pytest.mark.parametrize("hq,hkv,d,window,layout,lens,qn,mask", [
    # four row blocks, one key part: many key blocks, every layout, a prefix mask
    (16, 8, 128, 0, "contig", [1000, 1100, 1000, 1013], 1000, 0), (16, 8, 128, 300, "ring", [1000] * 4, 1000, 0),
    (16, 8, 128, 0, "paged", [1000, 1003, 1100, 1000], 1000, 0), (16, 8, 128, 0, "contig", [1000] * 4, 1000, 200),
    (16, 8, 64, 0, "contig", [1200] * 4, 1200, 0), (16, 8, 64, 200, "ring", [1200] * 4, 1200, 0),
    (16, 8, 64, 0, "paged", [1200] * 4, 1200, 77),
    (8, 1, 256, 512, "ring", [1200] * 3, 1200, 0), (8, 1, 256, 0, "contig", [1400, 1500, 1400, 1400], 1400, 90),
    (8, 1, 256, 0, "paged", [1400] * 4, 1400, 0),
    # two row blocks x four key parts
    (16, 8, 128, 0, "contig", [947, 900, 800], 274, 0), (16, 8, 128, 700, "ring", [1500, 947, 800], 274, 0),
    (16, 8, 128, 0, "paged", [300, 217], 40, 150), (8, 2, 64, 0, "paged", [300, 217], 40, 0),
    # two x two, and one x four with a key split
    (16, 8, 64, 0, "contig", [300, 333, 400, 420], 300, 0), (16, 8, 64, 150, "ring", [700] * 4, 300, 0),
    (16, 8, 128, 0, "contig", [700, 2000], 24, 120), (16, 8, 64, 0, "contig", [700], 24, 0),
    # PAGED over few keys: one part, then two
    (16, 8, 128, 0, "paged", [32, 13], 12, 0), (8, 2, 64, 0, "paged", [33, 160], 20, 30),
])
def test_prefill_launch_shapes(hq, hkv, d, window, layout, lens, qn, mask):
    _sampled(hq, hkv, d, window, layout, lens, qn, mask)


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("hq,hkv,window,layout,lens,qn,mask", [
    # tiles of 16 queries x 32 keys: one short, full, one over; 1 to 4 heads per
    # workgroup and groups of 5 and 6; rings that have wrapped; prefix masks
    (8, 4, 0, "contig", [15, 31], 15, 0), (8, 4, 0, "contig", [16, 32], 16, 0), (8, 4, 0, "contig", [17, 33], 17, 0),
    (4, 4, 0, "contig", [65, 96, 97], 40, 0), (16, 8, 0, "contig", [128, 150, 129], 33, 70),
    (6, 2, 0, "contig", [100, 64], 50, 20), (5, 1, 0, "contig", [60], 9, 0), (6, 1, 0, "contig", [64, 33], 20, 0),
    (8, 2, 0, "contig", [64, 50], 31, 31), (16, 8, 40, "ring", [900, 70], 50, 0), (8, 8, 100, "ring", [150, 333], 18, 60),
    (6, 2, 33, "ring", [500, 45], 45, 0), (16, 8, 0, "contig", [300, 310, 290, 305], 200, 100),
    # two query blocks on the same tiles: 1, 2, 3 and 4 heads
    (8, 8, 0, "contig", [320] * 4, 300, 0), (16, 8, 0, "contig", [150] * 8, 140, 64), (16, 8, 64, "ring", [500] * 8, 140, 0),
    (24, 8, 0, "contig", [170] * 8, 170, 0), (32, 8, 0, "contig", [150] * 8, 150, 33),
])
def test_prefill_over_few_keys(d, hq, hkv, window, layout, lens, qn, mask):
    _sampled(hq, hkv, d, window, layout, lens, qn, mask)


@pytest.mark.parametrize("hq,hkv,d,window,layout,n_rows,qn,keys", [
    # four 32-row blocks per workgroup: 64 queries of 2 heads, 128 of one, 16 of 8
    (2, 1, 512, 0, "contig", 300, 100, 264 + 300), (1, 1, 512, 0, "contig", 300, 130, 298 + 300),
    (8, 1, 512, 40, "contig", 500, 20, (39 + 16) + (39 + 4)),
    # 16-query blocks, four and two heads per workgroup
    (4, 1, 128, 0, "contig", 60, 20, 56 + 60), (8, 4, 128, 0, "contig", 60, 20, 4 * (56 + 60)),
])
def test_attended_counters_are_the_rows_read(hq, hkv, d, window, layout, n_rows, qn, keys):
    rt, _, q = _setup(hq, hkv, d, window, layout, [n_rows - qn], qn, seed=1)
    before = rt.counters()
    rt.attend_prefill(0, q.cuda(), [0], 0.1)
    after = rt.counters()
    assert after["attended_keys"] - before["attended_keys"] == keys
    assert after["attended_bytes"] - before["attended_bytes"] == keys * d * 4
