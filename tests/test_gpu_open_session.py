"""Opening a session in one launch (``KVRuntime.import_session``) against the
reset and the single imports: stored bytes, lengths, generations, refusals."""
from __future__ import annotations

import pytest
import torch

from tests.helpers import randn_bf16

pytestmark = pytest.mark.gpu


def _runtime(n_slots=2, capacity=300):
    from kvrt import KVRuntime, LayerSpec

    return KVRuntime([
        LayerSpec(kv_heads=8, head_dim=64),
        LayerSpec(kv_heads=1, head_dim=256, layout="ring", window=33, ring_rows=37),
        LayerSpec(kv_heads=3, head_dim=128),
        LayerSpec(kv_heads=1, head_dim=256, shared_src=1),
        LayerSpec(kv_heads=2, head_dim=512, layout="ring", window=100, ring_rows=128),
    ], n_slots, capacity, max_q=1, device="cuda")


def _dirty(rt):
    for layer in (0, 1, 2, 4):
        for t in rt.storage(layer)[:2]:
            t.normal_()


# rows per layer: none, one, a ring exactly full, wrapped by one row and more, capacity
@pytest.mark.parametrize("rows", [(0, 0, 0, 0), (1, 1, 1, 1), (37, 37, 37, 128), (36, 38, 100, 129), (300, 300, 299, 255)])
@pytest.mark.parametrize("given", [5, 3])  # layers past the given ones are emptied
def test_one_launch_matches_reset_and_imports(rows, given):
    gen = torch.Generator().manual_seed(sum(rows) + given)
    rt, one = _runtime(), _runtime()
    kv = []
    for spec, s in zip(rt.layers, rows[:3] + (0,) + rows[3:]):
        # K and V rows as views of a longer, wider buffer
        wide = [randn_bf16(gen, (1, spec.kv_heads, s + 3, spec.head_dim + 64)).cuda() for _ in range(2)]
        kv.append(tuple(w[:, :, 1:1 + s, 64:] for w in wide))
    kv[3] = (None, None)
    for r in (rt, one):
        _dirty(r)
    for t, u in zip(_stores(rt), _stores(one)):
        u.copy_(t)
    rt.reset_slot(1)
    for layer in (l for l in (0, 1, 2, 4) if l < given):
        rt.import_(1, layer, *kv[layer])
    launches = one.counters()["launches"]
    g = one.import_session(1, kv[:given])
    assert one.counters()["launches"] == launches + 1
    assert g == rt.slot_generation(1) == one.slot_generation(1)
    for t, u in zip(_stores(rt), _stores(one)):
        assert torch.equal(t[1], u[1]) and torch.equal(t[0], u[0])
    for r in (rt, one):
        r.sync_lengths()
    assert [rt.seq_length(1, l) for l in range(5)] == [one.seq_length(1, l) for l in range(5)]
    assert one.health() == 0


def _stores(rt):
    return [t for layer in (0, 1, 2, 4) for t in rt.storage(layer)[:2]]


def test_prefix_mask_and_own_rows():
    gen = torch.Generator().manual_seed(9)
    rt = _runtime()
    kv = [(randn_bf16(gen, (1, s.kv_heads, 40, s.head_dim)).cuda(),) * 2 for s in rt.layers]
    rt.import_session(0, kv, torch.ones(8, dtype=torch.int64))
    assert rt.slot_info(0)["prefix_len"] == 8
    # a session opened from its own slot's rows: the reset comes first
    rt.import_session(0, [rt.layer_view(0, 0)])
    assert rt.slot_info(0)["prefix_len"] == 0 and rt.seq_length(0, 0) == 40 and rt.seq_length(0, 2) == 0
    assert not rt.storage(0)[0][0].any()


def test_refusals_are_those_of_the_single_calls():
    from kvrt import KVRTError

    rt = _runtime()
    ok = torch.zeros((1, 8, 5, 64), dtype=torch.bfloat16, device="cuda")
    bad = torch.zeros((1, 2, 5, 256), dtype=torch.bfloat16, device="cuda")
    with pytest.raises(KVRTError) as e:
        rt.import_session(0, [(ok, ok), (bad, bad)])
    assert e.value.code == -1
    assert rt.seq_length(0, 0) == 5 and rt.seq_length(0, 1) == 0  # the layers before it are in
    with pytest.raises(ValueError):
        rt.import_session(0, [(ok.cpu(), ok.cpu())])
    assert rt.seq_length(0, 0) == 0
    with pytest.raises(KVRTError):
        rt.import_session(7, [(ok, ok)])
    assert rt.health() == 0


@pytest.mark.parametrize("n_layers", [48, 49, 100])
def test_more_layers_than_one_launch_takes(n_layers):
    """48 layers per launch: a topology past them opens in as few launches as
    hold it, every layer's rows, zeros and lengths in place."""
    from kvrt import KVRuntime, LayerSpec

    gen = torch.Generator().manual_seed(n_layers)
    rt = KVRuntime([LayerSpec(kv_heads=1 + l % 3, head_dim=64) for l in range(n_layers)], 2, 24, max_q=1, device="cuda")
    for l in range(n_layers):
        for t in rt.storage(l)[:2]:
            t.normal_()
    other = [t[0].clone() for l in range(n_layers) for t in rt.storage(l)[:2]]
    kv = [tuple(randn_bf16(gen, (1, 1 + l % 3, 5 + l % 19, 64)).cuda() for _ in range(2)) for l in range(n_layers)]
    before = rt.counters()["launches"]
    rt.import_session(1, kv, None)
    assert rt.counters()["launches"] - before == (n_layers + 47) // 48
    rt.sync_lengths()
    for l in range(n_layers):
        rows = 5 + l % 19
        assert rt.seq_length(1, l) == rows
        for t, src in zip(rt.storage(l)[:2], kv[l]):
            assert torch.equal(t[1, :, :rows], src[0]) and not t[1, :, rows:].any()
    assert all(torch.equal(a, b[0]) for a, b in zip(other, (t for l in range(n_layers) for t in rt.storage(l)[:2])))
    assert rt.health() == 0
