"""The native calls (kvrt_pycall) against the general ctypes path: the same
outputs, lengths and refusals for every form of argument either accepts."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from tests.helpers import randn_bf16


class _General:
    """Stands in for the native module: every call takes the general path."""

    def __getattr__(self, name):
        return lambda *a: 1


def _outcome(fn):
    try:
        r = fn()
        return [t for t in (r if isinstance(r, tuple) else (r,)) if t is not None]
    except Exception as e:  # noqa: BLE001 - the refusal itself is compared
        return (type(e), str(e))


def test_cpu_tensors_take_the_general_path():
    """Nothing but plain GPU tensors is read: 1, with nothing done."""
    from kvrt.runtime import calls

    c, t = calls(), torch.zeros((1, 2, 1, 64), dtype=torch.bfloat16)
    assert c.append_attend(1, 0, 0, [0], 1.0, t, t, t, t) == 1
    assert c.attend_tensors(0, 1.0, 0, t, t, t, t, t) == 1
    assert c.attend(1, 0, 0, [0], 1.0, None, t) == 1 and c.attend() == 1
    assert c.write_positions(1, 0, 2 ** 40, [0], [[0]], t, t) == 1


FORMS = {
    "plain": {},
    "tuple slots": {"slots": (0, 1)},
    "numpy slots": {"slots": np.array([0, 1])},
    "int scale": {"scale": 1},
    "strided q": {"q": lambda q: q.transpose(1, 2).contiguous().transpose(1, 2)},
    "parameter": {"q": lambda q: torch.nn.Parameter(q, requires_grad=False)},
    "float16 q": {"q": lambda q: q.half()},
    "fp32 q": {"q": lambda q: q.float()},
    "cpu q": {"q": lambda q: q.cpu()},
    "bad slot": {"slots": [0, 7]},
    "twice": {"slots": [1, 1]},
    "too few": {"slots": [0]},
    "bad layer": {"layer": 9},
    "nan": {"scale": float("nan")},
    "5 dims": {"q": lambda q: q.unsqueeze(0)},
}


@pytest.mark.gpu
@pytest.mark.parametrize("form", list(FORMS))
def test_native_calls_match_the_general_path(form):
    from kvrt import KVRuntime, LayerSpec, TalkerMask, attend_tensors
    from kvrt import runtime as R

    f = FORMS[form]
    layer, slots, scale = f.get("layer", 0), f.get("slots", [0, 1]), f.get("scale", 0.1)
    gen = torch.Generator().manual_seed(5)
    hq, hkv, d, n = 4, 2, 128, 300
    held = randn_bf16(gen, (1, hkv, n, d)).cuda()
    q = f.get("q", lambda t: t)(randn_bf16(gen, (2, hq, 2, d)).cuda())
    k, v = randn_bf16(gen, (2, hkv, 2, d)).cuda(), randn_bf16(gen, (2, hkv, 2, d)).cuda()
    masks = [TalkerMask(prefix_start=100, audio_start=150, prefix_position=120, audio_position=n + 1)] * 2
    got = {}
    native = R.calls()
    for path, mod in (("native", native), ("general", _General())):
        rt = KVRuntime([LayerSpec(kv_heads=hkv, head_dim=d)], 2, n + 8, max_q=2, device="cuda")
        rt._call = R._calls = mod
        try:
            for s in (0, 1):
                rt.import_(s, 0, held, held)
            dst = [torch.zeros((2, hkv, n + 8, d), dtype=torch.bfloat16, device="cuda") for _ in range(2)]
            lens = torch.tensor([n, n - 7], dtype=torch.int32, device="cuda")
            got[path] = [
                _outcome(lambda: rt.append_attend(layer, q, k, v, slots, scale)),
                _outcome(lambda: rt.attend(layer, q, slots, scale)),
                _outcome(lambda: rt.write_positions(layer, k, v, slots, [[n, n + 1], [n - 3, n + 1]])),
                _outcome(lambda: rt.write_positions(layer, k, v, slots, [[n], [n]])),
                _outcome(lambda: rt.attend_talker(layer, q, slots, scale, masks)),
                _outcome(lambda: rt.attend_talker(layer, q, slots, scale, masks[:1])),
                _outcome(lambda: rt.append_gather(layer, k, v, slots, out=tuple(dst))),
                _outcome(lambda: attend_tensors(q, dst[0], dst[1], lens, scale)),
                [torch.tensor([rt.seq_length(s, 0) for s in (0, 1)])],
            ]
            torch.cuda.synchronize()
            rt.close()
            got[path].append(_outcome(lambda: rt.attend(0, k, [0, 1], 0.1)))
        finally:
            R._calls = native
    for a, b in zip(got["native"], got["general"]):
        if isinstance(a, tuple):
            assert a == b
        else:
            assert len(a) == len(b) and all(torch.equal(x, y) for x, y in zip(a, b))
