"""The native call module's own error handling, without a GPU: the entry points
are replaced by host functions and the tensors are GPU tensors in name only
(their storage is host memory that nothing reads)."""
from __future__ import annotations

import subprocess
import sys
import textwrap
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]

PROGRAM = """
import ctypes, sys, threading
sys.path.insert(0, {pkg!r})
import torch
from kvrt import TalkerMask, _lib

mod = _lib.load_calls()
host = torch.zeros(4096, dtype=torch.uint8)
storage = torch._C._construct_storage_from_data_pointer(host.data_ptr(), torch.device("cuda", 0), 4096)

def gpu(size, stride, dtype=torch.bfloat16):
    return torch._C._construct_CUDA_Tensor_From_Storage_And_Metadata(
        dict(size=size, stride=stride, dtype=dtype, storage_offset=0), storage)

ok = ctypes.CFUNCTYPE(ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p)(lambda c, s: 0)
addr = lambda f: ctypes.cast(f, ctypes.c_void_p).value
cxx = ctypes.CDLL("libstdc++.so.6")
t = gpu((1, 2, 1, 64), (128, 64, 64, 1))
lens = gpu((1,), (1,), torch.int32)
mask = TalkerMask(prefix_start=0, audio_start=4, prefix_position=2, audio_position=6)
calls = dict(
    append_attend=lambda: mod.append_attend(8, 0, 0, [0], 0.5, t, t, t, t),
    attend=lambda: mod.attend(8, 0, 0, (0,), 0.5, t, t),
    attend_talker=lambda: mod.attend_talker(8, 0, 0, [0], 0.5, t, t, [mask]),
    write_positions=lambda: mod.write_positions(8, 0, 0, [0], [[3]], t, t),
    append_gather=lambda: mod.append_gather(8, 0, 0, [0], t, t, t, t, None),
    attend_tensors=lambda: mod.attend_tensors(0, 0.5, 0, t, t, t, lens, t),
)
for thrown in ("_ZSt17__throw_bad_allocv", "_ZSt16__throw_bad_castv"):
    f = addr(getattr(cxx, thrown))
    mod.connect(TalkerMask, addr(ok), f, f, f, f, f, f)
    for name, call in calls.items():
        assert call() == -3, name
        # the interpreter lock is held again: other threads and calls run
        seen = []
        th = threading.Thread(target=lambda: seen.append(call()))
        th.start()
        th.join()
        assert seen == [-3], name
# a bind that refuses leaves the call to the general path, nothing run
no = ctypes.CFUNCTYPE(ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p)(lambda c, s: -2)
mod.connect(TalkerMask, addr(no), f, f, f, f, f, f)
assert [c() for n, c in calls.items() if n != "attend_tensors"] == [1] * 5
print("done")
"""


def test_an_exception_from_a_call_is_an_error_and_keeps_the_interpreter_lock():
    """A C++ exception out of an entry point (its vectors can fail to allocate) is
    a device error, never a retry: the call may have enqueued work."""
    prog = textwrap.dedent(PROGRAM.format(pkg=str(ROOT / "gemma-4-omni_amd")))
    res = subprocess.run([sys.executable, "-c", prog], capture_output=True, text=True, timeout=300)
    assert res.returncode == 0 and res.stdout.strip().endswith("done"), (res.returncode, res.stderr[-2000:])
