"""The BERT driver's allocations, on host memory: the driver and the library run on a HIP runtime without kernels
(modules/host_hip.cpp) that counts allocations and refuses the one it is told to."""
import json
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PRELUDE = r"""
import ctypes, importlib, json, sys
import numpy as np
sys.path.insert(0, {root!r})
hip = ctypes.CDLL({shim!r}, mode=ctypes.RTLD_GLOBAL)   # in front of the real runtime
hip.hostHipLiveBytes.restype = ctypes.c_size_t
hip.hostHipFailAt.argtypes = [ctypes.c_long]
hip.hostHipAllocations.restype = hip.hostHipLaunches.restype = ctypes.c_long
rt = importlib.import_module("hands-on-mlir_amd.hom_runtime")
drv, lib = rt.load_driver(), rt.load_runtime()
L, H, HEADS, F, B, S, V = 3, 128, 2, 256, 2, 33, 50
def create():
    return drv.homBertCreate(L, H, HEADS, F, B, S, V, 1, 0)
def upload(e):
    for l in range(L):
        for which, n in enumerate((3 * H * H, H * H, H * F, H * F)):
            assert drv.homBertUpload(e, l, which, np.zeros(n, np.float16).ctypes.data, n) == 0
    for which, n in ((4, V * H), (5, S * H)):
        assert drv.homBertUpload(e, 0, which, np.zeros(n, np.float16).ctypes.data, n) == 0
"""


@pytest.fixture(scope="module")
def on_host(tmp_path_factory):
    shim = str(tmp_path_factory.mktemp("hip") / "libhost_hip.so")
    res = subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                          os.path.join(ROOT, "tests", "modules", "host_hip.cpp"), "-o", shim],
                         capture_output=True, text=True, timeout=300)
    assert res.returncode == 0, res.stderr

    def run(code):
        p = subprocess.run([sys.executable, "-c", PRELUDE.format(root=ROOT, shim=shim) + code], capture_output=True,
                           text=True, timeout=300)
        assert p.returncode == 0, p.stderr
        return json.loads(p.stdout.strip().splitlines()[-1])
    return run


def test_failed_allocation_is_reported_at_creation(on_host):
    """Whichever allocation fails, the encoder is not handed out and nothing is left behind; an encoder that was
    handed out allocates nothing in its forwards."""
    out = on_host(r"""
lib.homSetErrorMode(1)
hip.hostHipFailAt(-1)
e = create()
n = hip.hostHipAllocations()
upload(e)
hip.hostHipFailAt(-1)
drv.homBertForward(e, 1)
later, launches = hip.hostHipAllocations(), hip.hostHipLaunches()
packed = drv.homBertUsesPacked(e)
drv.homBertDestroy(e)
left = hip.hostHipLiveBytes()
refused, leaks = [], []
for k in range(n):
    hip.hostHipFailAt(k)
    e = create()
    refused.append(not e)
    if e:
        drv.homBertDestroy(e)
    leaks.append(hip.hostHipLiveBytes())
print(json.dumps(dict(n=n, later=later, launches=launches, packed=packed, left=left, refused=refused, leaks=leaks)))
""")
    assert out["packed"] == 1 and out["launches"] >= 5 * 3 and out["n"] > 10
    assert out["later"] == 0, "a forward allocates"
    assert out["left"] == 0 and not any(out["leaks"]), "memory left behind"
    # (one allocation is the first buffer of the pool of results, without which results take pageable memory)
    assert out["refused"].count(False) == 1


def test_layer_weights_are_held_once(on_host):
    """On packed weights the row-major layer weights and activations are not kept beside the packed ones, whatever a
    forward starts from; an encoder that a pinned kernel takes off them gives everything back when it goes."""
    out = on_host(r"""
L = 64
e = create()
upload(e)
drv.homBertForward(e, 1)
drv.homBertForward(e, 0)
assert drv.homBertUsesPacked(e) == 1
weights, live = L * (4 * H * H + 2 * H * F) * 2, hip.hostHipLiveBytes()
assert drv.homBertSetGemmChoice(e, 1, 1, 1) == 0 and drv.homBertUsesPacked(e) == 0
upload(e)
drv.homBertForward(e, 0)
drv.homBertDestroy(e)
# no memory for the row-major tensors: refused, and still on packed weights
lib.homSetErrorMode(1)
e = create()
hip.hostHipFailAt(5)
refused = [drv.homBertSetGemmChoice(e, 1, 1, 1), drv.homBertUsesPacked(e)]
hip.hostHipFailAt(-1)
drv.homBertDestroy(e)
print(json.dumps(dict(weights=weights, live=live, left=hip.hostHipLiveBytes(), refused=refused)))
""")
    assert out["weights"] < out["live"] < 1.2 * out["weights"]
    assert out["left"] == 0
    assert out["refused"] == [-3, 1]


def test_result_buffers_from_several_threads(on_host):
    """The pool of result buffers: no two threads hold the same memory at a time, buffers given back serve others,
    more than the pool hands out is refused, and nothing stays behind the last encoder."""
    out = on_host(r"""
import threading
e = create()
start, errors, seen = hip.hostHipLiveBytes(), [], set()
hip.hostHipFailAt(-1)
def work(t):
    rng = np.random.default_rng(t)
    held = []
    for i in range(600):
        if held and rng.random() < 0.5:
            p, n, v = held.pop(int(rng.integers(len(held))))
            if (np.ctypeslib.as_array((ctypes.c_ubyte * n).from_address(p)) != v).any():
                errors.append((t, i))
            drv.homHostBufferRelease(p)
        elif len(held) < 6:
            n, v = int(rng.integers(1, 300000)), int(rng.integers(256))
            p = drv.homHostBufferAcquire(n)
            ctypes.memset(p, v, n)
            held.append((p, n, v))
            seen.add(p)
    for p, n, v in held:
        drv.homHostBufferRelease(p)
threads = [threading.Thread(target=work, args=(t,)) for t in range(8)]
[t.start() for t in threads]; [t.join() for t in threads]
allocated, idle = hip.hostHipAllocations(), hip.hostHipLiveBytes() - start
kept = drv.homHostBufferAcquire(1000)
drv.homHostBufferRelease(12345)                   # (not a buffer of the pool)
big = drv.homHostBufferAcquire((1 << 30) + 1)
drv.homBertDestroy(e)
behind = hip.hostHipLiveBytes()
drv.homHostBufferRelease(kept)
print(json.dumps(dict(errors=errors, allocated=allocated, idle=idle, big=big, behind=behind, left=hip.hostHipLiveBytes())))
""")
    assert out["errors"] == [] and out["big"] is None
    assert out["allocated"] <= 8 * 6 * 5, "buffers given back are not used again"   # (five sizes of 64 KiB steps)
    assert 0 < out["idle"] <= 256 << 20
    assert 0 < out["behind"] <= 1 << 19 and out["left"] == 0   # the buffer still held, then nothing


def test_uploads_and_pins_leave_the_library_alone(on_host):
    """Another thread may be enqueueing on the library's stream: uploading and pinning launch nothing and never set
    it; an upload with no memory for it is refused; what they leave to do happens once, with the next forward."""
    out = on_host(r"""
e = create()
marker = ctypes.c_void_p(77)
lib.homSetStream(marker)
upload(e)
assert drv.homBertSetGemmChoice(e, 1, 10**6, 1) < 0   # (no such kernel: stays on packed weights)
quiet = [hip.hostHipLaunches(), lib.homGetStream()]
def forward():
    before = hip.hostHipLaunches()
    drv.homBertForward(e, 1)
    return hip.hostHipLaunches() - before
first, second = forward(), forward()
upload(e)
again = forward()
hip.hostHipFailAt(0)
refused = drv.homBertUpload(e, 0, 0, np.zeros(3 * H * H, np.float16).ctypes.data, 3 * H * H)
hip.hostHipFailAt(-1)
third = forward()
before = hip.hostHipLaunches()
assert drv.homBertSetGemmChoice(e, 1, 1, 1) == 0
n = 3 * H * H
assert drv.homBertUpload(e, 1, 0, np.zeros(n, np.float16).ctypes.data, n) == 0
quiet.append(hip.hostHipLaunches() - before)
left, pinned = forward(), forward()
bad = drv.homBertUpload(e, 0, -1, np.zeros(1, np.float16).ctypes.data, 1)
drv.homBertDestroy(e)
print(json.dumps(dict(quiet=quiet, stream=lib.homGetStream(), first=first, second=second, again=again, refused=refused,
                      third=third, left=left, pinned=pinned, bad=bad, live=hip.hostHipLiveBytes())))
""")
    assert out["quiet"] == [0, 77, 0] and out["stream"] == 77
    assert out["first"] - out["second"] == 6 * 3 == out["again"] - out["second"]   # 4 to pack, 2 column sums a layer
    assert out["refused"] == -3 and out["third"] == out["second"] and out["bad"] == -1
    assert out["left"] - out["pinned"] == 4 * 3 - 1   # unpacked but for the one uploaded since
    assert out["live"] == 0
