"""The library's choice of a GEMM kernel, which needs no GPU: every size gets a kernel that takes it."""
import ctypes
import random
import re

import pytest


def choice(lib, select, M, N, K, act):
    idx, sk = ctypes.c_int64(-1), ctypes.c_int32(0)
    getattr(lib, select)(M, N, K, act, ctypes.byref(idx), ctypes.byref(sk))
    return idx.value, sk.value


# few tiles (the wavefronts split K), some, more 64 x 64 tiles than CUs, and vectors, dwords and odd rows
@pytest.mark.parametrize("largest", [200, 1500, 20000])
@pytest.mark.parametrize("step", [8, 2, 1])
def test_every_size_gets_a_kernel_that_takes_it(rt, largest, step):
    lib = rt.load_runtime()
    kernels = {i: (n, lib.homGemmManifestAlignment(i)) for i, n, _, _ in rt.manifest()}
    rng, seen = random.Random(largest + step), set()
    for _ in range(150):
        M, N, K = (rng.randint(1, largest), max(step, rng.randint(1, 5000) // step * step),
                   max(step, rng.randint(1, 5000) // step * step))
        for select in ("homGemmSelect", "homGemmSelectNvte"):
            for act, epilogues in ((0, ("linear",)), (1, ("gelu", "gelutanh")), (2, ("gelutanh",))):
                idx, sk = choice(lib, select, M, N, K, act)
                name, alignment = kernels[idx]
                assert name.rsplit("_", 1)[1] in epilogues, (name, M, N, K, act)
                assert alignment == 1 or (K % 8 == 0 and N % 2 == 0), (name, M, N, K)
                assert 1 <= sk <= 16
                if "k8_w1x1_" in name:  # all workgroups resident at once
                    rows, cols = map(int, re.search(r"f16_(\d+)x(\d+)_", name).groups())
                    assert -(-M // rows) * -(-N // cols) * sk <= 256, (name, sk, M, N, K)
                    seen.add(rows)
    assert largest > 1500 or seen == {16, 32}
