"""The library's choice of a GEMM kernel, which needs no GPU: every size gets a kernel that takes it."""
import ctypes
import os
import random
import re
import subprocess

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


def test_shipped_table_answers_first(rt):
    lib = rt.load_runtime()
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    with open(os.path.join(root, "hands-on-mlir_amd", "csrc", "gemm_tuned_table.inc")) as f:
        rows = re.findall(r'\{(\d+), (\d+), (\d+), (\d), "(\w+)", (\d+), "(\w+)", (\d+), (\d)\}', f.read())
    assert len(rows) == 51
    for M, N, K, act, *kernels, prefers in rows:
        size = tuple(map(int, (M, N, K, act)))
        for select, kernel, split in (("homGemmSelect", *kernels[:2]), ("homGemmSelectNvte", *kernels[2:])):
            if select == "homGemmSelectNvte" and act == "1":
                continue  # (GELU is the tanh form there)
            idx, sk = ctypes.c_int64(-1), ctypes.c_int32(0)
            assert getattr(lib, select)(*size, ctypes.byref(idx), ctypes.byref(sk)) == 1, size
            assert (lib.homGemmManifestName(idx.value).decode(), sk.value) == (kernel, int(split)), size
        assert lib.homGemmPrefersNvte(*size) == int(prefers), size


# Few tiles: the wavefronts split K where there are slabs of 64 for most of them, on rows off 16 bytes earlier
@pytest.mark.parametrize("M,N", [(6, 72), (37, 952), (141, 168), (10, 320)])
@pytest.mark.parametrize("select", ["homGemmSelect", "homGemmSelectNvte"])
def test_few_slabs_stay_with_the_pipelines(rt, M, N, select):
    lib = rt.load_runtime()
    split = lambda n, K: "k8_w1x1_" in lib.homGemmManifestName(choice(lib, select, M, n, K, 0)[0]).decode()  # noqa: E731
    assert [split(N, K) for K in (8, 80, 136, 264, 384, 512, 696)] == [False] * 5 + [True] * 2
    assert [split(N + 2, K) for K in (80, 128, 192, 384, 512)] == [False] * 2 + [M > 16] + [True] * 2
    for source in (1, 2):  # which costs the pipelines more where the rows of C and D are off 16 bytes and not a few
        idx, sk = ctypes.c_int64(-1), ctypes.c_int32(0)
        lib.homGemmSelectWithSource(M, N + 2, 80, 0, int(select.endswith("Nvte")), source, ctypes.byref(idx), ctypes.byref(sk))
        assert ("k8_w1x1_" in lib.homGemmManifestName(idx.value).decode()) == (M > 16)
    assert split(N + 1, 63) and split(N + 2, 93)  # (any alignment)
    assert not split(N, 60) and not split(N, 85) and split(N, 133)


# Problems of more 64 x 64 tiles than CUs, no source or a bias row, all seven tiles timed on an MI355X: those within 5 % of
# the fastest (sizes, activation, tiles)
@pytest.mark.parametrize("M,N,K,act,tiles", [
    (15866, 3288, 328, 1, "128x256"), (15440, 4040, 336, 1, "128x256"), (13520, 3656, 176, 2, "128x256 256x128"),
    (13802, 3536, 56, 2, "128x256 256x128"), (9165, 424, 1176, 0, "128x256"), (10289, 912, 1256, 1, "256x256"),
    (16873, 440, 1016, 0, "256x256"), (3037, 2920, 880, 2, "256x256"), (5339, 296, 712, 0, "64x128"),
    (8930, 1728, 96, 0, "128x256 256x128"), (6580, 4168, 344, 0, "128x256 256x128"), (8534, 272, 32, 0, "64x64 64x128"),
    (588, 4184, 16, 0, "64x64 64x128"), (3396, 1608, 176, 1, "128x256"),
    # rows off 16 bytes
    (19540, 420, 112, 1, "64x64"), (2673, 3938, 8, 2, "64x64"), (17143, 86, 80, 0, "64x64"), (2356, 2588, 64, 2, "64x64")])
def test_large_problems_take_a_fast_tile(rt, M, N, K, act, tiles):
    lib = rt.load_runtime()
    idx, sk = choice(lib, "homGemmSelect", M, N, K, act)
    name = lib.homGemmManifestName(idx).decode()
    assert sk == 1 and re.search(r"f16_(\d+x\d+)_64x2r", name).group(1) in tiles.split(), name


# The same with a full matrix as source, whose price changes the fastest tile (the one named first is 9 % slower at least)
@pytest.mark.parametrize("M,N,K,act,without,tile", [
    (5945, 2312, 1408, 0, "256x256", "128x256"), (5475, 1576, 408, 0, "256x256", "64x128"), (3925, 2576, 608, 1, "256x256", "128x128"),
    (9658, 1728, 80, 0, "128x256", "64x128"), (8967, 1208, 392, 1, "128x256", "128x128")])
@pytest.mark.parametrize("nk", [0, 1])
def test_a_source_is_priced(rt, M, N, K, act, without, tile, nk):
    lib = rt.load_runtime()
    idx, sk = ctypes.c_int64(-1), ctypes.c_int32(0)
    for source, expected in ((0, without), (1, without), (2, tile)):
        assert lib.homGemmSelectWithSource(M, N, K, act, nk, source, ctypes.byref(idx), ctypes.byref(sk)) == 0
        assert f"f16_{expected}_64x2r" in lib.homGemmManifestName(idx.value).decode()
        if not source:
            assert (idx.value, sk.value) == choice(lib, "homGemmSelectNvte" if nk else "homGemmSelect", M, N, K, act)


# The layer-norm pair's tiles where all that fit were timed on an MI355X and one is 8 % faster at least than the others:
# (second GEMM, source: 0 none, 1 a bias row, 2 a full matrix; sizes, the fastest)
PAIR_TILES = [(0, 0, 5535, 2408, 2960, 256), (0, 0, 16384, 4096, 1024, 256), (0, 0, 5189, 1968, 728, 256),
              (0, 0, 9572, 3432, 24, 128), (0, 0, 1772, 3336, 240, 128), (0, 0, 306, 2256, 440, 64),
              (0, 1, 6000, 4000, 2000, 256), (0, 1, 16332, 2152, 360, 256), (0, 1, 13371, 1072, 1392, 128),
              (0, 1, 4400, 4096, 512, 128), (0, 1, 14553, 312, 344, 64), (0, 1, 350, 2696, 568, 64),
              (0, 2, 5535, 2408, 2960, 256), (0, 2, 16124, 3256, 1624, 256), (0, 2, 2500, 3072, 1024, 128),
              (0, 2, 5713, 3072, 1088, 128), (0, 2, 3368, 96, 192, 64), (1, 0, 4096, 4096, 1024, 256),
              (1, 0, 8015, 3880, 136, 256), (1, 0, 4224, 4096, 256, 128), (1, 0, 8192, 768, 768, 128),
              (1, 0, 1890, 776, 64, 64), (1, 1, 12925, 3200, 544, 256), (1, 1, 3796, 2400, 968, 256),
              (1, 1, 8400, 2048, 1024, 128), (1, 1, 2500, 3072, 1024, 128), (1, 1, 2534, 1712, 584, 64),
              (1, 2, 4924, 1864, 3176, 256), (1, 2, 5189, 1968, 728, 256), (1, 2, 6755, 2632, 328, 128),
              (1, 2, 4224, 4096, 256, 128), (1, 2, 254, 2064, 176, 64)]


def test_layernorm_pair_takes_the_fastest_tile(tmp_path):
    csrc = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "hands-on-mlir_amd", "csrc")
    source, program = tmp_path / "tiles.cpp", tmp_path / "tiles"
    calls = "".join(f'printf("%d\\n", hom::pairTileEdge({M}, {N}, {K}, {second}, hom::PairSource({form}), 256));'
                    for second, form, M, N, K, _ in PAIR_TILES)
    source.write_text(f'#include "pair_tile.h"\n#include <stdio.h>\nint main() {{ {calls} }}\n')
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", csrc, str(source), "-o", str(program)], check=True, timeout=60)
    edges = subprocess.run([str(program)], capture_output=True, text=True, check=True, timeout=10).stdout.split()
    assert list(map(int, edges)) == [case[-1] for case in PAIR_TILES]
