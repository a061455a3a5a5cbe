"""The sizes in packed_shapes.py reach every kernel that homPackedGemmF16 chooses from, in every kind of call."""
import ctypes
import math
import random

import pytest
from packed_shapes import FEW_ROWS, FROM_REGISTERS, MANY_ROWS, NORMALISED_MANY, TILES


def selected(lib, M, N, K, act=0, norm=0, source=0, packing=5, ahead=0):
    """("tile" | "registers", key of packed_shapes, tiles of the busiest CU > those it works on at a time)."""
    out = [ctypes.c_int32() for _ in range(3)]
    kind = lib.homPackedGemmSelect(M, N, K, act, norm, source, packing, ahead, *map(ctypes.byref, out))
    rows, cols, k = (v.value for v in out)
    if kind == 0:
        return "registers", (rows, cols, k, K <= 8 * k), False
    assert kind == 1
    return "tile", (rows, cols, k), -(-M // rows) * -(-N // cols) > 256 * TILES[rows, cols, k][1]


# the calls test_packed_gemm and test_packed_gemm_many_rows make: kind -> arguments
CALLS = {"source": dict(source=1, ahead=1), "linear": {}, "gelu": dict(act=1), "norm": dict(norm=1),
         "norm + gelu": dict(norm=1, act=1)}


def check_coverage(lib):
    tiles, several = set(), set()
    for size in MANY_ROWS:
        for call, args in CALLS.items():
            kind, key, more = selected(lib, *size, **dict(args, packing=7 if "source" in args else 5))
            if kind == "tile":
                tiles.add((key, call))
                several.add((key, more))
    assert tiles == {(t, c) for t, (norm, _) in TILES.items() for c in CALLS if norm or "norm" not in c}
    assert several == {(t, more) for t in TILES for more in (False, True)}
    norm = {selected(lib, *size, norm=1)[:2] for size in NORMALISED_MANY}
    assert norm >= {("tile", t) for t, (folds, _) in TILES.items() if folds}
    regs = set()
    for size in FEW_ROWS:
        for call in ("source", "norm", "norm + gelu"):
            for packing in (0, 7, 3, 5):
                args = dict(CALLS[call], packing=packing if call == "source" else packing & ~2)
                kind, key, _ = selected(lib, *size, **args)
                if kind == "registers":
                    regs.add((key, call, packing & 1))
    want = {(r, c, a) for r in FROM_REGISTERS for c in ("source", "norm", "norm + gelu") for a in (0, 1)
            if a or r[:2] != (64, 64)}  # (64 x 64 takes A in fragment order only)
    assert regs == want


def test_sizes_reach_every_packed_kernel(rt):
    check_coverage(rt.load_runtime())


@pytest.mark.gpu
def test_sizes_reach_every_packed_kernel_on_this_gpu(gpu):
    check_coverage(gpu)


def test_selection_knows_no_other_kernel(rt):
    """Over the sizes the entry point takes, nothing but what packed_shapes.py lists is ever selected."""
    lib, rng = rt.load_runtime(), random.Random(5)
    log = lambda lo, hi: int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))  # noqa: E731
    for _ in range(20000):
        M, N, K = log(1, 30000), max(1, log(16, 8192) // 32) * 32, max(1, log(32, 8192) // 32) * 32
        if max(M * max(K, N), K * N) >= 1 << 30:
            continue
        args = dict(rng.choice(list(CALLS.values())), packing=rng.choice([0, 1, 3, 4, 5, 7]), ahead=rng.choice([0, 1]))
        kind, key, _ = selected(lib, M, N, K, **args)
        assert key in (TILES if kind == "tile" else FROM_REGISTERS), (M, N, K, args)
        assert kind == "registers" or not args.get("norm") or TILES[key][0], (M, N, K, args)
    # (multiples of 16 columns, and what is not a problem for it)
    assert selected(lib, 5, 48, 64, packing=0) == ("registers", (16, 16, 96, True), False)
    for bad in ((0, 32, 32), (5, 24, 32), (5, 32, 33), (1 << 20, 2048, 2048)):
        assert lib.homPackedGemmSelect(*bad, 0, 0, 0, 0, 0, None, None, None) == -1
    assert lib.homPackedGemmSelect(5, 48, 32, 0, 0, 0, 5, 0, None, None, None) == -1   # D packed needs N % 32 == 0
    assert lib.homPackedGemmSelect(5, 32, 32, 1, 0, 1, 0, 0, None, None, None) == -1   # no activation with a source
