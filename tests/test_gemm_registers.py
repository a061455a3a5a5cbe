"""GEMM kernels from what they compile to: register use of the 64 x 64 ones, as problems of many tiles are walked by as
many workgroups as the registers leave room for, of the 256 x 256 ones for a bias row, and the cache policy of the latter's
results."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "hands-on-mlir_amd", "csrc")

# (slabs in flight, epilogue, [N, K] weights, staged by DMA, any alignment, early partial slab) -> wavefronts per SIMD
KERNELS = {(2, 0, 0, 0, 0, 0): 3, (2, 0, 1, 0, 0, 0): 3, (2, 1, 0, 0, 0, 0): 3, (2, 2, 1, 0, 0, 0): 3, (2, 0, 0, 0, 1, 0): 3,
           (2, 0, 1, 0, 1, 0): 3, (2, 1, 0, 0, 1, 0): 3, (3, 0, 0, 1, 0, 0): 4, (3, 0, 1, 1, 0, 0): 4, (2, 3, 0, 0, 0, 0): 4,
           (2, 4, 0, 0, 0, 0): 4, (2, 0, 0, 0, 0, 1): 2, (2, 0, 0, 0, 1, 1): 2, (2, 0, 1, 0, 1, 1): 3, (2, 1, 1, 0, 1, 1): 3}


def compiled(path, lines):
    """Assembly of gemm_pipe.h with these explicit instantiations."""
    flags = subprocess.run(["make", "-s", "-C", CSRC, "flags"], capture_output=True, text=True, timeout=60)
    assert flags.returncode == 0, flags.stderr
    source, out = path / "kernels.hip", path / "kernels.s"
    source.write_text("\n".join(['#include "gemm_pipe.h"', "namespace hom { namespace gemmk {", *lines, "} }"]))
    res = subprocess.run(flags.stdout.split() + ["--offload-device-only", "-S", "-I", CSRC, str(source), "-o", str(out)],
                         capture_output=True, text=True, timeout=600)
    assert res.returncode == 0, res.stderr
    return out.read_text()


@pytest.fixture(scope="module")
def registers(tmp_path_factory):
    """kernel -> registers of a wavefront (architectural and accumulation ones share the file)."""
    bools = ("false", "true")
    lines = [f"template __global__ void gemmPipeKernel<64, 64, 2, 2, {d}, {e}, {bools[nk]}, {bools[dma]}, {bools[any_]}, "
             f"{bools[early]}>("
             "const _Float16 *, const _Float16 *, int, int, int, int, int, int, int, uint32_t, uint32_t, int, GemmParams);"
             for d, e, nk, dma, any_, early in KERNELS]
    found = {}
    for name, body in re.findall(r"\.amdhsa_kernel (\S+)(.*?)\.end_amdhsa_kernel",
                                 compiled(tmp_path_factory.mktemp("asm"), lines), re.S):
        key = re.search(r"gemmPipeKernelILi64ELi64ELi2ELi2ELi(\d)ELi(\d)ELb(\d)ELb(\d)ELb(\d)ELb(\d)E", name).groups()
        found[tuple(map(int, key))] = int(re.search(r"next_free_vgpr (\d+)", body).group(1))
    return found


@pytest.mark.parametrize("kernel", KERNELS)
def test_wavefronts_per_simd(registers, kernel):
    assert 512 // (-(-registers[kernel] // 8) * 8) >= KERNELS[kernel], registers[kernel]


@pytest.mark.parametrize("epilogue,dma", [(0, "true"), (1, "true"), (0, "false")])
def test_results_stay_in_the_last_level_cache(tmp_path, epilogue, dma):
    """The next operator reads a GEMM's result from there, so no store passes it by."""
    text = compiled(tmp_path, [
        f"template __global__ void gemmPipeKernel<256, 256, 2, 4, 1, {epilogue}, false, {dma}>("
        "const _Float16 *, const _Float16 *, int, int, int, int, int, int, int, uint32_t, uint32_t, int, GemmParams);"])
    stores = re.findall(r"^\s*(?:buffer|global)_store_dwordx4 .*$", text, re.M)
    assert stores and not [s for s in stores if re.search(r"\bnt\b", s)]


@pytest.mark.parametrize("any_", ["false", "true"])
def test_bias_row_without_spills(tmp_path, any_):
    """256 x 256 linear tiles, results by lane exchanges: with the code for every source one kernel keeps some thirty
    registers in memory, the one for a bias row alone (last argument) next to none."""
    text = compiled(tmp_path, [
        f"template __global__ void gemmPipeKernel<256, 256, 2, 4, 1, 0, false, false, {any_}, false, {mode}>("
        "const _Float16 *, const _Float16 *, int, int, int, int, int, int, int, uint32_t, uint32_t, int, GemmParams);"
        for mode in (-1, 1)])
    spilled = list(map(int, re.findall(r"\.vgpr_spill_count: (\d+)", text)))
    assert spilled[1] <= 8 and spilled[1] < spilled[0], spilled
