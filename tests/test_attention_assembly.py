"""The attention kernels' hand-waited LDS reads, on their compiled form: between a transposing read and the wait that
covers it no instruction may touch what it writes, a copy or a spill by the register allocator included."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "hands-on-mlir_amd", "csrc")


def registers(text):
    """{("v", 3), ("a", 7), ..} of an operand list."""
    regs = set()
    for kind, lo, hi, one in re.findall(r"\b([va])(?:\[(\d+):(\d+)\]|(\d+)\b)", text):
        regs |= {(kind, i) for i in (range(int(lo), int(hi) + 1) if lo else [int(one)])}
    return regs


def early_uses(lines):
    """(reads, violations): LDS operations come back in order, lgkmcnt(n) leaves the n newest outstanding."""
    reads, bad, pending = 0, [], []  # pending: (registers written, transposing read?) in order of issue
    for line in lines:
        text = line.split(";")[0].strip()
        if not text or text.startswith(".") and not text.endswith(":"):
            continue
        if text.endswith(":") or text.startswith(("s_cbranch", "s_branch", "s_endpgm")):
            if any(tr for _, tr in pending):  # (a wait in another block would have to be followed through branches)
                bad.append(f"outstanding at {text}")
            pending = []
            continue
        op, _, args = text.partition(" ")
        if op == "s_waitcnt":
            count = re.search(r"lgkmcnt\((\d+)\)", text)
            if count:
                pending = pending[len(pending) - int(count.group(1)):] if int(count.group(1)) < len(pending) else pending
            continue
        used = registers(args)
        if any(tr and used & dst for dst, tr in pending):
            bad.append(text)
        if op.startswith("ds_"):
            tr = op == "ds_read_b64_tr_b16"
            reads += tr
            pending.append((registers(args.split(",")[0]) if op.startswith("ds_read") else set(), tr))
    return reads, bad


def test_the_check_sees_early_uses():
    code = ["ds_read_b64_tr_b16 v[2:3], v1", "ds_read_b64_tr_b16 v[4:5], v1 offset:64", "s_waitcnt lgkmcnt(1)",
            "v_mov_b32 v9, v3", "s_waitcnt vmcnt(0) lgkmcnt(0)", "v_mov_b32 v9, v4"]
    assert early_uses(code) == (2, [])
    assert early_uses(code[:3] + ["v_mov_b32 v9, v5"]) == (2, ["v_mov_b32 v9, v5"])
    assert early_uses(code[:2] + ["scratch_store_dwordx2 off, v[2:3], s0"])[1]
    assert early_uses(code[:3] + ["v_mfma_f32_32x32x16_f16 a[0:15], v[4:7], v[8:11], a[0:15]"])[1]
    assert early_uses(code[:1] + ["s_cbranch_scc1 .LBB0_1"])[1]


@pytest.fixture(scope="module")
def assembly(tmp_path_factory):
    flags = subprocess.run(["make", "-s", "-C", CSRC, "flags"], capture_output=True, text=True, timeout=60)
    assert flags.returncode == 0, flags.stderr
    out = str(tmp_path_factory.mktemp("asm") / "attention.s")
    res = subprocess.run(flags.stdout.split() + ["--offload-device-only", "-S", os.path.join(CSRC, "attention.hip"), "-o", out],
                         capture_output=True, text=True, timeout=600)
    assert res.returncode == 0, res.stderr
    return open(out).read()


def test_no_use_of_a_transposing_read_before_its_wait(assembly):
    kernels = re.findall(r"^(_ZN3hom\S*bertAttentionKernel\S*):\s*;.*?$(.*?)^\.Lfunc_end", assembly, re.M | re.S)
    dma = 0
    for name, body in kernels:
        reads, bad = early_uses(body.splitlines())
        assert reads > 0 and not bad, (name, bad)
        dma += "buffer_load_dwordx4" in body and " lds" in body
    assert len(kernels) >= 12 and dma >= 8, (len(kernels), dma)


def test_priorities_and_stores_by_variant(assembly):
    """Priorities are raised where the chunks come by DMA at head size 64, and nowhere else; results leave in stores that
    the compiler places, not in statements of their own."""
    kernels = re.findall(r"^(_ZN3hom\S*bertAttentionKernelILi\d+ELi\d+ELi(\d+)ELb(\d)ELb(\d)E\S*):\s*;.*?$(.*?)^\.Lfunc_end",
                         assembly, re.M | re.S)
    assert len(kernels) >= 12
    for name, head, fragments, dma, body in kernels:
        assert ("s_setprio" in body) == (head == "64" and dma == "1"), name
        stores = re.findall(r"^\s+(global_store_\w+)", body, re.M)
        assert stores and "#ASMSTART\n\tglobal_store" not in body, name
        assert ("global_store_dwordx2" in stores) == (fragments == "1"), name
