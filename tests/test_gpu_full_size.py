"""The BERT-large kernel shapes (M = 32 x 512 = 16384 rows) through the C-ABI.

The oracle is too slow for whole tensors of this size, so each operator is checked
(a) against the oracle on a sample of rows / (batch, head) pairs, which touches
every tile column and a spread of tile rows, and (b) through properties that hold
for the whole tensor whatever its size: column-sum checksums for GEMM, constant-V
and key-permutation invariance for attention, idempotence and unit statistics for
layer norm, commutativity for add.  Tolerances are the ones of test_gpu_parity.
"""
import ctypes
import importlib

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

GEMM_TOL = dict(rtol=1e-3, atol=1e-2)
LN_TOL = dict(rtol=2e-3, atol=1e-3)
ROWS = 32 * 512


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def host(t):
    torch.cuda.synchronize()
    return t.cpu().numpy()


def assert_close(got, want, rtol, atol, what=""):
    got = np.asarray(got, np.float64)
    want = np.asarray(want, np.float64)
    err = np.abs(got - want)
    bad = err > atol + rtol * np.abs(want)
    assert not bad.any(), (f"{what}: {bad.sum()} of {bad.size} outside rtol={rtol} atol={atol}; "
                           f"max abs err {err.max():.3e} at {np.unravel_index(err.argmax(), err.shape)}")


def sample_rows(g, rows, count=48):
    """First and last rows, rows either side of 256-row tile edges, and random ones."""
    fixed = [0, 1, 255, 256, 257, rows // 2 - 1, rows // 2, rows - 257, rows - 256, rows - 1]
    return np.unique(np.concatenate([fixed, g.integers(0, rows, size=count - len(fixed))]))


@pytest.mark.parametrize("tile", ["256x256_64q1_w2x4", "256x256_64x2r1_w2x4", "256x128_64x2r2_w4x2",
                                  "128x128_64x2r2_w2x4", "256x96_64x2r2_w4x1"])
@pytest.mark.parametrize("act", [0, 1])
@pytest.mark.parametrize("source", ["none", "bias", "full"])
@pytest.mark.parametrize("M,N", [(15501, 4080),  # several tiles a workgroup
                                 (301, 264)])   # edges in both directions inside a wavefront's blocks
def test_gemm_results_by_lane_exchange(gpu, rt, tile, act, source, M, N):
    """Every output of the epilogues without LDS: a block misplaced by an exchange shows as an error
    of the size of the values.  Operands of K = 64 are exact in fp32, so the bound is one rounding to fp16
    plus the activation's 3e-7."""
    kernel = f"hom_gfx950_mfma_f16_s32x32x16gemm_f16_{tile}_nn_align8_{'gelu' if act else 'linear'}"
    num = gpu.homGemmManifestFind(kernel.encode())
    assert num >= 0
    K, mr = 64, rt.MemRef.from_tensor
    g = torch.Generator(device="cuda")
    g.manual_seed(M + N)
    rnd = lambda *s: torch.randint(-8, 9, s, generator=g, device="cuda").to(torch.float16) / 16  # noqa: E731
    A, B, C = rnd(1, M, K), rnd(1, K, N), {"bias": rnd(1, 1, N), "full": rnd(1, M, N), "none": None}[source]
    D = torch.full((1, M, N), float("nan"), dtype=torch.float16, device="cuda")
    gpu.cutlassGemmF16(*mr(A).args(), False, *mr(B).args(), False, *mr(D if C is None else C).args(),
                       *mr(D).args(), act, 1.0, 0.0 if C is None else 1.0, num + 1, 1)
    torch.cuda.synchronize()
    want = A[0].float() @ B[0].float()
    if C is not None:
        want = want + C[0].float()
    if act:
        want = torch.nn.functional.gelu(want)
    err = (D[0].float() - want).abs()
    assert bool((err <= 2.0 ** -11 * want.abs() + 1e-6).all()), f"max {err.max().item()}"


# linear 256 x 256 tiles with a bias row have kernels of their own, aligned and any alignment: nothing but a partial slab,
# full slabs and a partial one, slices of K, several tiles a workgroup
@pytest.mark.parametrize("tile,step", [("256x256_64x2r1_w2x4_nn_align8", 8), ("256x256_64x2u1_w2x4_nn_align1", 1)])
@pytest.mark.parametrize("M,N,K,slices", [(301, 264, 40, 1), (301, 520, 64, 1), (515, 264, 200, 1), (301, 264, 200, 2),
                                          (15501, 4080, 72, 1)])
def test_gemm_bias_row_of_its_own(gpu, rt, tile, step, M, N, K, slices):
    num = gpu.homGemmManifestFind(f"hom_gfx950_mfma_f16_s32x32x16gemm_f16_{tile}_linear".encode())
    assert num >= 0
    mr, K = rt.MemRef.from_tensor, K + (step == 1)
    g = torch.Generator(device="cuda")
    g.manual_seed(M + N + K)
    rnd = lambda *s: torch.randint(-8, 9, s, generator=g, device="cuda").to(torch.float16) / 16  # noqa: E731
    A, B, C = rnd(1, M, K), rnd(1, K, N), rnd(1, 1, N)
    want = A[0].float() @ B[0].float() + 0.5 * C[0].float()  # (exact: multiples of 2^-8 below 2^6)
    D = torch.full((1, M, N), float("nan"), dtype=torch.float16, device="cuda")
    gpu.cutlassGemmF16(*mr(A).args(), False, *mr(B).args(), False, *mr(C).args(), *mr(D).args(), 0, 1.0, 0.5, num + 1,
                       slices)
    torch.cuda.synchronize()
    err = (D[0].float() - want).abs()
    assert bool((err <= 2.0 ** -11 * want.abs()).all()), f"max {err.max().item()}"


@pytest.mark.parametrize("N,K,act,beta", [
    (4096, 1024, 1, 0.0),   # FFN1 + GELU-erf
    (1024, 4096, 0, 1.0),   # FFN2 + residual, in place
    (3072, 1024, 0, 0.0),   # QKV projection
])
def test_gemm_bert_large_shapes(gpu, rt, oracle, N, K, act, beta):
    M = rt.MemRef.from_tensor
    g = np.random.default_rng(N + K)
    a = g.standard_normal((32, 512, K), dtype=np.float32).astype(np.float16)
    b = (g.standard_normal((1, K, N), dtype=np.float32) * 0.03).astype(np.float16)
    res = g.standard_normal((32, 512, N), dtype=np.float32).astype(np.float16)
    ta, tb = dev(a), dev(b)
    td = dev(res) if beta else torch.zeros((32, 512, N), dtype=torch.float16, device="cuda")
    gpu.cutlassGemmF16(*M(ta).args(), False, *M(tb).args(), False, *M(td).args(), *M(td).args(),
                       act, 1.0, beta, 0, 1)
    got = host(td).reshape(ROWS, N)
    rows = sample_rows(g, ROWS)
    want = oracle.gemm(a.reshape(ROWS, K)[rows], b[0], res.reshape(ROWS, N)[rows] if beta else None,
                       beta=beta, act="gelu_erf" if act else "linear")
    assert_close(got[rows], want, **GEMM_TOL, what=f"sampled rows of 16384x{N}x{K}")
    if not act:
        # checksum over every row: sum_j D[i, j] = A[i, :] . rowsum(B) (+ sum_j C[i, j]); the
        # stored values carry one fp16 rounding each (relative 2^-11, independent)
        a64 = a.reshape(ROWS, K).astype(np.float64)
        check = a64 @ b[0].astype(np.float64).sum(axis=1)
        if beta:
            check += res.reshape(ROWS, N).astype(np.float64).sum(axis=1)
        got64 = got.astype(np.float64)
        noise = 2.0 ** -11 * np.sqrt((got64 ** 2).sum(axis=1))
        assert (np.abs(got64.sum(axis=1) - check) <= 6 * noise + 1e-3).all(), "row checksum"
    assert np.isfinite(got.astype(np.float32)).all()


def run_attention(gpu, rt, qkv, lens, heads, scale):
    M = rt.MemRef.from_tensor
    bs, seq, w = qkv.shape
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    tq, tc = dev(qkv), dev(cu)
    out = torch.full((bs, seq, w // 3), 7.0, dtype=torch.float16, device="cuda")
    gpu.nvteBertAttentionF16(*M(tq).args(), *M(tc).args(), *M(out).args(), scale, heads)
    return host(out), cu


def test_attention_bert_large_shape(gpu, rt, oracle):
    bs, seq, heads = 32, 512, 16
    g = np.random.default_rng(7)
    qkv = g.standard_normal((bs, seq, 3 * heads * 64), dtype=np.float32).astype(np.float16)
    lens = g.integers(1, seq + 1, size=bs).astype(np.int32)
    lens[:4] = [512, 1, 511, 65]
    got, cu = run_attention(gpu, rt, qkv, lens, heads, 0.125)
    # oracle on a sample of sequences (all heads of each)
    for b in (0, 1, 2, 3, 17, 31):
        one_cu = np.array([0, lens[b]], np.int32)
        want = oracle.attention(qkv[b:b + 1], one_cu, heads, 0.125)
        assert_close(got[b:b + 1], want, **GEMM_TOL, what=f"attention sequence {b} (len {lens[b]})")
    for b, n in enumerate(lens):
        assert not got[b, n:].any(), "padded query rows must be zeros"

    # rows of P sum to 1: a V that is constant over the keys comes out unchanged
    v5 = qkv.reshape(bs, seq, 3, heads, 64).copy()
    const = g.standard_normal((bs, 1, heads, 64), dtype=np.float32).astype(np.float16)
    v5[:, :, 2] = const
    out_c, _ = run_attention(gpu, rt, v5.reshape(bs, seq, -1), lens, heads, 0.125)
    out_c = out_c.reshape(bs, seq, heads, 64)
    for b, n in enumerate(lens):
        assert_close(out_c[b, :n], np.broadcast_to(const[b], (n, heads, 64)), rtol=2e-3, atol=2e-3,
                     what=f"constant V, sequence {b}")

    # permuting the valid keys (K and V rows together) changes nothing but the summation order
    perm5 = qkv.reshape(bs, seq, 3, heads, 64).copy()
    for b, n in enumerate(lens):
        p = g.permutation(n)
        perm5[b, :n, 1:] = perm5[b, p, 1:]
    out_p, _ = run_attention(gpu, rt, perm5.reshape(bs, seq, -1), lens, heads, 0.125)
    assert_close(out_p, got, rtol=2e-3, atol=4e-3, what="key permutation")


def test_layernorm_bert_large_shape(gpu, rt, oracle):
    g = np.random.default_rng(11)
    x = (g.standard_normal((32, 512, 1024), dtype=np.float32) * 1.7 + 0.4).astype(np.float16)
    t = dev(x)
    gpu.nvteLayernormF16(*rt.MemRef.from_tensor(t).args(), 1e-12)
    once = host(t).reshape(ROWS, 1024)
    rows = sample_rows(g, ROWS)
    assert_close(once[rows], oracle.layernorm_f16(x.reshape(ROWS, 1024)[rows], 1e-12), **LN_TOL)
    o64 = once.astype(np.float64)
    assert np.abs(o64.mean(axis=1)).max() <= 2e-3
    assert np.abs(o64.var(axis=1) - 1.0).max() <= 5e-3
    gpu.nvteLayernormF16(*rt.MemRef.from_tensor(t).args(), 1e-12)   # idempotent up to rounding
    assert_close(host(t).reshape(ROWS, 1024), once, **LN_TOL, what="layer norm twice")


def test_elementwise_gather_cu_seqlens_bert_large_shapes(gpu, rt, oracle):
    M = rt.MemRef.from_tensor
    g = np.random.default_rng(13)
    a = g.standard_normal((32, 512, 1024), dtype=np.float32).astype(np.float16)
    b = g.standard_normal((32, 512, 1024), dtype=np.float32).astype(np.float16)
    ta, tb = dev(a), dev(b)
    ab, ba = torch.empty_like(ta), torch.empty_like(ta)
    gpu.thrustElementwiseAddF16(*M(ta).args(), *M(tb).args(), *M(ab).args())
    gpu.thrustElementwiseAddF16(*M(tb).args(), *M(ta).args(), *M(ba).args())
    assert torch.equal(ab, ba)
    rows = sample_rows(g, ROWS)
    want = oracle.elementwise("add", a.reshape(ROWS, 1024)[rows], b.reshape(ROWS, 1024)[rows])
    assert np.array_equal(host(ab).reshape(ROWS, 1024)[rows], want.astype(np.float16))

    vocab = 30522
    table = g.standard_normal((1, vocab, 1024), dtype=np.float32).astype(np.float16)
    ids = g.integers(0, vocab, size=(32, 512)).astype(np.int64)
    ids[0, :3] = [0, vocab - 1, 0]
    tt, ti = dev(table), dev(ids)
    out = torch.empty((32, 512, 1024), dtype=torch.float16, device="cuda")
    gpu.thrustGatherF16(*M(ti).args(), *M(tt).args(), *M(out).args())
    assert np.array_equal(host(out), table[0][ids])

    lens = g.integers(0, 513, size=32)
    mask = (np.arange(512)[None, :] < lens[:, None]).astype(np.int64)
    tm = dev(mask)
    cu = torch.empty(33, dtype=torch.int32, device="cuda")
    gpu.thrustCuSeqLenI64(*M(tm).args(), *M(cu).args())
    assert np.array_equal(host(cu), np.concatenate([[0], np.cumsum(lens)]).astype(np.int32))


def test_driver_measurement_helpers(gpu, rt):
    """The probes behind the figures on operand-dependent matrix-core rates run and give plausible numbers
    (their exact values are a property of the box; the relations asserted here are kept loose)."""
    drv = rt.load_driver()
    zero, rnd = drv.homMfmaCeilingProbe(0, 0), drv.homMfmaCeilingProbe(1, 0)
    assert 300 < rnd < 2600 and 300 < zero < 2600, (zero, rnd)
    assert zero >= 0.9 * rnd, (zero, rnd)
    assert 300 < drv.homMfmaCeilingProbe(1, 4) < 2600
    idx, sk = ctypes.c_int64(), ctypes.c_int32()
    gpu.homGemmSelect(ROWS, 1024, 4096, 0, ctypes.byref(idx), ctypes.byref(sk))
    t_rnd = drv.homTimeGemm(ROWS, 1024, 4096, 0, 0, idx.value + 1, sk.value, 10, 3)
    t_zero = drv.homTimeGemmZeroOperands(ROWS, 1024, 4096, 0, 0, idx.value + 1, sk.value, 10, 3)
    assert 0.03 < t_zero < 1.0 and 0.03 < t_rnd < 1.0, (t_zero, t_rnd)
    assert t_zero <= 1.1 * t_rnd, (t_zero, t_rnd)
    # a node of a replayed graph of empty kernels: a microsecond or two, never zero
    node_ms = drv.homTimeEmptyGraphNodes(88, 256, 50)
    assert 2e-4 < node_ms < 2e-2, node_ms
    assert drv.homTimeEmptyGraphNodes(0, 256, 50) < 0
