"""Sizes off the vector width, broadcast forms and edges of the dispatch rules, against numpy and the oracle."""
import ctypes

import numpy as np
import pytest
import torch
from packed_shapes import FEW_ROWS, MANY_ROWS, NORMALISED_FEW, NORMALISED_MANY

pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def host(t):
    torch.cuda.synchronize()
    return t.cpu().numpy()


# A's shape, B's shape: same, bias row, row per batch, value per row, repeating values, all the same, a pattern
# only the generic walk takes; rows of whole vectors and not, totals with and without a remainder, streaming size
@pytest.mark.parametrize("a,b", [
    ((3, 5, 16), (3, 5, 16)), ((3, 5, 7), (3, 5, 7)), ((4, 6, 16), (1, 1, 16)), ((4, 6, 13), (1, 1, 13)),
    ((4, 6, 16), (1, 6, 16)), ((4, 6, 24), (4, 1, 24)), ((4, 6, 9), (4, 1, 9)), ((4, 6, 16), (4, 6, 1)),
    ((4, 6, 11), (4, 6, 1)), ((4, 6, 8), (1, 6, 1)), ((4, 6, 3), (1, 6, 1)), ((4, 6, 5), (4, 1, 1)),
    ((2, 3, 4, 8), (2, 1, 4, 1)), ((2, 3, 4, 8), (1, 3, 1, 8)), ((4, 6, 5), (1, 1, 1)), ((1, 1, 1), (1, 1, 1)),
    ((9, 1001, 1023), (9, 1001, 1)), ((9, 1000, 1024), (9, 1, 1024))])
@pytest.mark.parametrize("sfx,dtype", [("F16", np.float16), ("F32", np.float32)])
def test_elementwise_broadcast_forms(gpu, rt, a, b, sfx, dtype):
    g = np.random.default_rng(len(a) + sum(a))
    x, y = g.standard_normal(a).astype(dtype), g.standard_normal(b).astype(dtype)
    M = rt.MemRef.from_tensor
    for op, want in (("Mul", x * y), ("Sub", x - y)):
        tx, ty, out = dev(x), dev(y), torch.zeros(a, dtype=torch.from_numpy(x).dtype, device="cuda")
        getattr(gpu, f"thrustElementwise{op}{sfx}")(*M(tx).args(), *M(ty).args(), *M(out).args())
        np.testing.assert_array_equal(host(out), want)
        getattr(gpu, f"thrustElementwise{op}{sfx}")(*M(tx).args(), *M(ty).args(), *M(tx).args())  # in place
        np.testing.assert_array_equal(host(tx), want)


@pytest.mark.parametrize("bs,seq", [(1, 1), (1, 64), (3, 65), (17, 511), (64, 513), (257, 33), (600, 5)])
def test_cu_seqlens_many_rows(gpu, rt, bs, seq):
    mask = (np.random.default_rng(bs).random((bs, seq)) < 0.7)
    want = np.concatenate([[0], np.cumsum(mask.sum(1))]).astype(np.int32)
    M = rt.MemRef.from_tensor
    for sfx, dt in (("I64", np.int64), ("I32", np.int32)):
        t, out = dev(mask.astype(dt)), torch.zeros(bs + 1, dtype=torch.int32, device="cuda")
        getattr(gpu, "thrustCuSeqLen" + sfx)(*M(t).args(), *M(out).args())
        np.testing.assert_array_equal(host(out), want)


@pytest.mark.parametrize("H", [1, 7, 8, 9, 129, 768, 1001])
@pytest.mark.parametrize("sfx,dtype", [("F16", np.float16), ("F32", np.float32)])
def test_gather_row_lengths(gpu, rt, H, sfx, dtype):
    g = np.random.default_rng(H)
    table, ids = g.standard_normal((1, 50, H)).astype(dtype), g.integers(0, 50, (3, 11)).astype(np.int64)
    ids[0, 0], ids[2, 10] = 49, 0
    t, i, out = dev(table), dev(ids), torch.zeros((3, 11, H), dtype=torch.from_numpy(table).dtype, device="cuda")
    M = rt.MemRef.from_tensor
    getattr(gpu, "thrustGather" + sfx)(*M(i).args(), *M(t).args(), *M(out).args())
    np.testing.assert_array_equal(host(out), table[0][ids])


# row lengths at the edges of the kernel variants (fp16: 1, 2, 4 vectors per lane of a wavefront, 2, 4, 8 of a workgroup)
@pytest.mark.parametrize("H", [3, 8, 9, 511, 513, 1025, 2047, 2056, 4097, 8191, 16391, 16400])
def test_layernorm_row_lengths(gpu, rt, oracle, H):
    g = np.random.default_rng(H)
    rows = 5
    x, r = (g.standard_normal((rows, H)).astype(np.float16) for _ in range(2))
    ga, be = (1 + 0.1 * g.standard_normal(H)).astype(np.float16), g.standard_normal(H).astype(np.float16)
    M = rt.MemRef.from_tensor
    tx, tr, tg, tb, out = dev(x), dev(r), dev(ga), dev(be), torch.zeros((rows, H), dtype=torch.float16, device="cuda")
    gpu.homAddLayernormF16(*M(tx).args(), *M(tr).args(), *M(tg).args(), *M(tb).args(), *M(out).args(), 1e-12)
    want = oracle.layernorm_f16(x, 1e-12, res=r, gamma=ga, beta=be)
    np.testing.assert_allclose(host(out).astype(np.float64), want, rtol=2e-3, atol=2e-3)
    gpu.nvteLayernormF16(*M(tx).args(), 1e-12)
    np.testing.assert_allclose(host(tx).astype(np.float64), oracle.layernorm_f16(x, 1e-12), rtol=2e-3, atol=1e-3)
    y = torch.from_numpy(g.standard_normal((rows, H)).astype(np.float32)).cuda()
    want32 = torch.nn.functional.layer_norm(y.cpu().double(), (H,), eps=1e-6).numpy()
    gpu.nvteLayernormF32(*M(y).args(), 1e-6)
    np.testing.assert_allclose(host(y), want32, rtol=1e-4, atol=1e-5)


# one, two and four vectors per lane, partial last vectors, the step-by-step form (H off 8, H > 2048), row counts
# around a wavefront's four rows and a workgroup's 64, more sequences than one pass of the length scan
@pytest.mark.parametrize("b,s,H", [(1, 1, 8), (1, 3, 512), (5, 13, 520), (8, 128, 768), (2, 33, 1032), (3, 7, 2048),
                                   (2, 5, 2056), (2, 5, 100), (300, 3, 64)])
@pytest.mark.parametrize("pinned", [False, True])
def test_embed_equals_its_steps(gpu, rt, b, s, H, pinned):
    g = np.random.default_rng(b + s + H)
    V = 97
    word, pos = g.standard_normal((1, V, H)).astype(np.float16), g.standard_normal((1, s, H)).astype(np.float16)
    ids, mask = g.integers(0, V, (b, s)), (g.random((b, s)) < 0.8).astype(np.int64)
    ids.flat[0], ids.flat[-1] = -3, V + 5  # clamped to the table
    tw, tp = dev(word), dev(pos)
    ti, tm = (torch.from_numpy(a).pin_memory() if pinned else dev(a) for a in (ids, mask))
    M = rt.MemRef.from_tensor
    new = lambda *shape, dt=torch.float16: torch.zeros(shape, dtype=dt, device="cuda")  # noqa: E731
    out, cu = new(b, s, H), new(b + 1, dt=torch.int32)
    gpu.homEmbedF16(*M(ti).args(), *M(tm).args(), *M(tw).args(), *M(tp).args(), *M(out).args(), *M(cu).args(), 1e-12, 0)
    rows, want, wantCu = new(b, s, H), new(b, s, H), new(b + 1, dt=torch.int32)
    gpu.thrustCuSeqLenI64(*M(dev(mask)).args(), *M(wantCu).args())
    gpu.thrustGatherF16(*M(dev(ids)).args(), *M(tw).args(), *M(rows).args())
    gpu.thrustElementwiseAddF16(*M(rows).args(), *M(tp).args(), *M(want).args())
    gpu.nvteLayernormF16(*M(want).args(), 1e-12)
    np.testing.assert_array_equal(host(cu), host(wantCu))
    np.testing.assert_array_equal(host(out), host(want))


def test_results_kept_by_the_caller_stay_apart(synth):
    import importlib
    bert = importlib.import_module("hands-on-mlir_amd.bert")
    m = synth.bert_encoder(layers=1, hidden=128, heads=2, ffn=256, bs=2, seq=17, vocab=50, config=4)
    d = m["dims"]
    enc = bert.BertEncoder(d["layers"], d["hidden"], d["heads"], d["ffn"], d["bs"], d["seq"], d["vocab"])
    enc.load(m)
    enc.set_inputs(ids=m["ids"], mask=m["mask"])
    enc.capture()
    kept = []
    for k in range(6):
        enc.set_inputs(ids=(m["ids"] + k) % d["vocab"])
        enc.replay()
        kept.append(enc.output())
    copies = [a.copy() for a in kept]
    del kept[1], kept[3]  # these buffers may serve later results
    enc.set_inputs(ids=m["ids"])
    enc.replay()
    again = enc.output()
    np.testing.assert_array_equal(again, copies[0])
    for a, c in zip(kept, [copies[0], copies[2], copies[3], copies[5]]):
        np.testing.assert_array_equal(a, c)
    enc.close()
    np.testing.assert_array_equal(again, copies[0])  # outlives the encoder


# the any-alignment GEMM tiles: K and N around whole slabs, vectors and tiles, remainders that a shifted last vector
# serves, split-K whose last slice is all remainder, and operands that start at odd elements
@pytest.mark.parametrize("tile", ["64x64_64x2u2_w2x2", "128x128_64x2u2_w2x4", "256x256_64x2u1_w2x4"])
@pytest.mark.parametrize("M,N,K", [(5, 9, 8), (64, 65, 9), (70, 127, 63), (130, 71, 64), (65, 1001, 65), (33, 64, 127),
                                   (257, 259, 128), (100, 513, 129), (3, 8, 200), (260, 77, 321)])
def test_gemm_any_alignment(gpu, rt, oracle, tile, M, N, K):
    g = np.random.default_rng(M + N + K)
    num = {n.rsplit("_", 1)[1]: i + 1 for i, n, _, _ in rt.manifest() if f"_{tile}_" in n}
    A, B = g.standard_normal((1, M, K)).astype(np.float16), (g.standard_normal((1, K, N)) * 0.1).astype(np.float16)
    R, bias = g.standard_normal((1, M, N)).astype(np.float16), g.standard_normal((1, 1, N)).astype(np.float16)
    Mr = rt.MemRef.from_tensor

    def odd(a):  # on the device, one element off any alignment
        t = torch.zeros(a.size + 1, dtype=torch.float16, device="cuda")[1:].view(a.shape)
        t.copy_(torch.from_numpy(a))
        return t

    for place in (dev, odd):
        ta, tb, tr, tbias = place(A), place(B), place(R), place(bias)
        for sk in (1, 2, 5):
            td = place(np.zeros((1, M, N), np.float16))
            gpu.cutlassGemmF16(*Mr(ta).args(), False, *Mr(tb).args(), False, *Mr(tr).args(), *Mr(td).args(), 0, 1.0,
                               0.5, num["linear"], sk)
            want = oracle.gemm(A[0], B[0], R[0], beta=0.5)
            np.testing.assert_allclose(host(td)[0].astype(np.float64), want, rtol=1e-3, atol=1e-2)
            gpu.cutlassGemmF16(*Mr(ta).args(), False, *Mr(tb).args(), False, *Mr(tbias).args(), *Mr(td).args(), 0, 1.0,
                               1.0, num["gelu"], sk)
            want = oracle.gemm(A[0], B[0], bias[0], beta=1.0, act="gelu_erf")
            np.testing.assert_allclose(host(td)[0].astype(np.float64), want, rtol=1e-3, atol=1e-2)
    # [N, K] weights, the library's own choice
    Bt = np.ascontiguousarray(B[0].T)[None]
    tb, td = odd(Bt), odd(np.zeros((1, M, N), np.float16))
    gpu.nvteGemmF16(*Mr(odd(A)).args(), False, *Mr(tb).args(), True, *Mr(td).args(), *Mr(td).args(), 0, 1.0, 0.0, 0, 0)
    np.testing.assert_allclose(host(td)[0].astype(np.float64), oracle.gemm(A[0], B[0]), rtol=1e-3, atol=1e-2)


# 64 x 64 tiles with a partial slab: requested ahead of the full ones (up to two workgroups per CU), or behind them
@pytest.mark.parametrize("tile,step", [("64x64_64x2r2_w2x2_nn_align8", 8), ("64x64_64x2u2_w2x2_nn_align1", 1)])
@pytest.mark.parametrize("tilesM,tilesN", [(2, 3), (16, 32), (19, 27), (40, 39)])
@pytest.mark.parametrize("K", [8, 72, 120, 392])
def test_gemm_partial_slab_early_and_late(gpu, rt, monkeypatch, tile, step, tilesM, tilesN, K):
    M, N, K = tilesM * 64 - 5, tilesN * 64 - step, K + (step == 1)
    num, name = next((i + 1, n) for i, n, _, _ in rt.manifest() if f"_{tile}_linear" in n)
    g = torch.Generator("cuda").manual_seed(M + K)
    A = torch.randn(1, M, K, device="cuda", generator=g).half()
    B = (torch.randn(1, K, N, device="cuda", generator=g) * 0.1).half()
    want = (A[0].double() @ B[0].double()).cpu().numpy()
    Mr, D, Bt = rt.MemRef.from_tensor, torch.zeros(1, M, N, dtype=torch.float16, device="cuda"), B[0].t().contiguous()[None]
    for sk in (1, 2):
        gpu.cutlassGemmF16(*Mr(A).args(), False, *Mr(B).args(), False, *Mr(D).args(), *Mr(D).args(), 0, 1.0, 0.0, num, sk)
        # (half a unit of the fp16 result, and fp32 sums of up to 393 products of about 0.1)
        np.testing.assert_allclose(host(D)[0].astype(np.float64), want, rtol=2**-10, atol=1e-4)
        D.zero_()
        monkeypatch.setenv("HOM_NVTE_GEMM_KERNEL", f"{name},{sk}")
        gpu.nvteGemmF16(*Mr(A).args(), False, *Mr(Bt).args(), True, *Mr(D).args(), *Mr(D).args(), 0, 1.0, 0.0, 0, 0)
        np.testing.assert_allclose(host(D)[0].astype(np.float64), want, rtol=2**-10, atol=1e-4)


# the kernels whose wavefronts split K: tiles and slabs of 64 and, rows at odd elements, of 63; remainders of a vector,
# fewer slabs than wavefronts and more than two rounds of them, slices across workgroups with a short last one.  What
# lies around the operands is NaN: nothing read from there may reach a result, and nothing may be written there.
@pytest.mark.parametrize("tile", ["16x64_64x2r2k8_w1x1_nn_align1", "32x64_64x2r2k8_w1x1_nn_align1"])
@pytest.mark.parametrize("M,N,K", [(1, 8, 8), (16, 64, 64), (17, 63, 63), (33, 65, 126), (5, 127, 127), (40, 130, 1032),
                                   (31, 66, 1150), (64, 126, 1009), (15, 1001, 777), (70, 72, 2002)])
def test_gemm_waves_split_k(gpu, rt, oracle, monkeypatch, tile, M, N, K):
    g = np.random.default_rng(M + N + K)
    names = {n.rsplit("_", 1)[1]: (i + 1, n) for i, n, _, _ in rt.manifest() if f"_{tile}_" in n}
    A, B = g.standard_normal((1, M, K)).astype(np.float16), (g.standard_normal((1, K, N)) * 0.1).astype(np.float16)
    R, bias = g.standard_normal((1, M, N)).astype(np.float16), g.standard_normal((1, 1, N)).astype(np.float16)
    Bt = np.ascontiguousarray(B[0].T)[None]
    Mr = rt.MemRef.from_tensor
    full, erf, plain = (oracle.gemm(A[0], B[0], R[0], beta=0.5),
                        oracle.gemm(A[0], B[0], bias[0], beta=1.0, act="gelu_erf"), oracle.gemm(A[0], B[0]))

    def place(a, off):  # between NaN, `off` elements behind a 256-byte boundary
        t = torch.full((a.size + 256,), float("nan"), dtype=torch.float16, device="cuda")
        v = t[128 + off:128 + off + a.size].view(a.shape)
        v.copy_(torch.from_numpy(a))
        return t, v

    def check(t, v, want):
        np.testing.assert_allclose(host(v)[0].astype(np.float64), want, rtol=1e-3, atol=1e-2)
        assert int(torch.isnan(t).sum()) == 256

    for off in (0, 1, 2):
        (_, ta), (_, tb), (_, tr), (_, tbias), (_, tbt) = (place(x, off) for x in (A, B, R, bias, Bt))
        for sk in (1, 2, 5):
            t, td = place(np.zeros((1, M, N), np.float16), off)
            gpu.cutlassGemmF16(*Mr(ta).args(), False, *Mr(tb).args(), False, *Mr(tr).args(), *Mr(td).args(), 0, 1.0,
                               0.5, names["linear"][0], sk)
            check(t, td, full)
            gpu.cutlassGemmF16(*Mr(ta).args(), False, *Mr(tb).args(), False, *Mr(tbias).args(), *Mr(td).args(), 0, 1.0,
                               1.0, names["gelu"][0], sk)
            check(t, td, erf)
            monkeypatch.setenv("HOM_NVTE_GEMM_KERNEL", f"{names['linear'][1]},{sk}")
            gpu.nvteGemmF16(*Mr(ta).args(), False, *Mr(tbt).args(), True, *Mr(td).args(), *Mr(td).args(), 0, 1.0, 0.0,
                            0, 0)
            check(t, td, plain)


# their slices added by the second kernel, with the in-kernel form off and where the caller brings the workspace: the sums
# of the in-kernel form bit for bit; tiles of 64 and of 63 columns, ragged rows and columns, a short last slice
@pytest.mark.parametrize("tile", ["16x64_64x2r2k8_w1x1_nn_align1", "32x64_64x2r2k8_w1x1_nn_align1"])
@pytest.mark.parametrize("M,N,K", [(40, 130, 1032), (33, 1001, 777), (17, 63, 2002), (70, 72, 2002), (5, 127, 1150)])
def test_gemm_waves_split_k_second_kernel(gpu, rt, oracle, monkeypatch, tile, M, N, K):
    g = np.random.default_rng(M + N + K)
    names = {n.rsplit("_", 1)[1]: (i + 1, n) for i, n, _, _ in rt.manifest() if f"_{tile}_" in n}
    A, B = g.standard_normal((1, M, K)).astype(np.float16), (g.standard_normal((1, K, N)) * 0.1).astype(np.float16)
    R = g.standard_normal((1, M, N)).astype(np.float16)
    Mr, ta, tb, tr, tbt = rt.MemRef.from_tensor, dev(A), dev(B), dev(R), dev(np.ascontiguousarray(B[0].T)[None])
    t = torch.full((M * N + 256,), float("nan"), dtype=torch.float16, device="cuda")
    td = t[128:128 + M * N].view(1, M, N)

    def result(fn, name, sk):
        td.zero_()
        if fn == "nvte":
            monkeypatch.setenv("HOM_NVTE_GEMM_KERNEL", f"{names[name][1]},{sk}")
            gpu.nvteGemmF16(*Mr(ta).args(), False, *Mr(tbt).args(), True, *Mr(td).args(), *Mr(td).args(), 0, 1.0, 0.0, 0, 0)
        else:
            getattr(gpu, fn)(*Mr(ta).args(), False, *Mr(tb).args(), False, *Mr(tr).args(), *Mr(td).args(), 0, 1.0, 0.5,
                             names[name][0], sk)
        out = host(td).copy()
        assert int(torch.isnan(t).sum()) == 256
        return out

    for sk in (2, 5):
        calls = [("cutlassGemmF16", "linear", sk), ("cutlassGemmF16", "gelu", sk), ("nvte", "linear", sk)]
        launches = gpu.homSplitKInKernelLaunches()
        in_kernel = [result(*c) for c in calls]
        assert gpu.homSplitKInKernelLaunches() == launches + 3
        np.testing.assert_allclose(in_kernel[0][0].astype(np.float64), oracle.gemm(A[0], B[0], R[0], beta=0.5), rtol=1e-3,
                                   atol=1e-2)
        try:
            gpu.homSetSplitKInKernel(0)
            for c, want in zip(calls, in_kernel):
                np.testing.assert_array_equal(result(*c), want)
        finally:
            gpu.homSetSplitKInKernel(3)
        assert gpu.homSplitKInKernelLaunches() == launches + 3
        for c, want in zip(calls[:2], in_kernel):
            np.testing.assert_array_equal(result("homGemmF16NoAlloc", *c[1:]), want)


# both halves of the layer-norm pair on each of their tiles (64, 128 and 256 on a side, ragged rows, columns and K),
# without a source, with a bias row (column sums and row sums by the general epilogue) and with a full matrix
@pytest.mark.parametrize("M,N,K", [(70, 136, 72), (1100, 2056, 200), (2500, 3080, 712), (4100, 2568, 136),
                                   (4090, 4096, 520)])
@pytest.mark.parametrize("source", ["none", "bias", "full"])
def test_layernorm_pair_tiles_and_sources(gpu, rt, M, N, K, source):
    g = torch.Generator(device="cuda").manual_seed(M)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    A, B = rand(1, M, K).half(), (rand(1, K, N) * 0.1).half()
    var, mean = (1 + 0.2 * rand(1, M, 1)).half(), (0.5 * rand(1, M, 1)).half()
    D = torch.zeros(1, M, N, dtype=torch.float16, device="cuda")
    C = {"none": D, "bias": rand(1, 1, N).half(), "full": rand(1, M, N).half()}[source]
    beta = 0.0 if source == "none" else 0.75
    add = 0.0 if source == "none" else beta * C[0].double()
    Mr = rt.MemRef.from_tensor
    gpu.cutlassLayernormGemmF16(*Mr(A).args(), *Mr(B).args(), *Mr(C).args(), *Mr(D).args(), *Mr(var).args(),
                                *Mr(mean).args(), 1.5, beta, 0)
    want = 1.5 * ((A[0].double() * var[0].double() + mean[0].double()) @ B[0].double()) + add
    # half a unit of the fp16 result; fp32 sums of K products and of K column values, a few units of their sizes
    np.testing.assert_allclose(host(D)[0].astype(np.float64), want.cpu().numpy(), rtol=2**-10, atol=2e-3)
    v, m = torch.zeros_like(var), torch.zeros_like(mean)
    D.zero_()
    gpu.cutlassGemmWithVarMeanF16(*Mr(A).args(), *Mr(B).args(), *Mr(C).args(), *Mr(D).args(), *Mr(v).args(),
                                  *Mr(m).args(), 1.5, beta, 0, 1e-6)
    want = 1.5 * (A[0].double() @ B[0].double()) + add
    np.testing.assert_allclose(host(D)[0].astype(np.float64), want.cpu().numpy(), rtol=2**-10, atol=2e-3)
    x = D[0].double()  # the statistics are those of the stored values
    rstd = 1 / torch.sqrt(x.var(1, unbiased=False) + 1e-6)
    np.testing.assert_allclose(host(v)[0, :, 0].astype(np.float64), rstd.cpu().numpy(), rtol=2**-10)
    np.testing.assert_allclose(host(m)[0, :, 0].astype(np.float64), (-x.mean(1) * rstd).cpu().numpy(), rtol=2**-10,
                               atol=1e-5)


# a first call inside a capture: a split across workgroups would need memory that cannot be allocated there
def test_gemm_waves_split_k_first_call_captured(gpu, rt, oracle):
    M, N, K = 33, 1001, 3001
    idx, sk = ctypes.c_int64(), ctypes.c_int32()
    gpu.homGemmSelect(M, N, K, 0, ctypes.byref(idx), ctypes.byref(sk))
    assert "k8_w1x1_" in gpu.homGemmManifestName(idx.value).decode() and sk.value > 1
    g = np.random.default_rng(3)
    A, B = g.standard_normal((1, M, K)).astype(np.float16), (g.standard_normal((1, K, N)) * 0.1).astype(np.float16)
    Mr = rt.MemRef.from_tensor
    ta, tb, td = dev(A), dev(B), torch.zeros((1, M, N), dtype=torch.float16, device="cuda")
    calls = [Mr(ta), Mr(tb), Mr(td)]
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    try:
        gpu.homSetStream(ctypes.c_void_p(stream.cuda_stream))
        with torch.cuda.graph(graph, stream=stream):
            gpu.cutlassGemmF16(*calls[0].args(), False, *calls[1].args(), False, *calls[2].args(), *calls[2].args(), 0,
                               1.0, 0.0, 0, 1)
    finally:
        gpu.homSetStream(None)
    want = oracle.gemm(A[0], B[0])
    for _ in range(3):
        td.zero_()
        graph.replay()
        np.testing.assert_allclose(host(td)[0].astype(np.float64), want, rtol=1e-3, atol=1e-2)


# a first call inside a capture on a stream that takes over another one's memory: the split, and the bits, of an eager call
def test_gemm_waves_split_k_captured_on_handed_on_memory(gpu, rt):
    M, N, K = 33, 1001, 3001
    g = torch.Generator("cuda").manual_seed(5)
    ta, tb = torch.randn(1, M, K, device="cuda", generator=g).half(), torch.randn(1, K, N, device="cuda", generator=g).half()
    eager, td = (torch.zeros((1, M, N), dtype=torch.float16, device="cuda") for _ in range(2))
    Mr = rt.MemRef.from_tensor

    def call(out):
        gpu.cutlassGemmF16(*Mr(ta).args(), False, *Mr(tb).args(), False, *Mr(out).args(), *Mr(out).args(), 0, 1.0, 0.0, 0, 1)

    first, second, graph = torch.cuda.Stream(), torch.cuda.Stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    try:
        gpu.homSetStream(ctypes.c_void_p(first.cuda_stream))
        call(eager)
        torch.cuda.synchronize()
        gpu.homReleaseStreamScratch(ctypes.c_void_p(first.cuda_stream))
        gpu.homSetStream(ctypes.c_void_p(second.cuda_stream))
        with torch.cuda.graph(graph, stream=second):
            call(td)
    finally:
        gpu.homSetStream(None)
    for _ in range(3):
        td.zero_()
        graph.replay()
        np.testing.assert_array_equal(host(td), host(eager))
    del graph
    gpu.homReleaseStreamScratch(ctypes.c_void_p(second.cuda_stream))


def fragment_order(a):
    """[rows, cols] -> blocks of 16 rows x 32 columns as the packed GEMM takes them (rows padded to 16)."""
    rows, cols = a.shape
    p = np.zeros((-(-rows // 16) * 16, cols), a.dtype)
    p[:rows] = a
    return np.ascontiguousarray(p.reshape(-1, 16, cols // 32, 4, 8).transpose(0, 2, 3, 1, 4)).reshape(-1)


# every kernel for few rows (test_packed_selection.py), both orders of every operand
@pytest.mark.parametrize("M,N,K", FEW_ROWS)
@pytest.mark.parametrize("packing", [0, 7, 3, 5])
def test_packed_gemm(gpu, rt, oracle, M, N, K, packing):
    g = np.random.default_rng(M + N + K + packing)
    A = (g.standard_normal((M, K)) + 0.3).astype(np.float16)
    B, C = (g.standard_normal((K, N)) * 0.03).astype(np.float16), g.standard_normal((M, N)).astype(np.float16)
    stats = np.stack([0.5 + g.random(M), g.standard_normal(M)], 1).astype(np.float32)
    Mr, R = rt.MemRef, -(-M // 16) * 16

    def place(a, flag):
        t = dev(fragment_order(a) if packing & flag else np.concatenate([a, np.zeros((R - M, a.shape[1]), a.dtype)]))
        return t, Mr(t.data_ptr(), [1, M, a.shape[1]])

    def result(t):
        v = host(t)
        if not packing & 4:
            return v.reshape(R, N)[:M]
        return v.reshape(-1, N // 32, 4, 16, 8).transpose(0, 3, 1, 2, 4).reshape(R, N)[:M]

    tb = dev(B[None])
    packed = torch.zeros(K * N, dtype=torch.float16, device="cuda")
    gpu.homPackWeightF16(*Mr.from_tensor(tb).args(), packed.data_ptr())
    np.testing.assert_array_equal(host(packed), fragment_order(np.ascontiguousarray(B.T)))
    colsum = dev(B.astype(np.float32).sum(0))
    (ta, ma), (tc, mc), ts = place(A, 1), place(C, 2), dev(stats)
    td, out = torch.zeros(R * N, dtype=torch.float16, device="cuda"), torch.zeros((M, 2), device="cuda")
    md = Mr(td.data_ptr(), [1, M, N])
    x = A.astype(np.float64)
    rstd = 1 / np.sqrt(x.var(1) + 1e-6)
    ln = (x - x.mean(1, keepdims=True)) * rstd[:, None]
    # residual of normalised rows
    gpu.homPackedGemmF16(*ma.args(), packed.data_ptr(), *mc.args(), *md.args(), 0, 0, 1e-6, None, ts.data_ptr(), None,
                         packing, None, 0)
    want = x @ B.astype(np.float64) + C.astype(np.float64) * stats[:, :1] + stats[:, 1:]
    np.testing.assert_allclose(result(td).astype(np.float64), want, rtol=1e-3, atol=1e-2)
    # plain residual, reading ahead
    gpu.homPackedGemmF16(*ma.args(), packed.data_ptr(), *mc.args(), *md.args(), 0, 0, 1e-6, None, None, None, packing,
                         packed.data_ptr(), 2 * K * N)
    want = x @ B.astype(np.float64) + C.astype(np.float64)
    np.testing.assert_allclose(result(td).astype(np.float64), want, rtol=1e-3, atol=1e-2)
    # normalised A with both activations, and the row statistics
    for act, name in ((1, "gelu_erf"), (2, "gelu_tanh"), (0, "linear")):
        gpu.homPackedGemmF16(*ma.args(), packed.data_ptr(), 0, None, *md.args(), act, 1, 1e-6, colsum.data_ptr(), None,
                             out.data_ptr(), packing & ~2, None, 0)
        z = oracle.gemm(ln.astype(np.float32).astype(np.float16), B, act=name)  # (A rounded: within the tolerance)
        np.testing.assert_allclose(result(td).astype(np.float64), z, rtol=2e-3, atol=1e-2)
        np.testing.assert_allclose(host(out)[:, 0], rstd, rtol=1e-4)
        np.testing.assert_allclose(host(out)[:, 1], -x.mean(1) * rstd, rtol=1e-3, atol=1e-4)


# every tile of the packed GEMM for many rows, with one tile and with several of them per workgroup
# (test_packed_selection.py)
@pytest.mark.parametrize("M,N,K", MANY_ROWS)
def test_packed_gemm_many_rows(gpu, rt, M, N, K):
    g = torch.Generator("cuda").manual_seed(M)
    Mr, R = rt.MemRef, -(-M // 16) * 16

    def rand(*shape, std=1.0):
        return (torch.randn(shape, device="cuda", generator=g) * std).half()

    def order(a):
        p = torch.zeros(R, a.shape[1], dtype=a.dtype, device="cuda")
        p[:M] = a
        return p.view(-1, 16, a.shape[1] // 32, 4, 8).permute(0, 2, 3, 1, 4).contiguous().view(-1)

    A, B, C = rand(M, K) + 0.3, rand(K, N, std=0.05), rand(M, N)
    packed, stats = torch.zeros(K * N, dtype=torch.float16, device="cuda"), torch.rand(M, 2, device="cuda", generator=g)
    gpu.homPackWeightF16(*Mr(B.data_ptr(), [1, K, N]).args(), packed.data_ptr())
    ta, tc, td = order(A), order(C), torch.zeros(R * N, dtype=torch.float16, device="cuda")
    ma, mc, md = (Mr(t.data_ptr(), [1, M, w]) for t, w in ((ta, K), (tc, N), (td, N)))
    out, colsum = torch.zeros(M, 2, device="cuda"), B.float().sum(0)

    def check(want, rtol):
        got = td.view(-1, N // 32, 4, 16, 8).permute(0, 3, 1, 2, 4).reshape(R, N)[:M].double()
        torch.testing.assert_close(got, want, rtol=rtol, atol=1e-2)

    x, w = A.double(), B.double()
    gpu.homPackedGemmF16(*ma.args(), packed.data_ptr(), *mc.args(), *md.args(), 0, 0, 1e-6, None, stats.data_ptr(), None,
                         7, packed.data_ptr(), 2 * K * N)
    check(x @ w + C.double() * stats[:, :1].double() + stats[:, 1:].double(), 1e-3)
    rstd = (x.var(1, unbiased=False) + 1e-6).rsqrt()
    z = ((x - x.mean(1, keepdim=True)) * rstd[:, None]) @ w
    for act, fn in ((0, lambda v: v), (1, torch.nn.functional.gelu), (2, lambda v: torch.nn.functional.gelu(v, approximate="tanh"))):
        gpu.homPackedGemmF16(*ma.args(), packed.data_ptr(), 0, None, *md.args(), act, 1, 1e-6, colsum.data_ptr(), None,
                             out.data_ptr(), 5, None, 0)
        check(fn(z), 2e-3)
        torch.testing.assert_close(out[:, 0].double(), rstd, rtol=1e-4, atol=0)
        gpu.homPackedGemmF16(*ma.args(), packed.data_ptr(), 0, None, *md.args(), act, 0, 1e-6, None, None, None, 5, None, 0)
        check(fn(x @ w), 1e-3)


@pytest.mark.parametrize("M,H", [(1, 32), (17, 96), (33, 768), (16, 800), (50, 1024), (15, 1056), (100, 2048)])
def test_packed_layernorm(gpu, rt, M, H):
    x = (np.random.default_rng(M + H).standard_normal((M, H)) * 2 + 0.5).astype(np.float16)
    Mr, R = rt.MemRef, -(-M // 16) * 16
    t, rows = dev(fragment_order(x)), torch.zeros((M, H), dtype=torch.float16, device="cuda")
    m = Mr(t.data_ptr(), [1, M, H])
    want = torch.nn.functional.layer_norm(torch.from_numpy(x).double(), (H,), eps=1e-6).numpy()
    gpu.homPackedLayernormF16(*m.args(), *Mr(rows.data_ptr(), [1, M, H]).args(), 1e-6, 1)
    np.testing.assert_allclose(host(rows), want, rtol=1e-3, atol=2e-3)
    gpu.homPackedLayernormF16(*m.args(), *m.args(), 1e-6, 5)
    got = host(t).reshape(-1, H // 32, 4, 16, 8).transpose(0, 3, 1, 2, 4).reshape(R, H)[:M]
    np.testing.assert_array_equal(got, host(rows))


# every way of the attention kernel; batch entries that start inside a row block, chunk ends inside one
@pytest.mark.parametrize("bs,seq,heads", [(1, 1, 1), (3, 33, 2), (2, 64, 12), (5, 99, 16), (2, 300, 4), (24, 128, 12),
                                          (40, 200, 8), (257, 17, 3), (44, 100, 12)])
def test_attention_in_fragment_order(gpu, rt, bs, seq, heads):
    g, H = np.random.default_rng(bs + seq), heads * 64
    rows, Mr = bs * seq, rt.MemRef
    R = -(-rows // 16) * 16
    qkv = g.standard_normal((rows, 3 * H)).astype(np.float16)
    lens = g.integers(1, seq + 1, bs)
    cu = dev(np.concatenate([[0], np.cumsum(lens)]).astype(np.int32))
    a, out = dev(qkv.reshape(bs, seq, 3 * H)), torch.zeros((bs, seq, H), dtype=torch.float16, device="cuda")
    gpu.nvteBertAttentionF16(*Mr.from_tensor(a).args(), *Mr.from_tensor(cu).args(), *Mr.from_tensor(out).args(), 0.125, heads)
    p, packed = dev(fragment_order(qkv)), torch.zeros(R * H, dtype=torch.float16, device="cuda")
    gpu.homBertAttentionF16(*Mr(p.data_ptr(), [bs, seq, 3 * H]).args(), *Mr.from_tensor(cu).args(),
                            *Mr(packed.data_ptr(), [bs, seq, H]).args(), 0.125, heads, 5, p.data_ptr(), 6 * rows * H)
    got = host(packed).reshape(-1, H // 32, 4, 16, 8).transpose(0, 3, 1, 2, 4).reshape(R, H)[:rows].reshape(bs, seq, H)
    want = host(out)
    for b in range(bs):
        np.testing.assert_allclose(got[b, :lens[b]].astype(np.float32), want[b, :lens[b]].astype(np.float32), rtol=2e-3,
                                   atol=1e-3)


@pytest.mark.parametrize("bs,seq", [(300, 128), (340, 127)])
def test_encoder_many_rows_equals_row_major(synth, bs, seq):
    """Enough rows for packed layer norms of their own, against the same weights on the row-major path."""
    import importlib
    bert = importlib.import_module("hands-on-mlir_amd.bert")
    model = synth.bert_encoder(layers=2, hidden=128, heads=2, ffn=512, bs=bs, seq=seq, vocab=1000, config=40)
    got = []
    for layout in (None, {"qkv": "kn"}):
        enc = bert.BertEncoder(2, 128, 2, 512, bs, seq, 1000, gemm_mode=1, gelu_form="erf", role_layout=layout)
        try:
            enc.load(model)
            enc.set_inputs(ids=model["ids"], mask=model["mask"])
            enc.forward()
            got.append(enc.output().astype(np.float32))
        finally:
            enc.close()
    live = np.asarray(model["mask"]).astype(bool)
    np.testing.assert_allclose(got[0][live], got[1][live], rtol=1e-2, atol=1e-2)


# the result is stored 16 bytes a lane from any 8-byte boundary: the same values there, padding rows included, and
# nothing beside them (each way of the dispatch)
@pytest.mark.parametrize("bs,seq,heads,d", [(1, 50, 2, 64), (3, 100, 4, 64), (30, 128, 12, 64), (2, 300, 4, 64),
                                            (2, 200, 4, 128), (3, 130, 3, 192), (2, 70, 2, 256), (8, 384, 16, 256),
                                            (44, 100, 12, 64)])
def test_attention_result_on_8_bytes(gpu, rt, bs, seq, heads, d):
    g = torch.Generator(device="cuda").manual_seed(seq)
    qkv = torch.randn(bs, seq, 3 * heads * d, generator=g, device="cuda").half()
    lens = torch.randint(1, seq + 1, (bs,), generator=g, device="cuda")
    cu = torch.zeros(bs + 1, dtype=torch.int32, device="cuda")
    cu[1:] = torch.cumsum(lens, 0)
    n, Mr, results = bs * seq * heads * d, rt.MemRef.from_tensor, []
    for off in (0, 4):
        t = torch.full((n + 64,), float("nan"), dtype=torch.float16, device="cuda")
        out = t[32 + off:32 + off + n].view(bs, seq, heads * d)
        gpu.nvteBertAttentionF16(*Mr(qkv).args(), *Mr(cu).args(), *Mr(out).args(), d ** -0.5, heads)
        results.append(host(out))
        assert int(torch.isnan(t).sum()) == 64
    np.testing.assert_array_equal(results[0], results[1])
    for b in range(bs):
        assert not results[0][b, int(lens[b]):].any()


# every way the attention is split, lengths around its chunk ends; what lies behind a sequence must not matter
@pytest.mark.parametrize("bs,seq,heads,d", [(2, 60, 4, 64), (3, 100, 4, 64), (30, 128, 12, 64), (2, 300, 4, 64),
                                            (40, 200, 8, 64), (2, 64, 4, 128), (3, 130, 4, 128), (40, 256, 8, 128),
                                            (2, 70, 3, 192), (16, 129, 9, 192), (2, 70, 3, 256), (16, 129, 9, 256),
                                            (5, 193, 2, 256), (44, 100, 12, 64)])
def test_attention_splits(gpu, rt, bs, seq, heads, d):
    g = torch.Generator("cuda").manual_seed(seq + d)
    qkv = torch.randn(bs, seq, 3, heads, d, device="cuda", generator=g).half()
    lens = torch.randint(1, seq + 1, (bs,), device="cuda", generator=g)
    lens[0], lens[-1] = seq, min(seq, 65)
    live = torch.arange(seq, device="cuda")[None, :] < lens[:, None]
    q, k, v = qkv.float().permute(2, 0, 3, 1, 4).contiguous()
    s = torch.matmul(q, k.transpose(2, 3).contiguous()) / d ** 0.5
    want = torch.matmul(s.masked_fill(~live[:, None, None, :], float("-inf")).softmax(-1), v).permute(0, 2, 1, 3)
    want = want.reshape(bs, seq, heads * d) * live[:, :, None]
    qkv[~live] = float("nan")
    cu = torch.zeros(bs + 1, dtype=torch.int32, device="cuda")
    cu[1:] = lens.cumsum(0)
    out = torch.full((bs, seq, heads * d), 7.0, dtype=torch.float16, device="cuda")
    Mr = rt.MemRef
    gpu.nvteBertAttentionF16(*Mr.from_tensor(qkv.view(bs, seq, -1)).args(), *Mr.from_tensor(cu).args(),
                             *Mr.from_tensor(out).args(), d ** -0.5, heads)
    torch.testing.assert_close(out.float(), want, rtol=2e-3, atol=2e-3)


# lengths at the ends of 32-key blocks and 64-key chunks: split keys (64, 128, 256), whole rows (128; 64 up to 128
# tokens with more tiles than half the CUs), split keys between one and 1.4 tiles a CU, chunks through registers (64 with
# more than two tiles a CU, 256 from half a tile on), and both ways of 192 at the line between them
@pytest.mark.parametrize("bs,seq,heads,d", [(13, 200, 2, 64), (13, 200, 2, 128), (13, 200, 2, 256), (48, 200, 2, 128),
                                            (48, 100, 4, 64), (13, 200, 11, 128), (13, 200, 11, 64), (7, 64, 2, 128),
                                            (10, 192, 2, 256), (13, 160, 11, 64), (13, 160, 11, 128), (48, 100, 11, 64),
                                            (48, 200, 2, 256), (16, 100, 8, 192), (13, 200, 5, 192)])
def test_attention_chunk_ends(gpu, rt, bs, seq, heads, d):
    g = torch.Generator("cuda").manual_seed(seq + d)
    qkv = torch.randn(bs, seq, 3, heads, d, device="cuda", generator=g)
    qkv[:, :, 1] *= 1.0 + 4.0 * torch.arange(seq, device="cuda")[None, :, None, None] / seq  # the reference moves
    qkv = qkv.half()
    ends = [1, 31, 32, 33, 63, 64, 65, 96, 97, 128, 129, 192, 200]
    lens = torch.tensor([min(seq, ends[i % 13]) for i in range(bs)], device="cuda")
    live = torch.arange(seq, device="cuda")[None, :] < lens[:, None]
    q, k, v = qkv.float().permute(2, 0, 3, 1, 4).contiguous()
    s = torch.matmul(q, k.transpose(2, 3).contiguous()) / d ** 0.5
    want = torch.matmul(s.masked_fill(~live[:, None, None, :], float("-inf")).softmax(-1), v).permute(0, 2, 1, 3)
    want = want.reshape(bs, seq, heads * d) * live[:, :, None]
    qkv[~live] = float("nan")
    cu = torch.zeros(bs + 1, dtype=torch.int32, device="cuda")
    cu[1:] = lens.cumsum(0)
    out = torch.full((bs, seq, heads * d), 7.0, dtype=torch.float16, device="cuda")
    Mr = rt.MemRef
    gpu.nvteBertAttentionF16(*Mr.from_tensor(qkv.view(bs, seq, -1)).args(), *Mr.from_tensor(cu).args(),
                             *Mr.from_tensor(out).args(), d ** -0.5, heads)
    # probabilities and result in fp16: 2 * 2^-11 of values up to about 4
    torch.testing.assert_close(out.float(), want, rtol=2e-3, atol=4e-3)


@pytest.mark.parametrize("K,N", [(32, 16), (96, 48), (768, 2304), (1056, 320)])
def test_pack_weight_and_back(gpu, rt, K, N):
    B = np.random.default_rng(K + N).standard_normal((1, K, N)).astype(np.float16)
    Mr, tb = rt.MemRef, dev(B)
    packed, back = (torch.zeros(K * N, dtype=torch.float16, device="cuda") for _ in range(2))
    gpu.homPackWeightF16(*Mr.from_tensor(tb).args(), packed.data_ptr())
    gpu.homUnpackWeightF16(packed.data_ptr(), *Mr(back.data_ptr(), [1, K, N]).args())
    np.testing.assert_array_equal(host(back).reshape(1, K, N), B)


@pytest.mark.parametrize("b,s,H", [(1, 1, 32), (1, 16, 64), (3, 11, 96), (5, 33, 768), (2, 100, 2048)])
def test_pack_rows(gpu, rt, b, s, H):
    a = np.random.default_rng(s + H).standard_normal((b, s, H)).astype(np.float16)
    Mr, R = rt.MemRef, -(-b * s // 16) * 16
    ta, out = dev(a), torch.full((R * H + 8,), 7.0, dtype=torch.float16, device="cuda")
    gpu.homPackRowsF16(*Mr.from_tensor(ta).args(), *Mr(out.data_ptr(), [b, s, H]).args())
    np.testing.assert_array_equal(host(out)[:R * H], fragment_order(a.reshape(b * s, H)))
    assert (host(out)[R * H:] == 7).all()


# few rows, the tile kernels with folded layer norms, and layer norms of their own
@pytest.mark.parametrize("bs,seq", [(1, 16), (3, 33), (8, 128), (340, 127)])
def test_encoder_from_hidden_states_equals_from_ids(gpu, rt, synth, bs, seq):
    """Hidden states given to the encoder take the same kernels as those its embedding front makes: the same bits."""
    import importlib
    bert = importlib.import_module("hands-on-mlir_amd.bert")
    m = synth.bert_encoder(layers=2, hidden=128, heads=2, ffn=512, bs=bs, seq=seq, vocab=100, config=43)
    enc = bert.BertEncoder(2, 128, 2, 512, bs, seq, 100, gemm_mode=1, gelu_form="erf")
    try:
        enc.load(m)
        assert enc.uses_packed()
        Mr = rt.MemRef.from_tensor
        ids, mask, word, pos = dev(m["ids"].astype(np.int64)), dev(m["mask"].astype(np.int64)), dev(m["word"][None]), dev(m["pos_type"][None])
        h, cu = torch.zeros(bs, seq, 128, dtype=torch.float16, device="cuda"), torch.zeros(bs + 1, dtype=torch.int32, device="cuda")
        gpu.homEmbedF16(*Mr(ids).args(), *Mr(mask).args(), *Mr(word).args(), *Mr(pos).args(), *Mr(h).args(),
                        *Mr(cu).args(), 1e-12, 0)
        hidden = host(h)
        enc.set_inputs(ids=m["ids"], mask=m["mask"])
        enc.forward()
        want = enc.output()
        enc.set_inputs(hidden=hidden)
        enc.forward(from_ids=False)
        np.testing.assert_array_equal(enc.output(), want)
        enc.set_inputs(hidden=hidden)
        enc.capture(from_ids=False)
        for _ in range(3):
            enc.set_inputs(hidden=hidden)
            enc.replay()
            np.testing.assert_array_equal(enc.output(), want)
            enc.forward()
            np.testing.assert_array_equal(enc.output(), want)
    finally:
        enc.close()


@pytest.mark.parametrize("pin", [False, True])
def test_weights_uploaded_again(gpu, rt, synth, pin):
    """Weights uploaded between a capture and its replays take effect, on packed weights and after a pinned kernel
    has taken the encoder off them; a graph captured on packed weights still runs then."""
    import importlib
    bert = importlib.import_module("hands-on-mlir_amd.bert")
    a, b = (synth.bert_encoder(layers=2, hidden=128, heads=2, ffn=512, bs=3, seq=33, vocab=100, config=c) for c in (50, 51))
    number = {n: i + 1 for i, n, _, _ in rt.manifest()}
    tile = "hom_gfx950_mfma_f16_s32x32x16gemm_f16_128x64_64x2r2_w2x2_nn_align8_linear"

    def make(m):
        enc = bert.BertEncoder(2, 128, 2, 512, 3, 33, 100, gemm_mode=1, gelu_form="erf")
        enc.load(m)
        enc.set_inputs(ids=a["ids"], mask=a["mask"])
        return enc

    def result(enc):
        enc.replay()
        return enc.output()

    want = []
    for m in (a, b):  # encoders that never saw other weights
        enc = make(m)
        if pin:
            enc.set_gemm_choice("out", number[tile])
        enc.capture()
        want.append(result(enc))
        enc.close()
    assert not np.array_equal(*want)
    enc = make(a)
    try:
        enc.capture()
        if pin:
            packed = result(enc)
            enc.set_gemm_choice("out", number[tile])
            np.testing.assert_array_equal(result(enc), packed)  # the graph from before
            enc.capture()
        np.testing.assert_array_equal(result(enc), want[0])  # (unpacked weights are the uploaded ones)
        for m, w in ((b, want[1]), (a, want[0])):
            enc.load(m)
            for _ in range(2):
                np.testing.assert_array_equal(result(enc), w)
    finally:
        enc.close()


# few rows (both orders of A, all of K at once and in rounds) and every tile that folds a layer norm
@pytest.mark.parametrize("M,N,K,packing", [(*size, packing) for packing in (0, 5) for size in NORMALISED_FEW] +
                         [(*size, 5) for size in NORMALISED_MANY])
@pytest.mark.parametrize("sigmas", [0, 3, 5, 60, 300])
def test_packed_gemm_of_rows_far_from_zero(gpu, rt, M, N, K, packing, sigmas):
    """A folded layer norm on rows whose mean is `sigmas` times their spread, mixed with rows around zero, constant
    rows and rows of one value among zeros: the statistics as close to 64 bits as sums of 32 allow, the result as
    close as its rounding to fp16 and the sum that cancels (sigmas x 2^-24 x some ten) allow."""
    g = torch.Generator("cuda").manual_seed(M + sigmas)
    Mr, R = rt.MemRef, -(-M // 16) * 16
    A = torch.randn(M, K, device="cuda", generator=g)
    A[::3] += sigmas
    A[1::5] -= sigmas
    A[2::16] = 0
    A[2::16, 1] = 5
    if sigmas:
        A[3::16] = 0.1  # constant
    A, B = A.half(), (torch.randn(K, N, device="cuda", generator=g) * 0.05).half()
    ta = torch.full((R, K), 3.0, device="cuda").half()  # (what fills the last row block is not a row)
    ta[:M] = A
    if packing & 1:
        ta = ta.view(R // 16, 16, K // 32, 4, 8).permute(0, 2, 3, 1, 4).contiguous()
    packed, td = torch.zeros(K * N, dtype=torch.float16, device="cuda"), torch.zeros(R * N, dtype=torch.float16, device="cuda")
    out, colsum = torch.full((M + 1, 2), 7.0, device="cuda"), B.double().sum(0).float()
    gpu.homPackWeightF16(*Mr(B.data_ptr(), [1, K, N]).args(), packed.data_ptr())
    gpu.homPackedGemmF16(*Mr(ta.data_ptr(), [1, M, K]).args(), packed.data_ptr(), 0, None,
                         *Mr(td.data_ptr(), [1, M, N]).args(), 0, 1, 1e-6, colsum.data_ptr(), None, out.data_ptr(), packing,
                         None, 0)
    got = td.view(R, N) if not packing & 4 else td.view(-1, N // 32, 4, 16, 8).permute(0, 3, 1, 2, 4).reshape(R, N)
    x = A.double()
    mean = x.mean(1, keepdim=True)
    rstd = (((x - mean) ** 2).mean(1, keepdim=True) + 1e-6).rsqrt()
    keep = torch.ones(M, dtype=torch.bool, device="cuda")
    if sigmas:
        keep[3::16] = False  # (there eps alone is left, and the mean's last place divided by it)
        assert torch.isfinite(got[:M]).all()
    # one pass serves up to 4 sigma: there (1 + 16) / 2 times what a sum of 256 terms in a row loses, sqrt(256) x 2^-24
    # and for the worst of thousands of rows at most twice that, 1.6e-5
    torch.testing.assert_close(out[:M][keep][:, :1].double(), rstd[keep], rtol=2e-5, atol=0)
    torch.testing.assert_close(out[:M][keep][:, 1:].double(), (-mean * rstd)[keep], rtol=2e-5, atol=1e-5)
    assert (out[M] == 7).all()
    want = ((x - mean) * rstd) @ B.double()
    rel = ((got[:M].double() - want)[keep].norm() / want[keep].norm()).item()
    assert rel <= 3.5e-4 + 1e-6 * sigmas, rel
