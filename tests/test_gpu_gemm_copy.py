"""Products on rounded copies, one and the two gradients of a product in one launch, against whole-number products in float64, bit
for bit, on every workgroup tile. The library reads NZHIP_GEMM_COPY and NZHIP_GEMM_COPY_PLAN ("tile,parts") per call, so products
and plans it would choose only at large sizes can be forced."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TILES = range(6)         # 64 x 64, 64 x 64 with two groups of waves, 128 x 64, 64 x 128, 128 x 128, 128 x 256


@pytest.fixture(scope="module")
def nz():
    import torch
    assert torch.cuda.is_available(), "these tests need the MI355X"
    from neuzephyr_amd import capi
    capi.load()
    return capi


def whole(rng, *shape):
    return rng.integers(-2, 3, shape).astype(np.float32)


def embedded(a):
    """a at an odd offset in NaN-filled storage: (storage, view)"""
    import torch
    buf = torch.full((a.size + 14,), float("nan"), device="cuda")
    buf[7:7 + a.size] = torch.from_numpy(np.ascontiguousarray(a).ravel()).cuda()
    return buf, buf[7:7 + a.size].view(a.shape)


def untouched(buf, n):
    import torch
    return bool(torch.isnan(buf[:7]).all() and torch.isnan(buf[7 + n:]).all())


# one over and one under the tiles; k of one step, of a unit less, of a unit more; nine panels of tile columns
SHAPES = [(65, 63, 129), (9, 72, 16), (130, 9, 67), (257, 200, 255), (64, 64, 64), (33, 577, 33), (200, 65, 600), (3, 129, 5)]


@pytest.mark.parametrize("a_trans,b_trans", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("tile", TILES)
def test_every_tile_and_layout_is_bit_exact_on_whole_numbers(nz, monkeypatch, tile, a_trans, b_trans):
    import torch
    monkeypatch.setenv("NZHIP_GEMM_COPY", "1")
    for M, K, N in SHAPES:
        rng = np.random.default_rng(M + 3 * K + 5 * N + tile)
        A, B, old, b = whole(rng, M, K), whole(rng, K, N), whole(rng, M, N), whole(rng, M * N)
        want = A.astype(np.float64) @ B
        a, bb = embedded(A.T if a_trans else A)[1], embedded(B.T if b_trans else B)[1]
        for parts in (1, 2, 3):
            monkeypatch.setenv("NZHIP_GEMM_COPY_PLAN", f"{tile},{parts}")
            tag = (M, K, N, parts)
            buf, out = embedded(np.full((M, N), np.nan, np.float32))
            nz.gemm(a, bb, a_trans=a_trans, b_trans=b_trans, out=out)
            assert np.array_equal(out.cpu().numpy(), want) and untouched(buf, M * N), tag
            for strides, bias in (((0, 1), b[:N][None, :]), ((1, 0), b[:M][:, None]), ((N, 1), b.reshape(M, N)), ((1, M), b.reshape(N, M).T)):
                nz.gemm(a, bb, a_trans=a_trans, b_trans=b_trans, bias=embedded(b)[1], bias_strides=strides, relu=True, out=out)
                assert np.array_equal(out.cpu().numpy(), np.maximum(want + bias, 0)) and untouched(buf, M * N), (tag, strides)
            buf, out = embedded(old)                                   # accumulating in place
            nz.gemm(a, bb, a_trans=a_trans, b_trans=b_trans, bias=out, bias_strides=(N, 1), out=out)
            assert np.array_equal(out.cpu().numpy(), want + old) and untouched(buf, M * N), tag


@pytest.mark.parametrize("K", [512, 576, 16384])
@pytest.mark.parametrize("tile", TILES)
def test_a_long_contraction_is_summed_in_chains_of_512(nz, monkeypatch, tile, K):
    """Unsplit: bit-exact on whole numbers, and the error of chains, not of one long sum. Each addition of a chain of n terms of equal variance
    rounds a partial sum of i terms by u sqrt(i / n) at most, evenly distributed: relative variance n u^2 / 6, with u = 2^-24. n = 512 for the
    chains, K / 512 for their sum: 5.7e-7 at 16384 (one sum: up to 3.1e-6, 8e-7 as MFMAs add several terms at once)."""
    import torch
    monkeypatch.setenv("NZHIP_GEMM_COPY", "1")
    monkeypatch.setenv("NZHIP_GEMM_COPY_PLAN", f"{tile},1")
    rng = np.random.default_rng(K + tile)
    A, B = whole(rng, 70, K), whole(rng, K, 130)
    assert np.array_equal(nz.gemm(torch.from_numpy(A).cuda(), torch.from_numpy(B).cuda()).cpu().numpy(), A.astype(np.float64) @ B)
    A, B = (rng.standard_normal(x.shape).astype(np.float16).astype(np.float32) for x in (A, B))
    want = A.astype(np.float64) @ B
    err = nz.gemm(torch.from_numpy(A).cuda(), torch.from_numpy(B).cuda()).cpu().numpy() - want
    assert np.linalg.norm(err) <= np.linalg.norm(want) * 2.0 ** -24 * np.sqrt((512 + K / 512) / 6)


@pytest.mark.parametrize("K", [1, 64, 65, 128, 129, 192, 257, 1000])
def test_waves_that_take_turns_are_bit_exact_on_whole_numbers(nz, monkeypatch, K):
    """128 x 256 tiles, 100 of them side by side, of one to 16 steps: fewer than the ring's three, as many, one more, many."""
    import torch
    monkeypatch.setenv("NZHIP_GEMM_COPY", "1")
    monkeypatch.setenv("NZHIP_GEMM_COPY_PLAN", "5,1")
    rng = np.random.default_rng(K)
    A, B = whole(rng, 1270, K), whole(rng, K, 2500)
    want = A @ B                                                       # whole numbers below 2^24: exact in fp32
    a, b = torch.from_numpy(A).cuda(), torch.from_numpy(B).cuda()
    for a_trans in (False, True):
        for b_trans in (False, True):
            aa, bb = a.T.contiguous() if a_trans else a, b.T.contiguous() if b_trans else b
            assert np.array_equal(nz.gemm(aa, bb, a_trans=a_trans, b_trans=b_trans).cpu().numpy(), want), (a_trans, b_trans)


@pytest.mark.parametrize("S,inputs,outputs", [(29, 466, 640), (64, 848, 786), (48, 880, 1984), (16, 792, 2752)])
def test_gradients_of_few_samples_are_as_exact_as_one_product_after_the_other(nz, monkeypatch, S, inputs, outputs):
    """Error in the 2-norm against float64 on operands that fp16 holds exactly: only the order of the fp32 sums counts."""
    import torch
    rng = np.random.default_rng(S)
    W, x, dz = (rng.standard_normal(s).astype(np.float16).astype(np.float32) for s in ((1, 1, outputs, inputs), (S, 1, inputs, 1), (S, 1, outputs, 1)))
    want = dz[:, 0, :, 0].T.astype(np.float64) @ x[:, 0, :, 0], dz[:, 0, :, 0].astype(np.float64) @ W[0, 0]
    err = {}
    for route in ("0", "1"):
        monkeypatch.setenv("NZHIP_GEMM_COPY", route)
        gw, gx = torch.zeros(W.shape, device="cuda"), torch.zeros(x.shape, device="cuda")
        nz.matmul_backward(gw, gx, *(torch.from_numpy(a).cuda() for a in (W, x, dz)))
        err[route] = [np.linalg.norm(g.cpu().numpy().reshape(r.shape) - r) / np.linalg.norm(r) for g, r in zip((gw, gx), want)]
    assert all(now <= 1.05 * before for now, before in zip(err["1"], err["0"])), err      # (the norm moves by a few hundredths with the order)


@pytest.mark.parametrize("S,inputs,outputs", [(65, 130, 63), (9, 300, 200), (257, 65, 10), (128, 64, 256), (40, 9, 600)])
@pytest.mark.parametrize("tile", TILES)
def test_both_gradients_of_a_linear_layer_are_bit_exact_on_whole_numbers(nz, monkeypatch, tile, S, inputs, outputs):
    monkeypatch.setenv("NZHIP_GEMM_COPY", "1")
    rng = np.random.default_rng(S + inputs + outputs)
    W, x, dz = whole(rng, 1, 1, outputs, inputs), whole(rng, S, 1, inputs, 1), whole(rng, S, 1, outputs, 1)
    dW0, dx0 = whole(rng, *W.shape), whole(rng, *x.shape)
    dW = dz[:, 0, :, 0].T.astype(np.float64) @ x[:, 0, :, 0] + dW0[0, 0]
    dx = dz[:, 0, :, 0].astype(np.float64) @ W[0, 0] + dx0[:, 0, :, 0]
    for parts in (1, 3):
        monkeypatch.setenv("NZHIP_GEMM_COPY_PLAN", f"{tile},{parts}")
        (bw, gw), (bx, gx) = embedded(dW0), embedded(dx0)
        nz.matmul_backward(gw, gx, embedded(W)[1], embedded(x)[1], embedded(dz)[1])
        assert np.array_equal(gw.cpu().numpy()[0, 0], dW) and untouched(bw, W.size)
        assert np.array_equal(gx.cpu().numpy()[:, 0, :, 0], dx) and untouched(bx, x.size)


def test_gradients_that_share_memory_with_an_operand_are_computed_one_after_the_other(nz, monkeypatch):
    # dA = the output gradient's memory: the second product reads what the first one wrote, as it did with two launches
    import torch
    rng = np.random.default_rng(3)
    A, B, dC = whole(rng, 1, 1, 96, 96), whole(rng, 1, 1, 96, 96), whole(rng, 1, 1, 96, 96)
    dB = np.zeros_like(B)
    want_dA = dC[0, 0] + dC[0, 0] @ B[0, 0].T
    want_dB = A[0, 0].T @ want_dA
    monkeypatch.setenv("NZHIP_GEMM_COPY", "1")
    cu = lambda a: torch.from_numpy(a.copy()).cuda()
    shared, gB = cu(dC), cu(dB)
    nz.matmul_backward(shared, gB, cu(A), cu(B), shared)
    assert np.array_equal(shared.cpu().numpy()[0, 0], want_dA) and np.array_equal(gB.cpu().numpy()[0, 0], want_dB)


@pytest.mark.parametrize("special", [float("inf"), float("nan"), 7e4])             # 7e4 is infinite in fp16
@pytest.mark.parametrize("a_trans,b_trans", [(False, False), (True, True)])
def test_a_special_value_stays_in_its_row_or_column(nz, monkeypatch, special, a_trans, b_trans):
    import torch
    monkeypatch.setenv("NZHIP_GEMM_COPY", "1")
    M, K, N = 70, 75, 66                                              # 75: a unit that is partly past the end of k
    rng = np.random.default_rng(4)
    A, B = rng.integers(1, 3, (M, K)).astype(np.float32), rng.integers(1, 3, (K, N)).astype(np.float32)
    want = A.astype(np.float64) @ B
    cu = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    run = lambda a, b: nz.gemm(cu(a.T if a_trans else a), cu(b.T if b_trans else b), a_trans=a_trans, b_trans=b_trans).cpu().numpy()
    for m, k in ((0, 0), (M - 1, K - 1), (5, 72)):
        a = A.copy()
        a[m, k] = special
        got, rest = run(a, B), np.arange(M) != m
        assert not np.isfinite(got[m]).any() and np.array_equal(got[rest], want[rest])
    for k, n in ((0, 0), (K - 1, N - 1), (72, 5)):
        b = B.copy()
        b[k, n] = special
        got, rest = run(A, b), np.arange(N) != n
        assert not np.isfinite(got[:, n]).any() and np.array_equal(got[:, rest], want[:, rest])


@pytest.mark.parametrize("M,K,N,b_trans", [(1235, 1116, 1766, True), (1000, 777, 513, False), (2831, 1296, 1001, False)])
def test_chosen_plans_are_bit_exact_on_whole_numbers(nz, M, K, N, b_trans):
    import torch
    rng = np.random.default_rng(M)
    A, B = whole(rng, M, K), whole(rng, K, N)
    got = nz.gemm(torch.from_numpy(A).cuda(), torch.from_numpy(np.ascontiguousarray(B.T if b_trans else B)).cuda(), b_trans=b_trans)
    assert np.array_equal(got.cpu().numpy(), A.astype(np.float64) @ B)


@pytest.mark.parametrize("b_trans", [False, True])
@pytest.mark.parametrize("M,K,N", [(2831, 1296, 2781), (2000, 777, 2001), (1801, 801, 1803), (3072, 768, 3072)])
def test_a_kept_image_gives_the_bits_of_the_plain_call(nz, M, K, N, b_trans):
    """The plain call multiplies copies, the one that keeps B's image takes the two-pass kernel: one sum over k in either."""
    import torch
    rng = np.random.default_rng(M)
    A, B, b = (torch.from_numpy(rng.standard_normal(s).astype(np.float32)).cuda() for s in ((M, K), (N, K) if b_trans else (K, N), (N,)))
    for how in ({}, {"bias": b, "bias_strides": (0, 1), "relu": True}):
        h = nz.Prepared()
        try:
            assert torch.equal(nz.gemm(A, B, b_trans=b_trans, prepared_b=h, **how), nz.gemm(A, B, b_trans=b_trans, **how))
            assert h.fills() == 1                                     # else the handle was not used, and both calls were the same one
        finally:
            h.close()


@pytest.mark.parametrize("S,inputs,outputs,copies", [(4096, 4096, 4096, False), (5000, 3000, 3500, False), (8192, 2048, 8192, False),
                                                     (4096, 1024, 4096, True), (1024, 4096, 4096, True)])
def test_gradients_of_large_layers_take_the_faster_way(nz, monkeypatch, S, inputs, outputs, copies):
    """Both in one launch on copies are summed in chains of 512, one after the other in one sum: other bits."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(S)
    W, x, dz = (torch.randn(s, device="cuda", generator=g) for s in ((1, 1, outputs, inputs), (S, 1, inputs, 1), (S, 1, outputs, 1)))

    def gradients(route):
        monkeypatch.setenv("NZHIP_GEMM_COPY", route) if route else monkeypatch.delenv("NZHIP_GEMM_COPY")
        return nz.matmul_backward(torch.zeros_like(W), torch.zeros_like(x), W, x, dz)

    one_launch, two, chosen = gradients("1"), gradients("0"), gradients(None)
    for way, taken in ((one_launch, copies), (two, not copies)):
        assert all(torch.equal(a, b) for a, b in zip(way, chosen)) == taken


@pytest.mark.parametrize("M,K,N", [(200, 5000, 5000), (1000, 777, 513), (381, 3820, 2880)])
def test_the_call_without_allocations_gives_the_same_bits(nz, M, K, N):
    import torch
    rng = np.random.default_rng(M)
    A, B = (torch.from_numpy(rng.standard_normal(s).astype(np.float32)).cuda() for s in ((M, K), (K, N)))
    assert torch.equal(nz.gemm(A, B, static=True), nz.gemm(A, B))
