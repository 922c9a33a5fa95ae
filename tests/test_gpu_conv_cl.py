"""The Conv2d kernels on channel-last fp16 copies (forward, data gradient, weight gradient) against float64 convolutions of
whole numbers, bit for bit, on every workgroup tile and with and without parts. The library reads NZHIP_CONV_CL and
NZHIP_CONV_CL_PLAN ("tile,parts") per call, so layers and plans it would choose only at large sizes can be forced."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TILES = range(5)          # 64 x 64, 64 x 64 with two groups of waves, 128 x 64, 64 x 128, 128 x 128


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


def oihw(w, C, K_h, K_w):
    """the library's [copy, 1, (c, r, s), o] as [copy][o][c][r][s]"""
    return w.reshape(w.shape[0], C, K_h, K_w, w.shape[3]).transpose(0, 4, 1, 2, 3)


def reference(x, w, dy, K_h, K_w, stride, pad):
    """forward sums and both gradients in float64 (whole numbers: exact)"""
    import torch
    import torch.nn.functional as F
    X = torch.from_numpy(x.astype(np.float64)).requires_grad_()
    Wt = torch.from_numpy(oihw(w, x.shape[1], K_h, K_w).astype(np.float64).copy()).requires_grad_()
    per = Wt.shape[0] > 1
    y = torch.cat([F.conv2d(X[n:n + 1], Wt[n if per else 0], stride=stride, padding=pad) for n in range(x.shape[0])])
    y.backward(torch.from_numpy(dy.astype(np.float64)))
    dw = Wt.grad.numpy().transpose(0, 2, 3, 4, 1).reshape(w.shape)
    return y.detach().numpy(), X.grad.numpy(), dw


# N, C, H, W, O, K_h, K_w, stride, pad, copies
LAYERS = [
    (2, 8, 9, 11, 64, 3, 3, 1, 1, 1),          # one group of 8 channels; 198 pixels: part of every tile
    (3, 13, 8, 8, 65, 3, 3, 1, 1, 3),          # 13 channels in 16, a copy per image, a second channel tile with one row
    (1, 3, 7, 7, 5, 7, 7, 2, 3, 1),            # 3 channels in 8, 49 taps, more taps than pixels
    (5, 20, 6, 5, 17, 5, 5, 1, 2, 1),          # kernel as large as the image
    (2, 70, 14, 14, 130, 3, 3, 2, 1, 1),       # stride 2: four sums of 1, 2, 2 and 4 taps
    (3, 20, 29, 31, 12, 3, 3, 2, 1, 1),        # four sums of 720 to 630 pixels, 12 to 10 tiles
    (2, 33, 10, 13, 9, 3, 3, 3, 0, 2),         # stride 3, no padding, columns that no window reaches
    (2, 17, 12, 12, 24, 2, 2, 3, 0, 1),        # kernel below the stride: sums without a tap
    (1, 9, 1, 40, 8, 1, 1, 1, 0, 1),           # no window at all, one row
    (4, 40, 4, 4, 72, 4, 4, 2, 3, 1),          # even kernel, padding up to its edge, 16-pixel images
    (1, 130, 23, 3, 66, 3, 3, 1, 2, 1),        # output larger than the input
]


@pytest.mark.parametrize("layer", LAYERS)
@pytest.mark.parametrize("tile", TILES)
def test_every_tile_is_bit_exact_on_whole_numbers(nz, monkeypatch, tile, layer):
    import torch
    N, C, H, W, O, K_h, K_w, stride, pad, copies = layer
    rng = np.random.default_rng(sum(layer) + tile)
    Ho, Wo = (H + 2 * pad - K_h) // stride + 1, (W + 2 * pad - K_w) // stride + 1
    x, w, dy = whole(rng, N, C, H, W), whole(rng, copies, 1, C * K_h * K_w, O), whole(rng, N, O, Ho, Wo)
    b, old_dx, old_dw = whole(rng, 1, 1, Ho * Wo, O), whole(rng, *x.shape), whole(rng, *w.shape)
    y64, dx64, dw64 = reference(x, w, dy, K_h, K_w, stride, pad)
    bias = b.reshape(Ho * Wo, O).T.reshape(1, O, Ho, Wo)
    monkeypatch.setenv("NZHIP_CONV_CL", "1")
    X, Wt, DY, B = embedded(x)[1], embedded(w)[1], embedded(dy)[1], embedded(b)[1]
    for parts in (1, 3):
        monkeypatch.setenv("NZHIP_CONV_CL_PLAN", f"{tile},{parts}")
        buf, out = embedded(np.full(y64.shape, np.nan, np.float32))
        nz.conv2d_forward(X, Wt, B, K_h, K_w, stride, pad, bias_strides=(O, 1), relu=True, out=out)
        assert np.array_equal(out.cpu().numpy(), np.maximum(y64 + bias, 0)) and untouched(buf, y64.size)
        nz.conv2d_forward(X, Wt, torch.from_numpy(b.ravel()[:O].copy()).cuda(), K_h, K_w, stride, pad, bias_strides=(0, 1), out=out)
        assert np.array_equal(out.cpu().numpy(), y64 + b.ravel()[:O].reshape(1, O, 1, 1))
        nz.conv2d_forward(X, Wt, None, K_h, K_w, stride, pad, out=out)
        assert np.array_equal(out.cpu().numpy(), y64) and untouched(buf, y64.size)
        if K_h == K_w and pad <= K_h - 1:
            buf, dx = embedded(np.full(x.shape, np.nan, np.float32))
            nz.conv2d_backward_data(dx, DY, Wt, K_h, K_w, stride, pad, accumulate=False)
            assert np.array_equal(dx.cpu().numpy(), dx64) and untouched(buf, x.size)
            buf, dx = embedded(old_dx)
            nz.conv2d_backward_data(dx, DY, Wt, K_h, K_w, stride, pad)
            assert np.array_equal(dx.cpu().numpy(), dx64 + old_dx) and untouched(buf, x.size)
        buf, dw = embedded(old_dw)
        nz.conv2d_backward_weights(dw, X, DY, K_h, K_w, stride, pad)
        assert np.array_equal(dw.cpu().numpy(), dw64 + old_dw) and untouched(buf, w.size)


# N, C, H, W, O, K, pad, copies: rows of an odd and an even number of columns, of two and three; one row; no tap for the even columns, for the odd
# ones; a second channel tile of one row; more columns than windows reach
PAIRS = [(2, 8, 9, 11, 24, 3, 1, 1), (3, 65, 8, 12, 13, 3, 1, 3), (2, 5, 7, 2, 9, 3, 1, 1), (2, 5, 6, 3, 9, 3, 0, 2), (1, 9, 1, 40, 8, 1, 0, 1),
         (2, 12, 10, 9, 17, 1, 0, 1), (2, 4, 14, 15, 8, 7, 3, 1), (4, 40, 4, 4, 72, 4, 3, 1), (2, 33, 10, 13, 9, 2, 1, 2), (5, 20, 6, 6, 17, 5, 0, 1)]


@pytest.mark.parametrize("layer", PAIRS)
@pytest.mark.parametrize("tile", TILES)
def test_columns_in_pairs_are_bit_exact_on_whole_numbers(nz, monkeypatch, tile, layer):
    N, C, H, W, O, K, pad, copies = layer
    rng = np.random.default_rng(sum(layer) + tile)
    Ho, Wo = (H + 2 * pad - K) // 2 + 1, (W + 2 * pad - K) // 2 + 1
    x, w, dy, old = np.zeros((N, C, H, W), np.float32), whole(rng, copies if copies == 1 else N, 1, C * K * K, O), whole(rng, N, O, Ho, Wo), whole(rng, N, C, H, W)
    _, dx64, _ = reference(x, w, dy, K, K, 2, pad)
    monkeypatch.setenv("NZHIP_CONV_CL", "1")
    monkeypatch.setenv("NZHIP_CONV_CL_PAIRED", "1")
    for parts in (1, 2):
        monkeypatch.setenv("NZHIP_CONV_CL_PLAN", f"{tile},{parts}")
        for accumulate in (False, True):
            buf, dx = embedded(old if accumulate else np.full(x.shape, np.nan, np.float32))
            nz.conv2d_backward_data(dx, embedded(dy)[1], embedded(w)[1], K, K, 2, pad, accumulate=accumulate)
            assert np.array_equal(dx.cpu().numpy(), dx64 + (old if accumulate else 0)) and untouched(buf, x.size), (parts, accumulate)


@pytest.mark.parametrize("special", [float("inf"), float("nan"), -7e4])
@pytest.mark.parametrize("K,W", [(3, 10), (3, 11), (5, 10)])
def test_a_special_weight_reaches_only_its_columns_of_a_pair(nz, monkeypatch, special, K, W):
    import torch
    N, C, H, O, pad = 2, 70, 11, 20, K // 2
    rng = np.random.default_rng(7)
    Ho, Wo = (H + 2 * pad - K) // 2 + 1, (W + 2 * pad - K) // 2 + 1
    x, dy, w = np.zeros((N, C, H, W), np.float32), rng.integers(1, 3, (N, O, Ho, Wo)).astype(np.float32), rng.integers(1, 3, (1, 1, C * K * K, O)).astype(np.float32)
    _, dx64, _ = reference(x, w, dy, K, K, 2, pad)
    monkeypatch.setenv("NZHIP_CONV_CL", "1")
    monkeypatch.setenv("NZHIP_CONV_CL_PAIRED", "1")
    for c, tap, o in ((0, 0, 0), (C - 1, K * K - 1, O - 1), (33, K // 2 * K, 7), (64, 1, 8)):
        ws, mark = w.copy(), np.zeros_like(w)
        ws[0, 0, c * K * K + tap, o], mark[0, 0, c * K * K + tap, o] = special, 1
        _, hit, _ = reference(x, mark, dy, K, K, 2, pad)
        dx = torch.ones(x.shape, device="cuda")
        nz.conv2d_backward_data(dx, torch.from_numpy(dy).cuda(), torch.from_numpy(ws).cuda(), K, K, 2, pad)
        got = dx.cpu().numpy()
        assert np.array_equal(np.isfinite(got), hit == 0) and np.array_equal(got[hit == 0], dx64[hit == 0] + 1), (c, tap, o)


@pytest.mark.parametrize("special", [float("inf"), float("nan"), 7e4])             # 7e4 is infinite in fp16
@pytest.mark.parametrize("K,stride,pad", [(3, 1, 1), (3, 2, 1), (5, 1, 2)])
def test_a_special_value_stays_in_the_sums_it_is_a_term_of(nz, monkeypatch, special, K, stride, pad):
    import torch
    N, C, H, W, O = 2, 9, 11, 10, 20                                  # 9 channels in 16, pixel counts that fill no tile
    rng = np.random.default_rng(5)
    Ho, Wo = (H + 2 * pad - K) // stride + 1, (W + 2 * pad - K) // stride + 1
    x = rng.integers(1, 3, (N, C, H, W)).astype(np.float32)
    w, dy = rng.integers(1, 3, (1, 1, C * K * K, O)).astype(np.float32), rng.integers(1, 3, (N, O, Ho, Wo)).astype(np.float32)
    monkeypatch.setenv("NZHIP_CONV_CL", "1")
    at = (1, 4, H - 1, W - 1)                                         # the last pixel: beside the padding, before the next plane
    xs, mark = x.copy(), np.zeros_like(x)
    xs[at], mark[at] = special, 1
    y_hit, _, dw_hit = reference(mark, w, dy, K, K, stride, pad)
    y64, dx64, dw64 = reference(x, w, dy, K, K, stride, pad)
    cu = lambda a: torch.from_numpy(a).cuda()
    y = nz.conv2d_forward(cu(xs), cu(w), None, K, K, stride, pad).cpu().numpy()
    assert np.array_equal(np.isfinite(y), y_hit == 0) and np.array_equal(y[y_hit == 0], y64[y_hit == 0])
    dw = torch.zeros(w.shape, device="cuda")
    nz.conv2d_backward_weights(dw, cu(xs), cu(dy), K, K, stride, pad)
    dw = dw.cpu().numpy()
    assert np.array_equal(np.isfinite(dw), dw_hit == 0) and np.array_equal(dw[dw_hit == 0], dw64[dw_hit == 0])
    dys, mark = dy.copy(), np.zeros_like(dy)
    dys[1, 3, Ho - 1, Wo - 1], mark[1, 3, Ho - 1, Wo - 1] = special, 1
    _, dx_hit, _ = reference(x, w, mark, K, K, stride, pad)
    dx = nz.conv2d_backward_data(torch.empty(x.shape, device="cuda"), cu(dys), cu(w), K, K, stride, pad, accumulate=False).cpu().numpy()
    assert np.array_equal(np.isfinite(dx), dx_hit == 0) and np.array_equal(dx[dx_hit == 0], dx64[dx_hit == 0])
    dw = torch.zeros(w.shape, device="cuda")
    nz.conv2d_backward_weights(dw, cu(x), cu(dys), K, K, stride, pad)
    dw = dw.cpu().numpy()
    dw_hit = np.broadcast_to(np.arange(O) == 3, dw.shape)              # padding is a term too: the column matrix holds zeros there, 0 x Inf
    assert np.array_equal(np.isfinite(dw), ~dw_hit) and np.array_equal(dw[~dw_hit], dw64[~dw_hit])


@pytest.mark.parametrize("special", [float("inf"), float("nan"), -7e4])            # -7e4 is infinite in fp16
@pytest.mark.parametrize("tile,parts", [(0, 1), (1, 3), (2, 1), (3, 2), (4, 1)])
@pytest.mark.parametrize("K,stride,pad,copies", [(3, 2, 1, 1), (3, 1, 1, 2), (5, 2, 2, 1), (4, 3, 2, 2)])
def test_a_special_weight_reaches_only_the_data_gradients_it_is_a_term_of(nz, monkeypatch, special, tile, parts, K, stride, pad, copies):
    """At the border of dx some taps lie outside dy: no terms of the sum, whatever their weight."""
    import torch
    N, C, H, W, O = 2, 70, 11, 10, 20
    rng = np.random.default_rng(6)
    Ho, Wo = (H + 2 * pad - K) // stride + 1, (W + 2 * pad - K) // stride + 1
    x, dy, old = np.zeros((N, C, H, W), np.float32), rng.integers(1, 3, (N, O, Ho, Wo)).astype(np.float32), whole(rng, N, C, H, W)
    w = rng.integers(1, 3, (copies, 1, C * K * K, O)).astype(np.float32)
    _, dx64, _ = reference(x, w, dy, K, K, stride, pad)
    monkeypatch.setenv("NZHIP_CONV_CL", "1")
    monkeypatch.setenv("NZHIP_CONV_CL_PLAN", f"{tile},{parts}")
    cu = lambda a: torch.from_numpy(a.copy()).cuda()
    for c, tap, o in ((0, 0, 0), (C - 1, K * K - 1, O - 1), (33, K // 2 * K, 7), (64, 1, 8)):
        at = (copies - 1, 0, c * K * K + tap, o)
        ws, mark = w.copy(), np.zeros_like(w)
        ws[at], mark[at] = special, 1
        _, hit, _ = reference(x, mark, dy, K, K, stride, pad)
        assert (hit != 0).any() and (hit[:, c] == 0).any()
        for accumulate in (False, True):
            dx = cu(old)
            nz.conv2d_backward_data(dx, cu(dy), cu(ws), K, K, stride, pad, accumulate=accumulate)
            got, want = dx.cpu().numpy(), dx64 + (old if accumulate else 0)
            assert np.array_equal(np.isfinite(got), hit == 0) and np.array_equal(got[hit == 0], want[hit == 0]), (at, accumulate)


@pytest.mark.parametrize("H,W,pad", [(0, 0, 3), (0, 0, 2), (0, 5, 2), (3, 0, 2)])
def test_an_empty_plane_is_all_padding(nz, H, W, pad):
    """y is the bias (here nothing), not what a copy of the same size left in the workspace; dw gets nothing."""
    import torch
    N, C, O, K = 2, 16, 24, 3
    lib, stream = nz.load(), torch.cuda.current_stream().cuda_stream
    Ho, Wo = H + 2 * pad - K + 1, W + 2 * pad - K + 1
    w = torch.ones(1, 1, C * K * K, O, device="cuda")
    nz.conv2d_forward(torch.ones(N, C, H + 2 * pad, W + 2 * pad, device="cuda"), w, None, K, K, 1, 0)
    y, dw, one = torch.full((N, O, Ho, Wo), 7.0, device="cuda"), torch.full_like(w, 3.0), torch.ones(64, device="cuda")
    nz.check(lib.nzhip_conv2d_forward(y.data_ptr(), one.data_ptr(), w.data_ptr(), None, N, C, H, W, O, K, K, 1, pad, 1, 0, 1, 0, stream))
    assert bool((y == 0).all())
    nz.check(lib.nzhip_conv2d_backward_weights(dw.data_ptr(), one.data_ptr(), y.data_ptr(), N, C, H, W, O, K, K, 1, pad, 1, stream))
    assert bool((dw == 3).all())


# N, C, H, W, O, K, stride, pad, copies: short sums, sums of 64 parts, strided gradients of many short sums, long sums
PRECISION = [(8, 13, 16, 16, 128, 7, 2, 3, 1), (1, 32, 23, 23, 15, 5, 1, 2, 1), (8, 8, 48, 48, 8, 7, 2, 3, 8), (4, 16, 32, 32, 16, 3, 1, 1, 1), (4, 32, 48, 48, 33, 3, 2, 1, 4),
             (16, 16, 30, 30, 113, 7, 2, 3, 1), (4, 160, 65, 65, 16, 3, 2, 1, 1), (16, 272, 17, 17, 99, 5, 1, 2, 16), (16, 256, 14, 14, 256, 3, 1, 1, 1)]


@pytest.mark.parametrize("layer", PRECISION)
def test_sums_are_as_exact_as_those_of_the_kernels_that_round_as_they_stage(nz, monkeypatch, layer):
    """Error in the 2-norm against float64 on operands that fp16 holds exactly, so that only the order of the fp32 sums counts."""
    import torch
    N, C, H, W, O, K, stride, pad, copies = layer
    rng = np.random.default_rng(7)
    Ho, Wo = (H + 2 * pad - K) // stride + 1, (W + 2 * pad - K) // stride + 1
    x, w, dy = (rng.standard_normal(s).astype(np.float16).astype(np.float32) for s in ((N, C, H, W), (copies, 1, C * K * K, O), (N, O, Ho, Wo)))
    want = reference(x, w, dy, K, K, stride, pad)
    X, Wt, DY = (torch.from_numpy(a).cuda() for a in (x, w, dy))
    err = {}
    for route in ("0", "1"):
        monkeypatch.setenv("NZHIP_CONV_CL", route)
        dw = torch.zeros(w.shape, device="cuda")
        nz.conv2d_backward_weights(dw, X, DY, K, K, stride, pad)
        dx = nz.conv2d_backward_data(torch.empty(x.shape, device="cuda"), DY, Wt, K, K, stride, pad, accumulate=False)
        got = nz.conv2d_forward(X, Wt, None, K, K, stride, pad), dx, dw
        err[route] = [np.linalg.norm(g.cpu().numpy() - r) / np.linalg.norm(r) for g, r in zip(got, want)]
    for name, before, now in zip(("y", "dx", "dw"), err["0"], err["1"]):
        assert now <= 1.05 * before, (name, before, now)              # (the 2-norm over thousands of elements moves by a few hundredths with their order)


@pytest.mark.parametrize("layer", [(16, 256, 14, 14, 256, 3, 1, 1, 1), (2, 208, 16, 16, 144, 5, 1, 2, 2), (4, 64, 48, 48, 45, 7, 2, 3, 1),
                                   (1, 16, 192, 96, 24, 3, 2, 1, 1)])
def test_chosen_plans_are_bit_exact_on_whole_numbers(nz, layer):
    import torch
    N, C, H, W, O, K, stride, pad, copies = layer
    rng = np.random.default_rng(sum(layer))
    Ho, Wo = (H + 2 * pad - K) // stride + 1, (W + 2 * pad - K) // stride + 1
    x, w, dy = whole(rng, N, C, H, W), whole(rng, copies, 1, C * K * K, O), whole(rng, N, O, Ho, Wo)
    y64, dx64, dw64 = reference(x, w, dy, K, K, stride, pad)
    cu = lambda a: torch.from_numpy(a).cuda()
    handle, weights = nz.Prepared(), cu(w)
    for _ in range(2):                                                # the second time on the kept copy of the weights
        y = nz.conv2d_forward(cu(x), weights, None, K, K, stride, pad, prepared_w=handle)
        assert np.array_equal(y.cpu().numpy(), y64)
    dx = nz.conv2d_backward_data(torch.empty(x.shape, device="cuda"), cu(dy), cu(w), K, K, stride, pad, accumulate=False)
    assert np.array_equal(dx.cpu().numpy(), dx64)
    dw = torch.zeros(w.shape, device="cuda")
    nz.conv2d_backward_weights(dw, cu(x), cu(dy), K, K, stride, pad)
    assert np.array_equal(dw.cpu().numpy(), dw64)


# direction, layer (N, C, H, W, O, K, stride, pad, copies), a bias per pixel, whether the kernels on copies are the faster ones
CHOICES = [
    ("weights", (16, 128, 56, 56, 112, 3, 1, 1, 1), False, False), ("weights", (16, 128, 56, 56, 128, 3, 1, 1, 1), False, False),
    ("weights", (16, 128, 56, 56, 64, 3, 1, 1, 1), False, True), ("weights", (16, 128, 56, 56, 136, 3, 1, 1, 1), False, True),
    ("weights", (8, 15, 96, 96, 242, 3, 1, 1, 1), False, False), ("weights", (32, 6, 48, 48, 160, 3, 1, 1, 1), False, True),
    ("weights", (16, 6, 32, 180, 192, 5, 1, 2, 16), False, False), ("weights", (16, 7, 32, 32, 128, 5, 1, 2, 1), False, True),
    ("weights", (16, 7, 64, 64, 84, 3, 2, 1, 16), False, False), ("weights", (16, 6, 32, 32, 225, 3, 2, 1, 16), False, True),
    ("forward", (8, 128, 64, 64, 64, 3, 1, 1, 1), False, False), ("forward", (8, 128, 64, 64, 64, 3, 1, 1, 1), True, True),
    ("forward", (10, 64, 32, 32, 60, 3, 1, 1, 1), False, True),
    ("forward", (16, 4, 12, 12, 425, 5, 1, 2, 16), False, False), ("forward", (16, 5, 16, 16, 403, 5, 1, 2, 16), False, True),
    ("forward", (16, 4, 176, 176, 64, 3, 1, 1, 16), False, False), ("forward", (10, 4, 160, 160, 192, 3, 1, 1, 10), False, True),
    ("forward", (16, 352, 64, 64, 128, 3, 1, 1, 1), False, False), ("forward", (10, 287, 128, 128, 32, 3, 1, 1, 1), False, True),
    ("data", (16, 212, 64, 64, 208, 3, 1, 1, 16), False, False), ("data", (16, 352, 64, 64, 128, 3, 1, 1, 1), False, True),
    ("data", (8, 480, 80, 80, 32, 3, 2, 1, 1), False, True), ("data", (10, 48, 144, 144, 5, 3, 2, 1, 10), False, True), ("data", (32, 3, 144, 144, 27, 3, 2, 1, 1), False, False),
]


@pytest.mark.parametrize("direction,layer,pixel_bias,copies", CHOICES)
def test_layers_take_the_faster_kernels(nz, monkeypatch, direction, layer, pixel_bias, copies):
    """Told apart by their bits: the kernels leave a chain of sums at other places."""
    import torch
    N, C, H, W, O, K, stride, pad, w_copies = layer
    g = torch.Generator(device="cuda").manual_seed(sum(layer))
    normal = lambda *s: torch.randn(s, device="cuda", generator=g)
    Ho, Wo = (H + 2 * pad - K) // stride + 1, (W + 2 * pad - K) // stride + 1
    x, w, dy = normal(N, C, H, W), normal(w_copies, 1, C * K * K, O), normal(N, O, Ho, Wo)
    b, strides = (normal(1, 1, Ho * Wo, O), (O, 1)) if pixel_bias else (normal(O), (0, 1))

    def result(route):
        monkeypatch.setenv("NZHIP_CONV_CL", route) if route else monkeypatch.delenv("NZHIP_CONV_CL")
        if direction == "forward": return nz.conv2d_forward(x, w, b, K, K, stride, pad, bias_strides=strides)
        if direction == "data": return nz.conv2d_backward_data(torch.empty_like(x), dy, w, K, K, stride, pad, accumulate=False)
        return nz.conv2d_backward_weights(torch.zeros_like(w), x, dy, K, K, stride, pad)

    on_copies, other, chosen = result("1"), result("0"), result(None)
    assert torch.equal(on_copies, chosen) == copies and torch.equal(other, chosen) == (not copies)


PLANS = r"""
import sys, torch
from neuzephyr_amd import capi
for line in sys.stdin:
    n, C, H, O, K, copies = (int(v) for v in line.split())
    Ho = (H + 2 * (K // 2) - K) // 2 + 1
    print("layer", file=sys.stderr, flush=True)
    capi.conv2d_backward_data(torch.zeros(n, C, H, H, device="cuda"), torch.zeros(n, O, Ho, Ho, device="cuda"), torch.zeros(copies, 1, C * K * K, O, device="cuda"), K, K, 2, K // 2)
"""


def test_plans_of_columns_in_pairs_are_what_is_launched():
    """The parts that the estimate was for, in layers whose two sums differ in length; and not on 128 x 64 tiles, on which pairs are slow."""
    import os
    import re
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    env = {k: v for k, v in os.environ.items() if not k.startswith("NZHIP_")}
    layers = [(1, 233, 25, 352, 5, 1), (8, 32, 80, 480, 7, 1), (32, 13, 44, 288, 7, 1), (4, 256, 16, 288, 5, 1), (16, 352, 26, 38, 7, 16)]
    p = subprocess.run([sys.executable, "-c", PLANS], input="\n".join(" ".join(map(str, v)) for v in layers), capture_output=True, text=True, timeout=100, cwd=root,
                       env={**env, "NZHIP_TRACE": "1", "NZHIP_CONV_CL": "1", "NZHIP_CONV_CL_PAIRED": "1", "PYTHONPATH": root})
    assert p.returncode == 0, p.stderr[-2000:]
    plans = re.findall(r"channel-last copies, tile (\d), (\d+) part\(s\), planned (\d+), columns in pairs", p.stderr)
    assert len(plans) == len(layers)
    assert all(parts == planned for _, parts, planned in plans), plans
    assert max(int(parts) for _, parts, _ in plans) > 1 and plans[-1][0] != "2", plans
