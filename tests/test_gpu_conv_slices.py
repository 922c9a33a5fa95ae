"""The one-launch convolutions of few tiles (nzhip_conv_slices.hip), forward and data gradient, against float64 convolutions of whole numbers, bit for
bit, in both workgroup shapes. The library reads NZHIP_CONV_SLICES per call: 0 never, 1 and 2 one of the shapes wherever it fits."""
import numpy as np
import pytest

from test_gpu_conv_cl import LAYERS, embedded, nz, reference, untouched, whole  # noqa: F401

pytestmark = pytest.mark.gpu

# one unit of 16 channels; an odd number of units; more chunks than waves; outputs and channels just past a tile; 1x1 at strides
MORE = [(2, 16, 6, 6, 32, 1, 1, 1, 0, 1), (1, 17, 8, 4, 33, 3, 3, 1, 1, 1), (3, 5, 20, 19, 40, 1, 1, 2, 0, 3), (1, 200, 7, 7, 31, 3, 3, 1, 1, 1), (2, 30, 16, 16, 4, 7, 7, 2, 3, 2)]


@pytest.mark.parametrize("layer", LAYERS + MORE)
@pytest.mark.parametrize("shape", [1, 2])
def test_bit_exact_on_whole_numbers(nz, monkeypatch, shape, layer):  # noqa: F811
    import torch
    N, C, H, W, O, K_h, K_w, stride, pad, copies = layer
    rng = np.random.default_rng(sum(layer) + shape)
    Ho, Wo = (H + 2 * pad - K_h) // stride + 1, (W + 2 * pad - K_w) // stride + 1
    x, w, dy = whole(rng, N, C, H, W), whole(rng, copies, 1, C * K_h * K_w, O), whole(rng, N, O, Ho, Wo)
    b, old_dx = whole(rng, 1, 1, Ho * Wo, O), whole(rng, *x.shape)
    y64, dx64, _ = reference(x, w, dy, K_h, K_w, stride, pad)
    bias = b.reshape(Ho * Wo, O).T.reshape(1, O, Ho, Wo)
    monkeypatch.setenv("NZHIP_CONV_SLICES", str(shape))
    X, Wt, DY, B = embedded(x)[1], embedded(w)[1], embedded(dy)[1], embedded(b)[1]
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


@pytest.mark.parametrize("special", [float("inf"), float("nan"), -7e4])            # -7e4 is infinite in fp16
@pytest.mark.parametrize("shape", [1, 2])
@pytest.mark.parametrize("K,stride,pad,copies", [(3, 2, 1, 1), (3, 1, 1, 2), (5, 2, 2, 1), (1, 2, 0, 1)])
def test_a_special_value_stays_in_the_sums_it_is_a_term_of(nz, monkeypatch, special, shape, K, stride, pad, copies):  # noqa: F811
    """Channels that fill a unit up and taps outside dy (also between the pixels of a stride) are no terms, whatever they are multiplied with."""
    import torch
    N, C, H, W, O = 2, 35, 11, 10, 20
    rng = np.random.default_rng(6)
    Ho, Wo = (H + 2 * pad - K) // stride + 1, (W + 2 * pad - K) // stride + 1
    x, dy = rng.integers(1, 3, (N, C, H, W)).astype(np.float32), rng.integers(1, 3, (N, O, Ho, Wo)).astype(np.float32)
    w = rng.integers(1, 3, (copies, 1, C * K * K, O)).astype(np.float32)
    y64, dx64, _ = reference(x, w, dy, K, K, stride, pad)
    monkeypatch.setenv("NZHIP_CONV_SLICES", str(shape))
    cu = lambda a: torch.from_numpy(a.copy()).cuda()
    dx_of = lambda dy_, w_: nz.conv2d_backward_data(torch.empty(x.shape, device="cuda"), cu(dy_), cu(w_), K, K, stride, pad, accumulate=False).cpu().numpy()

    def marked(a, at):
        b, mark = a.copy(), np.zeros_like(a)
        b[at], mark[at] = special, 1
        return b, mark

    xs, mark = marked(x, (1, C - 1, (Ho - 1) * stride - pad + (pad if K > 1 else 0), (Wo - 1) * stride - pad + (pad if K > 1 else 0)))
    hit, _, _ = reference(mark, w, dy, K, K, stride, pad)
    got = nz.conv2d_forward(cu(xs), cu(w), None, K, K, stride, pad).cpu().numpy()
    assert (hit != 0).any() and np.array_equal(np.isfinite(got), hit == 0) and np.array_equal(got[hit == 0], y64[hit == 0])
    dys, mark = marked(dy, (1, O - 1, Ho - 1, Wo - 1))
    _, hit, _ = reference(x, w, mark, K, K, stride, pad)
    got = dx_of(dys, w)
    assert np.array_equal(np.isfinite(got), hit == 0) and np.array_equal(got[hit == 0], dx64[hit == 0])
    for c, tap, o in ((0, 0, 0), (C - 1, K * K - 1, O - 1), (33, K // 2 * K, 7)):
        ws, mark = marked(w, (copies - 1, 0, c * K * K + tap, o))
        _, hit, _ = reference(x, mark, dy, K, K, stride, pad)
        got = dx_of(dy, ws)
        assert (hit[:, c] == 0).any() and np.array_equal(np.isfinite(got), hit == 0) and np.array_equal(got[hit == 0], dx64[hit == 0]), (c, tap, o)


@pytest.mark.parametrize("layer", [(16, 4, 10, 10, 25, 3, 1, 1, 16), (2, 11, 16, 16, 79, 7, 2, 3, 2), (4, 104, 64, 64, 19, 3, 1, 1, 1), (8, 240, 8, 8, 235, 3, 1, 1, 8), (8, 31, 39, 39, 19, 3, 2, 1, 8)])
def test_sums_are_as_exact_as_those_of_the_other_kernels(nz, monkeypatch, layer):  # noqa: F811
    """Error in the 2-norm against float64 on operands that fp16 holds exactly, so that only the order of the fp32 sums counts."""
    import torch
    N, C, H, W, O, K, stride, pad, copies = layer
    rng = np.random.default_rng(7)
    Ho, Wo = (H + 2 * pad - K) // stride + 1, (W + 2 * pad - K) // stride + 1
    x, w, dy = (rng.standard_normal(s).astype(np.float16).astype(np.float32) for s in ((N, C, H, W), (copies, 1, C * K * K, O), (N, O, Ho, Wo)))
    want = reference(x, w, dy, K, K, stride, pad)[:2]
    X, Wt, DY = (torch.from_numpy(a).cuda() for a in (x, w, dy))
    err = {}
    for route in ("0", "2"):
        monkeypatch.setenv("NZHIP_CONV_SLICES", route)
        got = nz.conv2d_forward(X, Wt, None, K, K, stride, pad), nz.conv2d_backward_data(torch.empty(x.shape, device="cuda"), DY, Wt, K, K, stride, pad, accumulate=False)
        err[route] = [np.linalg.norm(g.cpu().numpy() - r) / np.linalg.norm(r) for g, r in zip(got, want)]
    for name, before, now in zip(("y", "dx"), err["0"], err["2"]):
        assert now <= 1.05 * before, (name, before, now)              # (the 2-norm over thousands of elements moves by a few hundredths with their order)


# n, C, H, O, K, stride, weight copies, bias per pixel: layers that other ways compute in less time, and neighbours on which this one does
RULE = [((16, 112, 16, 283, 3, 2, 1, False), False), ((2, 3, 107, 318, 3, 2, 1, True), False), ((32, 7, 11, 336, 3, 1, 1, True), False), ((16, 40, 16, 283, 3, 2, 1, False), True),
        ((10, 48, 7, 384, 5, 1, 10, True), True), ((8, 3, 90, 24, 3, 1, 1, False), True), ((4, 112, 48, 237, 1, 1, 4, True), True)]


@pytest.mark.parametrize("layer,taken", RULE)
def test_which_forwards_run_on_it(nz, monkeypatch, layer, taken):  # noqa: F811
    """Told by the bits: the sums of the ways are in different order."""
    import torch
    N, C, H, O, K, stride, copies, pixel = layer
    Ho = (H + 2 * (K // 2) - K) // stride + 1
    g = torch.Generator().manual_seed(sum(layer))
    x, w, b = (torch.randn(*s, generator=g).cuda() for s in ((N, C, H, H), (copies, 1, C * K * K, O), (1, 1, Ho * Ho, O)))
    run = lambda: nz.conv2d_forward(x, w, b, K, K, stride, K // 2, bias_strides=(O if pixel else 0, 1))
    got = run()
    monkeypatch.setenv("NZHIP_CONV_SLICES", "0")
    other = run()
    monkeypatch.setenv("NZHIP_CONV_SLICES", "1")
    here = [run()]
    monkeypatch.setenv("NZHIP_CONV_SLICES", "2")
    here.append(run())
    assert not any(torch.equal(other, h) for h in here)
    assert any(torch.equal(got, h) for h in here) if taken else torch.equal(got, other)


@pytest.mark.parametrize("layer,taken", [((16, 96, 16, 4, 7, 1, 1), False), ((4, 223, 27, 4, 5, 1, 1), False), ((16, 40, 16, 4, 7, 1, 1), True), ((4, 100, 27, 40, 3, 1, 1), True)])
def test_which_gradients_run_on_it(nz, monkeypatch, layer, taken):  # noqa: F811
    import torch
    N, C, H, O, K, stride, copies = layer
    g = torch.Generator().manual_seed(sum(layer))
    dy, w = (torch.randn(*s, generator=g).cuda() for s in ((N, O, H, H), (copies, 1, C * K * K, O)))
    run = lambda: nz.conv2d_backward_data(torch.empty(N, C, H, H, device="cuda"), dy, w, K, K, stride, K // 2, accumulate=False)
    got = run()
    monkeypatch.setenv("NZHIP_CONV_SLICES", "0")
    other = run()
    monkeypatch.setenv("NZHIP_CONV_SLICES", "1")
    here = [run()]
    monkeypatch.setenv("NZHIP_CONV_SLICES", "2")
    here.append(run())
    assert not any(torch.equal(other, h) for h in here)
    assert any(torch.equal(got, h) for h in here) if taken else torch.equal(got, other)
