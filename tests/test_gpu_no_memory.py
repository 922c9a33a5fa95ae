"""Calls whose fp16 copies do not fit the memory that is left take the ways that need less, with their results. Almost all of the device's
memory is held by tensors meanwhile; what is asked for and not there is refused with an error that the library handles."""
import pytest

pytestmark = pytest.mark.gpu

PIECE = 16 << 20                                                     # bytes


def test_calls_without_memory_for_copies_take_the_ways_without_them(monkeypatch):
    import torch
    assert torch.cuda.is_available(), "these tests need the MI355X"
    from neuzephyr_amd import capi as nz
    g = torch.Generator(device="cuda").manual_seed(1)
    normal = lambda *s: torch.randn(s, device="cuda", generator=g)
    N, C, S, O = 8, 64, 256, 64                                      # 68 MB of copies of x, as much of dy
    x, dy, w, y, dx, dw = normal(N, C, S, S), normal(N, O, S, S), normal(1, 1, C * 9, O), normal(N, O, S, S), normal(N, C, S, S), normal(1, 1, C * 9, O)
    A, B, P = normal(100, 100000), normal(100000, 256), normal(100, 256)                             # 71 MB
    W, v, dz, dW, dv = normal(1, 1, 5000, 5000), normal(70, 1, 5000, 1), normal(70, 1, 5000, 1), normal(1, 1, 5000, 5000), normal(70, 1, 5000, 1)      # 50 MB of W
    calls = {"forward": (y, lambda: nz.conv2d_forward(x, w, None, 3, 3, 1, 1, out=y)),
             "data gradient": (dx, lambda: nz.conv2d_backward_data(dx, dy, w, 3, 3, 1, 1, accumulate=False)),
             "weight gradient": (dw, lambda: nz.conv2d_backward_weights(dw.zero_(), x, dy, 3, 3, 1, 1)),
             "product": (P, lambda: nz.gemm(A, B, out=P)),
             "gradients of a layer": (dv, lambda: nz.matmul_backward(dW.zero_(), dv.zero_(), W, v, dz))}

    def results(copies):
        monkeypatch.setenv("NZHIP_CONV_CL", copies)
        monkeypatch.setenv("NZHIP_GEMM_COPY", copies)
        out = {}
        for name, (result, call) in calls.items():
            call()
            out[name] = result.cpu()
        return out

    without, copies = results("0"), results("1")
    torch.cuda.synchronize()
    nz.check(nz.load().nzhip_allocator_trim())
    torch.cuda.empty_cache()
    held = [torch.empty(torch.cuda.mem_get_info()[0] - 4 * PIECE, dtype=torch.uint8, device="cuda")]
    try:
        for _ in range(1000):                                        # until no more is there, whatever is said to be free
            try:
                held.append(torch.empty(PIECE, dtype=torch.uint8, device="cuda"))
            except torch.OutOfMemoryError:
                break
        del held[-2:]                                                # 32 to 48 MB
        torch.cuda.empty_cache()
        starved = results("1")
        torch.cuda.synchronize()
    finally:
        held.clear()
        torch.cuda.empty_cache()
    for name in calls:
        assert torch.equal(starved[name], without[name]) and not torch.equal(starved[name], copies[name]), name
