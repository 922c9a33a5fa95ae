"""The kernel for products of few tiles (nzhip_gemm_slices.hip) at the edges of its tiles, chunks and rules: exact on integers, nothing read or
written outside the operands' rows, errors no larger than those of the kernels that take the same products otherwise. The library reads
NZHIP_GEMM_SLICES per call: 0 never, 1 to 3 one of its workgroup shapes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def nz():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from neuzephyr_amd import capi
    capi.load()
    return capi


# M, K, N: one row and column; the tiles' edges; chunks of 32 k cut anywhere; fewer chunks than waves, and more
SIZES = [(1, 4, 1), (1, 33, 70), (33, 5, 2), (31, 31, 33), (32, 32, 32), (64, 64, 65), (65, 127, 63), (70, 130, 2), (3, 259, 129), (128, 1029, 96)]


@pytest.mark.parametrize("shape", [1, 2, 3])
@pytest.mark.parametrize("a_trans", [False, True])
@pytest.mark.parametrize("b_trans", [False, True])
@pytest.mark.parametrize("size", SIZES)
def test_exact_on_integers_inside_larger_buffers(nz, monkeypatch, size, a_trans, b_trans, shape):
    """Rows of odd length and offset inside buffers of NaN: what lies between the rows or past them must enter no sum."""
    import torch
    monkeypatch.setenv("NZHIP_GEMM_SLICES", str(shape))
    M, K, N = size
    rng = np.random.default_rng(M * 31 + K * 7 + N)
    A, B, bias = (rng.integers(-3, 4, s).astype(np.float32) for s in ((M, K), (K, N), (M, N)))
    want = (A.astype(np.int64) @ B.astype(np.int64)).astype(np.float32)

    def embed(x, slack, offset):
        rows, cols = x.shape
        buf = torch.full((offset + rows * (cols + slack) + 3,), float("nan"), device="cuda")
        view = buf[offset:offset + rows * (cols + slack)].view(rows, cols + slack)[:, :cols]
        view.copy_(torch.from_numpy(np.ascontiguousarray(x)))
        return buf, view

    import ctypes as C
    keep = [embed(A.T if a_trans else A, 1, 1), embed(B.T if b_trans else B, 2, 3), embed(np.full((M, N), 9, np.float32), 3, 2), embed(bias, 0, 1)]
    (_, a), (_, b), (cbuf, c), (_, bv) = keep
    for form in ("none", "bias, ReLU", "column bias", "added to"):
        cbuf.fill_(float("nan"))
        c.fill_(4.0)
        d = nz.GemmDesc(A=a.data_ptr(), B=b.data_ptr(), C=c.data_ptr(), M=M, N=N, K=K, lda=a.stride(0), ldb=b.stride(0), ldc=c.stride(0),
                        a_layout=int(a_trans), b_layout=int(b_trans), batch_n=1, batch_c=1)
        expect = want
        if form == "bias, ReLU":
            d.bias, d.bias_stride_row, d.bias_stride_col, d.activation = bv.data_ptr(), bv.stride(0), 1, 1
            expect = np.maximum(want + bias, 0)
        elif form == "column bias":
            d.bias, d.bias_stride_row, d.bias_stride_col = bv.data_ptr(), 0, 1
            expect = want + bias[:1]
        elif form == "added to":
            d.bias, d.bias_stride_row, d.bias_stride_col = c.data_ptr(), c.stride(0), 1
            expect = want + 4
        nz.check(nz.load().nzhip_gemm(C.byref(d), torch.cuda.current_stream().cuda_stream))
        assert np.array_equal(c.cpu().numpy(), expect), form
        c.fill_(float("nan"))
        assert bool(torch.isnan(cbuf).all()), form


@pytest.mark.parametrize("shape", [1, 2, 3])
@pytest.mark.parametrize("sa,sb", [((3, 2, 40, 70), (3, 2, 70, 50)), ((1, 4, 33, 36), (5, 1, 36, 65)), ((4, 1, 64, 64), (1, 1, 64, 32))])
def test_batches_with_broadcasts(nz, monkeypatch, sa, sb, shape):
    import torch
    monkeypatch.setenv("NZHIP_GEMM_SLICES", str(shape))
    rng = np.random.default_rng(3)
    A, B = (rng.integers(-3, 4, s).astype(np.float32) for s in (sa, sb))
    got = nz.tensorcore_gemm(torch.from_numpy(A).cuda(), torch.from_numpy(B).cuda())
    assert np.array_equal(got.cpu().numpy(), np.matmul(A, B))


def test_infinities_and_nans_stay_in_their_rows_and_columns(nz, monkeypatch):
    """K = 45: the last chunk is filled up with zeros, which must meet no infinity."""
    import torch
    A, B = torch.ones(40, 45, device="cuda"), torch.ones(45, 70, device="cuda")
    A[7, 44], B[44, 11], B[0, 69] = float("inf"), float("nan"), 7e4                      # 7e4 is beyond fp16
    for shape in (1, 2, 3):
        for a_trans in (False, True):
            for b_trans in (False, True):
                monkeypatch.setenv("NZHIP_GEMM_SLICES", str(shape))
                got = nz.gemm(A.T.contiguous() if a_trans else A, B.T.contiguous() if b_trans else B, a_trans=a_trans, b_trans=b_trans)
                want = A.half().float().cpu() @ B.half().float().cpu()
                assert torch.equal(got.cpu().nan_to_num(nan=-1.0), want.nan_to_num(nan=-1.0)), (shape, a_trans, b_trans)


# one-tile and many-tile products, long and short sums, each with the shape that the rule picks
@pytest.mark.parametrize("M,K,N", [(64, 64, 64), (256, 256, 256), (300, 300, 300), (100, 1000, 200), (48, 1943, 112), (16, 1520, 18), (1, 416, 3072), (700, 300, 900), (1024, 1024, 1024)])
@pytest.mark.parametrize("b_trans", [False, True])
def test_sums_are_as_exact_as_those_of_the_other_kernels(nz, monkeypatch, M, K, N, b_trans):
    """Error in the 2-norm against float64 on operands that fp16 holds exactly."""
    import torch
    g = torch.Generator().manual_seed(M + K + N)
    A, B = torch.randn(M, K, generator=g).half().float().cuda(), torch.randn(*((N, K) if b_trans else (K, N)), generator=g).half().float().cuda()
    want = A.double() @ (B.T if b_trans else B).double()
    err = {}
    for route in ("0", None):
        monkeypatch.setenv("NZHIP_GEMM_SLICES", route) if route else monkeypatch.delenv("NZHIP_GEMM_SLICES")
        err[route] = float((nz.gemm(A, B, b_trans=b_trans).double() - want).norm() / want.norm())
    assert err[None] <= 1.05 * err["0"], err                        # (the 2-norm of a few thousand elements moves by a few hundredths with their order)


ROUTES = r"""
import sys, torch
from neuzephyr_amd import capi
for line in sys.stdin:
    M, K, N, at, bt = (int(v) for v in line.split())
    A, B = torch.zeros((K, M) if at else (M, K), device="cuda"), torch.zeros((N, K) if bt else (K, N), device="cuda")
    print("product", file=sys.stderr, flush=True)
    capi.gemm(A, B, a_trans=bool(at), b_trans=bool(bt))
"""

# M, K, N, a_trans, b_trans and the shape: none where the kernels before take less time; 32 x 32 tiles of 4 and 8 waves, 64 x 64
RULE = [((2064, 1136, 1, 1, 1), None), ((2, 1424, 2688, 0, 0), None), ((528, 256, 1, 0, 0), None), ((1, 208, 2, 0, 1), None), ((2, 465, 1, 0, 0), None),
        ((1264, 8, 1, 1, 1), None), ((64, 16, 1, 1, 1), None), ((2, 8, 368, 0, 0), None), ((588, 1441, 1136, 0, 1), None), ((1, 1760, 6000, 0, 0), 1),
        ((1, 100, 300, 0, 1), 0), ((1, 323, 128, 1, 1), 1), ((96, 16, 1, 0, 0), 0), ((378, 352, 2, 0, 1), 1), ((2, 40, 300, 0, 0), 0), ((588, 1200, 1136, 0, 1), 2),
        ((900, 300, 900, 0, 0), 0), ((3056, 421, 304, 0, 1), 2), ((736, 648, 1088, 0, 1), 2), ((1135, 276, 874, 1, 1), 2), ((356, 426, 2167, 0, 0), 2)]


def test_which_products_run_on_it():
    """The lines of its rule: rows and columns that a streaming kernel reads in one launch, a fourth round of small tiles, long sums of large ones."""
    import os
    import re
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    env = {k: v for k, v in os.environ.items() if not k.startswith("NZHIP_")}
    p = subprocess.run([sys.executable, "-c", ROUTES], input="\n".join(" ".join(map(str, s)) for s, _ in RULE), capture_output=True, text=True, timeout=100, cwd=root,
                       env={**env, "NZHIP_TRACE": "1", "PYTHONPATH": root})
    assert p.returncode == 0, p.stderr[-2000:]
    taken = [re.search(r"sliced kernel, shape (\d)", t) for t in p.stderr.split("product\n")[1:]]
    assert [int(t[1]) if t else None for t in taken] == [shape for _, shape in RULE]


# samples, inputs, outputs of a Linear layer, and whether its two gradients take less time as a pair on rounded copies than one after the other
PAIRS = [(201, 1168, 292, True), (457, 3888, 208, True), (562, 1008, 821, True), (1008, 1632, 128, False), (848, 352, 48, False), (736, 134, 8, False)]


@pytest.mark.parametrize("S,I,O,pair", PAIRS)
def test_gradients_of_a_layer_go_the_faster_way(nz, monkeypatch, S, I, O, pair):
    """Told by the bits: the sums of the two ways are in different order."""
    import torch
    g = torch.Generator().manual_seed(S + I + O)
    W, x, dz = (torch.randn(*s, generator=g).cuda() for s in ((1, 1, O, I), (S, 1, I, 1), (S, 1, O, 1)))

    def gradients():
        dW, dx = torch.ones(1, 1, O, I, device="cuda"), torch.ones(S, 1, I, 1, device="cuda")
        nz.matmul_backward(dW, dx, W, x, dz)
        return dW.view(O, I), dx.view(S, I)

    def one_by_one():
        dW, dx = torch.ones(O, I, device="cuda"), torch.ones(S, I, device="cuda")
        nz.gemm(dz.view(S, O), x.view(S, I), a_trans=True, bias=dW, bias_strides=(I, 1), out=dW)
        nz.gemm(dz.view(S, O), W.view(O, I), bias=dx, bias_strides=(I, 1), out=dx)
        return dW, dx

    same = lambda p, q: all(torch.equal(a, b) for a, b in zip(p, q))
    got, apart = gradients(), one_by_one()
    monkeypatch.setenv("NZHIP_GEMM_COPY", "1")
    together = gradients()
    assert not same(apart, together)
    assert same(got, together if pair else apart)
