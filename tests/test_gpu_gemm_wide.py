"""The GEMM of BF16 operands in 16-byte layouts against the element-wise one.

Operands stored as FP32 holding BF16 values take the element-wise kernel, the
same values stored as BF16 the wide one; both round nothing, multiply the same
pairs in the same order of k, and so must give the same bits in every output.
Sizes: around the edges of a 64- or 128-row tile, of a 64-deep K step, of the
chunks inside one, single rows and columns, K splits that leave parts empty,
and enough rows for the larger tile.  Nothing may be written outside [M, N]."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


def _run(lib, TL, A, B, M, N, K, lda, ldb, ldc, ta, tb, epi, ns, crow, extra, bf):
    dev = A.device
    nan = float("nan")
    outs = [torch.full((M, ldc), nan, device=dev) for _ in range(3)]
    work = torch.full((ns * M * ldc,), nan, device=dev) if ns > 1 else None
    p = lambda t: None if t is None else t.data_ptr()
    f = dict(M=M, N=N, K=K, A=p(A), lda=lda, B=p(B), ldb=ldb, C=p(outs[0]), ldc=ldc, work=p(work),
             crow=p(crow))
    bias, w4, s, x1, x2, ym = extra
    if epi == 1:
        f.update(bias=p(bias), aux=p(outs[1]), x1=p(w4), out2=p(outs[2]))
    elif epi == 2:
        f.update(s=p(s), aux=p(outs[1]), x1=p(w4), x2=p(ym), out2=p(outs[2]))
    elif epi == 3:
        f.update(s=p(s), x1=p(x1), x2=p(x2))
    elif ns == 1:
        f.update(bias=p(bias))
    arr = (TL.GemmGroup * 1)(TL.GemmGroup(**f))
    lib.tm_gemm_bf16_grouped(1, ctypes.cast(arr, ctypes.c_void_p), ta, tb, epi, int(bf), 1.5, ns,
                             torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    return outs


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("M,N,K,ns", [(1, 4, 8, 1), (63, 128, 64, 1), (64, 132, 56, 1),
                                      (65, 260, 72, 1), (129, 64, 200, 1), (127, 1, 136, 1),
                                      (130, 3, 520, 1), (131100, 128, 72, 1), (129, 36, 2056, 5),
                                      (513, 1, 1032, 8), (40, 516, 64, 6), (17, 8, 0, 1)])
def test_wide_gemm_equals_elementwise(cuda, ta, tb, M, N, K, ns):
    from tensormol_amd import _lib as TL
    lib = TL.lib()
    g = torch.Generator().manual_seed(M + 3 * N + 7 * K)
    up = lambda n: (n + 7) // 8 * 8 + 8

    def operand(rows, cols, trans):   # stored [cols, ld] when transposed, else [rows, ld]
        r, c = (cols, rows) if trans else (rows, cols)
        ld = 1 if trans and rows == 1 else up(c)
        X = (0.3 * torch.randn(max(r, 1), ld, generator=g)).to(cuda).bfloat16()
        return X, X.float(), ld

    A16, A32, lda = operand(M, K, ta)
    B16, B32, ldb = operand(N, K, not tb)
    ldc = (N + 3) // 4 * 4 + 4
    rnd = lambda *s: torch.randn(*s, generator=g).to(cuda)
    extra = (rnd(N), rnd(N), torch.rand(M, ldc, generator=g).to(cuda), rnd(M, ldc), rnd(M, ldc),
             rnd(M))
    for epi in ((0,) if ns > 1 else (0, 1, 2, 3)):
        args = (M, N, K, lda, ldb, ldc, ta, tb, epi, ns)
        crow = None
        if epi == 0 and ns == 1 and M > 1:
            crow = torch.randperm(M, generator=g).to(torch.int32).to(cuda)
        ref = _run(lib, TL, A32, B32, *args, crow, extra, False)
        out = _run(lib, TL, A16, B16, *args, crow, extra, True)
        for r, o in zip(ref, out):
            assert torch.equal(r.nan_to_num(7.25e9), o.nan_to_num(7.25e9)), epi
            assert o[:, N:].isnan().all()
        assert not out[0][:, :N].isnan().any()
