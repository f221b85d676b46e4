"""Grouped row copies: single columns (256 rows a block), rows in 16-byte loads
around three of them per lane (768 columns), rows whose length, stride or start
does not allow those, sets without an index, more sets than one launch takes,
gather and scatter, FP32 and BF16 outputs.  Copies and roundings are exact."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scatter", [0, 1])
@pytest.mark.parametrize("M,cols,pad,shift", [(1, 1, 0, 0), (257, 1, 2, 0), (5, 4, 0, 0),
                                              (6, 768, 16, 0), (7, 772, 4, 0), (3, 1540, 0, 0),
                                              (9, 768, 1, 0), (4, 766, 2, 0), (8, 64, 8, 1)])
def test_row_sets(cuda, M, cols, pad, shift, scatter):
    from tensormol_amd import _lib as TL
    lib = TL.lib()
    g = torch.Generator().manual_seed(M + cols)
    ld, rows = cols + pad, 2 * M + 3
    keep, sets, checks = [], [], []
    for k in range(40):
        half, mapped = k % 2, k % 4 < 2
        src = torch.randn(rows, ld, generator=g).to(cuda)
        out = torch.full((rows * ld + 8,), 9.0, device=cuda,
                         dtype=torch.bfloat16 if half else torch.float32)
        idx = torch.randperm(rows, generator=g)[:M].to(torch.int32).to(cuda)
        m = 0 if k == 5 else M
        keep += [src, out, idx]
        first = src.view(-1)[shift:]
        sets.append(TL.RowsGroup(m, cols - (shift if cols > 1 else 0),
                                 idx.data_ptr() if mapped else None, first.data_ptr(), ld,
                                 out.data_ptr(), ld, half))
        checks.append((m, cols - (shift if cols > 1 else 0), idx.long() if mapped else
                       torch.arange(M, device=cuda), src, out))
    arr = (TL.RowsGroup * len(sets))(*sets)
    lib.tm_rows_grouped(len(sets), ctypes.cast(arr, ctypes.c_void_p), scatter,
                        torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    for m, c, at, src, out in checks:
        ref = torch.full_like(out, 9.0)
        view = ref[:rows * ld].view(rows, ld)
        if m:
            val = (src[:M] if scatter else src[at])[:, shift:shift + c].to(out.dtype)
            view[at if scatter else torch.arange(M, device=cuda), :c] = val
        assert torch.equal(out, ref)
