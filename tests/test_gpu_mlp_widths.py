"""MFMA MLP kernel at widths and row counts where its tiling can go wrong:
descriptor lengths and hidden widths that are odd multiples of 64 (the short
weight ring, a half descriptor chunk), waves without features of their own, and
segments that end inside a tile.

A network and the same network padded with zero weights to widths that are
multiples of 128 (the sizes test_gpu_mlp.py compares with FP32 torch) have the
same products in the same order plus exact zeros, so their outputs are equal
bit for bit, as are those of 64-row and 32-row tiles."""
from types import SimpleNamespace

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _run(device, D, H, nets, G, counts, precision, ncu):
    """(y [2, N], dG [2, N, D]) of the element networks `nets` (per net and
    element) on rows that are element-sorted already."""
    from tensormol_amd import _lib
    from tensormol_amd.mlp_mfma import MFMAWeights
    eles = list(range(len(counts)))
    model = SimpleNamespace(sym=SimpleNamespace(D=D), hidden=[H] * 3, eles=eles, alpha=1.0,
                            energy_nets=nets[0], charge_nets=nets[1])
    eng = SimpleNamespace(model=model, device=device, lib=_lib.lib(), nele=len(eles),
                          _stream=lambda: _lib.P(torch.cuda.current_stream().cuda_stream))
    w = MFMAWeights(eng, precision)
    w.ncu = ncu
    N = sum(counts)
    ws = SimpleNamespace(N=N, G=G, eoff=np.concatenate([[0], np.cumsum(counts)]),
                         perm=torch.arange(N, dtype=torch.int32, device=device),
                         Y2=torch.zeros(2 * N, device=device),
                         J2=torch.zeros(2 * N * D, device=device))
    ws.mlp_ws = w.workspace(ws)
    w.run(ws)
    torch.cuda.synchronize()
    return ws.Y2.view(2, N), ws.J2.view(2, N, D), ws.mlp_ws["n64"]


def _pad(nets, D, H, Dp, Hp):
    sizes, psizes = [D, H, H, H, 1], [Dp, Hp, Hp, Hp, 1]
    out = {}
    for e, layers in nets.items():
        out[e] = []
        for k, (W, b) in enumerate(layers):
            Wp, bp = np.zeros((psizes[k], psizes[k + 1])), np.zeros(psizes[k + 1])
            Wp[:sizes[k], :sizes[k + 1]] = W
            bp[:sizes[k + 1]] = b
            out[e].append((Wp, bp))
    return out


@pytest.mark.parametrize("precision", ["bf16", "fp16", "bf16x2", "fp16x2", "bf16x3f", "bf16x3"])
@pytest.mark.parametrize("D,H", [(256, 64), (64, 320), (320, 512), (192, 448), (832, 64)])
def test_widths(cuda, precision, D, H):
    rng = np.random.default_rng(D + H)
    counts = [161, 65, 1]   # 2 * 64 + 33 rows, 64 + 1, one
    sizes = [D, H, H, H, 1]
    nets = [{e: [(rng.normal(size=(a, b)) / np.sqrt(a), 0.1 * rng.normal(size=b))
                 for a, b in zip(sizes[:-1], sizes[1:])] for e in range(3)} for _ in range(2)]
    G = torch.tensor(rng.uniform(0.0, 1.0, (sum(counts), D)), dtype=torch.float32, device=cuda)
    y, dG, _ = _run(cuda, D, H, nets, G, counts, precision, 1 << 20)      # 32-row tiles only
    y2, dG2, n64 = _run(cuda, D, H, nets, G, counts, precision, 2)         # and 64-row tiles
    assert n64 > 0 or precision == "bf16x3"
    assert torch.equal(y, y2) and torch.equal(dG, dG2)
    Dp, Hp = -(-D // 128) * 128, -(-H // 128) * 128
    Gp = torch.zeros(sum(counts), Dp, device=cuda)
    Gp[:, :D] = G
    yp, dGp, _ = _run(cuda, Dp, Hp, [_pad(n, D, H, Dp, Hp) for n in nets], Gp, counts, precision, 2)
    assert torch.equal(y, yp) and torch.equal(dG, dGp[:, :, :D])
    assert y.abs().max() > 0 and dG.abs().max() > 0
