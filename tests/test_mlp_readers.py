"""Weight readers in the MLP tile tables: one per XCD and weight blob where
tiles and readers have a CU each, none past that, and the same results."""
import numpy as np
import pytest
import torch

from tensormol_amd.mlp_mfma import NXCD, with_readers, xcd_order


def _tiles(counts):
    return np.array([(s, 32 * t) for s, n in enumerate(counts) for t in range(n)],
                    dtype=np.int32).reshape(-1, 2)


@pytest.mark.parametrize("counts", [[], [1], [1, 1], [3, 1, 2], [1] * 8, [20, 1, 7, 30], [31] * 8,
                                    [120, 120], [128, 128], [250], [9, 300]])
def test_with_readers(counts):
    til = xcd_order(_tiles(counts))
    out = with_readers(til, 256)
    np.testing.assert_array_equal(out[:len(til)], til)
    extra = out[len(til):]
    assert len(out) % NXCD == 0 and out.dtype == np.int32
    assert not len(extra) or len(out) <= 256
    need = [sorted({int(s) for s in til[x::NXCD, 0] if s >= 0}) for x in range(NXCD)]
    if not len(extra):
        assert not len(til) or len(til) + NXCD * max(map(len, need)) > 256
        return
    for x in range(NXCD):
        have = [-2 - int(s) for s in extra[x::NXCD, 0] if s < -1]
        assert sorted(have) == need[x]


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["bf16x3f", "bf16x3", "bf16", "fp16"])
@pytest.mark.parametrize("eles,natom", [([1, 8], 1), ([1, 8], 70), ([1, 6, 7, 8], 333)])
def test_readers_change_nothing(cuda, eles, natom, precision, monkeypatch):
    from tensormol_amd import mlp_mfma
    from tensormol_amd.engine import BPEEEngine
    from tensormol_amd.model import BPEEModel
    rng = np.random.default_rng(natom)
    Z = rng.choice(eles, natom)
    eng = BPEEEngine(BPEEModel(eles, hidden=[192] * 3), precision=precision)
    out = []
    for readers in (True, False):
        if not readers:
            monkeypatch.setattr(mlp_mfma, "with_readers", lambda til, ncu: til)
        ws = eng.prepare(Z, np.array([0, natom]), pos0=rng.normal(size=(natom, 3)))
        g = np.random.default_rng(1).uniform(0, 1, (natom, eng.D))
        ws.G.copy_(torch.tensor(g, dtype=torch.float32))
        ws.Y2.fill_(float("nan"))
        ws.J2.fill_(float("nan"))
        eng.networks(ws)
        torch.cuda.synchronize()
        out.append((ws.mlp_ws["n32"], ws.Y2.clone(), ws.J2.clone()))
    assert out[0][0] > out[1][0]
    for a, b in zip(out[0][1:], out[1][1:]):
        assert not torch.isnan(b).any() and torch.equal(a, b)
