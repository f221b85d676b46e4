"""Which launches a batch's electrostatics take: charges and sweep in one for
small molecules, separate ones where a batch holds many candidates (its sweep
pays for loading raw charges), and on a cell grid; and that both give the same."""
import numpy as np
import pytest
import torch

from tests import helpers as H


class _Calls:
    def __init__(self):
        self.names = []

    def __getattr__(self, name):
        return lambda *args: self.names.append(name)


@pytest.mark.parametrize("sizes,one", [([1], True), ([256], True), ([8, 0, 256] * 37, True),
                                       ([2000, 2000], True), ([3000, 3000], False),
                                       ([256] * 160, False), ([60] * 2000, False),
                                       ([60] * 100 + [4000], False)])
def test_route(sizes, one, monkeypatch):
    from tensormol_amd.engine import BPEEEngine
    eng = BPEEEngine(H.water_model(), device="cpu", precision="fp32", ldr=2, lda=2)
    N = sum(sizes)
    ws = eng.prepare(np.ones(N, int), np.concatenate([[0], np.cumsum(sizes)]))
    assert not ws.use_cells
    eng.lib = calls = _Calls()
    monkeypatch.setattr(eng, "_raw_stream", lambda: 0)
    monkeypatch.setattr(eng, "_stream", lambda: None)
    eng.electrostatics(ws, torch.zeros(N, 3, dtype=torch.float64))
    head = ["tm_coulomb_raw"] if one else ["tm_mol_sum_f32", "tm_charges", "tm_coulomb"]
    assert calls.names == head + ["tm_mol_sum_f64"]


@pytest.mark.gpu
@pytest.mark.parametrize("sizes,edge", [([2500, 2500], None), ([300] * 110, None), ([2500] * 2, 33.0)])
def test_routes_agree(cuda, sizes, edge):
    """The tolerance is that of the raw sweep's own test: charges may round to
    the neighbouring FP32 value, 2e-7 of the sums of the terms' magnitudes."""
    from tensormol_amd.engine import BPEEEngine
    rng = np.random.default_rng(4)
    N, B = sum(sizes), len(sizes)
    eng = BPEEEngine(H.water_model(), precision="fp32")
    x = rng.uniform(0, 33.0, (N, 3))
    ws = eng.prepare(rng.choice([1, 8], N), np.concatenate([[0], np.cumsum(sizes)]),
                     None if edge is None else np.full((B, 3), edge))
    pos = torch.tensor(x, device=cuda)
    ws.qraw.copy_(torch.tensor(rng.normal(size=N), dtype=torch.float32))
    assert not ws.raw_sweep
    out = []
    for raw in (False, True):
        for n in ("qmean", "q", "qx", "phi", "gradc", "eatom", "phimean", "xq"):
            getattr(ws, n).fill_(float("nan"))
        ws.raw_sweep = raw
        eng.electrostatics(ws, pos)
        torch.cuda.synchronize()
        out.append({n: getattr(ws, n).double().clone()
                    for n in ("qmean", "q", "qx", "phi", "gradc", "eatom", "phimean", "xq")})
    for n, ref in out[0].items():
        assert not ref.isnan().any() and not out[1][n].isnan().any(), n
        bound = 2e-7 * ref.abs().max().item() * max(sizes)
        assert (out[1][n] - ref).abs().max().item() <= bound, n
