"""The total energy is a torch sum where the workspace is not on the current
GPU: the launch that replaces it goes to the current device's stream."""
import numpy as np
import torch

from tests import helpers as H


class _Elsewhere:
    """A tensor that says it lives on another GPU than the current one."""
    is_cuda, device = True, torch.device("cuda", 1)

    def __init__(self, t):
        self.t = t

    def __getitem__(self, k):
        return self.t[k]


def test_energy_tensor_off_the_current_device(monkeypatch):
    from tensormol_amd.engine import BPEEEngine
    eng = BPEEEngine(H.water_model(), device="cpu", precision="fp32", ldr=2, lda=2)
    ws = eng.prepare(np.ones(7, int), np.array([0, 3, 4, 7]))
    rng = np.random.default_rng(0)
    ws.Ebp.copy_(torch.tensor(rng.normal(size=3)))
    ws.Eext.copy_(torch.tensor(rng.normal(size=(3, 2))))
    want = (ws.Ebp + ws.Eext[:, 0]) + ws.Eext[:, 1]
    assert torch.equal(eng.energy_tensor(ws), want)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    ws.Ebp = _Elsewhere(ws.Ebp)
    assert torch.equal(eng.energy_tensor(ws), want)
