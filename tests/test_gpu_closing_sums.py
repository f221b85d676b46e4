"""run()'s combined force gather and closing sums against adjoint() and
reductions(), and the total energy against its parts: the same sums in the same
order, so equal bits.  Sizes around a block of the sums (1024 atoms, 2048 for
the switch to several blocks), molecules of one atom, without atoms, larger
than a block, and repeated calls (the completion counter must return to zero)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [[1], [3, 0, 300, 1], [256], [257, 40], [2048], [2049], [3500]])
def test_run_equals_stages(cuda, sizes):
    from tensormol_amd.engine import BPEEEngine
    from tensormol_amd.model import BPEEModel
    rng = np.random.default_rng(sum(sizes))
    N, ms = sum(sizes), np.concatenate([[0], np.cumsum(sizes)])
    # a grid of atoms 1.5 A apart, jittered
    k = int(np.ceil(N ** (1 / 3)))
    g = np.stack(np.meshgrid(*[np.arange(k)] * 3, indexing="ij"), -1).reshape(-1, 3)[:N]
    x = 1.5 * g + rng.uniform(-0.2, 0.2, (N, 3))
    eng = BPEEEngine(BPEEModel([1, 8], hidden=[64] * 3, seed=1), precision="fp32", ldr=256, lda=128)
    ws = eng.prepare(rng.choice([1, 8], N), ms, pos0=x)
    pos = torch.tensor(x, device=cuda)
    names = ("Ebp", "Eext", "dipole", "grad", "force")
    eng.build_lists(ws, pos)
    eng.descriptors(ws, pos)
    eng.networks(ws)
    eng.electrostatics(ws, pos)
    eng.adjoint(ws, pos)
    eng.reductions(ws)
    torch.cuda.synchronize()
    ref = {n: getattr(ws, n).clone() for n in names}
    for _ in range(3):
        for n in names:
            getattr(ws, n).fill_(float("nan"))
        eng.run(ws, pos, check=True)
        E = eng.energy_tensor(ws)
        torch.cuda.synchronize()
        for n in names:
            B = ref[n].shape[0]
            assert torch.equal(getattr(ws, n)[:B], ref[n]), n
        assert torch.equal(E, ws.Ebp[:ws.B] + ws.Eext[:ws.B, 0] + ws.Eext[:ws.B, 1])
