"""The tabulated sweep at sizes around the rounds where a two-element system's
tables are read from memory instead of LDS (workgroups of eight atoms that leave
a round of 256 CUs half empty): equal, bit for bit, to a model with elements
that do not occur, whose tables are always in memory."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("natom", [2048, 2049, 3072, 3073, 4099, 5121, 7169, 8193])
@pytest.mark.parametrize("edge", [None, 46.2])
def test_rounds(cuda, natom, edge):
    from tensormol_amd.engine import BPEEEngine
    from tensormol_amd.model import BPEEModel
    rng = np.random.default_rng(natom)
    k = int(np.ceil(natom ** (1 / 3)))
    g = np.stack(np.meshgrid(*[np.arange(k)] * 3, indexing="ij"), -1).reshape(-1, 3)[:natom]
    x = (2.2 if edge is None else edge / k) * (g + rng.uniform(-0.15, 0.15, (natom, 3)))
    Z, q = rng.choice([1, 8], natom), torch.tensor(rng.normal(size=natom), dtype=torch.float32)
    pos = torch.tensor(x, device=cuda)
    outs = []
    for eles in ([1, 8], [1, 6, 8]):
        eng = BPEEEngine(BPEEModel(eles, hidden=[64] * 3), precision="fp32", ldr=256, lda=256)
        ws = eng.prepare(Z, [0, natom], None if edge is None else np.full((1, 3), edge), pos0=x)
        eng.build_lists(ws, pos)
        ws.qraw.copy_(q)
        for t in (ws.phi, ws.gradc, ws.eatom):
            t.fill_(float("nan"))
        eng.electrostatics(ws, pos)
        torch.cuda.synchronize()
        outs.append([t.clone() for t in (ws.phi, ws.gradc, ws.eatom)])
    for a, b in zip(*outs):
        assert not a.isnan().any() and torch.equal(a, b)
