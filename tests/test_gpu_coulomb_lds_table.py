"""The tabulated sweep with its tables in LDS (two elements, 1,024 entries) and
in memory (more elements): the same atoms under models that differ in elements
that do not occur read equal entries in equal order, so the results are equal
bit for bit.  Sizes: one more than the smallest cell system, workgroups of 4 and
8 waves partly filled, rounds whose candidates fit the list and rounds that do
not (a dense cluster)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("natom,spacing,edge", [(257, 2.6, None), (523, 2.2, None), (1031, 1.1, None),
                                                (1000, 3.2, 32.0), (1728, 2.6, 31.2)])
def test_lds_tables_equal_memory_tables(cuda, natom, spacing, edge):
    from tensormol_amd.engine import BPEEEngine
    from tensormol_amd.model import BPEEModel
    rng = np.random.default_rng(natom)
    k = int(np.ceil(natom ** (1 / 3)))
    g = np.stack(np.meshgrid(*[np.arange(k)] * 3, indexing="ij"), -1).reshape(-1, 3)[:natom]
    x = spacing * (g + rng.uniform(-0.15, 0.15, (natom, 3)))
    Z = rng.choice([1, 8], natom)
    q = torch.tensor(rng.normal(size=natom), dtype=torch.float32)
    pos = torch.tensor(x, device=cuda)
    box = None if edge is None else np.full((1, 3), edge)
    outs = []
    for eles in ([1, 8], [1, 6, 8], [1, 6, 7, 8]):
        eng = BPEEEngine(BPEEModel(eles, hidden=[64] * 3), precision="fp32", ldr=256, lda=256)
        assert eng.coulomb_tables
        small = (1 + len(eles) * (len(eles) + 1) // 2) * eng.cl_nint <= 1024
        assert small == (len(eles) == 2)
        ws = eng.prepare(Z, [0, natom], box, pos0=x)
        assert ws.use_cells
        eng.build_lists(ws, pos)
        ws.qraw.copy_(q)
        for t in (ws.phi, ws.gradc, ws.eatom):
            t.fill_(float("nan"))
        eng.electrostatics(ws, pos)
        torch.cuda.synchronize()
        outs.append([t.clone() for t in (ws.phi, ws.gradc, ws.eatom)])
        assert not any(t.isnan().any() for t in outs[-1])
    for other in outs[1:]:
        for a, b in zip(outs[0], other):
            assert torch.equal(a, b)
