"""Candidate sweeps over the cell grid against brute force, on grids where a
stencil can go wrong: axes that the cutoff wraps whole, mixed and long boxes,
unwrapped coordinates, rows far longer than the candidate list, few atoms.

The tabulated Coulomb sweep runs with the constant table K = 1 and charges 1,
so phi counts the pairs inside the cutoff exactly.  It tests FP32 distances: a
pair within 1e-3 A of the cutoff may be counted or not (FP32 positions up to
130 A are rounded by at most 8e-6 A).  The neighbour rows are compared with the
FP64 predicate without that allowance."""
import numpy as np
import pytest
import torch

from tests import helpers as H

pytestmark = pytest.mark.gpu


def _system(name, rng):
    if name.startswith("box"):
        edges = {"box_full": (31.06, 31.06, 31.06), "box_mixed": (33.0, 47.3, 62.0),
                 "box_long": (30.5, 30.5, 129.0), "box_unwrapped": (45.0, 38.0, 51.0)}[name]
        n = int(0.05 * np.prod(edges))
        x = rng.uniform(0.0, 1.0, (n, 3)) * edges
        if name == "box_unwrapped":
            x = x + rng.integers(-3, 4, (n, 3)) * np.array(edges)
        return x, np.array(edges)
    if name == "dense":    # every stencil row holds hundreds of atoms
        return rng.uniform(0.0, 9.0, (3000, 3)), None
    if name == "flat":
        return rng.uniform(0.0, 1.0, (2500, 3)) * (90.0, 60.0, 3.0), None
    return rng.uniform(0.0, 40.0, (257, 3)), None   # few: the smallest system on a grid


@pytest.mark.parametrize("name", ["box_full", "box_mixed", "box_long", "box_unwrapped", "dense",
                                  "flat", "few"])
def test_sweeps_count_brute_force(cuda, name):
    from tensormol_amd import _lib
    from tensormol_amd.engine import BPEEEngine
    x, edges = _system(name, np.random.default_rng(7))
    N = len(x)
    eng = BPEEEngine(H.model_for("water"), precision="fp32", ldr=256, lda=256,
                     check_overflow=False)
    ws = eng.prepare(np.where(np.arange(N) % 3 == 0, 8, 1), np.array([0, N]),
                     None if edges is None else edges[None], pos0=x)
    assert ws.use_cells
    pos = torch.tensor(x, dtype=torch.float64, device=cuda)
    eng.build_lists(ws, pos)
    order = ws.cell_atoms.long()
    ws.xqc[:, :3] = pos[order].float()
    ws.xqc[:, 3] = 1.0
    ws.elc.copy_(ws.elem[:N][order])
    _, inv_h, u0 = eng._cl_table()
    tab = torch.zeros(1 + eng.nele * (eng.nele + 1) // 2, eng.cl_nint, 4, device=cuda)
    tab[0, :, 0] = 1.0
    P = _lib.ptr
    g = eng._grid_args(ws)
    eng.lib.tm_coulomb_tab(N, P(ws.box), g[0], g[1], g[2], *g[6:15], ws.periodic, 15.0, eng.nele,
                           P(tab), eng.cl_nint, inv_h, u0, P(ws.xqc), P(ws.elc), P(ws.phi),
                           P(ws.gradc), P(ws.eatom), P(ws.flags), eng._stream())
    torch.cuda.synchronize()
    phi, ncnt = ws.phi[:N].cpu(), ws.ncnt[:N].cpu()
    lo, hi, short = (torch.zeros(N, dtype=torch.float64) for _ in range(3))
    L = None if edges is None else torch.tensor(edges, device=cuda)
    for s in range(0, N, 512):
        d = pos[s:s + 512, None] - pos[None]
        if L is not None:
            d = d - L * torch.round(d / L)
        r = torch.sqrt((d[..., 0] ** 2 + d[..., 1] ** 2) + d[..., 2] ** 2)
        r[torch.arange(len(r)), torch.arange(s, s + len(r))] = 1e9
        lo[s:s + 512] = (r < 15.0 - 1e-3).sum(1).cpu().double()
        hi[s:s + 512] = (r < 15.0 + 1e-3).sum(1).cpu().double()
        short[s:s + 512] = (r + 1e-13 < 4.6).sum(1).cpu().double()
    assert torch.all(phi == torch.round(phi))
    assert torch.all(phi >= lo) and torch.all(phi <= hi)
    assert hi.max() > 0
    if name != "dense":   # rows there exceed their stride
        assert torch.equal(ncnt.double(), short)
