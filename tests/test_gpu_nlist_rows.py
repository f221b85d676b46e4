"""Neighbour rows against brute force in float64, entry for entry: molecules of
one atom, around whole chunks of 64, several in a batch, dense rows (lengths
around multiples of 4 and 64, up to more than 128), one system on a cell grid,
open and periodic with atoms outside the box, and rows that overflow.  The lists
are integers, so the comparison is exact; positions are random, which keeps
pairs away from the cutoff by far more than float64 rounding."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _rows(x, elem, ms, edge, rc):
    """(neighbours by (element, index), of these the places closer than 3.1) per atom."""
    out = []
    for m in range(len(ms) - 1):
        for i in range(ms[m], ms[m + 1]):
            d = x[ms[m]:ms[m + 1]] - x[i]
            if edge is not None:
                d = d - edge * np.round(d / edge)
            r = np.sqrt((d * d).sum(1))
            js = [j for j in range(ms[m], ms[m + 1]) if j != i and r[j - ms[m]] < rc[0]]
            js.sort(key=lambda j: (elem[j], j))
            out.append((js, [k for k, j in enumerate(js) if r[j - ms[m]] < rc[1]]))
    return out


@pytest.mark.parametrize("sizes,width,edge,ldr", [
    ([1], 1.0, None, 128), ([2, 64, 65, 3], 9.0, None, 128), ([128, 129], 12.0, None, 128),
    ([34], 3.0, None, 128), ([66], 3.5, None, 128), ([130], 4.0, None, 256),
    ([700], 24.0, None, 128), ([900], 90.0, 31.0, 128), ([300], 40.0, None, 128)])
def test_rows(cuda, sizes, width, edge, ldr):
    from tensormol_amd.engine import BPEEEngine
    from tensormol_amd.model import BPEEModel
    rng = np.random.default_rng(sum(sizes))
    N, ms = sum(sizes), np.concatenate([[0], np.cumsum(sizes)])
    x = rng.uniform(0, width, (N, 3))
    Z = rng.choice([1, 6, 8], N)
    model = BPEEModel([1, 6, 8], hidden=[64] * 3)
    eng = BPEEEngine(model, precision="fp32", ldr=ldr, lda=ldr)
    box = None if edge is None else np.full((len(sizes), 3), edge)
    ws = eng.prepare(Z, ms, box, pos0=x)
    eng.build_lists(ws, torch.tensor(x, device=cuda))
    eng.check_flags(ws)
    nbr = ws.nbr.view(-1, ldr).cpu().numpy()
    ang = ws.ang.view(-1, ldr).cpu().numpy()
    ncnt, acnt = ws.ncnt.cpu().numpy(), ws.acnt.cpu().numpy()
    rseg, aseg = (t.view(-1, 4).cpu().numpy() for t in (ws.rseg, ws.aseg))
    elem = model.element_index(Z)
    ref = _rows(x, elem, ms, edge, (model.sym.rr, model.sym.ra))
    assert max(len(r) for r, _ in ref) <= ldr
    for i, (row, sub) in enumerate(ref):
        assert ncnt[i] == len(row) and list(nbr[i, :ncnt[i]]) == row
        assert acnt[i] == len(sub) and list(ang[i, :acnt[i]]) == sub
        e = [int(elem[j]) for j in row]
        assert list(rseg[i]) == [sum(v < k for v in e) for k in range(4)]
        assert list(aseg[i]) == [sum(e[s] < k for s in sub) for k in range(4)]


@pytest.mark.parametrize("natom", [130, 300])
def test_rows_overflow(cuda, natom):
    """More neighbours than the row, or than the candidates a wave keeps, raise."""
    from tensormol_amd.engine import BPEEEngine, NeighbourOverflow
    from tensormol_amd.model import BPEEModel
    x = np.random.default_rng(natom).uniform(0, 2.5, (natom, 3))
    eng = BPEEEngine(BPEEModel([1, 8], hidden=[64] * 3), precision="fp32", ldr=128, lda=64)
    ws = eng.prepare(np.full(natom, 8), [0, natom], pos0=x)
    eng.build_lists(ws, torch.tensor(x, device=cuda))
    with pytest.raises(NeighbourOverflow):
        eng.check_flags(ws)
    assert int(ws.ncnt[:natom].max()) == 128
