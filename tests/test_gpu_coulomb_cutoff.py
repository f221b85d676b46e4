"""Pairs at the last digit of the Coulomb cutoff.  Whether one counts moves the
FP32 lane sums of every pair behind it, so the tabulated sweep takes the same
decision in all of its loops: r^2 = fma(z, z, fma(x, x, y y)) < 15^2.  Each
separation here falls on different sides of the cutoff when x and y change
places in that form; with charges 1 and the constant table K = 1, phi counts
pairs: 300 atoms at one place and one atom that separation away."""
from fractions import Fraction

import numpy as np
import pytest
import torch

from tests import helpers as H

pytestmark = pytest.mark.gpu

NEAR = [(2.403212547302246, -12.271933555603027, 8.28397274017334),
        (-11.464350700378418, 7.605044841766357, -5.977621078491211),
        (3.926193952560425, 14.476249694824219, -0.15231658518314362),
        (-4.818249225616455, 13.60537052154541, -4.083914756774902),
        (-3.3940958976745605, -14.554965019226074, 1.2779312133789062),
        (-6.5701446533203125, -13.006075859069824, 3.560222625732422)]
ATOMS = 300


def _fma(a, b, c):
    """a b + c rounded once to float32 (to nearest, ties to even)."""
    v = Fraction(float(a)) * Fraction(float(b)) + Fraction(float(c))
    x = np.float32(float(v))
    near = [np.nextafter(x, np.float32(-np.inf)), x, np.nextafter(x, np.float32(np.inf))]
    return min(near, key=lambda t: (abs(Fraction(float(t)) - v), int(t.view(np.int32)) & 1))


def _inside(x, y, z):
    return _fma(z, z, _fma(x, x, _fma(y, y, 0.0))) < np.float32(225.0)


@pytest.mark.parametrize("model,edge", [("water", None), ("water", 40.0), ("chno", None),
                                        ("chno", 40.0)])
def test_cutoff_decision(cuda, model, edge):
    from tensormol_amd import _lib
    from tensormol_amd.engine import BPEEEngine
    eng = BPEEEngine(H.model_for(model), precision="fp32", check_overflow=False)
    tab = torch.zeros(1 + eng.nele * (eng.nele + 1) // 2, eng.cl_nint, 4, device=cuda)
    tab[0, :, 0] = 1.0
    _, inv_h, u0 = eng._cl_table()
    P, N = _lib.ptr, ATOMS + 1
    sides = set()
    for v in NEAR:
        d = np.array(v, dtype=np.float32)
        inside, swapped = _inside(*d), _inside(d[1], d[0], d[2])
        assert inside != swapped
        sides.add(bool(inside))
        x = np.zeros((N, 3))
        x[1:] = d
        ws = eng.prepare(np.where(np.arange(N) % 3 == 0, 8, 1), np.array([0, N]),
                         None if edge is None else np.full((1, 3), edge), pos0=x)
        pos = torch.tensor(x, device=cuda)
        eng.build_lists(ws, pos)
        order = ws.cell_atoms.long()
        ws.xqc[:, :3] = pos[order].float()
        ws.xqc[:, 3] = 1.0
        ws.elc.copy_(ws.elem[:N][order])
        g = eng._grid_args(ws)
        eng.lib.tm_coulomb_tab(N, P(ws.box), g[0], g[1], g[2], *g[6:15], ws.periodic, 15.0, eng.nele,
                               P(tab), eng.cl_nint, inv_h, u0, P(ws.xqc), P(ws.elc), P(ws.phi),
                               P(ws.gradc), P(ws.eatom), P(ws.flags), eng._stream())
        phi = ws.phi[:N].cpu().numpy()
        assert phi[0] == (ATOMS if inside else 0), v
        assert np.all(phi[1:] == ATOMS - 1 + (1 if inside else 0)), v
    assert sides == {True, False}
