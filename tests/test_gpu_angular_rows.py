"""Descriptors and their tangent where the angular pass splits its work: no pair,
55 / 66 triples (one chunk of 64 and two), 120 / 136, more members than lanes;
one to four elements, with elements that a centre has none of (empty pairs) and
one that holds a single atom.

References: the oracle's float64 descriptors, and for the tangent their
float64 directional derivative.  Tolerance: a term is a product of a few FP32
factors, the largest relative error being that of a Gaussian whose exponent
(up to 4 (4.6)^2 = 85) is rounded, 85 * 6e-8 = 5e-6; 2e-5 allows four such
factors.  Descriptors are sums of positive terms, so it holds for each (with
1e-7 for values that underflow); the tangent's terms cancel, so it is taken in
the 2-norm against the sum of the terms' magnitudes, which is at least the
norm of the result."""
import numpy as np
import pytest
import torch

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _ball(n, rng):
    """n points at least 0.35 A apart in a ball of radius 1.5 A: all within 3.1 A."""
    pts = []
    while len(pts) < n:
        c = rng.uniform(-1.5, 1.5, 3)
        if c @ c < 1.5 ** 2 and all((c - p) @ (c - p) > 0.35 ** 2 for p in pts):
            pts.append(c)
    return np.array(pts)


@pytest.mark.parametrize("eles,used", [([8], [8]), ([1, 8], [1, 8]), ([1, 6, 7, 8], [1, 6, 7, 8]),
                                       ([1, 6, 7, 8], [6]), ([1, 6, 7, 8], [1, 8])])
@pytest.mark.parametrize("natom", [1, 2, 3, 12, 13, 17, 18, 67])
def test_angular_rows(cuda, natom, eles, used):
    from tensormol_amd.engine import BPEEEngine
    from tensormol_amd.model import BPEEModel
    rng = np.random.default_rng(100 * natom + len(eles) + used[0])
    x = _ball(natom, rng)
    Z = rng.choice(used, natom)
    Z[0] = used[-1]
    if natom > 3 and len(used) > 2:
        Z[Z == used[1]] = used[0]
        Z[1] = used[1]          # an element with one atom
    model = BPEEModel(eles, hidden=[64] * 3)
    eng = BPEEEngine(model, precision="fp32", ldr=128, lda=128)
    ms = np.array([0, natom])
    ws = eng.prepare(Z, ms, pos0=x)
    pos = torch.tensor(x, dtype=torch.float64, device=cuda)
    du = torch.tensor(rng.normal(size=(natom, 3)), dtype=torch.float64, device=cuda)
    V = torch.empty(natom, eng.D, dtype=torch.float32, device=cuda)
    ws.G.fill_(float("nan"))
    eng.build_lists(ws, pos)
    eng.check_flags(ws)
    assert int(ws.acnt[0]) == natom - 1
    eng.descriptors(ws, pos)
    eng.descriptor_jvp(ws, pos, du, V)
    sp = O.SymParams(model.eles)
    lists = O.build_lists(x, Z, ms, sp)

    def descr(xt):
        Gr = torch.zeros(natom, len(eles) * sp.nr_r, dtype=torch.float64) + 0.0 * xt.sum()
        Ga = torch.zeros(natom, eng.D - Gr.shape[1], dtype=torch.float64) + 0.0 * xt.sum()
        if len(lists.pi):
            Gr = O.sym_radial(xt, lists.pi, lists.pj, lists.pl, natom, sp)
        if len(lists.ti):
            Ga = O.sym_angular(xt, lists.ti, lists.tj, lists.tk, lists.tp, natom, sp)
        return torch.cat([Gr, Ga], 1)

    ref = descr(torch.tensor(x)).numpy()
    got = ws.G[:natom].double().cpu().numpy()
    assert (np.abs(got - ref) <= 2e-5 * np.abs(ref) + 1e-7).all()
    # d/dt G(x + t u) by a second derivative: v -> grad(v . G) is linear in v
    xt = torch.tensor(x, requires_grad=True)
    v = torch.zeros(natom, eng.D, dtype=torch.float64, requires_grad=True)
    (gx,) = torch.autograd.grad((descr(xt) * v).sum(), xt, create_graph=True)
    (tan,) = torch.autograd.grad((gx * du.cpu()).sum(), v)
    # |dG/dx| is at most about 2 eta 4.6 + zeta + pi / 3.1 < 50 per term of G, and
    # |du_j - du_i| a few: magnitudes of the terms from the descriptors themselves
    scale = np.maximum(tan.abs().numpy(), 50.0 * np.abs(ref))
    assert np.linalg.norm(V.double().cpu().numpy() - tan.numpy()) <= 2e-5 * np.linalg.norm(scale)
