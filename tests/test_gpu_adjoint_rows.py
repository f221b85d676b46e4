"""Descriptor adjoint on rows of every length its windows split differently: one
to a few members, 16 / 17 (120 and 136 triples: one window and two), more
members than lanes (65, 100, 128), and radial shell counts that leave the
angular part unaligned.

Reference: float64 autograd of the oracle's descriptors.  Tolerance: every term
is a product of a few FP32 factors, of which the Gaussians carry the largest
relative error, the rounding of exponents up to 4 (4.6)^2 = 85, i.e. 85 * 6e-8
= 5e-6; sums of at most 128 of them keep that size in the 2-norm.  2e-5 allows
four such factors."""
import copy

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


@pytest.mark.parametrize("nr", [32, 31])
@pytest.mark.parametrize("natom", [1, 2, 3, 4, 12, 17, 18, 30, 65, 66, 101, 129])
def test_adjoint_rows(cuda, natom, nr):
    from tensormol_amd.engine import BPEEEngine
    from tensormol_amd.model import BPEEModel
    from tensormol_amd.params import PARAMS
    rng = np.random.default_rng(natom)
    x = _ball(natom, rng)
    Z = rng.choice([1, 6, 8], natom)
    p = copy.deepcopy(dict(PARAMS))
    p["AN1_num_r_Rs"] = nr
    model = BPEEModel([1, 6, 8], hidden=[64] * 3, p=p)
    eng = BPEEEngine(model, precision="fp32", ldr=128 if natom < 100 else 256, lda=128)
    ms = np.array([0, natom])
    ws = eng.prepare(Z, ms, pos0=x)
    pos = torch.tensor(x, dtype=torch.float64, device=cuda)
    gE = torch.tensor(rng.normal(size=(natom, eng.D)), dtype=torch.float32, device=cuda)
    grad = torch.zeros(natom, 3, dtype=torch.float64, device=cuda)
    eng.build_lists(ws, pos)
    eng.check_flags(ws)
    assert int(ws.acnt[0]) == natom - 1
    eng.descriptor_vjp(ws, pos, gE, grad)
    sp = O.SymParams(model.eles, nr_r=nr)
    lists = O.build_lists(x, Z, ms, sp)
    xt = torch.tensor(x, requires_grad=True)
    w = gE.double().cpu()
    E = 0.0 * xt.sum()
    if len(lists.pi):
        Gr = O.sym_radial(xt, lists.pi, lists.pj, lists.pl, natom, sp)
        E = E + (Gr * w[:, :Gr.shape[1]]).sum()
    if len(lists.ti):
        Ga = O.sym_angular(xt, lists.ti, lists.tj, lists.tk, lists.tp, natom, sp)
        E = E + (Ga * w[:, w.shape[1] - Ga.shape[1]:]).sum()
    (ref,) = torch.autograd.grad(E, xt)
    err = (grad.cpu() - ref).norm().item()
    assert err <= 2e-5 * ref.norm().item()
