"""Descriptors and tangents written as BF16 rows by the kernels that form them:
no, one and several workgroups, elements with one atom, both row capacities,
rows at places of any order and stride; what lies between the rows stays.

A descriptor row holds the rounding (to nearest even) of the FP32 values of the
same launch, so it is compared bit for bit.  A tangent row is compared with the
FP32 tangent of another launch: half a BF16 ulp is 2^-9 relative, 2^-8 leaves
room for the last FP32 bits, 1e-6 of the largest value for cancelling sums."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ldr", [128, 256])
@pytest.mark.parametrize("eles,natom", [([8], 1), ([1, 8], 2), ([1, 8], 5), ([1, 6, 7, 8], 37),
                                        ([1, 6, 7, 8], 131)])
def test_descriptor_rows(cuda, eles, natom, ldr):
    from tensormol_amd.engine import BPEEEngine
    from tensormol_amd.model import BPEEModel
    rng = np.random.default_rng(natom + ldr)
    grid = np.array([[i, j, k] for i in range(6) for j in range(6) for k in range(6)])[:natom]
    x = 1.3 * grid + rng.uniform(-0.2, 0.2, (natom, 3))
    Z = rng.choice(eles, natom)
    Z[0] = eles[-1]
    eng = BPEEEngine(BPEEModel(eles, hidden=[64] * 3), precision="fp32", ldr=ldr, lda=ldr)
    ws = eng.prepare(Z, np.array([0, natom]), pos0=x)
    pos = torch.tensor(x, dtype=torch.float64, device=cuda)
    du = torch.tensor(rng.normal(size=(natom, 3)), dtype=torch.float64, device=cuda)
    ybar = torch.tensor(rng.normal(size=natom), dtype=torch.float32, device=cuda)
    D, ld = eng.D, eng.D + 9   # an odd stride: rows at two-byte alignment
    X = torch.full((2 * natom, ld), -3.0, dtype=torch.bfloat16, device=cuda)
    yf = torch.full((natom,), -3.0, dtype=torch.float32, device=cuda)
    yh = torch.full((2 * natom,), -3.0, dtype=torch.bfloat16, device=cuda)
    order = rng.permutation(natom)   # atom i writes row order[i]
    places = torch.tensor(np.stack([X.data_ptr() + 2 * ld * order,
                                    X.data_ptr() + 2 * ld * (natom + order),
                                    yf.data_ptr() + 4 * order, yh.data_ptr() + 2 * order], 1),
                          dtype=torch.int64, device=cuda)
    V = torch.empty(natom, D, dtype=torch.float32, device=cuda)
    eng.build_lists(ws, pos)
    eng.check_flags(ws)
    eng.descriptors(ws, pos)
    G, rev = ws.G[:natom].clone(), ws.rev.clone()
    eng.descriptor_jvp(ws, pos, du, V)
    ws.G.fill_(float("nan"))
    eng.descriptor_rows(ws, pos, places)
    assert torch.equal(X[natom:], torch.full_like(X[natom:], -3.0))
    eng.descriptor_jvp_rows(ws, pos, du, ybar, places)
    eng.check_flags(ws)
    at = torch.tensor(order, device=cuda)
    torch.testing.assert_close(ws.G[:natom], G, rtol=2e-6, atol=1e-30)
    assert torch.equal(X[at, :D], ws.G[:natom].to(torch.bfloat16))
    n = torch.arange(ldr, device=cuda) < ws.ncnt[:natom, None]
    assert torch.equal(ws.rev.view(-1, ldr)[:natom][n], rev.view(-1, ldr)[:natom][n])
    err = (X[natom + at, :D].float() - V).abs()
    assert bool((err <= V.abs() * 2.0 ** -8 + 1e-6 * V.abs().max()).all())
    assert torch.equal(X[:, D:], torch.full_like(X[:, D:], -3.0))
    assert torch.equal(yf[at], ybar) and torch.equal(yh[at], ybar.to(torch.bfloat16))
    assert torch.equal(yh[natom:], torch.full_like(yh[natom:], -3.0))
