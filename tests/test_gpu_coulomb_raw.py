"""Molecule electrostatics from raw charges in one launch against the mean,
charge and sweep launches: molecules of one atom, of whole and partial chunks of
64, without atoms, wider than the cutoff, and in periodic boxes.

Both form the same FP32 pair terms in the same order; the molecule means sum in
another order, 1e-16 apart, which can round a charge to the neighbouring FP32
value.  Tolerance: 2e-7 of the sums of the terms' magnitudes, of which the
largest value of an output array times the atoms of a molecule is a bound."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes,width,edge", [([1], 2.0, None), ([5, 0, 1, 64, 0], 6.0, None),
                                              ([63, 65, 128, 130, 3], 8.0, None),
                                              ([40, 200], 30.0, None), ([70, 30], 40.0, 40.0)])
def test_raw_equals_separate_launches(cuda, sizes, width, edge):
    from tensormol_amd import _lib
    from tensormol_amd.engine import BPEEEngine
    from tensormol_amd.model import BPEEModel
    L, P = _lib.lib(), _lib.ptr
    rng = np.random.default_rng(sum(sizes))
    model = BPEEModel([1, 8], hidden=[64] * 3)
    eng = BPEEEngine(model, precision="fp32")
    N, B = sum(sizes), len(sizes)
    ms = np.concatenate([[0], np.cumsum(sizes)])
    box = None if edge is None else np.full((B, 3), edge)
    x = rng.uniform(0, width, (N, 3))
    ws = eng.prepare(rng.choice([1, 8], N), ms, box, pos0=x)
    if ws.use_cells:
        pytest.skip("a cell grid sweeps this one")
    pos = torch.tensor(x, device=cuda)
    ws.qraw.copy_(torch.tensor(rng.normal(size=N), dtype=torch.float32))
    st = torch.cuda.current_stream().cuda_stream
    for t in (ws.qmean, ws.q, ws.qx, ws.phi, ws.gradc, ws.eatom, ws.phimean, ws.xq):
        t.fill_(float("nan"))
    eng.electrostatics(ws, pos)
    torch.cuda.synchronize()
    names = ("qmean", "q", "qx", "phi", "gradc", "eatom", "phimean", "xq")
    got = {n: getattr(ws, n).clone() for n in names}
    L.tm_mol_sum_f32(B, P(ws.mol_start), 1, P(ws.qraw), 1, P(ws.qmean), 1, P(ws.red), N, st)
    L.tm_charges(N, P(ws.mol), None, P(ws.qmean), P(ws.qraw), P(pos), P(ws.xq), P(ws.q), P(ws.qx),
                 None, None, None, None, st)
    L.tm_coulomb(N, P(ws.xq), P(ws.elem), P(ws.mol), P(ws.mol_start), P(ws.box), None, None, None,
                 None, None, 1, 1, 1, 1.0, 1.0, 1.0, 0.0, 0.0, 0.0, ws.periodic,
                 eng.dsf.ctypes.data_as(_lib.P), model.ee_off, eng.vdw_width, 1,
                 int(model.has_vdw), eng.nele, eng.c6.ctypes.data_as(_lib.P),
                 eng.r0.ctypes.data_as(_lib.P), None, None, P(ws.phi), P(ws.gradc), P(ws.eatom),
                 P(ws.flags), st)
    L.tm_mol_sum_f64(B, P(ws.mol_start), 1, P(ws.phi), 1, P(ws.phimean), 1, P(ws.red), N, st)
    torch.cuda.synchronize()
    for n in names:
        ref = getattr(ws, n).double()
        assert not got[n].isnan().any(), n
        bound = 2e-7 * max(ref.abs().max().item(), 1e-30) * max(sizes)
        assert (got[n].double() - ref).abs().max().item() <= bound, n
