"""The cell build that clears the status flags itself against the clearing launch
and the plain build: same cells, same flags whatever they held before; fewer
atoms than flags, one and several blocks, both scans, atoms outside an open
grid, non-finite coordinates.  Integers throughout, so everything is equal."""
import numpy as np
import pytest
import torch

from tensormol_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("periodic", [0, 1])
@pytest.mark.parametrize("bad", ["none", "outside", "nan", "both"])
@pytest.mark.parametrize("N,n", [(1, 2), (7, 3), (257, 5), (3000, 40)])
def test_cell_build_fresh(cuda, N, n, bad, periodic):
    L = _lib.lib()
    rng = np.random.default_rng(N)
    x = rng.uniform(0, 12.0, (N, 3))
    if bad in ("outside", "both"):
        x[N - 1, 1] = -0.5
    if bad in ("nan", "both"):
        x[N // 2, 2] = np.nan if bad == "nan" else np.inf
    pos = torch.tensor(x, dtype=torch.float64, device=cuda)
    mol = torch.zeros(N, dtype=torch.int32, device=cuda)
    i32 = dict(dtype=torch.int32, device=cuda)
    cs, out = 12.0 / n, []
    for fresh in (False, True):
        t = dict(of=torch.full((N,), -1, **i32), count=torch.zeros(n ** 3, **i32),
                 start=torch.full((n ** 3 + 1,), -1, **i32), fill=torch.full((N,), -1, **i32),
                 atoms=torch.full((N,), -1, **i32), cpos=torch.full((N,), -1, **i32))
        posc = torch.zeros(N, 3, dtype=torch.float64, device=cuda)
        flags = torch.arange(1, 9, **i32)
        if not fresh:
            L.tm_zero_i32(8, _lib.ptr(flags), None)
        build = L.tm_cell_build_fresh if fresh else L.tm_cell_build
        for _ in range(2 if fresh else 1):   # a second build clears the first one's flags
            build(N, _lib.ptr(pos), _lib.ptr(mol), 0.0, 0.0, 0.0, cs, cs, cs, n, n, n, periodic,
                  _lib.ptr(t["of"]), _lib.ptr(t["count"]), _lib.ptr(t["start"]),
                  _lib.ptr(t["fill"]), _lib.ptr(t["atoms"]), _lib.ptr(t["cpos"]),
                  _lib.ptr(posc), None, _lib.ptr(flags), None)
        torch.cuda.synchronize()
        del t["fill"]   # staging, in the order of the atomics
        out.append((t, posc.cpu().numpy(), flags.cpu().numpy()))
    (t0, p0, f0), (t1, p1, f1) = out
    for k in t0:
        assert torch.equal(t0[k], t1[k]), k
    np.testing.assert_array_equal(p0, p1)
    np.testing.assert_array_equal(f0, f1)
    assert bool(f1[3]) == (bad in ("nan", "both"))
    if not periodic and bad == "outside":
        assert f1[2] == 1
