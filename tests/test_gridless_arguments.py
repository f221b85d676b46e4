"""Sweeps without a cell grid (cell_atoms NULL) do not look at the grid's sizes:
a caller may pass zeros for them, with open and periodic molecules."""
import os
import subprocess
import sys

import numpy as np
import pytest
import torch

from tensormol_amd import _lib

ZERO, ONE = (0, 0, 0) + (0.0,) * 6, (1, 1, 1) + (1.0,) * 3 + (0.0,) * 3
NELE, LDR = 2, 64


def calls(sizes, periodic, N, bufs, P, stream):
    """The sweeps of N atoms in one molecule, on buffers `bufs`."""
    from tensormol_amd.engine import dsf_constants, nl_threshold
    L, b = _lib.lib(), {k: P(v) for k, v in bufs.items()}
    dsf = dsf_constants(0.2, 4.6, 15.0)
    c6, r0 = np.full(NELE, 0.5), np.full(NELE, 2.5)
    box = b["box"] if periodic else None
    yield lambda: L.tm_nl_build(
        N, b["pos"], b["elem"], b["mol"], b["ms"], box, *([None] * 6), *sizes, periodic, NELE, 4.6,
        nl_threshold(4.6), nl_threshold(3.1), LDR, LDR, b["nbr"], b["ncnt"], b["rseg"], b["ang"],
        b["acnt"], b["aseg"], None, b["flags"], stream)
    yield lambda: L.tm_pairs(
        N, b["pos"], b["mol"], b["ms"], None, box, *([None] * 6), *sizes, periodic, 4.6,
        nl_threshold(4.6), 0, b["count"], None, None, b["flags"], stream)
    yield lambda: L.tm_coulomb(
        N, b["xq"], b["elem"], b["mol"], b["ms"], box, *([None] * 5), *sizes, periodic,
        dsf.ctypes.data, 15.0, 8.7, 1, 1, NELE, c6.ctypes.data, r0.ctypes.data, None, None, b["phi"],
        b["grad"], b["eatom"], b["flags"], stream)


def buffers(N, device):
    rng = np.random.default_rng(2)
    i32, f64 = dict(dtype=torch.int32, device=device), dict(dtype=torch.float64, device=device)
    pos = torch.tensor(rng.uniform(0, 12, (N, 3)), **f64)
    return dict(pos=pos, elem=torch.arange(N, **i32) % NELE, mol=torch.zeros(N, **i32),
                ms=torch.tensor([0, N], **i32), box=torch.full((1, 3), 31.0, **f64),
                xq=torch.cat([pos.float(), torch.ones(N, 1, device=device)], 1).contiguous(),
                nbr=torch.zeros(N * LDR, **i32), ncnt=torch.zeros(N, **i32),
                rseg=torch.zeros(N * (NELE + 1), **i32), ang=torch.zeros(N * LDR, **i32),
                acnt=torch.zeros(N, **i32), aseg=torch.zeros(N * (NELE + 1), **i32),
                flags=torch.zeros(8, **i32), count=torch.zeros(N, **i32),
                phi=torch.zeros(N, **f64), grad=torch.zeros(N, 3, **f64),
                eatom=torch.zeros(N, 2, **f64))


def _host():
    """Without a device every call must come back with the launch's error."""
    for periodic in (0, 1):
        for call in calls(ZERO, periodic, 8, buffers(8, "cpu"), _lib.ptr, None):
            try:
                call()
                raise SystemExit("launched without a device")
            except RuntimeError as e:
                assert "launch" in str(e), e


@pytest.mark.skipif(torch.cuda.is_available(), reason="looks at the host side alone")
def test_host_side_survives_zero_sizes():
    r = subprocess.run([sys.executable, "-c", "from tests.test_gridless_arguments import _host; _host()"],
                       cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                       stdout=subprocess.PIPE, stderr=subprocess.STDOUT)
    assert r.returncode == 0, (r.returncode, r.stdout.decode())


@pytest.mark.gpu
@pytest.mark.parametrize("periodic", [0, 1])
def test_zero_sizes_change_nothing(cuda, periodic):
    N, out = 150, []
    for sizes in (ZERO, ONE):
        b = buffers(N, cuda)
        for call in calls(sizes, periodic, N, b, _lib.ptr, None):
            call()
        torch.cuda.synchronize()
        assert int(b["ncnt"].max()) > 10 and torch.equal(b["count"], b["ncnt"])
        out.append(b)
    for k, v in out[0].items():
        assert torch.equal(v, out[1][k]), k
