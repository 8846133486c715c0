"""The transforms in LDS at the edges of what they take: every radix, rows and
columns that end inside a tile, an odd number of rows, lines beyond 64 KB of
LDS, ghosts wider than the box; and the lengths beside them that go to the
library.

Each transform rounds to a few ulp of the largest mode. The operator's smallest
mode is about (pi / n)^2 of its largest one, so that its relative error, and
with it the solution's, is a few (n / pi)^2 ulp: 8 of them, or 1e-12 as in
test_gpu_fourier.py where that is more.
"""
import numpy as np
import pytest
import torch

from conftest import STC7
from nga2_amd import fourier, incomp
from nga2_amd.config import Config, uniform
from oracle import fourier3d_ref as F3

pytestmark = pytest.mark.gpu

SHAPES = [
    ((2, 2, 2), 1),
    ((64, 30, 28), 1),
    ((77, 26, 40), 1),       # 7 x 11, 2 x 13, 5 x 8
    ((121, 65, 22), 2),
    ((169, 7, 3), 1),        # an odd number of rows
    ((126, 1, 9), 1),        # no y transform
    ((8, 1024, 2), 1),       # 144 KB of LDS a workgroup
    ((4, 2, 512), 1),        # 72 KB: 512 threads
    ((4, 1001, 3), 1),       # 7 x 11 x 13 in 141 KB: 512 threads of more registers
    ((1024, 2, 1), 1),
    ((143, 63, 49), 1),      # three row pairs a workgroup, the last with one and a half
    ((1001, 65, 32), 1),     # long rows, two pairs a workgroup
    ((1024, 33, 64), 1),
    ((16, 16, 17), 1),       # a prime factor above 13: the library
    ((8, 1026, 2), 1),
    ((1, 16, 24), 1),        # no x transform: the library
    ((4, 2, 3), 3),          # ghosts wider than the box
]


def problem(n, no):
    per = tuple(m > 1 for m in n)
    cfg = Config(*(uniform(m, m / max(n)) for m in n), no=no, xper=per[0], yper=per[1], zper=per[2])
    opr = incomp.laplacian(incomp.Metrics(cfg))
    rng = np.random.default_rng(11)
    rhs, sol0 = (np.asfortranarray(rng.standard_normal(cfg.shape)) for _ in range(2))
    ref = F3.solve(cfg, F3.setup(cfg, opr, STC7, fourier.circ_tol(cfg)), rhs, sol0)
    return cfg, opr, rhs, sol0, ref


def up(a):
    return torch.from_numpy(np.ascontiguousarray(a.ravel(order="F"))).cuda()


@pytest.mark.parametrize("n,no", SHAPES)
def test_solve_matches_oracle(n, no):
    print(f"\n[fourier tiles {n} ghosts {no}]", flush=True)
    cfg, opr, rhs, sol0, ref = problem(n, no)
    ds = fourier.DeviceFourier(cfg)
    ds.setup(up(opr))
    d_rhs, d_sol = up(rhs), up(sol0)
    ds.solve(d_rhs, d_sol)
    got = d_sol.cpu().numpy().reshape(cfg.shape, order="F")
    tol = max(1e-12, 8 * 2.0 ** -52 * (max(n) / np.pi) ** 2)
    assert np.abs(got - ref).max() <= tol * np.abs(ref).max()
    # ghosts: exactly the images of the returned interior
    chk = got.copy()
    cfg.sync(chk)
    assert np.array_equal(chk, got)
    assert torch.equal(d_rhs, up(rhs))
    ds.destroy()


def test_handles_of_long_and_shorter_lines():
    """The LDS a kernel may use is a limit of the kernel: a handle made later
    for shorter lines (still over 64 KB) leaves an older one's as it is."""
    made = []
    for n in ((8, 1024, 2), (8, 576, 2)):
        print(f"\n[fourier handles {n}]", flush=True)
        cfg, opr, rhs, sol0, ref = problem(n, 1)
        ds = fourier.DeviceFourier(cfg)
        ds.setup(up(opr))
        made.append((ds, n, cfg, rhs, sol0, ref))
    for ds, n, cfg, rhs, sol0, ref in made:
        d_rhs, d_sol = up(rhs), up(sol0)
        ds.solve(d_rhs, d_sol)
        got = d_sol.cpu().numpy().reshape(cfg.shape, order="F")
        tol = max(1e-12, 8 * 2.0 ** -52 * (max(n) / np.pi) ** 2)
        assert np.abs(got - ref).max() <= tol * np.abs(ref).max()
        ds.destroy()
