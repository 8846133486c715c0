"""The V-cycle against the same cycle put together from the kernels of its
levels, one launch each, through the hooks: the same bits. This holds the fused
launches to the kernels they replace: the sweep pairs, the three transfers over
skipped levels (k_gather3, k_prolong3) and the small levels in one workgroup
(k_bottom).

The shapes reach: chains of all orders of directions that the coarsening
produces, odd and even lengths, walled and periodic directions side by side,
one-cell directions, and the first levels that the bottom takes in either
precision. Levels of at most 1024 cells with rows of 64 FP64 (128 FP32) cells and
more are left out: there k_bottom and the residual of long rows, k_stencil_rw,
round one product differently.
"""
import numpy as np
import pytest

from nga2_amd._lib import MIXED
from test_gpu_parity import _box, _solver

pytestmark = pytest.mark.gpu


def relaxed(hk, skip):
    """The levels that the cycle smooths (set_relax on a uniform grid)."""
    out = []
    for l in range(hk.nlevels):
        if not skip or l == 0 or l == hk.nlevels - 1:
            out.append(True)
            continue
        n, _ = hk.level_info(l)
        co = hk.level_coefs(l)
        s = [np.abs(co[a]).sum() for a, m in zip(("ax", "ay", "az"), n) if m > 1]
        s = [v for v in s if v > 0.0]
        out.append(len(s) < 2 or max(s) <= 2.0 * (1.0 + 1e-6) * min(s))
    return out


def chains(hk, relax):
    """Levels from which three transfers along three directions pass over two skipped levels."""
    d = [hk.level_info(l)[1] for l in range(hk.nlevels)]
    return [l for l in range(hk.nlevels - 3)
            if not relax[l + 1] and not relax[l + 2] and len(set(d[l:l + 3])) == 3]


def composed(hk, r, relax, nu, prec):
    """One V(nu, nu) cycle from a zero guess, level by level: red first on the way down, black on the way up."""
    nl = hk.nlevels

    def cycle(l, f):
        if l == nl - 1:
            return hk.coarse_solve(f, prec=prec)
        v = np.zeros_like(f)
        if relax[l]:
            v = hk.rbgs(l, f, v, 2, prec=prec)
            for _ in range(nu - 1):
                v = hk.rbgs(l, f, v, 0, prec=prec)
        v = hk.prolong_add(l, cycle(l + 1, hk.resid_restrict(l, f, v, prec=prec)), v, prec=prec)
        if relax[l]:
            for _ in range(nu):
                v = hk.rbgs(l, f, v, 1, prec=prec)
        return v

    return cycle(0, r)


SHAPES = [
    # shape, periodic, chains with skipped levels
    ((66, 50, 38), (False, False, False), True),
    ((67, 49, 35), (False, False, False), True),     # an odd last cell in every direction
    ((64, 64, 48), (True, True, True), True),
    ((48, 64, 37), (True, True, False), True),       # periodic and walled directions in one chain
    ((37, 48, 64), (False, True, True), True),
    ((130, 3, 130), (False, False, False), True),    # a direction of three cells
    ((64, 1, 48), (True, True, True), False),        # one cell in y
    ((16, 16, 16), (True, True, True), True),        # first coarse level: 2048 cells
    ((15, 17, 16), (False, False, False), True),
    ((1, 1, 1000), (True, True, False), False),      # a line
]


def check(shape, per, nu, skip, L, precs, chain=None):
    P = _box(*shape, per, walls=not all(per), L=L)
    ps = _solver(P, precision=MIXED, nu_pre=nu, nu_post=nu, skip_relax=skip, coarsest_max=20)
    hk = ps.hooks()
    relax = relaxed(hk, skip)
    if chain is not None:
        assert bool(chains(hk, relax)) == chain
    rng = np.random.default_rng(3)
    r = rng.standard_normal(int(np.prod(shape)))
    r -= r.mean()
    r = r.astype(np.float32).astype(np.float64)
    dims = [hk.level_info(l)[0] for l in range(hk.nlevels)]
    for prec in precs:
        got, want = hk.vcycle(r, prec=prec), composed(hk, r, relax, nu, prec)
        assert np.isfinite(want).all()
        assert np.array_equal(got, want), (prec, np.abs(got - want).max() / np.abs(want).max())
    ps.destroy()
    return dims


@pytest.mark.parametrize("skip", [0, 1])
@pytest.mark.parametrize("nu", [1, 2])
@pytest.mark.parametrize("shape,per,chain", SHAPES)
def test_cycle_equals_its_levels(shape, per, chain, nu, skip):
    print(f"\n[cycle bits {shape} {per} nu {nu} skip {skip}]", flush=True)
    check(shape, per, nu, skip, tuple(n / max(shape) for n in shape), (0, 1), chain if skip else None)


@pytest.mark.parametrize("nu", [1, 2])
def test_long_rows(nu):
    """A level of 2048 cells with rows of 128, too long for the FP32 bottom, and one of 1024 with rows of 64."""
    print(f"\n[cycle bits, long rows, nu {nu}]", flush=True)
    dims = check((256, 4, 4), (False, False, False), nu, 0, (0.25, 4 / 256, 4 / 256), (1,))
    assert dims[1:3] == [(128, 4, 4), (64, 4, 4)]
