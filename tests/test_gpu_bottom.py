"""The small-level bottom of the V-cycle at the edges of what it takes: levels
of odd lengths, one or two cells wide, the largest first levels it accepts in
either precision and one just beyond, skipped levels, several sweeps.

The FP64 cycle issues the oracle's operations in the oracle's order, level by
level; only the coarsest inverse and fused multiply-adds round differently, a
few ulp amplified by the cycle's own O(1) factors: 1e-9 of max|z|, as in
test_gpu_parity.py. The FP32 cycle rounds each of about 100 operations per cell
and level to 2^-24: 1e-3, as there.
"""
import numpy as np
import pytest

from nga2_amd._lib import MIXED
from oracle.orc import Oracle
from test_gpu_parity import _box, _close, _solver

pytestmark = pytest.mark.gpu

SHAPES = [
    ((15, 17, 16), (False, False, False)),   # odd lengths all the way down
    ((16, 16, 16), (True, True, True)),      # first coarse level: 2048 cells
    ((31, 16, 16), (False, True, True)),     # odd rows beside periodic directions
    ((16, 16, 8), (True, True, True)),       # first coarse level: 1024 cells
    ((17, 16, 9), (False, True, False)),
    ((1, 40, 52), (True, False, False)),     # one cell wide: half of the places hold no cell
    ((2, 32, 64), (True, True, False)),      # a periodic direction of two cells
    ((64, 2, 31), (False, False, False)),
    ((1, 1, 1000), (True, True, False)),     # a line
]


@pytest.mark.parametrize("skip", [0, 1])
@pytest.mark.parametrize("nu", [1, 2])
@pytest.mark.parametrize("shape,per", SHAPES)
def test_cycle_matches_oracle(shape, per, nu, skip):
    print(f"\n[bottom {shape} {per} nu {nu} skip {skip}]", flush=True)
    P = _box(*shape, per, walls=not all(per), L=tuple(n / max(shape) for n in shape))
    o = Oracle.from_cfg(P.cfg, P.opr, skip_relax=skip, coarsest_max=20, nu_pre=nu, nu_post=nu)
    ps = _solver(P, precision=MIXED, nu_pre=nu, nu_post=nu, skip_relax=skip, coarsest_max=20)
    rng = np.random.default_rng(3)
    r = rng.standard_normal(o.N)
    r -= r.mean()
    zo = o.vcycle(r)
    assert _close(ps.hooks().vcycle(r), zo, 1e-9)
    assert _close(ps.hooks().vcycle(r, prec=1), zo, 1e-3)
    ps.destroy()
    o.close()
