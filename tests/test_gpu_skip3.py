"""Three transfers in one launch over skipped levels: the cycle against the
oracle's, which goes level by level, on boxes of odd and even lengths, periodic
and walled, whose first chains lie above the levels that run in one workgroup.
Tolerances as in test_gpu_bottom.py.
"""
import numpy as np
import pytest

from nga2_amd._lib import MIXED
from oracle.orc import Oracle
from test_gpu_parity import _box, _close, _solver

pytestmark = pytest.mark.gpu

SHAPES = [
    ((66, 50, 38), (False, False, False)),
    ((67, 49, 35), (False, False, False)),   # an odd last cell in every direction
    ((64, 64, 48), (True, True, True)),
    ((50, 66, 37), (True, True, False)),     # odd periodic coarse lengths
    ((130, 3, 130), (False, True, False)),   # a direction of three cells
]


@pytest.mark.parametrize("shape,per", SHAPES)
def test_cycle_matches_oracle(shape, per):
    print(f"\n[skip3 {shape} {per}]", flush=True)
    per = tuple(p and n % 2 == 0 for p, n in zip(per, shape))
    P = _box(*shape, per, walls=not all(per), L=tuple(n / max(shape) for n in shape))
    o = Oracle.from_cfg(P.cfg, P.opr, skip_relax=1, coarsest_max=20, nu_pre=1, nu_post=1)
    ps = _solver(P, precision=MIXED, nu_pre=1, nu_post=1, skip_relax=1, coarsest_max=20)
    rng = np.random.default_rng(3)
    r = rng.standard_normal(o.N)
    r -= r.mean()
    zo = o.vcycle(r)
    assert _close(ps.hooks().vcycle(r), zo, 1e-9)
    assert _close(ps.hooks().vcycle(r, prec=1), zo, 1e-3)
    ps.destroy()
    o.close()
