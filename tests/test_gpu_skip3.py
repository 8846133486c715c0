"""Three transfers in one launch over skipped levels: the cycle against the
oracle's, which goes level by level, on boxes of odd and even lengths, periodic
and walled, all with a chain of three directions above the levels that run in one
workgroup. (Periodic directions are halved while their length is a multiple of 4,
so no level has an odd periodic length of three or more.) Tolerances as in
test_gpu_bottom.py; the bits are held in test_gpu_cycle_bits.py.
"""
import numpy as np
import pytest

from nga2_amd._lib import MIXED
from oracle.orc import Oracle
from test_gpu_cycle_bits import chains, relaxed
from test_gpu_parity import _box, _close, _solver

pytestmark = pytest.mark.gpu

SHAPES = [
    ((66, 50, 38), (False, False, False)),
    ((67, 49, 35), (False, False, False)),   # an odd last cell in every direction
    ((64, 64, 48), (True, True, True)),
    ((48, 64, 37), (True, True, False)),     # two periodic directions and a walled one
    ((37, 96, 64), (False, True, True)),
    ((130, 3, 130), (False, False, False)),  # a direction of three cells
]


@pytest.mark.parametrize("shape,per", SHAPES)
def test_cycle_matches_oracle(shape, per):
    print(f"\n[skip3 {shape} {per}]", flush=True)
    P = _box(*shape, per, walls=not all(per), L=tuple(n / max(shape) for n in shape))
    o = Oracle.from_cfg(P.cfg, P.opr, skip_relax=1, coarsest_max=20, nu_pre=1, nu_post=1)
    ps = _solver(P, precision=MIXED, nu_pre=1, nu_post=1, skip_relax=1, coarsest_max=20)
    hk = ps.hooks()
    # a chain whose two skipped levels lie above the bottom kernel's (at most 2048 cells)
    assert any(np.prod(hk.level_info(l + 2)[0]) > 2048 for l in chains(hk, relaxed(hk, 1)))
    rng = np.random.default_rng(3)
    r = rng.standard_normal(o.N)
    r -= r.mean()
    zo = o.vcycle(r)
    assert _close(hk.vcycle(r), zo, 1e-9)
    assert _close(hk.vcycle(r, prec=1), zo, 1e-3)
    ps.destroy()
    o.close()
