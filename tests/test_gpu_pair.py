"""The fused pair of FP32 sweeps with two cells per lane against the one-cell
form on every level of boxes at the edges of its tiles (output core 56 x 24
cells, chunks of whole 6 planes): cores filled exactly, one pair or row more,
boxes smaller than the ring, directions of two cells, periodic and walled. Both
issue the same operations in the same order: the same bits. (Levels with odd
rows, one plane or one periodic cell in y or z have the one-cell form only.)
"""
import numpy as np
import pytest

from nga2_amd._lib import MIXED
from test_gpu_parity import _box, _solver

pytestmark = pytest.mark.gpu

SHAPES = [
    ((56, 24, 6), (False, False, False)),
    ((58, 25, 7), (False, False, False)),
    ((112, 49, 13), (True, False, False)),
    ((64, 32, 12), (True, True, True)),
    ((2, 2, 2), (True, True, True)),
    ((2, 3, 2), (False, False, False)),
    ((6, 4, 34), (False, True, True)),
    ((62, 8, 5), (False, True, False)),
    ((200, 70, 40), (False, False, True)),
    ((30, 6, 8), (False, True, True)),       # 6 periodic rows: a tile wraps around the box five times
    ((48, 64, 24), (True, True, False)),     # periodic directions that coarsen
]


@pytest.mark.parametrize("shape,per", SHAPES)
def test_pair_matches_one_cell_form(shape, per):
    print(f"\n[pair {shape} {per}]", flush=True)
    P = _box(*shape, per, walls=not all(per), L=tuple(n / max(shape) for n in shape))
    ps = _solver(P, precision=MIXED, coarsest_max=20)
    hk = ps.hooks()
    rng = np.random.default_rng(5)
    for l in range(hk.nlevels):
        n = int(np.prod(hk.level_info(l)[0]))
        f, x = rng.standard_normal(n), rng.standard_normal(n)
        for order in (0, 1):
            for pair in (4, 6):
                got = hk.rbgs(l, f, x, pair | order, prec=1)
                want = hk.rbgs(l, f, x, 8 | pair | order, prec=1)
                assert np.isfinite(want).all()
                assert np.array_equal(got, want), (l, order, pair)
    ps.destroy()
