"""The skinny product over more row tiles than the chip holds at once (a head's rows): every tile once
whatever the tiles leave over a round of workgroups, ragged last tiles, the packed second column tile's edge (24 rows),
narrow K (several workgroups a CU) and K in two ranges (the second adds to the first's sums)."""
import numpy as np
import pytest

import pyoracle as po

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols,M,add", [
    (16400, 2048, 17, False), (16401, 2048, 24, False), (16640, 2048, 25, False), (32771, 2048, 32, False),
    (16400, 2048, 1, False), (16401, 2048, 8, False), (32784, 2048, 9, False), (32771, 2048, 16, False),
    (16400, 6144, 5, False), (65552, 512, 4, False), (131104, 128, 3, False), (17000, 2048, 5, True),
    (70000, 512, 17, False), (131104, 128, 18, True), (20496, 4096, 24, False), (17000, 2048, 17, True)])
def test_gemv_many_tiles(rows, cols, M, add):
    import geode_amd as gv

    gv.init(0)
    wq, s2 = po.q4_random(31 + rows + cols, rows, cols)
    m = gv.Q4Matrix(wq, rows, cols, s2)
    x = po.normal(41 + M, M * cols, 1.0).reshape(M, cols)
    base = po.normal(79, M * rows).reshape(M, rows) if add else None
    got = gv.gemv(m, x, accumulate_into=base)
    want = np.stack([po.matvec_q(wq, cols, s2, x[t]) for t in range(M)])
    if add:
        want = base + want
    # the integer block sums are exact; cols / 16 of them in fp32 in another order: the bound of the other products' tests
    assert np.abs(got - want).max() <= 1e-5 * np.abs(want).max()
