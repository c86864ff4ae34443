"""The reference's noise stream at the sizes where its parallel generation can go wrong: grids of
one row, self-conjugate planes of odd and even sizes, both parities of the row's last cell, many
seeds (normals that straddle chunk boundaries by far), and a grid whose normals need more groups
of chunks than are chained at a time.  The stream is defined bit for bit, so is the test."""
import numpy as np
import pytest

import crava_amd as C
import oracle as O

pytestmark = pytest.mark.gpu

# the last one draws 17.3 M normals: 132 groups and more, past the 128 that are chained at a time
SHAPES = [(1, 5, 4), (2, 3, 2), (3, 4, 5), (5, 8, 6), (6, 1, 9), (7, 9, 1), (64, 30, 33), (31, 64, 128),
          (352, 256, 192)]


@pytest.mark.parametrize("shape", SHAPES)
def test_reference_noise_edges(ctx, shape):
    nxp, nyp, nzp = shape
    print("reference noise", shape, flush=True)
    g = C.FFTGrid(ctx, nxp, nyp, nzp, nxp, nyp, nzp, C.PARAMETER)
    cells = nxp * nyp * nzp
    for seed in (0, 23665, 4294967295) if cells > 1 << 20 else [7919 * k for k in range(24)]:
        state = np.array([seed], dtype=np.uint32)
        after = g.fillInComplexNoiseReference(seed)
        want = O.fill_complex_noise(nxp, nyp, nzp, state)
        assert np.array_equal(g.download_complex().view(np.uint32), want.view(np.uint32)), seed
        assert after == int(state[0]), seed
    g.close()
