"""The density filter's tile kernel at the edges of its tiles (32 x 8 x 4 and
32 x 8 x 8 outputs), for every reach of the taps, and on cells too short for
the weight sums' distance classes, against the oracle's FP64 loops."""
import numpy as np
import pytest

import opentm_amd as otm

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (3, 2, 1), (3, 4, 5), (4, 8, 32), (5, 9, 33), (9, 7, 31), (8, 17, 65), (96, 90, 70)]


@pytest.mark.parametrize("kind", [0, 1])
@pytest.mark.parametrize("radius,reach", [(0.7, 0), (1.5, 1), (2.5, 2), (3.4, 3)])
@pytest.mark.parametrize("periodic", [False, True])
def test_filter_tiles(orc, kind, radius, reach, periodic):
    """Sums of at most 171 positive terms in FP32: held to the 2e-6 of the
    other filter tests."""
    rng = np.random.default_rng(17)
    for shape in SHAPES:  # (nz, ny, nx)
        if reach > min(shape):
            continue
        x = rng.uniform(0.05, 1.0, shape).astype(np.float32)
        for adjoint in (False, True):
            got = otm.conv_filter(x, kind, radius, periodic, adjoint=adjoint)
            ref = (orc.filter_adj if adjoint else orc.filter_fwd)(x, kind, radius, periodic)
            err = float(np.abs(got - ref).max() / np.abs(ref).max())
            print("[case]", shape, kind, radius, periodic, adjoint, err, flush=True)
            assert err < 2e-6
