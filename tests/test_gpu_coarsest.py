"""The coarsest level's dense inverse and its product at the sizes where
their tiling changes: the one-workgroup inverse up to 64 nodes, the tiled
one above (tiles of 64, steps of 32 pivots, ragged last tile and step), alone
and batched, against numpy in FP64."""
import numpy as np
import pytest

import opentm_amd as otm

from test_gpu_components import make, shape_of
from test_oracle_mg import dense

pytestmark = pytest.mark.gpu

# (resolution, min_coarse): nodes of the coarsest level
CELLS = [((12, 12, 12), 3), ((8, 8, 8), 4), ((10, 8, 8), 4), ((12, 8, 8), 4), ((10, 10, 10), 4), ((16, 8, 8), 4),
         ((10, 12, 14), 4), ((18, 22, 14), 4), ((22, 22, 22), 4)]  # 27 64 80 96 125 128 210 693 1331


def conductivity(reso):
    rng = np.random.default_rng(sum(reso))
    return rng.uniform(1e-3, 1.0, reso[::-1]).astype(np.float32)


@pytest.mark.parametrize("reso,min_coarse", CELLS)
def test_coarsest_inverse_and_product(reso, min_coarse):
    """u = (K0 + tr/n^2 1 1^T)^-1 f. Everything is FP64 but the FP32 result:
    2^-24 relative, and 1e-16 times the condition number (below 1e5 here)."""
    hom = make(reso, min_coarse=min_coarse)
    hom.update(conductivity(reso))
    L = len(hom.levels()) - 1
    shape = shape_of(hom.levels()[L])
    n = int(np.prod(shape))
    K = dense(hom.stencil(L).astype(np.float64), shape)
    K = 0.5 * (K + K.T)
    K -= np.diag(np.diag(K))
    K -= np.diag(K.sum(axis=1))
    B = K + np.trace(K) / n ** 2
    f = np.random.default_rng(n).standard_normal((3, n)).astype(np.float32)
    u = hom.coarsest_solve(f).reshape(3, n).astype(np.float64)
    ref = np.linalg.solve(B, f.astype(np.float64).T).T
    err = np.abs(u - ref).max() / np.abs(ref).max()
    print("[case]", reso, "n", n, "err", err, flush=True)
    assert err < 2.0 ** -24 + 1e-11


def test_batched_inverse_is_the_single_cells():
    """Cells of every path in one batched setup: the same bits as alone."""
    homs = [make(reso, min_coarse=mc) for reso, mc in CELLS]
    kappas = [conductivity(reso) for reso, _ in CELLS]
    alone = []
    rng = np.random.default_rng(3)
    fs = []
    for h, k in zip(homs, kappas):
        h.update(k)
        n = int(np.prod(h.levels()[-1]))
        fs.append(rng.standard_normal((3, n)).astype(np.float32))
        alone.append(h.coarsest_solve(fs[-1]))
        h.update(np.ones_like(k))  # another inverse in between
    batch = otm.Batch()
    batch.update(homs, kappas)
    for h, f, a in zip(homs, fs, alone):
        assert np.array_equal(h.coarsest_solve(f), a)
    batch.close()


@pytest.mark.parametrize("fp16", [0, 1])
@pytest.mark.parametrize("reso,min_coarse", [((16, 16, 16), 4), ((12, 12, 12), 3), ((12, 12, 28), 3), ((28, 12, 12), 3),
                                             ((12, 16, 20), 3)])
def test_tail_is_its_parts(reso, min_coarse, fp16):
    """The V-cycle whose last two levels run in the one-workgroup tail (8^3
    and edges that are no power of two, whose rows wrap inside a wave) against
    the same V-cycle put together from the level entry points. About ten
    FP32 parts, each held to 2e-6 by its own tests."""
    hom = make(reso, min_coarse=min_coarse, exact_smoother=1, fp16_stencils=fp16)
    hom.update(conductivity(reso))
    assert len(hom.levels()) == 3
    n = int(np.prod(reso))
    r = np.random.default_rng(n).standard_normal((3, n)).astype(np.float32)
    r -= r.mean(axis=1, keepdims=True)
    r = r.reshape(-1)
    z = hom.smooth_level(0, r, np.zeros_like(r), sweeps=2, mode=0)
    f1 = hom.restrict(1, r - hom.apply_level(0, z))
    u1 = hom.smooth_level(1, f1, np.zeros_like(f1), sweeps=2, mode=0)
    u1 = hom.prolong_add(2, hom.coarsest_solve(hom.restrict(2, f1 - hom.apply_level(1, u1))), u1)
    u1 = hom.smooth_level(1, f1, u1, sweeps=2, mode=1)
    z = hom.smooth_level(0, r, hom.prolong_add(1, u1, z), sweeps=2, mode=1)
    got = hom.vcycle(r)
    err = np.abs(got - z).max() / np.abs(z).max()
    print("[case] tail", reso, "fp16", fp16, "err", err, flush=True)
    assert err < 2e-5
