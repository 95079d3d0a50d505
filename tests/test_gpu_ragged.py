"""The fine smoother on cells whose edges are no multiples of its tiles: the
tiles' overhang at every axis, both widths, one tile and several, alone (one
and three load cases per workgroup) and batched."""
import numpy as np
import pytest

import opentm_amd as otm

from test_gpu_components import make, rel, shape_of

pytestmark = pytest.mark.gpu

# resolution of a two-level cell, tile width
CELLS = [((10, 8, 8), 16), ((12, 12, 14), 16), ((16, 10, 8), 16), ((18, 10, 10), 32), ((20, 12, 14), 32),
         ((34, 12, 10), 16), ((46, 8, 12), 16), ((50, 8, 10), 32), ((64, 10, 8), 32), ((66, 14, 22), 16)]


def conductivity(reso):
    return np.random.default_rng(sum(reso)).uniform(1e-3, 1.0, reso[::-1]).astype(np.float32)


@pytest.mark.parametrize("reso,bx", CELLS)
def test_ragged_smoother_matches_block_restatement(orc, reso, bx):
    """The V-cycle of a two-level cell against its parts, with the oracle's
    block Gauss-Seidel (bx x 4 x 8 blocks cut at the edges) as the smoother
    (the pre-smoother runs the colours in the oracle's reverse order).
    Six FP32 parts, each held to 2e-6 by its own tests."""
    hom = make(reso, min_coarse=3)
    k = conductivity(reso)
    hom.update(k)
    assert len(hom.levels()) == 2 and hom.fine_tile()[0] == -1
    shape = shape_of(hom.levels()[0])
    n = int(np.prod(shape))
    A = orc.assemble(k.astype(np.float64) + 1e-9)
    r = np.random.default_rng(n).standard_normal((3, n)).astype(np.float32)
    r -= r.mean(axis=1, keepdims=True)
    z = orc.brick_gs(shape, A, r, np.zeros_like(r), (bx, 4, 8), sweeps=2, reverse=True).astype(np.float32)
    d = r.reshape(-1) - hom.apply_level(0, z.reshape(-1)).reshape(-1)
    z = hom.prolong_add(1, hom.coarsest_solve(hom.restrict(1, d)), z.reshape(-1))
    ref = orc.brick_gs(shape, A, r, z.reshape(3, n), (bx, 4, 8), sweeps=2)
    got = hom.vcycle(r.reshape(-1)).reshape(3, n)
    errs = [rel(got[c], ref[c]) for c in range(3)]
    print("[case] ragged", reso, "err", max(errs), flush=True)
    assert max(errs) < 2e-5


def test_ragged_cells_batched_are_the_single_cells():
    """Ragged cells of both widths with whole ones in one batch: the same
    bits as alone (104 x 88 x 48 takes three load cases per workgroup alone)."""
    cells = [(20, 24, 28), (12, 12, 12), (40, 48, 56), (32, 32, 32), (56, 24, 40), (104, 88, 48), (48, 16, 16)]
    homs = [make(reso) for reso in cells]
    kappas = [conductivity(reso) for reso in cells]
    alone = []
    for h, k in zip(homs, kappas):
        h.update(k)
        alone.append((h.heatMatrix(), h.get_chi(), h.solve_stats()[0]))
        h.reset_displacement()
    batch = otm.Batch()
    batch.update(homs, kappas)
    C = batch.heat_matrix(homs)
    for i, h in enumerate(homs):
        assert np.array_equal(np.asarray(C[i]), np.asarray(alone[i][0]))
        assert np.array_equal(h.get_chi(), alone[i][1])
        assert list(h.solve_stats()[0]) == list(alone[i][2])
    batch.close()
