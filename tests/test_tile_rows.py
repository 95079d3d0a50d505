"""The fine post-smoother's r.z partial sums: a row per tile in a buffer of
at most 65536 rows, so a cell of more tiles forms r.z apart, alone and
batched."""
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_rows_cover_the_tiles_of_every_cell(tmp_path):
    from opentm_amd.build import HIPCC, HIPFLAGS
    exe = tmp_path / "rows"
    flags = [f for f in HIPFLAGS if f not in ("-Xclang", "-target-feature", "-packed-fp32-ops")]
    r = subprocess.run([HIPCC] + flags + ["-x", "hip", "--offload-host-only", "-I",
                                          os.path.join(ROOT, "opentm_amd", "csrc"),
                                          os.path.join(ROOT, "tests", "cxx", "tile_rows_check.cpp"), "-o", str(exe)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120).stdout.splitlines()
    rows = [line.split() for line in out]
    cells, fused, apart, bad = (int(v) for v in rows[0][1:])
    assert cells == 509 ** 3 and fused > 0 and apart > 0
    assert bad == 0
    cubes = {int(n): (int(t), int(have), int(ok)) for _, n, t, have, ok in rows[1:]}
    assert cubes[256] == (16384, 32769, 1)       # 256^3 / 1024 tiles, one row per 512 nodes
    assert cubes[400] == (125000, 65536, 0)      # 16-wide tiles
    assert cubes[384] == (55296, 65536, 1)
    assert cubes[416] == (70304, 65536, 0)
    assert cubes[512] == (131072, 65536, 0)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [160, 416])
def test_batched_cell_forms_rz_as_alone(n):
    """160^3 (4000 tiles): r.z from the post-smoother, more rows than the
    final sum's slots. 416^3 (70304 tiles): no row for each tile, r.z in a
    pass of its own. Batched as alone: the same iterations and tensor."""
    import opentm_amd as otm
    from test_gpu_components import make
    reso = (n, n, n)
    hom = make(reso)
    k = np.random.default_rng(n).random(reso, dtype=np.float32) * np.float32(0.9) + np.float32(0.1)
    hom.update(k)
    alone, its = np.asarray(hom.heatMatrix()), list(hom.solve_stats()[0])
    print("[case] alone", n, its, flush=True)
    hom.reset_displacement()
    batch = otm.Batch()
    batch.update([hom], [k])
    got = np.asarray(batch.heat_matrix([hom])[0])
    print("[case] batched", list(hom.solve_stats()[0]), flush=True)
    batch.close()
    assert list(hom.solve_stats()[0]) == its
    assert np.array_equal(got, alone)
