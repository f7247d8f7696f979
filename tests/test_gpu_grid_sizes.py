"""ud2_scene_build_grids against the oracle's maps at the sizes where its blocks and receptor chunks end: axes one
point past a block and shorter than one, receptors of one atom and around a chunk of 1,024, one probe type and
all twenty (several radii, in an order of their own)."""
import dataclasses

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_rec,size,probes", [
    (1, (4.0, 2.5, 1.0), [4]),
    (1023, (6.0, 8.0, 4.5), [15, 2, 10, 4]),
    (1025, (8.0, 3.5, 6.0), [13, 1]),
    (2000, (3.5, 4.0, 8.0), list(range(20, 0, -1))),
])
def test_grid_sizes(gpu, receptor, n_rec, size, probes):
    from unidock_engine import topology as T
    print(f"grid maps: {n_rec} receptor atoms, box {size}, {len(probes)} types", flush=True)
    keep = np.argsort(np.linalg.norm(receptor.xyz - np.array([31.0, -3.0, 7.25], np.float32), axis=1), kind="stable")
    keep = np.sort(keep[:n_rec])  # the atoms nearest a point of the shell, in receptor order
    rec = dataclasses.replace(receptor, xyz=receptor.xyz[keep], types=receptor.types[keep])
    sc = gpu.Scene(rec, T.Box.from_center_size((29.0, -3.0, 7.25), size))
    sc.build_grids(0.5, probes)
    n, org, sp, nt = sc.grid_info()
    assert nt == len(probes)
    got = sc.download_maps()
    ref = O.grid_build(rec, n, org, sp, probes, nthreads=8)
    assert np.abs(ref).max() > 0.0
    err = np.abs(got.astype(np.float64) - ref) / np.maximum(np.abs(ref), 1.0)
    assert err.max() < 1e-5, err.max()
