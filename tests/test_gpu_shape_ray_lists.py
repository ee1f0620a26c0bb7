"""Rays against their own shapes where the lists of rays on hulls and on capsules have their edges: counts
around a wavefront and a listing block, sets of one kind only, solid shapes and hollow ones (whose
rays from inside are cast again from behind), against the oracle bit for bit."""
import numpy as np
import pytest
import torch

import ncollide_amd as ncx
from ncollide_amd import workloads
from ncollide_amd.math import to_oracle_poses
from tests.test_gpu_parity import oracle_shapes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("solid", [True, False])
@pytest.mark.parametrize("types", [[0, 1, 2, 3], [3], [2], [0, 1], [1, 2]])
@pytest.mark.parametrize("n", [1, 63, 65, 1023, 1024, 1025, 4099])
def test_rays_listed_by_kind(ctx, orc, n, types, solid):
    rng = np.random.default_rng(n)
    w = workloads.full_pipeline(seed=21, n=800, box=20.0, nclusters=3)
    rec = w["records"][np.isin(w["records"]["type"], types)]
    poses = w["poses"][np.isin(w["records"]["type"], types)]
    idx = rng.integers(0, len(rec), n).astype(np.uint32)
    centre = poses[idx, :3]
    o = centre + workloads.unit_vectors(rng, n) * rng.choice([0.02, 0.2, 3.0], (n, 1))  # a third well inside
    d = np.where(rng.random((n, 1)) < 0.7, centre + rng.normal(0, 0.1, (n, 3)) - o, rng.normal(0, 1, (n, 3)))
    o, d = o.astype(np.float32), (d * rng.uniform(0.2, 3.0, (n, 1))).astype(np.float32)
    ss = ncx.ShapeSet(records=rec, pool=w["pool"], ctx=ctx)
    r = orc.shape_rays(oracle_shapes(orc, rec, w["pool"]), to_oracle_poses(poses), idx, o, d, np.float32(2.0), solid,
                       nthreads=8)
    g = ncx.query.cast_rays(ss, torch.as_tensor(poses, device=ctx.device), idx.astype(np.int32), o, d, 2.0, solid=solid)
    for name, a, b in zip(("toi", "normal", "feature"), g, r):
        assert np.array_equal(a.cpu().numpy().view(np.uint32), np.asarray(b).view(np.uint32)), name
    assert n < 1000 or ((r[0] >= 0).any() and (r[0] < 0).any() and (solid or (r[0][r[0] >= 0] > 0).any()))
