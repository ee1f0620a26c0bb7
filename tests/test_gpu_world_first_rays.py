"""First hits of world rays where the traversal's scheduling has its edges: worlds of one and two
proxies, ray counts around a wavefront, a block and a refill, and a crowd in which every ray
reaches many capsules and hulls (more than a lane keeps, so that leaves go back onto its stack).
The oracle casts every shape whose stored box the ray enters and takes the least (toi, handle)."""
import numpy as np
import pytest
import torch

import ncollide_amd as ncx
from ncollide_amd import workloads
from ncollide_amd.math import to_oracle_poses
from ncollide_amd.world import World
from tests.test_gpu_parity import oracle_shapes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nshapes,nrays,box", [(1, 1, 1.0), (1, 63, 1.0), (2, 65, 1.0), (3, 129, 1.0),
                                               (400, 1, 4.0), (400, 127, 2.0), (400, 3000, 2.0),
                                               (2000, 100003, 12.0)])
def test_world_first_rays_edges(ctx, orc, nshapes, nrays, box):
    w = workloads.full_pipeline(seed=50 + nshapes, n=nshapes, box=box, nclusters=1)
    ss = ncx.ShapeSet(records=w["records"], pool=w["pool"], ctx=ctx)
    world = World(ss, margin=0.05, prediction=0.0, max_pairs=1 << 18)
    p = w["poses"]
    poses = torch.as_tensor(p, device=ctx.device)
    world.step(poses)
    world.sync()
    stored = world.stored_aabbs().cpu().numpy().T.copy()
    rng = np.random.default_rng(nrays)
    tgt = p[rng.integers(0, nshapes, nrays), :3]
    ro = (tgt + rng.normal(0, 3, (nrays, 3))).astype(np.float32)
    ro[::5] = tgt[::5]  # from inside
    rd = ((tgt - ro) * rng.uniform(0.2, 1.5, (nrays, 1))).astype(np.float32)
    rd[::5] = rng.normal(size=(len(rd[::5]), 3)).astype(np.float32)
    oss = oracle_shapes(orc, w["records"], w["pool"])
    rh, rt, rn = orc.world_rays(oss, to_oracle_poses(p), stored, ro, rd, np.float32(20.0), 0)
    for o, d in ((ro, rd), (torch.as_tensor(ro, device=ctx.device), torch.as_tensor(rd, device=ctx.device))):
        h, t, n = world.first_interference_with_rays(poses, o, d, 20.0)
        assert np.array_equal(h.cpu().numpy().view(np.uint32), rh)
        assert np.array_equal(t.cpu().numpy().view(np.uint32), rt.view(np.uint32))
        assert np.array_equal(n.cpu().numpy().view(np.uint32), rn.view(np.uint32))
