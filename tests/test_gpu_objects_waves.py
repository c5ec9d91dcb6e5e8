"""Object queries at the edges of their kernels' forms: trees whose node-group
stacks fit the small LDS stack and the large one only
(meshes at geometric scales, 13 and 20 levels), with and without a world tree
and with a world tree alone, so that lanes of one wave meet in every mix of
phases; ray counts about a wave, a workgroup and the refill line.  Hits and
occlusion against the oracle, bit for bit."""
import numpy as np
import pytest
import torch

import oracle
from rise_amd import raycast, scenes
from tests.conftest import log_case
from tests.test_gpu_objects import _manager, _tmax

pytestmark = pytest.mark.gpu


def _scales(n, seed):
    g = np.random.default_rng(seed)
    s = 1.3 ** -np.arange(float(n)).repeat(20)[:, None]
    c = s * g.uniform(0.7, 1.0, (len(s), 3))
    e1, e2 = g.normal(0, 0.1, (2, len(s), 3)) * s
    return np.ascontiguousarray(np.concatenate([c, c + e1, c + e2], 1), np.float32)


@pytest.mark.parametrize("arith", ["ieee", "fast"])
@pytest.mark.parametrize("levels,n_objects,n_identity", [(0, 9, 2), (60, 6, 1), (110, 6, 1), (110, 4, 0), (0, 2, 2), (0, 1, 0)])
def test_gpu_object_waves(cuda, levels, n_objects, n_identity, arith):
    meshes, objs = scenes.instanced_scene(2, n_objects, 1500, seed=41, n_identity=n_identity)
    if levels:
        meshes[0] = _scales(levels, 42)
    rays = scenes.object_rays(meshes, objs, 4097, seed=43)
    tmax = _tmax(rays.shape[1], 44)
    om = _manager(meshes, objs, {"ieee": raycast.ARITH_IEEE, "fast": raycast.ARITH_X86_FMA}[arith])
    o = oracle.objects_closest(meshes, objs, rays, arith=arith)
    occ = oracle.objects_any(meshes, objs, rays, tmax, arith=arith)
    assert 0.2 < (o["prim_id"] >= 0).mean() < 1.0
    for n in (1, 9, 55, 57, 64, 65, 129, rays.shape[1]):
        log_case(f"{n_objects} objects, {levels} scales, {arith}, n={n}")
        r = torch.from_numpy(np.ascontiguousarray(rays[:, :n])).to(cuda)
        g = raycast.hit_fields(om.intersect_ray_ex(r, raycast.FACES_BOTH))
        hit = o["prim_id"][:n] >= 0
        assert np.array_equal(g["prim_id"], o["prim_id"][:n]) and np.array_equal(g["mesh"], o["object"][:n])
        assert np.array_equal(g["range"][hit], o["range"][:n][hit])
        assert np.array_equal(g["point"][hit], o["point"][:n][hit].astype(np.float32))
        pid, t = om.intersect_ray(r)
        assert np.array_equal(pid.cpu().numpy(), g["prim_id"])
        assert np.array_equal(t.cpu().numpy(), g["range"].astype(np.float32))
        got = om.intersect_shadow_ray(r, how_far=torch.from_numpy(tmax[:n].copy()).to(cuda))
        assert np.array_equal(got.cpu().numpy(), occ[:n])
    om.release()
