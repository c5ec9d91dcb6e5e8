"""Ray counts at the edges of the persistent kernels' item fetch: one wave and
its neighbours, one workgroup, less and more than the resident lanes, and
counts that leave the last claimed chunk partly filled.  Ids, distances and
occlusion against the kernels' per-ray code on host threads (itself compared
with the oracle in test_host_traversal.py), bit for bit."""
import numpy as np
import pytest
import torch

from rise_amd import raycast, scenes
from tests.conftest import log_case

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def scene(cuda):
    tris = scenes.soup_triangles(6000, seed=11, sigma=0.02)
    om = raycast.ObjectManager()
    om.add_mesh(tris)
    om.prepare_for_rendering()
    rays = scenes.incoherent_rays(700_001, 12)
    far = np.random.default_rng(13).uniform(0.01, 1.0, rays.shape[1]).astype(np.float32)
    pid, t, _, _ = raycast.host_trace(tris, rays)
    occ, _, _ = raycast.host_trace(tris, rays, mode=1, tmax=far)
    yield om, rays, far, pid, t, occ
    om.release()


@pytest.mark.parametrize("n", [1, 7, 63, 64, 65, 127, 129, 4097, 327_679, 327_681, 700_001])
def test_gpu_ray_counts(cuda, scene, n):
    log_case(f"n={n}")
    om, rays, far, pid, t, occ = scene
    r = torch.from_numpy(np.ascontiguousarray(rays[:, :n])).to(cuda)
    gp, gt = om.intersect_ray(r)
    assert np.array_equal(gp.cpu().numpy(), pid[:n])
    assert np.array_equal(gt.cpu().numpy(), t[:n])
    go = om.intersect_shadow_ray(r, torch.from_numpy(far[:n].copy()).to(cuda))
    assert np.array_equal(go.cpu().numpy(), occ[:n])
