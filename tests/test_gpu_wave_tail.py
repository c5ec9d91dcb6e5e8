"""The ends of traversal launches, where eight lanes share a ray, and launches
of so few rays that they start that way: ray counts around a wave's share (8),
a workgroup's (16) and the resident lanes' (the line to one lane a ray lies
where a device's lanes / 8 run out), with coincident triangles of equal
distance (lower id wins, over slots, lanes and leaves of several triangles),
axis-parallel rays and rays in the triangles' planes.  Ids, distances and
occlusion against the kernels' per-ray code on host threads, bit for bit."""
import numpy as np
import pytest
import torch

from rise_amd import raycast, scenes
from tests.conftest import log_case

pytestmark = pytest.mark.gpu

N = 41_000  # more than 2560 workgroups' 16 rays


def _grid_of_copies():
    """Axis-aligned quads on a lattice, each three times, and a soup around them."""
    g = np.random.default_rng(21)
    c = np.stack(np.meshgrid(*[np.arange(9) / 8.0] * 3, indexing="ij"), -1).reshape(-1, 3)
    quads = np.concatenate([np.concatenate([c, c + a, c + b], 1) for a, b in
                            (((.1, 0, 0), (0, .1, 0)), ((0, .1, 0), (0, 0, .1)))])
    tris = np.concatenate([quads] * 3 + [scenes.soup_triangles(3000, seed=22, sigma=0.03).reshape(-1, 9)])
    return np.ascontiguousarray(tris[g.permutation(len(tris))], np.float32)


def _rays():
    g = np.random.default_rng(23)
    o = g.uniform(-0.2, 1.2, (N, 3))
    d = g.normal(size=(N, 3))
    axis = g.integers(0, 3, N)
    par = np.arange(N) % 3 == 0
    d[par] = np.eye(3)[axis[par]] * g.choice([-1.0, 1.0], par.sum())[:, None]
    lat = np.arange(N) % 6 == 0
    o[lat] = g.integers(-1, 10, (lat.sum(), 3)) / 8.0 + 0.05 * g.integers(0, 2, (lat.sum(), 3))
    return scenes.rays_from_rows(o, d)


@pytest.fixture(scope="module")
def scene(cuda):
    tris, rays = _grid_of_copies(), _rays()
    om = raycast.ObjectManager()
    om.add_mesh(tris)
    om.prepare_for_rendering()
    far = np.random.default_rng(24).uniform(0.01, 1.0, N).astype(np.float32)
    pid, t, _, _ = raycast.host_trace(tris, rays)
    occ, _, _ = raycast.host_trace(tris, rays, mode=1, tmax=far)
    assert 0.2 < (pid >= 0).mean() < 1.0
    yield om, rays, far, pid, t, occ
    om.release()


@pytest.mark.parametrize("n", [1, 2, 7, 8, 9, 15, 16, 17, 33, 1000, 40_959, 40_960, 40_961, N])
def test_gpu_few_rays(cuda, scene, n):
    log_case(f"n={n}")
    om, rays, far, pid, t, occ = scene
    # The last n rays, so that every count meets other rays.
    r = torch.from_numpy(np.ascontiguousarray(rays[:, N - n:])).to(cuda)
    gp, gt = om.intersect_ray(r)
    assert np.array_equal(gp.cpu().numpy(), pid[N - n:])
    assert np.array_equal(gt.cpu().numpy(), t[N - n:])
    go = om.intersect_shadow_ray(r, torch.from_numpy(far[N - n:].copy()).to(cuda))
    assert np.array_equal(go.cpu().numpy(), occ[N - n:])


@pytest.mark.parametrize("faces", [raycast.FACES_FRONT, raycast.FACES_BACK, raycast.FACES_BOTH])
@pytest.mark.parametrize("arith", [raycast.ARITH_IEEE, raycast.ARITH_X86_FMA])
@pytest.mark.parametrize("vertices", [np.float32, np.float64])
def test_gpu_few_rays_forms(cuda, vertices, arith, faces):
    """The same ends under a face selection, with records, double vertices (off the float grid) and both arithmetic
    models, against the per-ray code of a scene with one identity object on host threads."""
    tris, rays = _grid_of_copies().astype(vertices), _rays()
    if vertices is np.float64:
        tris *= 1.0 + np.random.default_rng(25).uniform(-1e-9, 1e-9, tris.shape)
    far = np.random.default_rng(24).uniform(0.01, 1.0, N).astype(np.float32)
    objs = raycast.make_objects([(0, *raycast.object_matrices())])
    want = raycast.host_trace_objects([tris], objs, rays, faces=faces, arith=arith)
    occ = raycast.host_trace_objects([tris], objs, rays, mode=1, faces=faces, tmax=far, arith=arith)
    hit = want["prim_id"] >= 0
    assert 0.1 < hit.mean() < 1.0
    om = raycast.ObjectManager(arith)
    om.add_mesh(tris)
    om.prepare_for_rendering()
    for n in (1, 7, 8, 9, 15, 16, 17, 33, 1000, 40_959, 40_961, N):
        log_case(f"{vertices.__name__} {arith} faces {faces} n={n}")
        r = torch.from_numpy(np.ascontiguousarray(rays[:, N - n:])).to(cuda)
        g, h = raycast.hit_fields(om.intersect_ray_ex(r, faces)), hit[N - n:]
        assert np.array_equal(g["prim_id"], want["prim_id"][N - n:])
        for field in ("range", "alpha", "beta", "point", "geom_normal"):
            assert np.array_equal(g[field][h], want[field][N - n:][h]), field
        go = om.intersect_shadow_ray_ex(r, faces, torch.from_numpy(far[N - n:].copy()).to(cuda))
        assert np.array_equal(go.cpu().numpy(), occ[N - n:])
        if faces == raycast.FACES_BOTH:
            gp, gt = om.intersect_ray(r)
            assert np.array_equal(gp.cpu().numpy(), want["prim_id"][N - n:])
            assert np.array_equal(gt.cpu().numpy()[h], want["range"][N - n:][h].astype(np.float32))
    om.release()
