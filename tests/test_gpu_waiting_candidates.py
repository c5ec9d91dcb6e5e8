"""Closest hits on scenes in units of hundreds (test_waiting_candidates.py: the
pre-filter's range test decides between triangles at or near one distance), where
a ray's id and distance are those of one lane that certifies each candidate at
once, whatever rays share its wave and its launch: few rays (eight lanes each),
many, permuted ones; plain, counted, record and allocation-free queries; float
and double vertices; objects; and films of small passes, large ones and one
ray a thread."""
import dataclasses

import numpy as np
import pytest
import torch

from rise_amd import _lib, pt_scene, raycast, scenes
from rise_amd.render import PathTracingSpectralRasterizer, RenderBatch
from tests.conftest import log_case
from tests.test_waiting_candidates import SCENES, copies_tris

pytestmark = pytest.mark.gpu

N = 60_000


@pytest.mark.parametrize("arith", [raycast.ARITH_IEEE, raycast.ARITH_X86_FMA])
@pytest.mark.parametrize("vertices", [np.float32, np.float64])
@pytest.mark.parametrize("extent", [100.0, 1000.0])
@pytest.mark.parametrize("name", sorted(SCENES))
def test_gpu_waiting_world(cuda, name, extent, vertices, arith):
    make_tris, make_rays = SCENES[name]
    tris, rays = make_tris(extent), make_rays(extent, N, 5)
    om = raycast.ObjectManager(arith)
    om.add_mesh(tris.astype(vertices))  # the same triangles, so the same hits
    om.prepare_for_rendering()
    pid, t, _, _ = raycast.host_trace(tris, rays, arith=arith)
    perm = np.random.default_rng(6).permutation(N)
    for n, order in ((1, slice(0, 1)), (7, slice(0, 7)), (1000, slice(0, 1000)), (17_001, slice(0, 17_001)),
                     (N, slice(0, N)), (N, perm)):
        log_case(f"{name} {extent} {vertices.__name__} {arith} n={n}")
        r = torch.from_numpy(np.ascontiguousarray(rays[:, order])).to(cuda)
        gp, gt = om.intersect_ray(r)
        assert np.array_equal(gp.cpu().numpy(), pid[order]), (gp.cpu().numpy() != pid[order]).sum()
        assert np.array_equal(gt.cpu().numpy(), t[order])
        cp, ct = om.intersect_ray(r, counters=torch.zeros(2, dtype=torch.int64, device=cuda))
        assert torch.equal(cp, gp) and torch.equal(ct, gt)
        h = raycast.hit_fields(om.intersect_ray_ex(r, raycast.FACES_BOTH))
        assert np.array_equal(h["prim_id"], pid[order])
        assert np.array_equal(h["range"].astype(np.float32), t[order])
        np_, nt = torch.empty_like(gp), torch.empty_like(gt)
        _lib.check(_lib.lib().rise_hip_intersect_closest_noalloc(om.handle, r.data_ptr(), n, np_.data_ptr(),
                                                                 nt.data_ptr(), None))
        torch.cuda.synchronize()
        assert torch.equal(np_, gp) and torch.equal(nt, gt)
    om.release()


@pytest.mark.parametrize("n_identity", [0, 2])
def test_gpu_waiting_objects(cuda, n_identity):
    meshes, objs = scenes.instanced_scene(2, 6, 10, seed=41, n_identity=n_identity)
    meshes = [copies_tris(2.0, 2000, 7 + k) - np.float32(1.0) for k in range(2)]
    scale = 500.0
    for o in objs:  # every object 500 times as far and as large
        tw = np.array(o["to_world"], np.float64).reshape(4, 4)
        tw[3, :3] *= scale
        o["to_world"] = tw.reshape(o["to_world"].shape)
        to = np.array(o["to_object"], np.float64).reshape(4, 4)
        to[3, :3] *= scale
        o["to_object"] = to.reshape(o["to_object"].shape)
    meshes = [np.ascontiguousarray(m * np.float32(scale)) for m in meshes]
    rays = scenes.object_rays(meshes, objs, N, seed=43, spread=6.0 * scale)
    want = raycast.host_trace_objects(meshes, objs, rays)
    assert (want["prim_id"] >= 0).mean() > 0.3
    om = raycast.ObjectManager(raycast.ARITH_IEEE)
    for m in meshes:
        om.add_mesh(m)
    for ob in objs:
        om.add_object(int(ob["mesh"]), ob["to_world"], ob["to_object"])
    om.prepare_for_rendering()
    for n in (1, 65, 20_000, N):
        log_case(f"objects, {n_identity} identity, n={n}")
        r = torch.from_numpy(np.ascontiguousarray(rays[:, :n])).to(cuda)
        g = raycast.hit_fields(om.intersect_ray_ex(r, raycast.FACES_BOTH))
        for field in ("prim_id", "mesh", "range"):
            assert np.array_equal(g[field], want[field][:n]), (field, (g[field] != want[field][:n]).sum())
    om.release()


def test_gpu_waiting_films(cuda):
    s, r = pt_scene.cornell_box()
    extent = 1000.0
    tris = copies_tris(extent, 3000, 9)
    s.objects = [pt_scene.Object(np.ascontiguousarray(tris[k::3]), k, double_sided=True) for k in range(3)]
    s.objects.append(pt_scene.Object(pt_scene.quad(*[tuple(extent * np.array(p)) for p in
                                                    ((0, 1.5, 0), (1, 1.5, 0), (1, 1.5, 1), (0, 1.5, 1))]), 3))
    s.camera = dataclasses.replace(s.camera, position=(1.8 * extent, 0.6 * extent, 1.9 * extent),
                                   look_at=(0.5 * extent,) * 3)
    rast = PathTracingSpectralRasterizer(s)
    small = dataclasses.replace(r, width=96, height=80, spp=2, seed=3)
    big = dataclasses.replace(r, width=512, height=512, spp=1, seed=4)
    films = {}
    for label, reqs, tuning in (("alone", [small], None), ("with 512x512", [small, big], None),
                                ("one ray a thread", [small, big], {"persistent": 2})):
        log_case(label)
        b = RenderBatch([(rast, q) for q in reqs], tuning=tuning)
        b.launch()
        torch.cuda.synchronize()
        films[label] = [f.cpu().numpy() for f in b.films]
        b.release()
    assert films["alone"][0].any()
    assert np.array_equal(films["alone"][0], films["with 512x512"][0])
    for a, b in zip(films["with 512x512"], films["one ray a thread"]):
        assert np.array_equal(a, b)
    rast.release()
