"""Which launches a batch consists of under its tuning, counted in its captured
graph: a small batch of automatic shapes is a few launches (k_finish); one with
a chosen workgroup size, stack or schedule launches every bounce's kernels in
that shape, so the choice has its effect whatever the batch's size."""
import ctypes
import dataclasses

import numpy as np
import pytest
import torch

from rise_amd import _lib, pt_scene
from rise_amd.render import PathTracingSpectralRasterizer, RenderBatch
from tests.conftest import log_case

pytestmark = pytest.mark.gpu


def _launches(batch):
    g = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(g):
        batch.launch()
    n = ctypes.c_size_t(0)
    assert _lib.lib().hipGraphGetNodes(ctypes.c_void_p(g.raw_cuda_graph()), None, ctypes.byref(n)) == 0
    return n.value


def test_gpu_tuning_launches(cuda):
    s, r = pt_scene.cornell_box()
    rast = PathTracingSpectralRasterizer(s)
    q = dataclasses.replace(r, width=40, height=30, spp=2, seed=3)  # 6 bounces
    films = []
    for tuning, few in ((None, True), ({"max_paths": 1 << 20}, True), ({"persistent": 1}, False),
                        ({"persistent": 2}, False), ({"trace_block": 64}, False), ({"stack": 16}, False),
                        ({"stack": -1}, False)):
        log_case(f"{tuning}")
        b = RenderBatch([(rast, q)], tuning=tuning)
        b.launch()
        torch.cuda.synchronize()
        films.append(b.films[0].cpu().numpy())
        n = _launches(b)
        assert n <= 7 if few else n >= 6 + 6 * 4, (tuning, n)
        b.release()
    assert films[0].any() and all(np.array_equal(f, films[0]) for f in films)
    rast.release()
