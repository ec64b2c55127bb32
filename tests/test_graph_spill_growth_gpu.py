"""A pass captured after the caller has raised waves_per_cu: the traversals' spill area grows before the capture.

Workloads with more rays than the default grid holds at once (20 waves on each CU), so that 32 waves need a larger
area than the one that creating the object allocated.  Bar: captured passes equal eager ones, to the bit.
"""
import numpy as np
import pytest
import torch

from vermeer_amd import pathtrace, render, scenes

pytestmark = pytest.mark.gpu


def _junk():
    junk = torch.randn(4096, device="cuda").sum()   # the program's own work between replays
    torch.cuda.synchronize()
    assert torch.isfinite(junk)


@pytest.mark.parametrize("sort", [0, 4])
def test_render_pass(sort):
    W = 256
    desc = scenes.box_spheres_scene(nseg=16, nring=8)
    c = desc["camera"]
    cam = render.lookat_camera(c["from"], c["to"], c["up"], c["fov"], c["focal"], W, W)
    scr = torch.from_numpy(scenes.pixel_scrambles(W, W, seed=4).view(np.int64).reshape(-1).copy()).cuda()
    st = torch.cuda.current_stream().cuda_stream
    films = []
    for graph in (False, True):
        R = render.Renderer(desc, W, W, cam)
        R.scene.set_trace_config(64, 12, 32, sort=sort)
        film = torch.zeros(W * W * 3, device="cuda")
        print(f"[case] render graph={graph} sort={sort}", flush=True)
        for it in range(1, 5):
            R.render_pass_device(scr.data_ptr(), it, film.data_ptr(), stream=st, graph=graph)
            _junk()
        R.scene.status(st)
        films.append(film.cpu().numpy().tobytes())
        R.close()
    assert films[0] == films[1]


def test_path_pass():
    W = 640
    d = scenes.guided_room_scene(res=5, nboxes=500)
    st = torch.cuda.current_stream().cuda_stream
    sums = []
    for graph in (False, True):
        p = pathtrace.PathTracer(d, W, W, max_depth=3, seed=3)
        p.scene.set_trace_config(64, 12, 32)
        acc = torch.zeros(W * W * 3, dtype=torch.float64, device="cuda")
        print(f"[case] path graph={graph}", flush=True)
        for k in range(4):
            p.render_pass_device(acc.data_ptr(), k, stream=st, graph=graph)
            _junk()
        p.scene.status(st)
        sums.append(acc.cpu().numpy().tobytes())
        p.close()
    assert sums[0] == sums[1]
