"""The scene's ray sort on the shading passes' shadow rays, which are traced from a list of the slots in use.

Workload: the feature scene (mirrors, two lights: four levels of shadow rays a pass) at an odd size and at one with
more listed rays than a wavefront grid holds at once.  Bars: the sort runs (its share of the scene's timing is that of
its five launches, against two adjacent events without it), and film, sample and shadow-ray count equal the oracle's,
whose renderer knows no list, for each grid size; a captured pass with the sort replays to the same bits.
"""
import numpy as np
import pytest
import torch

import oracle
import vermeer_amd as va
from vermeer_amd import render, scenes

pytestmark = pytest.mark.gpu


def _scene(w, h):
    desc = scenes.feature_scene(nseg=24, nring=12)
    c = desc["camera"]
    M, ttf = oracle.camera_lookat(c["from"], c["to"], c["up"], c["fov"], c["focal"])
    cam = np.zeros((), va._lib.CAMERA_DTYPE)
    cam["M"], cam["tan_theta_focal"], cam["aspect"], cam["focal"] = M, ttf, w / h, c["focal"]
    return desc, cam, M, ttf


@pytest.mark.parametrize("w,h", [(37, 29), (160, 121)])
def test_sorted_shadow_rays_match_the_oracle(w, h):
    oracle.set_normalize_ieee(True)
    try:
        desc, cam, M, ttf = _scene(w, h)
        R = render.Renderer(desc, w, h, cam)
        o = oracle.OracleRenderer(desc, w, h, M, ttf, desc["camera"]["focal"])
        scr = scenes.pixel_scrambles(w, h)
        for it, sort in ((1, 0), (2, 3), (3, 6)):
            print(f"[case] {w}x{h} sort {sort}", flush=True)
            R.scene.set_trace_config(64, 12, 20, sort=sort)
            n, samp = R.render_pass(scr, it, want_sample=True)
            m, ref = o.render_pass(scr, it, want_sample=True)
            assert n == m > 0
            a, b = samp.view(np.uint32), np.ascontiguousarray(ref, np.float32).view(np.uint32)
            assert np.all((a == b) | (np.isnan(samp) & np.isnan(ref)))
        R.close()
    finally:
        oracle.set_normalize_ieee(False)


def test_the_sort_runs_on_listed_rays():
    w, h = 160, 121
    desc, cam, _, _ = _scene(w, h)
    R = render.Renderer(desc, w, h, cam)
    scr = scenes.pixel_scrambles(w, h)
    share = {}
    for sort in (0, 5):
        R.scene.set_trace_config(64, 12, 20, sort=sort)
        R.render_pass(scr, 1)
        R.scene.set_timing(True)
        R.render_pass(scr, 2)
        trace, took, launches = R.scene.timing()
        R.scene.set_timing(False)
        assert launches == 4 and trace > 0   # one listed trace a level
        share[sort] = took / launches
    print(f"[case] sort a launch: {share[0] * 1e3:.1f} us without, {share[5] * 1e3:.1f} us with", flush=True)
    # five launches one after another, 2 us at least each, against two events with nothing between
    assert share[5] > 0.010 and share[5] > 2 * share[0]
    R.close()


def test_a_captured_pass_sorts():
    w, h = 96, 64
    desc, cam, _, _ = _scene(w, h)
    st = torch.cuda.current_stream().cuda_stream
    scr = torch.from_numpy(scenes.pixel_scrambles(w, h).view(np.int64).reshape(-1).copy()).cuda()
    films = []
    for sort, graph in ((0, False), (4, True)):
        R = render.Renderer(desc, w, h, cam)
        R.scene.set_trace_config(64, 12, 20, sort=sort)
        film = torch.zeros(w * h * 3, device="cuda")
        per_pass = []
        for it in range(1, 6):
            R.render_pass_device(scr.data_ptr(), it, film.data_ptr(), stream=st, graph=graph)
            junk = torch.randn(4096, device="cuda").sum()
            torch.cuda.synchronize()
            assert torch.isfinite(junk)
            per_pass.append(film.cpu().numpy().tobytes())
        R.scene.status(st)
        films.append(per_pass)
        R.close()
    assert films[0] == films[1]
