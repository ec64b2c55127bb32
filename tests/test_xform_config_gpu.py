"""Launch configuration of scenes with transforms: one block and LDS depth, the caller's waves per CU.

The spill area that a scene's first trace allocates has 120 entries of 8 bytes for every lane of the grid, so the
memory it takes shows the waves per CU that were launched.  Hits do not depend on them.
"""
import numpy as np
import pytest
import torch

import vermeer_amd as va
from vermeer_amd import render, scenes

pytestmark = pytest.mark.gpu

N = 300_001   # more rays than 16 waves on each of 256 CUs hold


def _renderer():
    desc = scenes.instance_scene()
    c = desc["camera"]
    return render.Renderer(desc, 8, 8, render.lookat_camera(c["from"], c["to"], c["up"], c["fov"], c["focal"], 8, 8))


def _rays():
    g = np.random.default_rng(4)
    rays = np.zeros(N, va.RAY_DTYPE)
    rays["P"] = g.uniform((-0.9, 0.1, -0.9), (0.9, 1.9, 0.9), (N, 3))
    d = g.normal(size=(N, 3))
    rays["D"] = d / np.linalg.norm(d, axis=1, keepdims=True)
    rays["tmax"] = np.inf
    rays["time"] = g.uniform(0, 1, N)
    return torch.from_numpy(rays.view(np.uint8).copy()).cuda()


def test_waves_per_cu_takes_effect():
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    dr = _rays()
    ref = None
    for waves in (24, None, 1, 4, 24):   # the first is not measured: the runtime allocates the kernel's scratch then
        R = _renderer()
        assert R.scene.trace_config()["waves_per_cu"] == 16
        if waves:
            R.scene.set_trace_config(block=256, lds_stack=16, waves_per_cu=waves)
        dh = torch.empty(N, 4, dtype=torch.int32, device="cuda")
        torch.cuda.synchronize()
        before = torch.cuda.mem_get_info()[0]
        R.scene.trace_device(dr.data_ptr(), N, dh.data_ptr())
        torch.cuda.synchronize()
        took = before - torch.cuda.mem_get_info()[0]
        lanes = min(cus * 64 * (waves or 16), (N + 255) // 256 * 256)
        print(f"[case] waves {waves}: {took / 1e6:.1f} MB for {lanes} lanes", flush=True)
        # the allocator rounds to 2 MB; what the renderer's 64 pixels already held is less than one such step
        assert ref is None or abs(took - lanes * 120 * 8) <= 3 * (2 << 20) + (1 << 20)
        R.scene.status()
        hits = dh.cpu().numpy()
        ref = hits if ref is None else ref
        assert np.array_equal(hits, ref)
        R.close()


def test_autotuner_keeps_the_shape():
    R = _renderer()
    dr = _rays()
    dh = torch.empty(N, 4, dtype=torch.int32, device="cuda")
    st = torch.cuda.current_stream().cuda_stream
    R.scene.trace_device(dr.data_ptr(), N, dh.data_ptr(), stream=st)
    ref = dh.clone()
    cfg, ms = R.scene.autotune(dr.data_ptr(), N, dh.data_ptr(), stream=st)
    print(f"[case] tuned {cfg} {ms:.3f} ms", flush=True)
    assert (cfg["block"], cfg["lds_stack"]) == (64, 12) and cfg == R.scene.trace_config()
    dh.zero_()
    R.scene.trace_device(dr.data_ptr(), N, dh.data_ptr(), stream=st)
    torch.cuda.synchronize()
    assert torch.equal(dh, ref)
    R.close()
