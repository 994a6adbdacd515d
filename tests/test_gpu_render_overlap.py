"""The render loop with its launches per bounce, each bounce's any hit on the
side stream beside the next closest hit: what a default render of more than
262144 paths runs (smaller ones run as one launch, MT_RENDER_PROFILE keeps the
stages in one stream).  Just above that size, over every kind of light.  Bar:
images, ray counts and the light grid's sums bit-exact against the oracle,
uncaptured and replayed from a capture with eager work between the replays."""
import numpy as np
import pytest
import torch

from mambatracer_amd import _lib, api
from mambatracer_amd import workloads as W
from oracle import orc_py as orc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def soup():
    points, faces, nodes, bounds, depth = W.soup_scene(20_000, 61)
    emit = W.material_records(np.full((1, 3), 0.5), 0.04, 0.5, 0.5, emission=np.full((1, 3), 1.0), emission_power=20.0)
    mats = np.concatenate([W.c1_materials(), emit])
    faces[::400, 9] = mats.shape[0] - 1
    rgba = W.env_map()
    lum, sat = orc.env_lum_sat(rgba.reshape(-1, 4), 1024, 512)
    return (points, faces, nodes, bounds, depth), mats, rgba, (rgba.reshape(-1, 4), lum, sat, 1024, 512)


def _bits(x):
    return np.ascontiguousarray(x).view(np.int32)


@pytest.mark.parametrize("w,h,spp,bounces", [(331, 397, 2, 8), (512, 513, 1, 3), (91, 97, 30, 1)])
@pytest.mark.parametrize("light", ["env", "mesh", "both", "guided", "guided_tile_pdf"])
def test_overlapped_loop(ctx, soup, light, w, h, spp, bounces):
    print(f"[case] overlapped loop {w}x{h}x{spp} bounces={bounces} light={light}", flush=True)
    (points, faces, nodes, bounds, depth), mats, rgba, oenv = soup
    assert w * h * spp > 262144
    sc = api.Scene(ctx, points, faces, nodes, bounds, depth)
    dm = ctx.to_device(mats)
    job = W.soup_job(W.JobSpec(0, 0, 8, spp, 900))
    job.width, job.height, job.max_bounces = w, h, bounces
    lf = nl = olf = env = grid = og = None
    if light in ("mesh", "both"):
        lf, nl = api.mesh_lights(ctx, sc, dm)
        torch.cuda.synchronize()
        olf = lf.cpu().numpy()[:int(nl.item())].copy()
        job.flags |= _lib.MT_RENDER_PICKED_LIGHT
    if light != "mesh":
        env = api.CEnvironment(ctx)
        env.setEnvironmentMap(rgba)
    mode = 0
    if light.startswith("guided"):
        mode = 2 if light.endswith("pdf") else 1
        job.flags |= _lib.MT_RENDER_LIGHTGRID_ENV | (_lib.MT_RENDER_LIGHTGRID_TILE_PDF if mode == 2 else 0)
        tile = api.lightgrid_seed_tile(oenv[1], 1024, 512)
        grid = api.CAdaptiveEnvironment(ctx)
        grid.setHDRLuminance(tile)
        grid.setCameraPosition(job.pos)
        env.attachLightGrid(grid)
        og = orc.LightGrid(tile, cam=job.pos)
    pids = np.arange(w * h * spp, dtype=np.int32)
    graph = api.RenderGraph(ctx, sc, dm, env, job, light_faces=lf, num_lights=nl)

    def reseed():
        if grid is not None:
            grid.clearBuffers()
            grid.setHDRLuminance(tile)

    for seed in (900, 17):
        job.seed = seed
        if og is not None:
            og = orc.LightGrid(tile, cam=job.pos)
        L, rays = orc.render_paths(points, None, faces, nodes, bounds, mats, None if light == "mesh" else oenv, job,
                                   pids, light_faces=olf, grid=og, grid_mode=mode)
        oimg = orc.resolve(L, w, h, spp)
        if og is not None:
            og.fold()
        for captured in (False, True, True):
            reseed()
            if captured:
                graph.launch(seed)
                st, img = graph.stats(), graph.image
            else:
                img, st = api.render(ctx, sc, dm, env, job, light_faces=lf, num_lights=nl)
            torch.cuda.synchronize()
            assert (int(st.extension_rays), int(st.shadow_rays)) == (int(rays[0]), int(rays[1]))
            np.testing.assert_array_equal(_bits(img.cpu().numpy()[:, :3]), _bits(oimg))
            if grid is not None:
                np.testing.assert_array_equal(_bits(grid.read_arrays()[0].reshape(-1)), _bits(og.accum))
                assert og.accum.sum() > 0
            torch.rand(100_000, device="cuda").sum().item()  # eager work between replays
    graph.close()
