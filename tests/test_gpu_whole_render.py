"""Small renders run all of their bounces in one launch; MT_RENDER_PROFILE
keeps the launches per bounce.  Both against each other, and the late-bounce
launch with few lanes per wave, at the numbers of paths where the lanes per
wave change (4096 waves of 2, 4 .. 64 lanes) and where the one launch ends.
Bar: the image's bits, the ray counts and the paths per bounce are the same
(both are compared with the oracle in test_gpu_render.py, the per-bounce loop
with its side stream in test_gpu_render_overlap.py)."""
import numpy as np
import pytest

from mambatracer_amd import _lib, api
from mambatracer_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def soup():
    return W.soup_scene(20_000, 61)


@pytest.fixture(scope="module")
def spheres():
    return W.c1_scene(count=8)


@pytest.mark.parametrize("bounces", [1, 8])
@pytest.mark.parametrize("w,h,spp", [(1, 1, 1), (3, 1, 1), (8192, 1, 1), (8193, 1, 1), (181, 181, 1), (129, 127, 8),
                                     (512, 512, 1), (52429, 5, 1)])
def test_one_launch_and_per_bounce_agree(ctx, soup, spheres, w, h, spp, bounces):
    print(f"[case] whole render {w}x{h}x{spp} bounces {bounces}", flush=True)
    emit = W.material_records(np.full((1, 3), 0.5), 0.04, 0.5, 0.5, emission=np.full((1, 3), 1.0), emission_power=20.0)
    for scene in ("soup", "spheres"):
        mats = W.c1_materials()
        lf = nl = env = None
        if scene == "soup":  # lit by its own triangles
            points, faces, nodes, bounds, depth = soup
            mats = np.concatenate([mats, emit])
            faces = faces.copy()
            faces[::400, 9] = mats.shape[0] - 1
            sc = api.Scene(ctx, points, faces, nodes, bounds, depth)
            dm = ctx.to_device(mats)
            lf, nl = api.mesh_lights(ctx, sc, dm)
            base = W.soup_job(W.JobSpec(0, 0, 64, spp, 77))
            base.width, base.height = w, h
        else:
            points, normals, faces, nodes, bounds, depth = spheres
            sc = api.Scene(ctx, points, faces, nodes, bounds, depth, normals=normals)
            dm = ctx.to_device(mats)
            env = api.CEnvironment(ctx)
            env.setEnvironmentMap(W.env_map())
            base = W.RenderJob(width=w, height=h, spp=spp, pos=(0.0, 0.5, -8.0), look=(0.0, -1.0, 0.0), seed=5)
        base.max_bounces = bounces
        out = []
        for flags in (_lib.MT_RENDER_PROFILE, 0, _lib.MT_RENDER_TAIL_FROM(1)):
            base.flags = flags
            img, st = api.render(ctx, sc, dm, env, base, light_faces=lf, num_lights=nl)
            out.append((img.cpu().numpy().view(np.int32),
                        [int(st.extension_rays), int(st.shadow_rays), int(st.paths), *st.bounce_counts]))
        assert out[0][1][2] == w * h * spp == out[0][1][3]
        for img, st in out[1:]:
            np.testing.assert_array_equal(img, out[0][0])
            assert st == out[0][1]
