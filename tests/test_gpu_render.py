"""GPU path tracer against the oracle (the CPU restatement of
src/lib/Graphics/Bling/Integrator/Path.hs:41-87 and what it calls).

Bar: per-pixel means within 3 sigma of the oracle at equal spp.  With the same
seed both sides draw the same sample values, so almost every path is the
same path and the pixel means agree far more tightly; with different seeds
the comparison is purely statistical (expected fraction beyond 3 sigma is
0.27% for normal errors; the test allows 1%).
"""
import numpy as np
import pytest

from bling_amd import abi, scenes
from bling_amd.runtime import GpuRenderer, Job, JobSpec
from oracle import pyoracle
from tests.imagestats import compare, mean_se

pytestmark = pytest.mark.gpu


def render_gpu(ctx, flat, spec):
    gs = ctx.scene(flat)
    try:
        img, sq = GpuRenderer(spec).render_plain(gs)
    finally:
        gs.close()
    return img, sq


def test_cornell_same_seed_tracks_oracle(gpu_ctx):
    flat = scenes.cornell(64)
    spec = JobSpec(spp_nu=4, spp_nv=4, max_depth=5, sample_depth=3, rr_start_depth=3, passes=2,
                   seed=7, variance=True)
    g, gsq = render_gpu(gpu_ctx, flat, spec)
    o, osq, _ = pyoracle.render(flat, spec)
    assert np.array_equal(g[..., 0], o[..., 0]), "sample weights per pixel differ"
    frac, zmean, zmax = compare(g, gsq, o, osq)
    assert frac < 0.003, (frac, zmean, zmax)
    mg, _ = mean_se(g, gsq)
    mo, _ = mean_se(o, osq)
    rel = np.abs(mg - mo) / np.maximum(np.abs(mo), 1e-3)
    # same sample streams: most pixels agree to float rounding
    assert np.median(rel) < 1e-4, np.median(rel)


def test_cornell_independent_seeds_3sigma(gpu_ctx):
    flat = scenes.cornell(64)
    spec_g = JobSpec(spp_nu=4, spp_nv=4, max_depth=5, sample_depth=3, rr_start_depth=3, passes=4,
                     seed=11, variance=True)
    spec_o = JobSpec(spp_nu=4, spp_nv=4, max_depth=5, sample_depth=3, rr_start_depth=3, passes=4,
                     seed=12, variance=True)
    g, gsq = render_gpu(gpu_ctx, flat, spec_g)
    o, osq, _ = pyoracle.render(flat, spec_o)
    frac, zmean, zmax = compare(g, gsq, o, osq)
    assert frac < 0.01, (frac, zmean, zmax)
    assert abs(zmean) < 0.05, zmean


def _view_spec(flat, w, h, spp, seed, **kw):
    return JobSpec(spp_nu=spp, spp_nv=spp, sample_depth=3, seed=seed, view=flat.view(w, h),
                   **{"max_depth": 5, "rr_start_depth": 3, **kw})


def _same_samples(got, want, spp):
    """The same samples' sums in another order: equal box-filter weights (1 a
    sample; up to 1e-3 of the samples lie on a pixel's edge by rounding and
    count for both pixels or the next one)."""
    assert np.array_equal(got[..., 0], want[..., 0])
    n = spp * got.shape[0] * got.shape[1]
    assert abs(got[..., 0].sum(dtype=np.float64) - n) <= 1e-3 * n + 1e-6
    assert np.linalg.norm(got[..., 1:] - want[..., 1:]) <= 1e-6 * np.linalg.norm(want[..., 1:])


def test_render_sizes_on_one_engine(gpu_ctx):
    """An engine sizes its launches by the work: renders larger than the pool
    and smaller than a block, in turn and of both integrators, lose no sample
    and give a fresh engine's sums."""
    from bling_amd.runtime import Context
    flat = scenes.cornell(64)
    sizes = [(700, 400, 2, "path"), (7, 5, 1, "path"), (333, 201, 4, "direct"), (1, 1, 1, "direct"), (512, 512, 3, "path"),
             (16, 16, 1, "path")]
    gs = gpu_ctx.scene(flat)
    try:
        for k, (w, h, spp, integ) in enumerate(sizes):
            spec = _view_spec(flat, w, h, spp, 40 + k, integrator=integ)
            got, _ = GpuRenderer(spec).render_plain(gs)
            with Context(0) as ctx:
                other = ctx.scene(flat)
                want, _ = GpuRenderer(spec).render_plain(other)
                other.close()
            _same_samples(got, want, spp * spp)
    finally:
        gs.close()


def test_served_jobs_arriving_in_anothers_tail(gpu_ctx):
    """Once no samples wait, the iterations cover the paths last seen active
    only: jobs that arrive then, tiny or larger than the pool, lose no sample
    and neither does the job in its tail."""
    import time
    flat = scenes.cornell(64)
    gs = gpu_ctx.scene(flat)
    try:
        for k, delay in enumerate((0.0, 0.0005, 0.001, 0.002, 0.004)):
            specs = [_view_spec(flat, 400, 300, 2, 60 + k, max_depth=40, rr_start_depth=40),
                     _view_spec(flat, 9, 4, 1, 70 + k), _view_spec(flat, 640, 500, 2, 80 + k)]
            want = [GpuRenderer(s).render_plain(gs)[0] for s in specs]
            jobs = []
            for s in specs:
                jobs.append(Job(gs, s))
                time.sleep(delay)
            for j, s, w in zip(jobs, specs, want):
                j.wait(timeout=120)
                _same_samples(j.poll()[0], w, s.spp_nu * s.spp_nv)
                j.release()
    finally:
        gs.close()


@pytest.mark.parametrize("mix", ["cornell", "with_sky"])
def test_served_jobs_match_plain(gpu_ctx, mix):
    """Each job's result is the same alone (plain path) and in the mix
    (served path, several jobs and scenes in flight).  With a sun/sky scene
    resident, every job in flight runs the kernels that evaluate the sky,
    the Cornell boxes' included."""
    from tests import cases
    flats = [scenes.cornell(48), scenes.cornell(32, light_radiance=8.0)]
    if mix == "with_sky":
        flats.append(cases.sun_sky_scene(False, res=32))
    specs = [JobSpec(spp_nu=2, spp_nv=2, max_depth=4, sample_depth=3, passes=2, seed=s, variance=True)
             for s in (1, 2, 3)]
    gss = [gpu_ctx.scene(f) for f in flats]
    try:
        plain = {}
        for si, gs in enumerate(gss):
            for k, sp in enumerate(specs):
                plain[(si, k)] = GpuRenderer(sp).render_plain(gs)
        jobs = {}
        for si, gs in enumerate(gss):
            for k, sp in enumerate(specs):
                jobs[(si, k)] = Job(gs, sp)
        for key, j in jobs.items():
            j.wait(timeout=120)
            img, sq, done, state = j.poll()
            assert state == abi.JOB_DONE and done == specs[key[1]].passes
            p_img, p_sq = plain[key]
            assert np.array_equal(img[..., 0], p_img[..., 0])
            # film sums are accumulated with atomics in a different order
            np.testing.assert_allclose(img, p_img, rtol=1e-4, atol=1e-5)
            assert j.latency_ms() > 0.0
            j.release()
    finally:
        for gs in gss:
            gs.close()


def test_progressive_passes_and_cancel(gpu_ctx):
    flat = scenes.cornell(32)
    gs = gpu_ctx.scene(flat)
    try:
        spec = JobSpec(spp_nu=2, spp_nv=2, max_depth=3, sample_depth=2, passes=6, seed=5)
        seen = []

        def report(ev):
            seen.append(ev.pass_num)
            assert ev.final_img.shape == (32, 32, 4)
            return ev.pass_num < 3  # stop after the third pass

        GpuRenderer(spec).render(gs, report)
        assert seen and seen[0] >= 1 and max(seen) >= 3
        # cancelling a queued/running job ends it as CANCELLED
        big = JobSpec(spp_nu=8, spp_nv=8, max_depth=8, sample_depth=3, passes=200, seed=9)
        j = Job(gs, big)
        j.cancel()
        with pytest.raises(abi.BgpuError) as e:
            j.wait(timeout=120)
        assert e.value.code == abi.E_CANCELLED
        j.release()
    finally:
        gs.close()


def test_invalid_job_rejected(gpu_ctx):
    flat = scenes.cornell(16)
    gs = gpu_ctx.scene(flat)
    try:
        for bad in (JobSpec(spp_nu=0), JobSpec(passes=0), JobSpec(max_depth=-1)):
            with pytest.raises(abi.BgpuError) as e:
                GpuRenderer(bad).render_plain(gs)
            assert e.value.code == abi.E_INVALID
        # 30001^2 extent pixels x 8 samples in one pass exceed the 32-bit pass
        # counters: refused before the film is touched
        import ctypes as C
        big = JobSpec(spp_nu=4, spp_nv=2, view=flat.view(30000, 30000))
        tiny = np.zeros(16, np.float32)
        for call in (lambda: gpu_ctx.lib.bgpu_render(gs.h, C.byref(big.desc()), tiny.ctypes.data, None),
                     lambda: gpu_ctx.lib.bgpu_job_submit(gs.h, C.byref(big.desc()), C.byref(C.c_void_p()))):
            assert call() == abi.E_INVALID
    finally:
        gs.close()


def _y_mean(img, sq):
    m, se = mean_se(img, sq)
    return m[..., 1].mean(), np.sqrt((se[..., 1] ** 2).sum()) / m[..., 1].size


def test_analytic_radiance_on_gpu(gpu_ctx):
    from tests import cases
    spec = JobSpec(spp_nu=8, spp_nv=8, max_depth=1, sample_depth=1, passes=8, seed=5, variance=True)
    y, s = _y_mean(*render_gpu(gpu_ctx, cases.plane_under_sky(rho=0.5, sky=1.0), spec))
    assert abs(y - 0.5) < 4 * s + 5e-5, (y, s)
    R, D, Le, rho = 0.25, 2.0, 4.0, 0.5
    y, s = _y_mean(*render_gpu(gpu_ctx, cases.sphere_light_over_plane(rho=rho, Le=Le, R=R, D=D), spec))
    want = rho * Le * (R / D) ** 2
    assert abs(y - want) < 4 * s + 1e-4 * want, (y, want, s)
    img, _ = render_gpu(gpu_ctx, cases.sky_only(sky=2.0), JobSpec(spp_nu=2, spp_nv=2, passes=1))
    from bling_amd.scene import const, spectrum_to_xyz
    np.testing.assert_allclose(img[..., 1:] / img[..., :1],
                               np.broadcast_to(np.array(spectrum_to_xyz(const(2.0))), img[..., 1:].shape),
                               rtol=1e-6)


@pytest.mark.parametrize("env", [False, True])
def test_materials_scene_matches_oracle(gpu_ctx, env):
    from tests import cases
    flat = cases.materials_scene(res=48, env=env)
    spec = JobSpec(spp_nu=4, spp_nv=4, max_depth=8, sample_depth=3, rr_start_depth=3, passes=4,
                   seed=21, variance=True)
    g, gsq = render_gpu(gpu_ctx, flat, spec)
    o, osq, _ = pyoracle.render(flat, spec)
    assert np.isfinite(g).all()
    frac, zmean, zmax = compare(g, gsq, o, osq)
    assert frac < 0.01, (frac, zmean, zmax)
    spec2 = JobSpec(spp_nu=4, spp_nv=4, max_depth=8, sample_depth=3, rr_start_depth=3, passes=4,
                    seed=22, variance=True)
    o2, osq2, _ = pyoracle.render(flat, spec2)
    frac, zmean, zmax = compare(g, gsq, o2, osq2)
    assert frac < 0.015, (frac, zmean, zmax)
    assert abs(zmean) < 0.08, zmean


def test_job_view_tracks_oracle_and_scene_film(gpu_ctx):
    """A job's own camera and film: same image as a scene described at that
    size, on the plain and the served path, and tracking the oracle."""
    import dataclasses
    other = scenes.cornell(48)
    direct = scenes.cornell(40, height=24)
    spec = JobSpec(spp_nu=2, spp_nv=2, max_depth=4, sample_depth=3, rr_start_depth=3, passes=2,
                   seed=13, variance=True, view=other.view(40, 24))
    g, gsq = render_gpu(gpu_ctx, other, spec)
    assert g.shape == (24, 40, 4)
    o, osq, _ = pyoracle.render(other, spec)
    assert np.array_equal(g[..., 0], o[..., 0])
    mg, _ = mean_se(g, gsq)
    mo, _ = mean_se(o, osq)
    rel = np.abs(mg - mo) / np.maximum(np.abs(mo), 1e-3)
    assert np.median(rel) < 1e-4, np.median(rel)
    d, _ = render_gpu(gpu_ctx, direct, dataclasses.replace(spec, view=None))
    np.testing.assert_allclose(g, d, rtol=1e-4, atol=1e-5)
    gs = gpu_ctx.scene(other)
    try:
        j = Job(gs, spec)
        j.wait(timeout=120)
        img, _, done, state = j.poll()
        assert state == abi.JOB_DONE and img.shape == (24, 40, 4)
        np.testing.assert_allclose(img, g, rtol=1e-4, atol=1e-5)
        j.release()
        bad = other.view(16, 16)
        bad.film.width = 0
        with pytest.raises(abi.BgpuError) as e:
            GpuRenderer(dataclasses.replace(spec, view=bad)).render_plain(gs)
        assert e.value.code == abi.E_INVALID
    finally:
        gs.close()


def test_tuning_knobs_keep_results(gpu_ctx):
    """Kernel block size, pool size and the shading kernel's occupancy variant
    change scheduling only: the image is the same up to film-atomic order."""
    flat = scenes.cornell(32)
    spec = JobSpec(spp_nu=2, spp_nv=2, max_depth=5, sample_depth=3, rr_start_depth=3, seed=4)
    base, _ = render_gpu(gpu_ctx, flat, spec)
    defaults = {k: gpu_ctx.config_get(k) for k in ("pt.block", "pt.pool", "pt.shade_waves", "pt.persistent",
                                                   "pt.sort", "pt.diffuse_waves", "pt.stack", "pt.walk",
                                                   "pt.light_variants")}
    try:
        for key, val in (("pt.shade_waves", 0), ("pt.block", 64), ("pt.block", 256), ("pt.pool", 4096),
                         ("pt.persistent", 0), ("pt.persistent", 1), ("pt.sort", 0), ("pt.sort", 1),
                         ("pt.diffuse_waves", 0), ("pt.diffuse_waves", 4), ("pt.stack", 8), ("pt.stack", 24),
                         ("pt.walk", 16), ("pt.walk", 1), ("pt.light_variants", 0)):
            gpu_ctx.config_set(key, val)
            assert gpu_ctx.config_get(key) == val
            img, _ = render_gpu(gpu_ctx, flat, spec)
            assert np.array_equal(img[..., 0], base[..., 0]), key
            np.testing.assert_allclose(img, base, rtol=1e-4, atol=1e-5, err_msg=key)
            gpu_ctx.config_set(key, defaults[key])
        with pytest.raises(abi.BgpuError) as e:
            gpu_ctx.config_set("pt.block", 96)
        assert e.value.code == abi.E_INVALID
        with pytest.raises(abi.BgpuError) as e:
            gpu_ctx.config_set("no.such.key", 1)
        assert e.value.code == abi.E_INVALID
        gs = gpu_ctx.scene(flat)
        try:
            j = Job(gs, spec)
            with pytest.raises(abi.BgpuError) as e:
                gpu_ctx.config_set("pt.pool", 8192)  # a served job handle is live
            assert e.value.code == abi.E_STATE
            j.wait(timeout=120)
            j.release()
            gpu_ctx.config_set("pt.pool", 8192)
            gpu_ctx.config_set("pt.pool", defaults["pt.pool"])
        finally:
            gs.close()
    finally:
        for k, v in defaults.items():
            gpu_ctx.config_set(k, v)


def test_shiny_metal_matches_oracle(gpu_ctx):
    """shinyMetal spheres (mkShinyMetal, Material.hs:98-109: a microfacet and
    a specular reflection, conductor terms approximated from ks and kr) on
    a matte floor under a quad light and a sky: the same seed tracks the
    oracle."""
    from bling_amd.scene import Material, SceneBuilder, rgb_illum, rgb_refl
    from bling_amd import transform as T
    sb = SceneBuilder()
    floor = sb.material(Material.matte(rgb_refl(0.6, 0.6, 0.6)))
    sb.shape(abi.SHAPE_QUAD, (4.0, 4.0), o2w=T.rotate_x(90), material=floor)
    for x, (kr, ks, rough) in zip((-1.2, 0.0, 1.2), ((rgb_refl(0.9, 0.6, 0.3), rgb_refl(0.8, 0.8, 0.8), 0.02),
                                                     (rgb_refl(0.3, 0.3, 0.3), rgb_refl(0.9, 0.7, 0.2), 0.3),
                                                     (rgb_refl(0.95, 0.95, 0.95), rgb_refl(0.1, 0.1, 0.1), 0.0))):
        m = sb.material(Material.shiny_metal(kr, ks, rough))
        sb.shape(abi.SHAPE_SPHERE, (0.5,), o2w=T.translate((x, 0.5, 0.0)), material=m)
    sb.shape(abi.SHAPE_QUAD, (1.0, 1.0), o2w=T.rotate_x(-90) @ T.translate((0.0, 3.0, 0.0)), material=floor,
             emission=rgb_illum(8.0, 8.0, 8.0))
    sb.infinite_light(np.tile(rgb_illum(0.4, 0.4, 0.5), (2, 4, 1)))
    sb.look(T.look_at((0.0, 1.5, -4.0), (0.0, 0.5, 0.0), (0, 1, 0)), 50.0, 48, 48)
    flat = sb.build()
    spec = JobSpec(spp_nu=4, spp_nv=4, max_depth=6, sample_depth=3, rr_start_depth=3, passes=2, seed=45,
                   variance=True)
    g, gsq = render_gpu(gpu_ctx, flat, spec)
    o, osq, _ = pyoracle.render(flat, spec)
    assert np.isfinite(g).all()
    assert np.array_equal(g[..., 0], o[..., 0])
    mg, _ = mean_se(g, gsq)
    mo, _ = mean_se(o, osq)
    rel = np.abs(mg - mo) / np.maximum(np.abs(mo), 1e-3)
    assert np.median(rel) < 1e-4, np.median(rel)
    frac, zmean, zmax = compare(g, gsq, o, osq)
    assert frac < 0.01, (frac, zmean, zmax)


def test_delta_lights_closed_forms_and_oracle(gpu_ctx):
    """Point and directional lights (Light.hs:53-61,142-150): the closed
    forms of a Lambertian plane below each, and a scene that mixes them with
    an area light and a sky over matte, plastic and glass spheres, against
    the oracle at the same seed."""
    from tests import cases
    from bling_amd.scene import Material, SceneBuilder, const, rgb_illum, rgb_refl
    from bling_amd import transform as T
    spec1 = JobSpec(spp_nu=2, spp_nv=2, max_depth=1, sample_depth=1, seed=5, variance=True)
    rho, I, D = 0.5, 3.0, 2.0
    g, gsq = render_gpu(gpu_ctx, cases.delta_light_over_plane("point", rho=rho, I=I, D=D), spec1)
    m, _ = mean_se(g, gsq)
    np.testing.assert_allclose(m[..., 1], rho * I / (np.pi * D * D), rtol=1e-4)
    g, gsq = render_gpu(gpu_ctx, cases.delta_light_over_plane("directional", rho=rho, I=I, theta=60.0), spec1)
    m, _ = mean_se(g, gsq)
    np.testing.assert_allclose(m[..., 1], rho * I * 0.25 / np.pi, rtol=1e-4)
    sb = SceneBuilder()
    floor = sb.material(Material.matte(rgb_refl(0.6, 0.6, 0.6)))
    sb.shape(abi.SHAPE_QUAD, (4.0, 4.0), o2w=T.rotate_x(90), material=floor)
    mats = [Material.matte(rgb_refl(0.7, 0.3, 0.2), 0.3), Material.plastic(rgb_refl(0.2, 0.4, 0.7),
            rgb_refl(0.5, 0.5, 0.5), 0.05), Material.glass(1.5, const(1.0), const(1.0))]
    for x, m in zip((-1.2, 0.0, 1.2), mats):
        sb.shape(abi.SHAPE_SPHERE, (0.5,), o2w=T.translate((x, 0.5, 0.0)), material=sb.material(m))
    sb.shape(abi.SHAPE_QUAD, (0.5, 0.5), o2w=T.rotate_x(-90) @ T.translate((1.5, 3.0, 0.0)), material=floor,
             emission=rgb_illum(6.0, 6.0, 6.0))
    sb.point_light(rgb_illum(4.0, 3.0, 2.0), (-1.0, 2.5, -1.0))
    sb.directional_light(rgb_illum(1.0, 1.0, 1.2), (0.3, 1.0, -0.4))
    sb.infinite_light(np.tile(rgb_illum(0.2, 0.2, 0.3), (2, 4, 1)))
    sb.look(T.look_at((0.0, 1.5, -4.0), (0.0, 0.5, 0.0), (0, 1, 0)), 50.0, 48, 48)
    flat = sb.build()
    spec = JobSpec(spp_nu=4, spp_nv=4, max_depth=6, sample_depth=3, rr_start_depth=3, passes=2, seed=46,
                   variance=True)
    g, gsq = render_gpu(gpu_ctx, flat, spec)
    o, osq, _ = pyoracle.render(flat, spec)
    assert np.isfinite(g).all()
    assert np.array_equal(g[..., 0], o[..., 0])
    mg, _ = mean_se(g, gsq)
    mo, _ = mean_se(o, osq)
    rel = np.abs(mg - mo) / np.maximum(np.abs(mo), 1e-3)
    assert np.median(rel) < 1e-4, np.median(rel)
    frac, zmean, zmax = compare(g, gsq, o, osq)
    assert frac < 0.01, (frac, zmean, zmax)
    for integrator in ("direct",):
        sd = JobSpec(spp_nu=2, spp_nv=2, max_depth=4, sample_depth=3, rr_start_depth=3, passes=1, seed=47,
                     variance=True, integrator=integrator)
        g, gsq = render_gpu(gpu_ctx, flat, sd)
        o, osq, _ = pyoracle.render(flat, sd)
        assert np.array_equal(g[..., 0], o[..., 0])
        mg, _ = mean_se(g, gsq)
        mo, _ = mean_se(o, osq)
        rel = np.abs(mg - mo) / np.maximum(np.abs(mo), 1e-3)
        assert np.median(rel) < 1e-4, np.median(rel)


def test_environment_camera_matches_oracle(gpu_ctx):
    """The environment camera (Camera.hs:70-76) inside a lit room with a
    sky: the same seed tracks the oracle (the device's sinf/cosf may move a
    ray by an ulp, so pixels are compared by their median difference)."""
    from bling_amd.scene import Material, SceneBuilder, rgb_illum, rgb_refl
    from bling_amd import transform as T
    sb = SceneBuilder()
    scenes._lit_room(sb, 2.0)
    m = sb.material(Material.plastic(rgb_refl(0.3, 0.5, 0.7), rgb_refl(0.5, 0.5, 0.5), 0.05))
    sb.shape(abi.SHAPE_SPHERE, (0.5,), o2w=T.translate((0.8, 0.5, 0.6)), material=m)
    sb.infinite_light(np.tile(rgb_illum(0.3, 0.3, 0.4), (2, 4, 1)))
    sb.environment_camera(T.translate((0.0, 1.0, 0.0)), 64, 32)
    sb.set_film(64, 32)
    flat = sb.build()
    spec = JobSpec(spp_nu=4, spp_nv=4, max_depth=5, sample_depth=3, rr_start_depth=3, passes=2, seed=48,
                   variance=True)
    g, gsq = render_gpu(gpu_ctx, flat, spec)
    o, osq, _ = pyoracle.render(flat, spec)
    assert np.isfinite(g).all() and g[..., 2].sum() > 0
    assert np.array_equal(g[..., 0], o[..., 0])
    mg, _ = mean_se(g, gsq)
    mo, _ = mean_se(o, osq)
    rel = np.abs(mg - mo) / np.maximum(np.abs(mo), 1e-3)
    assert np.median(rel) < 1e-4, np.median(rel)
    frac, zmean, zmax = compare(g, gsq, o, osq)
    assert frac < 0.01, (frac, zmean, zmax)
    v = flat.view(32, 16)  # a job's view at another size keeps the camera kind
    assert v.camera.type == abi.CAMERA_ENVIRONMENT and (v.camera.xres, v.camera.yres) == (32.0, 16.0)


@pytest.mark.parametrize("env_camera", [False, True], ids=["perspective", "environment"])
def test_sun_sky_matches_oracle(gpu_ctx, env_camera):
    """An infinite light with a sun/sky map (SunSky.hs), evaluated per
    direction on the device, over matte, plastic and glass spheres: the same
    seed tracks the oracle.  The environment camera sees the whole map, the
    sun's disk included, directly."""
    from tests import cases
    flat = cases.sun_sky_scene(env_camera)
    spec = JobSpec(spp_nu=4, spp_nv=4, max_depth=6, sample_depth=3, rr_start_depth=3, passes=2, seed=51,
                   variance=True)
    g, gsq = render_gpu(gpu_ctx, flat, spec)
    o, osq, _ = pyoracle.render(flat, spec)
    assert np.isfinite(g).all() and g[..., 2].sum() > 0
    assert np.array_equal(g[..., 0], o[..., 0])
    mg, _ = mean_se(g, gsq)
    mo, _ = mean_se(o, osq)
    rel = np.abs(mg - mo) / np.maximum(np.abs(mo), 1e-3)
    assert np.median(rel) < 1e-4, np.median(rel)
    frac, zmean, zmax = compare(g, gsq, o, osq)
    assert frac < 0.01, (frac, zmean, zmax)
    if env_camera:  # the sun's disk is in view: some pixels hold sunR
        assert mg[..., 1].max() > 5 * np.median(mg[..., 1])


def test_sun_sky_direct_lighting_and_knob(gpu_ctx):
    """The direct-lighting integrator under a sun/sky map tracks the oracle,
    and with the light-kind variants switched off the engine still picks the
    kernels that evaluate the map (the same image as with them on, up to the
    order of the film's sums)."""
    from tests import cases
    flat = cases.sun_sky_scene(False, res=32)
    spec = JobSpec(spp_nu=2, spp_nv=2, max_depth=4, sample_depth=3, passes=2, seed=53, variance=True,
                   integrator="direct")
    g, gsq = render_gpu(gpu_ctx, flat, spec)
    o, osq, _ = pyoracle.render(flat, spec)
    assert np.array_equal(g[..., 0], o[..., 0])
    mg, _ = mean_se(g, gsq)
    mo, _ = mean_se(o, osq)
    rel = np.abs(mg - mo) / np.maximum(np.abs(mo), 1e-3)
    assert np.median(rel) < 1e-4, np.median(rel)
    spec = JobSpec(spp_nu=2, spp_nv=2, max_depth=5, sample_depth=3, rr_start_depth=3, seed=54, variance=True)
    a, _ = render_gpu(gpu_ctx, flat, spec)
    try:
        gpu_ctx.config_set("pt.light_variants", 0)
        b, _ = render_gpu(gpu_ctx, flat, spec)
    finally:
        gpu_ctx.config_set("pt.light_variants", 1)
    # the film's per-pixel sums take samples in either order: equal weights, close sums
    assert np.array_equal(a[..., 0], b[..., 0])
    np.testing.assert_allclose(a, b, rtol=1e-4, atol=1e-5)


def test_texel_light_map_orientation_matches_oracle(gpu_ctx):
    """A texel light map of distinct texels seen through the environment
    camera: the device's rgbfToTexMap lookup (IO/Bitmap.hs:21-28) and
    Dist2D pick the oracle's texels."""
    from bling_amd.scene import Material, SceneBuilder, rgb_illum, rgb_refl
    from bling_amd import transform as T
    rng = np.random.default_rng(12)
    sb = SceneBuilder()
    floor = sb.material(Material.matte(rgb_refl(0.5, 0.5, 0.5)))
    sb.shape(abi.SHAPE_SPHERE, (0.4,), o2w=T.translate((0.0, -0.6, 1.0)), material=floor)
    texels = np.stack([[rgb_illum(*rng.uniform(0.05, 2.0, 3)) for _ in range(12)] for _ in range(6)])
    sb.infinite_light(texels, T.rotate_y(30) @ T.rotate_x(-90))
    sb.environment_camera(T.Transform(), 72, 36)
    sb.set_film(72, 36)
    flat = sb.build()
    spec = JobSpec(spp_nu=2, spp_nv=2, max_depth=3, sample_depth=3, seed=52, variance=True)
    g, gsq = render_gpu(gpu_ctx, flat, spec)
    o, osq, _ = pyoracle.render(flat, spec)
    assert np.array_equal(g[..., 0], o[..., 0])
    mg, _ = mean_se(g, gsq)
    mo, _ = mean_se(o, osq)
    rel = np.abs(mg - mo) / np.maximum(np.abs(mo), 1e-3)
    assert np.median(rel) < 1e-4, np.median(rel)


def test_light_kind_variants_keep_results(gpu_ctx):
    """The diffuse shading kernel's light-kind variants (quad lights only;
    quad, sphere and infinite lights) give the all-kinds kernel's image:
    the Cornell box (one quad light), a lit room (a quad and a sphere
    light), a room under a sky map with a quad light, and one lit by a box
    (every kind)."""
    from bling_amd.scene import Material, SceneBuilder, rgb_illum, rgb_refl
    from bling_amd import transform as T

    def room(extra):
        sb = SceneBuilder()
        scenes._lit_room(sb, 2.0)
        m = sb.material(Material.matte(rgb_refl(0.5, 0.6, 0.7)))
        sb.shape(abi.SHAPE_SPHERE, (0.5,), o2w=T.translate((0.0, 0.5, 0.0)), material=m)
        extra(sb, m)
        sb.look(T.look_at((0.0, 2.0, -6.0), (0.0, 0.5, 0.0), (0, 1, 0)), 50.0, 32, 32)
        return sb.build()

    flats = {"quad": scenes.cornell(32),
             "quad+sphere": room(lambda sb, m: None),
             "sky": room(lambda sb, m: sb.infinite_light(np.tile(rgb_illum(0.3, 0.3, 0.3), (4, 8, 1)))),
             "box": room(lambda sb, m: sb.shape(abi.SHAPE_BOX, (-0.2, 0.0, -0.2, 0.2, 0.4, 0.2),
                                                  o2w=T.translate((1.0, 0.0, 0.5)), material=m,
                                                  emission=rgb_illum(2.0, 2.0, 2.0))),
             "point": room(lambda sb, m: sb.point_light(rgb_illum(3.0, 3.0, 3.0), (0.5, 2.0, -0.5)))}
    spec = JobSpec(spp_nu=2, spp_nv=2, max_depth=5, sample_depth=3, rr_start_depth=3, seed=8)
    try:
        for name, flat in flats.items():
            gpu_ctx.config_set("pt.light_variants", 1)
            a, _ = render_gpu(gpu_ctx, flat, spec)
            gpu_ctx.config_set("pt.light_variants", 0)
            b, _ = render_gpu(gpu_ctx, flat, spec)
            assert np.array_equal(a[..., 0], b[..., 0]), name
            np.testing.assert_allclose(a, b, rtol=1e-4, atol=1e-5, err_msg=name)
            assert a[..., 2].sum() > 0, name
    finally:
        gpu_ctx.config_set("pt.light_variants", 1)


def test_divergent_materials_matches_oracle(gpu_ctx):
    """The divergent-materials workload at reduced size (heightmap, tori,
    spheres of matte/plastic/metal/glass under a sky map, max depth 16):
    independent seeds agree within 3 sigma per pixel, the same seed tracks
    the oracle sample for sample."""
    flat = scenes.divergent_scene(res=40, hm=32, n_tori=4, torus_tris=800, n_spheres=30)
    mk = lambda seed: JobSpec(spp_nu=4, spp_nv=4, max_depth=16, sample_depth=3, rr_start_depth=3,
                              passes=4, seed=seed, variance=True)
    g, gsq = render_gpu(gpu_ctx, flat, mk(31))
    assert np.isfinite(g).all()
    o, osq, _ = pyoracle.render(flat, mk(32))
    frac, zmean, zmax = compare(g, gsq, o, osq)
    assert frac < 0.01, (frac, zmean, zmax)
    assert abs(zmean) < 0.08, zmean
    o1, o1sq, _ = pyoracle.render(flat, mk(31))
    assert np.array_equal(g[..., 0], o1[..., 0])
    mg, _ = mean_se(g, gsq)
    mo, _ = mean_se(o1, o1sq)
    rel = np.abs(mg - mo) / np.maximum(np.abs(mo), 1e-3)
    assert np.median(rel) < 1e-4, np.median(rel)
    # grouping the shading queue by material kind (on by default for this
    # mixed-material scene) changes the order of work only
    keep = gpu_ctx.config_get("pt.sort")
    try:
        for mode in (0, 1):
            gpu_ctx.config_set("pt.sort", mode)
            g2, _ = render_gpu(gpu_ctx, flat, mk(31))
            assert np.array_equal(g2[..., 0], g[..., 0]), mode
            np.testing.assert_allclose(g2, g, rtol=1e-4, atol=1e-5, err_msg=str(mode))
    finally:
        gpu_ctx.config_set("pt.sort", keep)


def test_batch_of_64_jobs(gpu_ctx):
    """64 jobs over 8 resident scenes of different sizes, resolutions and spp
    submitted at once: every job's image in the mix equals its image alone."""
    rng = np.random.default_rng(64)
    flats = [scenes.stack_scene(int(n), seed=k) if k % 2 == 0 else scenes.grid_scene(int(n), seed=k)
             for k, n in enumerate(np.exp(rng.uniform(np.log(1e3), np.log(5e4), 8)))]
    gss = [gpu_ctx.scene(f) for f in flats]
    try:
        jobs = []
        for k in range(64):
            si = int(rng.integers(8))
            res = int(rng.choice([16, 24, 32, 48]))
            spp = [(1, 1), (2, 1), (2, 2), (4, 2)][int(rng.integers(4))]
            spec = JobSpec(spp_nu=spp[0], spp_nv=spp[1], max_depth=5, sample_depth=3, rr_start_depth=3,
                           passes=1, seed=1000 + k, view=flats[si].view(res, res))
            jobs.append((si, spec))
        handles = [Job(gss[si], spec) for si, spec in jobs]
        for (si, spec), h in zip(jobs, handles):
            h.wait(timeout=120)
            img, _, done, state = h.poll()
            h.release()
            alone, _ = GpuRenderer(spec).render_plain(gss[si])
            assert state == abi.JOB_DONE and img.shape == alone.shape
            assert np.array_equal(img[..., 0], alone[..., 0])
            np.testing.assert_allclose(img, alone, rtol=1e-4, atol=1e-5)
    finally:
        for gs in gss:
            gs.close()


def test_chunked_jobs_match_plain_overtake_and_cancel(gpu_ctx):
    """With a small path pool every job reaches the device in many chunks:
    chunked jobs equal their plain renders, a short job submitted after a
    long one finishes first, and a long job cancelled part-way ends as
    CANCELLED with its complete passes kept."""
    import time
    keep = gpu_ctx.config_get("pt.pool")
    gpu_ctx.config_set("pt.pool", 4096)  # chunks of 2048 samples
    flat = scenes.cornell(48)
    gs = gpu_ctx.scene(flat)
    try:
        specs = [JobSpec(spp_nu=2, spp_nv=2, max_depth=4, sample_depth=3, passes=3, seed=21),
                 JobSpec(spp_nu=1, spp_nv=1, max_depth=4, sample_depth=3, passes=1, seed=22,
                         view=flat.view(16, 16)),
                 JobSpec(spp_nu=4, spp_nv=2, max_depth=4, sample_depth=3, passes=2, seed=23,
                         view=flat.view(40, 24))]
        handles = [Job(gs, sp) for sp in specs]
        for sp, h in zip(specs, handles):
            h.wait(timeout=120)
            img, _, done, state = h.poll()
            h.release()
            alone, _ = GpuRenderer(sp).render_plain(gs)
            assert state == abi.JOB_DONE and done == sp.passes
            assert np.array_equal(img[..., 0], alone[..., 0])
            np.testing.assert_allclose(img, alone, rtol=1e-4, atol=1e-5)

        big = Job(gs, JobSpec(spp_nu=4, spp_nv=4, max_depth=6, sample_depth=3, passes=50, seed=24))
        small = Job(gs, JobSpec(spp_nu=1, spp_nv=1, max_depth=4, sample_depth=3, passes=1, seed=25,
                                view=flat.view(16, 16)))
        small.wait(timeout=120)
        assert small.poll(want_image=False)[3] == abi.JOB_DONE
        assert big.poll(want_image=False)[3] == abi.JOB_RUNNING  # overtaken
        small.release()
        t0 = time.time()
        while big.poll(want_image=False)[2] < 1 and time.time() - t0 < 60:
            time.sleep(0.002)
        big.cancel()
        with pytest.raises(abi.BgpuError) as e:
            big.wait(timeout=120)
        assert e.value.code == abi.E_CANCELLED
        img, _, done, state = big.poll()
        assert state == abi.JOB_CANCELLED and 1 <= done < 50
        assert np.isfinite(img).all()
        big.release()
    finally:
        gs.close()
        gpu_ctx.config_set("pt.pool", keep)


def test_bling_file_renders_like_the_procedural_scene(gpu_ctx):
    """The Cornell box read from its .bling text (tests/golden/cornell_c1.bling)
    renders the image of the procedurally built scene: same seed, same
    samples (film sums agree up to atomic order and the signed zeros the
    reference's transform composition leaves in the camera matrix)."""
    import os
    from bling_amd import bling_format
    b = bling_format.load(os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden",
                                       "cornell_c1.bling"))
    spec = b.spec(seed=7)
    flat = scenes.cornell(256)
    a_img, _ = render_gpu(gpu_ctx, flat, spec)
    b_img, _ = render_gpu(gpu_ctx, b.flat, spec)
    assert np.array_equal(a_img[..., 0], b_img[..., 0])
    np.testing.assert_allclose(b_img, a_img, rtol=1e-4, atol=1e-5)
    assert b_img[..., 2].mean() > 0.01


def test_textured_scene_matches_oracle(gpu_ctx):
    """Checker and graph-paper selectors on triangles (uv from the mesh),
    spheres, quads, uv and planar mappings, and a material with both
    spectra textured: same seed tracks the oracle, another seed is within
    3 sigma."""
    from tests import cases
    flat = cases.textured_scene(res=48)
    spec = JobSpec(spp_nu=4, spp_nv=4, max_depth=6, sample_depth=3, rr_start_depth=3, passes=4,
                   seed=31, variance=True)
    g, gsq = render_gpu(gpu_ctx, flat, spec)
    o, osq, _ = pyoracle.render(flat, spec)
    assert np.isfinite(g).all()
    frac, zmean, zmax = compare(g, gsq, o, osq)
    assert frac < 0.01, (frac, zmean, zmax)
    mg, _ = mean_se(g, gsq)
    mo, _ = mean_se(o, osq)
    rel = np.abs(mg - mo) / np.maximum(np.abs(mo), 1e-3)
    assert np.median(rel) < 1e-4, np.median(rel)
    spec2 = JobSpec(spp_nu=4, spp_nv=4, max_depth=6, sample_depth=3, rr_start_depth=3, passes=4,
                    seed=32, variance=True)
    o2, osq2, _ = pyoracle.render(flat, spec2)
    frac, zmean, zmax = compare(g, gsq, o2, osq2)
    assert frac < 0.015, (frac, zmean, zmax)
    assert abs(zmean) < 0.08, zmean


def test_scene_file_renders_like_the_flat_scene(gpu_ctx, tmp_path):
    """A scene loaded from its flat binary file (bgpu_scene_load) renders
    the image of the scene created from the descriptor."""
    from tests import cases
    flat = cases.textured_scene(res=32)
    path = tmp_path / "t.bgs"
    flat.save(path)
    spec = JobSpec(spp_nu=2, spp_nv=2, max_depth=5, sample_depth=3, rr_start_depth=3, passes=2,
                   seed=13, variance=True)
    a, _ = render_gpu(gpu_ctx, flat, spec)
    gs = gpu_ctx.load_scene(path)
    try:
        b, _ = GpuRenderer(spec).render_plain(gs)
    finally:
        gs.close()
    assert np.array_equal(a[..., 0], b[..., 0])
    np.testing.assert_allclose(b, a, rtol=1e-5, atol=1e-6)


def test_direct_lighting_matches_oracle(gpu_ctx):
    """The direct-lighting integrator (Integrator/DirectLighting.hs) on the
    materials scene, whose glass and mirror spheres branch: the same seed
    tracks the oracle, another seed is within 3 sigma."""
    from tests import cases
    flat = cases.materials_scene(res=40, env=True)
    spec = JobSpec(spp_nu=4, spp_nv=4, max_depth=5, sample_depth=0, passes=4, seed=41, variance=True,
                   integrator="direct")
    before = gpu_ctx.stats()["branches_dropped"]
    g, gsq = render_gpu(gpu_ctx, flat, spec)
    assert gpu_ctx.stats()["branches_dropped"] == before, "a pending specular branch was dropped"
    o, osq, _ = pyoracle.render(flat, spec)
    assert np.isfinite(g).all()
    assert np.array_equal(g[..., 0], o[..., 0])
    frac, zmean, zmax = compare(g, gsq, o, osq)
    assert frac < 0.01, (frac, zmean, zmax)
    mg, _ = mean_se(g, gsq)
    mo, _ = mean_se(o, osq)
    rel = np.abs(mg - mo) / np.maximum(np.abs(mo), 1e-3)
    assert np.median(rel) < 1e-4, np.median(rel)
    spec2 = JobSpec(spp_nu=4, spp_nv=4, max_depth=5, sample_depth=0, passes=4, seed=42, variance=True,
                    integrator="direct")
    o2, osq2, _ = pyoracle.render(flat, spec2)
    frac, zmean, zmax = compare(g, gsq, o2, osq2)
    assert frac < 0.015, (frac, zmean, zmax)
    assert abs(zmean) < 0.08, zmean


def test_direct_lighting_mirror_closed_form(gpu_ctx):
    """r Le (w + 1) through a mirror under a quad light (the oracle's pin of
    the same scene), r Le w at maxDepth 1."""
    from tests.test_oracle_pins import mirror_under_light
    r, Le, theta = 0.9, 3.0, 60.0
    c = np.cos(np.radians(theta))
    pdf_l = (3.0 / c) ** 2 / (c * (4 * 100.0 * 100.0))
    w = 1.0 / (1.0 + pdf_l ** 2)
    flat = mirror_under_light(r=r, Le=Le, theta=theta)
    for md, want in ((1, r * Le * w), (2, r * Le * (w + 1.0)), (5, r * Le * (w + 1.0))):
        spec = JobSpec(spp_nu=2, spp_nv=2, max_depth=md, sample_depth=0, passes=1, seed=3, integrator="direct")
        img, _ = render_gpu(gpu_ctx, flat, spec)
        np.testing.assert_allclose(img[..., 2] / img[..., 0], want, rtol=1e-5)


def test_direct_and_path_jobs_served_together(gpu_ctx):
    """Direct-lighting and path jobs in flight together on the served path
    each give their plain result; a direct-lighting job deeper than the
    branch stacks hold is refused."""
    from tests import cases
    flat = cases.materials_scene(res=24, env=True)
    specs = [JobSpec(spp_nu=2, spp_nv=2, max_depth=5, sample_depth=0, passes=2, seed=s, integrator="direct")
             for s in (1, 2)]
    specs += [JobSpec(spp_nu=2, spp_nv=2, max_depth=5, sample_depth=3, passes=2, seed=3)]
    gs = gpu_ctx.scene(flat)
    try:
        plain = [GpuRenderer(sp).render_plain(gs) for sp in specs]
        jobs = [Job(gs, sp) for sp in specs]
        for sp, j, (p_img, _) in zip(specs, jobs, plain):
            j.wait(timeout=120)
            img, _, done, state = j.poll()
            assert state == abi.JOB_DONE and done == sp.passes
            assert np.array_equal(img[..., 0], p_img[..., 0])
            np.testing.assert_allclose(img, p_img, rtol=1e-4, atol=1e-5)
            j.release()
        assert gpu_ctx.config_get("pt.dl_depth") == 4
        deep = JobSpec(spp_nu=1, spp_nv=1, max_depth=6, passes=1, integrator="direct")
        with pytest.raises(abi.BgpuError) as e:
            GpuRenderer(deep).render_plain(gs)
        assert e.value.code == abi.E_INVALID and "pt.dl_depth" in str(e.value)
    finally:
        gs.close()


HEIGHTMAP_BLING = """
imageSize 48 48
filter box
transform { lookAt { pos 0 3 -3 look 0 0 0 up 0 1 0 } }
camera { perspective fov 50 lensRadius 0 focalDistance 1 }
newTransform { }
material { plastic kd { constant rgbR 0.3 0.5 0.2 } ks { constant rgbR 0.4 0.4 0.4 } rough { constant 0.05 } }
prim { heightMap 40 30 { scale 0.6 { fbm 0 octaves 4 omega 0.5 } } { translate -0.5 0 -0.5 scale 4 1 4 } }
material { blackbody }
emission { rgbI 6 6 6 }
transform { rotateX -90 translate 0 3 0 }
prim { shape { quad 0.7 0.7 } }
emission { none }
renderer { sampler sampled { sampler { stratified 4 4 } integrator { path maxDepth 5 sampleDepth 3 } } }
"""


def test_heightmap_bling_scene_matches_oracle(gpu_ctx):
    """A heightMap primitive from .bling text (fBm elevation baked into a
    mesh with shading normals and uvs, Primitive/Heightmap.hs) renders on
    the GPU as in the oracle."""
    from bling_amd import bling_format
    b = bling_format.parse(HEIGHTMAP_BLING)
    assert b.flat.num_triangles == 39 * 29 * 2 and b.flat.normals is not None
    spec = b.spec(passes=2, seed=17)
    spec.variance = True
    g, gsq = render_gpu(gpu_ctx, b.flat, spec)
    o, osq, _ = pyoracle.render(b.flat, spec)
    assert np.isfinite(g).all() and g[..., 2].mean() > 0
    frac, zmean, zmax = compare(g, gsq, o, osq)
    assert frac < 0.01, (frac, zmean, zmax)
    mg, _ = mean_se(g, gsq)
    mo, _ = mean_se(o, osq)
    assert np.median(np.abs(mg - mo) / np.maximum(np.abs(mo), 1e-3)) < 1e-4


def test_translucent_matte_matches_oracle_and_closed_form(gpu_ctx):
    """transMatte's transmission lobe (brdfToBtdf of a Lambertian): a
    translucent plane under a surrounding uniform sky has direct radiance
    (kr + kt (1 - kr)) L; the same seed tracks the oracle."""
    from bling_amd.scene import Material, const
    from tests import cases
    kr, kt = 0.3, 0.7
    flat = cases.plane_under_sky(sky=1.0, material=Material.trans_matte(const(kr), const(kt), 0.0))
    spec = JobSpec(spp_nu=8, spp_nv=8, max_depth=1, sample_depth=1, passes=8, seed=5, variance=True)
    g, gsq = render_gpu(gpu_ctx, flat, spec)
    o, osq, _ = pyoracle.render(flat, spec)
    mg, se = mean_se(g, gsq)
    mo, _ = mean_se(o, osq)
    y = mg[..., 1].mean()
    s = np.sqrt((se[..., 1] ** 2).sum()) / mg[..., 1].size
    want = kr + kt * (1 - kr)
    assert abs(y - want) < 4 * s + 1e-4, (y, want, s)
    np.testing.assert_allclose(mg, mo, rtol=1e-4, atol=1e-6)


SUBSTRATE_BLING = """
imageSize 64 36
filter box
renderer { sampler sampled { sampler { stratified 2 2 } integrator { path maxDepth 5 sampleDepth 3 } } }
transform { lookAt { pos -5 12 -12 look 0 2 1 up 0 1 0 } }
camera { perspective fov 33 lensRadius 0 focalDistance 8.6 }
newTransform { }
material { matte kd { graphPaper 0.02 map { uv 15 15 0 0 } tex1 { constant rgbR 0.8 0.8 0.8 }
                      tex2 { constant rgbR 0.05 0.05 0.05 } } sigma { constant 0.005 } }
newTransform { rotateX 90 }
prim { shape { quad 50 50 } }
emission { rgbI 10 10 10 }
newTransform { rotateX -90 translate 0 20 0 }
prim { shape { quad 4 4 } }
emission { none }
newTransform { translate -3 2 0 }
material { substrate kd { constant rgbR 0.6 0.1 0.05 } ks { constant rgbR 0.8 0.8 0.8 }
           ka { constant rgbR 0.7 0.7 0.7 } urough { constant 0.005 } vrough { constant 0.0002 }
           depth { constant 0 } }
prim { shape { sphere radius 2 } }
transform { translate 6 0 0 }
material { substrate kd { constant rgbR 0.1 0.3 0.6 } ks { constant rgbR 0.5 0.5 0.5 }
           ka { constant rgbR 0.7 0.2 0.2 } urough { constant 0.0002 } vrough { constant 0.005 }
           depth { constant 0.5 } }
prim { shape { sphere radius 2 } }
newTransform { translate 0 2.5 4 }
material { substrate kd { graphPaper 0.1 map { uv 8 8 0 0 } tex1 { constant rgbR 0.7 0.7 0.2 }
                          tex2 { constant rgbR 0.02 0.02 0.02 } } ks { constant rgbR 0.3 0.3 0.3 }
           ka { constant rgbR 0.3 0.3 0.3 } urough { constant 0.05 } vrough { constant 0.05 }
           depth { constant 0.05 } }
prim { shape { sphere radius 2.5 } }
"""


def test_substrate_scene_matches_oracle(gpu_ctx):
    """substrate (FresnelBlend over the anisotropic distribution,
    Material.hs:111-127, Microfacet.hs:56-196) from .bling text: anisotropy
    along either axis, coatings with and without absorption, a textured
    diffuse layer; the same seed tracks the oracle, another seed is within
    3 sigma."""
    from bling_amd import bling_format
    b = bling_format.parse(SUBSTRATE_BLING)
    kinds = sorted({m.type for m in b.flat.materials})
    assert kinds == [abi.MAT_MATTE, abi.MAT_SUBSTRATE]
    spec = b.spec(passes=4, seed=23)
    spec.variance = True
    g, gsq = render_gpu(gpu_ctx, b.flat, spec)
    o, osq, _ = pyoracle.render(b.flat, spec)
    assert np.isfinite(g).all() and g[..., 2].mean() > 0
    frac, zmean, zmax = compare(g, gsq, o, osq)
    assert frac < 0.01, (frac, zmean, zmax)
    mg, _ = mean_se(g, gsq)
    mo, _ = mean_se(o, osq)
    assert np.median(np.abs(mg - mo) / np.maximum(np.abs(mo), 1e-3)) < 1e-4
    spec2 = b.spec(passes=4, seed=24)
    spec2.variance = True
    o2, osq2, _ = pyoracle.render(b.flat, spec2)
    frac, zmean, zmax = compare(g, gsq, o2, osq2)
    assert frac < 0.015, (frac, zmean, zmax)
    assert abs(zmean) < 0.08, zmean
    # the direct-lighting integrator's shading kernel on the same materials
    spec3 = b.spec(passes=4, seed=25)
    spec3.variance = True
    spec3.integrator = "direct"
    g3, gsq3 = render_gpu(gpu_ctx, b.flat, spec3)
    o3, osq3, _ = pyoracle.render(b.flat, spec3)
    assert np.isfinite(g3).all() and g3[..., 2].mean() > 0
    frac, zmean, zmax = compare(g3, gsq3, o3, osq3)
    assert frac < 0.01, (frac, zmean, zmax)
    mg, _ = mean_se(g3, gsq3)
    mo, _ = mean_se(o3, osq3)
    assert np.median(np.abs(mg - mo) / np.maximum(np.abs(mo), 1e-3)) < 1e-4


def test_path_recursion_two_mirrors_closed_form(gpu_ctx):
    """Two mirrors under a uniform sky (the oracle's pin of the path
    recursion, Integrator/Path.hs:66-87): r^2 L (1 + w) from maxDepth 2 on,
    0 at maxDepth 1, with and without Russian roulette from depth 1 (the
    stratified roulette sample continues exactly 3 of a pixel's 4 paths,
    each weighted 1 / 0.75)."""
    from tests import cases
    r, L = 0.9, 2.0
    flat = cases.two_mirrors_under_sky(r=r, sky=L)
    pdf_l = 1.0 / (2 * np.pi ** 2)
    w = 1.0 / (1.0 + pdf_l ** 2)
    for rr in (7, 0):
        for md, want in ((1, 0.0), (2, r * r * L * (1 + w)), (5, r * r * L * (1 + w))):
            spec = JobSpec(spp_nu=2, spp_nv=2, max_depth=md, sample_depth=3, rr_start_depth=rr, passes=1, seed=9)
            img, _ = render_gpu(gpu_ctx, flat, spec)
            np.testing.assert_allclose(img[..., 2] / img[..., 0], want, rtol=1e-5, atol=1e-6)


@pytest.mark.parametrize("name", ["gauss", "mitchell", "sinc", "triangle", "box"])
def test_film_filters_track_oracle(gpu_ctx, name):
    """Non-box filters splat a sample over several pixels, clipped to the
    16 x 16 tile prender renders it in (mkImageTile / addTile,
    Image.hs:108-120,178-199).  Same seed on both sides: per-pixel weight
    sums agree to float rounding (GPU atomics add in another order) and the
    pixel means track the oracle's."""
    from tests.test_oracle_closed_forms import FILTERS
    kind, p = FILTERS[name]
    flat = scenes.cornell(48)
    view = flat.view(45, 38)
    view.film.filter = kind
    for k in range(4):
        view.film.fparams[k] = p[k]
    spec = JobSpec(spp_nu=2, spp_nv=2, max_depth=4, sample_depth=3, rr_start_depth=3, passes=2, seed=17,
                   variance=True, view=view)
    g, gsq = render_gpu(gpu_ctx, flat, spec)
    o, osq, _ = pyoracle.render(flat, spec)
    assert np.isfinite(g).all()
    np.testing.assert_allclose(g[..., 0], o[..., 0], rtol=1e-5, atol=1e-5)
    mg = g[..., 1:] / g[..., :1]
    mo = o[..., 1:] / o[..., :1]
    ok = np.abs(o[..., 0]) > 1e-3
    rel = np.abs(mg - mo)[ok] / np.maximum(np.abs(mo[ok]), 1e-3)
    assert np.median(rel) < 1e-4, np.median(rel)


@pytest.mark.parametrize("filt, params, size, n", [
    (abi.FILTER_GAUSS, (5.0, 4.5, 0.2, 0.0), (33, 19), 1),     # 11 x 10 pixels a sample: several passes of a wave
    (abi.FILTER_GAUSS, (2.0, 2.0, 2.0, 0.0), (7, 5), 3),       # a film smaller than a tile and a run of pixels
    (abi.FILTER_TRIANGLE, (0.75, 3.1, 0.0, 0.0), (40, 17), 2),  # one column or two, clipped rows
])
def test_wide_filter_splats_keep_their_weights(gpu_ctx, filt, params, size, n):
    """Splats over several pixels are summed per wave before they reach the
    film; the same seed gives the oracle's weights and XYZ sums.  The weights
    are positive, and at most ~1000 of them meet in a pixel, so two orders of
    their float sums differ by less than 1000 * 2^-24 = 6e-5."""
    flat = scenes.cornell(48)
    view = flat.view(*size)
    view.film.filter = filt
    for k in range(4):
        view.film.fparams[k] = params[k]
    spec = JobSpec(spp_nu=n, spp_nv=n, max_depth=3, sample_depth=3, rr_start_depth=3, passes=2, seed=23,
                   variance=True, view=view)
    g, gsq = render_gpu(gpu_ctx, flat, spec)
    o, osq, _ = pyoracle.render(flat, spec)
    np.testing.assert_allclose(g[..., 0], o[..., 0], rtol=6e-5, atol=1e-7)
    for a, b in ((g[..., 1:], o[..., 1:]), (gsq, osq)):
        assert np.median(np.abs(a - b) / np.maximum(np.abs(b), 1e-3)) < 1e-4


@pytest.mark.parametrize("hidden", ["oren", "translucent", "glass", "textured"])
@pytest.mark.parametrize("lights", ["quad", "quad+sphere+sky", "disk+point+directional", "none"])
def test_lambert_kernel_matches_general_ones(gpu_ctx, lights, hidden):
    """Scenes of plain Lambert materials have a shading kernel of their own.
    A sphere walled in where no ray can reach it makes a scene take the
    general kernels (whole queue, or grouped with the Lambert classes split
    off) for the same paths: equal weights, and sums that differ by the order
    of the film's atomics only.  Matte, checkered and black surfaces, depths
    past the roulette."""
    from bling_amd import transform as T
    from bling_amd.scene import Material, SceneBuilder, const, rgb_refl
    from bling_amd.textures import Map3d, Tex

    def build(extra):
        sb = SceneBuilder()
        grey = sb.material(Material.matte(rgb_refl(0.7, 0.6, 0.5)))
        check = sb.material(Material.matte(rgb_refl(0.7, 0.7, 0.7)).textured(0, abi.TEX_CHECKER, (2.0, 2.0, 2.0),
                                                                              rgb_refl(0.1, 0.2, 0.6)))
        black = sb.material(Material.black())
        sb.mesh(np.array([[-4, 0, -4], [4, 0, -4], [4, 0, 4], [-4, 0, 4]], np.float32),
                np.array([[0, 1, 2], [0, 2, 3]]), material=check)
        v, f = scenes.unit_box()
        for k, m in enumerate((grey, black, grey)):
            sb.mesh(v, f, o2w=T.rotate_y(20 * k) @ T.translate((-1.5 + 1.5 * k, 0.5, 0.2 * k)), material=m)
        if extra:
            m = {"oren": Material.matte(const(0.5), sigma=0.5), "glass": Material.glass(1.5, const(1.0), const(1.0)),
                 "translucent": Material.trans_matte(const(0.3), const(0.3)),
                 "textured": Material.matte(const(0.5)).textured_inputs(
                     scalar={0: Tex.scale(0.3, 0.2, Tex.fbm(3, 0.5, Map3d.identity()))})}[extra]
            sb.shape(abi.SHAPE_SPHERE, (0.1,), o2w=T.translate((-1.5, 0.5, 0.0)), material=sb.material(m))
        up = T.rotate_x(-90) @ T.translate((0.5, 3.0, 0.0))
        if "quad" in lights:
            sb.shape(abi.SHAPE_QUAD, (0.5, 0.4), o2w=up, material=grey, emission=const(9.0))
        if "sphere" in lights:
            sb.shape(abi.SHAPE_SPHERE, (0.2,), o2w=T.translate((-1.0, 2.0, -1.0)), material=grey, emission=const(20.0))
        if "disk" in lights:
            sb.shape(abi.SHAPE_DISK, (0.0, 0.5, 0.0, 6.2831855), o2w=up, material=grey, emission=const(9.0))
        if "sky" in lights:
            sb.infinite_light(scenes.sky_gradient(16, 8), w2l=T.rotate_x(90))
        if "point" in lights:
            sb.point_light(const(6.0), (1.0, 2.0, -2.0))
            sb.directional_light(const(1.0), (0.3, 1.0, -0.2))
        sb.look(T.look_at((0.5, 2.2, -4.5), (0.0, 0.4, 0.0), (0, 1, 0)), 45.0, 45, 37)
        return sb.build()

    spec = JobSpec(spp_nu=3, spp_nv=3, max_depth=8, sample_depth=2, rr_start_depth=2, seed=31)
    a, _ = render_gpu(gpu_ctx, build(None), spec)
    b, _ = render_gpu(gpu_ctx, build(hidden), spec)
    assert np.array_equal(a[..., 0], b[..., 0])
    assert np.linalg.norm(a[..., 1:] - b[..., 1:]) <= 1e-6 * np.linalg.norm(b[..., 1:])
    assert lights == "none" or a[..., 2].sum() > 0


def _bumpy_obj(n=6):
    """An n x n grid of quads over [-1, 1]^2 (y up, a bump in the middle),
    with per-vertex normals and uvs; the second half of the faces under
    `usemtl gloss`, and a last `usemtl` with no faces after it."""
    lines = []
    for j in range(n + 1):
        for i in range(n + 1):
            x, z = -1 + 2 * i / n, -1 + 2 * j / n
            y = 0.4 * np.exp(-3 * (x * x + z * z))
            g = -2 * 3 * y
            nx, ny, nz = -g * x, 1.0, -g * z
            lines += ["v %.6f %.6f %.6f" % (x, y, z), "vn %.6f %.6f %.6f" % (nx, ny, nz),
                      "vt %.6f %.6f" % (i / n, j / n)]
    faces = []
    for j in range(n):
        for i in range(n):
            a = j * (n + 1) + i + 1
            q = (a, a + 1, a + n + 2, a + n + 1)
            faces.append("f " + " ".join("%d/%d/%d" % (k, k, k) for k in q))
    half = len(faces) // 2
    lines += faces[:half] + ["usemtl gloss"] + faces[half:] + ["usemtl unused"]
    return ("\n".join(lines) + "\n").encode()


def test_wavefront_bling_scene_matches_oracle(gpu_ctx, tmp_path):
    """A Wavefront mesh from .bling text (IO/WaveFront.hs: fans, untransformed
    normals, the second corner's uv and normal on the third, per-usemtl
    materials) renders on the GPU as in the oracle."""
    from bling_amd import bling_format
    (tmp_path / "bumpy.obj").write_bytes(_bumpy_obj())
    text = """
imageSize 48 48
filter box
transform { lookAt { pos 0 2.5 -3 look 0 0.2 0 up 0 1 0 } }
camera { perspective fov 50 lensRadius 0 focalDistance 1 }
newTransform { rotateY 20 translate 0 0 0.2 }
material { matte kd { graphPaper 0.1 map { uv 4 4 0 0 } tex1 { constant rgbR 0.8 0.3 0.2 } tex2 { constant rgbR 0.2 0.3 0.8 } } sigma { constant 0 } }
prim { waveFront "bumpy.obj" materials { "gloss" { plastic kd { constant rgbR 0.3 0.5 0.2 } ks { constant rgbR 0.4 0.4 0.4 } rough { constant 0.05 } } } }
newTransform { }
material { blackbody }
emission { rgbI 6 6 6 }
transform { rotateX -90 translate 0 3 0 }
prim { shape { quad 0.7 0.7 } }
emission { none }
light { infinite { } l { constant rgbI 0.2 0.2 0.3 } }
renderer { sampler sampled { sampler { stratified 4 4 } integrator { path maxDepth 5 sampleDepth 3 } } }
"""
    b = bling_format.parse(text, base=str(tmp_path))
    assert b.flat.num_triangles == 72 and b.flat.normals is not None
    spec = b.spec(passes=2, seed=19)
    spec.variance = True
    g, gsq = render_gpu(gpu_ctx, b.flat, spec)
    o, osq, _ = pyoracle.render(b.flat, spec)
    assert np.isfinite(g).all() and g[..., 2].mean() > 0
    assert np.array_equal(g[..., 0], o[..., 0])
    mg, _ = mean_se(g, gsq)
    mo, _ = mean_se(o, osq)
    assert np.median(np.abs(mg - mo) / np.maximum(np.abs(mo), 1e-3)) < 1e-4
    frac, zmean, zmax = compare(g, gsq, o, osq)
    assert frac < 0.01, (frac, zmean, zmax)
