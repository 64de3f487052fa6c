"""GPU path tracer vs the oracle on identical seeded inputs.

Both sides draw the same Owen-scrambled Sobol / ZSobol samples (pure
functions of pixel, sample index, dimension and seed), traverse the same
BVHs with bit-identical hit rules, evaluate the same elementary functions
(include/mtx_fmath.h) and run the same integrator with the same FP64
accumulation order, so at equal spp the accumulators agree bit for bit.
Bar (written here): FP64 sums and sample counts identical; the radiance
relMSE = mean((gpu - ref)^2 / (ref^2 + 1e-2)) is also reported and must be
<= 1e-4 (the tolerance the accuracy target states). Every case runs on both
the wavefront kernels (default) and the megakernel.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

REL_MSE_MAX = 1e-4


@pytest.fixture(scope="module")
def env():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    from mutracer_amd import render, scene
    return torch, render, scene


def rel_mse(a, b):
    return float(np.mean((a - b) ** 2 / (b * b + 1e-2)))


KERNELS = ["wavefront", "megakernel"]


def _both(orc, render, sc, w, h, spp, batches=None, **kw):
    rs = render.RenderScene(sc)
    tgt = render.RenderTarget(rs, w, h, **kw)
    for n in (batches or [spp]):
        tgt.render(n)
    tgt.synchronize()
    sums, counts = tgt.read_accumulators()
    okw = dict(bounces=kw.get("bounces", 8), candidates=kw.get("direct_light_candidates", 1),
               pattern=kw.get("pattern", "sobol"), seed=kw.get("sequence_seed", 0),
               max_samples=kw.get("max_samples", spp), clamping=kw.get("clamping", 0.0),
               sample_offset=kw.get("sample_sequence_offset", 0))
    ref = orc.OracleRenderer(sc, w, h, **okw).render(0, spp)
    return sums, counts, ref, tgt


def _check(sums, counts, ref, spp):
    assert np.all(counts == spp), "sample counts differ"
    g = sums / spp
    r = ref / spp
    err = rel_mse(g[..., 0:3], r[..., 0:3])
    print(f"relMSE={err:.3e}  mean gpu={g[..., 0:3].mean():.6f} ref={r[..., 0:3].mean():.6f}")
    assert err <= REL_MSE_MAX, f"radiance relMSE {err:.3e} > {REL_MSE_MAX}"
    assert np.abs(g[..., 4:11] - r[..., 4:11]).max() <= 1e-4, "albedo/normal AOVs differ"
    assert np.array_equal(g[..., 11], r[..., 11])
    assert np.array_equal(sums, ref), "FP64 accumulators differ from the oracle's"
    return err


@pytest.mark.parametrize("kernel", KERNELS)
def test_cornell_sobol(env, orc, kernel):
    torch, render, scene = env
    sc = scene.cornell_box()
    sums, counts, ref, _ = _both(orc, render, sc, 96, 96, 32, bounces=8, max_samples=32, kernel=kernel)
    _check(sums, counts, ref, 32)


@pytest.mark.parametrize("kernel", KERNELS)
def test_cornell_zsobol_candidates(env, orc, kernel):
    torch, render, scene = env
    sc = scene.cornell_box()
    sums, counts, ref, _ = _both(orc, render, sc, 64, 64, 16, bounces=8, pattern="zsobol", max_samples=64,
                                 direct_light_candidates=4, sequence_seed=7, kernel=kernel)
    _check(sums, counts, ref, 16)


@pytest.mark.parametrize("kernel", KERNELS)
def test_batches_equal_single_launch(env, orc, kernel):
    """Samples split over launches (and over wavefront generations) continue
    the per-pixel Sobol index."""
    torch, render, scene = env
    sc = scene.cornell_box()
    rs = render.RenderScene(sc)
    a = render.RenderTarget(rs, 48, 40, bounces=6, max_samples=12, kernel=kernel)
    a.render(12)
    b = render.RenderTarget(rs, 48, 40, bounces=6, max_samples=12, kernel=kernel,
                            max_paths_in_flight=48 * 40 * 2 + 7)
    for n in (5, 1, 6):
        b.render(n)
    sa, ca = a.read_accumulators()
    sb, cb = b.read_accumulators()
    assert np.array_equal(ca, cb)
    assert np.array_equal(sa, sb), "split launches must reproduce the single launch bit-exactly"
    assert b.stats()["samples"] == 12


@pytest.mark.parametrize("kernel", KERNELS)
def test_instanced_field_env(env, orc, kernel):
    """Reduced config-2 scene: metal / glass / coated instances, sky+sun env."""
    torch, render, scene = env
    sc = scene.instanced_field(n_instances=9, freq=10, env_size=(256, 128))
    sums, counts, ref, _ = _both(orc, render, sc, 96, 54, 8, bounces=12, max_samples=8, kernel=kernel,
                                 direct_light_candidates=4)
    _check(sums, counts, ref, 8)


@pytest.mark.parametrize("kernel", KERNELS)
def test_clamping_and_offset(env, orc, kernel):
    torch, render, scene = env
    sc = scene.instanced_field(n_instances=4, freq=6, env_size=(64, 32))
    sums, counts, ref, _ = _both(orc, render, sc, 40, 30, 6, bounces=5, max_samples=6, clamping=4.0,
                                 sample_sequence_offset=17, direct_light_candidates=2, kernel=kernel)
    _check(sums, counts, ref, 6)


@pytest.mark.parametrize("kernel", KERNELS)
def test_thin_lens(env, orc, kernel):
    """Aperture > 0: lens samples from the CAMERA_LENS dimension, focus plane
    perpendicular to the view direction (rayTrace.compute.ts:1196-1205)."""
    torch, render, scene = env
    sc = scene.instanced_field(n_instances=6, freq=6, env_size=(64, 32))
    sc.camera.aperture = 0.4
    sc.camera.focus_distance = 12.0
    sums, counts, ref, _ = _both(orc, render, sc, 48, 32, 6, bounces=6, max_samples=8, kernel=kernel,
                                 direct_light_candidates=2)
    _check(sums, counts, ref, 6)


@pytest.mark.parametrize("kernel", KERNELS)
def test_fuzz_materials(env, orc, kernel):
    """Fuzz layered over diffuse, metal, coated and glass bases."""
    torch, render, scene = env
    sc = scene.instanced_field(n_instances=8, freq=6, env_size=(64, 32))
    for k, m in enumerate(sc.materials):
        if k % 2 == 0:
            m.fuzz_weight = 0.3 + 0.1 * (k % 5)
            m.fuzz_color = (0.9, 0.5 + 0.05 * k, 0.3)
            m.fuzz_roughness = 0.2 + 0.15 * (k % 4)
    sums, counts, ref, _ = _both(orc, render, sc, 48, 32, 6, bounces=8, max_samples=6, kernel=kernel,
                                 direct_light_candidates=2)
    _check(sums, counts, ref, 6)


@pytest.mark.parametrize("kernel", KERNELS)
def test_thin_walled_and_subsurface(env, orc, kernel):
    """Thin-walled glass (smooth and rough, tinted), subsurface boundaries
    of solids and thin subsurface sheets, some under a coat."""
    torch, render, scene = env
    sc = scene.instanced_field(n_instances=10, freq=6, env_size=(64, 32))
    for k, m in enumerate(sc.materials):
        if k % 3 == 0:
            m.thin_walled = True
            m.transmission_weight = 1.0 if k % 2 == 0 else 0.0
            m.subsurface_weight = 0.0 if k % 2 == 0 else 0.7
            m.transmission_color = (0.9, 0.7, 0.5)
            m.specular_roughness = 0.05 * (k % 4)
        elif k % 3 == 1:
            m.subsurface_weight = 0.6
            m.subsurface_color = (0.8, 0.4, 0.3)
            m.coat_weight = 0.5 if k % 2 else 0.0
    sums, counts, ref, _ = _both(orc, render, sc, 48, 32, 6, bounces=10, max_samples=6, kernel=kernel,
                                 direct_light_candidates=3)
    _check(sums, counts, ref, 6)


@pytest.mark.parametrize("kernel", KERNELS)
def test_random_pattern(env, orc, kernel):
    """Random pattern: Halton jitter per sample index, one pcg4d stream per
    path drawn in the reference's call order (lens, alpha coverage, NEE
    candidates with the discarded replacement draw, BSDF, roulette), over
    split launches and a sample offset."""
    torch, render, scene = env
    sc = scene.instanced_field(n_instances=6, freq=6, env_size=(64, 32))
    sc.camera.aperture = 0.3
    sc.camera.focus_distance = 12.0
    sums, counts, ref, _ = _both(orc, render, sc, 48, 32, 6, batches=[2, 1, 3], bounces=8, max_samples=6,
                                 kernel=kernel, pattern="random", sequence_seed=3, direct_light_candidates=3,
                                 sample_sequence_offset=5)
    _check(sums, counts, ref, 6)


@pytest.mark.parametrize("tail_paths", [0, 1500])
def test_random_pattern_tail_kernel(env, orc, tail_paths):
    """The pcg4d state of each path passes between the wavefront kernels and
    the tail kernel through device memory."""
    torch, render, scene = env
    sc = scene.cornell_box()
    rs = render.RenderScene(sc)
    t = render.RenderTarget(rs, 40, 30, bounces=8, direct_light_candidates=2, max_samples=4, pattern="random",
                            sequence_seed=21)
    t.set_tuning(tail_paths=tail_paths)
    t.render(4)
    sums, counts = t.read_accumulators()
    ref = orc.OracleRenderer(sc, 40, 30, bounces=8, candidates=2, max_samples=4, pattern="random",
                             seed=21).render(0, 4)
    assert np.all(counts == 4)
    assert np.array_equal(sums, ref)


@pytest.mark.parametrize("kernel", KERNELS)
def test_all_light_types(env, orc, kernel):
    """Rect, sphere, point, spot (point and finite), directional, disk and
    cylinder lights together with the environment: NEE candidates pick
    among all of them, BSDF continuations hit the hittable ones."""
    torch, render, scene = env
    sc = scene.instanced_field(n_instances=6, freq=6, env_size=(64, 32))
    sc.lights = [
        scene.RectLight(position=(2.0, 4.0, 0.0), u=(1.0, 0.0, 0.0), v=(0.0, 0.0, 1.0), intensity=6.0),
        scene.SphereLight(position=(-3.0, 3.0, 1.0), radius=0.5, color=(1.0, 0.8, 0.6), intensity=4.0),
        scene.SphereLight(position=(0.0, 5.0, -2.0), radius=0.0, intensity=20.0),
        scene.SpotLight(position=(4.0, 4.0, 4.0), direction=(-1.0, -1.0, -1.0), inner_angle=15, outer_angle=30,
                        intensity=40.0),
        scene.SpotLight(position=(-4.0, 3.0, -4.0), direction=(1.0, -1.0, 1.0), radius=0.3, inner_angle=25,
                        outer_angle=40, intensity=30.0),
        scene.DirectionalLight(direction=(0.3, -1.0, 0.2), color=(1.0, 0.9, 0.8), intensity=1.5),
        scene.DiskLight(position=(0.0, 3.5, 3.0), direction=(0.0, -1.0, -0.3), radius=0.6, intensity=5.0),
        scene.CylinderLight(position=(-2.0, 2.5, -3.0), axis=(1.0, 0.0, 0.2), radial=(0.0, 1.0, 0.0), radius=0.2,
                            length=2.0, intensity=6.0, normalize=False),
    ]
    sums, counts, ref, _ = _both(orc, render, sc, 64, 40, 6, bounces=6, max_samples=8, kernel=kernel,
                                 direct_light_candidates=4)
    _check(sums, counts, ref, 6)


@pytest.mark.parametrize("kernel", KERNELS)
def test_emissive_instances(env, orc, kernel):
    """Emissive meshes are triangle lights (NEE over their world-space
    triangles, MIS-weighted emission on BSDF hits) next to the environment
    and an analytic light."""
    torch, render, scene = env
    sc = scene.instanced_field(n_instances=6, freq=4, env_size=(64, 32))
    sc.materials[2].emission = (4.0, 3.0, 2.0)
    sc.materials[4].emission = (0.5, 2.0, 6.0)
    sc.materials[4].double_sided = True
    sc.lights = [scene.SphereLight(position=(1.0, 4.0, 2.0), radius=0.3, intensity=8.0)]
    sums, counts, ref, _ = _both(orc, render, sc, 48, 32, 6, bounces=6, max_samples=8, kernel=kernel,
                                 direct_light_candidates=4)
    _check(sums, counts, ref, 6)


def _resolve_expected(sums):
    """The output pass of WGPURayTraceOutput.ts:32-92 on the sums (bottom row
    first), evaluated per pixel in Python floats."""
    h, w, _ = sums.shape
    out = {k: np.zeros((h, w, 4)) for k in ("color", "albedo", "normal")}
    for y in range(h):
        for x in range(w):
            s = [float(v) for v in sums[y, x]]
            n, hit = s[11], s[7]
            if n <= 0:
                continue
            total = max(n, 1.0)
            div = hit if hit > 0 else total
            out["color"][y, x] = [s[0] / div, s[1] / div, s[2] / div, s[3] / total]
            out["albedo"][y, x] = [s[4] / total, s[5] / total, s[6] / total, min(max(hit / total, 0.0), 1.0)]
            if s[8] * s[8] + s[9] * s[9] + s[10] * s[10] > 0.1:
                out["normal"][y, x] = [s[8] / total * 0.5 + 0.5, s[9] / total * 0.5 + 0.5,
                                       s[10] / total * 0.5 + 0.5, 1.0]
    return {k: v[::-1].astype(np.float32) for k, v in out.items()}


def test_read_pixels_resolve(env, orc):
    """Sky pixels without an environment are blank (hit count 0): their color
    divides by the sample count, geometry pixels by the hit count."""
    torch, render, scene = env
    sc = scene.instanced_field(n_instances=4, freq=4, env_size=(64, 32))
    sc.env = None
    rs = render.RenderScene(sc)
    t = render.RenderTarget(rs, 48, 32, bounces=4, max_samples=4)
    t.render(3)
    sums, counts = t.read_accumulators()
    assert (sums[..., 7] == 0).any() and (sums[..., 7] > 0).any()
    exp = _resolve_expected(sums)
    for kind in ("color", "albedo", "normal"):
        assert np.array_equal(t.read_pixels(kind), exp[kind]), kind
    assert t.stats()["rays"] > 0
    t.restart_samples()
    assert not t.read_pixels("color").any()  # no samples: zeros


@pytest.mark.parametrize("kernel", KERNELS)
def test_counted_launch_matches_plain(env, orc, kernel):
    """The instrumented launch renders the same samples as the plain one."""
    torch, render, scene = env
    sc = scene.instanced_field(n_instances=6, freq=8, env_size=(64, 32))
    rs = render.RenderScene(sc)
    a = render.RenderTarget(rs, 64, 48, bounces=6, direct_light_candidates=2, max_samples=4, kernel=kernel)
    b = render.RenderTarget(rs, 64, 48, bounces=6, direct_light_candidates=2, max_samples=4, kernel=kernel)
    if kernel == "wavefront":
        b.set_tuning(tail_paths=3000)  # the tail kernel takes over mid-generation
    a.render(4)
    work = b.render_counted(4)
    sa, _ = a.read_accumulators()
    sb, _ = b.read_accumulators()
    assert np.array_equal(sa, sb)
    rays = b.stats()["rays"]
    assert 0 < work["hits"] <= rays - work["shadow_rays"]
    assert work["box_tests"] > work["tri_tests"] > 0
    assert work["instance_visits"] >= work["hits"]
    assert work["shadow_box_tests"] > work["shadow_tri_tests"] > 0
    assert work["closest_rays"] + work["shadow_rays"] == rays
    assert work["wavefront"]["box_tests"] + work["tail"]["box_tests"] == work["box_tests"]
    if kernel == "wavefront":
        assert work["wavefront"]["closest_rays"] > 0 and work["tail"]["closest_rays"] > 0


def test_wavefront_equals_megakernel_large(env, orc):
    """Both kernel forms on a 1M-triangle-class scene at 256x144, 4 spp."""
    torch, render, scene = env
    sc = scene.instanced_field(n_instances=64, freq=28, env_size=(1024, 512))
    rs = render.RenderScene(sc)
    out = []
    for kernel in KERNELS:
        t = render.RenderTarget(rs, 256, 144, bounces=12, direct_light_candidates=4, max_samples=4, kernel=kernel)
        t.render(4)
        out.append(t.read_accumulators())
    assert np.array_equal(out[0][1], out[1][1])
    assert np.array_equal(out[0][0], out[1][0])


# A wave of the shade kernel takes 64 paths at a time from 2048 waves' shares
# of the queue: a partial wave, one share each, two (a class fills once), five
# (classes fill repeatedly, two at once, leftovers of several).
@pytest.mark.parametrize("w,h,spp", [(9, 5, 1), (256, 128, 4), (320, 200, 4), (400, 250, 6)])
@pytest.mark.parametrize("tail_paths", [0, 1 << 16])
def test_shading_classes_match_oracle(env, orc, w, h, spp, tail_paths):
    """Paths shaded grouped by what they hit (diffuse, coat, metal, glass,
    nothing) give the oracle's sums, with the shadow rays of an event in the
    next event's launch (no tail) and in their own."""
    torch, render, scene = env
    sc = scene.instanced_field(n_instances=13, freq=5, env_size=(64, 32))
    t = render.RenderTarget(render.RenderScene(sc), w, h, bounces=3, direct_light_candidates=2, max_samples=spp)
    t.set_tuning(tail_paths=tail_paths)
    t.render(spp)
    sums, counts = t.read_accumulators()
    ref = orc.OracleRenderer(sc, w, h, bounces=3, candidates=2, max_samples=spp).render(0, spp)
    assert np.all(counts == spp)
    assert np.array_equal(sums, ref)


@pytest.mark.parametrize("kind", ["diffuse", "glass", "masked", "subsurface"])
@pytest.mark.parametrize("bounces", [0, 1, 2, 7])
def test_event_limit_of_opaque_scenes(env, orc, kind, bounces):
    """Scenes that let no path past `bounces` + 1 events launch no more of
    them; one transmitting, masked or subsurface material lifts that."""
    torch, render, scene = env
    sc = scene.cornell_box()
    more = dict(diffuse={}, glass=dict(transmission_weight=1.0, specular_roughness=0.1),
                masked=dict(alpha_mode="mask", opacity=0.2, alpha_cutoff=0.5),
                subsurface=dict(subsurface_weight=0.6))[kind]
    sc.materials.append(scene.Material(base_color=(0.7, 0.8, 0.9), **more))
    sc.instance_material[-1] = len(sc.materials) - 1
    t = render.RenderTarget(render.RenderScene(sc), 40, 32, bounces=bounces, max_samples=4)
    t.render(4)
    sums, _ = t.read_accumulators()
    assert np.array_equal(sums, orc.OracleRenderer(sc, 40, 32, bounces=bounces, candidates=1, max_samples=4).render(0, 4))


# One pixel, a partial block, a block edge, rows that straddle blocks.
@pytest.mark.parametrize("w,h", [(1, 1), (7, 5), (256, 1), (131, 4)])
def test_read_pixels_kinds(env, w, h):
    """Every pixel kind from the accumulators' sums in f64, rounded once."""
    torch, render, scene = env
    t = render.RenderTarget(render.RenderScene(scene.cornell_box()), w, h, bounces=3, max_samples=3)
    t.render(3)
    sums, counts = t.read_accumulators()
    sums, n = sums[::-1], counts[::-1].astype(np.float64)[..., None]
    total, hit = np.maximum(sums[..., 11:12], 1.0), sums[..., 7:8]
    lum = (0.2126 * sums[..., 0:1] + 0.7152 * sums[..., 1:2] + 0.0722 * sums[..., 2:3]) / n
    var = np.maximum(0.0, sums[..., 12:13] / n - lum * lum) / n
    nrm = sums[..., 8:11]
    valid = (nrm[..., 0:1] * nrm[..., 0:1] + nrm[..., 1:2] * nrm[..., 1:2] + nrm[..., 2:3] * nrm[..., 2:3]) > 0.1
    zero, one = np.zeros_like(n), np.ones_like(n)
    exp = dict(color=np.concatenate([sums[..., 0:3] / np.where(hit > 0, hit, total), sums[..., 3:4] / total], 2),
               albedo=np.concatenate([sums[..., 4:7] / total, np.clip(hit / total, 0, 1)], 2),
               normal=np.where(valid, np.concatenate([nrm / total * 0.5 + 0.5, one], 2), 0.0),
               variance=np.concatenate([var, zero, zero, one], 2))
    for kind, e in exp.items():
        assert np.array_equal(t.read_pixels(kind), e.astype(np.float32)), kind


def test_read_pixels_of_partly_sampled_images(env):
    """Pixels with fewer samples than others and with none: per-pixel sample
    targets of 0 to 3 (zero resolves to 0; the variance's alpha is 1)."""
    torch, render, scene = env
    w, h = 61, 37
    t = render.RenderTarget(render.RenderScene(scene.cornell_box()), w, h, bounces=3, max_samples=3)
    targets = np.random.default_rng(4).integers(0, 4, (h, w)).astype(np.float32)
    t.set_sample_targets(targets)
    t.render(3)
    sums, counts = t.read_accumulators()
    assert np.array_equal(counts, targets.astype(counts.dtype)) and len(np.unique(counts)) == 4
    none = (counts == 0)[::-1]
    sums, n = sums[::-1], np.maximum(counts[::-1], 1).astype(np.float64)
    color = sums[..., 0:4] / np.maximum(sums[..., 11:12], 1.0)
    hit = sums[..., 7]
    color[..., 0:3] = np.where(hit[..., None] > 0, sums[..., 0:3] / np.where(hit > 0, hit, 1.0)[..., None], color[..., 0:3])
    lum = (0.2126 * sums[..., 0] + 0.7152 * sums[..., 1] + 0.0722 * sums[..., 2]) / n
    var = np.maximum(0.0, sums[..., 12] / n - lum * lum) / n
    got = {k: t.read_pixels(k) for k in ("color", "albedo", "normal", "variance")}
    assert np.array_equal(got["color"], color.astype(np.float32))
    assert np.array_equal(got["variance"][..., 0], var.astype(np.float32)) and np.all(got["variance"][..., 3] == 1)
    for k in ("color", "albedo", "normal"):
        assert np.all(got[k][none] == 0) and np.any(got[k][~none] != 0), k


@pytest.mark.parametrize("h,kept", [(2048, 64), (2049, 0)])
def test_read_pixels_keeps_at_most_64_mib(env, h, kept):
    """The device image of read_pixels stays for the next call up to 2048 x
    2048 pixels; a larger one is given back."""
    torch, render, scene = env
    rs = render.RenderScene(scene.cornell_box())
    small = render.RenderTarget(rs, 8, 8, bounces=1)
    small.read_pixels()  # the kernel's code is loaded
    t = render.RenderTarget(rs, 2048, h, bounces=1)
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    for kind in ("color", "albedo"):
        assert not t.read_pixels(kind).any()
        assert abs((free - torch.cuda.mem_get_info()[0]) / 2**20 - kept) <= 4


@pytest.mark.parametrize("tuning", [
    dict(lds_stack=16),
    dict(trace_kernel=1, use_graphs=0),
    dict(lds_stack=24, trace_oversubscription=2),
    dict(lds_stack=32, shade_oversubscription=3, max_paths_in_flight=3000),
    dict(shade_waves_per_simd=2),
    dict(shade_waves_per_simd=4, shade_oversubscription=2),
    dict(tail_paths=0),
    dict(tail_paths=1500),
    dict(tail_paths=1 << 30),
    dict(use_graphs=0, tail_paths=3000, max_paths_in_flight=9000),
    dict(lds_stack_closest=16),
    dict(lds_stack_closest=32, lds_stack=24),
    dict(queue_sort=1),
    dict(queue_sort=1, tail_paths=0, max_paths_in_flight=9000),
])
def test_wavefront_tunings_match_oracle(env, orc, tuning):
    """Every launch shape of the wavefront kernels yields the oracle's sums,
    wherever the tail kernel takes over (never, mid-generation, at event 0)."""
    torch, render, scene = env
    sc = scene.instanced_field(n_instances=12, freq=12, env_size=(128, 64))
    rs = render.RenderScene(sc)
    t = render.RenderTarget(rs, 80, 45, bounces=10, direct_light_candidates=3, max_samples=6)
    t.set_tuning(**tuning)
    got = t.tuning()
    assert all(got[k] == v for k, v in tuning.items())
    t.render(6)
    sums, counts = t.read_accumulators()
    ref = orc.OracleRenderer(sc, 80, 45, bounces=10, candidates=3, max_samples=6).render(0, 6)
    assert np.all(counts == 6)
    assert np.array_equal(sums, ref)


def test_graph_replays_match_eager(env, orc):
    """Captured generations replayed between unrelated eager work give the
    eager launches' bits (and the oracle's)."""
    torch, render, scene = env
    sc = scene.cornell_box()
    rs = render.RenderScene(sc)
    kw = dict(bounces=6, max_samples=8, max_paths_in_flight=48 * 40 * 2)
    g = render.RenderTarget(rs, 48, 40, **kw)
    e = render.RenderTarget(rs, 48, 40, **kw)
    e.set_tuning(use_graphs=0)
    for k in range(4):
        g.render(2)
        junk = torch.randn(1 << 16, device="cuda").cumsum(0)
        e.render(2)
        torch.cuda.synchronize()
        assert float(junk[-1]) == float(junk[-1])
        sg, cg = g.read_accumulators()
        se, ce = e.read_accumulators()
        assert np.array_equal(cg, ce) and np.array_equal(sg, se), f"replay {k} differs"
    t = g.tuning()
    assert t["graph_captures"] == 1 and t["graph_replays"] == 4
    assert e.tuning()["graph_replays"] == 0
    ref = orc.OracleRenderer(sc, 48, 40, bounces=6, max_samples=8).render(0, 8)
    assert np.array_equal(g.read_accumulators()[0], ref)


def test_targets_rendering_side_by_side(env):
    """Two targets whose renders are in flight together on the default stream
    (their graphs run on streams of their own, the traversal stacks' spill
    memory is shared), with ray queries of another thread in between, give
    the sums each gives alone."""
    import threading
    torch, render, scene = env
    from mutracer_amd import accel, workloads as W
    scenes = [scene.instanced_field(n_instances=n, freq=f, env_size=(64, 32)) for n, f in ((20, 16), (9, 22))]
    kw = dict(bounces=6, direct_light_candidates=2, max_samples=12)
    targets = [render.RenderTarget(render.RenderScene(sc), 200, 120, **kw) for sc in scenes]
    alone = []
    for t in targets:
        for _ in range(6):
            t.render(2)
        alone.append(t.read_accumulators()[0])
        t.restart_samples()
    pos, idx = W.random_triangles(30000, seed=3)
    acc = accel.Accel([accel.Blas(pos, idx)], [0], [W.identity_transform()])
    rays = torch.from_numpy(W.pinhole_rays(300)).cuda()
    expect = torch.zeros((rays.shape[0], 8), dtype=torch.int32, device="cuda")
    acc.trace_closest(rays, expect)
    hits = [torch.zeros_like(expect) for _ in range(12)]
    torch.cuda.synchronize()
    bad = []

    def ask():
        try:
            for h in hits:
                acc.trace_closest(rays, h)
        except Exception as e:
            bad.append(e)

    other = threading.Thread(target=ask)
    other.start()
    for _ in range(6):
        for t in targets:
            t.render(2)
    other.join()
    torch.cuda.synchronize()
    assert not bad and all(torch.equal(h, expect) for h in hits)
    for t, ref in zip(targets, alone):
        sums, counts = t.read_accumulators()
        assert np.all(counts == 12) and np.array_equal(sums, ref)


def test_autotune(env, orc, tmp_path):
    torch, render, scene = env
    from mutracer_amd import autotune
    sc = scene.instanced_field(n_instances=6, freq=8, env_size=(64, 32))
    rs = render.RenderScene(sc)
    t = render.RenderTarget(rs, 96, 64, bounces=6, direct_light_candidates=2, max_samples=4)
    best = autotune.tune(t, samples=1, cache_path=str(tmp_path / "tune.json"))
    for k, v in best.items():
        if k in autotune.SPACE:
            assert v in autotune.SPACE[k] or k == "lds_stack"
    again = autotune.tune(t, samples=1, cache_path=str(tmp_path / "tune.json"))
    assert again == best
    t.restart_samples()
    t.render(4)
    ref = orc.OracleRenderer(sc, 96, 64, bounces=6, candidates=2, max_samples=4).render(0, 4)
    assert np.array_equal(t.read_accumulators()[0], ref)


def test_autotune_measures_replayed_graphs(env):
    torch, render, scene = env
    from mutracer_amd import autotune
    t = render.RenderTarget(render.RenderScene(scene.cornell_box()), 32, 24, bounces=3, max_samples=2)
    before = t.tuning()
    assert autotune.probe(t, before, 2) > 0.0
    after = t.tuning()
    assert after["graph_captures"] == 1 and after["graph_replays"] >= 4


@pytest.mark.parametrize("kernel", KERNELS)
def test_adaptive_converge(env, orc, kernel):
    """Pilot moments -> per-tile plan (the reference formula, recomputed here
    in numpy) -> final pass whose pixels stop at their targets and continue
    the Sobol sequence after the pilot samples (checked against the oracle)."""
    torch, render, scene = env
    sc = scene.cornell_box()
    rs = render.RenderScene(sc)
    W, H, S, pilot = 40, 32, 24, 4
    t = render.RenderTarget(rs, W, H, bounces=5, max_samples=S, kernel=kernel)
    t.render(pilot)
    sums, counts = t.read_accumulators()
    mx, avg, tv = t.plan_adaptive(S, tile_size=8, absolute_error=0.05, relative_error=0.1)
    # reference formula (offlineAdaptive.compute.ts:29-106), per 8x8 tile
    n = counts.astype(np.float64)
    mean = (0.2126 * sums[..., 0] + 0.7152 * sums[..., 1] + 0.0722 * sums[..., 2]) / n
    var = np.maximum(sums[..., 12] / n - mean * mean, 0) * n / (n - 1)
    want = np.zeros((H, W))
    for ty in range(H // 8):
        for tx in range(W // 8):
            sl = (slice(ty * 8, ty * 8 + 8), slice(tx * 8, tx * 8 + 8))
            tol = 0.05 + 0.1 * abs(mean[sl].mean())
            req = np.ceil(1.96 ** 2 * var[sl].max() / max(tol * tol, 1e-16))
            want[sl] = min(S, max(16, req))
            assert abs(tv[ty, tx] - var[sl].max()) <= 1e-12 * max(1.0, var[sl].max())
    assert mx == int(want.max()) and abs(avg - want.mean()) < 1e-9
    t.restart_samples()
    t.set_sample_offset(pilot)
    t.render(mx)
    sums2, counts2 = t.read_accumulators()
    assert np.array_equal(counts2, want.astype(np.uint32))
    for v in np.unique(want):
        ref = orc.OracleRenderer(sc, W, H, bounces=5, max_samples=S, sample_offset=pilot).render(0, int(v))
        sel = want == v
        assert np.array_equal(sums2[sel], ref[sel])
    t.set_sample_offset(0)
    img, info = render.Render(t).converge(S, adaptive=dict(pilot_samples=pilot, tile_size=8, absolute_error=0.05,
                                                            relative_error=0.1))
    assert info["adaptive"] and info["samples"] == mx
    assert np.array_equal(t.read_accumulators()[0], sums2)
