"""GPU two-level traversal vs the oracle: bit-exact closest-hit IDs and t.

For identical f32 rays the HIP traversal must return the same hit flag,
source instance, source triangle, t bits and barycentric bits as the
oracle's reference-order traversal (intersect.wgsl.ts getBVHTraverseCode).
Any-hit occlusion and the per-ray visit counters are compared as well.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def env():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    from mutracer_amd import accel, workloads
    return torch, accel, workloads


def _gpu_closest(torch, acc, rays, double_sided=False):
    r = torch.from_numpy(rays).cuda()
    h = torch.zeros((rays.shape[0], 8), dtype=torch.int32, device="cuda")
    acc.trace_closest(r, h, double_sided=double_sided)
    torch.cuda.synchronize()
    return h.cpu().numpy().view(np.uint32)


def _compare(scene, ref_hits, gpu_hits, orc):
    hit, inst, tri, tbits = orc.hits_to_ids(scene, ref_hits)
    g = gpu_hits
    assert np.array_equal(g[:, 0].astype(bool), hit), "hit flags differ"
    assert np.array_equal(g[hit, 1].view(np.int32), inst[hit]), "instance ids differ"
    assert np.array_equal(g[hit, 2].view(np.int32), tri[hit]), "triangle ids differ"
    assert np.array_equal(g[hit, 3], tbits[hit]), "t bits differ"
    assert np.array_equal(g[hit, 4:7], ref_hits[hit, 4:7]), "barycentric bits differ"
    return hit.mean()


def _c3_scene(orc, accel, W, ntris, res, bins=32):
    pos, idx = W.random_triangles(ntris, seed=3)
    scene = orc.assemble_scene([dict(positions=pos, indices=idx)],
                               dict(mesh=[0], transform=[W.identity_transform()], material=[0]),
                               blas_bins=bins, material_double_sided=[1])
    blas = accel.Blas(pos, idx, bins)
    acc = accel.Accel([blas], [0], [W.identity_transform()], material=[0], double_sided=[1])
    return pos, idx, scene, acc, blas


@pytest.mark.parametrize("ntris,res", [(2000, 64), (100000, 192)])
def test_microbench_scaled_bit_exact(orc, env, ntris, res):
    torch, accel, W = env
    print(f"microbench ntris={ntris} res={res}", flush=True)
    pos, idx, scene, acc, _ = _c3_scene(orc, accel, W, ntris, res)
    prim = W.pinhole_rays(res)
    ref = scene.closest(prim)
    got = _gpu_closest(torch, acc, prim)
    frac = _compare(scene, ref, got, orc)
    assert frac > (0.2 if ntris >= 100000 else 0.005)
    # bounce rays from the primary hits, about the geometric normal
    hit = ref[:, 0].astype(bool)
    t = ref[hit, 3].view(np.float32)
    p = prim[hit, 0:3] + prim[hit, 4:7] * t[:, None]
    tri = scene.record_triangle[ref[hit, 2]]
    v = pos[idx.reshape(-1, 3)[tri]]
    n = np.cross(v[:, 1] - v[:, 0], v[:, 2] - v[:, 0])
    n *= np.where((n * prim[hit, 4:7]).sum(1, keepdims=True) > 0, -1, 1)
    bounce = W.hemisphere_bounces(p, n, prim.shape[0], seed=0)
    ref_b = scene.closest(bounce)
    got_b = _gpu_closest(torch, acc, bounce)
    _compare(scene, ref_b, got_b, orc)


def test_single_sided_culling_and_any_hit(orc, env):
    torch, accel, W = env
    pos, idx = W.sphere_mesh(40, 20, radius=0.4)
    pos = pos + np.float32(0.5)
    scene = orc.assemble_scene([dict(positions=pos, indices=idx)],
                               dict(mesh=[0], transform=[W.identity_transform()], material=[0]),
                               material_double_sided=[0])
    acc = accel.Accel([accel.Blas(pos, idx)], [0], [W.identity_transform()], material=[0], double_sided=[0])
    rays = W.pinhole_rays(96)
    # from inside the sphere too: back faces are culled for single-sided materials
    inner = rays.copy()
    inner[:, 0:3] = 0.5
    for rr in (rays, inner):
        _compare(scene, scene.closest(rr), _gpu_closest(torch, acc, rr), orc)
        _compare(scene, scene.closest(rr, double_sided=True), _gpu_closest(torch, acc, rr, True), orc)
    short = rays.copy()
    short[:, 3] = np.linspace(0.0, 2.5, short.shape[0], dtype=np.float32)
    r = torch.from_numpy(short).cuda()
    occ = torch.zeros(short.shape[0], dtype=torch.int32, device="cuda")
    acc.trace_any(r, occ)
    torch.cuda.synchronize()
    assert np.array_equal(occ.cpu().numpy().astype(np.uint32), scene.any(short))


def test_instanced_scene_bit_exact(orc, env):
    torch, accel, W = env
    rng = np.random.default_rng(7)
    meshes = [W.sphere_mesh(24, 12), W.random_triangles(4000, seed=5), W.sphere_mesh(8, 4)]
    n = 48
    mesh_idx = rng.integers(0, 3, n)
    tr = []
    for i in range(n):
        q = rng.normal(size=4)
        q /= np.linalg.norm(q)
        tr.append(W.trs(rng.random(3) * 6 - 3, q, float(rng.lognormal(0, 0.3))))
    tr = np.array(tr)
    mats = rng.integers(0, 2, n)
    ds = [0, 1]
    scene = orc.assemble_scene([dict(positions=m[0], indices=m[1]) for m in meshes],
                               dict(mesh=mesh_idx, transform=tr, material=mats), material_double_sided=ds)
    blases = [accel.Blas(m[0], m[1]) for m in meshes]
    acc = accel.Accel(blases, mesh_idx, tr, material=mats, double_sided=[ds[m] for m in mats])
    rays = W.pinhole_rays(160, eye=(0, 0, -9), target=(0, 0, 0), fov_deg=50)
    frac = _compare(scene, scene.closest(rays), _gpu_closest(torch, acc, rays), orc)
    assert frac > 0.05
    # counters equal the oracle's instrumented traversal
    r = torch.from_numpy(rays).cuda()
    cnt = torch.zeros((rays.shape[0], 3), dtype=torch.int32, device="cuda")
    acc.trace_counters(r, cnt)
    torch.cuda.synchronize()
    _, st = scene.closest(rays, stats=True)
    assert np.array_equal(cnt.cpu().numpy().astype(np.uint32), st)


@pytest.fixture(scope="module")
def queue_scene(orc, env):
    """Instances in TLAS leaves of one and of several (coincident ones cannot
    be split), meshes whose root is a leaf, both cullings; rays that start
    inside and outside, short, with zero, infinite and NaN components."""
    torch, accel, W = env
    rng = np.random.default_rng(21)
    one = (np.array([[-1, -1, 0], [1, -1, 0], [0, 1, 0]], np.float32), np.arange(3, dtype=np.uint32))
    meshes = [W.sphere_mesh(20, 10), W.random_triangles(1500, mu=-2.0, seed=9), one]
    mesh_idx, tr = [], []
    for i in range(24):
        q = rng.normal(size=4)
        q /= np.linalg.norm(q)
        t = W.trs(rng.random(3) * 5 - 2.5, q, float(rng.lognormal(0, 0.3)))
        for _ in range(5 if i % 8 == 0 else 1):
            mesh_idx.append(i % 3)
            tr.append(t)
    tr = np.array(tr)
    mats = rng.integers(0, 2, len(mesh_idx))
    scene = orc.assemble_scene([dict(positions=m[0], indices=m[1]) for m in meshes],
                               dict(mesh=mesh_idx, transform=tr, material=mats), material_double_sided=[0, 1])
    acc = accel.Accel([accel.Blas(m[0], m[1]) for m in meshes], mesh_idx, tr, material=mats,
                      double_sided=[int(m) for m in mats])
    n = 400_000
    rays = np.zeros((n, 8), np.float32)
    rays[:, 0:3] = rng.uniform(-4, 4, (n, 3))
    rays[:, 4:7] = rng.normal(size=(n, 3))
    rays[:, 3] = rng.uniform(0.0, 4.0, n)
    bad = rng.integers(0, n, 4000)
    rays[bad[:1500], rng.integers(4, 7, 1500)] = 0.0
    rays[bad[1500:2000], 4:7] = 0.0
    rays[bad[2000:3000], rng.integers(0, 7, 1000)] = np.nan
    rays[bad[3000:], rng.integers(0, 7, 1000)] = np.inf
    unbounded = rays.copy()  # closest-hit queries ignore tmax
    unbounded[:, 3] = 9999.0
    return scene, acc, rays, scene.closest(unbounded), scene.any(rays)


# One ray, partial and full waves, one ray a wave on the whole grid and just
# beyond, every lane used, chunks handed out dynamically.
@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 129, 2560, 5121, 40_000, 163_840, 163_841, 400_000])
def test_query_sizes_bit_exact(orc, env, queue_scene, n):
    torch, accel, W = env
    scene, acc, rays, ref, occ = queue_scene
    print(f"query of {n} rays", flush=True)
    got = _gpu_closest(torch, acc, rays[:n])
    _compare(scene, ref[:n], got, orc)
    miss = got[:, 0] == 0
    assert np.all(got[miss, 1:3] == 0xffffffff) and np.all(got[miss, 3].view(np.float32) == 9999.0)
    assert np.all(got[miss, 4:8] == 0)
    r = torch.from_numpy(rays[:n]).cuda()
    o = torch.full((n + 1,), 7, dtype=torch.int32, device="cuda")
    acc.trace_any(r, o)
    torch.cuda.synchronize()
    o = o.cpu().numpy()
    assert np.array_equal(o[:n].astype(np.uint32), occ[:n]) and o[n] == 7


def test_any_hit_threads_on_one_stream(orc, env, queue_scene):
    """Occlusion queries of two threads on the default stream, with more rays
    than the waves start with: every query answers all of its rays."""
    import threading
    torch, accel, W = env
    scene, acc, rays, ref, occ = queue_scene
    reps, bad = 60, []
    dev = [torch.from_numpy(np.tile(rays[k::2], (4, 1))).cuda() for k in range(2)]
    exp = [torch.from_numpy(np.tile(occ[k::2].astype(np.int32), 4)).cuda() for k in range(2)]
    outs = [torch.full((reps, d.shape[0]), 7, dtype=torch.int32, device="cuda") for d in dev]
    torch.cuda.synchronize()

    def ask(k):
        try:
            for i in range(reps):
                acc.trace_any(dev[k], outs[k][i])
        except Exception as e:
            bad.append(e)

    threads = [threading.Thread(target=ask, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not bad
    for k in range(2):
        assert bool((outs[k] == exp[k]).all())


# The waves' first chunks only, and a second chunk for some of them.
@pytest.mark.parametrize("n", [1, 6145, 393_217, 400_000])
def test_any_hit_recorded(orc, env, queue_scene, n):
    """An occlusion query recorded into a graph, replayed between eager work."""
    torch, accel, W = env
    scene, acc, rays, ref, occ = queue_scene
    r = torch.from_numpy(rays[:n]).cuda()
    o = torch.full((n + 1,), 7, dtype=torch.int32, device="cuda")
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        acc.trace_any(r, o, stream=s)  # the stream's scratch
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        acc.trace_any(r, o, stream=s)
    for _ in range(3):
        o.fill_(7)
        g.replay()
        acc.trace_any(r[:1], o[:1])
        torch.cuda.synchronize()
        got = o.cpu().numpy()
        assert np.array_equal(got[:n].astype(np.uint32), occ[:n]) and got[n] == 7


@pytest.fixture(scope="module")
def shallow_scene(orc, env):
    """A scene whose traversal stacks fit in LDS (spilled ones belong to a
    stream), rays and which of them are occluded."""
    torch, accel, W = env
    pos, idx = W.sphere_mesh(20, 10)
    scene = orc.assemble_scene([dict(positions=pos, indices=idx)],
                               dict(mesh=[0], transform=[W.identity_transform()], material=[0]))
    blas = accel.Blas(pos, idx)
    assert blas.info()["max_depth"] < 16
    acc = accel.Accel([blas], [0], [W.identity_transform()])
    rng = np.random.default_rng(5)
    rays = np.zeros((50_000, 8), np.float32)
    rays[:, 0:3], rays[:, 4:7] = rng.uniform(-1.5, 1.5, (50_000, 3)), rng.normal(size=(50_000, 3))
    rays[:, 3] = rng.uniform(0.0, 2.0, 50_000)
    return acc, rays, scene.any(rays).astype(np.int32)


def test_any_hit_on_per_thread_streams(env, shallow_scene):
    """Occlusion queries of two threads on hipStreamPerThread (handle 2)."""
    import threading
    import types
    torch, accel, W = env
    acc, rays, occ = shallow_scene
    reps, bad = 40, []
    dev = [torch.from_numpy(np.tile(rays[k::2], (40, 1))).cuda() for k in range(2)]
    exp = [torch.from_numpy(np.tile(occ[k::2], 40)).cuda() for k in range(2)]
    outs = [torch.full((reps, d.shape[0]), 7, dtype=torch.int32, device="cuda") for d in dev]
    acc.trace_any(dev[0], outs[0][0])
    torch.cuda.synchronize()

    def ask(k):
        try:
            for i in range(reps):
                acc.trace_any(dev[k], outs[k][i], stream=types.SimpleNamespace(cuda_stream=2))
            torch.cuda.synchronize()
        except Exception as e:
            bad.append(e)

    threads = [threading.Thread(target=ask, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not bad
    for k in range(2):
        assert bool((outs[k] == exp[k]).all())


def test_any_hit_graphs_side_by_side(env, shallow_scene):
    """Two occlusion queries recorded on one stream, replayed on two at once."""
    torch, accel, W = env
    acc, rays, occ = shallow_scene
    rec, streams, work = torch.cuda.Stream(), [torch.cuda.Stream(), torch.cuda.Stream()], []
    for k in range(2):
        r = torch.from_numpy(np.tile(rays[k::2], (40, 1))).cuda()
        e = torch.from_numpy(np.tile(occ[k::2], 40)).cuda()
        o = torch.full((r.shape[0],), 7, dtype=torch.int32, device="cuda")
        acc.trace_any(r, o, stream=rec)
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=rec):
            acc.trace_any(r, o, stream=rec)
        work.append((g, r, o, e))
    for _ in range(5):
        for g, r, o, e in work:
            o.fill_(7)
        torch.cuda.synchronize()
        for _ in range(4):
            for s, (g, r, o, e) in zip(streams, work):
                with torch.cuda.stream(s):
                    g.replay()
        torch.cuda.synchronize()
        for g, r, o, e in work:
            assert bool((o == e).all())


# One ray a wave on part of the grid, on all of it, eight a wave.
@pytest.mark.parametrize("n,mib", [(1000, 4), (4096, 8), (40_000, 40)])
def test_spill_memory_of_short_queries(env, queue_scene, n, mib):
    """A stream's first queries allocate stack memory for the rays they have
    (576 bytes a ray), not for every lane of the grid."""
    torch, accel, W = env
    scene, acc, rays, ref, occ = queue_scene
    r = torch.from_numpy(rays[:n]).cuda()
    h = torch.zeros((n, 8), dtype=torch.int32, device="cuda")
    o = torch.zeros((n,), dtype=torch.int32, device="cuda")
    acc.trace_closest(r, h)  # the kernels' code is loaded
    acc.trace_any(r, o)
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    acc.trace_closest(r, h, stream=s)
    acc.trace_any(r, o, stream=s)
    torch.cuda.synchronize()
    assert free - torch.cuda.mem_get_info()[0] <= mib << 20
    assert np.array_equal(o.cpu().numpy().astype(np.uint32), occ[:n])
