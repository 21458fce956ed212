"""The wide walk (trace_wide.hip, the default on triangle scenes, single frame octrees and brick sets)
and the multi-octree kernel (trace_multi.hip) against the binary walk, record for record: tile and batch edges, instances, first-hit and any-hit rays,
rays and scenes that fall back to the sequential walk, trees deeper than the LDS stack, the refitted
instance level, graph replay, several streams and the allocation-free entry point. Both scenes of a comparison
say which walk they take."""
import numpy as np
import pytest

import test_wide_cpu as cpu
from conftest import assert_sdf_parity, raw_equal, sdf_check

pytestmark = pytest.mark.gpu
MO_VOXEL_COUNT = 24   # MULTI_RENDER_MODE_MO_VOXEL_COUNT


@pytest.fixture(scope="module")
def torch_dev():
    import torch
    assert torch.cuda.is_available()
    torch.cuda.set_device(0)
    return torch


def trace(torch, g, s, pos, dirs, fn="trace_closest"):
    hits = torch.full((pos.shape[0], 8), -5, dtype=torch.int32, device="cuda")
    getattr(s, fn)(pos, dirs, hits)
    torch.cuda.synchronize()
    return hits.cpu().numpy().view(g.HIT_DTYPE).reshape(-1)


def flags(torch, s, pos, dirs):
    out = torch.full((pos.shape[0],), 7, dtype=torch.int32, device="cuda")
    s.trace_any(pos, dirs, out)
    torch.cuda.synchronize()
    return out.cpu().numpy()


LDS_STACK = 12   # WIDE_LDS_STACK (wide_walk.h): deeper trees spill


class Both:
    """The same scene twice: the wide form, also for batches that crowd into a small scene, and the binary walk.
    tree: the wide walk's, or none (multi-octrees and scenes without a wide form)."""

    def __init__(self, g, build, tree=True, wide=True):
        self.g = g
        self.wide, self.binary = build(), build()
        self.wide.set_walk(g.WALK_WIDE)
        self.binary.set_launch_config(256, 16, True)
        self.binary.set_tail_config(0, 1024)
        self.binary.set_leaf_postponement(0)   # the sequential walk, leaf by leaf
        self.walk = g.WALK_WIDE if wide else g.WALK_BINARY
        assert bool(self.wide.get_array("wide_blocks").size) == tree

    def levels(self):
        root = int(self.wide.get_array("wide_root").view(np.uint32)[0])
        return cpu.tree_levels(self.wide.get_array("wide_blocks").view(np.uint32).reshape(-1, 16), root)

    def check(self, torch, pos, dirs, fn="trace_closest", any_hit=True):
        n = pos.shape[0]
        assert self.wide.walk_of_call(n) == self.walk and self.binary.walk_of_call(n) == self.g.WALK_BINARY
        a, b = (trace(torch, self.g, s, pos, dirs, fn) for s in (self.wide, self.binary))
        assert raw_equal(a, b), int((a.view(np.uint8).reshape(-1, 32) != b.view(np.uint8).reshape(-1, 32)).any(1).sum())
        if any_hit:
            assert np.array_equal(flags(torch, self.wide, pos, dirs), flags(torch, self.binary, pos, dirs))
        return a


def mesh(g, n, mats=(None,), seed=1, build="cbvh_embree2"):
    def make():
        s = g.SceneRT(build_name=build)
        gid = s.AddGeom_Triangles3f(*g.gen_geodesic(n, 0.05, 4.0, seed))
        for m in mats:
            s.AddInstance(gid, m)
        s.CommitScene()
        return s
    return make


def random_rays(torch, n, seed, extent=1.5, far=100.0):
    rng = np.random.default_rng(seed)
    pos = np.concatenate([rng.uniform(-extent, extent, (n, 3)), np.full((n, 1), 1e-4)], 1).astype(np.float32)
    d = rng.normal(size=(n, 3))
    dirs = np.concatenate([d / np.linalg.norm(d, axis=1, keepdims=True), np.full((n, 1), far)], 1).astype(np.float32)
    return torch.from_numpy(pos).cuda(), torch.from_numpy(dirs).cuda()


def mats(n, seed, extent):
    rng = np.random.default_rng(seed)
    out = []
    for _ in range(n):
        m = np.eye(4, dtype=np.float32)
        q, r = np.linalg.qr(rng.normal(size=(3, 3)))
        m[:3, :3] = q * rng.uniform(0.5, 2.0)
        m[:3, 3] = rng.uniform(-extent, extent, 3)
        out.append(m)
    return out


@pytest.mark.parametrize("n_rays", [1, 63, 64, 65, 4097, 700001])
@pytest.mark.parametrize("n", [1, 7, 64])
def test_mesh(lrt, torch_dev, n, n_rays):
    b = Both(lrt, mesh(lrt, n))
    pos, dirs = random_rays(torch_dev, n_rays, n_rays)
    hits = b.check(torch_dev, pos, dirs)
    if n_rays > 60:
        assert 0 < (hits["primId"] != lrt.MISS).sum()


@pytest.mark.parametrize("build", ["cbvh_embree1", "cbvh_embree4", "gpu_lbvh2"])
def test_builders(lrt, torch_dev, build):
    Both(lrt, mesh(lrt, 20, build=build)).check(torch_dev, *random_rays(torch_dev, 50000, 3))


@pytest.mark.parametrize("n_inst", [2, 6, 7, 300])
def test_instances(lrt, torch_dev, n_inst):
    b = Both(lrt, mesh(lrt, 12, mats(n_inst, n_inst, 4.0)))
    b.check(torch_dev, *random_rays(torch_dev, 200003, 5, extent=5.0))


def test_first_hit_and_short_rays(lrt, torch_dev):
    b = Both(lrt, mesh(lrt, 12, mats(20, 4, 3.0)))
    pos, dirs = random_rays(torch_dev, 30000, 6, extent=4.0, far=0.7)
    dirs[::3, 3] *= -1   # stops at the sequential walk's first hit
    dirs[::7, 3] = 0.0
    b.check(torch_dev, pos, dirs)
    pos[:, 3] = 0.5   # near plane inside the scene
    b.check(torch_dev, pos, dirs)


def test_special_rays(lrt, torch_dev):
    b = Both(lrt, mesh(lrt, 9, mats(3, 4, 1.0) + [None]))
    pos, dirs = random_rays(torch_dev, 9000, 7)
    dirs[0::9, 0] = 0.0
    dirs[1::9, :2] = 0.0
    dirs[2::9, 1] = -0.0
    dirs[3::9, 2] = 1e-30
    pos[4::9, 0] = float("inf")
    pos[5::9, 1] = float("nan")
    dirs[6::9, 2] = float("nan")
    dirs[7::9, 3] = float("inf")
    pos[8::9, 3] = -1.0
    b.check(torch_dev, pos, dirs)


def test_ties(lrt, torch_dev):
    """Every surface twice, and coplanar tessellations: equal distances are the sequential walk's call."""
    v, f = lrt.gen_geodesic(8, 0.05, 4.0, 2)

    def make():
        s = lrt.SceneRT()
        gid = s.AddGeom_Triangles3f(np.concatenate([v, v]), np.concatenate([f, f + v.shape[0]]))
        s.AddInstance(gid)
        s.AddInstance(gid)
        x, y = np.meshgrid(np.arange(9, dtype=np.float32), np.arange(9, dtype=np.float32), indexing="ij")
        grid = np.stack([x.ravel() - 4, y.ravel() - 4, np.full(81, 0.25, np.float32)], 1)
        q = (np.arange(8)[:, None] * 9 + np.arange(8)).ravel()
        tri = np.concatenate([np.stack([q, q + 9, q + 1], 1), np.stack([q + 1, q + 9, q + 10], 1)]).astype(np.uint32)
        s.AddInstance(s.AddGeom_Triangles3f(grid, tri))
        s.CommitScene()
        return s

    b = Both(lrt, make)
    pos, dirs = random_rays(torch_dev, 40000, 8, extent=3.0)
    b.check(torch_dev, pos, dirs)
    # through the lattice's vertices and edges
    t = np.random.default_rng(1).integers(-4, 5, (5000, 2)).astype(np.float32)
    p = pos[:5000].clone()
    d = torch_dev.from_numpy(np.concatenate([t, np.full((5000, 1), 0.25, np.float32)], 1)).cuda() - p[:, :3]
    dirs[:5000, :3] = d / d.norm(dim=1, keepdim=True)
    b.check(torch_dev, p, dirs[:5000].contiguous())


def aimed_rays(torch, n, seed, at, octaves=30, far=100.0):
    """Rays from around `at` to places nearer and nearer to it."""
    rng = np.random.default_rng(seed)
    pos = np.concatenate([rng.uniform(-0.2, 0.2, (n, 3)) + at, np.full((n, 1), 1e-4)], 1).astype(np.float32)
    d = at + rng.normal(size=(n, 3)) * 0.5 ** rng.uniform(0, octaves, (n, 1)) - pos[:, :3]
    dirs = np.concatenate([d / np.linalg.norm(d, axis=1, keepdims=True), np.full((n, 1), far)], 1).astype(np.float32)
    return torch.from_numpy(pos).cuda(), torch.from_numpy(dirs).cuda()


@pytest.mark.parametrize("n,ratio,n_inst,levels", [(66, 0.5, 1, 11), (200, 0.7, 1, 28), (200, 0.7, 12, 30), (200, 0.7, 60, 39),
                                                   (200, 0.7, 100, None)])
def test_deep_tree(lrt, torch_dev, n, ratio, n_inst, levels):
    """Triangles whose sizes fall by a ratio each, alone and as instances whose sizes fall: a chain of nodes, up to
    three times as many levels as stack entries in LDS. Batches whose rays are handed over in parts and batches
    that fill the device; 100 instances have no tree (more than 40 levels)."""
    def make():
        s = lrt.SceneRT()
        gid = s.AddGeom_Triangles3f(*cpu.chain_mesh(n, ratio))
        for m in cpu.shrinking(n_inst):
            s.AddInstance(gid, m)
        s.CommitScene()
        return s

    b = Both(lrt, make, tree=levels is not None, wide=levels is not None)
    assert levels is None or b.levels() == levels
    for n_rays in (1, 100, 20000, 300001):
        pos, dirs = aimed_rays(torch_dev, n_rays, 9, np.zeros(3))
        if levels is None:   # (the two-pass scheme's hits are within some ulp here: triangles in front of their boxes)
            b.wide.set_tail_config(0, 1024)
        hits = b.check(torch_dev, pos, dirs)
        assert n_rays == 1 or (hits["primId"] != lrt.MISS).mean() > 0.05
        if n_rays <= 20000:
            assert raw_equal(trace(torch_dev, lrt, b.wide, pos, dirs, "trace_closest_noalloc"), hits)


@pytest.mark.parametrize("kind", ["frame", 1, 2, "indexed"])
def test_deep_sdf_trees(lrt, torch_dev, kind):
    """A frame octree and brick sets refined towards one point: more levels than stack entries in LDS, for traces
    and, with the indexed set, for the differentiable calls (whose small batches take whole waves of rays then)."""
    torch = torch_dev

    def make():
        s = lrt.SceneRT()
        s.AddInstance(s.AddGeom_SdfFrameOctree(cpu.corner_octree(15)) if kind == "frame" else
                      s.AddGeom_SdfSBS(*cpu.corner_bricks(15, kind)))
        s.CommitScene()
        return s

    b = Both(lrt, make)
    assert b.levels() > LDS_STACK
    point = np.full(3, 2 * 0.333 - 1.0)   # the bits of the path are 1 0 1 0 ...: a third or two thirds of the cube
    for at in (point, -point):
        for n in (1, 100, 20000, 150001):
            pos, dirs = aimed_rays(torch, n, 5, at)
            dirs[::7, 3] = 0.15
            hits = b.check(torch, pos, dirs)
            assert n < 100 or (hits["primId"] != lrt.MISS).any()
        if kind == "indexed":   # (fewer rays into the smallest bricks: short sums)
            for n in (1, 100, 4097):
                adjoint_agrees(torch, b, *aimed_rays(torch, n, 6, at, octaves=12))


@pytest.mark.parametrize("depth", [2, 5, 8])
def test_frame_octree(lrt, torch_dev, depth):
    rng = np.random.default_rng(2)
    sph = np.concatenate([rng.uniform(-0.8, 0.8, (24, 3)), rng.uniform(0.1, 0.3, (24, 1))], 1).astype(np.float32)
    nodes = lrt.sdf_spheres_frame_octree(sph, depth)

    for mode in (lrt.SDF_OCTREE_NODE_INTERSECT_ANALYTIC, lrt.SDF_OCTREE_NODE_INTERSECT_BBOX):
        for m in (None, mats(1, 3, 0.3)[0]):
            def make():
                s = lrt.SceneRT()
                s.AddInstance(s.AddGeom_SdfFrameOctree(nodes), m)
                p = lrt.default_preset()
                p["sdf_node_intersect"] = mode
                s.SetPreset(p)
                s.CommitScene()
                return s

            b = Both(lrt, make)
            pos, dirs = random_rays(torch_dev, 100003, 10, extent=2.0)
            dirs[::5, 3] *= -1
            dirs[::11, 0] = 0.0
            hits = b.check(torch_dev, pos, dirs)
            assert (hits["primId"] != lrt.MISS).sum() > 100


def test_instance_updates(lrt, torch_dev):
    start, moved, far_off = mats(40, 1, 4.0), mats(40, 2, 4.0), mats(40, 3, 60.0)
    b = Both(lrt, mesh(lrt, 10, start))
    pos, dirs = random_rays(torch_dev, 60000, 11, extent=5.0)
    b.check(torch_dev, pos, dirs)
    for step, kind in ((moved, 1), (far_off, 2), (start, None)):
        for s in (b.wide, b.binary):
            for i, m in enumerate(step):
                s.UpdateInstance(i, m)
            s.CommitScene()
        if kind is not None:
            assert b.wide.commit_info()["kind"] == kind
        b.check(torch_dev, pos, dirs)
    one = Both(lrt, mesh(lrt, 10, start[:1]))
    for s in (one.wide, one.binary):
        s.UpdateInstance(0, moved[0])
        s.CommitScene()
    one.check(torch_dev, pos, dirs)


@pytest.mark.parametrize("x,steps", [(9e29, ((1.2e30, 1), (9e29, 1), (1e31, 1))), (1.0, ((1e31, 2), (1.0, 1)))])
def test_boxes_that_cannot_be_packed(lrt, torch_dev, x, steps):
    """An instance far away moved past what a node's planes can hold (1e30) and back, by refits: the nodes above it
    let every ray through meanwhile, and the exact boxes of instances decide as before. Where the instance tree is
    built again with such a box, the scene goes without the wide walk."""
    start = mats(40, 1, 4.0)
    start[7][0, 3] = x
    b = Both(lrt, mesh(lrt, 10, start))
    pos, dirs = random_rays(torch_dev, 30000, 11, extent=5.0)
    b.check(torch_dev, pos, dirs)
    for x, kind in steps:
        m = start[7].copy()
        m[0, 3] = x
        for s in (b.wide, b.binary):
            s.UpdateInstance(7, m)
            s.CommitScene()
            assert s.commit_info()["kind"] == kind
        if kind == 2:
            b.walk = lrt.WALK_BINARY
        b.check(torch_dev, pos, dirs)


def test_streams(lrt, torch_dev):
    """One scene traced on several streams at once, with rays for the second pass: each stream has its own queue
    and counters."""
    torch = torch_dev
    bricks = Both(lrt, brick_scene(lrt, 4, 8, "indexed"))
    for b in (Both(lrt, mesh(lrt, 40, mats(9, 1, 2.0))), bricks):
        batches = []
        for k, n in enumerate((60000, 999, 200001, 64)):
            pos, dirs = random_rays(torch, n, 20 + k, extent=2.0)
            dirs[::17, 1] = 0.0
            batches.append((pos, dirs, b.check(torch, pos, dirs)))
        streams = [torch.cuda.Stream() for _ in batches]
        out = [torch.zeros((p.shape[0], 8), dtype=torch.int32, device="cuda") for p, _, _ in batches]
        torch.cuda.synchronize()
        for _ in range(5):
            for h in out:
                h.fill_(-1)
            torch.cuda.synchronize()
            for _ in range(4):
                for (pos, dirs, _), st, h in zip(batches, streams, out):
                    b.wide.trace_closest(pos, dirs, h, stream=st.cuda_stream)
            torch.cuda.synchronize()
            for (_, _, want), h in zip(batches, out):
                assert raw_equal(h.cpu().numpy().view(lrt.HIT_DTYPE).reshape(-1), want)
    # the differentiable calls, too
    params = torch.from_numpy(bricks.wide.get_array("sbs_data_f")).cuda()
    want = [torch.zeros((p.shape[0], 4), device="cuda") for p, _, _ in batches]
    got = [torch.full_like(c, -7.0) for c in want]
    for (pos, dirs, _), c in zip(batches, want):
        bricks.wide.sbs_forward(0, params, pos, dirs, c)
    torch.cuda.synchronize()
    for _ in range(4):
        for (pos, dirs, _), st, c in zip(batches, streams, got):
            bricks.wide.sbs_forward(0, params, pos, dirs, c, stream=st.cuda_stream)
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(want, got))


def test_graph_replay_and_noalloc(lrt, torch_dev):
    torch = torch_dev
    b = Both(lrt, mesh(lrt, 16, mats(9, 1, 2.0)))
    pos, dirs = random_rays(torch, 60000, 12, extent=3.0)
    dirs[::17, 1] = 0.0   # some rays take the second pass
    want = b.check(torch, pos, dirs)
    assert raw_equal(trace(torch, lrt, b.wide, pos, dirs, "trace_closest_noalloc"), want)
    hits = torch.zeros((pos.shape[0], 8), dtype=torch.int32, device="cuda")
    side, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        b.wide.trace_closest(pos, dirs, hits, stream=side.cuda_stream)
        torch.cuda.synchronize()
        with torch.cuda.graph(graph, stream=side):
            b.wide.trace_closest(pos, dirs, hits, stream=torch.cuda.current_stream().cuda_stream)
    for k in range(3):
        hits.fill_(-1)
        graph.replay()
        torch.cuda.synchronize()
        assert raw_equal(hits.cpu().numpy().view(lrt.HIT_DTYPE).reshape(-1), want)
        pos2, dirs2 = random_rays(torch, 1000 + k, k)
        b.check(torch, pos2, dirs2)


def brick_scene(g, depth, bs, kind, pad=0, m=None, seed=2):
    rng = np.random.default_rng(seed)
    sph = np.concatenate([rng.uniform(-0.8, 0.8, (64, 3)), rng.uniform(0.05, 0.2, (64, 1))], 1).astype(np.float32)

    def make():
        s = g.SceneRT()
        if kind == "indexed":
            h, nodes, vals, vf, _ = g.sdf_spheres_sbs_indexed(sph, depth, bs, 3)
            gid = s.AddGeom_SdfSBS(h, nodes, vals, vf)
        else:
            h = np.zeros((), g.SBS_HEADER_DTYPE)
            h["brick_size"], h["brick_pad"], h["bytes_per_value"] = bs, pad, kind
            h["aux_data"] = g.SDF_SBS_NODE_LAYOUT_DX_RGB8
            nodes, vals = g.sdf_spheres_sbs(sph, depth, h, 0, 5)
            gid = s.AddGeom_SdfSBS(h, nodes, vals)
        s.AddInstance(gid, m)
        s.CommitScene()
        return s
    return make


# depth 5 holds bricks of two sizes, whose binary tree has overlapping siblings
@pytest.mark.parametrize("depth,bs,kind", [(2, 1, 1), (3, 4, 2), (5, 2, 4), (5, 8, "indexed"), (4, 3, "indexed")])
def test_bricks(lrt, torch_dev, depth, bs, kind):
    for m in (None, mats(1, 3, 0.3)[0]):
        b = Both(lrt, brick_scene(lrt, depth, bs, kind, pad=1 if kind == 2 else 0, m=m))
        pos, dirs = random_rays(torch_dev, 150001, depth, extent=2.0)
        dirs[::11, 0] = 0.0
        dirs[::5, 3] = 0.6
        hits = b.check(torch_dev, pos, dirs)
        assert (hits["primId"] != lrt.MISS).sum() > 0


def adjoint_agrees(torch, b, pos, dirs):
    """Colour bit for bit, gradient and loss up to the order of the atomics (fp32 sums of up to 50,000 terms
    in another order: 1e-5 of the norm)."""
    n = pos.shape[0]
    params = torch.from_numpy(b.wide.get_array("sbs_data_f")).cuda()
    params += 0.002 * torch.randn(params.shape, device="cuda", generator=torch.Generator("cuda").manual_seed(1))
    target = torch.rand((n, 4), device="cuda", generator=torch.Generator("cuda").manual_seed(2))
    got = []
    for s in (b.wide, b.binary):
        c = [torch.full((n, 4), -7.0, device="cuda") for _ in range(2)]
        grads = [torch.zeros_like(params) for _ in range(3)]
        loss = [torch.zeros(1, device="cuda") for _ in range(2)]
        s.sbs_forward(0, params, pos, dirs, c[0])
        s.sbs_backward(0, params, pos, dirs, target, grads[0])
        s.sbs_l2_backward(0, params, pos, dirs, target, grads[1], loss[0])
        s.sbs_render_l2_backward(0, params, pos, dirs, target, c[1], grads[2], loss[1])
        torch.cuda.synchronize()
        assert s.sbs_recompute_misses() == 0
        got.append((c, grads, loss))
    for x, y in zip(got[0][0], got[1][0]):
        assert torch.equal(x, y)
    for x, y in zip(got[0][1] + got[0][2], got[1][1] + got[1][2]):
        assert float((x - y).norm()) <= 1e-5 * float(y.norm()) + 1e-12


@pytest.mark.parametrize("depth,n", [(3, 1), (3, 63), (4, 4097), (5, 50000)])
def test_adjoint(lrt, torch_dev, depth, n):
    b = Both(lrt, brick_scene(lrt, depth, 8, "indexed"))
    pos, dirs = random_rays(torch_dev, n, depth, extent=2.0)
    dirs[::13, 1] = 0.0
    adjoint_agrees(torch_dev, b, pos, dirs)


@pytest.mark.parametrize("other", [1, 2, "indexed"])
def test_adjoint_of_another_set(lrt, torch_dev, other):
    """Two brick sets, the first (of packed codes or indices) or the second one instanced, the second one
    differentiated: rays that hit the first have no colour, no gradient and a loss against 0."""
    torch, g = torch_dev, lrt
    rng = np.random.default_rng(2)
    sph = np.concatenate([rng.uniform(-0.8, 0.8, (64, 3)), rng.uniform(0.05, 0.2, (64, 1))], 1).astype(np.float32)

    def add(s, kind, depth):
        if kind == "indexed":
            return s.AddGeom_SdfSBS(*g.sdf_spheres_sbs_indexed(sph, depth, 8, 3)[:4])
        h = np.zeros((), g.SBS_HEADER_DTYPE)
        h["brick_size"], h["bytes_per_value"], h["aux_data"] = 4, kind, g.SDF_SBS_NODE_LAYOUT_DX
        return s.AddGeom_SdfSBS(h, *g.sdf_spheres_sbs(sph, depth, h))

    n = 5001
    pos, dirs = random_rays(torch, n, 4, extent=2.0)
    dirs[::13, 1] = 0.0   # some rays take the sequential walk
    target = torch.rand((n, 4), device="cuda", generator=torch.Generator("cuda").manual_seed(2))
    for instanced in (0, 1):
        def make():
            s = g.SceneRT()
            s.AddInstance((add(s, other, 3), add(s, "indexed", 4))[instanced])
            s.CommitScene()
            return s
        b = Both(g, make)
        assert (b.check(torch, pos, dirs)["primId"] != g.MISS).sum() > 300
        params = torch.from_numpy(b.wide.get_array("sbs_data_f")).cuda()
        got = []
        for s in (b.wide, b.binary):
            c = [torch.full((n, 4), -7.0, device="cuda") for _ in range(2)]
            grads = [torch.zeros_like(params) for _ in range(3)]
            loss = [torch.zeros(1, device="cuda") for _ in range(2)]
            s.sbs_forward(1, params, pos, dirs, c[0])
            s.sbs_backward(1, params, pos, dirs, target, grads[0])
            s.sbs_l2_backward(1, params, pos, dirs, target, grads[1], loss[0])
            s.sbs_render_l2_backward(1, params, pos, dirs, target, c[1], grads[2], loss[1])
            torch.cuda.synchronize()
            assert s.sbs_recompute_misses() == 0
            if instanced == 0:
                # the loss: an fp32 sum of n terms in any order, each step of which rounds by 2^-24
                want = float((target[:, :3].double() ** 2).sum())
                assert all(not x.any() for x in c + grads)
                assert all(abs(float(x) - want) <= n * 2.0 ** -24 * want for x in loss)
            got.append((c, grads + loss))
        for x, y in zip(got[0][0], got[1][0]):
            assert torch.equal(x, y)
        for x, y in zip(got[0][1], got[1][1]):
            assert float((x - y).norm()) <= 1e-5 * float(y.norm()) + 1e-12


@pytest.mark.parametrize("sizes", [((3, 1000), (5, 6400), (2, 1), (4, 0), (4, 65)),
                                   ((2, 300001), (15, 777), (3, 130000), (2, 64))])
def test_batch_forms_agree(lrt, torch_dev, sizes):
    """The batched run in the wide form (its default) against the binary one: ragged items, and a batch of several
    rounds of the waves with a set whose tree is deeper than the LDS stack (depth 15)."""
    torch = torch_dev
    items = []
    for k, (depth, n) in enumerate(sizes):
        if depth == 15:
            s = lrt.SceneRT()
            s.AddInstance(s.AddGeom_SdfSBS(*cpu.corner_bricks(15, "indexed")))
            s.CommitScene()
        else:
            s = brick_scene(lrt, depth, 8, "indexed", seed=k)()
        pos, dirs = random_rays(torch, max(n, 1), k, extent=2.0)
        pos, dirs = pos[:n].contiguous(), dirs[:n].contiguous()
        dirs[::9, 2] = 0.0
        params = torch.from_numpy(s.get_array("sbs_data_f")).cuda()
        items.append({"scene": s, "geom_id": 0, "params": params, "grad": torch.full_like(params, 9.0),
                      "loss": torch.full((1,), 9.0, device="cuda"), "pos": pos, "dir": dirs,
                      "target": torch.full((n, 4), 0.3, device="cuda"), "colour": torch.full((n, 4), -7.0, device="cuda")})
    runs = []
    for wide in (True, False):
        if not wide:
            for it in items:
                it["scene"].set_launch_config(256, 16, True)
        batch = lrt.SbsBatch(items)
        for _ in range(2):
            batch.run()
        torch.cuda.synchronize()
        runs.append([[it[k].clone() for k in ("colour", "grad", "loss")] for it in items])
    for a, b in zip(*runs):
        assert torch.equal(a[0], b[0])
        for x, y in zip(a[1:], b[1:]):   # fp32 sums in another order; the loss of 300,001 rays: as many steps of 2^-24
            assert float((x - y).norm()) <= max(1e-5, a[0].shape[0] * 2.0 ** -24) * float(y.norm()) + 1e-12
    batch.set_walk(lrt.WALK_WIDE)
    assert batch.get_walk() == lrt.WALK_BINARY   # the plan of scenes on the binary walk has no other
    for it in items:
        it["scene"].set_walk(lrt.WALK_AUTO)
    batch = lrt.SbsBatch(items)
    assert batch.get_walk() == lrt.WALK_WIDE
    r = batch.autotune()
    assert r["walk"] == batch.get_walk()
    batch.configure(r["lds_stack"], r["record"], r["grid"])
    assert batch.get_walk() == lrt.WALK_BINARY
    batch.set_walk(r["walk"])
    assert batch.get_walk() == r["walk"]


@pytest.mark.parametrize("n", [1, 65, 300001])
def test_batch_loss(lrt, torch_dev, n):
    """The batch's losses against float64 sums over the rendered colours. A term rounds by at most 5 steps of 2^-24
    (difference, square, two sums), a chunk's sum by 6, the result by one; the chunks are summed in 64 bits."""
    torch = torch_dev
    items = []
    for k, m in enumerate((n, 4097)):
        s = brick_scene(lrt, 3, 8, "indexed", seed=k)()
        pos, dirs = random_rays(torch, m, k, extent=2.0)
        params = torch.from_numpy(s.get_array("sbs_data_f")).cuda()
        items.append({"scene": s, "geom_id": 0, "params": params, "grad": torch.zeros_like(params),
                      "loss": torch.full((1,), 9.0, device="cuda"), "pos": pos, "dir": dirs,
                      "target": torch.rand((m, 4), device="cuda", generator=torch.Generator("cuda").manual_seed(k)),
                      "colour": torch.zeros((m, 4), device="cuda")})
    batch = lrt.SbsBatch(items)
    assert batch.get_walk() == lrt.WALK_WIDE
    for _ in range(3):
        batch.run()
        torch.cuda.synchronize()
        for it in items:
            want = float(((it["colour"][:, :3].double() - it["target"][:, :3].double()) ** 2).sum())
            assert abs(float(it["loss"]) - want) <= 12 * 2.0 ** -24 * want


@pytest.mark.parametrize("depth,count,lod,n", [(2, 1, 0.0, 1), (3, 2, 0.0, 63), (6, 1, 3.0, 70000), (7, 3, 0.0, 100001),
                                               (8, 1, 0.0, 400000)])
def test_multi_octrees(lrt, torch_dev, depth, count, lod, n):
    """Small and large batches, several instances, levels of detail, first-hit and any-hit rays, axis-parallel
    rays, the modes that put node properties into the record, graph replay."""
    torch, g = torch_dev, lrt
    rng = np.random.default_rng(4)
    sph = np.concatenate([rng.uniform(-0.7, 0.7, (48, 3)), rng.uniform(0.05, 0.25, (48, 1))], 1).astype(np.float32)
    nodes, values = g.sdf_spheres_multi_octree(sph, depth)

    def make():
        s = g.SceneRT()
        for _ in range(min(count, 2)):
            gid = s.AddGeom_SdfMultiOctree(nodes, values)
        for k, m in enumerate(mats(count, 3, 0.4)):
            s.AddInstance(k % (gid + 1), m if count > 1 else None)
        s.CommitScene()
        return s
    b = Both(g, make, tree=False)
    pos, dirs = random_rays(torch, n, depth, extent=2.0)
    dirs[::11, 0] = 0.0
    dirs[::5, 3] = 0.6
    dirs[::7, 3] *= -1.0
    for mode in (g.MULTI_RENDER_MODE_LAMBERT_NO_TEX, MO_VOXEL_COUNT):
        preset = g.default_preset()
        preset["render_mode"] = mode
        if lod:
            preset["fixed_lod"], preset["level_of_detail"] = 1, lod
        for s in (b.wide, b.binary):
            s.SetPreset(preset)
        hits = b.check(torch, pos, dirs)
        assert n < 63 or (hits["geomId"] != g.MISS).sum() > 0
    if n <= 65536:
        assert raw_equal(trace(torch, g, b.wide, pos, dirs, "trace_closest_noalloc"), hits)
    out = torch.zeros((n, 8), dtype=torch.int32, device="cuda")
    side, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        b.wide.trace_closest(pos, dirs, out, stream=side.cuda_stream)
        torch.cuda.synchronize()
        with torch.cuda.graph(graph, stream=side):
            b.wide.trace_closest(pos, dirs, out, stream=torch.cuda.current_stream().cuda_stream)
    for _ in range(3):
        out.fill_(-1)
        graph.replay()
        torch.cuda.synchronize()
        assert raw_equal(out.cpu().numpy().view(g.HIT_DTYPE).reshape(-1), hits)


# the lines of Scene::rays_crowd: 65,536 rays, 128 a triangle up to 7,168 triangles, 8,192 a brick up to 256 bricks
@pytest.mark.parametrize("kind,size,line", [("mesh", 1, 65536), ("mesh", 6, 92160), ("mesh", 18, 829440), ("mesh", 19, None),
                                            ("bricks", 2, 524288), ("bricks", 3, None)])
def test_crowded_batches(lrt, torch_dev, kind, size, line):
    """Both sides of the line where default calls leave the wide walk, and batches beyond it with the walk set."""
    b = Both(lrt, mesh(lrt, size) if kind == "mesh" else brick_scene(lrt, size, 1, 1))
    for n in (line - 1, line) if line else (1000003,):
        pos, dirs = random_rays(torch_dev, n, 1)
        for b.walk, setting in ((lrt.WALK_BINARY if n == line else lrt.WALK_WIDE, lrt.WALK_AUTO),
                                (lrt.WALK_WIDE, lrt.WALK_WIDE)):
            b.wide.set_walk(setting)
            b.check(torch_dev, pos, dirs)


@pytest.mark.parametrize("kind", ["crowded mesh", "instances", "multi", "mixed"])
def test_tuned_walk_is_kept(lrt, torch_dev, kind):
    """The tuner times the walk it names and a scene of the same make takes its result over: shape, then walk."""
    torch = torch_dev

    def make():
        s = lrt.SceneRT()
        if kind in ("multi", "mixed"):
            s.AddInstance(s.AddGeom_SdfMultiOctree(*lrt.sdf_spheres_multi_octree(
                np.array([[0.2, 0.1, -0.3, 0.4], [-0.3, 0.1, 0.3, 0.3]], np.float32), 4)))
        if kind != "multi":
            gid = s.AddGeom_Triangles3f(*lrt.gen_geodesic(2, 0.05, 4.0, 2))
            for m in mats(9 if kind == "instances" else 1, 4, 2.0):
                s.AddInstance(gid, m)
        s.CommitScene()
        return s
    n = 70001
    pos, dirs = random_rays(torch, n, 2, extent=2.5)
    s, other = make(), make()
    assert (s.walk_of_call(n) == lrt.WALK_WIDE) == (kind in ("instances", "multi"))
    want = trace(torch, lrt, s, pos, dirs)
    hits = torch.zeros((n, 8), dtype=torch.int32, device="cuda")
    r = s.autotune(pos, dirs, hits)
    assert r["walk"] == s.get_walk() == s.walk_of_call(n) != lrt.WALK_AUTO
    assert kind != "mixed" or r["walk"] == lrt.WALK_BINARY
    other.set_launch_config(r["block"], r["lds_stack"], bool(r["xcd_remap"]))
    other.set_tail_config(r["budget"], r["tail_waves"])
    other.set_ray_interleave(r["ray_interleave"])
    other.set_persistent(bool(r["persistent"]))
    other.set_walk(r["walk"])
    assert other.walk_of_call(n) == r["walk"]
    for x in (s, other):
        assert raw_equal(trace(torch, lrt, x, pos, dirs), want)


@pytest.mark.parametrize("first", [False, True])
@pytest.mark.parametrize("voxels", [0, 1])
def test_multi_octree_of_one_node(lrt, orc, torch_dev, first, voxels):
    """A root without children is a leaf (or empty), as the only octree and behind another one, in the default
    and the one-ray-a-lane kernels and beside a mesh."""
    node = np.zeros(1, lrt.MULTI_NODE_DTYPE)
    node["voxel_count"] = voxels
    values = np.array([((i >> 2) + (i >> 1 & 1) + (i & 1) - 1.4) * 0.5 for i in range(8)], np.float32)
    more = lrt.sdf_spheres_multi_octree(np.array([[0.2, 0.1, -0.3, 0.4]], np.float32), 3)
    for beside in (False, True):
        def make():
            s = lrt.SceneRT()
            if first:
                s.AddInstance(s.AddGeom_SdfMultiOctree(*more), mats(1, 3, 1.0)[0])
            s.AddInstance(s.AddGeom_SdfMultiOctree(node, values))
            if beside:
                s.AddInstance(s.AddGeom_Triangles3f(*lrt.gen_geodesic(3, 0.05, 4.0, 2)), mats(1, 5, 2.0)[0])
            s.CommitScene()
            return s
        b = Both(lrt, make, tree=False, wide=not beside)
        pos, dirs = random_rays(torch_dev, 20001, 3, extent=2.5)
        dirs[::11, 0] = 0.0
        got = b.check(torch_dev, pos, dirs)
        p, d = pos.cpu().numpy(), dirs.cpu().numpy()
        want, _ = orc.trace_closest(orc.Scene.from_scene(b.wide), p, d)
        r = sdf_check(got, want, p, d)
        assert_sdf_parity(r, got, want)
        assert bool(((got["geomId"] & lrt.GEOM_ID_MASK) == int(first)).any()) == bool(voxels)


@pytest.mark.parametrize("n", [1, 4096, 4097])
def test_host_staging(lrt, torch_dev, n):
    """Host calls staged in pinned memory (up to 4,096 rays) and by copies give the device call's records."""
    s = mesh(lrt, 12)()
    pos, dirs = random_rays(torch_dev, n, 3)
    want = trace(torch_dev, lrt, s, pos, dirs)
    for _ in range(2):
        assert raw_equal(s.trace_closest_host(pos.cpu().numpy(), dirs.cpu().numpy()), want)


def test_host_staging_across_scenes_and_threads(lrt, torch_dev):
    """Scenes that come and go share the staging memory of host calls, one block a call: threads on scenes of
    their own, on one scene, and calls after most scenes are gone give the device call's records."""
    import threading
    pos, dirs = random_rays(torch_dev, 300, 3)
    p, d = pos.cpu().numpy(), dirs.cpu().numpy()
    scenes = [mesh(lrt, 3 + k)() for k in range(6)]
    want = [trace(torch_dev, lrt, s, pos, dirs) for s in scenes]
    bad = []

    def work(k, own):
        for r in range(20):
            s = mesh(lrt, 3 + k)() if own else scenes[k]
            if not raw_equal(s.trace_closest_host(p, d), want[k]):
                bad.append((k, own, r))
    threads = [threading.Thread(target=work, args=(k % 6, k % 4 == 3)) for k in range(12)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
    del scenes[1:]
    assert raw_equal(scenes[0].trace_closest_host(p, d), want[0])
    scenes.clear()   # the last scene gives the memory back
    assert raw_equal(mesh(lrt, 4)().trace_closest_host(p, d), want[1])
