"""The engine-exact walk (csrc/walk.h) decides boxes from float products with a margin and settles near ties in
further stages; its hits must stay the oracle's bit for bit where those ties are common: flat boxes, planes shared by
both children, rays along axes and through edges, distances equal to the current hit, tmin in and on boxes, directions
outside the margin's premises, stacks deeper than the LDS rows; and over the launch shapes' edges (rays per wave,
chunks of 64, coherent or incoherent batches)."""
import numpy as np
import pytest

import atlas_rt
import oracle_rt
import rt_cases
from atlas_rt import _abi
from atlas_rt import workloads as W

pytestmark = pytest.mark.gpu


def boxes_mesh(g, n=700):
    """Axis-aligned boxes on a coarse lattice: flat triangles' boxes, many shared and coincident planes."""
    lo = g.integers(-10, 10, (n, 3)).astype(np.float64) * 0.5
    hi = lo + g.integers(1, 4, (n, 3)) * 0.5
    tris = []
    for a, b in zip(lo, hi):
        p = [np.array([(a, b)[i & 1][0], (a, b)[(i >> 1) & 1][1], (a, b)[i >> 2][2]]) for i in range(8)]
        for q in ((0, 1, 3, 2), (4, 5, 7, 6), (0, 1, 5, 4), (2, 3, 7, 6), (0, 2, 6, 4), (1, 3, 7, 5)):
            tris.append(np.concatenate([p[q[0]], p[q[1]], p[q[2]]]))
            tris.append(np.concatenate([p[q[0]], p[q[2]], p[q[3]]]))
    return np.asarray(tris, np.float32)


def strip_mesh(n=3000):
    """Triangles of growing size along x: a tree as deep as the builder makes it."""
    x = np.cumsum(1.02 ** np.arange(n) * 1e-3)
    t = np.zeros((n, 9))
    t[:, 0], t[:, 3], t[:, 6] = x, x * 1.01, x
    t[:, 4], t[:, 8] = x * 0.02, x * 0.02
    return t.astype(np.float32)


def meshes(g):
    return {"soup": W.triangle_soup(3000, g), "boxes": boxes_mesh(g), "height": W.heightfield(64), "strip": strip_mesh(),
            "one": W.triangle_soup(1, g), "two": W.triangle_soup(2, g)}


def hard_rays(g, verts, n):
    """Rays at the decisions' edges, an eighth of each kind."""
    rays = W.random_rays(n, g)
    v = verts.reshape(-1, 3).astype(np.float64)
    lo, hi = v.min(axis=0), v.max(axis=0)
    size = np.maximum(hi - lo, 1e-3)
    o = lo - 0.2 * size + g.uniform(0, 1.4, (n, 3)) * size
    target = v[g.integers(0, len(v), n)]
    d = target - o
    kind = np.arange(n) % 8
    o[kind == 1] = target[kind == 1]                                     # from a vertex
    d[kind == 1] = g.standard_normal((np.count_nonzero(kind == 1), 3))
    axis = g.integers(0, 3, n)
    along = np.eye(3)[axis] * g.choice([-1.0, 1.0], n)[:, None]
    k = kind == 2                                                         # along an axis, towards a vertex's line
    d[k] = along[k]
    o[k] = target[k] - along[k] * size.max() * g.uniform(0, 2, k.sum())[:, None]
    k = kind == 3                                                         # in a lattice plane: a zero component
    d[k] = d[k] * (1 - np.abs(along[k]))
    o[k] = np.round(o[k] * 2) / 2
    k = kind == 4                                                         # steep: subnormal and tiny components
    d[k] = d[k] * np.where(np.abs(along[k]) > 0, g.choice([1e-45, 1e-39, 1e-30, 1e-8], k.sum())[:, None], 1.0)
    k = kind == 5                                                         # long and short directions
    d[k] = d[k] * g.choice([1e-30, 1e-10, 1e10, 1e38], k.sum())[:, None]
    rays["origin"] = o.astype(np.float32)
    with np.errstate(over="ignore"):
        rays["direction"] = d.astype(np.float32)
    rays["tmin"] = g.choice(np.array([0.0, 1e-4, 1.0, -1.0], np.float32), n)
    rays["tmax"] = g.choice(np.array([1e12, np.inf, 2.0, 0.0], np.float32), n)
    k = kind == 6                                                         # tmax, then tmin, on the vertex itself
    rays["direction"][k] = (target[k] - o[k]).astype(np.float32)
    rays["tmax"][k] = 1.0
    k = kind == 7
    rays["tmin"][k] = 1.0
    return rays


def trace(torch, blas, rays, kernel):
    d = torch.from_numpy(rays.view(np.float32).reshape(-1, 8).copy()).cuda()
    h = torch.full((len(rays), 4), -7.0, device="cuda")
    s = torch.full((len(rays),), -7, dtype=torch.int32, device="cuda")
    blas.trace_closest(d, h, s, kernel=kernel)
    a = torch.full((len(rays),), -7, dtype=torch.int32, device="cuda")
    blas.trace_any(d, a)
    torch.cuda.synchronize()
    return h.cpu().numpy().view(atlas_rt.HIT_DTYPE).reshape(-1), s.cpu().numpy(), a.cpu().numpy().astype(np.uint32)


@pytest.mark.parametrize("name", ["soup", "boxes", "height", "strip", "one", "two"])
def test_hard_rays_bit_exact(torch_cuda, name):
    g = W.rng(5, 1)
    verts = meshes(g)[name]
    blas = atlas_rt.Blas.build(verts)
    nodes, tris, orig = blas.export()
    rays = hard_rays(g, verts, 70001)
    ref, slots = oracle_rt.trace_closest(nodes, tris, orig, rays)
    any_ref = oracle_rt.trace_any(nodes, tris, rays)
    for kernel in (0, 1, 2, 2 | _abi.KERNEL_LEAF_BATCH):
        h, s, a = trace(torch_cuda, blas, rays, kernel)
        bad = np.nonzero(np.any(rt_cases.hit_bits(h) != rt_cases.hit_bits(ref), axis=1) | (s != slots))[0]
        assert len(bad) == 0, f"{name} kernel {kernel}: {len(bad)} rays, first {bad[:4]} {rays[bad[:2]]} {h[bad[:2]]} {ref[bad[:2]]}"
    bad = np.nonzero(a != any_ref)[0]
    assert len(bad) == 0, f"{name} any: {len(bad)} rays, first {bad[:4]} {rays[bad[:2]]}"


def test_hard_rays_batched_bit_exact(torch_cuda):
    torch = torch_cuda
    g = W.rng(5, 4)
    M = list(meshes(g).values())
    blases = [atlas_rt.Blas.build(v) for v in M]
    n = 20011
    rays = np.concatenate([hard_rays(g, v, n) for v in M])
    rays["direction"][::97] = np.nan
    bs = atlas_rt.BatchSet(blases, [(k, k * n, n, 0) for k in range(len(M))])
    ref = np.zeros(len(rays), atlas_rt.HIT_DTYPE)
    for k, b in enumerate(blases):
        ref[k * n:(k + 1) * n] = oracle_rt.trace_closest(*b.export(), rays[k * n:(k + 1) * n])[0]
    d = torch.from_numpy(rays.view(np.float32).reshape(-1, 8).copy()).cuda()
    for kernel in (1, 2, 2 | _abi.KERNEL_LEAF_BATCH):
        for block in (64, 128, 256):
            print("case hard rays batched", kernel, block, flush=True)
            h = torch.full((len(rays), 4), -7.0, device="cuda")
            bs.trace_closest(d, h, kernel=kernel, block=block, refill=32)
            h = h.cpu().numpy().view(atlas_rt.HIT_DTYPE).reshape(-1)
            bad = np.nonzero(np.any(rt_cases.hit_bits(h) != rt_cases.hit_bits(ref), axis=1))[0]
            assert len(bad) == 0, f"{kernel} {block}: {len(bad)} rays, first {bad[:4]} {rays[bad[:2]]} {h[bad[:2]]} {ref[bad[:2]]}"


def transforms(g, size):
    """Instance matrices: as they are, turned by a quarter (components that become exactly 0), any rotation, mirrored
    and scaled unevenly, flat, tiny (object-space directions of 1e30) and as large as finite boxes of a mesh of this
    size allow (directions of 1e-35 and less, subnormal components among them)."""
    quarter = np.array([[0, 0, 1.0], [0, 1, 0], [-1, 0, 0]])
    c, s = np.cos(0.7), np.sin(0.7)
    turn = np.array([[c, -s, 0], [s, c, 0], [0, 0, 1.0]])
    linear = [np.eye(3), quarter, turn, np.diag([-1.0, 2.0, 0.25]), turn @ np.diag([1.0, 1e-3, 1.0]), np.eye(3) * 1e-30,
              quarter * (1e36 / size), np.eye(3), turn @ quarter]
    m = np.zeros((len(linear), 3, 4))
    for k, a in enumerate(linear):
        m[k, :, :3] = a
        m[k, :, 3] = np.round(g.uniform(-6, 6, 3) * 2) / 2 if k else 0.0
    return m


@pytest.mark.parametrize("name", ["soup", "boxes", "height", "strip", "one", "chain"])
def test_hard_rays_through_worlds_bit_exact(torch_cuda, name):
    """Overlapping instances, so that walks leave instances with TLAS entries on the stack; some masked from one of
    the two masks.  The chain's walks hold 80 entries above the TLAS's."""
    torch = torch_cuda
    g = W.rng(5, 5)
    if name == "chain":
        nodes, tris, _ = rt_cases.chain_tree(80)
        first = atlas_rt.Blas.create(nodes, tris)
        verts = np.concatenate([tris["v0"][:, :3], tris["v1"][:, :3], tris["v2"][:, :3]], axis=1)
    else:
        verts = meshes(g)[name]
        first = atlas_rt.Blas.build(verts)
    second = atlas_rt.Blas.build(boxes_mesh(g, 40))
    xf = transforms(g, np.abs(verts).max())
    xf = np.concatenate([xf, xf[:4]])
    xf[-4:, :, 3] += 0.5
    descs = atlas_rt.instance_descs(xf, [0] * 9 + [1] * 4)
    descs["mask"][[2, 7, 10]] = _abi.MASK_ALL
    descs["mask"][[3, 11]] = _abi.MASK_SHADOW
    w = atlas_rt.World()
    w.update(descs, [first, second])
    tl, inst, order = w.export()
    bl = [first.export(), second.export()]
    rays = hard_rays(g, verts, 30011)
    if name == "chain":
        rays[::2] = np.resize(rt_cases.chain_tree(80)[2], len(rays[::2]))
    rays["direction"][::97] = np.nan
    d = torch.from_numpy(rays.view(np.float32).reshape(-1, 8).copy()).cuda()
    for mask in (_abi.MASK_ALL, _abi.MASK_SHADOW):
        print("case hard rays world", name, mask, flush=True)
        h = torch.full((len(rays), 4), -7.0, device="cuda")
        gi = torch.full((len(rays),), -7, dtype=torch.int32, device="cuda")
        w.trace_closest_rays(d, h, gi, mask=mask)
        h = h.cpu().numpy().view(atlas_rt.HIT_DTYPE).reshape(-1)
        ref, _, ri = oracle_rt.trace_world(tl, inst, bl, rays, mask=mask)
        ri = np.where(ri >= 0, order[np.maximum(ri, 0)].astype(np.int32), -1)
        bad = np.nonzero(np.any(rt_cases.hit_bits(h) != rt_cases.hit_bits(ref), axis=1) | (gi.cpu().numpy() != ri))[0]
        assert len(bad) == 0, f"{len(bad)} rays, first {bad[:4]} {rays[bad[:2]]} {h[bad[:2]]} {ref[bad[:2]]}"
        assert (ri >= 0).sum() > 1000
        for flags, mode in ((_abi.ANY_ENGINE_HITANY, oracle_rt.WORLD_ANY),
                            (_abi.ANY_RESTORE_ALWAYS, oracle_rt.WORLD_ANY_RESTORE)):
            a = torch.full((len(rays),), -7, dtype=torch.int32, device="cuda")
            w.trace_any_rays(d, a, mask=mask, flags=flags)
            ar, _, _ = oracle_rt.trace_world(tl, inst, bl, rays, mask=mask, mode=mode)
            bad = np.nonzero(a.cpu().numpy() != ar["prim_id"])[0]
            assert len(bad) == 0, f"any {flags}: {len(bad)} rays, first {bad[:4]} {rays[bad[:2]]}"


@pytest.mark.parametrize("count", [1, 2, 63, 64, 65, 2048, 2049, 5003, 65535, 65536, 65537, 131073])
@pytest.mark.parametrize("coherent", [False, True])
def test_launch_shapes_bit_exact(torch_cuda, count, coherent):
    g = W.rng(5, 2)
    verts = W.heightfield(64)
    blas = atlas_rt.Blas.build(verts)
    nodes, tris, orig = blas.export()
    if coherent:
        rays = W.pinhole_rays(512, 257, (31.0, 60.0, -9.0), 0.0, 30.0)[:count]
    else:
        rays = W.random_rays(count, g, extent=40.0)
    rays["direction"][::97] = np.nan
    ref, slots = oracle_rt.trace_closest(nodes, tris, orig, rays)
    h, s, a = trace(torch_cuda, blas, rays, 0)
    assert np.array_equal(rt_cases.hit_bits(h), rt_cases.hit_bits(ref)) and np.array_equal(s, slots)
    assert np.array_equal(a, oracle_rt.trace_any(nodes, tris, rays))


@pytest.mark.parametrize("more", [-1, 0, 4097])
@pytest.mark.parametrize("coherent", [False, True])
def test_any_hit_shapes_bit_exact(torch_cuda, more, coherent):
    """Any-hit rays are refilled, if incoherent, from 2^33 / nodes of them on."""
    print("case any-hit shapes", more, coherent, flush=True)
    torch = torch_cuda
    blas = atlas_rt.Blas.build(W.heightfield(129))
    nodes, tris, orig = blas.export()
    count = -(-2**33 // min(len(nodes), 16384)) + more
    if coherent:
        rays = W.pinhole_rays(1024, 517, (64.0, 60.0, -19.0), 0.0, 30.0)[:count]
    else:
        rays = W.random_rays(count, W.rng(5, 6), extent=80.0)
    assert len(rays) == count
    d = torch.from_numpy(rays.view(np.float32).reshape(-1, 8).copy()).cuda()
    a = torch.full((count,), -7, dtype=torch.int32, device="cuda")
    blas.trace_any(d, a)
    ref = oracle_rt.trace_any(nodes, tris, rays)
    assert ref.mean() > 0.05 and np.array_equal(a.cpu().numpy().astype(np.uint32), ref)


def chain_rays(depth, n):
    """A tree whose walks hold `depth` stack entries, and n rays that need them all (their tmax ends some early)."""
    nodes, tris, rays = rt_cases.chain_tree(depth)
    rays = np.tile(rays, -(-n // len(rays)))[:n]
    rays["tmax"][1::3] = np.random.default_rng(depth).uniform(90.0, 110.0 + depth, len(rays[1::3])).astype(np.float32)
    return nodes, tris, rays


# the walk's stack rows: 14 in LDS (20 or 30 with a wave per ray set and in worlds), 32 of the lane's own, then spill rows
@pytest.mark.parametrize("depth", [12, 13, 14, 15, 18, 19, 20, 28, 29, 30, 31, 44, 45, 46, 47, 50, 51, 52, 60, 61, 62, 63, 80])
def test_stack_rows_bit_exact(torch_cuda, depth):
    print("case stack rows", depth, flush=True)
    torch = torch_cuda
    nodes, tris, rays = chain_rays(depth, 65536)
    blas = atlas_rt.Blas.create(nodes, tris)
    nodes, tris, orig = blas.export()
    ref, slots = oracle_rt.trace_closest(nodes, tris, orig, rays)
    any_ref = oracle_rt.trace_any(nodes, tris, rays)
    assert (slots >= 0).mean() > 0.5
    for n, kernel in ((65536, 0), (1024, 0), (1024, 1), (65536, 2), (1024, 2 | _abi.KERNEL_LEAF_BATCH)):
        h, s, a = trace(torch, blas, rays[:n], kernel)
        assert np.array_equal(rt_cases.hit_bits(h), rt_cases.hit_bits(ref[:n])) and np.array_equal(s, slots[:n]), kernel
        assert np.array_equal(a, any_ref[:n]), kernel
    d = torch.from_numpy(rays.view(np.float32).reshape(-1, 8).copy()).cuda()
    bs = atlas_rt.BatchSet([blas], [(0, 0, len(rays), 0)])
    for kernel in (1, 2, 2 | _abi.KERNEL_LEAF_BATCH):
        for block in (64, 256):
            hits = torch.full((len(rays), 4), -7.0, device="cuda")
            bs.trace_closest(d, hits, kernel=kernel, block=block, refill=32)
            h = hits.cpu().numpy().view(atlas_rt.HIT_DTYPE).reshape(-1)
            assert np.array_equal(rt_cases.hit_bits(h), rt_cases.hit_bits(ref)), (kernel, block)
    xf = np.zeros((1, 3, 4))
    xf[0, :, :3] = np.eye(3)
    w = atlas_rt.World()
    w.update(atlas_rt.instance_descs(xf, np.zeros(1, np.int64)), [blas])
    hits = torch.full((len(rays), 4), -7.0, device="cuda")
    w.trace_closest_rays(d, hits)
    h = hits.cpu().numpy().view(atlas_rt.HIT_DTYPE).reshape(-1)
    assert np.array_equal(rt_cases.hit_bits(h), rt_cases.hit_bits(ref))


@pytest.mark.parametrize("limit", [1, 2, 12, 13, 14, 18, 19, 20, 21, 28, 29, 30, 31, 44, 45, 46, 47, 50, 51, 52])
def test_stack_limits_at_the_rows_edges(torch_cuda, limit):
    """A walk of a chain of d levels holds d entries: a limit of d is enough for it and one of d - 1 stops every ray,
    on each side of the rows' edges, in every shape."""
    print("case stack limit", limit, flush=True)
    torch = torch_cuda
    for depth in (limit, limit + 1):
        nodes, tris, rays = rt_cases.chain_tree(depth)
        rays = np.tile(rays, 64)
        blas = atlas_rt.Blas.create(nodes, tris)
        blas.set_stack_limit(limit)
        for n, kernel in ((len(rays), 0), (1024, 0), (1024, 1), (1024, 2), (1024, 2 | _abi.KERNEL_LEAF_BATCH)):
            h, s, a = trace(torch, blas, rays[:n], kernel)
            assert blas.trace_status() == (_abi.OK if depth == limit else _abi.E_STACK_OVERFLOW), (depth, kernel)
            if depth == limit:
                assert np.all(h["prim_id"] >= 0) and np.all(s >= 0) and np.all(a == 1), (depth, kernel)
            else:
                assert np.all(h["prim_id"] == -1) and np.all(s == -1) and np.all(a == 0), (depth, kernel)
                assert np.array_equal(h["t"], rays["tmax"][:n])


def test_traces_allocate_nothing(torch_cuda):
    """Once a handle has been traced at all, traces of more rays take no more device memory, so they can be
    captured; the trees are 19 and more levels deep."""
    print("case traces without allocation", flush=True)
    torch = torch_cuda
    g = W.rng(5, 3)
    verts = W.triangle_soup(65536, g)
    rays = W.random_rays(1 << 20, g)
    d = torch.from_numpy(rays.view(np.float32).reshape(-1, 8).copy()).cuda()
    hits = torch.empty((len(rays), 4), device="cuda")
    occluded = torch.empty(len(rays), dtype=torch.int32, device="cuda")
    xf = np.zeros((1, 3, 4))
    xf[0, :, :3] = np.eye(3)

    def handles():
        blas = atlas_rt.Blas.build(verts)
        assert blas.info()[2] >= 19
        w = atlas_rt.World()
        w.update(atlas_rt.instance_descs(xf, np.zeros(1, np.int64)), [blas])
        few = atlas_rt.BatchSet([blas], [(0, 0, 100, 0)])
        return blas, w, few, atlas_rt.BatchSet([blas], [(0, 0, len(rays), 0)])

    def traces(blas, w, sets, n):
        blas.trace_closest(d[:n], hits[:n])
        blas.trace_any(d[:n], occluded[:n])
        blas.trace_closest(d[:n], hits[:n], kernel=1)
        w.trace_closest_rays(d[:n], hits[:n])
        w.trace_any_rays(d[:n], occluded[:n])
        sets.trace_closest(d, hits, kernel=1, block=64)
        sets.trace_closest(d, hits, kernel=2, block=64)

    warm = handles()  # the runtime's own memory for these kernels
    traces(*warm[:2], warm[3], len(rays))
    blas, w, few, sets = handles()
    traces(blas, w, few, 100)
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    traces(blas, w, sets, len(rays))
    torch.cuda.synchronize()
    assert before - torch.cuda.mem_get_info()[0] < 4 << 20  # of 29 MB that one trace's spill rows would take
    nodes, tris, orig = blas.export()
    n = 100000
    ref, _ = oracle_rt.trace_closest(nodes, tris, orig, rays[:n])
    # a small trace, then larger ones captured and replayed beside eager work
    blas2, w2, few2, sets2 = handles()
    traces(blas2, w2, few2, 100)
    sets2.trace_closest(d, hits, kernel=2, block=64)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        blas2.trace_closest(d, hits)
    for rep in range(3):
        hits.fill_(-3.0)
        graph.replay()
        torch.cuda.synchronize()
        h = hits[:n].cpu().numpy().view(atlas_rt.HIT_DTYPE).reshape(-1)
        assert np.array_equal(rt_cases.hit_bits(h), rt_cases.hit_bits(ref)), rep
        blas2.trace_closest(d, hits, kernel=1)
        blas2.trace_any(d, occluded)
