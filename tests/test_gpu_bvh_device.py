"""rt_bvh_build_device (the BVH built on the GPU from device arrays, the
arrangement of the reference's BVH constructor, cuda_libraries/BVH.cu:
314-341) against the oracle's restatement of the same build
(oracle/lbvh.c): the exported two-wide nodes, triangles and four-wide nodes
are bitwise equal and the reported figures match; traces on the device-built
tree agree with brute force on every unambiguous ray; transparency and the
error paths work as on the host-built tree."""
import ctypes as C
import importlib

import numpy as np
import pytest
import torch

from test_oracle_lbvh import soup

pytestmark = pytest.mark.gpu


def to_dev(arrs):
    return [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in arrs]


def device_bvh(rt, ctx, xyz, idx, max_leaf=4, width=4):
    x = torch.from_numpy(np.ascontiguousarray(xyz, np.float32).reshape(-1, 3)).cuda()
    i = torch.from_numpy(np.ascontiguousarray(idx, np.uint32).reshape(-1, 3).view(np.int32)).cuda()
    if x.shape[0] == 0:  # the entry point wants a vertex for any triangle; none here
        x = torch.zeros((1, 3), dtype=torch.float32, device="cuda")
    return rt.Bvh.from_device(ctx, x, i, max_leaf=max_leaf, width=width)


CASES = [(0, 4, 4, False), (1, 4, 4, False), (2, 4, 2, False), (3, 4, 4, False), (5, 1, 4, False),
         (100, 4, 2, False), (1000, 8, 4, False), (3000, 1, 4, True), (4096, 4, 4, False),
         (50000, 4, 4, False), (50000, 4, 2, False), (200000, 2, 4, True)]


@pytest.mark.parametrize("n,max_leaf,width,dup", CASES)
def test_device_build_equals_oracle(rt, orc, gpu_ctx, n, max_leaf, width, dup):
    print(f"[bvh device] n={n} max_leaf={max_leaf} width={width} dup={dup}", flush=True)
    xyz, idx = soup(rt, n, seed=n + 3, dup=dup)
    bvh = device_bvh(rt, gpu_ctx, xyz, idx, max_leaf, width)
    inf = bvh.info()
    nodes, tris = bvh.export()
    want, wn, wt, w4 = orc.lbvh_build(xyz, idx, max_leaf=max_leaf, wide=width == 4)
    assert (inf.num_nodes, inf.num_leaves, inf.max_depth) == (want["num_nodes"], want["num_leaves"],
                                                              want["max_depth"])
    assert inf.num_tris == n and inf.width == width
    assert np.array_equal(nodes.view(np.uint32), wn.view(np.uint32))
    assert np.array_equal(tris.view(np.uint32), wt.view(np.uint32))
    if width == 4:
        assert (inf.num_nodes4, inf.depth4, inf.stack_cap) == (want["num_nodes4"], want["depth4"],
                                                               want["max_stack4"] + 1)
        assert np.array_equal(bvh.export4().view(np.uint32), w4.view(np.uint32))
    else:
        assert inf.num_nodes4 == 0 and inf.stack_cap == want["max_depth"] + 1
    print(f"[bvh device] n={n}: {inf.num_nodes} nodes, depth {inf.max_depth}, sah {inf.sah_cost:.2f}, "
          f"{inf.build_ms:.2f} ms", flush=True)
    bvh.close()


def chain(rt, n):
    """Triangles halving their distance to a corner bit by bit (a radix tree
    that is a chain down to the last code bit) and n equal ones at its end (equal
    boxes: the wide nodes open one side only, so the wide tree is about as deep
    as the two-wide one)."""
    steps = [0.75 * 2.0**-k * np.eye(3)[a] for k in range(10) for a in range(3)]
    at = np.concatenate([np.array(steps), np.zeros((n, 3)), np.ones((1, 3))])
    shape = np.array([[0, 0, 0], [1, 0, 0], [0, 1, 1]]) * 2.0**-13
    xyz = (at[:, None, :] + shape[None]).astype(np.float32).reshape(-1, 3)
    return xyz, np.arange(xyz.shape[0], dtype=np.uint32).reshape(-1, 3)


@pytest.mark.parametrize("kind,n,max_leaf,width", [
    # one leaf more and less than one, two and three runs of 512 leaves
    ("soup", 511, 4, 4), ("soup", 512, 1, 4), ("soup", 513, 4, 4), ("soup", 1025, 8, 2), ("soup", 1537, 4, 4),
    # more wide levels than are launched before a look (16), at small and large sizes
    ("chain", 3, 1, 4), ("chain", 513, 1, 4), ("chain", 1 << 17, 1, 4),
    # a level of more entries than one tile per block (512 x 256)
    ("soup", 1 << 20, 1, 4)])
def test_runs_and_levels_equal_the_oracle(rt, orc, gpu_ctx, kind, n, max_leaf, width):
    print(f"[bvh device] {kind} n={n} max_leaf={max_leaf} width={width}", flush=True)
    xyz, idx = chain(rt, n) if kind == "chain" else rt.gen_soup(n, seed=n)
    bvh = device_bvh(rt, gpu_ctx, xyz, idx, max_leaf, width)
    inf = bvh.info()
    nodes, tris = bvh.export()
    want, wn, wt, w4 = orc.lbvh_build(xyz, idx, max_leaf=max_leaf, wide=width == 4)
    assert (inf.num_nodes, inf.max_depth) == (want["num_nodes"], want["max_depth"])
    assert np.array_equal(nodes.view(np.uint32), wn.view(np.uint32))
    assert np.array_equal(tris.view(np.uint32), wt.view(np.uint32))
    if width == 4:
        assert (inf.num_nodes4, inf.depth4, inf.stack_cap) == (want["num_nodes4"], want["depth4"],
                                                               want["max_stack4"] + 1)
        assert np.array_equal(bvh.export4().view(np.uint32), w4.view(np.uint32))
    bvh.close()


@pytest.mark.parametrize("width", [4, 2])
@pytest.mark.parametrize("n", [1, 5, 4096, 32768])
def test_traces_on_device_tree_match_brute_force(rt, orc, gpu_ctx, n, width):
    print(f"[bvh device trace] n={n} width={width}", flush=True)
    xyz, idx = soup(rt, n, seed=100 + n)
    rays = rt.gen_rays(64, 48, n_incoherent=4096, seed=n)
    bvh = device_bvh(rt, gpu_ctx, xyz, idx, width=width)
    prim, t = bvh.trace_closest(*to_dev(rays))
    torch.cuda.synchronize()
    prim, t = prim.cpu().numpy(), t.cpu().numpy()
    bp, bt, fl = orc.brute_trace(xyz, idx, rays)
    clean = fl == 0
    assert clean.mean() > 0.99
    assert np.array_equal(prim[clean], bp[clean])
    assert np.array_equal(t[clean], bt[clean])
    bvh.close()


def test_any_hit_with_transparency_on_device_tree(rt, orc, gpu_ctx):
    print("[bvh device any-hit]", flush=True)
    xyz, idx = rt.gen_soup(8192, seed=9, edge_mu=0.03)
    rays = rt.gen_rays(32, 32, n_incoherent=6000, seed=10)
    rng = np.random.default_rng(2)
    transparent = (rng.uniform(size=idx.shape[0]) < 0.3).astype(np.uint8)
    bp, bt, fl = orc.brute_trace(xyz, idx, rays, transparent=transparent, check_shadow=True)
    tmax = np.where(bp >= 0, bt * rng.choice([0.5, 2.0], bp.shape), 5.0).astype(np.float32)
    bvh = device_bvh(rt, gpu_ctx, xyz, idx)
    bvh.set_transparent(transparent)
    occ = bvh.trace_any(*to_dev(rays), torch.from_numpy(tmax).cuda())
    torch.cuda.synchronize()
    occ = occ.cpu().numpy().astype(bool)
    want = (bp >= 0) & (bt <= tmax)
    clean = fl == 0
    assert np.array_equal(occ[clean], want[clean])
    assert want.sum() > 100 and (~want).sum() > 100
    # the flags land on the exported records by triangle id
    _, tris = bvh.export()
    ids = tris[:-1, 3].copy().view(np.int32)
    assert np.array_equal(tris[:-1, 7].copy().view(np.uint32), transparent[ids].astype(np.uint32))
    bvh.close()


def test_bad_input_is_refused(rt, gpu_ctx):
    print("[bvh device errors]", flush=True)
    xyz, idx = rt.gen_soup(64, seed=1)
    bad = idx.copy()
    bad[3, 1] = xyz.shape[0]  # one past the last vertex: the kernel reads vertex 0 instead and reports it
    with pytest.raises(RuntimeError, match="out of range"):
        device_bvh(rt, gpu_ctx, xyz, bad)
    x2 = xyz.copy()
    x2[5, 0] = np.inf
    with pytest.raises(RuntimeError, match="non-finite"):
        device_bvh(rt, gpu_ctx, x2, idx)
    h = C.c_void_p()
    opts = rt.BvhOpts(9, 32, 1.2, 4)
    assert rt.lib().rt_bvh_build_device(gpu_ctx.h, None, 0, None, 0, C.byref(opts), C.byref(h)) != 0
    # the context still works
    bvh = device_bvh(rt, gpu_ctx, xyz, idx)
    assert bvh.info().num_tris == 64
    bvh.close()


def test_full_size_device_build(rt, orc, gpu_ctx):
    """The 1M-triangle soup (seed 7): the device build equals the oracle's
    record for record, and the kernel's closest hits on it agree with the
    restated traversal of the same tree except on rays brute force flags as
    ambiguous."""
    print("[bvh device full size] 1M soup", flush=True)
    xyz, idx = rt.gen_soup(1 << 20, seed=7)
    bvh = device_bvh(rt, gpu_ctx, xyz, idx)
    inf = bvh.info()
    print(f"[bvh device full size] {inf.build_ms:.1f} ms, {inf.num_nodes} nodes, depth {inf.max_depth}, "
          f"wide {inf.num_nodes4} depth4 {inf.depth4} stack {inf.stack_cap}, sah {inf.sah_cost:.2f}", flush=True)
    nodes, tris = bvh.export()
    nodes4 = bvh.export4()
    want, wn, wt, w4 = orc.lbvh_build(xyz, idx)
    assert np.array_equal(nodes.view(np.uint32), wn.view(np.uint32))
    assert np.array_equal(tris.view(np.uint32), wt.view(np.uint32))
    assert np.array_equal(nodes4.view(np.uint32), w4.view(np.uint32))
    coh = rt.gen_rays(4096, 2048, seed=7)
    inc = rt.gen_rays(0, 0, n_incoherent=1 << 15, seed=7)
    sel = np.random.default_rng(0).choice(4096 * 2048, 1 << 15, replace=False)
    rays = [np.concatenate([a[sel], b]) for a, b in zip(coh, inc)]
    prim, t = bvh.trace_closest(*to_dev(rays))
    torch.cuda.synchronize()
    prim, t = prim.cpu().numpy(), t.cpu().numpy()
    p2, t2, _, _, _ = orc.bvh4_trace(nodes4, tris, rays, nthreads=16)
    dk = np.nonzero((prim != p2) | (t != t2))[0]
    print(f"[bvh device full size] kernel vs restated traversal: {dk.size} rays differ", flush=True)
    assert dk.size <= 1e-4 * prim.size
    if dk.size:
        _, _, fk = orc.brute_trace(xyz, idx, [a[dk] for a in rays], nthreads=16)
        assert np.all(fk != 0), dk[fk == 0][:10]
    bvh.close()


def deep_chain(n):
    """Thirty steps towards a corner, each with four triangles larger than all
    that follows, and n equal ones at its end: the wide nodes open the steps'
    triangles, so up to three entries are pending per level."""
    rng = np.random.default_rng(1)
    out = []
    for k in range(10):
        for a in range(3):
            p = 0.75 * 2.0**-k * np.eye(3)[a]
            for j in range(4):
                t = rng.uniform(-1, 1, (3, 3))
                lo, hi = t.min(0), t.max(0)
                t = (t - (lo + hi) / 2) / (hi - lo) * 2  # the cube [-1, 1]^3 bounds it
                out.append(p + 1.5 * 2.0**-(k + a / 3) * (1 + 0.02 * j) * t)
    s = np.array([[0, 0, 0], [1, 0, 0], [0, 1, 1]]) * 2.0**-13
    out += [s] * n + [1 + s]
    xyz = np.array(out).astype(np.float32).reshape(-1, 3)
    return xyz, np.arange(xyz.shape[0], dtype=np.uint32).reshape(-1, 3)


def corner_rays(n, seed):
    """Rays that pass close by the corner from near and far."""
    rng = np.random.default_rng(seed)
    o = rng.normal(0, 1e-4, (n, 3))
    d = rng.normal(0, 1, (n, 3))
    d /= np.linalg.norm(d, axis=1)[:, None]
    o -= d * rng.choice([0, 1e-3, 3.0], (n, 1))
    return [np.ascontiguousarray(v[:, c].astype(np.float32)) for v in (o, d) for c in range(3)]


@pytest.mark.parametrize("n,cap", [(1, 92), (4096, 124), (16381, 128)])
def test_traversal_stack_bound(rt, orc, gpu_ctx, n, cap):
    """Trees that need a deep stack, up to the largest that is accepted (129
    entries of every lane in LDS with the mark at the bottom).  The restated
    walk's pending entries stay within the bound, and the kernels' hits are
    its hits: distances, and ids where no equal triangle ties."""
    xyz, idx = deep_chain(n)
    bvh = device_bvh(rt, gpu_ctx, xyz, idx, max_leaf=1)
    assert bvh.info().stack_cap == cap
    rays = corner_rays(5000, n)
    p2, t2, _, _, msp = orc.bvh4_trace(bvh.export4(), bvh.export()[1], rays)
    print(f"[bvh device] deep chain n={n}: {msp} entries of {cap}", flush=True)
    assert 80 <= msp <= cap - 1  # the rays use most of it
    prim, t = bvh.trace_closest(*to_dev(rays))
    occ = bvh.trace_any(*to_dev(rays), torch.full((5000,), 10.0, device="cuda"))
    torch.cuda.synchronize()
    prim, t, occ = prim.cpu().numpy(), t.cpu().numpy(), occ.cpu().numpy().astype(bool)
    assert np.array_equal(t, t2)
    steps = 120
    same = (p2 < steps) | (prim < steps)
    assert np.array_equal(prim[same], p2[same]) and np.all((prim >= steps) == (p2 >= steps))
    assert np.array_equal(occ, (p2 >= 0) & (t2 <= 10.0))
    bvh.close()
    two = device_bvh(rt, gpu_ctx, xyz, idx, max_leaf=1, width=2)
    t = two.trace_closest(*to_dev(rays))[1]
    torch.cuda.synchronize()
    assert np.array_equal(t.cpu().numpy(), t2)
    two.close()
    # one entry more is refused
    if cap == 128:
        with pytest.raises(rt.RtError):
            device_bvh(rt, gpu_ctx, *deep_chain(n + 2), max_leaf=1)


def test_deep_stack_in_the_renderer(rt, gpu_ctx):
    """The path tracer keeps 24 stack entries in LDS and the rest in private
    memory: a scene whose tree needs 124 gives the image of the same scene
    under a host-built tree, on (almost) every pixel."""
    scenes = importlib.import_module("2023_render_engine_amd.scenes")
    xyz, idx = deep_chain(4096)
    d = scenes.cornell(width=64, height=64, spp=4)
    d.xyz, d.idx, d.tri_mat = xyz, idx, (np.arange(len(idx)) % 3).astype(np.uint32)
    d.tri_mat[120:] = 0
    d.spheres, d.lights = [], [((-1.7, 0.4, 0.3), (1, 1, 1), 10.0), ((-1.5, -0.5, 0.6), (1, 1, 1), 10.0)]
    out = []
    for kw in (dict(), dict(bvh_on_device=True, bvh_max_leaf=1), dict(bvh_on_device=True, bvh_max_leaf=1, bvh_width=2)):
        sc = rt.Scene(gpu_ctx, d, **kw)
        film = sc.new_film()
        sc.render(film)
        torch.cuda.synchronize()
        out.append((film[0].cpu().numpy().reshape(-1, 3), film[1].cpu().numpy()))
        sc.close()
    assert out[0][0].mean() > 0
    for a, n in out[1:]:
        same = np.all(a == out[0][0], axis=1)
        print(f"[bvh device] deep stack in the renderer: {same.mean():.4f} of pixels equal", flush=True)
        assert np.array_equal(n, out[0][1])
        assert same.mean() >= 0.99
