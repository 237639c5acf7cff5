"""GPU parity of the traversal path, through the C ABI, against the CPU oracle.

Bar (closest hit): the GPU hit index equals the oracle's on >= 99.99% of rays,
where a differing index counts as agreeing only at a near-tie, i.e. both hit
and |t_gpu - t_cpu| <= 1e-6 * t (the agreement tolerance of this path). On
the small test meshes the reference's own 1e-5 absolute slop
(IndexedTriangle.cpp:114-115, under which the first triangle found wins) also
counts as a tie; the 1.33M-triangle sets are held to the 1e-6 relative rule
alone on all of their rays, and report the rest by cause. Any-hit: occlusion bits equal on
>= 99.99% of rays. The oracle is the C++ restatement of the reference's
triangle test and BVHMesh / BasicMesh traversal.
"""
import os

import numpy as np
import pytest

from tests import meshgen

pytestmark = pytest.mark.gpu

F32MAX = float(np.finfo(np.float32).max)


def _compare_closest(ph, th, pc, tc, label):
    n = len(ph)
    same = ph == pc
    both = (ph >= 0) & (pc >= 0)
    dt = np.abs(th.astype(np.float64) - tc.astype(np.float64))
    near = both & ((dt <= 1e-6 * np.maximum(tc, 1e-30)) | (dt <= 1e-5))
    agree = same | near
    frac = agree.mean()
    print(f"[{label}] n={n} index-equal={same.mean():.6f} agree(incl. near-ties)={frac:.6f} "
          f"hit-rate gpu={np.mean(ph >= 0):.4f} cpu={np.mean(pc >= 0):.4f}", flush=True)
    bad = np.nonzero(~agree)[0][:5]
    for i in bad:
        print(f"   ray {i}: gpu ({ph[i]}, {th[i]!r}) cpu ({pc[i]}, {tc[i]!r})", flush=True)
    return frac


def _small_scene():
    sp, si = meshgen.icosphere(4)
    tp, ti = meshgen.random_triangles(2000, seed=5, extent=1.5)
    bp, bi = meshgen.quad([-3, -1.2, -3], [-3, -1.2, 3], [3, -1.2, 3], [3, -1.2, -3])
    return meshgen.merge([(sp, si), (tp, ti), (bp, bi)])


@pytest.mark.parametrize("builder,fmt,width", [(0, 0, 4), (1, 0, 4), (2, 0, 4), (3, 0, 4), (4, 0, 4), (0, 1, 4),
                                               (1, 1, 4), (4, 1, 4), (0, 0, 2), (0, 0, 8), (1, 0, 8), (2, 0, 8)])
def test_closest_matches_oracle_brute_force(gpu_ctx, ilm, orc, builder, fmt, width):
    pos, idx = _small_scene()
    rays = np.concatenate([meshgen.rays_toward(30000, pos, seed=7), meshgen.random_rays(20000, seed=8)])
    n = len(rays)
    m = ilm.Mesh(gpu_ctx, pos, idx)
    info = m.build(builder=builder, node_format=fmt, width=width)
    assert info["width"] == width
    rb = ilm.rays_to_device(gpu_ctx, rays)
    hb = gpu_ctx.buffer(n * 16)
    m.trace_closest(rb, n, hb)
    gpu_ctx.sync()
    h = hb.download(ilm.HIT_DTYPE, n)
    om = orc.Mesh(pos, idx)
    pc, tc = om.trace(rays, mode=0, accel=0)
    assert _compare_closest(h["prim"], h["t"], pc, tc, f"brute b{builder} f{fmt} w{width}") >= 0.9999
    # barycentrics reproduce the hit point on the triangle
    ok = h["prim"] >= 0
    tri = pos[idx[h["prim"][ok]]]
    P = rays[ok, 0:3] + h["t"][ok, None] * rays[ok, 4:7]
    Q = (1 - h["u"][ok] - h["v"][ok])[:, None] * tri[:, 0] + h["u"][ok, None] * tri[:, 1] + h["v"][ok, None] * tri[:, 2]
    assert np.abs(P - Q).max() < 1e-4
    for b in (rb, hb):
        b.free()
    m.close()


@pytest.mark.parametrize("builder,fmt,width", [(0, 0, 4), (1, 0, 4), (0, 1, 4), (0, 0, 2), (0, 0, 8)])
def test_room_fixture(gpu_ctx, ilm, builder, fmt, width):
    """The committed box-room fixture (closest hits and shadow occlusion of
    the oracle's brute force, pinned by float64 rectangle geometry)."""
    g = np.load(os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "room_rays_4096.npz"))
    m = ilm.Mesh(gpu_ctx, g["pos"], g["idx"])
    m.build(builder=builder, node_format=fmt, width=width)
    n = len(g["closest_rays"])
    rb = ilm.rays_to_device(gpu_ctx, g["closest_rays"])
    sb = ilm.rays_to_device(gpu_ctx, g["shadow_rays"])
    hb, ob = gpu_ctx.buffer(n * 16), gpu_ctx.buffer(n)
    m.trace_closest(rb, n, hb)
    m.trace_any(sb, n, ob)
    gpu_ctx.sync()
    h = hb.download(ilm.HIT_DTYPE, n)
    # every ray agrees (the boxes' bottom faces lie on the floor: exact ties may go either way)
    assert _compare_closest(h["prim"], h["t"], g["closest_prim"], g["closest_t"], f"room b{builder} f{fmt} w{width}") == 1.0
    assert np.array_equal(ob.download(np.uint8, n), g["shadow_occluded"])
    for b in (rb, sb, hb, ob):
        b.free()
    m.close()


@pytest.mark.parametrize("builder,fmt,width", [(0, 0, 4), (1, 0, 4), (0, 1, 4), (4, 0, 4)])
def test_rays_along_box_faces(gpu_ctx, ilm, orc, builder, fmt, width):
    """Rays with a zero direction component in the plane of box faces: the
    GPU's slab test (fminf/fmaxf drop the NaN of 0 * inf) finds what the
    oracle's BasicMesh finds, also on the reference topology, where the
    oracle's BVHMesh loses the hits."""
    from tests.test_oracle import zero_direction_fans
    P, idx, rays = zero_direction_fans()
    m = ilm.Mesh(gpu_ctx, P, idx)
    m.build(builder=builder, node_format=fmt, width=width)
    n = len(rays)
    rb = ilm.rays_to_device(gpu_ctx, rays)
    hb = gpu_ctx.buffer(n * 16)
    m.trace_closest(rb, n, hb)
    gpu_ctx.sync()
    h = hb.download(ilm.HIT_DTYPE, n)
    pb, tb = orc.Mesh(P, idx).trace(rays, 0, 0)
    assert (h["prim"] >= 0).all() and np.allclose(h["t"], tb, rtol=1e-6, atol=0)
    for b in (rb, hb):
        b.free()
    m.close()


@pytest.mark.parametrize("builder,fmt,width", [(0, 0, 4), (2, 0, 4), (4, 0, 4), (0, 1, 4), (0, 0, 2), (0, 0, 8)])
def test_any_matches_oracle(gpu_ctx, ilm, orc, builder, fmt, width):
    pos, idx = _small_scene()
    rays = meshgen.rays_toward(40000, pos, seed=17)
    rays[:, 7] = np.random.default_rng(3).uniform(0.5, 4.0, len(rays)).astype(np.float32)  # finite segments
    n = len(rays)
    m = ilm.Mesh(gpu_ctx, pos, idx)
    m.build(builder=builder, node_format=fmt, width=width)
    rb = ilm.rays_to_device(gpu_ctx, rays)
    ob = gpu_ctx.buffer(n)
    m.trace_any(rb, n, ob)
    gpu_ctx.sync()
    occ = ob.download(np.uint8, n)
    om = orc.Mesh(pos, idx)
    pc, _ = om.trace(rays, mode=1, accel=0)
    if builder == 2:
        # the KDTreeMesh restatement's any-hit agrees with brute force too
        om.kd_build(1, 10, 35)
        pk, _ = om.trace(rays, mode=1, accel=2)
        assert ((pk >= 0) == (pc >= 0)).mean() >= 0.9999
    agree = (occ == (pc >= 0)).mean()
    print(f"[any] agree={agree:.6f} occluded={occ.mean():.4f}")
    assert agree >= 0.9999
    m.close()


def test_space_matches_oracle_basicspace(gpu_ctx, ilm, orc):
    # One flattened world-space BVH against the BasicSpace restatement, which
    # transforms every ray into every primitive's object space.
    inst = meshgen.instances(seed=1)
    space = orc.Space()
    keep = []
    sp = ilm.Space(gpu_ctx)
    for pos, idx, rot, scl, trn in inst:
        m = orc.Mesh(pos, idx)
        m.build(10, 35)
        keep.append(m)
        space.add(m, rot, scl, trn)
        sp.add(pos, idx, None, rot, scl, trn)
    sp.build()
    wp, _, _, _ = meshgen.flatten_instances(inst)
    rays = np.concatenate([meshgen.rays_toward(30000, wp, seed=3, dist=6.0), meshgen.random_rays(10000, seed=4)])
    n = len(rays)
    rb = ilm.rays_to_device(gpu_ctx, rays)
    hb, pb_, lb, ob = gpu_ctx.buffer(n * 16), gpu_ctx.buffer(n * 4), gpu_ctx.buffer(n * 4), gpu_ctx.buffer(n)
    sp.mesh.trace_closest(rb, n, hb)
    sp.resolve(hb, n, pb_, lb)
    sp.mesh.trace_any(rb, n, ob)
    gpu_ctx.sync()
    h = hb.download(ilm.HIT_DTYPE, n)
    gp, gl, occ = pb_.download(np.int32, n), lb.download(np.int32, n), ob.download(np.uint8, n)
    p, tr, t = space.trace(rays, mode=0)
    key_g = np.where(gp >= 0, gp * 100000 + gl, -1)
    key_c = np.where(p >= 0, p * 100000 + tr, -1)
    assert _compare_closest(key_g, h["t"], key_c, t, "space") >= 0.9999
    pa, _, _ = space.trace(rays, mode=1)
    assert (occ == (pa >= 0)).mean() >= 0.9999
    for b in (rb, hb, pb_, lb, ob):
        b.free()
    sp.close()


@pytest.mark.parametrize("ntri", [1, 3, 5, 2000, 100000])
def test_lbvh_structure(gpu_ctx, ilm, ntri):
    # The device builder's BVH4: every triangle in exactly one leaf, leaves of
    # at most max_leaf triangles, every child box containing its subtree, and
    # every node reachable once from the root.
    pos, idx = meshgen.random_triangles(ntri, seed=ntri, extent=2.0, size=0.05)
    m = ilm.Mesh(gpu_ctx, pos, idx)
    info = m.build(builder=ilm.ILM_BUILDER_LBVH, max_leaf=4)
    nodes, order = m.export()
    boxes, child = ilm.decode_bvh4(nodes)
    assert len(boxes) == info["nodes"] and np.array_equal(np.sort(order), np.arange(ntri))
    tri = pos[idx]
    tlo, thi = tri.min(axis=1), tri.max(axis=1)
    seen = np.zeros(ntri, np.int64)
    visited = np.zeros(len(boxes), np.int64)
    stack = [(0, None)]
    while stack:
        ni, pbox = stack.pop()
        visited[ni] += 1
        for k in range(4):
            c = int(child[ni, k])
            b = boxes[ni, k]
            if c & 0x80000000:
                cnt, first = c & 31, (c & 0x7FFFFFFF) >> 5
                if cnt == 0:
                    continue
                assert cnt <= 4
                ids = order[first:first + cnt]
                seen[ids] += 1
                assert (tlo[ids] >= b[:3]).all() and (thi[ids] <= b[3:]).all()
            else:
                stack.append((c, b))
            if pbox is not None:
                assert (b[:3] >= pbox[:3]).all() and (b[3:] <= pbox[3:]).all()
    assert (seen == 1).all() and (visited == 1).all()
    assert info["max_leaf"] <= 4 and info["build_ms"] > 0
    m.close()


def test_empty_and_tiny_inputs(gpu_ctx, ilm):
    pos, idx = meshgen.quad([0, 0, 0], [1, 0, 0], [1, 1, 0], [0, 1, 0])
    m = ilm.Mesh(gpu_ctx, pos, idx)
    info = m.build()
    assert info["nodes"] == 1
    rays = np.array([[0.25, 0.5, 1, 0, 0, 0, -1, F32MAX],      # hits
                     [0.25, 0.5, 1, 0, 0, 0, 1, F32MAX],       # points away
                     [0.25, 0.5, 1, 0, 0, 0, -1, 0.5],         # segment too short
                     [2.0, 0.5, 1, 0, 0, 0, -1, F32MAX]], np.float32)  # beside
    rb = ilm.rays_to_device(gpu_ctx, rays)
    hb = gpu_ctx.buffer(4 * 16)
    m.trace_closest(rb, 0, hb)          # n = 0 is a no-op
    m.trace_closest(rb, 4, hb)
    gpu_ctx.sync()
    h = hb.download(ilm.HIT_DTYPE, 4)
    assert h["prim"][0] in (0, 1) and h["t"][0] == 1.0
    assert (h["prim"][1:] == -1).all()
    m.close()


def test_every_ray_traced_once_for_any_count(gpu_ctx, ilm, orc):
    """Launches split their rays into eight segments with their own fetch
    counters (one per XCD) and only the first ceil(n / 64) waves take part:
    for counts around those boundaries every ray is traced (no hit record
    keeps its sentinel) and hits equal brute force; any hits too."""
    pos, idx = _small_scene()
    rays_all = meshgen.rays_toward(5000, pos, seed=21)
    m = ilm.Mesh(gpu_ctx, pos, idx)
    m.build()
    om = orc.Mesh(pos, idx)
    pc_all, tc_all = om.trace(rays_all, mode=0, accel=0)
    oc_all, _ = om.trace(rays_all, mode=1, accel=0)
    rb = ilm.rays_to_device(gpu_ctx, rays_all)
    hb = gpu_ctx.buffer(len(rays_all) * 16)
    ob = gpu_ctx.buffer(len(rays_all))
    sentinel = np.zeros(len(rays_all), ilm.HIT_DTYPE)
    sentinel["prim"] = -7
    for n in (1, 2, 7, 8, 9, 15, 63, 64, 65, 127, 129, 511, 512, 513, 1000, 4095, 4097, 5000):
        hb.upload(sentinel)
        ob.upload(np.full(len(rays_all), 9, np.uint8))
        m.trace_closest(rb, n, hb)
        m.trace_any(rb, n, ob)
        gpu_ctx.sync()
        h = hb.download(ilm.HIT_DTYPE, len(rays_all))
        occ = ob.download(np.uint8, len(rays_all))
        assert (h["prim"][:n] != -7).all() and (h["prim"][n:] == -7).all(), n
        assert (occ[:n] != 9).all() and (occ[n:] == 9).all(), n
        assert _compare_closest(h["prim"][:n], h["t"][:n], pc_all[:n], tc_all[:n], f"n={n}") >= 0.999
        assert (occ[:n] == (oc_all[:n] >= 0)).mean() >= 0.999
    for b in (rb, hb, ob):
        b.free()
    m.close()


@pytest.fixture(scope="module")
def c2(gpu_ctx, ilm):
    from illuminaprt_amd import workloads
    pos, idx = workloads.intersection_scene()
    m = ilm.Mesh(gpu_ctx, pos, idx)
    info = m.build()
    rs = workloads.intersection_rays(gpu_ctx, m)
    print(f"[c2] tris={len(idx)} bvh={info} centre_hits={rs.centre_hits} replaced={rs.replaced}", flush=True)
    yield pos, idx, m, rs
    rs.free()
    m.close()


@pytest.fixture(scope="module")
def c2_oracle(c2, orc):
    """The oracle's BVHMesh over the 1,334,720 triangles (reference topology:
    128-bin count heuristic, leaves of at most 10, depth 35)."""
    pos, idx, _, _ = c2
    om = orc.Mesh(pos, idx)
    om.build(10, 35)
    return om


def _classify_disagreements(orc, om, pos, idx, rays, ph, th, pc, tc):
    """Rays whose index differs from the oracle's BVHMesh and are not
    near-ties under the 1e-6 relative rule, by cause. The oracle's BasicMesh
    (brute force over every triangle, BasicMesh.cpp:16-64) traces each such
    ray again:
    'bvhmesh' BasicMesh finds the GPU's hit (or a 1e-6 near-tie of it) where
    BVHMesh does not: the reference's traversal loses a closer hit. The known
    cause is the slab test's 0 * inf = NaN (BoundingBox.cpp:212-232 with
    Maths::Min/Max's argument order): a ray with a zero direction component
    whose origin lies on a box face is rejected by that box;
    'slop' both hit within the reference's 1e-5 absolute window
    (IndexedTriangle.cpp:114-115: a later triangle within 1e-5 of the current
    hit cannot replace it, so the first one found wins);
    'leak' the GPU's triangle is one the reference's Shirley test misses for
    this ray (a ray through a shared edge or vertex that the Shirley test lets
    through, while the watertight test counts it); 'other' the rest.
    Returns (fraction equal or a near-tie of BVHMesh, fraction equal or a
    near-tie of BVHMesh or of BasicMesh, counts by cause, 'other' rays,
    rays of the 'bvhmesh' class with a zero direction component)."""
    both = (ph >= 0) & (pc >= 0)
    dt = np.abs(th.astype(np.float64) - tc.astype(np.float64))
    ns = (ph == pc) | (both & (dt <= 1e-6 * np.maximum(np.abs(tc.astype(np.float64)), 1e-30)))
    out = {"bvhmesh": 0, "slop": 0, "leak": 0, "other": 0}
    others = []
    bad = np.nonzero(~ns)[0]
    pb, tb = om.trace(rays[bad], mode=0, accel=0) if len(bad) else (np.zeros(0, np.int32), np.zeros(0, np.float32))
    zero_dir = 0
    for j, i in enumerate(bad):
        dtb = abs(float(th[i]) - float(tb[j]))
        if ph[i] == pb[j] or (ph[i] >= 0 and pb[j] >= 0 and dtb <= 1e-6 * max(abs(float(tb[j])), 1e-30)):
            out["bvhmesh"] += 1
            zero_dir += bool((rays[i, 4:7] == 0).any())
            continue
        if both[i] and dt[i] <= 1e-5:
            out["slop"] += 1
            continue
        if ph[i] >= 0:
            tri = pos[idx[ph[i]]]
            hit = orc.tri_intersect(tri[0], tri[1], tri[2], rays[i, 0:3], rays[i, 4:7], rays[i, 7])
            if not hit[0]:
                out["leak"] += 1
                continue
        out["other"] += 1
        others.append(int(i))
    n = len(ph)
    return ns.mean(), (ns.sum() + out["bvhmesh"]) / n, out, others, zero_dir


@pytest.mark.parametrize("power", [-51, -40, 0, 40, 60])
def test_hits_do_not_depend_on_a_power_of_two_scale(power, gpu_ctx, ilm):
    """Geometry and rays scaled by a power of two: every product and quotient
    of the ray set-up and the triangle test scales exactly, so t, u, v and the
    triangle are the same bit for bit, whichever division (the plain one, or
    the general one for determinants outside [1e-30, 1e30]) is taken."""
    pos, idx = meshgen.icosphere(3)
    rays = meshgen.rays_toward(6000, pos, seed=6)
    d = np.abs(rays[:, 4:7])
    rays = rays[d.min(axis=1) > 0.01 * d.max(axis=1)]   # no component near the 1e-18 that stands for 0
    hits = []
    for e in (0, power):
        k = np.float32(2.0 ** e)
        m = ilm.Mesh(gpu_ctx, pos * k, idx)
        m.build()
        scaled = rays.copy()
        scaled[:, 0:3] *= k
        scaled[:, 4:7] *= k
        rb, hb = ilm.rays_to_device(gpu_ctx, scaled), gpu_ctx.buffer(len(rays) * 16)
        m.trace_closest(rb, len(rays), hb)
        gpu_ctx.sync()
        hits.append(hb.download(ilm.HIT_DTYPE, len(rays)))
        rb.free()
        hb.free()
        m.close()
    assert (hits[0]["prim"] >= 0).mean() > 0.3
    assert np.array_equal(hits[0].view(np.uint32), hits[1].view(np.uint32))


@pytest.mark.parametrize("any_hit", [False, True])
def test_ray_counts_around_the_shares_of_a_launch(any_hit, gpu_ctx, ilm):
    """A launch deals its rays out to the waves (1 to 64 each) and fetches the
    rest of a long one by counters: at counts around each of these lines every
    output equals, bit for bit, that of the same ray in short launches, and
    nothing past the last is written. The shares depend on the CU count; the
    grid has at most 8 workgroups of 256 per CU."""
    pos, idx = meshgen.icosphere(3)
    m = ilm.Mesh(gpu_ctx, pos, idx)
    cus = gpu_ctx.cu_count
    most = 3 * cus * 8 * 256 + 77
    rng = np.random.default_rng(3)
    few = meshgen.rays_toward(4000, pos, seed=4)
    rays = few[rng.integers(len(few), size=most)]
    rb, fb = ilm.rays_to_device(gpu_ctx, rays), ilm.rays_to_device(gpu_ctx, few)
    size = 1 if any_hit else 16
    out, ref = gpu_ctx.buffer((most + 64) * size), gpu_ctx.buffer(len(few) * size)
    kind = np.dtype(np.uint8) if any_hit else ilm.HIT_DTYPE
    lines = [8 * cus, 64 * 8 * cus] + [64 * 4 * k * cus for k in range(4, 9)] + [2 * 64 * 4 * 7 * cus]
    counts = sorted({n + d for n in lines for d in (-1, 0, 1, 13)} | {most})
    for width, fmt in ((4, 0), (4, 1), (2, 0)):
        m.build(node_format=fmt, width=width)
        trace = m.trace_any if any_hit else m.trace_closest
        for at in range(0, len(few), 500):      # short launches of 500
            part, o = gpu_ctx.to_device(few[at:at + 500]), gpu_ctx.buffer(500 * size)
            trace(part, 500, o)
            gpu_ctx.sync()
            ref.upload(o.download(np.uint8, 500 * size), at * size)
            part.free()
            o.free()
        want = ref.download(kind, len(few))
        rng = np.random.default_rng(3)
        want = want[rng.integers(len(few), size=most)]
        for n in counts:
            out.upload(np.full((most + 64) * size, 0xA5, np.uint8))
            trace(rb, n, out)
            gpu_ctx.sync()
            got = out.download(np.uint8, (n + 64) * size)
            assert np.array_equal(got[:n * size], want[:n].view(np.uint8)), (width, fmt, n)
            assert (got[n * size:] == 0xA5).all(), (width, fmt, n)
    for x in (rb, fb, out, ref):
        x.free()
    m.close()


@pytest.mark.parametrize("ntri", [5, 8, 255, 256, 257, 511, 513, 65535, 65537, 140001])
def test_lbvh_boxes_are_tight(ntri, gpu_ctx, ilm):
    """Every child's box is exactly the union of its triangles' boxes (unions
    of floats do not round), at triangle counts around the aligned runs of 256
    and 65,536 sorted leaves that the boxes are made from; the reported
    largest leaf and depth are those of the tree."""
    pos, idx = meshgen.random_triangles(ntri, seed=ntri, extent=2.0, size=0.05)
    m = ilm.Mesh(gpu_ctx, pos, idx)
    info = m.build(builder=ilm.ILM_BUILDER_LBVH, max_leaf=3)
    nodes, order = m.export()
    boxes, child = ilm.decode_bvh4(nodes)
    tri = pos[idx]
    tlo, thi = tri.min(axis=1), tri.max(axis=1)
    levels, largest, seen = [np.array([0])], 0, 0
    while len(levels[-1]):
        c = child[levels[-1]]
        levels.append(c[(c & 0x80000000) == 0])
    lo, hi = np.full((len(boxes), 3), np.inf, np.float32), np.full((len(boxes), 3), -np.inf, np.float32)
    for level in reversed(levels[:-1]):
        for k in range(4):
            c = child[level, k]
            blo, bhi = np.full((len(level), 3), np.inf, np.float32), np.full((len(level), 3), -np.inf, np.float32)
            leaf = (c & 0x80000000) != 0
            blo[~leaf], bhi[~leaf] = lo[c[~leaf]], hi[c[~leaf]]
            cnt, first = c & 31, (c & 0x7FFFFFFF) >> 5
            for j in range(int(cnt[leaf].max(initial=0))):
                has = leaf & (cnt > j)
                ids = order[first[has] + j]
                blo[has], bhi[has] = np.minimum(blo[has], tlo[ids]), np.maximum(bhi[has], thi[ids])
                seen += int(has.sum())
            largest = max(largest, int(cnt[leaf].max(initial=0)))
            used = ~leaf | (cnt > 0)
            assert np.array_equal(blo[used], boxes[level, k, :3][used])
            assert np.array_equal(bhi[used], boxes[level, k, 3:][used])
            lo[level], hi[level] = np.minimum(lo[level], blo), np.maximum(hi[level], bhi)
    assert seen == ntri and sum(len(x) for x in levels) == info["nodes"]
    assert info["depth"] == len(levels) - 1 and info["max_leaf"] == largest
    m.close()


@pytest.mark.parametrize("node_format", [0, 1])
def test_lbvh_builds_reuse_the_workspace(node_format, gpu_ctx, ilm):
    """Builds of growing and shrinking sizes, whose scratch is kept between
    them, leave every mesh's own tree intact: hits equal the SAH tree's."""
    built = []
    for ntri in (3000, 60000, 2, 500, 60001):
        pos, idx = meshgen.random_triangles(ntri, seed=ntri, extent=2.0, size=0.05)
        m = ilm.Mesh(gpu_ctx, pos, idx)
        m.build(builder=ilm.ILM_BUILDER_LBVH, node_format=node_format)
        built.append((pos, idx, m))
    for pos, idx, m in built:
        ref = ilm.Mesh(gpu_ctx, pos, idx)
        ref.build(node_format=node_format)
        rays = meshgen.rays_toward(3000, pos, seed=2)
        rb, ha, hb = ilm.rays_to_device(gpu_ctx, rays), gpu_ctx.buffer(3000 * 16), gpu_ctx.buffer(3000 * 16)
        m.trace_closest(rb, 3000, ha)
        ref.trace_closest(rb, 3000, hb)
        gpu_ctx.sync()
        a, b = ha.download(ilm.HIT_DTYPE, 3000), hb.download(ilm.HIT_DTYPE, 3000)
        assert _compare_closest(a["prim"], a["t"], b["prim"], b["t"], f"lbvh {len(idx)}") >= 0.9999
        for x in (rb, ha, hb):
            x.free()
        ref.close()
        m.close()


@pytest.mark.parametrize("kind", ["primary", "incoherent"])
def test_c2_closest_matches_oracle_bvhmesh(c2, c2_oracle, gpu_ctx, ilm, orc, kind):
    """1,334,720 triangles: GPU closest hit vs the oracle's BVHMesh (reference
    topology, unordered recursive traversal) on every one of the 4,194,304
    rays of the set. The bar: index equal, or both hit with
    |t_gpu - t_cpu| <= 1e-6 t, on >= 99.99% of rays, against the reference's
    CPU Intersect: BVHMesh, or BasicMesh on the rays where the two
    reference meshes disagree (BVHMesh's slab test loses hits on rays with a
    zero direction component: the pixel-centre rays of the camera's middle
    column). The rest are counted by cause."""
    pos, idx, m, rs = c2
    buf = rs.primary if kind == "primary" else rs.incoherent
    n = rs.n
    hb = gpu_ctx.buffer(n * 16)
    m.trace_closest(buf, n, hb)
    gpu_ctx.sync()
    h = hb.download(ilm.HIT_DTYPE, n)
    rays = buf.download(np.float32, 8 * n).reshape(n, 8)
    if kind == "primary":
        assert (h["prim"] >= 0).all()   # the primary set is made of hitting rays
    pc, tc = c2_oracle.trace(rays, mode=0, accel=1)
    strict, frac, cls, others, zero_dir = _classify_disagreements(orc, c2_oracle, pos, idx, rays, h["prim"], h["t"],
                                                                  pc, tc)
    loose = _compare_closest(h["prim"], h["t"], pc, tc, f"c2 {kind} (all rays)")
    print(f"[c2 {kind}] 1e-6-relative rule: vs BVHMesh {strict:.7f}, vs BVHMesh or BasicMesh {frac:.7f}; "
          f"the rest by cause {cls}; BVHMesh-lost hits on rays with a zero direction component: {zero_dir}",
          flush=True)
    for i in others[:5]:
        print(f"   other ray {i}: gpu ({h['prim'][i]}, {h['t'][i]!r}) cpu ({pc[i]}, {tc[i]!r})", flush=True)
    assert frac >= 0.9999 and loose >= strict
    hb.free()


def test_c2_quantized_matches_float(c2, gpu_ctx, ilm):
    """64-byte quantised nodes find the same closest hits as the float nodes
    of the same tree on all 4,194,304 incoherent rays (near-ties aside)."""
    pos, idx, m, rs = c2
    n = rs.n
    mq = ilm.Mesh(gpu_ctx, pos, idx)
    info = mq.build(node_format=ilm.ILM_NODES_QUANTIZED)
    print(f"[c2 quantised] {info}", flush=True)
    ha, hb = gpu_ctx.buffer(n * 16), gpu_ctx.buffer(n * 16)
    m.trace_closest(rs.incoherent, n, ha)
    mq.trace_closest(rs.incoherent, n, hb)
    gpu_ctx.sync()
    a, b = ha.download(ilm.HIT_DTYPE, n), hb.download(ilm.HIT_DTYPE, n)
    assert _compare_closest(b["prim"], b["t"], a["prim"], a["t"], "c2 quantised vs float") >= 0.99999
    for x in (ha, hb):
        x.free()
    mq.close()


def test_c2_lbvh_matches_sah(c2, gpu_ctx, ilm):
    """The device-built tree finds the same closest hits as the host SAH tree
    on all 4,194,304 incoherent rays (near-ties aside)."""
    pos, idx, m, rs = c2
    n = rs.n
    ml = ilm.Mesh(gpu_ctx, pos, idx)
    info = ml.build(builder=ilm.ILM_BUILDER_LBVH)
    print(f"[c2 lbvh] {info}", flush=True)
    ha, hb = gpu_ctx.buffer(n * 16), gpu_ctx.buffer(n * 16)
    m.trace_closest(rs.incoherent, n, ha)
    ml.trace_closest(rs.incoherent, n, hb)
    gpu_ctx.sync()
    a, b = ha.download(ilm.HIT_DTYPE, n), hb.download(ilm.HIT_DTYPE, n)
    assert _compare_closest(b["prim"], b["t"], a["prim"], a["t"], "c2 lbvh vs sah") >= 0.99999
    for x in (ha, hb):
        x.free()
    ml.close()


def test_c2_shadow_matches_oracle_and_closest(c2, c2_oracle, gpu_ctx, ilm, orc):
    pos, idx, m, rs = c2
    n = rs.n
    ob = gpu_ctx.buffer(n)
    m.trace_any(rs.shadow, n, ob)
    hb = gpu_ctx.buffer(n * 16)
    m.trace_closest(rs.shadow, n, hb)
    gpu_ctx.sync()
    occ = ob.download(np.uint8, n)
    h = hb.download(ilm.HIT_DTYPE, n)
    # size-independent property over all 4,194,304 rays: any-hit == closest-hit exists
    assert np.array_equal(occ.astype(bool), h["prim"] >= 0)
    rays = rs.shadow.download(np.float32, 8 * n).reshape(n, 8)
    # segment endpoints lie on the 0.5 x 0.5 light at y = 2.5
    end = rays[:, 0:3] + rays[:, 4:7]
    assert np.abs(end[:, 1] - 2.5).max() < 1e-5
    assert (np.abs(end[:, 0]) <= 0.25 + 1e-5).all() and (np.abs(end[:, 2]) <= 0.25 + 1e-5).all()
    # every one of the 4,194,304 segments against the oracle's any hit
    pc, _ = c2_oracle.trace(rays, mode=1, accel=1)
    diff = occ.astype(bool) != (pc >= 0)
    agree = 1.0 - diff.mean()
    # a differing segment: does the oracle's BasicMesh (brute force) agree
    # with the GPU, and does the oracle's Shirley test miss the triangle the GPU found?
    dix = np.nonzero(diff)[0]
    pb, _ = c2_oracle.trace(rays[dix], mode=1, accel=0) if len(dix) else (np.zeros(0, np.int32), None)
    basic = int(((pb >= 0) == occ[dix].astype(bool)).sum())
    leak = 0
    for i in np.nonzero(diff & (h["prim"] >= 0))[0]:
        tri = pos[idx[h["prim"][i]]]
        leak += not orc.tri_intersect(tri[0], tri[1], tri[2], rays[i, 0:3], rays[i, 4:7], rays[i, 7])[0]
    print(f"[c2 shadow] all {n} segments: agree={agree:.7f} occluded={occ.mean():.4f} differing={int(diff.sum())} "
          f"(gpu occluded, cpu not: {int((diff & occ.astype(bool)).sum())}, of which the oracle's test misses "
          f"the gpu's triangle: {leak}; cpu occluded, gpu not: {int((diff & ~occ.astype(bool)).sum())}; "
          f"BasicMesh agrees with the gpu on {basic} of them)", flush=True)
    assert agree >= 0.9999
    ob.free()
    hb.free()


def test_c2_determinism_and_hit_geometry(c2, gpu_ctx, ilm):
    pos, idx, m, rs = c2
    n = rs.n
    a, b = gpu_ctx.buffer(n * 16), gpu_ctx.buffer(n * 16)
    m.trace_closest(rs.incoherent, n, a)
    m.trace_closest(rs.incoherent, n, b)
    gpu_ctx.sync()
    ha, hb = a.download(ilm.HIT_DTYPE, n), b.download(ilm.HIT_DTYPE, n)
    assert np.array_equal(ha.view(np.uint32), hb.view(np.uint32))   # bit-identical runs
    rays = rs.incoherent.download(np.float32, 8 * n).reshape(n, 8)
    ok = ha["prim"] >= 0
    tri = pos[idx[ha["prim"][ok]]]
    P = rays[ok, 0:3] + ha["t"][ok, None] * rays[ok, 4:7]
    nrm = np.cross(tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 0])
    nrm /= np.linalg.norm(nrm, axis=1, keepdims=True)
    assert np.abs(np.einsum("ij,ij->i", P - tri[:, 0], nrm)).max() < 1e-4   # on the plane
    assert (ha["u"][ok] >= -1e-6).all() and (ha["v"][ok] >= -1e-6).all() and \
        (ha["u"][ok] + ha["v"][ok] <= 1 + 1e-6).all()
    # incoherent directions are unit and cosine-distributed about the normal
    d = rays[:, 4:7]
    assert np.abs(np.linalg.norm(d, axis=1) - 1).max() < 1e-5
    a.free()
    b.free()


def test_compaction_and_camera(gpu_ctx, ilm, orc):
    from illuminaprt_amd import workloads
    cam = workloads.intersection_camera()
    W = H = 256
    rb = gpu_ctx.buffer(W * H * 32)
    gpu_ctx.raygen_camera(cam, W, H, rb)
    gpu_ctx.sync()
    rays = rb.download(np.float32, W * H * 8).reshape(-1, 8)
    for (x, y) in [(0, 0), (128, 128), (255, 17), (3, 250)]:
        o, d = orc.camera_ray(cam.as_list(), W, H, x, y, 0.5, 0.5)
        r = rays[y * W + x]
        assert np.allclose(r[0:3], o) and np.allclose(r[4:7], d, atol=2e-7)
    # compaction: hits with prim >= 0, in index order
    n = 100003
    prim = np.where(np.random.default_rng(0).random(n) < 0.3, 1, -1).astype(np.int32)
    hits = np.zeros(n, ilm.HIT_DTYPE)
    hits["prim"] = prim
    hb = gpu_ctx.to_device(hits)
    ib = gpu_ctx.buffer(n * 4)
    c = gpu_ctx.compact_hits(hb, n, ib)
    want = np.nonzero(prim >= 0)[0]
    assert c == len(want)
    assert np.array_equal(ib.download(np.int32, c), want)


def test_refill_threshold_is_the_callers(ilm):
    """A threshold that the caller sets is that of every later launch but a
    frame's camera rays; the default lets a frame's launches with shadow
    segments wait for 28 idle lanes."""
    ctx = ilm.Context(0)
    assert ctx.trace_refill() == (24, 28)
    for lanes in (1, 4, 23, 25, 28, 61, 64):
        ctx.set_trace_refill(lanes)
        assert ctx.trace_refill() == (lanes, lanes)
    for lanes in (0, 65, -1):
        with pytest.raises(ilm.IlmError):
            ctx.set_trace_refill(lanes)
    assert ctx.trace_refill() == (64, 64)
    ctx.set_trace_refill(24)
    assert ctx.trace_refill() == (24, 28)
    ctx.close()


@pytest.mark.parametrize("caller", ["spill", "alloc", "trim"])
def test_kept_build_scratch_makes_room(caller, ilm):
    """A device build's scratch stays with the context: an allocation that
    finds the device full (the traversal's spill area, a buffer) takes it back
    and succeeds, and so can the program. It is about 300 bytes a triangle."""
    ctx = ilm.Context(0)
    ntri = 400000
    pos, idx = meshgen.random_triangles(ntri, seed=5, extent=2.0, size=0.02)
    m = ilm.Mesh(ctx, pos, idx)
    m.build(builder=ilm.ILM_BUILDER_LBVH)
    rays = meshgen.rays_toward(5000, pos, seed=2)
    rb, hb = ilm.rays_to_device(ctx, rays), ctx.buffer(len(rays) * 16)
    before = ctx.memory()[0]
    if caller == "trim":
        ctx.trim()
        ctx.trim()
    else:
        ctx.fail_allocations(0, 1)
    if caller == "alloc":
        ctx.buffer(1 << 20).free()
    m.trace_closest(rb, len(rays), hb)
    ctx.sync()
    ctx.fail_allocations()
    assert ctx.memory()[0] - before > 200 * ntri - (32 << 20)   # less the spill area
    a = hb.download(ilm.HIT_DTYPE, len(rays))
    m.build(builder=ilm.ILM_BUILDER_LBVH)
    m.trace_closest(rb, len(rays), hb)
    ctx.sync()
    b = hb.download(ilm.HIT_DTYPE, len(rays))
    assert (a["prim"] >= 0).mean() > 0.1 and np.array_equal(a.view(np.uint32), b.view(np.uint32))
    ctx.fail_allocations(0, 1000)
    with pytest.raises(ilm.IlmError):
        ctx.buffer(1 << 20)
    ctx.fail_allocations()
    ctx.buffer(1 << 20).free()
    m.close()
    ctx.close()


@pytest.mark.parametrize("instances", [False, True])
def test_short_launches_share_one_spill_area(instances, ilm):
    """Once one ray has been traced, launches of up to 256 rays for each
    workgroup of a short launch (2 per CU) allocate nothing: a launch captured
    in a graph keeps a valid spill area whatever short launches follow."""
    ctx = ilm.Context(0)
    pos, idx = meshgen.icosphere(3)
    m = ilm.Mesh(ctx, pos, idx)
    m.build()
    most = 2 * ctx.cu_count * 256
    rays = np.resize(meshgen.rays_toward(5000, pos, seed=9), (most, 8))
    rb, hb, ib = ilm.rays_to_device(ctx, rays), ctx.buffer(most * 16), ctx.buffer(most * 4)
    table = ilm.Instances(ctx, [m])
    table.set([(0, None, None, None)])
    run = (lambda n: table.trace_closest(rb, n, hb, ib)) if instances else (lambda n: m.trace_closest(rb, n, hb))
    run(1)
    ctx.fail_allocations(0, 1000)
    for n in (100, 250, 257, 2000, 8 * ctx.cu_count + 1, 50000, most):
        run(n)
    ctx.sync()
    ctx.fail_allocations()
    table.close()
    m.close()
    ctx.close()


@pytest.mark.parametrize("instances", [False, True])
def test_short_launch_without_memory_for_the_wide_grid(instances, ilm):
    """A short launch spread over the chip asks for a larger spill area than
    its rays need; refused that, it traces with as many workgroups as its rays
    fill, to the same hits, and fails only when that is refused too."""
    pos, idx = meshgen.icosphere(4)
    n = 3000
    rays = meshgen.rays_toward(n, pos, seed=8)
    hits = []
    for refused in (0, 1, 1000):
        ctx = ilm.Context(0)
        m = ilm.Mesh(ctx, pos, idx)
        m.build()
        rb, hb, ib = ilm.rays_to_device(ctx, rays), ctx.buffer(n * 16), ctx.buffer(n * 4)
        table = ilm.Instances(ctx, [m]) if instances else None
        if instances:
            table.set([(0, None, None, None)])
        run = (lambda: table.trace_closest(rb, n, hb, ib)) if instances else (lambda: m.trace_closest(rb, n, hb))
        ctx.fail_allocations(0, refused)
        if refused == 1000:
            with pytest.raises(ilm.IlmError):
                run()
            ctx.fail_allocations()
        run()
        ctx.sync()
        ctx.fail_allocations()
        hits.append(hb.download(ilm.HIT_DTYPE, n))
        if instances:
            table.close()
        m.close()
        ctx.close()
    assert (hits[0]["prim"] >= 0).mean() > 0.3
    for h in hits[1:]:
        assert np.array_equal(h.view(np.uint32), hits[0].view(np.uint32))


def test_threads_building_in_one_context(ilm):
    """Device builds of several threads in one context: one holds the kept
    scratch, the others take their own; every tree traces to its own hits."""
    import threading
    ctx = ilm.Context(0)
    ntri = (40000, 60001, 25000, 90000)
    meshes = [meshgen.random_triangles(n, seed=n, extent=2.0, size=0.03) for n in ntri]
    built, failed = {}, []

    def build(k):
        try:
            for _ in range(4):
                m = ilm.Mesh(ctx, *meshes[k])
                m.build(builder=ilm.ILM_BUILDER_LBVH)
                if k in built:
                    built[k].close()
                built[k] = m
        except Exception as e:  # noqa: BLE001 (reported by the test's own thread)
            failed.append(e)
    threads = [threading.Thread(target=build, args=(k,)) for k in range(len(meshes))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed, failed
    for k, (pos, idx) in enumerate(meshes):
        rays = meshgen.rays_toward(3000, pos, seed=k)
        rb, hb = ilm.rays_to_device(ctx, rays), ctx.buffer(len(rays) * 16)
        built[k].trace_closest(rb, len(rays), hb)
        ctx.sync()
        got = hb.download(ilm.HIT_DTYPE, len(rays))
        ref = ilm.Mesh(ctx, pos, idx)
        ref.build()
        ref.trace_closest(rb, len(rays), hb)
        ctx.sync()
        want = hb.download(ilm.HIT_DTYPE, len(rays))
        assert _compare_closest(got["prim"], got["t"], want["prim"], want["t"], f"threads {k}") >= 0.9999
        ref.close()
        built[k].close()
    ctx.close()
