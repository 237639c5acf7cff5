"""The GPU irradiance cache (ilm_ic_*) against the restatement in
oracle/icache.py and against closed forms.

- Octree and lookups: records inserted through the C ABI give the same tree
  (node count, children, per-node record lists) as the restatement, and GPU
  lookups equal the restatement's weighted means (float tolerance; a record
  whose weight is within rounding of 0 may flip).
- Records: in a closed box whose walls all emit Le with albedo rho, a small
  reflector in the middle receives Le from every direction plus what the
  walls reflect. A gather path (PathLi: next-event estimation at each of its
  RayDepth vertices, no emission) then has mean Le * sum_{k=1..D} rho^k, so
  every record's irradiance must be that number; its Ri must be the
  harmonic-mean hit distance, which the restatement's stratified cosine
  directions give by ray casting against the box.
- Images: the reflector's pixels are direct light rho_q * Le plus
  indirect_factor * rho_q * E, with the reference's 1/pi factor or 1.
"""
import numpy as np
import pytest

from oracle import icache as oic
from tests.test_gpu_pt import _closed_box

pytestmark = pytest.mark.gpu


def _room(ilm, ctx):
    from illuminaprt_amd import workloads as w
    pos, nrm, idx, tm, tl, mats, lights = w.box_room()
    m = ilm.Mesh(ctx, pos, idx)
    m.build()
    return m, ilm.Scene(ctx, m, nrm, tm, tl, mats, lights), pos


@pytest.mark.parametrize("variant", [0, 1])
def test_octree_and_lookups_match_restatement(gpu_ctx, ilm, variant):
    m, sc, pos = _room(ilm, gpu_ctx)
    ic = ilm.IrradianceCache(sc, cache_depth=8, error_threshold=0.5, ambient_resolution=0.01, ambient_multiplier=0.3,
                             variant=variant)
    info = ic.info()
    lo, hi, L = oic.root_cell(pos)
    assert np.array_equal(info["root"], np.concatenate([lo, hi]))
    assert info["rmin"] == np.float32(L * np.float32(0.01)) and info["rmax"] == np.float32(L * np.float32(0.3))
    rng = np.random.default_rng(7)
    n = 3000
    P = rng.random((n, 3)).astype(np.float32)
    N = rng.normal(size=(n, 3))
    N = (N / np.linalg.norm(N, axis=1, keepdims=True)).astype(np.float32)
    E = rng.random((n, 3)).astype(np.float32)
    Ri = (0.005 + 0.4 * rng.random(n) ** 3).astype(np.float32)
    ic.insert(np.concatenate([P, N, E, Ri[:, None]], axis=1))
    t = oic.Octree(lo, hi, 8, ["ward", "tabelion"][variant])
    rc = np.clip(Ri, info["rmin"], info["rmax"]).astype(np.float32)
    for i in range(n):
        t.insert(P[i], N[i], E[i], rc[i])
    info = ic.info()
    assert info["records"] == n and info["nodes"] == len(t.lo)
    assert info["refs"] == sum(len(r) for r in t.recs)
    for node in range(len(t.lo)):
        child, recs = ic.node(node)
        assert child == t.child[node] and recs.tolist() == t.recs[node], node
    recs = ic.records()
    np.testing.assert_array_equal(recs[:, 10], rc)
    # lookups at random points, half of them with a record's normal
    q = 20000
    qp = rng.random((q, 3)).astype(np.float32)
    k = rng.integers(n, size=q)
    qn = np.where(rng.random((q, 1)) < 0.5, N[k], rng.normal(size=(q, 3))).astype(np.float32)
    qn = (qn / np.linalg.norm(qn, axis=1, keepdims=True)).astype(np.float32)
    got = ic.lookup(np.concatenate([qp, qn], axis=1))
    agree = 0
    for i in range(q):
        e, den, _ = t.lookup(qp[i], qn[i], 0.5)
        ok = (den == 0 and got[i, 3] == 0) or (den > 0 and abs(got[i, 3] - den) <= 1e-4 * den + 1e-5 and
                                                np.allclose(got[i, :3], e, rtol=1e-4, atol=1e-6))
        agree += ok
    covered = float((got[:, 3] > 0).mean())
    print(f"[ic lookup] agreement {agree / q:.5f}, covered {covered:.3f}", flush=True)
    # Tabelion weights accept a record only within half its radius and ~6
    # degrees of its normal at this threshold, so fewer points are covered
    assert agree / q >= 0.999 and covered > (0.3 if variant == 0 else 0.1)
    ic.close()
    sc.close()
    m.close()


def _furnace_with_reflector(rho, le, rho_q, half=0.02):
    pos, nrm, idx, tm, tl, mats, lights = _closed_box(rho, le)
    # a small quad at the centre facing -z (the camera), material 1 (non-emissive)
    q = np.array([[0.5 - half, 0.5 - half, 0.5], [0.5 + half, 0.5 - half, 0.5], [0.5 + half, 0.5 + half, 0.5],
                  [0.5 - half, 0.5 + half, 0.5]], np.float32)
    b = len(pos)
    pos = np.concatenate([pos, q])
    nrm = np.concatenate([nrm, np.tile([[0, 0, -1]], (4, 1)).astype(np.float32)])
    # winding with cross(p1 - p0, p2 - p0) along -z
    idx = np.concatenate([idx, np.array([[b, b + 3, b + 2], [b, b + 2, b + 1]], np.int32)])
    tm = np.concatenate([tm, [1, 1]]).astype(np.int32)
    tl = np.concatenate([tl, [-1, -1]]).astype(np.int32)
    mats = np.concatenate([mats, np.array([[rho_q] * 3 + [0, 0, 0, 1, 0]], np.float32)])
    return pos, nrm, idx, tm, tl, mats, lights


def _cube_exit_distance(o, d):
    t = np.full(len(d), np.inf)
    for k in range(3):
        with np.errstate(divide="ignore", invalid="ignore"):
            tk = np.where(d[:, k] > 0, (1 - o[k]) / d[:, k], np.where(d[:, k] < 0, -o[k] / d[:, k], np.inf))
        t = np.minimum(t, tk)
    return t


@pytest.mark.parametrize("factor", [0.0, 1.0])
def test_records_and_image_in_furnace(gpu_ctx, ilm, factor):
    rho, le, rho_q, depth = 0.5, 1.0, 0.6, 6
    arr = _furnace_with_reflector(rho, le, rho_q)
    m = ilm.Mesh(gpu_ctx, arr[0], arr[2])
    m.build()
    sc = ilm.Scene(gpu_ctx, m, arr[1], *arr[3:])
    # every pixel of the first pass makes a record (stride 1): a few hundred
    # records of 512 gather paths each pin the record mean to ~0.2%
    ic = ilm.IrradianceCache(sc, ray_depth=depth, azimuth_strata=32, altitude_strata=16, error_threshold=0.3,
                             indirect_factor=factor, placement_stride=1)
    cam = ilm.Camera.make((0.5, 0.5, 0.1), (0.5, 0.5, 1.0), (0, 1, 0), 8.0, 1.0)  # the quad fills the middle
    W = H = 32
    acc = gpu_ctx.buffer(W * H * 24).zero()
    spp = 64
    st = ic.render(cam, W, H, spp, acc, seed=3)
    recs = ic.records()
    print(f"[ic furnace] {st} records {len(recs)}", flush=True)
    assert st["records_created"] == len(recs) > 0
    want_e = le * sum(rho ** k for k in range(1, depth + 1))
    e = recs[:, 6:9].mean()
    print(f"[ic furnace] record E {e:.5f} vs {want_e:.5f}; per-record spread {recs[:, 6:9].std():.4f}", flush=True)
    assert len(recs) > 200 and abs(e - want_e) < 0.01 * want_e
    # Ri: harmonic mean of the hit distances of cosine-distributed rays from
    # the quad's centre toward -z, by ray casting against the unit cube
    rng = np.random.default_rng(1)
    u, v = rng.random(400000), rng.random(400000)
    alt, az = rng.integers(16, size=u.shape), rng.integers(32, size=u.shape)
    dl = oic.cosine_stratified(u, v, alt, az, 16, 32)
    d = np.stack([dl[:, 0], dl[:, 1], -dl[:, 2]], axis=1)
    want_ri = 1.0 / np.mean(1.0 / _cube_exit_distance(np.array([0.5, 0.5, 0.5]), d))
    ri = np.mean(recs[:, 9])
    print(f"[ic furnace] Ri {ri:.4f} vs {want_ri:.4f}", flush=True)
    assert abs(ri - want_ri) < 0.05 * want_ri
    # the quad's pixels: direct rho_q Le plus factor * rho_q * E (factor 0 = 1/pi)
    img = acc.download(np.float64, W * H * 3).reshape(H, W, 3) / spp
    centre = img[12:20, 12:20].mean()
    f = factor if factor > 0 else 1 / np.pi
    want = rho_q * le + f * rho_q * want_e
    print(f"[ic furnace] quad pixels {centre:.5f} vs {want:.5f}", flush=True)
    assert abs(centre - want) < 0.015 * want
    # a second frame reuses the cache
    acc.zero()
    st2 = ic.render(cam, W, H, 1, acc, seed=4, spp_offset=1)
    assert st2["records_created"] <= st["records_created"] // 10
    ic.close()
    sc.close()
    m.close()
    acc.free()


@pytest.mark.parametrize("variant", [0, 1])
def test_room_image_converges_near_path_tracing(gpu_ctx, ilm, variant):
    """With the consistent indirect factor and a tight error threshold, the
    cache's image of the box room (closed scene front: camera rays that miss
    are excluded) stays within a modest relRMSE of a converged path-traced
    image: the cache's error is its interpolation bias, one bounce deep."""
    from illuminaprt_amd import workloads as w
    m, sc, pos = _room(ilm, gpu_ctx)
    W = H = 64
    cam = w.room_camera()
    acc = gpu_ctx.buffer(W * H * 24).zero()
    sc.render(cam, W, H, 1024, acc, seed=9, max_depth=6)
    ref = acc.download(np.float64, W * H * 3).reshape(H, W, 3) / 1024
    ic = ilm.IrradianceCache(sc, ray_depth=5, error_threshold=0.25, indirect_factor=1.0,
                             miss_radiance=(0.0, 0.0, 0.0), variant=variant)
    acc.zero()
    frames = 8
    for f in range(frames):
        ic.render(cam, W, H, 4, acc, seed=10 + f, spp_offset=4 * f)
    img = acc.download(np.float64, W * H * 3).reshape(H, W, 3) / (4 * frames)
    e = w.rel_rmse(img, ref)
    mean_ratio = img.mean() / ref.mean()
    print(f"[ic room v{variant}] relRMSE vs PT {e:.4f}, mean ratio {mean_ratio:.4f}, records {ic.info()['records']}",
          flush=True)
    assert e < 0.2 and abs(mean_ratio - 1) < 0.05
    ic.close()
    sc.close()
    m.close()
    acc.free()


@pytest.mark.parametrize("variant", [0, 1])
@pytest.mark.parametrize("count", [31, 32, 33, 64, 65, 129])
def test_lookups_at_list_lengths_around_the_masks(gpu_ctx, ilm, variant, count):
    """Lists just short of and past the length that gets cell masks, whole and
    part words, at thresholds below and above 1, with record normals and
    lookup normals longer than 1 (which reach further). The whole lists in 64
    bits give the sums; a weight w = 1 / x - 1 / threshold, x = d / RiClamp +
    1 - cos, is off by x's rounding (a few 2^-24 of its terms, each at most
    4 here) over x squared, plus its own, and a list's sum by its length
    times 2^-24."""
    m, sc, pos = _room(ilm, gpu_ctx)
    rng = np.random.default_rng(count)
    for threshold, scale in ((0.05, 1.0), (0.3, 1.0), (0.3, 1.5), (3.0, 1.0)):
        ic = ilm.IrradianceCache(sc, cache_depth=1, error_threshold=threshold, ambient_resolution=0.01,
                                 ambient_multiplier=10.0, variant=variant)
        # cache depth 1: every record lies in the lists of the root's children
        P = rng.random((count, 3)) * 0.4 + 0.05
        N = np.array([0, 1, 0]) + 0.1 * rng.normal(size=(count, 3))
        N *= scale / np.linalg.norm(N, axis=1, keepdims=True)
        R = np.concatenate([P, N, rng.random((count, 3)), 0.1 + 0.2 * rng.random((count, 1))], 1).astype(np.float32)
        ic.insert(R)
        lists = [ic.node(k)[1] for k in range(ic.info()["nodes"])]
        lo, hi = ic.info()["root"][:3], ic.info()["root"][3:]
        centre = lo + (hi - lo) * np.float32(0.5)
        q = 300
        qn = np.tile(np.array([0, 1.0, 0]), (q, 1))
        qn[::3] *= 2.0                             # beyond unit length: the whole list is walked
        Q = np.concatenate([rng.random((q, 3)) * 0.5, qn], 1).astype(np.float32)
        got = ic.lookup(Q).astype(np.float64)
        rc, Rd, Qd, inv = ic.records()[:, 10].astype(np.float64), R.astype(np.float64), Q.astype(np.float64), \
            float(np.float32(1) / np.float32(threshold))
        assert max(len(x) for x in lists) == count
        weighted = 0
        for i in range(q):
            b = Q[i, :3] > centre
            r = lists[1 + int(b[0]) + 2 * int(b[2]) + 4 * int(b[1])]
            d = np.linalg.norm(Rd[r, :3] - Qd[i, :3], axis=1) / rc[r]
            cos = Rd[r, 3:6] @ Qd[i, 3:]
            if variant == 0:
                x = d + 1 - cos
                w = np.where(cos > 0, 1 / x - inv, -1.0)
                off = 24 * 2.0 ** -24 / x ** 2 + 4 * 2.0 ** -24 * (np.abs(1 / x) + inv)
            else:
                w = 1 - inv * np.maximum(d, (1 - cos) * 9.0124)
                off = np.full(len(r), 48 * 2.0 ** -24 * (1 + inv))
            w0 = np.where(w > 0, w, 0)
            den = w0.sum()
            bound = off[w > -off].sum() + len(r) * 2.0 ** -23 * den
            assert abs(got[i, 3] - den) <= bound, (i, got[i, 3], den, bound)
            if den > 100 * bound:
                e = (w0[:, None] * Rd[r, 6:9]).sum(0) / den
                assert np.abs(got[i, :3] - e).max() <= 2 * bound / den + len(r) * 2.0 ** -23
                weighted += 1
        assert weighted > 20 or threshold < 0.1
        ic.close()
    sc.close()
    m.close()


@pytest.mark.parametrize("refused", range(6))
def test_lookups_after_an_allocation_was_refused(gpu_ctx, ilm, refused):
    """An insertion whose n-th device allocation (nodes, references, records,
    masks, their jobs; the sixth does not happen) is refused. Without masks
    the lists are walked whole, to the same sums bit for bit; without the
    others the insertion fails, lookups fail while memory is short, and the
    next one with memory sees every record."""
    m, sc, pos = _room(ilm, gpu_ctx)
    rng = np.random.default_rng(4)

    def records(n):
        N = np.array([0, 1, 0]) + 0.2 * rng.normal(size=(n, 3))
        N /= np.linalg.norm(N, axis=1, keepdims=True)
        return np.concatenate([rng.random((n, 3)), N, rng.random((n, 3)), 0.05 + 0.2 * rng.random((n, 1))],
                              1).astype(np.float32)
    first, second = records(50), records(4000)
    Q = np.concatenate([rng.random((2000, 3)), np.tile([0, 1.0, 0], (2000, 1))], 1).astype(np.float32)
    caches = [ilm.IrradianceCache(sc, cache_depth=4, error_threshold=0.3, ambient_resolution=0.01,
                                  ambient_multiplier=10.0) for _ in range(2)]
    for ic in caches:
        ic.insert(first)
    whole, short = caches
    whole.insert(second)
    want = whole.lookup(Q)
    assert (want[:, 3] > 0).mean() > 0.3
    points, out = gpu_ctx.to_device(Q), gpu_ctx.buffer(len(Q) * 16)
    lookup = lambda: ilm.load().ilm_ic_lookup(short.h, points.ptr, len(Q), out.ptr, None)
    try:
        if refused < 3:
            gpu_ctx.fail_allocations(refused, 1000)
            with pytest.raises(ilm.IlmError):
                short.insert(second)
            assert lookup() == -3  # ILM_ERR_NOMEM
            gpu_ctx.fail_allocations()
        else:
            gpu_ctx.fail_allocations(refused, 2)  # a context tries again after freeing what it keeps
            short.insert(second)
            gpu_ctx.fail_allocations()
        assert np.array_equal(short.lookup(Q).view(np.uint32), want.view(np.uint32))
        more = records(3)
        for ic in caches:
            ic.insert(more)
        assert np.array_equal(short.lookup(Q).view(np.uint32), whole.lookup(Q).view(np.uint32))
    finally:
        gpu_ctx.fail_allocations()
    for x in (points, out, *caches, sc, m):
        (x.free if hasattr(x, "free") else x.close)()


@pytest.mark.parametrize("variant", [0, 1])
@pytest.mark.parametrize("count", [1, 32, 33, 70])
def test_records_of_infinite_radius_keep_their_weight(gpu_ctx, ilm, variant, count):
    """An unbounded ambient_multiplier leaves a record whose gather rays all
    miss its infinite radius. Its distance then counts nothing and its weight
    is that of the normals alone, 1 / (1 - cos) - 1 / threshold (Ward) or 1 -
    9.0124 (1 - cos) / threshold: in 64 bits, off by the rounding of 1 - cos
    (four roundings of 2^-24) over its square, and of the sum."""
    m, sc, pos = _room(ilm, gpu_ctx)
    threshold = 0.5
    ic = ilm.IrradianceCache(sc, cache_depth=2, error_threshold=threshold, ambient_resolution=0.01,
                             ambient_multiplier=float("inf"), variant=variant)
    rng = np.random.default_rng(count)
    a = 0.15 + 0.2 * rng.random(count)                   # radians off the lookups' normal
    N = np.stack([np.sin(a), np.cos(a), np.zeros(count)], 1)
    R = np.concatenate([rng.random((count, 3)), N, rng.random((count, 3)), np.full((count, 1), np.inf)],
                       1).astype(np.float32)
    R[::5, 9] = 0.02                                     # and a few that reach no lookup
    if count == 1:
        R[0, 9] = np.inf
    ic.insert(R)
    far = np.isinf(ic.records()[:, 10])
    assert far.sum() >= max(1, 0.7 * count)
    q = 200
    Q = np.concatenate([np.full((q, 3), 0.98) + 0.01 * rng.random((q, 3)), np.tile([0, 1.0, 0], (q, 1))],
                       1).astype(np.float32)
    got = ic.lookup(Q).astype(np.float64)
    x = 1 - R[far, 4].astype(np.float64)
    w = 1 / x - 1 / threshold if variant == 0 else 1 - 9.0124 * x / threshold
    off = 4 * 2.0 ** -24 * ((1 / x ** 2 + 1 / x) if variant == 0 else np.full(len(x), 9.0124 / threshold + 1))
    w0 = np.maximum(w, 0)
    den, bound = w0.sum(), off.sum() + count * 2.0 ** -23 * w0.sum()
    assert den > 100 * bound
    clear = ~(np.linalg.norm(Q[:, None, :3] - R[None, ~far, :3], axis=2).min(axis=1, initial=9.0) < 0.02)
    assert clear.sum() > q / 2
    assert np.abs(got[clear, 3] - den).max() <= bound
    e = (w0[:, None] * R[far, 6:9]).sum(0) / den
    assert np.abs(got[clear, :3] - e).max() <= 2 * bound / den + count * 2.0 ** -23
    for x in (ic, sc, m):
        x.close()


@pytest.mark.parametrize("variant", [0, 1])
@pytest.mark.parametrize("threshold", [0.9, 0.95, 1.2, 1.25])
def test_lookups_on_both_sides_of_the_thresholds_of_the_walk(gpu_ctx, ilm, variant, threshold):
    """Lookups of points walk the lists by the records' reach, by the masks
    alone or whole, depending on the threshold. Lists of 33 and 150 records
    (with and without whole words of mask), against the sums in 64 bits: a
    weight 1 / x - 1 / threshold, x = d / RiClamp + 1 - cos, is off by x's
    rounding (24 roundings of its terms) over x squared and its own, Tabelion's
    by 48, and a list's sum by its length times 2^-23."""
    m, sc, pos = _room(ilm, gpu_ctx)
    rng = np.random.default_rng(12)
    inv = float(np.float32(1) / np.float32(threshold))
    for count in (33, 150):
        ic = ilm.IrradianceCache(sc, cache_depth=1, error_threshold=threshold, ambient_resolution=0.01,
                                 ambient_multiplier=10.0, variant=variant)
        N = np.array([0, 1, 0]) + 0.3 * rng.normal(size=(count, 3))
        N /= np.linalg.norm(N, axis=1, keepdims=True)
        R = np.concatenate([rng.random((count, 3)) * 0.4 + 0.05, N, rng.random((count, 3)),
                            0.02 + 0.1 * rng.random((count, 1))], 1).astype(np.float32)
        ic.insert(R)
        lists = [ic.node(k)[1] for k in range(ic.info()["nodes"])]
        lo, hi = ic.info()["root"][:3], ic.info()["root"][3:]
        centre = lo + (hi - lo) * np.float32(0.5)
        Q = np.concatenate([rng.random((400, 3)) * 0.5, np.tile([0, 1.0, 0], (400, 1))], 1).astype(np.float32)
        got = ic.lookup(Q).astype(np.float64)
        rc, Rd, Qd = ic.records()[:, 10].astype(np.float64), R.astype(np.float64), Q.astype(np.float64)
        weighted = 0
        for i in range(len(Q)):
            b = Q[i, :3] > centre
            r = lists[1 + int(b[0]) + 2 * int(b[2]) + 4 * int(b[1])]
            d = np.linalg.norm(Rd[r, :3] - Qd[i, :3], axis=1) / rc[r]
            cos = Rd[r, 3:6] @ Qd[i, 3:]
            if variant == 0:
                x = d + 1 - cos
                w = np.where(cos > 0, 1 / x - inv, -1.0)
                off = 24 * 2.0 ** -24 * np.maximum(d, 1) / x ** 2 + 4 * 2.0 ** -24 * (np.abs(1 / x) + inv)
            else:
                w = 1 - inv * np.maximum(d, (1 - cos) * 9.0124)
                off = 48 * 2.0 ** -24 * (1 + inv) * np.maximum(d, 1)
            w0 = np.where(w > 0, w, 0)
            den = w0.sum()
            bound = off[w > -off].sum() + len(r) * 2.0 ** -23 * den
            assert abs(got[i, 3] - den) <= bound, (count, i, got[i, 3], den, bound)
            if den > 100 * bound:
                e = (w0[:, None] * Rd[r, 6:9]).sum(0) / den
                assert np.abs(got[i, :3] - e).max() <= 2 * bound / den + len(r) * 2.0 ** -23
                weighted += 1
        assert weighted > 20
        ic.close()
    sc.close()
    m.close()


@pytest.mark.parametrize("variant", [0, 1])
@pytest.mark.parametrize("threshold", [0.3, 1.0, 3.0])
def test_frames_by_the_masks_equal_frames_over_whole_lists(gpu_ctx, ilm, variant, threshold):
    """Frames go by the masks at every threshold. A cache filled by one frame
    shows the same frame again; a second cache given the same records without
    memory for masks shows it over the whole lists: the same image bit for bit,
    and neither places a record, since every point is covered."""
    from illuminaprt_amd import workloads as w
    m, sc, pos = _room(ilm, gpu_ctx)
    cam = w.room_camera()
    width, height = 150, 90
    kw = dict(cache_depth=1, error_threshold=threshold, ambient_resolution=0.01, ambient_multiplier=0.08,
              indirect_factor=1.0, miss_radiance=(0.0, 0.0, 0.0), variant=variant, ray_depth=3)
    acc = gpu_ctx.buffer(width * height * 24)
    show = lambda ic: ic.render(cam, width, height, 1, acc, seed=5)
    masked, whole = ilm.IrradianceCache(sc, **kw), ilm.IrradianceCache(sc, **kw)
    acc.zero()
    show(masked)
    acc.zero()
    again = show(masked)
    want = acc.download(np.uint64, width * height * 3)
    assert again["records_created"] == 0 and again["lookups"] > 0
    lists = [len(masked.node(k)[1]) for k in range(masked.info()["nodes"])]
    assert max(lists) > 64   # lists of more than 32 records have masks
    gpu_ctx.fail_allocations(3, 2)   # nodes, references and records go ahead, masks do not
    whole.insert(masked.records()[:, :10])
    gpu_ctx.fail_allocations()
    acc.zero()
    stats = show(whole)
    assert stats["records_created"] == 0
    assert np.array_equal(acc.download(np.uint64, width * height * 3), want)
    for x in (masked, whole, sc, m):
        x.close()
    acc.free()
