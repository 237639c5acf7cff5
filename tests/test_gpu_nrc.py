"""GPU parity of the neural radiance cache kernels (bf16 MFMA forward,
backward, weight gradients and Adam) against the numpy oracle, through the
C ABI. Tolerances: the oracle rounds to bf16 at the same points as the GPU;
what remains is FP32 accumulation order (about 1e-3 relative per layer)."""
import numpy as np
import pytest

from oracle import nrc as onrc

pytestmark = pytest.mark.gpu

LO, HI = [-1.0, -1.0, -1.0], [1.0, 1.0, 1.0]


def _queries(n, seed):
    rng = np.random.default_rng(seed)
    q = np.zeros((n, 16), np.float32)
    q[:, 0:3] = rng.uniform(-1, 1, (n, 3))
    q[:, 3:7] = rng.uniform(0, 1, (n, 4))
    q[:, 7] = rng.uniform(0.1, 1, n)
    q[:, 8:14] = rng.uniform(0, 1, (n, 6))
    return q


def _rel(a, b):
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / max(np.linalg.norm(b), 1e-30))


def test_infer_matches_oracle(gpu_ctx, ilm):
    net = ilm.Nrc(gpu_ctx, LO, HI, seed=3)
    w = onrc.init_weights(5)
    net.set_weights(w)
    assert np.array_equal(net.weights(), w)
    n = 5003                                   # not a multiple of the 32-sample tile
    q = _queries(n, 1)
    qb = gpu_ctx.to_device(q)
    ob = gpu_ctx.buffer(n * 16)
    net.infer(qb, n, ob)
    gpu_ctx.sync()
    y = ob.download(np.float32, 4 * n).reshape(n, 4)[:, :3]
    x = onrc.encode(q, LO, HI)
    _, yb = onrc.forward(w, x, use_bf16=True)
    _, yf = onrc.forward(w, x, use_bf16=False)
    e_b, e_f = _rel(y, yb[:, :3]), _rel(y, yf[:, :3])
    print(f"[nrc infer] rel err vs bf16 oracle {e_b:.2e}, vs fp64 oracle {e_f:.2e}")
    assert e_b < 5e-3 and e_f < 3e-2
    net.close()


def test_gradients_and_adam_match_oracle(gpu_ctx, ilm):
    net = ilm.Nrc(gpu_ctx, LO, HI, lr=1e-3)
    w = onrc.init_weights(7)
    net.set_weights(w)
    n = 3001
    q = _queries(n, 2)
    rng = np.random.default_rng(4)
    t = np.zeros((n, 4), np.float32)
    t[:, :3] = rng.uniform(0, 2, (n, 3))
    t[:, 3] = 1.0
    qb, tb = gpu_ctx.to_device(q), gpu_ctx.to_device(t)
    lb = gpu_ctx.buffer(n * 4)
    net.train_step(qb, tb, n, lb)
    gpu_ctx.sync()
    g = net.gradients().astype(np.float64)
    w1 = net.weights().astype(np.float64)
    x = onrc.encode(q, LO, HI)
    loss, go = onrc.loss_grad(w, x, t, use_bf16=True)
    gl = lb.download(np.float32, n)
    print(f"[nrc grad] loss gpu {gl.sum() / (3 * n):.6f} oracle {loss:.6f}")
    assert abs(gl.sum() / (3 * n) - loss) < 1e-3 * loss
    off = 0
    for k, (o, i) in enumerate(onrc.SHAPES):
        s = slice(off, off + o * i)
        e = _rel(g[s], go[s])
        print(f"[nrc grad] layer {k} rel err {e:.2e} |g| {np.linalg.norm(go[s]):.3e}")
        assert e < 2e-2
        off += o * i
    # padding stays exactly zero
    ws = onrc.split(g)
    assert (ws[0][:, 83:] == 0).all() and (ws[5][3:, :] == 0).all()
    # Adam step 1 from the GPU's own gradient
    wa, _, _ = onrc.adam(w, g, 0, 0, 1, lr=1e-3, b1=0.9, b2=0.99, eps=1e-8)
    assert np.abs(w1 - wa).max() < 1e-6
    net.close()


@pytest.mark.parametrize("n", [1, 15, 17, 127, 128, 129, 1000, 32769])
def test_gradients_at_sample_counts_around_the_workgroups(gpu_ctx, ilm, n):
    """Part of a wave's 16 samples, part of a workgroup's 128, one and two
    rounds of workgroups, weights of 0 for some samples.

    Against the oracle: inputs that differ by a rounding (the encoding's sines)
    switch a hidden unit whose sum is within it of 0 on or off, in about one
    sample of a hundred; one unit of 64 in one sample of n is 1 / sqrt(64 n)
    of a layer's gradient norm (contributions of random signs); four such and
    the 2e-2 of many samples are allowed.

    Against itself: the samples moved behind as many of weight 0 (other lanes,
    waves and workgroups, twice the count: every gradient exactly half) give
    the same gradient up to the order of the sums, 1e-5."""
    net = ilm.Nrc(gpu_ctx, LO, HI, lr=1e-3)
    w = onrc.init_weights(9)
    net.set_weights(w)
    q = _queries(n, n)
    rng = np.random.default_rng(n + 1)
    t = np.zeros((n, 4), np.float32)
    t[:, :3] = rng.uniform(0, 2, (n, 3))
    t[:, 3] = rng.integers(0, 2, n) if n > 1 else 1
    qb, tb, lb = gpu_ctx.to_device(q), gpu_ctx.to_device(t), gpu_ctx.buffer(n * 4)
    net.train_step(qb, tb, n, lb)
    gpu_ctx.sync()
    g = net.gradients().astype(np.float64)
    loss, go = onrc.loss_grad(w, onrc.encode(q, LO, HI), t, weight=t[:, 3], use_bf16=True)
    gl = lb.download(np.float32, n)
    assert abs(gl.sum() / (3 * n) - loss) <= 2e-3 * loss
    off = 0
    for k, (o, i) in enumerate(onrc.SHAPES):
        s = slice(off, off + o * i)
        assert _rel(g[s], go[s]) < 2e-2 + 4 / np.sqrt(64 * n), k
        off += o * i
    q2, t2 = gpu_ctx.to_device(np.concatenate([q, q])), gpu_ctx.to_device(np.concatenate([t * [1, 1, 1, 0], t]).astype(np.float32))
    net.set_weights(w)
    net.train_step(q2, t2, 2 * n)
    gpu_ctx.sync()
    assert _rel(2 * net.gradients().astype(np.float64), g) < 1e-5
    for x in (qb, tb, lb, q2, t2):
        x.free()
    net.close()


def test_training_fits_a_smooth_field(gpu_ctx, ilm):
    """Online training on a fixed synthetic radiance field lowers the loss and
    generalises to held-out queries."""
    def field(q):
        p = q[:, 0:3]
        r = 0.6 + 0.3 * np.sin(2 * p[:, 0]) * np.cos(3 * p[:, 1]) + 0.2 * q[:, 8]
        gch = 0.4 + 0.3 * np.cos(2 * p[:, 2] + p[:, 0]) * q[:, 6]
        b = 0.2 + 0.15 * (p[:, 1] > 0) + 0.1 * q[:, 9]
        t = np.stack([r, gch, b, np.ones(len(q))], axis=1).astype(np.float32)
        return t

    net = ilm.Nrc(gpu_ctx, LO, HI, lr=1e-2, seed=11)
    n = 16384
    losses = []
    lb = gpu_ctx.buffer(n * 4)
    for step in range(300):
        q = _queries(n, 100 + step)
        qb, tb = gpu_ctx.to_device(q), gpu_ctx.to_device(field(q))
        net.train_step(qb, tb, n, lb)
        if step % 50 == 0 or step == 299:
            gpu_ctx.sync()
            losses.append(float(lb.download(np.float32, n).mean() / 3))
        qb.free()
        tb.free()
    q = _queries(4096, 99999)
    qb = gpu_ctx.to_device(q)
    ob = gpu_ctx.buffer(4096 * 16)
    net.infer(qb, 4096, ob)
    gpu_ctx.sync()
    y = ob.download(np.float32, 4 * 4096).reshape(-1, 4)[:, :3]
    t = field(q)[:, :3]
    err = float(np.sqrt(np.mean((y - t) ** 2)) / np.sqrt(np.mean(t ** 2)))
    print(f"[nrc fit] losses {losses} held-out rel RMS {err:.4f}")
    assert losses[-1] < losses[0] / 10
    assert err < 0.1
    net.close()


def test_trained_cache_beats_plain_pt_at_equal_time(gpu_ctx, ilm):
    """What the learned part gains: on the radiance-cache workload at
    1920 x 1080, cache rendering (trained online from a cold start) reaches a
    lower relRMSE than plain path tracing given the same GPU time, and the
    same renderer with training switched off is far worse (the untrained
    network's bias). Errors are against a 256-spp plain render whose own
    noise, estimated from two independent halves, is removed."""
    from illuminaprt_amd import workloads as w
    W, H, depth = 1920, 1080, 10
    pos, nrm, idx, tm, tl, mats, lights = w.cache_scene()
    m = ilm.Mesh(gpu_ctx, pos, idx)
    m.build()
    sc = ilm.Scene(gpu_ctx, m, nrm, tm, tl, mats, lights)
    cam = w.cache_camera(W / H)
    n3 = W * H * 3
    buf = gpu_ctx.buffer(n3 * 8)

    def mean_of(spp, seed, chunk=32):
        buf.zero()
        ms = 0.0
        for k in range(0, spp, chunk):
            ms += sc.render(cam, W, H, min(chunk, spp - k), buf, max_depth=depth, seed=seed, spp_offset=k)["ms"]
        return buf.download(np.float64, n3).reshape(H, W, 3) / spp, ms

    r1, _ = mean_of(128, 501)
    r2, _ = mean_of(128, 502)
    ref = 0.5 * (r1 + r2)
    noise2 = float(np.mean((r1 - r2) ** 2 / (ref ** 2 + 0.01)) / 4.0)

    def err(img):
        return float(np.sqrt(max(float(np.mean((img - ref) ** 2 / (ref ** 2 + 0.01))) - noise2, 0.0)))

    def cache_run(train_steps, frames=56, skip=16):
        net = ilm.Nrc(gpu_ctx, *w.CACHE_BOUNDS, lr=1e-2, seed=5)
        buf.zero()
        ms = 0.0
        for f in range(frames):
            st = sc.render_nrc(net, cam, W, H, 1, buf if f >= skip else None, seed=7000 + f, prefix_depth=2,
                               suffix_depth=depth - 2, train_fraction=1 / 16, train_batch=65536,
                               train_steps=train_steps)
            ms += st["ms"]
        net.close()
        return err(buf.download(np.float64, n3).reshape(H, W, 3) / (frames - skip)), ms

    e_nrc, t_nrc = cache_run(1)
    e_off, _ = cache_run(0)
    # plain PT given the cache's time
    spp_per_ms = 1.0 / (mean_of(4, 900)[1] / 4)
    spp = max(1, int(t_nrc * spp_per_ms))
    e_plain = err(mean_of(spp, 901)[0])
    print(f"[cache gain] ref noise {np.sqrt(noise2):.4f}; cache {e_nrc:.4f} in {t_nrc:.0f} ms; "
          f"plain {e_plain:.4f} at {spp} spp (same time); cache untrained {e_off:.4f}", flush=True)
    assert e_nrc < 0.85 * e_plain
    assert e_off > 2.0 * e_nrc
    buf.free()
    sc.close()
    m.close()
