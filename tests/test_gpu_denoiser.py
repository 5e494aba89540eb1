"""HIP denoiser (BF16 MFMA convolutions, FP32 accumulation) against the
float64 CPU oracle, and what training it on renders buys.

Bars: forward prediction (log space) within 3 % relative L2 of the oracle
run on the same BF16-rounded weights; loss within 2 %; gradient cosine
similarity >= 0.98 and relative L2 error <= 0.15 (BF16 activations and
operands); the film path equals the host path bit for bit; after training
on renders, the denoised 4-spp image has lower relMSE against a 1024-spp
render than the 4-spp input on held-out views."""
import ctypes as C
import os

import numpy as np
import pytest

import asuna_amd as A
from oracle import unet_ref as U

pytestmark = pytest.mark.gpu


def log(*a):
    print(*a, flush=True)


def bf16(x):
    """Round float32 values to BF16 (nearest even) and back."""
    u = np.ascontiguousarray(x, np.float32).view(np.uint32).astype(np.uint64)
    u = ((u + 0x7FFF + ((u >> 16) & 1)) >> 16) << 16
    return u.astype(np.uint32).view(np.float32)


def _raw(rng, n, h, w):
    rad = np.exp(rng.normal(-1.0, 1.0, size=(n, h, w, 3))).astype(np.float32)
    alb = rng.uniform(0, 1, size=(n, h, w, 3)).astype(np.float32)
    nrm = rng.normal(size=(n, h, w, 3)).astype(np.float32)
    nrm /= np.linalg.norm(nrm, axis=-1, keepdims=True)
    dep = rng.uniform(0.5, 5, size=(n, h, w, 1)).astype(np.float32)
    return np.concatenate([rad, alb, nrm, dep], -1)


def _features64(raw):
    return bf16(U.features(raw[..., :3], raw[..., 3:6], raw[..., 6:9], raw[..., 9]).astype(np.float32)).astype(np.float64)


def test_forward_matches_oracle():
    d = A.Denoiser(0, seed=7)
    assert d.num_params() == U.num_params()
    theta = d.get_params()
    rng = np.random.default_rng(3)
    raw = _raw(rng, 1, 32, 48)
    out = d.forward(raw)
    ref = U.forward(bf16(theta).astype(np.float64), _features64(raw))
    got = np.log1p(out.astype(np.float64))
    err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
    log(f"forward: relative L2 error {err:.4f}, |ref| mean {np.abs(ref).mean():.3f}")
    assert err <= 0.03
    d.close()


def test_gradient_matches_oracle():
    d = A.Denoiser(0, seed=11)
    theta = d.get_params()
    rng = np.random.default_rng(4)
    raw = _raw(rng, 2, 32, 32)
    target = np.exp(rng.normal(-1.0, 1.0, size=(2, 32, 32, 3))).astype(np.float32)
    loss, g = d.gradient(raw, target)
    rl, rg = U.loss_and_grad(bf16(theta).astype(np.float64), _features64(raw), np.log1p(target.astype(np.float64)))
    cos = float(g @ rg / (np.linalg.norm(g) * np.linalg.norm(rg)))
    rel = float(np.linalg.norm(g - rg) / np.linalg.norm(rg))
    log(f"gradient: loss {loss:.5f} vs {rl:.5f}, cosine {cos:.5f}, relative L2 {rel:.4f}")
    assert abs(loss - rl) <= 0.02 * rl
    assert cos >= 0.98 and rel <= 0.15
    # per-layer: the biggest layers carry the signal of every block of kernels
    k = 0
    for name, a, b, o, relu in U.layer_shapes():
        n = 9 * (a + b) * o + o
        gl, rl_ = g[k:k + n], rg[k:k + n]
        c = float(gl @ rl_ / (np.linalg.norm(gl) * np.linalg.norm(rl_) + 1e-30))
        assert c >= 0.95, (name, c)
        k += n
    d.close()


def _render_set(r, s, cams, pc, w, h, spp, chans):
    xs, ys = [], []
    for cam in cams:
        r.set_film(w, h)
        r.render(cam, pc, 0, spp)
        rad = r.read(0)[..., :3]
        feats = [rad]
        for ch, k in chans:
            img = r.read(ch + 1)
            feats.append(img[..., :k])
        xs.append(np.concatenate(feats, -1))
    return np.stack(xs)


def test_training_on_renders_reduces_relmse(spheres_small):
    s = A.HostScene(spheres_small)
    st = s.state
    _, pc = s.shot(0)
    chans = [(pc.diffuseOutChannel, 3), (pc.normalOutChannel, 3), (st.depth_out_channel, 1)]
    assert min(c for c, _ in chans) >= 0
    r = A.Renderer(0)
    r.upload(s)
    r.build()
    rng = np.random.default_rng(9)
    w = h = 96
    cams = []
    for _ in range(28):
        eye = rng.normal(size=3)
        eye = eye / np.linalg.norm(eye) * rng.uniform(1.5, 3.5)
        eye[1] = abs(eye[1]) + 0.3
        cams.append(A.camera_lookat(w, h, float(rng.uniform(35, 75)), tuple(eye), (0.0, 0.3, 0.0)))
    noisy, ref = [], []
    for cam in cams:
        r.set_film(w, h)
        r.render(cam, pc, 0, 4, depth_channel=st.depth_out_channel)
        x = [r.read(0)[..., :3], r.read(pc.diffuseOutChannel + 1)[..., :3], r.read(pc.normalOutChannel + 1)[..., :3],
             r.read(st.depth_out_channel + 1)[..., :1]]
        noisy.append(np.concatenate(x, -1))
        r.set_film(w, h)
        r.render(cam, pc, 0, 1024)
        ref.append(r.read(0)[..., :3])
    r.close()
    noisy, ref = np.stack(noisy), np.stack(ref)
    train_x, train_y, test_x, test_y = noisy[:24], ref[:24], noisy[24:], ref[24:]

    def relmse(a, b):
        return float(np.mean((a - b) ** 2 / (b ** 2 + 1e-2)))

    d = A.Denoiser(0, seed=5)
    losses = []
    for it in range(400):
        idx = rng.choice(24, 8, replace=False)
        oy, ox = rng.integers(0, h - 64 + 1, 2)
        xb = train_x[idx, oy:oy + 64, ox:ox + 64]
        yb = train_y[idx, oy:oy + 64, ox:ox + 64]
        if it % 2:
            xb, yb = xb[:, :, ::-1], yb[:, :, ::-1]
        losses.append(d.train_step(xb, yb, lr=2e-3 if it < 300 else 5e-4))
    den = d.forward(test_x)
    before, after = relmse(test_x[..., :3], test_y), relmse(den, test_y)
    log(f"training: loss {np.mean(losses[:20]):.4f} -> {np.mean(losses[-20:]):.4f}; held-out relMSE "
        f"4 spp {before:.4f} -> denoised {after:.4f}")
    assert np.mean(losses[-20:]) < np.mean(losses[:20])
    assert after < 0.8 * before
    d.close()


def test_film_path_equals_host_path(spheres_small):
    s = A.HostScene(spheres_small)
    st = s.state
    cam, pc = s.shot(0)
    w, h = s.film
    r = A.Renderer(0)
    r.upload(s)
    r.build()
    r.set_film(w, h)
    r.render(cam, pc, 0, 4, depth_channel=st.depth_out_channel)
    planes = [r.read(0)[..., :3], r.read(pc.diffuseOutChannel + 1)[..., :3], r.read(pc.normalOutChannel + 1)[..., :3],
              r.read(st.depth_out_channel + 1)[..., :1]]
    d = A.Denoiser(0, seed=2)
    out_img = 7
    ms = d.denoise_film(r, pc.diffuseOutChannel, pc.normalOutChannel, st.depth_out_channel, out_img)
    film = r.read(out_img)
    hp, wp = (h + 15) // 16 * 16, (w + 15) // 16 * 16
    x = np.zeros((1, hp, wp, 10), np.float32)
    x[0, :h, :w] = np.concatenate(planes, -1)
    host = d.forward(x)[0, :h, :w]
    log(f"film denoise {w}x{h}: {ms:.2f} ms")
    np.testing.assert_array_equal(film[..., :3], np.maximum(host, 0.0))
    assert (film[..., 3] == 1).all()
    d.close()
    r.close()


def test_film_1080p_workload(tmp_path):
    """Inference at the workload's size: the 1920x1080 procedural scene
    (5.24M triangles) rendered at 4 spp and denoised in HBM.  The film path
    equals the host path on the whole padded 1088x1920 frame bit for bit,
    and on four 128x128 crops of the same input planes the network's
    prediction is within the forward bar of the float64 oracle."""
    s = A.HostScene(A.generate_scene(1, str(tmp_path / "c2")))
    st = s.state
    cam, pc = s.shot(0)
    w, h = s.film
    assert (w, h) == (1920, 1080)
    r = A.Renderer(0)
    r.upload(s)
    r.build()
    r.set_film(w, h)
    r.render(cam, pc, 0, 4, depth_channel=st.depth_out_channel)
    planes = np.concatenate([r.read(0)[..., :3], r.read(pc.diffuseOutChannel + 1)[..., :3],
                             r.read(pc.normalOutChannel + 1)[..., :3], r.read(st.depth_out_channel + 1)[..., :1]], -1)
    d = A.Denoiser(0, seed=13)
    d.denoise_film(r, pc.diffuseOutChannel, pc.normalOutChannel, st.depth_out_channel, 7)  # warm
    ms = d.denoise_film(r, pc.diffuseOutChannel, pc.normalOutChannel, st.depth_out_channel, 7)
    film = r.read(7)
    r.close()
    x = np.zeros((1, 1088, 1920, 10), np.float32)
    x[0, :h, :w] = planes
    host = d.forward(x)[0, :h, :w]
    log(f"1080p film denoise: {ms:.2f} ms ({181_000 * 1920 * 1088 / (ms * 1e-3) / 1e12:.1f} TFLOP/s)")
    np.testing.assert_array_equal(film[..., :3], np.maximum(host, 0.0))
    theta = d.get_params()
    crops = np.stack([planes[y:y + 128, xo:xo + 128] for xo, y in ((0, 0), (896, 464), (1792, 952), (416, 208))])
    out = d.forward(crops)
    ref = U.forward(bf16(theta).astype(np.float64), _features64(crops))
    got = np.log1p(out.astype(np.float64))
    err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
    log(f"1080p crops forward: relative L2 error {err:.4f}")
    assert err <= 0.03
    d.close()


def test_gradients_and_training_are_reproducible():
    """The weight and bias gradients are summed in a fixed order (per-split
    partial sums added in split order), so the same batch gives the same
    gradient bit for bit, and two denoisers from one seed trained on the
    same batches end with identical parameters."""
    rng = np.random.default_rng(21)
    raw = _raw(rng, 4, 64, 64)
    target = np.exp(rng.normal(-1.0, 1.0, size=(4, 64, 64, 3))).astype(np.float32)
    d = A.Denoiser(0, seed=17)
    l1, g1 = d.gradient(raw, target)
    l2, g2 = d.gradient(raw, target)
    assert l1 == l2
    np.testing.assert_array_equal(g1, g2)
    d2 = A.Denoiser(0, seed=17)
    for it in range(4):
        xb, yb = raw[it % 2::2], target[it % 2::2]
        assert d.train_step(xb, yb, lr=1e-3) == d2.train_step(xb, yb, lr=1e-3)
    np.testing.assert_array_equal(d.get_params(), d2.get_params())
    d.close()
    d2.close()


@pytest.mark.parametrize("n,h,w", [(1, 16, 16), (3, 16, 48), (2, 48, 80), (1, 32, 336), (1, 272, 16), (5, 64, 64)])
def test_tile_edges_match_oracle(n, h, w):
    """Forward and gradient where tiles are cut: levels of one to a few
    pixels, widths of 8, 16 and 32-column tiles with remainders, one image and
    odd batches.  Bars: BF16 operands (2^-9 each) through 19 layers measure
    0.005 in the prediction and 0.005 - 0.01 in the gradient; four times that."""
    d = A.Denoiser(0, seed=23)
    theta = bf16(d.get_params()).astype(np.float64)
    rng = np.random.default_rng(n * 1000 + h + w)
    raw = _raw(rng, n, h, w)
    target = np.exp(rng.normal(-1.0, 1.0, size=(n, h, w, 3))).astype(np.float32)
    x = _features64(raw)
    ref = U.forward(theta, x)
    got = np.log1p(d.forward(raw).astype(np.float64))
    ferr = np.linalg.norm(got - ref) / np.linalg.norm(ref)
    loss, g = d.gradient(raw, target)
    rl, rg = U.loss_and_grad(theta, x, np.log1p(target.astype(np.float64)))
    gerr = np.linalg.norm(g - rg) / np.linalg.norm(rg)
    log(f"{n}x{h}x{w}: forward {ferr:.4f}, gradient {gerr:.4f}, loss {loss:.5f} vs {rl:.5f}")
    assert ferr <= 0.02 and gerr <= 0.04 and abs(loss - rl) <= 0.01 * rl
    # Biases, summed apart from the weights.  A bias gradient is a sum over its level's pixels, and a
    # pre-activation that BF16 rounds to the other side of zero drops or adds a whole pixel of a channel:
    # of a level's N h w co units about half are on, so four such flips are sqrt(4 / (units / 2)) of the
    # layer's bias gradient (0.14 on the 2 x 2 pixels x 96 channels of a 16 x 16 image), on top of the
    # 0.04 above.
    k = 0
    levels = [0, 0, 1, 1, 2, 2, 3, 3, 4, 4, 3, 3, 2, 2, 1, 1, 0, 0, 0]
    for lv, (name, a, b, o, relu) in zip(levels, U.layer_shapes()):
        k += 9 * (a + b) * o
        e = np.linalg.norm(g[k:k + o] - rg[k:k + o]) / (np.linalg.norm(rg[k:k + o]) + 1e-12)
        units = n * (h >> lv) * (w >> lv) * o
        assert e <= 0.04 + np.sqrt(8.0 / units), (name, e)
        k += o
    d.close()


def test_large_batch_equals_its_images():
    """A batch large enough for the large-tile kernels (0.5 M pixels) against
    its images one by one, which run on the small-tile ones: only the order of
    the FP32 sums differs, then the BF16 roundings it turns over, which travel
    through 19 layers (0.0035 in the prediction; bar 0.01), and the batch gradient is
    the images' mean."""
    n, h, w = 8, 256, 256
    d = A.Denoiser(0, seed=29)
    rng = np.random.default_rng(31)
    raw = _raw(rng, n, h, w)
    target = np.exp(rng.normal(-1.0, 1.0, size=(n, h, w, 3))).astype(np.float32)
    out = np.log1p(d.forward(raw))
    one = np.log1p(np.concatenate([d.forward(raw[i:i + 1]) for i in range(n)]))
    ferr = np.linalg.norm(out - one) / np.linalg.norm(one)
    loss, g = d.gradient(raw, target)
    parts = [d.gradient(raw[i:i + 1], target[i:i + 1]) for i in range(n)]
    mean = np.mean([p[1].astype(np.float64) for p in parts], 0)
    gerr = np.linalg.norm(g - mean) / np.linalg.norm(mean)
    log(f"batch of {n}: forward {ferr:.5f}, gradient {gerr:.5f}")
    assert ferr <= 0.01 and gerr <= 0.01
    assert abs(loss - np.mean([p[0] for p in parts])) <= 1e-4 * loss
    d.close()


def test_features_of_any_magnitude_reach_the_network():
    """Weights that hand the radiance features through every full-resolution
    layer unchanged: the output is expm1 of the BF16 rounding of log(1 + x), for x
    from 1e-36 to the largest finite number, in both feature kernels.  log(1 + x) is
    within 0.54 units of its last place, which rounds to the other BF16 neighbour
    for at most 2 x 0.54 / 2^16 of the values; bar 3 times that."""
    theta = np.zeros(U.num_params(), np.float32)
    k = 0
    for name, a, b, o, relu in U.layer_shapes():
        n = 9 * (a + b) * o
        if name in ("enc0a", "enc0b", "dec0a", "dec0b", "out"):
            W = theta[k:k + n].reshape(9, o, a + b)
            for c in range(3):
                W[4, c, (a if name == "dec0a" else 0) + c] = 1.0  # dec0a: from the skip tensor
        k += n + o
    d = A.Denoiser(0)
    d.set_params(theta)
    h = w = 256
    x = np.zeros((1, h, w, 10), np.float32)
    x[..., :3] = np.geomspace(1e-36, np.finfo(np.float32).max, 3 * h * w).astype(np.float32).reshape(1, h, w, 3)
    x[0, 0, 0, :3] = (0.0, 3.0e38, np.finfo(np.float32).max)
    out = d.forward(x)
    got = bf16(np.log1p(out.astype(np.float64)).astype(np.float32))[0]
    want = bf16(np.log1p(x[0, ..., :3].astype(np.float64)).astype(np.float32))
    assert np.isfinite(out).all()
    differ = got != want
    log(f"features: {int(differ.sum())} of {differ.size} round to the other BF16 neighbour")
    assert differ.mean() <= 3 * 2 * 0.54 / 2 ** 16
    np.testing.assert_allclose(got, want, rtol=2.0 ** -7)
    # and from a film's planes
    r = A.Renderer(0)
    r.set_film(w, h)
    rad = np.concatenate([x[0, ..., :3], np.ones((h, w, 1), np.float32)], -1)
    src, dst = r.output_device_ptr(0), r.output_device_ptr(7)
    assert C.CDLL("libamdhip64.so").hipMemcpy(C.c_void_p(src), C.c_void_p(rad.ctypes.data), C.c_size_t(rad.nbytes), 1) == 0
    d._check(A.lib().ash_denoise_planes(d._d, src, None, None, None, w, h, dst, C.byref(C.c_double())), "denoise_planes")
    np.testing.assert_array_equal(r.read(7)[..., :3], out[0])
    r.close()
    d.close()


@pytest.mark.parametrize("n,h,w", [(8, 272, 144), (12, 208, 176)])
def test_cut_tiles_of_large_batches_equal_their_images(n, h, w):
    """Batches whose two finest levels run on the 16-row tiles (16 x 32 pixels,
    and 16 x 16 by two output groups) and the next on 8 x 32, with remainders in
    both directions, against their images one by one, which run on the small
    tiles that are checked against the oracle.  Bars as for the large batch; the
    biases, summed tile by tile in the convolutions, per layer: 0.01, and two
    pre-activations of a level's n h w co units rounded to the other side of zero."""
    d = A.Denoiser(0, seed=37)
    rng = np.random.default_rng(n + h + w)
    raw = _raw(rng, n, h, w)
    target = np.exp(rng.normal(-1.0, 1.0, size=(n, h, w, 3))).astype(np.float32)
    out = np.log1p(d.forward(raw))
    one = np.log1p(np.concatenate([d.forward(raw[i:i + 1]) for i in range(n)]))
    ferr = np.linalg.norm(out - one) / np.linalg.norm(one)
    worst = max(np.linalg.norm(out[i] - one[i]) / np.linalg.norm(one[i]) for i in range(n))
    edge = np.linalg.norm(out[:, -16:, -32:] - one[:, -16:, -32:]) / np.linalg.norm(one[:, -16:, -32:])
    loss, g = d.gradient(raw, target)
    parts = [d.gradient(raw[i:i + 1], target[i:i + 1]) for i in range(n)]
    mean = np.mean([p[1].astype(np.float64) for p in parts], 0)
    gerr = np.linalg.norm(g - mean) / np.linalg.norm(mean)
    log(f"{n} x {h} x {w}: forward {ferr:.5f}, worst image {worst:.5f}, last corner {edge:.5f}, gradient {gerr:.5f}")
    assert ferr <= 0.01 and worst <= 0.01 and edge <= 0.01 and gerr <= 0.01
    assert abs(loss - np.mean([p[0] for p in parts])) <= 1e-4 * loss
    k = 0
    levels = [0, 0, 1, 1, 2, 2, 3, 3, 4, 4, 3, 3, 2, 2, 1, 1, 0, 0, 0]
    for lv, (name, a, b, o, relu) in zip(levels, U.layer_shapes()):
        m = 9 * (a + b) * o
        for what, s in (("weights", slice(k, k + m)), ("biases", slice(k + m, k + m + o))):
            e = np.linalg.norm(g[s] - mean[s]) / np.linalg.norm(mean[s])
            log(f"  {name} {what}: {e:.5f}")
            assert e <= 0.01 + np.sqrt(8.0 / (n * (h >> lv) * (w >> lv) * o)), (name, what, e)
        k += m + o
    d.close()
