"""Batched training of the denoiser: gradients at ragged sizes against the
float32 restatement of test_gpu_denoise.py, and a step on a batch against the
gradients of its images."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

from test_gpu_denoise import _rand_input, _torch_forward  # noqa: E402


@pytest.fixture(scope="module")
def dnmod():
    from mdwtracker_amd import denoise
    return denoise


# widths past one 32-column unit and one 64-pixel tile, heights that end inside
# an 8-row unit at every level, input widths of 8, 17 and 11 values
@pytest.mark.parametrize("channels,h,w", [(1, 36, 100), (10, 12, 68), (4, 44, 36)])
def test_gradient_of_pixels_at_the_edges(dnmod, channels, h, w):
    """The target is the prediction but at pixels on the edges of the image, of
    its row bands and of its column units, so the gradient comes from there
    alone. The bound is test_gradient_matches_torch_reference's, layer by layer."""
    print(f"[denoise] gradient {channels} channels {h} x {w}", flush=True)
    rng = np.random.default_rng(h * 1000 + w)
    dn = dnmod.Denoiser(w, h, channels=channels, seed=5)
    p = dn.get_params() + rng.normal(0, 0.02, dn.num_params()).astype(np.float32)
    dn.set_params(p)
    x = _rand_input(rng, h, w, channels)
    t, _ = dn.infer(x)
    y, layers = _torch_forward(p, x, channels)
    tr = y.detach().clone()
    for py in (0, 7, 8, h - 1):
        for px in (0, 31, 32, w - 1):
            e = rng.uniform(0.2, 0.6, 3).astype(np.float32)
            t[py, px] += e
            tr[py, px] += torch.tensor(e)
    g, loss = dn.gradient(x, t)
    ref = ((y - tr) ** 2).mean()
    ref.backward()
    assert abs(loss - float(ref.detach())) < 1e-2 * float(ref.detach())
    o = 0
    for i, (wt, b, _) in enumerate(layers):
        for r in (wt.grad.permute(2, 3, 0, 1).reshape(-1).numpy(), b.grad.numpy()):
            got = g[o:o + r.size]
            o += r.size
            cos = float(np.dot(got, r) / (np.linalg.norm(got) * np.linalg.norm(r) + 1e-30))
            rel = float(np.linalg.norm(got - r) / (np.linalg.norm(r) + 1e-30))
            assert cos > 0.999 and rel < 5e-2, (i, cos, rel)
    assert o == g.size
    dn.close()


# 5 images in one part; 1024 x 768 in two parts of one image each
@pytest.mark.parametrize("count,h,w", [(5, 36, 100), (2, 1024, 768)])
def test_batched_step_is_the_step_of_the_summed_gradients(dnmod, count, h, w):
    print(f"[denoise] batch of {count}, {h} x {w}", flush=True)
    rng = np.random.default_rng(count)
    xs = np.stack([_rand_input(rng, h, w) for _ in range(count)])
    ts = rng.uniform(0, 1, (count, h, w, 3)).astype(np.float32)
    wt = rng.uniform(0.5, 1.5, count).astype(np.float32)
    dn = dnmod.Denoiser(w, h, seed=5)
    p0 = dn.get_params()
    grads, losses = zip(*(dn.gradient(x, t) for x, t in zip(xs, ts)))
    g = sum(float(k) * a.astype(np.float64) for k, a in zip(wt, grads)) / count
    loss = dn.train_step(xs, ts, 1e-3, wt)
    p1 = dn.get_params()
    dn.close()
    # fp32 sums of at most 2^20 positive terms in another order
    assert abs(loss - np.mean(losses)) < 1e-4 * loss
    # Adam's first step is lr g / (|g| + 1e-8). The bf16 logit gradients carry the
    # weight before they are rounded (2^-8 relative), so compare where |g| is well
    # above its own rounding: there the step is lr within the sign and 1 %.
    big = np.abs(g) > 0.05 * np.abs(g).max()
    assert big.sum() > 100
    step = (p1 - p0)[big] / -1e-3
    np.testing.assert_allclose(step, np.sign(g[big]), atol=1e-2)
