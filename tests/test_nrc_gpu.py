"""GPU tests of the radiance cache's kernels (metal-vibe-tracer_amd/csrc/nrc.hip) against the FP64
oracle (oracle/nrc.py): MFMA forward outputs, the fused backward's gradients (the gradient check),
one Adam step, the averaged inference weights, ragged batch sizes, and that online training lowers
the loss."""
import numpy as np
import pytest

from oracle import nrc as onrc
import vt

pytestmark = pytest.mark.gpu


def _params(seed=0, scale=0.15):
    rng = np.random.default_rng(seed)
    p = rng.uniform(-scale, scale, onrc.N_PARAMS)
    Ws = onrc.split(p)
    Ws[0][:, 265:] = 0
    Ws[4][4:] = 0
    return np.concatenate([w.reshape(-1) for w in Ws]).astype(np.float32)


def _dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a, np.float32)).cuda()


@pytest.mark.parametrize("n", [1, 17, 1000, 4099, 65536])
def test_forward_matches_oracle(gpu_ctx, n):
    # Against the oracle that rounds weights and every layer input to bf16 as the kernel does, the
    # outputs agree to fp32 accumulation order except where a hidden activation's fp32 sum lies within
    # that order's rounding of a bf16 rounding boundary: the activation then rounds the other way (one
    # bf16 step, 2^-8 relative) and moves its query's outputs by up to about 1e-3 of the output scale.
    # Bars: 99.9% of outputs within 1e-3, the mean within 1e-5, every output within 5e-3 (a few such
    # steps in one query).
    cache = vt.NRC(gpu_ctx, seed=3)
    p = _params(1)
    cache.params = p
    x = np.random.default_rng(n).random((n, 11)).astype(np.float32)
    y = cache.infer(_dev(x)).cpu().numpy().astype(np.float64)
    ref, _ = onrc.forward(p.astype(np.float64), x, bf16=True)
    exact, _ = onrc.forward(p.astype(np.float64), x)
    scale = np.abs(exact).max() + 1e-6
    err = np.abs(y - ref) / scale
    err_exact = np.abs(y - exact).max() / scale
    print(f"n {n}: |gpu - oracle(bf16)| / scale max {err.max():.2e} p99.9 {np.quantile(err, 0.999):.2e} "
          f"mean {err.mean():.2e}, vs fp64 {err_exact:.2e}", flush=True)
    assert np.quantile(err, 0.999) < 1e-3 and err.mean() < 1e-5 and err.max() < 5e-3
    assert err_exact < 2e-2
    cache.close()


def test_gradient_check(gpu_ctx):
    cache = vt.NRC(gpu_ctx, seed=3)
    p = _params(2)
    cache.params = p
    rng = np.random.default_rng(5)
    n = 777
    x = rng.random((n, 11)).astype(np.float32)
    t = rng.random((n, 4)).astype(np.float32)
    g, loss = cache.gradients(_dev(x), _dev(t))
    ref = onrc.gradients(p.astype(np.float64), x, t, bf16=True)
    exact = onrc.gradients(p.astype(np.float64), x, t)
    y, _ = onrc.forward(p.astype(np.float64), x)
    rel = np.linalg.norm(g - ref) / np.linalg.norm(ref)
    rel_exact = np.linalg.norm(g - exact) / np.linalg.norm(exact)
    per_layer = []
    offsets = np.cumsum([0] + onrc.SIZES)
    for k in range(5):
        a, b = offsets[k], offsets[k + 1]
        per_layer.append(np.linalg.norm(g[a:b] - exact[a:b]) / np.linalg.norm(exact[a:b]))
    print(f"gradient rel error vs bf16 oracle {rel:.2e}, vs fp64 {rel_exact:.2e}, per layer "
          + " ".join(f"{e:.2e}" for e in per_layer), flush=True)
    assert rel < 3e-2 and rel_exact < 6e-2 and max(per_layer) < 0.1
    assert abs(loss / onrc.loss(y, t) - 1) < 2e-2
    # Padded inputs and unused outputs receive nothing.
    Gs = onrc.split(g)
    assert np.all(Gs[0][:, 265:] == 0) and np.all(Gs[4][4:] == 0)
    cache.close()


@pytest.mark.parametrize("n", [1, 15, 16, 17, 127, 128, 129, 300, 32769])
def test_gradients_at_tile_edges(gpu_ctx, n):
    # Around a wave's 16 samples, a block's 128 and one block's second group (256 blocks x 128 + 1).
    # Against the oracle that rounds where the kernel does, gradients agree to fp32 summation order but
    # for activations whose sum lies at a bf16 rounding boundary: each moves one of its sample's terms by
    # a bf16 step, 2^-8 relative, so the whole by less than that.
    cache = vt.NRC(gpu_ctx, seed=3)
    p = _params(2)
    cache.params = p
    rng = np.random.default_rng(n)
    x = rng.random((n, 11)).astype(np.float32)
    t = rng.random((n, 4)).astype(np.float32)
    g, loss = cache.gradients(_dev(x), _dev(t))
    ref = onrc.split(onrc.gradients(p.astype(np.float64), x, t, bf16=True))
    err = [np.linalg.norm(a - b) / np.linalg.norm(b) for a, b in zip(onrc.split(g), ref)]
    print(f"n {n}: per layer " + " ".join(f"{e:.1e}" for e in err), flush=True)
    assert max(err) < 2.0 ** -8
    again, _ = cache.gradients(_dev(x), _dev(t))
    assert np.array_equal(g, again)   # summed in a fixed order
    cache.close()


def test_adam_step_matches_oracle(gpu_ctx):
    cache = vt.NRC(gpu_ctx, seed=3)
    p = _params(4)
    cache.params = p
    rng = np.random.default_rng(6)
    x = rng.random((256, 11)).astype(np.float32)
    t = rng.random((256, 4)).astype(np.float32)
    g, _ = cache.gradients(_dev(x), _dev(t))
    cache.train(_dev(x), _dev(t), lr=1e-3)
    q = cache.params
    want, _, _ = onrc.adam(p.astype(np.float64), 0.0, 0.0, g.astype(np.float64), 1)
    assert np.abs(q - want).max() < 2e-6
    cache.close()


def test_inference_uses_averaged_weights(gpu_ctx):
    # After one large Adam step (every parameter moves by about lr), inference answers with
    # decay p0 + (1 - decay) p1, far from the network at p1.
    cache = vt.NRC(gpu_ctx, seed=3)
    p = _params(4)
    cache.params = p
    rng = np.random.default_rng(8)
    x = rng.random((256, 11)).astype(np.float32)
    t = rng.random((256, 4)).astype(np.float32)
    cache.train(_dev(x), _dev(t), lr=0.05)
    q = cache.params
    e = onrc.ema(p.astype(np.float64), q.astype(np.float64))
    y = cache.infer(_dev(x)).cpu().numpy()
    ref, _ = onrc.forward(e, x, bf16=True)
    raw, _ = onrc.forward(q.astype(np.float64), x, bf16=True)
    scale = np.abs(ref).max()
    err, sep = np.abs(y - ref).max() / scale, np.abs(raw - ref).max() / scale
    print(f"ema inference error {err:.2e}, distance to the raw weights' answer {sep:.2e}", flush=True)
    assert err < 1e-2 and sep > 0.2
    cache.close()


def test_online_training_lowers_the_loss(gpu_ctx):
    import torch
    cache = vt.NRC(gpu_ctx, seed=9)
    rng = np.random.default_rng(7)

    def target(x):
        # A smooth radiance-like field of position and direction.
        r = 0.5 + 0.4 * np.sin(3 * x[:, 0] + 2 * x[:, 1]) * np.cos(2 * x[:, 3])
        return np.stack([r, 0.8 * r, 0.6 * r + 0.1 * x[:, 2], 0.4 * r], 1).astype(np.float32)

    xv = rng.random((4096, 11)).astype(np.float32)
    tv = target(xv)
    _, before = cache.gradients(_dev(xv), _dev(tv))
    for step in range(300):
        xb = rng.random((8192, 11)).astype(np.float32)
        cache.train(_dev(xb), _dev(target(xb)), lr=1e-3)
    torch.cuda.synchronize()
    _, after = cache.gradients(_dev(xv), _dev(tv))
    print(f"relative L2 loss before {before:.4f} after 300 steps {after:.4f}", flush=True)
    assert after < 0.1 * before
    cache.close()
