"""GPU tests of what a radiance cache holds: the partial gradients' 31.5 MB from its first training on, also
where that training is recorded into a graph."""
import numpy as np
import pytest

import vt

pytestmark = pytest.mark.gpu
MB = 1 << 20


def _free():
    import torch
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def _batch(n, seed):
    import torch
    g = torch.Generator().manual_seed(seed)
    return torch.rand(n, 11, generator=g).cuda(), torch.rand(n, 4, generator=g).cuda()


def test_untrained_cache_is_small(gpu_ctx):
    # Eight caches that only infer: 0.74 MB each, where the partial gradients would be 252 MB in all.
    x, t = _batch(1000, 1)
    y = vt.NRC(gpu_ctx, seed=1)
    y.infer(x)
    before = _free()
    caches = [vt.NRC(gpu_ctx, seed=k) for k in range(8)]
    for c in caches:
        c.infer(x)
    held = before - _free()
    print(f"8 caches hold {held / MB:.1f} MB", flush=True)
    assert held < 32 * MB
    caches[0].train(x, t)
    assert before - _free() - held < 64 * MB
    for c in caches + [y]:
        c.close()


def test_first_training_in_a_graph(gpu_ctx):
    import torch
    x, t = _batch(3000, 2)
    eager = vt.NRC(gpu_ctx, seed=5)
    eager.train(x, t, lr=1e-3)
    ref = eager.params
    graphs, caches = [], [vt.NRC(gpu_ctx, seed=5) for _ in range(2)]
    start = caches[0].params
    for c in caches:
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            c.train(x, t, lr=1e-3, stream=torch.cuda.current_stream())
        graphs.append(g)
        assert np.array_equal(c.params, start)   # recorded, not run
    graphs[0].replay()
    torch.cuda.synchronize()
    assert np.array_equal(caches[0].params, ref)
    # Replays with the program's own work in between and one after another end in the same weights.
    for _ in range(2):
        eager.train(x, t)
        eager.infer(x)
        graphs[0].replay()
        torch.cuda.synchronize()
    for _ in range(3):
        graphs[1].replay()
    torch.cuda.synchronize()
    print(f"moved {np.abs(caches[0].params - start).max():.2e}", flush=True)
    assert np.array_equal(caches[0].params, caches[1].params)
    assert not np.array_equal(caches[0].params, ref)
    for c in caches + [eager]:
        c.close()
