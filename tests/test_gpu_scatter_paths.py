"""The hash-grid gradient scatter takes large levels with global atomics up to
a batch capacity of 8,192 samples and partitioned by table slice beyond it, in
passes of 2^18 samples.  A batch's gradients are the sum of its parts', so one
partitioned backward is compared with the sum of small backwards on a context
that never partitions, at batches on both sides of the chunk (1,024 samples),
pass and path boundaries.

Tolerance: both sides add the same FP32 products; the small backwards round
each of up to 33 partial gradients and their running sum to FP32, 2^-24
relative each, and atomics add a batch's up to 2^13 terms per entry in FP32:
1e-5 of a block's 2-norm."""
import numpy as np
import pytest

from insta_amd import synth
from insta_amd.capi import full_config

pytestmark = pytest.mark.gpu

PART = 8192


def _ctx(torch, cfg, av, params):
    from insta_amd.capi import Context
    ctx = Context(cfg)
    ctx.set_canonical_mesh(av.canonical, av.faces, av.masks)
    ctx.set_params(torch.from_numpy(params).cuda())
    return ctx


# growth 1.5 from 16: levels of 4,096 and 13,824 entries (LDS), a small dense one of 46,656, then hashed tables
@pytest.mark.parametrize("log2_t", [16, 19])
@pytest.mark.parametrize("n", [8193, 9216, 9217, 30001, (1 << 18) + 1])
def test_partitioned_backward_equals_the_sum_of_small_ones(log2_t, n):
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    cfg = full_config(max_frames=1, log2_hashmap_size=log2_t, cell_split=0)
    av = synth.small_sphere_avatar(seed=0)
    from insta_amd.capi import query_layout
    lay = query_layout(cfg)
    rng = np.random.default_rng(n + log2_t)
    params = synth.network_params(7, lay, cfg)
    params[lay.n_mlp_params:] = rng.uniform(-0.1, 0.1, lay.n_grid_params).astype(np.float32)
    c = np.zeros((n, 11), np.float32)
    c[:, 0:3] = rng.uniform(0.0, 1.0, (n, 3))
    c[: n // 2, 0:3] = 0.5 + 0.01 * rng.standard_normal((n // 2, 3))   # crowded entries
    d = rng.standard_normal((n, 3))
    c[:, 8:11] = (d / np.linalg.norm(d, axis=1, keepdims=True) + 1.0) * 0.5
    up = rng.standard_normal((n, 4)).astype(np.float32)
    coords, dout = torch.from_numpy(c).cuda(), torch.from_numpy(up).cuda()
    big = _ctx(torch, cfg, av, params)
    big.network_forward(coords)
    got = big.network_backward(coords, dout).double()
    small = _ctx(torch, cfg, av, params)
    small.reserve(train_samples=PART, train_batch=PART)
    ref = torch.zeros(lay.n_params, dtype=torch.float64, device="cuda")
    for s in range(0, n, PART):
        x = coords[s:s + PART].contiguous()
        small.network_forward(x)
        ref += small.network_backward(x, dout[s:s + PART].contiguous()).double()
    for l in range(cfg.n_levels):
        a = lay.n_mlp_params + 2 * lay.level_offset[l]
        b = a + 2 * lay.level_size[l]
        err = float((got[a:b] - ref[a:b]).norm() / ref[a:b].norm())
        assert err <= 1e-5, (l, err)
    a = lay.n_mlp_params
    assert float((got[:a] - ref[:a]).norm() / ref[:a].norm()) <= 1e-5
