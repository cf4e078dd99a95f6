"""The hash-grid gradient scatter partitions large levels by table slice, in
passes of 2^18 samples, or, where a table exceeds 2^19 entries, adds to them
with global FP64 atomics.  A batch's gradients are the sum of its parts', so one
backward is compared with the sum of small ones on a context reserved for no
more, at batches on both sides of the chunk (1,024 samples) and pass
boundaries.

Tolerance: both sides add the same FP32 products; the small backwards round
each of up to 33 partial gradients and their running sum to FP32, 2^-24
relative each: 1e-5 of a block's 2-norm."""
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


def _crowd(n, rng):
    """Coordinates within a hundredth of the cube's centre, upstream gradients of one sign: few entries, long sums."""
    c = np.zeros((n, 11), np.float32)
    c[:, 0:3] = 0.5 + 0.01 * rng.standard_normal((n, 3))
    d = rng.standard_normal((n, 3))
    c[:, 8:11] = (d / np.linalg.norm(d, axis=1, keepdims=True) + 1.0) * 0.5
    return c, (np.abs(rng.standard_normal((n, 4))) + 0.5).astype(np.float32)


def _scene(torch, log2_t, rng):
    from insta_amd.capi import query_layout
    cfg = full_config(max_frames=1, log2_hashmap_size=log2_t, cell_split=0)
    lay = query_layout(cfg)
    params = synth.network_params(7, lay, cfg)
    params[lay.n_mlp_params:] = rng.uniform(-0.1, 0.1, lay.n_grid_params).astype(np.float32)
    av = synth.small_sphere_avatar(seed=0)
    first_large = next(l for l in range(cfg.n_levels) if lay.level_size[l] > 16384)
    return lay, (lambda: _ctx(torch, cfg, av, params)), lay.n_mlp_params + 2 * lay.level_offset[first_large]


@pytest.mark.parametrize("log2_t", [16, 19])
@pytest.mark.parametrize("n", [512, 2048, 8192])
def test_sums_do_not_lengthen_with_a_small_reservation(log2_t, n):
    """The same batch under a reservation of its own size and under a large one: the sums of the large levels are
    exact but for one rounding each (2^-24; a chain of FP32 additions would be off by some 9e-7 at 8,192)."""
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    rng = np.random.default_rng(n + log2_t)
    lay, make, first = _scene(torch, log2_t, rng)
    c, up = _crowd(n, rng)
    x, g = torch.from_numpy(c).cuda(), torch.from_numpy(up).cuda()
    grads = []
    for reserve in (n, 100000):
        ctx = make()
        ctx.reserve(train_samples=reserve, train_batch=reserve)
        ctx.network_forward(x)
        grads.append(ctx.network_backward(x, g).double()[first:])
    assert float((grads[0] - grads[1]).norm() / grads[1].norm()) <= 2 ** -23


def test_atomic_sums_of_large_tables():
    """T = 2^20: a batch of crowded samples against the sum of its parts of 256.  Either side's entries are sums in
    FP64 of products, of which runs of neighbours were added in FP32 (at most six additions deep), rounded to FP32
    once per backward: 2^-24 of the parts' magnitudes a rounding, 2^-22 for all (FP32 chains: some 9e-7)."""
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    rng = np.random.default_rng(20)
    lay, make, first = _scene(torch, 20, rng)
    n = 8192
    c, up = _crowd(n, rng)
    x, g = torch.from_numpy(c).cuda(), torch.from_numpy(up).cuda()
    ctx = make()
    ctx.network_forward(x)
    got = ctx.network_backward(x, g).double()[first:]
    ref, size = torch.zeros_like(got), torch.zeros_like(got)
    for s in range(0, n, 256):
        y = x[s:s + 256].contiguous()
        ctx.network_forward(y)
        part = ctx.network_backward(y, g[s:s + 256].contiguous()).double()[first:]
        ref += part
        size += part.abs()
    assert float((got - ref).norm() / size.norm()) <= 2 ** -22
