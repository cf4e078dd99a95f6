"""The matrix-core network takes calls that would end in a short round of
256-sample tiles on the CUs (up to 40,960 samples, and some beyond 65,536) in
tiles of 64: an output depends on its own sample alone, so a call of any size
returns, bit for bit, what the same samples return within a larger call.  Sizes
at the edges of both tiles and on both sides of the lines, with positions inside
and outside the unit cube (where dense levels wrap)."""
import numpy as np
import pytest

from insta_amd import synth
from insta_amd.capi import PRECISION_BF16, PRECISION_FP16, PRECISION_FP32, full_config, small_config

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [PRECISION_FP32, PRECISION_FP16, PRECISION_BF16])
@pytest.mark.parametrize("config", [small_config, full_config])
def test_outputs_do_not_depend_on_the_tile(config, precision):
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from insta_amd.capi import Context
    cfg = config(max_frames=1, precision=precision, n_extra_dims=0)
    ctx = Context(cfg)
    p = synth.network_params(7, ctx.layout, cfg)
    p[ctx.layout.n_mlp_params:] = np.random.default_rng(3).uniform(
        -0.3, 0.3, ctx.layout.n_grid_params).astype(np.float32)
    ctx.set_params(torch.from_numpy(p).cuda())
    rng = np.random.default_rng(5)
    c = rng.uniform(0.0, 1.0, ((1 << 17) + 257, 11)).astype(np.float32)
    c[::7, :3] = rng.uniform(-0.5, 1.5, c[::7, :3].shape)
    c = torch.from_numpy(c).cuda()
    whole = ctx.network_inference(c)
    assert torch.isfinite(whole).all()
    for n in (1, 15, 17, 63, 64, 65, 255, 257, 4097, 40960, 40961, 1 << 16, (1 << 16) + 1, 81920, 81921, 106496, 106497,
              1 << 17):
        assert torch.equal(ctx.network_inference(c[:n].contiguous()), whole[:n]), n


@pytest.mark.parametrize("config", [small_config, full_config])
def test_features_do_not_depend_on_the_call(config):
    """Encodes of more than 2^18 positions fetch the corners of a cell one by one, smaller ones in pairs: bit for bit
    the same features, inside and outside the unit cube."""
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from insta_amd.capi import Context
    cfg = config(max_frames=1, n_extra_dims=0)
    ctx = Context(cfg)
    p = synth.network_params(7, ctx.layout, cfg)
    p[ctx.layout.n_mlp_params:] = np.random.default_rng(3).uniform(
        -0.3, 0.3, ctx.layout.n_grid_params).astype(np.float32)
    ctx.set_params(torch.from_numpy(p).cuda())
    rng = np.random.default_rng(6)
    n = (1 << 18) + 1
    x = rng.uniform(0.0, 1.0, (n, 3)).astype(np.float32)
    x[::7] = rng.uniform(-0.5, 1.5, x[::7].shape)
    x = torch.from_numpy(x).cuda()
    whole = ctx.encode(x)
    assert torch.equal(ctx.encode(x[:1 << 18].contiguous()), whole[:1 << 18])
    assert torch.equal(ctx.encode(x[n - 5:].contiguous()), whole[n - 5:])
