"""The network plugin's kernels take batches of up to 2^16 samples 64 to a
workgroup and larger ones 256, and cut the weight gradients' sums into chunks
that follow the batch.  A sample's output and input gradient depend on that
sample alone, so they are, bit for bit, those of a larger batch that starts
with it; the parameter gradients are those of the larger batch whose other
samples carry no gradient, up to the order of the sums (chains of at most
some 600 FP32 additions, 600 x 2^-24 = 3.6e-5 of the terms' magnitudes, and
gradients whose terms partly cancel: 1e-4 of the largest)."""
import numpy as np
import pytest

from insta_amd import synth
from insta_amd.capi import full_config, small_config

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("config,extra", [(small_config, 0), (small_config, 16), (full_config, 16)])
def test_batch_size_does_not_change_a_sample(config, extra):
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from insta_amd.capi import Context
    cfg = config(max_frames=1, n_extra_dims=extra)
    ctx = Context(cfg)
    p = synth.network_params(7, ctx.layout, cfg)
    p[ctx.layout.n_mlp_params:] = np.random.default_rng(3).uniform(
        -0.3, 0.3, ctx.layout.n_grid_params).astype(np.float32)
    ctx.set_params(torch.from_numpy(p).cuda())
    rng = np.random.default_rng(5)
    total = (1 << 16) + 300
    c = torch.from_numpy(rng.uniform(0.0, 1.0, (total, 11 + extra)).astype(np.float32)).cuda()
    g = torch.from_numpy(rng.standard_normal((total, 4)).astype(np.float32)).cuda()

    def run(n, upstream):
        x = c[:n].contiguous()
        out = ctx.network_forward(x).clone()
        din = torch.zeros_like(x)
        grads = ctx.network_backward(x, upstream, dL_dinput_dev=din).clone()
        return out, din, grads

    whole_out, whole_din, _ = run(total, g)
    for n in (1, 63, 65, 257, 4097, 1 << 16):
        out, din, grads = run(n, g[:n].contiguous())
        assert torch.equal(out, whole_out[:n]), n
        assert torch.equal(din, whole_din[:n]), n
        alone = g.clone()
        alone[n:] = 0.0
        ref = run(total, alone)[2]
        assert (grads - ref).abs().max() <= 1e-4 * ref.abs().max(), n
