"""A frame large enough evaluates its rays' samples in windows, and only while
a ray lives; a profiled render takes all that
fit the workspace in one round.  Each ray's
samples, and the order they are composited in, are the same either way, so the
images, depths and step counts are compared bit for bit: at sizes on both
sides of the threshold (2^15 pixels), with ragged tiles, for an opaque skin
(rays end early), a translucent volume (the second round takes the rest) and
an empty one (rays run to the box's far side)."""
import numpy as np
import pytest

from insta_amd import synth
from insta_amd.capi import PRECISION_FP16, PRECISION_FP32, make_camera, small_config

pytestmark = pytest.mark.gpu


def _params(lay, cfg, scene):
    p = synth.network_params(7, lay, cfg)
    rng = np.random.default_rng(3)
    p[lay.n_mlp_params:] = rng.uniform(-0.3, 0.3, lay.n_grid_params).astype(np.float32)
    w1 = 64 * lay.density_in           # row 0 of the density output: the density logit
    h = np.abs(p[w1:w1 + 64])          # the hidden layer is >= 0: the sign of the row is the logit's
    p[w1:w1 + 64] = {"opaque": 60.0, "translucent": 0.0, "empty": -60.0}[scene] * h
    return p


@pytest.mark.parametrize("precision", [PRECISION_FP32, PRECISION_FP16])
@pytest.mark.parametrize("scene", ["opaque", "translucent", "empty"])
@pytest.mark.parametrize("size", [(181, 181), (182, 181), (301, 257), (1, 32768)])
def test_windows_render_the_same_frame(size, scene, precision):
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from insta_amd.capi import Context
    cfg = small_config(max_frames=1, precision=precision)
    av = synth.small_sphere_avatar(seed=0, n_frames=1)
    ctx = Context(cfg)
    ctx.set_canonical_mesh(av.canonical, av.faces, av.masks)
    ctx.set_frames(0, torch.from_numpy(av.frames[0][None]).cuda())
    ctx.set_params(torch.from_numpy(_params(ctx.layout, cfg, scene)).cuda())
    ctx.build_occupancy(0, 0.05)
    w, h = size
    cam = make_camera(synth.random_camera(np.random.default_rng(5), 1.0), synth.focal_from_fov(max(h, 64), 30.0))
    ctx.set_profiling(True)
    whole = [t.clone() for t in ctx.render(cam, w, h, 0, 0)]
    one = ctx.render_stats()
    ctx.set_profiling(False)
    got = ctx.render(cam, w, h, 0, 0)
    many = ctx.render_stats()
    for g, r in zip(got, whole):
        assert np.array_equal(g.cpu().numpy(), r.cpu().numpy())
    assert many.n_samples == one.n_samples
    if w * h < 1 << 15:   # (more than one round only where a round's samples exceed the workspace)
        assert many.n_iterations == one.n_iterations
    if scene == "opaque" and w * h >= 1 << 15:
        assert many.n_samples_emitted < one.n_samples_emitted
    if scene == "empty":  # nothing ends the rays: two windows, then all that is left
        assert many.n_iterations <= one.n_iterations + 2
