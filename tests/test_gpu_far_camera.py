"""A camera so far away that a marching step is below the last bit of a ray's
t: the ray stands still.  In an occupied cell it samples the same position
until its step limit (the oracle's render, which never steps through an empty
cell here, says what it composites); in an empty cell, where a walk that waits
for the next voxel would never end, it ends without samples."""
import numpy as np
import pytest

from insta_amd import synth
from insta_amd.capi import make_camera, small_config
from tests.conftest import ensure_oracle

pytestmark = pytest.mark.gpu

FAR = 3.0e5   # a float's last bit there is 2^-5; the step is 1/256


def _scene(cfg, bits):
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    ensure_oracle()
    from insta_amd.capi import Context
    from oracle.oracle import Oracle
    av = synth.small_sphere_avatar(seed=0, n_frames=1)
    ctx, orc = Context(cfg), Oracle(cfg)
    for s in (ctx, orc):
        s.set_canonical_mesh(av.canonical, av.faces, av.masks)
    ctx.set_frames(0, torch.from_numpy(av.frames[0][None]).cuda())
    orc.set_frame(0, av.frames[0])
    p = synth.network_params(7, ctx.layout, cfg)
    ctx.set_params(torch.from_numpy(p).cuda())
    orc.set_params(p)
    ctx.set_occupancy(0, torch.from_numpy(bits).cuda())
    orc.set_occupancy(0, bits)
    return ctx, orc


def _camera(height):
    # along x, where the box ends at 0.9709 and the ray lands on a multiple of 2^-5 inside it
    cam = synth.look_at_camera(np.array([1.0, 0.0, 0.0]), FAR)
    return make_camera(cam, height * FAR)    # the image spans about one unit at the box


@pytest.mark.parametrize("size", [(24, 16), (200, 190)])   # one round, and windows (from 2^15 pixels)
def test_occupied_cells(size):
    cfg = small_config(max_frames=1)
    ctx, orc = _scene(cfg, np.full(cfg.grid_size ** 3 // 8, 255, np.uint8))
    w, h = size
    rgba, depth, steps = ctx.render(_camera(h), w, h, 0, 0)
    r_rgba, r_depth, r_steps, _ = orc.render(_camera(h), w, h, 0, 0)
    steps = steps.cpu().numpy().astype(np.uint32)
    assert steps.max() == cfg.max_steps
    assert np.array_equal(steps, r_steps)
    g, r = rgba.cpu().numpy().astype(np.float64), r_rgba.astype(np.float64)
    # up to 2^10 FP32 additions of positive terms: 2^10 x 2^-24 = 6e-5
    assert np.abs(g - r).max() <= 1e-4 * np.abs(r).max()


@pytest.mark.parametrize("size", [(24, 16), (200, 190)])
def test_empty_cells(size):
    cfg = small_config(max_frames=1)
    ctx, _ = _scene(cfg, np.zeros(cfg.grid_size ** 3 // 8, np.uint8))
    w, h = size
    rgba, _, steps = ctx.render(_camera(h), w, h, 0, 0)
    assert int(steps.sum()) == 0 and float(rgba.abs().sum()) == 0.0


def test_walk_of_a_position_at_a_time_is_the_walk_ahead():
    """The walk that far cameras take, at a distance where every step still moves the ray: the march of the
    oracle, step counts equal (empty and occupied cells, the mesh's own grid)."""
    cfg = small_config(max_frames=1, min_transmittance=0.0)
    ctx, orc = _scene(cfg, np.full(cfg.grid_size ** 3 // 8, 255, np.uint8))
    ctx.build_occupancy(0, 0.05)
    orc.build_occupancy(0, 0.05)
    for dist in (2.0e4, 32764.0):    # steps of 2^-8, last bits of 2^-9; the second is a far camera (from 2^15 on)
        w, h = 40, 33
        cam = make_camera(synth.look_at_camera(np.array([1.0, 0.0, 0.0]), dist), h * dist)
        steps = ctx.render(cam, w, h, 0, 0)[2].cpu().numpy().astype(np.uint32)
        r_steps = orc.render(cam, w, h, 0, 0)[2]
        assert r_steps.max() > 0
        assert np.array_equal(steps, r_steps), dist
