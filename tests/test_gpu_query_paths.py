"""Every way a nearest-triangle query is answered gives the same triangle.

Points of one call go to groups of lanes or to one lane each by their number,
and the samples of a render (or of the density grid) that exceed a lane's
budget go to a second pass with a wave each.  All are exact under the
(squared distance, face id) order, so their results are compared bit for bit:
with brute force, and with the counting build, which has no budget."""
import numpy as np
import pytest

from insta_amd import synth
from insta_amd.capi import full_config, make_camera
from tests.conftest import ensure_oracle

pytestmark = pytest.mark.gpu

N_FRAMES = 2


@pytest.fixture(scope="module")
def scenes():
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    ensure_oracle()
    from insta_amd.capi import Context
    from oracle.oracle import Oracle
    av = synth.head_avatar(seed=1, n_frames=N_FRAMES)
    out = {}
    for split in (0, 2, 4):
        cfg = full_config(max_frames=N_FRAMES, cell_split=split)
        ctx = Context(cfg)
        ctx.set_canonical_mesh(av.canonical, av.faces, av.masks)
        ctx.set_frames(0, torch.from_numpy(np.stack(av.frames)).cuda())
        ctx.set_params(torch.from_numpy(synth.network_params(7, ctx.layout, cfg)).cuda())
        for f in range(N_FRAMES):
            ctx.build_occupancy(f, 0.015)
        out[split] = ctx
    orc = Oracle(full_config(max_frames=N_FRAMES))
    orc.set_canonical_mesh(av.canonical, av.faces, av.masks)
    orc.set_frame(0, av.frames[0])
    return out, orc, av


def _points(av, n, seed):
    """Near the skin, at the mesh's pole (long lists), near the centre (most leaves) and anywhere."""
    rng = np.random.default_rng(seed)
    v = av.frames[0].astype(np.float64)
    near = v[rng.integers(0, len(v), n)] + rng.normal(0.0, 0.004, (n, 3))
    pole = v[0] + rng.normal(0.0, 0.006, (n, 3))
    centre = 0.5 + rng.normal(0.0, 0.01, (n, 3))
    far = rng.uniform(0.0, 1.0, (n, 3))
    pick = np.arange(n) % 4
    p = np.choose(pick[:, None], [near, far, centre, pole])
    return np.clip(p, 0.0, 1.0).astype(np.float32)


@pytest.mark.parametrize("n", [1, 7, 8, 9, 63, 65, 4099])
@pytest.mark.parametrize("split", [0, 4])
def test_grouped_points_equal_brute_force(scenes, split, n):
    import torch
    ctxs, orc, av = scenes
    pts = _points(av, n, n)
    ids, dist = ctxs[split].closest(0, torch.from_numpy(pts).cuda())
    rid, rd2 = orc.closest_brute(0, pts)
    assert np.array_equal(ids.cpu().numpy(), rid)
    assert np.array_equal(dist.cpu().numpy(), np.sqrt(rd2))


@pytest.mark.parametrize("split", [0, 4])
def test_many_points_equal_grouped_points(scenes, split):
    """One more than the largest grouped call (one lane each) against two grouped calls."""
    import torch
    ctxs, _, av = scenes
    n = (1 << 20) + 1
    pts = torch.from_numpy(_points(av, n, 5)).cuda()
    ids, dist = ctxs[split].closest(0, pts)
    for part in (slice(0, n // 2), slice(n // 2, n)):
        gi, gd = ctxs[split].closest(0, pts[part].contiguous())
        assert torch.equal(gi, ids[part]) and torch.equal(gd, dist[part])


def test_many_coords_equal_grouped_coords(scenes):
    import torch
    ctxs, _, av = scenes
    n = (1 << 18) + 1
    c = np.zeros((n, 11), np.float32)
    c[:, 0:3] = _points(av, n, 6)
    c[:, 4] = np.arange(n) % (N_FRAMES + 1)      # frame 2 is not built: left as they are
    c[:, 8:11] = np.random.default_rng(7).uniform(0.2, 0.8, (n, 3))
    a = torch.from_numpy(c).cuda()
    whole, part = a.clone(), a.clone()
    ctxs[4].deform_samples(whole)
    for s in (slice(0, n // 2), slice(n // 2, n)):
        p = part[s].contiguous()
        ctxs[4].deform_samples(p)
        part[s] = p
    assert torch.equal(whole, part)
    assert torch.equal(whole[2::3], a[2::3])


@pytest.mark.parametrize("split", [0, 2, 4])
def test_second_pass_equals_unbudgeted_queries(scenes, split):
    """The mesh's pole seen from above, where lists are long or overflow: the budgeted render against the
    counting build's."""
    ctx = scenes[0][split]
    cam = make_camera(synth.look_at_camera(np.array([0.2, 1.0, 0.3]), 0.4), synth.focal_from_fov(200, 30.0))
    ctx.set_profiling(True, count_traversal=True)
    ref = [t.clone() for t in ctx.render(cam, 203, 200, 0, 0)]
    ctx.set_profiling(False)
    got = ctx.render(cam, 203, 200, 0, 0)
    for g, r in zip(got, ref):
        assert np.array_equal(g.cpu().numpy(), r.cpu().numpy())


@pytest.mark.parametrize("n", [1 << 17, (1 << 17) + 1])
def test_coords_on_a_small_mesh(n):
    """The line lies lower for meshes of few triangles: both sides of it against calls far below it."""
    import torch
    from insta_amd.capi import Context, small_config
    av = synth.small_sphere_avatar(seed=0, n_frames=N_FRAMES)
    ctx = Context(small_config(max_frames=N_FRAMES, cell_split=0))
    ctx.set_canonical_mesh(av.canonical, av.faces, av.masks)
    ctx.set_frames(0, torch.from_numpy(np.stack(av.frames)).cuda())
    c = np.zeros((n, 11), np.float32)
    c[:, 0:3] = _points(av, n, 8)
    c[:, 4] = np.arange(n) % N_FRAMES
    c[:, 8:11] = np.random.default_rng(9).uniform(0.2, 0.8, (n, 3))
    whole, part = torch.from_numpy(c).cuda(), torch.from_numpy(c).cuda()
    ctx.deform_samples(whole)
    for s in (slice(0, 40000), slice(40000, 80000), slice(80000, n)):
        p = part[s].contiguous()
        ctx.deform_samples(p)
        part[s] = p
    assert torch.equal(whole, part)


@pytest.mark.parametrize("split", [0, 1, 4])
def test_wider_occupancy_than_the_lists(split):
    """Samples inside and outside the cells that have lists, side by side in a wave: the budgeted render against the
    counting build's."""
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from insta_amd.capi import Context
    av = synth.head_avatar(seed=1, n_frames=1)
    cfg = full_config(max_frames=1, cell_split=split)
    ctx = Context(cfg)
    ctx.set_canonical_mesh(av.canonical, av.faces, av.masks)
    ctx.set_frames(0, torch.from_numpy(np.stack(av.frames)).cuda())
    ctx.set_params(torch.from_numpy(synth.network_params(7, ctx.layout, cfg)).cuda())
    wide = ctx.build_occupancy(0, 0.04).clone()
    ctx.build_occupancy(0, 0.015)
    ctx.set_occupancy(-1, wide)
    cam = make_camera(synth.look_at_camera(np.array([0.4, 0.7, 0.6]), 0.4), synth.focal_from_fov(200, 30.0))
    ctx.set_profiling(True, count_traversal=True)
    ref = [t.clone() for t in ctx.render(cam, 203, 200, 0, -1)]
    tc = ctx.traversal_counts()
    ctx.set_profiling(False)
    assert tc["queries"] > tc["list_queries"] >= (1000 if split else 0)
    got = ctx.render(cam, 203, 200, 0, -1)
    for g, r in zip(got, ref):
        assert np.array_equal(g.cpu().numpy(), r.cpu().numpy())
