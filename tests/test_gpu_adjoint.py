"""Differentiable depth on the GPU: the vertex tape, the per-ray hit
vertices, tc_depth_adjoint against the FP64 adjoint and FP64 central
differences, and a 200-step Adam fit of a 512^2 height map."""
import numpy as np
import pytest

from adjoint_oracle import Problem
from vk_tessellated_clusters_amd import abi

pytestmark = pytest.mark.gpu

SIZE = 512


def _bilinear64(hmap, u, v):
    """FP32 sampler coordinates, FP64 weights (REPEAT)."""
    H, W = hmap.shape
    x = (u.astype(np.float32) * np.float32(W) - np.float32(0.5)).astype(np.float32)
    y = (v.astype(np.float32) * np.float32(H) - np.float32(0.5)).astype(np.float32)
    x0, y0 = np.floor(x), np.floor(y)
    fx, fy = (x - x0).astype(np.float64), (y - y0).astype(np.float64)
    xa, xb = x0.astype(np.int64) % W, (x0.astype(np.int64) + 1) % W
    ya, yb = y0.astype(np.int64) % H, (y0.astype(np.int64) + 1) % H
    h = hmap.astype(np.float64)
    return ((1 - fx) * (1 - fy) * h[ya, xa] + fx * (1 - fy) * h[ya, xb] + (1 - fx) * fy * h[yb, xa] +
            fx * fy * h[yb, xb])


@pytest.fixture(scope="module")
def frame():
    import torch
    from vk_tessellated_clusters_amd import diff, scene
    print(f"[adjoint] frame: {SIZE}^2 R32 heights (0.5 * fBm seed 5), target fBm seed 3", flush=True)
    hmap = (0.5 * scene.fbm_height(SIZE, 5, 4)).astype(np.float32)
    heights = torch.from_numpy(hmap).cuda().requires_grad_(True)
    target = diff.target_depth(SIZE, 3)
    r = diff.DepthRenderer(heights)
    t = diff.displaced_depth(heights, r)
    loss = diff.depth_loss(t, target)
    loss.backward()
    torch.cuda.synchronize()
    st = r.host_state()
    out = dict(st, hmap=hmap, grad=heights.grad.cpu().numpy(), t=t.detach().cpu().numpy(),
               target=target.cpu().numpy(), loss=float(loss))
    r.close()
    return out


def test_frame_capacity_and_coverage(frame):
    rb = frame["readback"]
    assert rb.numGenVertices > 0 and rb.numGenVertices <= abi.default_config().maxGeneratedVertices
    assert rb.numPartTriangles + rb.numFullClusters > 0
    hit = frame["t"] >= 0
    assert hit.mean() > 0.999, hit.mean()
    assert (frame["target"] >= 0).mean() > 0.999


def test_vertex_tape_reproduces_vertices(frame):
    tape, gv, hmap = frame["tape"], frame["genVertices"], frame["hmap"]
    assert (tape["texture"] == 0).all()
    np.testing.assert_allclose(tape["normal"], np.broadcast_to([0, 1, 0], tape["normal"].shape), atol=1e-7)
    h = _bilinear64(hmap, tape["u"], tape["v"])
    p = tape["base"].astype(np.float64) + tape["normal"].astype(np.float64) * (
        h * tape["heightScale"].astype(np.float64) + tape["heightOffset"].astype(np.float64))[:, None]
    np.testing.assert_allclose(gv.astype(np.float64), p, rtol=0, atol=2e-7)


def test_hit_vertices_span_the_hit_point(frame):
    hits, hv, rays, gv = frame["hits"], frame["hitVertices"].reshape(-1, 4), frame["rays"], frame["genVertices"]
    ok = hits["t"] >= 0
    assert (hv[ok, :3] < len(gv)).all() and (hv[~ok] == 0xFFFFFFFF).all()
    u, v = hits["u"][ok].astype(np.float64), hits["v"][ok].astype(np.float64)
    P = gv.astype(np.float64)[hv[ok, :3]]
    q = (1 - u - v)[:, None] * P[:, 0] + u[:, None] * P[:, 1] + v[:, None] * P[:, 2]
    x = rays["origin"][ok].astype(np.float64) + hits["t"][ok, None].astype(np.float64) * rays["direction"][ok]
    np.testing.assert_allclose(q, x, rtol=0, atol=2e-6)


def _problem(frame):
    return Problem(frame["rays"], frame["hits"], frame["hitVertices"], frame["tape"], [frame["hmap"]], frame["xforms"])


def _grad_t(frame, p):
    t64, tg = p.t64(), frame["target"].astype(np.float64)
    valid = (frame["t"] >= 0) & (frame["target"] >= 0)
    n = valid.sum()
    g = np.where(valid, 2.0 * (frame["t"].astype(np.float64) - tg) / n, 0.0)
    return g, 1.0 / n, t64


def test_gradient_matches_fp64_adjoint(frame):
    p = _problem(frame)
    g_t, _, t64 = _grad_t(frame, p)
    ok = frame["t"] >= 0
    # the plane distance of the frozen triangle agrees with the traced t
    np.testing.assert_allclose(t64[ok], frame["t"][ok], rtol=1e-5)
    (ref,) = p.adjoint64(g_t)
    g = frame["grad"].astype(np.float64)
    scale = np.abs(ref).max()
    assert scale > 0
    err = np.abs(g - ref)
    print(f"[adjoint] max |gpu - fp64 adjoint| / max|g| = {err.max() / scale:.3e}")
    assert (err <= 1e-3 * np.abs(ref) + 1e-5 * scale).all(), (err / (np.abs(ref) + 1e-5 * scale)).max()


def test_gradient_matches_fp64_central_differences(frame):
    p = _problem(frame)
    _, scale, _ = _grad_t(frame, p)
    rng = np.random.default_rng(0)
    texels = rng.choice(SIZE * SIZE, 256, replace=False).astype(np.uint64)
    fd = p.loss_fd64(frame["target"], scale, 0, texels, 1e-3)
    g = frame["grad"].reshape(-1)[texels.astype(np.int64)].astype(np.float64)
    floor = 1e-2 * np.sqrt(np.mean(fd * fd))
    assert floor > 0
    rel = np.abs(g - fd) / np.maximum(np.abs(fd), floor)
    print(f"[adjoint] 256 texels: max rel err vs FP64 central differences = {rel.max():.3e}, "
          f"median {np.median(rel):.3e}")
    assert rel.max() <= 1e-3


def test_adam_fit_200_steps():
    from vk_tessellated_clusters_amd import diff
    print("[adjoint] Adam fit: 200 steps", flush=True)
    heights, losses = diff.fit_heights(steps=200, lr=0.02)
    print(f"[adjoint] loss {losses[0]:.4e} -> {losses[-1]:.4e}")
    assert all(np.isfinite(losses))
    assert losses[-1] < 0.05 * losses[0]
    assert np.isfinite(heights.cpu().numpy()).all()


@pytest.mark.parametrize("rays", [32, 33, 256])
def test_gradient_of_scattered_rays(rays):
    """The adjoint sums a workgroup's 1024 rays per texel in LDS before it
    adds them to the map.  Rays in row order (many rays per texel) and the
    same rays in random order (more texels per workgroup than the table has
    slots) give one gradient: exactly 1024 rays (on the grid's own lines, where
    most miss and the table stays nearly empty), a remainder of 65, and 64
    workgroups.  Tolerance: each texel is a sum of at most K = 12 * rays^2 /
    texels * 16 (sixteen times the mean) or 256 float32 terms of one sign,
    so two orders differ by at most 2 K 2^-24 of the sum's size."""
    import torch
    from vk_tessellated_clusters_amd import diff, scene
    heights = torch.from_numpy((0.5 * scene.fbm_height(SIZE, 7, 4)).astype(np.float32)).cuda()
    r = diff.DepthRenderer(heights, rays=rays)
    try:
        t = r.render()
        gen = torch.Generator().manual_seed(rays)
        g = (torch.rand(rays * rays, generator=gen) + 0.5).cuda()
        want = r.adjoint(g)
        perm = torch.randperm(rays * rays, generator=gen).cuda()
        for name, width in (("rays", abi.RAY_DT.itemsize), ("hits", abi.HIT_DT.itemsize)):
            b = getattr(r, name).view(-1, width)
            b.copy_(b[perm].clone())
        hv = r.hit_vertices.view(-1, 4)
        hv.copy_(hv[perm].clone())
        got = r.adjoint(g[perm])
        torch.cuda.synchronize()
    finally:
        r.close()
    want, got = want.double().cpu().numpy(), got.double().cpu().numpy()
    assert rays == 32 or np.count_nonzero(want) > rays * rays / 4
    k = max(256.0, 12.0 * rays * rays / SIZE ** 2 * 16)
    assert (np.abs(got - want) <= 2 * k * 2.0 ** -24 * np.abs(want) + 1e-30).all()


@pytest.mark.parametrize("rays", [7, 64, 181, 182, 255, 256, 362, 363])
def test_gradient_by_ray_count_matches_fp64(rays):
    """Workgroups of 128, 256, 512 and 1024 rays, at both sides of each line
    (32, 64 and 128 thousand rays on 256 CUs) and for fewer rays than one
    workgroup: the gradient of the rays in row order and in random order (whose
    texels overflow the tables) against the FP64 adjoint, within the bounds of
    test_gradient_matches_fp64_adjoint."""
    import torch
    from vk_tessellated_clusters_amd import diff, scene
    hmap = (0.5 * scene.fbm_height(SIZE, 7, 4)).astype(np.float32)
    r = diff.DepthRenderer(torch.from_numpy(hmap).cuda(), rays=rays)
    rng = np.random.default_rng(rays)
    g = (rng.random(rays * rays) + 0.5).astype(np.float32)
    perm = rng.permutation(rays * rays)
    try:
        r.render()
        st = r.host_state()
        rows = r.adjoint(torch.from_numpy(g).cuda())
        dperm = torch.from_numpy(perm).cuda()
        for name, width in (("rays", abi.RAY_DT.itemsize), ("hits", abi.HIT_DT.itemsize)):
            b = getattr(r, name).view(-1, width)
            b.copy_(b[dperm].clone())
        hv = r.hit_vertices.view(-1, 4)
        hv.copy_(hv[dperm].clone())
        mixed = r.adjoint(torch.from_numpy(g[perm]).cuda())
        torch.cuda.synchronize()
    finally:
        r.close()
    assert (st["hits"]["t"] >= 0).mean() > 0.5  # (vertical rays on the lines of 7 x 7 lie in box planes and miss)
    (ref,) = Problem(st["rays"], st["hits"], st["hitVertices"], st["tape"], [hmap], st["xforms"]).adjoint64(g)
    scale = np.abs(ref).max()
    assert scale > 0
    for got in (rows, mixed):
        err = np.abs(got.double().cpu().numpy() - ref)
        assert (err <= 1e-3 * np.abs(ref) + 1e-5 * scale).all(), (err / (np.abs(ref) + 1e-5 * scale)).max()
