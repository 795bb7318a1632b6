"""Clusters without triangles.  The library's clusterizer makes none and
tc_cluster_template_order refuses them, but a caller that fills its own
tc_cluster and tc_clas_template records may: such a cluster gives a CLAS of its
vertices alone, as the oracle builds it."""
import copy

import numpy as np
import pytest

import harness
from vk_tessellated_clusters_amd import abi, device, scene

pytestmark = pytest.mark.gpu


@pytest.fixture
def empty_templates(monkeypatch):
    """Template words and sizes of geometries with empty clusters (the
    library's order for the others)."""
    real = device.cluster_templates

    def templates(geo, lib=None):
        some = geo.clusters["numTriangles"] > 0
        sub = copy.copy(geo)
        sub.clusters = geo.clusters[some]
        words, sizes = real(sub, lib)
        out = np.zeros(geo.num_clusters, np.uint32)
        out[some] = sizes
        for c in np.nonzero(~some)[0]:
            out[c] = (lib or abi.lib()).tc_clas_size(0, int(geo.clusters[c]["numVertices"]))
        return words, out

    monkeypatch.setattr(device, "cluster_templates", templates)
    monkeypatch.setattr(harness, "cluster_templates", templates)


def with_empty_clusters(geo, vertices):
    """`geo` with an empty cluster before each of its clusters: the first
    `vertices[k % len]` vertices of that one, no triangles."""
    g = copy.copy(geo)
    g.clusters = np.repeat(geo.clusters, 2)
    g.bboxes = np.repeat(geo.bboxes, 2)
    for k in range(geo.num_clusters):
        g.clusters[2 * k]["numTriangles"] = 0
        g.clusters[2 * k]["numVertices"] = min(int(geo.clusters[k]["numVertices"]), vertices[k % len(vertices)])
    return g


def mixed_scene(quads, px):
    """A displaced patch with empty clusters of 0 to 81 vertices between its
    own, and instances of one empty cluster alone above it."""
    geo = with_empty_clusters(scene.grid_patch(quads, quads, 8.0, 8.0), (5, 81, 0, 1, 64))
    lone = scene.grid_patch(2, 2, 4.0, 4.0)
    lone.clusters = lone.clusters.copy()
    lone.clusters[0]["numTriangles"] = 0
    insts = [scene.Instance(0, scene.rigid_transform(0.3 * k, [6.0 * (k % 2), 0.2 * k, 6.0 * (k // 2)]), displacement_index=0,
                            displacement_scale=0.4) for k in range(4)]
    insts += [scene.Instance(1, scene.rigid_transform(0.0, [3.0 * k, 2.0, 1.0])) for k in range(3)]
    heights = scene.to_r16(scene.fbm_height(64, 9, 3))
    cam = scene.Camera(eye=(4.0, 5.0, -5.0), center=(6.0, 0.0, 6.0), width=160, height=90, near=0.05, far=100.0)
    return scene.HostScene([geo, lone], insts, [(heights, abi.TEXTURE_R16_UNORM)], cam, px, "empty")


@pytest.mark.parametrize("quads,px", [(24, 400.0), (60, 1.0)])
def test_clas_without_triangles(empty_templates, quads, px):
    """Blocks of clusters without triangles hold their vertices, between
    blocks of whole clusters and of tessellated parts: every CLAS byte, size
    and list equals the oracle's."""
    host = mixed_scene(quads, px)
    cfg = harness.small_config()
    of = harness.OracleFrame(host, cfg)
    of.run(host.frame())
    ref = of.results()
    g = harness.GpuFrame(host, cfg)
    try:
        g.run(host.frame())
        res = g.results()
    finally:
        g.close()
    assert ref.counters["tempInstantiateCounter"] >= 4 * 2 * (-(-quads // 8)) ** 2 * 3 // 4
    harness.compare(res, ref)


@pytest.mark.parametrize("num", [300, 60000])
def test_trace_past_blocks_without_triangles(empty_templates, num):
    """Leaf steps whose lanes hold blocks without triangles beside others.
    Vertical rays take the general slab test, which an inverted box passes, so
    they enter such blocks in every tree; an instance of one such block alone
    is entered by all rays.  Few rays (shared waves) and many (whole waves), in
    one order and mixed: hits and decoded hits are the oracle's."""
    host = mixed_scene(24, 2.0)
    cfg = harness.small_config()
    rng = np.random.default_rng(num)
    rays = np.zeros(num, abi.RAY_DT)
    rays["origin"] = rng.uniform(-1.0, 15.0, (num, 3))
    rays["origin"][:, 1] = 6.0
    kind = np.arange(num) % 3
    rays["direction"] = np.where((kind == 0)[:, None], (0.0, -1.0, 0.0),
                                 rng.uniform(-0.4, 0.4, (num, 3)) * (1, 0, 1) + (0.003, -1.0, 0.002))
    rays["tMin"], rays["tMax"] = 0.0, 100.0
    of = harness.OracleFrame(host, cfg)
    of.run(host.frame())
    g = harness.GpuFrame(host, cfg)
    try:
        g.run(host.frame(), stages="accel")
        for order in (np.argsort(kind, kind="stable"), np.arange(num)):
            some = np.ascontiguousarray(rays[order])
            oh, od = of.trace(0, 0, 0, rays=some)
            assert (oh["t"] > 0).mean() > 0.3, "rays must meet the surface"
            for flags in (0, abi.TRACE_PRIVATE_STACK, abi.TRACE_PACKETS):
                gh, gd = g.trace(0, 0, flags, rays=some)
                harness.compare_hits(gh, oh, gd, od)
    finally:
        g.close()
