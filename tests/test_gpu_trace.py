"""Cluster acceleration structures and ray traversal on the GPU.

The BVH is validated on the host first (every CLAS reachable exactly once,
boxes equal to the unions of their subtrees, Morton order inside each
instance); only then are rays traced, and hits are compared with the CPU
oracle's hierarchy-free ray caster (closest hit over every CLAS, same
watertight test and tie-break): hit IDs must agree on >= 99.99 % of rays
and t within 1e-5 relative."""
import numpy as np
import pytest

import harness
from vk_tessellated_clusters_amd import abi, scene

pytestmark = pytest.mark.gpu


def small_scene():
    return scene.scene_grid_instances(num_instances=4, quads=64, patch_size=8.0, tex_size=256)


def clas_boxes(g, addrs):
    out = {}
    for a in np.unique(addrs):
        h = g.r.copy(int(a), 48).view(abi.CLAS_HEADER_DT)[0]
        out[int(a)] = (h["lo"].copy(), h["hi"].copy(), int(h["counts"]) | int(h["clusterID"]) << 32)
    return out


def check_blas(arr, boxes, inst):
    info = arr["infos"][inst]
    n = int(info["clusterReferencesCount"])
    first = int(info["clusterReferences"] - arr["sb"].blasClusterAddresses) // 8
    leaves = arr["blasLeaves"][first:first + n]
    assert sorted(leaves.tolist()) == sorted(arr["refs"][first:first + n].tolist())
    # the leaf info repeats each leaf's header counts and cluster ID
    assert [int(x) for x in arr["blasLeafInfo"][first:first + n]] == [boxes[int(a)][2] for a in leaves]
    if n == 1:
        return
    nodes = arr["blasNodes"][first:first + n - 1]
    seen_nodes, seen_leaves = set(), []

    def visit(word):
        if word & abi.BVH_LEAF:
            k = word & ~abi.BVH_LEAF
            assert k < n
            seen_leaves.append(k)
            return boxes[int(leaves[k])]
        assert word < n - 1 and word not in seen_nodes
        seen_nodes.add(word)
        nd = nodes[word]
        b0 = visit(int(nd["child0"]))
        b1 = visit(int(nd["child1"]))
        assert np.array_equal(nd["lo0"], b0[0]) and np.array_equal(nd["hi0"], b0[1])
        assert np.array_equal(nd["lo1"], b1[0]) and np.array_equal(nd["hi1"], b1[1])
        return np.minimum(b0[0], b1[0]), np.maximum(b0[1], b1[1])

    visit(0)
    assert len(seen_nodes) == n - 1 and sorted(seen_leaves) == list(range(n))
    check_wide(nodes, arr["blasNodes4"][first:first + n - 1])


def check_wide(nodes, wide):
    """Every four-wide record lists the node's leaf children and the
    children of its internal children, with the binary tree's boxes."""
    for i, nd in enumerate(nodes):
        want = []
        for c in (0, 1):
            ch, lo, hi = int(nd["child%d" % c]), nd["lo%d" % c], nd["hi%d" % c]
            if ch & abi.BVH_LEAF:
                want.append((ch, tuple(lo), tuple(hi)))
            else:
                g = nodes[ch]
                want += [(int(g["child0"]), tuple(g["lo0"]), tuple(g["hi0"])),
                         (int(g["child1"]), tuple(g["lo1"]), tuple(g["hi1"]))]
        w = wide[i]
        got = [(int(w["child"][k]), tuple(w["lo"][:, k]), tuple(w["hi"][:, k])) for k in range(4)
               if int(w["child"][k]) != abi.BVH4_EMPTY]
        assert got == want, i
        assert all(int(w["child"][k]) == abi.BVH4_EMPTY for k in range(len(want), 4))


def test_accel_structure():
    host = small_scene()
    g = harness.GpuFrame(host, harness.small_config())
    try:
        g.run(host.frame(), stages="accel")
        arr = g.accel_arrays()
        boxes = clas_boxes(g, arr["refs"])
        for i in range(len(host.instances)):
            check_blas(arr, boxes, i)
        assert harness.check_blas_key_order(g, arr) == len(arr["refs"])
        # TLAS reaches every instance once
        n = len(host.instances)
        seen = []

        def tvisit(word, depth=0):
            assert depth < 64
            if word & abi.BVH_LEAF:
                seen.append(word & ~abi.BVH_LEAF)
                return
            nd = arr["tlasNodes"][word]
            tvisit(int(nd["child0"]), depth + 1)
            tvisit(int(nd["child1"]), depth + 1)

        tvisit(arr["tlasRoot"])
        assert sorted(seen) == list(range(n))
        check_wide(arr["tlasNodes"][:n - 1], arr["tlasNodes4"][:n - 1])
    finally:
        g.close()


compare_hits = harness.compare_hits


def test_trace_parity_primary_and_shadow():
    host = small_scene()
    cfg = harness.small_config()
    of = harness.OracleFrame(host, cfg)
    of.run(host.frame())
    W, H = 160, 90
    oh, od = of.trace(W, H, abi.TRACE_CULL_BACK | abi.TRACE_SHADOW)
    g = harness.GpuFrame(host, cfg)
    try:
        g.run(host.frame(), stages="accel")
        gh, gd = g.trace(W, H, abi.TRACE_CULL_BACK | abi.TRACE_SHADOW)
        # the same traversal with the whole stack in private memory, and the
        # wave-wide packet traversal
        ph, pd = g.trace(W, H, abi.TRACE_CULL_BACK | abi.TRACE_SHADOW | abi.TRACE_PRIVATE_STACK)
        kh, kd = g.trace(W, H, abi.TRACE_CULL_BACK | abi.TRACE_SHADOW | abi.TRACE_PACKETS)
    finally:
        g.close()
    assert np.array_equal(ph.view(np.uint8), gh.view(np.uint8))
    assert np.array_equal(pd.view(np.uint8), gd.view(np.uint8))
    assert np.array_equal(kh.view(np.uint8), gh.view(np.uint8))
    assert np.array_equal(kd.view(np.uint8), gd.view(np.uint8))
    assert (oh["t"] > 0).mean() > 0.3, "camera must see geometry"
    agree = compare_hits(gh, oh, gd, od)
    print("hit agreement", agree, "hits", (oh["t"] > 0).sum(), "shadowed", od["shadowed"].sum())


def test_trace_parity_icosphere():
    host = scene.scene_icosphere()
    cfg = harness.small_config()
    of = harness.OracleFrame(host, cfg)
    of.run(host.frame())
    W, H = 128, 72
    oh, od = of.trace(W, H, abi.TRACE_CULL_BACK | abi.TRACE_SHADOW)
    g = harness.GpuFrame(host, cfg)
    try:
        g.run(host.frame(), stages="accel")
        gh, gd = g.trace(W, H, abi.TRACE_CULL_BACK | abi.TRACE_SHADOW)
    finally:
        g.close()
    # a radius-1 sphere at distance 3 under a 60 degree, 16:9 frustum covers
    # about 17% of the pixels
    assert 0.12 < (oh["t"] > 0).mean() < 0.25
    compare_hits(gh, oh, gd, od)


def test_trace_parity_transient_1x():
    """Hits on 1X transient CLAS decode to the base cluster and triangle."""
    host = scene.scene_grid_instances(num_instances=4, quads=64, patch_size=8.0, tex_size=256, tess_rate_pixels=16.0)
    cfg = harness.small_config(flags=abi.FLAG_DISPLACEMENT | abi.FLAG_CULLING | abi.FLAG_1X_TRANSIENT)
    of = harness.OracleFrame(host, cfg)
    of.run(host.frame())
    W, H = 160, 90
    oh, od = of.trace(W, H, abi.TRACE_CULL_BACK | abi.TRACE_SHADOW)
    g = harness.GpuFrame(host, cfg)
    try:
        g.run(host.frame(), stages="accel")
        gh, gd = g.trace(W, H, abi.TRACE_CULL_BACK | abi.TRACE_SHADOW)
    finally:
        g.close()
    assert ((oh["clusterID"] >> 30) == abi.RT_CLUSTER_MODE_1X_SUBSET_CLUSTER).sum() > 20
    agree = compare_hits(gh, oh, gd, od)
    print("hit agreement", agree)


def test_trace_parity_transient_2x():
    """Hits on 2X batch CLAS decode to the base cluster, triangle and
    sub-triangle (with 1X subsets in the same frame)."""
    host = scene.scene_grid_instances(num_instances=4, quads=64, patch_size=8.0, tex_size=256, tess_rate_pixels=8.0)
    cfg = harness.small_config(flags=abi.FLAG_DISPLACEMENT | abi.FLAG_CULLING | abi.FLAG_1X_TRANSIENT |
                               abi.FLAG_2X_TRANSIENT)
    of = harness.OracleFrame(host, cfg)
    of.run(host.frame())
    W, H = 160, 90
    oh, od = of.trace(W, H, abi.TRACE_CULL_BACK | abi.TRACE_SHADOW)
    g = harness.GpuFrame(host, cfg)
    try:
        g.run(host.frame(), stages="accel")
        gh, gd = g.trace(W, H, abi.TRACE_CULL_BACK | abi.TRACE_SHADOW)
    finally:
        g.close()
    assert ((oh["clusterID"] >> 30) == abi.RT_CLUSTER_MODE_2X_BATCHED_TESSELLATED).sum() > 50
    agree = compare_hits(gh, oh, gd, od)
    print("hit agreement", agree)


def test_tile_row_order_keeps_hits():
    """A renderer's camera traces time their tile rows, the next frame start
    ranks the rows (longest wave first), and that frame's traces of the same
    height take the rows in that order.  Hits and decoded records do not
    depend on the order: ordered traces, traces after a frame that traced
    another height (tile order again), and the 128- and 256-thread workgroup
    forms all equal the first trace byte for byte."""
    import ctypes as C
    host = small_scene()
    cfg = harness.small_config()
    flags = abi.TRACE_CULL_BACK | abi.TRACE_SHADOW
    W, H = 160, 90
    L = abi.lib()
    g = harness.GpuFrame(host, cfg)

    def frame_and_trace(w, h):
        g.run(host.frame(), stages="accel")
        return g.trace(w, h, flags)

    try:
        first = frame_and_trace(W, H)
        later = [frame_and_trace(W, H), frame_and_trace(W, H)]
        small = frame_and_trace(96, 54)
        small2 = frame_and_trace(96, 54)
        later += [frame_and_trace(W, H), frame_and_trace(W, H)]
        for threads in (128, 256):
            t = abi.Tuning()
            abi.check(L.tc_get_tuning(C.byref(t)))
            t.traceThreads = threads
            abi.check(L.tc_set_tuning(C.byref(t)))
            later += [frame_and_trace(W, H), frame_and_trace(W, H)]
    finally:
        abi.check(L.tc_set_tuning(None))
        g.close()
    assert (first[0]["t"] > 0).mean() > 0.3, "camera must see geometry"
    for h, d in later:
        assert np.array_equal(h.view(np.uint8), first[0].view(np.uint8))
        assert np.array_equal(d.view(np.uint8), first[1].view(np.uint8))
    assert np.array_equal(small2[0].view(np.uint8), small[0].view(np.uint8))
    assert np.array_equal(small2[1].view(np.uint8), small[1].view(np.uint8))


def test_packet_traversal_matches_per_ray():
    """Packet traversal gives the per-ray traversal's hits byte for byte,
    for camera rays (ragged tiles) and explicit rays in any directions."""
    host = scene.scene_icosphere()
    cfg = harness.small_config()
    g = harness.GpuFrame(host, cfg)
    rng = np.random.default_rng(7)
    rays = np.zeros(5000, abi.RAY_DT)
    rays["origin"] = rng.normal(0, 0.3, (5000, 3)) + np.array([0.0, 0.0, 3.0])
    dirs = rng.normal(size=(5000, 3)) + np.array([0.0, 0.0, -2.0])
    rays["direction"] = dirs / np.linalg.norm(dirs, axis=1, keepdims=True)
    rays["tMin"], rays["tMax"] = 0.0, 100.0
    try:
        g.run(host.frame(), stages="accel")
        for W, H in ((100, 60), (64, 64)):
            a = g.trace(W, H, abi.TRACE_CULL_BACK | abi.TRACE_SHADOW)
            b = g.trace(W, H, abi.TRACE_CULL_BACK | abi.TRACE_SHADOW | abi.TRACE_PACKETS)
            assert np.array_equal(a[0].view(np.uint8), b[0].view(np.uint8))
            assert np.array_equal(a[1].view(np.uint8), b[1].view(np.uint8))
        a = g.trace(0, 0, 0, rays=rays)
        b = g.trace(0, 0, abi.TRACE_PACKETS, rays=rays)
        assert (a[0]["t"] > 0).sum() > 500
        assert np.array_equal(a[0].view(np.uint8), b[0].view(np.uint8))
    finally:
        g.close()


def lattice_scene(n=1100, width=96, height=54):
    """n one-cluster patches (2 x 2 quads) on a square lattice with seeded
    yaw, one displacement map, and a camera looking down across the field:
    more instances than the one-workgroup TLAS build takes, so the TLAS is
    built by separate launches with a radix sort over instances."""
    geo = scene.grid_patch(2, 2, 1.4, 1.4)
    side = int(np.ceil(np.sqrt(n)))
    rng = np.random.default_rng(5)
    insts = []
    for k in range(n):
        x, z = 1.0 * (k % side - side / 2), 1.0 * (k // side - side / 2)
        insts.append(scene.Instance(0, scene.rigid_transform(float(rng.uniform(0, 6.28)), [x, 0.0, z]),
                                    displacement_index=0, displacement_scale=0.1))
    h = scene.to_r16(scene.fbm_height(64, 3, 3))
    cam = scene.Camera(eye=(0.0, 14.0, -22.0), center=(0.0, 0.0, 0.0), width=width, height=height, near=0.05,
                       far=500.0)
    return scene.HostScene([geo], insts, [(h, abi.TEXTURE_R16_UNORM)], cam, 8.0, "lattice")


def test_large_tlas_structure_and_trace():
    host = lattice_scene()
    n = len(host.instances)
    cfg = harness.small_config()
    W, H = host.camera.width, host.camera.height
    of = harness.OracleFrame(host, cfg)
    of.run(host.frame())
    oh, od = of.trace(W, H, abi.TRACE_CULL_BACK | abi.TRACE_SHADOW)
    g = harness.GpuFrame(host, cfg)
    try:
        g.run(host.frame(), stages="accel")
        arr = g.accel_arrays()
        # more than 256 instances: the key sort runs its instance digits
        assert harness.check_blas_key_order(g, arr) == len(arr["refs"])
        gh, gd = g.trace(W, H, abi.TRACE_CULL_BACK | abi.TRACE_SHADOW)
    finally:
        g.close()
    seen = []

    def tvisit(word, depth=0):
        assert depth < 64
        if word & abi.BVH_LEAF:
            seen.append(word & ~abi.BVH_LEAF)
            return
        nd = arr["tlasNodes"][word]
        tvisit(int(nd["child0"]), depth + 1)
        tvisit(int(nd["child1"]), depth + 1)

    tvisit(arr["tlasRoot"])
    assert sorted(seen) == list(range(n))
    check_wide(arr["tlasNodes"][:n - 1], arr["tlasNodes4"][:n - 1])
    assert (oh["t"] > 0).mean() > 0.3, "camera must see geometry"
    assert len(np.unique(oh["instanceID"][oh["t"] > 0])) > 200
    compare_hits(gh, oh, gd, od)


def test_large_tlas_with_clas_overflow():
    """The TLAS has key space of its own, so a scene with more instances
    (1100) than maxGeneratedClusters (1024) builds: the frame overflows its
    CLAS capacity exactly as the oracle's does, instances without accepted
    CLAS stay in the TLAS with empty BLAS, and hits match the oracle."""
    host = lattice_scene()
    n = len(host.instances)
    cfg = harness.small_config(maxGeneratedClusters=1024)
    W, H = host.camera.width, host.camera.height
    of = harness.OracleFrame(host, cfg)
    of.run(host.frame())
    ref = of.results()
    oh, od = of.trace(W, H, abi.TRACE_CULL_BACK | abi.TRACE_SHADOW)
    g = harness.GpuFrame(host, cfg)
    try:
        g.run(host.frame(), stages="accel")
        res = g.results()
        arr = g.accel_arrays()
        assert harness.check_blas_key_order(g, arr) == len(arr["refs"])
        gh, gd = g.trace(W, H, abi.TRACE_CULL_BACK | abi.TRACE_SHADOW)
    finally:
        g.close()
    harness.compare(res, ref)
    assert ref.counters["tempInstantiateCounter"] <= 1024 < n
    seen = []

    def tvisit(word, depth=0):
        assert depth < 64
        if word & abi.BVH_LEAF:
            seen.append(word & ~abi.BVH_LEAF)
            return
        nd = arr["tlasNodes"][word]
        tvisit(int(nd["child0"]), depth + 1)
        tvisit(int(nd["child1"]), depth + 1)

    tvisit(arr["tlasRoot"])
    assert sorted(seen) == list(range(n))
    compare_hits(gh, oh, gd, od)


@pytest.mark.parametrize("layout,num", [("parallel", 1), ("parallel", 4096), ("grazing", 63), ("grazing", 4097),
                                        ("scattered", 65), ("scattered", 6000)])
def test_shared_leaf_steps_match_packets(layout, num):
    """The leaf steps that share blocks over a wave's lanes give the packet
    traversal's hits (one lane per block) byte for byte: parallel rays onto
    whole clusters (every lane holds 32 groups, tested per lane), grazing rays
    in one plane (few lanes hold leaves, many leaves per ray) and scattered
    rays (blocks of all sizes in one wave: whole clusters and tessellated
    parts); ragged ray counts leave lanes without a ray; also with the whole
    stack in private memory."""
    host = scene.scene_grid_instances(num_instances=4, quads=60, patch_size=8.0, tex_size=256, tess_rate_pixels=6.0)
    rng = np.random.default_rng(num)
    rays = np.zeros(num, abi.RAY_DT)
    if layout == "parallel":
        rays["origin"] = rng.uniform(0.0, 14.0, (num, 3))
        rays["origin"][:, 1] = 5.0
        rays["direction"] = (0.01, -1.0, 0.02)
    elif layout == "grazing":
        rays["origin"] = (1.0, 0.35, -2.0)
        a = rng.uniform(-0.5, 0.5, num)
        rays["direction"] = np.stack([np.sin(a), rng.uniform(-0.02, 0.005, num), np.cos(a)], 1)
    else:
        rays["origin"] = rng.uniform(0.0, 14.0, (num, 3)) * (1.0, 0.1, 1.0) + (0.0, 0.7, 0.0)
        rays["direction"] = rng.normal(size=(num, 3))
    rays["tMin"], rays["tMax"] = 0.0, 200.0
    g = harness.GpuFrame(host, harness.small_config())
    try:
        g.run(host.frame(), stages="accel")
        want = g.trace(0, 0, abi.TRACE_PACKETS, rays=rays)
        got = [g.trace(0, 0, f, rays=rays) for f in (0, abi.TRACE_PRIVATE_STACK)]
    finally:
        g.close()
    if num > 1000:
        assert (want[0]["t"] > 0).mean() > 0.05, "rays must meet the surface"
        assert len(np.unique(want[0]["clusterID"] >> 30)) > 1 or layout != "scattered"
    for h, d in got:
        assert np.array_equal(h.view(np.uint8), want[0].view(np.uint8))
        assert np.array_equal(d.view(np.uint8), want[1].view(np.uint8))


@pytest.mark.gpu
@pytest.mark.parametrize("num", [64, 1000])
def test_ordered_and_general_slab_tests_agree(num):
    """Waves of regular rays load a node's planes in the order the ray meets
    them; a wave with a ray parallel to an axis, or with an origin that is not
    finite, takes the general slab test.  Rays of all eight octants give the
    same bytes both ways, and the irregular rays those of the packet traversal
    (which has only the general test)."""
    host = scene.scene_grid_instances(num_instances=4, quads=24, patch_size=8.0, tex_size=64, tess_rate_pixels=6.0)
    rng = np.random.default_rng(num)
    rays = np.zeros(num, abi.RAY_DT)
    target = rng.uniform(1.0, 13.0, (num, 3)) * (1.0, 0.02, 1.0)
    rays["direction"] = rng.choice([-1.0, 1.0], (num, 3)) * rng.uniform(0.1, 1.0, (num, 3))
    rays["origin"] = target - 3.0 * rays["direction"]
    rays["tMin"], rays["tMax"] = 0.0, 200.0
    mixed = rays.copy()
    odd = np.arange(0, num, 16)  # one or more in every wave
    mixed["direction"][odd, 1] = np.where(odd % 32 == 0, -1.0, mixed["direction"][odd, 1])
    mixed["direction"][odd[::2], 0] = 0.0
    mixed["direction"][odd[::4], 2] = -0.0
    mixed["origin"][odd[1::4], 1] = np.inf
    mixed["origin"][odd[3::4], 0] = np.nan
    g = harness.GpuFrame(host, harness.small_config())
    try:
        g.run(host.frame(), stages="accel")
        regular, _ = g.trace(0, 0, 0, rays=rays)
        general, _ = g.trace(0, 0, 0, rays=mixed)
        packets = [g.trace(0, 0, abi.TRACE_PACKETS, rays=r)[0] for r in (rays, mixed)]
    finally:
        g.close()
    if num == 1000:
        assert (regular["t"] > 0).mean() > 0.3, "rays must meet the surface"
    same = np.ones(num, bool)
    same[odd] = False
    assert np.array_equal(regular[same].view(np.uint8), general[same].view(np.uint8))
    assert np.array_equal(regular.view(np.uint8), packets[0].view(np.uint8))
    assert np.array_equal(general.view(np.uint8), packets[1].view(np.uint8))


@pytest.mark.gpu
@pytest.mark.parametrize("width,height", [(1, 1), (33, 17), (96, 54), (160, 90), (250, 130), (320, 180), (408, 224), (640, 360)])
def test_small_images_share_tiles(width, height):
    """Small images deal a tile's rays over 16, 8, 4, 2 or one wave; hits and
    decoded hits are those of the packet traversal (one wave a tile) byte for
    byte, each pixel written once."""
    host = scene.scene_grid_instances(num_instances=4, quads=24, patch_size=8.0, tex_size=64, tess_rate_pixels=6.0)
    g = harness.GpuFrame(host, harness.small_config())
    flags = abi.TRACE_CULL_BACK | abi.TRACE_SHADOW
    try:
        g.run(host.frame(), stages="accel")
        gh, gd = g.trace(width, height, flags)
        ph, pd = g.trace(width, height, flags | abi.TRACE_PACKETS)
    finally:
        g.close()
    assert width < 96 or (ph["t"] > 0).mean() > 0.2, "camera must see geometry"
    assert np.array_equal(gh.view(np.uint8), ph.view(np.uint8))
    assert np.array_equal(gd.view(np.uint8), pd.view(np.uint8))


@pytest.mark.gpu
@pytest.mark.parametrize("qx,qz,px", [(31, 16, 20.0), (40, 30, 20.0), (120, 90, 3.0), (760, 400, 0.7)])
def test_refit_of_one_instance(qx, qz, px):
    """Boxes and four-wide records of one instance whose leaves lie in one
    chunk of the refit, in three, in about twenty (climbs meet in LDS) and in
    more than 512 (in global memory): every node's boxes are its children's
    (the leaves' from their CLAS headers), checked in whole arrays, and the
    four-wide records of the first and of random nodes list the grandchildren."""
    geo = scene.grid_patch(qx, qz, 76.0, 40.0)
    cam = scene.Camera(eye=(38.0, 60.0, 19.0), center=(38.0, 0.0, 20.0), width=1920, height=1080, near=0.1, far=500.0)
    host = scene.HostScene([geo], [scene.Instance(0, np.eye(4))], [], cam, px, "one")
    tris = 2 * qx * qz
    cfg = harness.small_config(maxPartTriangles=tris + 1024, maxGeneratedClusters=tris + 32768,
                               maxGeneratedVertices=12 * tris + (1 << 16))
    g = harness.GpuFrame(host, cfg)
    try:
        g.run(host.frame(), stages="accel")
        arr = g.accel_arrays()
        sb = arr["sb"]
        n = int(arr["infos"][0]["clusterReferencesCount"])
        off = (arr["blasLeaves"][:n] - np.uint64(sb.genClusterData)).astype(np.int64)
        pool = g.r.copy(sb.genClusterData, int(off.max()) + 48).view(np.float32)
    finally:
        g.close()
    print("CLAS", n, flush=True)
    assert n > 0.9 * tris
    nodes, wide = arr["blasNodes"][:n - 1], arr["blasNodes4"][:n - 1]
    h = pool[(off // 4)[:, None] + np.arange(8)]
    leaf_lo, leaf_hi = h[:, 0:3], h[:, 4:7]
    lo = np.minimum(nodes["lo0"], nodes["lo1"])
    hi = np.maximum(nodes["hi0"], nodes["hi1"])
    seen = np.zeros(2 * n, np.int64)
    for c in ("0", "1"):
        word = nodes["child" + c]
        leaf = (word & abi.BVH_LEAF) != 0
        at = (word & ~np.uint32(abi.BVH_LEAF)).astype(np.int64)
        want_lo = np.where(leaf[:, None], leaf_lo[np.where(leaf, at, 0)], lo[np.where(leaf, 0, at)])
        want_hi = np.where(leaf[:, None], leaf_hi[np.where(leaf, at, 0)], hi[np.where(leaf, 0, at)])
        assert np.array_equal(nodes["lo" + c], want_lo) and np.array_equal(nodes["hi" + c], want_hi)
        np.add.at(seen, np.where(leaf, n + at, at), 1)
    assert seen[0] == 0 and (seen[1:n - 1] == 1).all() and (seen[n:] == 1).all()
    rng = np.random.default_rng(n)
    for i in [0, *rng.integers(0, n - 1, 2000)]:
        nd, want = nodes[i], []
        for c in ("0", "1"):
            ch = int(nd["child" + c])
            if ch & abi.BVH_LEAF:
                want.append((ch, tuple(nd["lo" + c]), tuple(nd["hi" + c])))
            else:
                want += [(int(nodes[ch]["child" + d]), tuple(nodes[ch]["lo" + d]), tuple(nodes[ch]["hi" + d])) for d in "01"]
        got = [(int(wide[i]["child"][k]), tuple(wide[i]["lo"][:, k]), tuple(wide[i]["hi"][:, k])) for k in range(len(want))]
        assert got == want
        assert all(int(wide[i]["child"][k]) == abi.BVH4_EMPTY for k in range(len(want), 4))


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 2, 3, 63, 65, 257, 512, 513, 1024])
def test_small_tlas_trees(n):
    """One-workgroup TLAS builds over instance counts at the edges of its rank
    shares (several threads, two and one thread to an instance): every instance
    is a leaf once, inner boxes are the unions below them, the four-wide records
    list the grandchildren."""
    host = lattice_scene(n)
    g = harness.GpuFrame(host, harness.small_config())
    try:
        g.run(host.frame(), stages="accel")
        arr = g.accel_arrays()
    finally:
        g.close()
    if n == 1:
        assert arr["tlasRoot"] == abi.BVH_LEAF
        return
    nodes = arr["tlasNodes"][:n - 1]
    seen, inner = [], set()

    def visit(word):
        assert word < n - 1 and word not in inner
        inner.add(word)
        nd = nodes[word]
        for c in ("0", "1"):
            ch = int(nd["child" + c])
            if ch & abi.BVH_LEAF:
                seen.append(ch & ~abi.BVH_LEAF)
            else:
                lo, hi = visit(ch)
                assert np.array_equal(nd["lo" + c], lo) and np.array_equal(nd["hi" + c], hi)
        return np.minimum(nd["lo0"], nd["lo1"]), np.maximum(nd["hi0"], nd["hi1"])

    assert arr["tlasRoot"] == 0
    visit(0)
    assert sorted(seen) == list(range(n)) and len(inner) == n - 1
    check_wide(nodes, arr["tlasNodes4"][:n - 1])


@pytest.mark.gpu
@pytest.mark.parametrize("width,height", [(480, 270), (568, 320), (592, 328), (600, 340)])
def test_halved_tiles_beyond_residency(width, height):
    """Tiles halved over more waves than are resident together, at both sides
    of the rule's line (24 waves a CU): hits and decoded hits are those of the
    packet traversal byte for byte."""
    host = scene.scene_grid_instances(num_instances=4, quads=24, patch_size=8.0, tex_size=64, tess_rate_pixels=6.0)
    g = harness.GpuFrame(host, harness.small_config())
    flags = abi.TRACE_CULL_BACK | abi.TRACE_SHADOW
    try:
        g.run(host.frame(), stages="accel")
        gh, gd = g.trace(width, height, flags)
        ph, pd = g.trace(width, height, flags | abi.TRACE_PACKETS)
    finally:
        g.close()
    assert (ph["t"] > 0).mean() > 0.2, "camera must see geometry"
    assert np.array_equal(gh.view(np.uint8), ph.view(np.uint8))
    assert np.array_equal(gd.view(np.uint8), pd.view(np.uint8))


@pytest.mark.gpu
@pytest.mark.parametrize("quads,px,vertices", [(1, 40.0, 2), (1, 40.0, 1 << 22), (12, 2.0, 1 << 22)])
def test_tlas_of_one_instance(quads, px, vertices):
    """The TLAS of one instance with no CLAS (its vertices are over the
    capacity), a single one (the BLAS root is a leaf) and 288: its record's
    fields, and the traced frame against the oracle's."""
    geo = scene.grid_patch(quads, quads, 1.0, 1.0)
    cam = scene.Camera(eye=(0.5, 2.0, 0.5), center=(0.5, 0.0, 0.5), up=(0.0, 0.0, -1.0), width=96, height=56, near=0.01,
                       far=100.0)
    host = scene.HostScene([geo], [scene.Instance(0, np.eye(4))], [], cam, px, "one")
    cfg = harness.small_config(maxGeneratedVertices=vertices)
    of = harness.OracleFrame(host, cfg)
    of.run(host.frame())
    oh, od = of.trace(96, 56, 0)
    g = harness.GpuFrame(host, cfg)
    try:
        g.run(host.frame(), stages="accel")
        arr = g.accel_arrays()
        gh, gd = g.trace(96, 56, 0)
    finally:
        g.close()
    n = int(of.sb.blasClusterCounter)
    assert n == (0 if vertices == 2 else 2 * quads * quads if quads > 1 else 1)
    ti, acc = arr["tlasInstances"][0], arr["accel"]
    assert arr["tlasRoot"] == abi.BVH_LEAF
    assert int(ti["numClusters"]) == n and int(ti["flags"]) == 1
    assert int(ti["blasRoot"]) == (abi.BVH_LEAF if n == 1 else 0)
    assert int(ti["blasNodes"]) == acc.blasNodes and int(ti["blasLeaves"]) == acc.blasLeaves
    assert np.array_equal(ti["objectToWorld"], np.eye(4, dtype=np.float32).reshape(-1)[:12])
    assert (gh["t"] >= 0).any() == (n > 0)
    compare_hits(gh, oh, gd, od)


def big_cluster_patch(n, q):
    """n x n clusters of q x q quads over [0, n]^2 (more triangles than the
    pipeline's 128 a cluster), with a bumpy surface."""
    ii, jj = np.meshgrid(np.arange(q + 1), np.arange(q + 1), indexing="xy")
    a = (jj[:-1, :-1] * (q + 1) + ii[:-1, :-1]).reshape(-1)
    tri = np.stack([np.stack([a, a + q + 1, a + 1], 1), np.stack([a + 1, a + q + 1, a + q + 2], 1)], 1).reshape(-1, 3)
    nv, nt = (q + 1) ** 2, 2 * q * q
    clusters, bboxes, pos = np.zeros(n * n, abi.CLUSTER_DT), np.zeros(n * n, abi.BBOX_DT), []
    for c in range(n * n):
        x, z = c % n + ii.reshape(-1) / q, c // n + jj.reshape(-1) / q
        p = np.stack([x, 0.1 * np.sin(7.0 * x) * np.cos(5.0 * z), z], 1)
        clusters[c] = (nv, nt, c * nt, c * nv, 3 * c * nt)
        bboxes[c] = (p.min(0), p.max(0), 0.0, 1.0)
        pos.append(p)
    pos = np.ascontiguousarray(np.concatenate(pos), np.float32)
    g = scene.Geometry(pos, np.tile(np.float32([0, 1, 0]), (len(pos), 1)), np.ascontiguousarray(pos[:, ::2] / n), clusters,
                       np.tile(tri.astype(np.uint8).reshape(-1), n * n), bboxes)
    g.lo, g.hi = pos.min(0), pos.max(0)
    return g


@pytest.mark.gpu
@pytest.mark.parametrize("q,num", [(8, 60000), (10, 300), (10, 60000), (11, 60000)])
def test_blocks_of_more_than_32_groups(q, num):
    """Clusters of 200 and 242 triangles (templates may hold that many) give
    blocks of 25 and 31 group pairs: a wave of parallel rays deals out more
    pairs than 64 lanes of whole pipeline clusters (8 x 8 quads) have.  Hits
    are the oracle's."""
    geo = big_cluster_patch(6, q)
    cam = scene.Camera(eye=(3.0, 4.0, 3.0), center=(3.0, 0.0, 3.0), up=(0.0, 0.0, -1.0), width=96, height=56, near=0.01,
                       far=100.0)
    insts = [scene.Instance(0, scene.rigid_transform(0.2, [0.0, 0.3 * k, 0.0])) for k in range(2)]
    host = scene.HostScene([geo], insts, [], cam, 4000.0, "big")
    cfg = harness.small_config()
    rng = np.random.default_rng(num)
    rays = np.zeros(num, abi.RAY_DT)
    rays["origin"] = rng.uniform(0.0, 6.0, (num, 3))
    rays["origin"][:, 1] = 5.0
    rays["direction"] = (0.01, -1.0, 0.02)
    rays["direction"][num // 2:] = (0.0, -1.0, 0.0)
    rays["tMin"], rays["tMax"] = 0.0, 100.0
    of = harness.OracleFrame(host, cfg)
    of.run(host.frame())
    oh, od = of.trace(0, 0, 0, rays=rays)
    assert of.sb.tempInstantiateCounter == 2 * 36 and (oh["t"] > 0).mean() > 0.5
    g = harness.GpuFrame(host, cfg)
    try:
        g.run(host.frame(), stages="accel")
        got = [g.trace(0, 0, f, rays=rays) for f in (0, abi.TRACE_PRIVATE_STACK)]
    finally:
        g.close()
    for gh, gd in got:
        harness.compare_hits(gh, oh, gd, od)
