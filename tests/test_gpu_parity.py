"""GPU parity of the tessellation stages through the C-ABI: the HIP
library and the CPU oracle run the same seeded frames and must agree bit
for bit on every counter, list, record, CLAS block and BLAS reference list,
and within 2 ULP on generated positions (the kernels reproduce the
oracle's float evaluation order, so the observed difference is 0 ULP)."""
import ctypes as C

import numpy as np
import pytest

import harness
from vk_tessellated_clusters_amd import abi, scene

pytestmark = pytest.mark.gpu


def run_both(host, cfg, **frame_kw):
    print("case:", host.name, len(host.instances), "instances", host.num_base_triangles, "tris", flush=True)
    of = harness.OracleFrame(host, cfg)
    of.run(host.frame(**frame_kw))
    ref = of.results()
    g = harness.GpuFrame(host, cfg)
    try:
        g.run(host.frame(**frame_kw))
        res = g.results()
    finally:
        g.close()
    return res, ref


def small_grid(**kw):
    return scene.scene_grid_instances(num_instances=4, quads=64, patch_size=8.0, tex_size=256, **kw)


def test_icosphere_parity():
    res, ref = run_both(scene.scene_icosphere(), harness.small_config())
    assert ref.readback["numTotalTriangles"] > 1280
    harness.compare(res, ref)


def test_grid_split_parity():
    res, ref = run_both(small_grid(), harness.small_config())
    assert ref.counters["splitWriteCounter"] > 0
    harness.compare(res, ref)


def test_pn_parity():
    res, ref = run_both(scene.scene_icosphere(segments=16), harness.small_config(flags=abi.FLAG_DISPLACEMENT | abi.FLAG_PN))
    harness.compare(res, ref)


def test_animation_parity():
    """Ripple animation after displacement (full clusters and part
    templates), after PN, and on 1X transient clusters."""
    anim = abi.FLAG_DISPLACEMENT | abi.FLAG_CULLING | abi.FLAG_ANIMATION
    res, ref = run_both(small_grid(), harness.small_config(flags=anim), animation_time=2.25)
    assert ref.counters["partTriangleCounter"] > 0
    harness.compare(res, ref)
    res, ref = run_both(scene.scene_icosphere(segments=16), harness.small_config(flags=anim | abi.FLAG_PN),
                        animation_time=0.75)
    harness.compare(res, ref)
    res, ref = run_both(small_grid(tess_rate_pixels=16.0), harness.small_config(flags=anim | abi.FLAG_1X_TRANSIENT),
                        animation_time=7.5)
    assert ref.counters["transBuildCounter"] > 0
    harness.compare(res, ref)


def test_culling_off_and_invisible_instances():
    host = small_grid()
    host.camera.center = (200.0, 0.0, -100.0)
    res, ref = run_both(host, harness.small_config())
    assert ref.readback["numFullClusters"] > 0
    harness.compare(res, ref)
    res, ref = run_both(small_grid(), harness.small_config(flags=abi.FLAG_DISPLACEMENT))
    harness.compare(res, ref)


def test_capacity_overflow_parity():
    cfg = harness.small_config(maxSplitTriangles=512, maxPartTriangles=4096, maxGeneratedVertices=40000,
                               maxGeneratedClusters=3000)
    res, ref = run_both(small_grid(), cfg)
    assert ref.readback["numPartTriangles"] > 4096
    harness.compare(res, ref)


def test_transient_1x_parity():
    """1X transient clusters: records, part slots at the top of the part
    list, index and mapping bytes, CLAS blocks and both insert passes."""
    cfg = harness.small_config(flags=abi.FLAG_DISPLACEMENT | abi.FLAG_CULLING | abi.FLAG_1X_TRANSIENT)
    res, ref = run_both(small_grid(tess_rate_pixels=16.0), cfg)
    assert len(ref.arrays["transBuilds"]) > 10
    harness.compare(res, ref)


def test_transient_2x_parity():
    """2X mini batches: batch records and part slots, member vertices,
    index and u16 mapping bytes, CLAS blocks and both insert passes; alone,
    with 1X subsets, with PN and with the ripple."""
    base = abi.FLAG_DISPLACEMENT | abi.FLAG_CULLING | abi.FLAG_2X_TRANSIENT
    for flags, kw in ((base, {}), (base | abi.FLAG_1X_TRANSIENT, {}), (base | abi.FLAG_PN, {}),
                      (base | abi.FLAG_1X_TRANSIENT | abi.FLAG_ANIMATION, {"animation_time": 3.5})):
        print("flags", hex(flags), flush=True)
        res, ref = run_both(small_grid(tess_rate_pixels=8.0), harness.small_config(flags=flags), **kw)
        modes = ref.arrays["transBuilds"]["clusterID"] >> 30
        assert (modes == abi.RT_CLUSTER_MODE_2X_BATCHED_TESSELLATED).sum() > 100
        harness.compare(res, ref)


def test_transient_2x_capacity_overflow_parity():
    # batch slots and parts share the part list; vertices run out part way
    flags = abi.FLAG_DISPLACEMENT | abi.FLAG_CULLING | abi.FLAG_1X_TRANSIENT | abi.FLAG_2X_TRANSIENT
    for kw in ({"maxPartTriangles": 12000}, {"maxGeneratedVertices": 60000}, {"maxGeneratedClusters": 1500},
               {"maxGeneratedClusterMegs": 1}):
        print("capacity", kw, flush=True)
        res, ref = run_both(small_grid(tess_rate_pixels=8.0), harness.small_config(flags=flags, **kw))
        harness.compare(res, ref)


def test_loaded_gltf_scene_parity(tmp_path):
    """A glTF scene (clusters from tc_clusterize_mesh, R16 height maps
    from PNG files, node transforms) through the GPU frame and the oracle."""
    from test_assets import gltf_doc
    from vk_tessellated_clusters_amd import assets
    path, _ = gltf_doc(tmp_path)
    host = assets.load_gltf_scene(str(path), width=640, height=360, tess_rate_pixels=2.0)
    res, ref = run_both(host, harness.small_config())
    assert ref.readback["numTotalTriangles"] > host.num_base_triangles
    harness.compare(res, ref)


def split_queue_error(g):
    """The persistent split's error word (a wait hit its bound)."""
    ws = g.r.bindings.workspace
    return int(g.r.copy(ws + 256 + 12, 4).view(np.uint32)[0])


def test_persistent_split_wait_bound_is_reported():
    """A persistent-split wait that reaches its bound ends every wait of the
    launch and flags the frame in tc_readback.errorFlags.  The bound is
    lowered from the host (tc_tuning.splitWaitLimit = 1 sleep), so every
    wait of the launch still ends at once.  Only classify and the split
    stage run on the flagged frame (the split list is reset to all-ones at
    frame start, so every item the launch reads is either valid or
    rejected); the next frame, with the default bound, is clean and matches
    the oracle."""
    host = small_grid(tess_rate_pixels=1.0)
    cfg = harness.small_config(flags=abi.FLAG_DISPLACEMENT | abi.FLAG_CULLING | abi.FLAG_PERSISTENT_SPLIT,
                               maxSplitFactor=2)
    of = harness.OracleFrame(host, cfg)
    of.run(host.frame())
    ref = of.results()
    L = abi.lib()
    fc = host.frame()
    g = harness.GpuFrame(host, cfg)
    try:
        g.run(fc)
        t = abi.Tuning()
        abi.check(L.tc_get_tuning(C.byref(t)))
        t.splitWaitLimit = 1
        abi.check(L.tc_set_tuning(C.byref(t)))
        r = g.r
        b = C.byref(r.bindings)
        print("forced wait bound: classify + persistent split only", flush=True)
        abi.check(L.tc_renderer_begin_frame(r.handle, C.byref(fc), None))
        abi.check(L.tc_instances_classify(b, cfg, None))
        abi.check(L.tc_clusters_cull(b, cfg, None))
        abi.check(L.tc_build_setup(b, cfg, abi.BUILD_SETUP_CLASSIFY, None))
        abi.check(L.tc_cluster_classify(b, cfg, None))
        abi.check(L.tc_build_setup(b, cfg, abi.BUILD_SETUP_SPLIT, None))
        abi.check(L.tc_triangle_split(b, cfg, None))
        abi.check(L.tc_device_synchronize())
        flagged = r.readback().errorFlags
        assert split_queue_error(g) == 1
        assert flagged == abi.READBACK_ERROR_SPLIT_WAIT
        abi.check(L.tc_set_tuning(None))
        g.run(fc)
        res = g.results()
    finally:
        abi.check(L.tc_set_tuning(None))
        g.close()
    assert res.readback["errorFlags"] == 0
    harness.compare(res, ref)


def test_persistent_split_parity():
    """TC_FLAG_PERSISTENT_SPLIT runs every split pass in one launch; the
    frame equals the multipass frame and the oracle bit for bit (lists,
    counters and SPLIT_PASS state), for 4 and 14 passes, with the split list
    overflowing, and with transient builds."""
    base = abi.FLAG_DISPLACEMENT | abi.FLAG_CULLING
    cases = [(4.0, {}, base), (1.0, {}, base), (1.0, {"maxSplitFactor": 2}, base),
             (1.0, {"maxSplitTriangles": 300}, base), (1.0, {}, base | abi.FLAG_1X_TRANSIENT | abi.FLAG_2X_TRANSIENT)]
    for rate, kw, flags in cases:
        host = small_grid(tess_rate_pixels=rate)
        multi = harness.small_config(flags=flags, **kw)
        pers = harness.small_config(flags=flags | abi.FLAG_PERSISTENT_SPLIT, **kw)
        print("case", rate, kw, hex(flags), flush=True)
        of = harness.OracleFrame(host, multi)
        of.run(host.frame())
        ref = of.results()
        out = []
        for cfg in (multi, pers):
            g = harness.GpuFrame(host, cfg)
            try:
                g.run(host.frame())
                g.run(host.frame())  # a second frame reuses the queue state
                out.append(g.results())
                if cfg is pers:
                    assert split_queue_error(g) == 0
            finally:
                g.close()
        assert ref.counters["splitWriteCounter"] > 0
        harness.compare(out[1], out[0], max_ulp=0)
        harness.compare(out[1], ref)


def test_transient_1x_capacity_overflow_parity():
    # the part list is shared by parts (from the bottom) and transient slots
    # (from the top); acceptance stays a prefix of the canonical order
    cfg = harness.small_config(flags=abi.FLAG_DISPLACEMENT | abi.FLAG_CULLING | abi.FLAG_1X_TRANSIENT,
                               maxPartTriangles=6000, maxGeneratedVertices=200000)
    res, ref = run_both(small_grid(tess_rate_pixels=16.0), cfg)
    assert ref.readback["numPartTriangles"] > 6000
    harness.compare(res, ref)


def test_many_instances_parity():
    host = scene.scene_grid_instances(num_instances=16, quads=32, patch_size=4.0, tex_size=128, cam_height=1.5)
    res, ref = run_both(host, harness.small_config())
    harness.compare(res, ref)


def test_repeat_frames_are_identical():
    host = small_grid()
    cfg = harness.small_config()
    g = harness.GpuFrame(host, cfg)
    try:
        g.run(host.frame())
        r1 = g.results()
        g.run(host.frame())
        r2 = g.results()
    finally:
        g.close()
    harness.compare(r2, r1, max_ulp=0)


def test_launch_shapes_do_not_change_results():
    """Work-queue kernels give identical frames, BVHs and hits for every
    launch shape the tuner may pick."""
    import numpy as np
    from vk_tessellated_clusters_amd import autotune
    host = small_grid()
    cfg = harness.small_config()
    shapes = [None, dict(classifyBlocksPerCU=1, splitBlocksPerCU=1, instantiateBlocksPerCU=1, clasWavesPerCU=4,
                         traceBlocksPerCU=2, traceThreads=64, bvhBlocksPerCU=1),
              dict(classifyBlocksPerCU=12, splitBlocksPerCU=16, instantiateBlocksPerCU=8, clasWavesPerCU=128,
                   traceBlocksPerCU=128, traceThreads=128, bvhBlocksPerCU=16)]
    out = []
    try:
        for shape in shapes:
            autotune.set_tuning(shape)
            g = harness.GpuFrame(host, cfg)
            try:
                g.run(host.frame(), stages="accel")
                res = g.results()
                arr = g.accel_arrays()
                hits, dec = g.trace(96, 54, abi.TRACE_CULL_BACK | abi.TRACE_SHADOW)
            finally:
                g.close()
            out.append((res, arr, hits, dec))
    finally:
        autotune.set_tuning(None)
    def written(a):
        """Node records that the build writes (n - 1 internal nodes per
        instance) and leaves as offsets into the CLAS pool."""
        sb, n = a["sb"], len(a["infos"])
        keep = np.zeros(len(a["blasNodes"]), bool)
        for info in a["infos"]:
            first = int(info["clusterReferences"] - sb.blasClusterAddresses) // 8
            keep[first:first + max(0, int(info["clusterReferencesCount"]) - 1)] = True
        return (a["blasNodes"][keep].view(np.uint8), a["blasNodes4"][keep].view(np.uint8),
                a["tlasNodes"][:n - 1].view(np.uint8), a["tlasNodes4"][:n - 1].view(np.uint8),
                a["blasLeaves"] - np.uint64(sb.genClusterData))

    r0, a0, h0, d0 = out[0]
    for r, a, h, d in out[1:]:
        harness.compare(r, r0, max_ulp=0)
        for x, y in zip(written(a), written(a0)):
            assert np.array_equal(x, y)
        assert np.array_equal(h.view(np.uint8), h0.view(np.uint8))
        assert np.array_equal(d.view(np.uint8), d0.view(np.uint8))


def test_graph_replays_match_eager_frames():
    """Graph replays with new frame constants (queued back to back, more
    than the pinned ring holds) end in the same state as an eager frame
    with the last constants."""
    import ctypes as C
    import numpy as np
    import torch
    host = small_grid()
    cfg = harness.small_config()
    frames = []
    for k in range(20):
        host.camera.eye = (8.0 + 0.3 * k, 2.5, -2.4 + 0.1 * k)
        frames.append(host.frame())
    g = harness.GpuFrame(host, cfg)
    try:
        g.run(frames[-1], stages="accel")
        eager = g.results()
        eh, ed = g.trace(64, 36, abi.TRACE_CULL_BACK)
        stream = torch.cuda.Stream()
        s = C.c_void_p(stream.cuda_stream)
        L = g.r.L
        abi.check(L.tc_renderer_graph_capture(g.r.handle, C.byref(frames[0]), None, s))
        for fc in frames:
            abi.check(L.tc_renderer_graph_launch(g.r.handle, C.byref(fc), s))
        stream.synchronize()
        replay = g.results()
        rh, rd = g.trace(64, 36, abi.TRACE_CULL_BACK)
    finally:
        g.close()
    ce, cr = eager.arrays["clasBlocks"], replay.arrays["clasBlocks"]
    if ce.shape == cr.shape and not np.array_equal(ce, cr):
        # name the first differing block and the part of it that differs
        off = 0
        for i, sz in enumerate(eager.arrays["tempClusterSizes"]):
            a, b = ce[off:off + int(sz)], cr[off:off + int(sz)]
            if not np.array_equal(a, b):
                d = np.nonzero(a != b)[0]
                print("block", i, "of", len(eager.arrays["tempClusterSizes"]), "size", int(sz), "differs at bytes",
                      d[:8], "count", d.size, "headers", a[:48].view(abi.CLAS_HEADER_DT), b[:48].view(abi.CLAS_HEADER_DT))
                break
            off += int(sz)
    harness.compare(replay, eager, max_ulp=0)
    assert np.array_equal(rh.view(np.uint8), eh.view(np.uint8))


def test_device_fbm_matches_numpy():
    """The device height-map generator reproduces the numpy generator texel
    for texel (R32 and R16)."""
    import numpy as np
    import torch
    L = abi.lib()
    for size, seed, octaves, fmt in ((64, 1, 6, abi.TEXTURE_R32_FLOAT), (256, 7, 4, abi.TEXTURE_R16_UNORM),
                                     (100, 3, 5, abi.TEXTURE_R32_FLOAT)):
        ref = scene.fbm_height(size, seed, octaves)
        if fmt == abi.TEXTURE_R16_UNORM:
            ref = scene.to_r16(ref)
        out = torch.zeros(size * size * ref.itemsize, dtype=torch.uint8, device="cuda")
        abi.check(L.tc_fbm_height(out.data_ptr(), size, seed, octaves, 8, fmt, None))
        torch.cuda.synchronize()
        got = out.cpu().numpy().view(ref.dtype).reshape(size, size)
        assert np.array_equal(got, ref)


@pytest.mark.parametrize("instances,quads", [(1, 24), (131, 64), (258, 64)])
def test_classify_tile_sizes(instances, quads):
    """Classify's tiles hold 8 clusters in small frames and up to 64 in large
    ones: 9 clusters (a full and a ragged tile of 8), 8384 (tiles of 16) and
    16,512 (tiles of 32, the last ragged) equal the oracle bit for bit."""
    host = scene.scene_grid_instances(num_instances=instances, quads=quads, patch_size=8.0, tex_size=64)
    cfg = harness.small_config(maxVisibleClusters=1 << 15, maxGeneratedClusters=1 << 17, maxPartTriangles=1 << 17)
    of = harness.OracleFrame(host, cfg)
    of.run(host.frame(), nthreads=8)
    g = harness.GpuFrame(host, cfg)
    try:
        g.run(host.frame())
        res = g.results()
    finally:
        g.close()
    harness.compare(res, of.results())


@pytest.mark.parametrize("quads,rate,stride", [(8, 4000.0, 12), (40, 3.0, 12), (40, 3.0, 16), (64, 1.0, 12)])
def test_clas_runs_and_rounds(quads, rate, stride):
    """CLAS blocks are built in runs of records whose rounds hold what fits
    LDS: one whole cluster alone, whole clusters (ragged ones among them)
    beside parts of every size, mostly parts of up to 121 triangles.  Blocks,
    sizes and padding equal the oracle byte for byte; vertex buffers with a
    stride of 16 bytes give the same blocks."""
    host = scene.scene_grid_instances(num_instances=1 if quads == 8 else 3, quads=quads, patch_size=6.0, tex_size=64,
                                      tess_rate_pixels=rate)
    cfg = harness.small_config()
    of = harness.OracleFrame(host, cfg)
    of.run(host.frame(), nthreads=8)
    g = harness.GpuFrame(host, cfg)
    try:
        g.run(host.frame())
        res = g.results()
        if stride != 12:
            # the same vertices spread to 16 bytes in a second buffer
            import torch
            nv = res.arrays["genVertices"].shape[0]
            wide = torch.zeros(nv, 4, dtype=torch.float32, device="cuda")
            wide[:, :3] = torch.from_numpy(res.arrays["genVertices"].copy()).cuda()
            sb = g.r.scene_building()
            n = sb.tempInstantiateCounter
            ti = g.r.copy(sb.tempInstantiations, 32 * n).view(abi.TEMPLATE_INSTANTIATE_INFO).copy()
            base = np.uint64(sb.genVertices)
            ti["vertexBufferAddress"] = np.uint64(wide.data_ptr()) + (ti["vertexBufferAddress"] - base) // np.uint64(12) * np.uint64(16)
            ti["vertexBufferStride"] = 16
            torch.cuda.synchronize()
            L = abi.lib()
            abi.check(L.tc_memcpy(C.c_void_p(sb.tempInstantiations), ti.ctypes.data, ti.nbytes), "tc_memcpy")
            abi.check(L.tc_clas_instantiate(C.byref(g.r.bindings), cfg, None), "tc_clas_instantiate")
            again = g.results()
            want, got = (x.arrays["clasBlocks"].view(np.uint32).copy() for x in (res, again))
            # the header's vertexBase names a source outside genVertices
            at = (res.arrays["tempClusterOffsets"].astype(np.int64) - int(res.arrays["tempClusterOffsets"][0])) // 4 + 8
            want[at] = got[at] = 0
            assert np.array_equal(want, got)
            assert np.array_equal(res.arrays["tempClusterSizes"], again.arrays["tempClusterSizes"])
    finally:
        g.close()
    harness.compare(res, of.results())


@pytest.mark.parametrize("instances,quads,rate,flags", [
    (1, 16, 0.25, 0), (2, 64, 1.5, 0), (4, 96, 0.6, 0), (4, 64, 1.0, abi.FLAG_1X_TRANSIENT | abi.FLAG_2X_TRANSIENT)])
def test_frame_sequence_tiles(instances, quads, rate, flags):
    """The frame sequence takes its stages' counters, tickets and epochs from
    the launches before them, and tiles of a size by the number of items
    (split: 16 to 64, instantiation: 256 to 1024 parts): few and many split
    triangles and parts equal the oracle, as do two frames in a row and the
    stage entry points with a prologue each."""
    host = scene.scene_grid_instances(num_instances=instances, quads=quads, patch_size=6.0, tex_size=64,
                                      tess_rate_pixels=rate)
    cfg = harness.small_config(maxPartTriangles=1 << 20, maxGeneratedClusters=(1 << 14) + (1 << 20), maxSplitTriangles=1 << 17,
                               maxGeneratedVertices=1 << 25, maxGeneratedClusterMegs=2048)
    cfg.flags |= flags
    of = harness.OracleFrame(host, cfg)
    of.run(host.frame(), nthreads=8)
    ref = of.results()
    print("split", ref.counters["splitWriteCounter"], "parts", ref.counters["partTriangleCounter"], flush=True)
    assert ref.counters["splitWriteCounter"] > 0
    g = harness.GpuFrame(host, cfg)
    L, b = abi.lib(), C.byref(g.r.bindings)
    try:
        g.run(host.frame())
        g.run(host.frame())
        harness.compare(g.results(), ref)
        abi.check(L.tc_renderer_begin_frame(g.r.handle, C.byref(host.frame()), None))
        abi.check(L.tc_instances_classify(b, cfg, None))
        abi.check(L.tc_clusters_cull(b, cfg, None))
        abi.check(L.tc_build_setup(b, cfg, abi.BUILD_SETUP_CLASSIFY, None))
        abi.check(L.tc_cluster_classify(b, cfg, None))
        abi.check(L.tc_build_setup(b, cfg, abi.BUILD_SETUP_SPLIT, None))
        passes = L.tc_num_split_passes(cfg.maxSplitFactor)
        for p in range(passes):
            abi.check(L.tc_triangle_split(b, cfg, None))
            if p + 1 < passes:
                abi.check(L.tc_build_setup(b, cfg, abi.BUILD_SETUP_SPLIT_PASS, None))
        abi.check(L.tc_build_setup(b, cfg, abi.BUILD_SETUP_INSTANTIATE_TESS, None))
        abi.check(L.tc_triangle_tess_template_instantiate(b, cfg, None))
        abi.check(L.tc_build_setup(b, cfg, abi.BUILD_SETUP_BUILD_BLAS, None))
        g.r.clas_and_blas()
        abi.check(L.tc_device_synchronize(), "synchronize")
        harness.compare(g.results(), ref)
    finally:
        g.close()


@pytest.mark.parametrize("instances,flags,capacity", [
    (1, 0, 0), (2, 0, 0), (256, 0, 0), (257, 0, 0), (600, 0, 0), (2, "trans", 0), (300, "trans", 0), (40, 0, 300),
    (300, "trans", 600)])
def test_insertion_with_keys_matches_stages(instances, flags, capacity):
    """tc_renderer_build_accel inserts and sorts in one sort whose digit bases
    come from the reference counts; the stage entry points (setup, insertion of
    both lists, keys, sort) give the same lists, counts, totals and trees: one
    and two instance digits and their borders, both CLAS lists, and a CLAS
    capacity that cuts the frame."""
    from test_gpu_trace import lattice_scene
    host = lattice_scene(instances)
    host.tess_rate_pixels /= 8.0  # eight parts a patch, or transient builds
    over = {"maxGeneratedClusters": capacity} if capacity else {}
    if flags:
        over["flags"] = (abi.FLAG_DISPLACEMENT | abi.FLAG_CULLING | abi.FLAG_1X_TRANSIENT | abi.FLAG_2X_TRANSIENT)
    g = harness.GpuFrame(host, harness.small_config(**over))
    L = abi.lib()
    out = []
    try:
        for staged in (False, True):
            g.r.tessellate(host.frame())
            if staged:
                g.r.clas_and_blas()
                accel, xforms = g.r.accel()
                abi.check(L.tc_accel_build(C.byref(g.r.bindings), g.cfg, C.byref(accel), C.c_void_p(xforms), None),
                          "tc_accel_build")
            else:
                g.r.build_accel()
            abi.check(L.tc_device_synchronize(), "synchronize")
            arr, rb = g.accel_arrays(), g.r.readback()
            sb = arr["sb"]
            keep = np.zeros(len(arr["blasNodes"]), bool)
            for info in arr["infos"]:
                first = int(info["clusterReferences"] - sb.blasClusterAddresses) // 8
                keep[first:first + max(0, int(info["clusterReferencesCount"]) - 1)] = True
            out.append([arr["refs"], arr["infos"], arr["blasLeaves"], arr["blasLeafInfo"], arr["blasNodes"][keep],
                        arr["blasNodes4"][keep], arr["tlasNodes"][:instances - 1], arr["tlasInstances"],
                        np.array([sb.blasClusterCounter, sb.tempInstantiateCounter, sb.transBuildCounter,
                                  rb.numBlasActualSizes, rb.numGenActualDatas])])
    finally:
        g.close()
    assert out[0][8][0] >= (capacity or instances) and bool(flags) == (out[0][8][2] > 0)
    for x, y in zip(*out):
        assert x.tobytes() == y.tobytes()


@pytest.mark.parametrize("fmt", ["r16", "r32"])
@pytest.mark.parametrize("w,h", [(1, 1), (2, 1), (1, 3), (2, 2), (3, 5), (64, 7)])
def test_height_map_edges(w, h, fmt):
    """Samples across a height map's edges wrap texel by texel; waves whose
    samples all lie inside read a row's two texels in one load.  Maps of one
    and two texels (every sample wraps, or one in nine does not), odd sizes and
    both formats against the oracle's vertices."""
    rng = np.random.default_rng(10 * w + h)
    heights = rng.random((h, w), np.float32)
    tex = (scene.to_r16(heights), abi.TEXTURE_R16_UNORM) if fmt == "r16" else (heights, abi.TEXTURE_R32_FLOAT)
    geo = scene.grid_patch(12, 12, 4.0, 4.0)
    cam = scene.Camera(eye=(2.0, 3.0, -1.0), center=(2.0, 0.0, 2.0), width=160, height=90, near=0.05, far=100.0)
    host = scene.HostScene([geo], [scene.Instance(0, np.eye(4), displacement_index=0, displacement_scale=0.3)], [tex], cam,
                           3.0, "edges")
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
    assert ref.counters["partTriangleCounter"] > 100
    harness.compare(res, ref)
