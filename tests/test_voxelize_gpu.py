"""GPU voxelizer (libnlod nlod_voxelize*) vs the CPU oracle: bit-exact tables.

Every case runs the default kernel choice and both kernel paths (direct:
one triangle per lane with global atomics; tiled: LDS tiles of voxel rows,
with triangles spanning many tiles handed to the direct kernel)."""
import numpy as np
import pytest
import torch

from neural_lod_amd import synthetic as S

pytestmark = pytest.mark.gpu


def _gpu_table(tris, res, **kw):
    from neural_lod_amd import voxelizer as V
    t = torch.from_numpy(np.ascontiguousarray(tris, np.float32)).cuda()
    table, info = V.voxelize(t, res, **kw)
    torch.cuda.synchronize()
    return table.cpu().numpy().view(np.uint32), info


def _assert_same(gpu, cpu, what):
    diff = np.nonzero(gpu != cpu)[0]
    assert diff.size == 0, f"{what}: {diff.size} words differ, first at {diff[:5]}"


def _check_paths(tris, res, cpu, what, **kw):
    for path in ("auto", "direct", "tiled"):
        gpu, info = _gpu_table(tris, res, path=path, **kw)
        _assert_same(gpu, cpu, f"{what} path={path}")
    return info


@pytest.mark.parametrize("solid", [False, True])
@pytest.mark.parametrize("pad", [False, True])
def test_blob_mesh_200k_256(oracle, cuda, solid, pad):
    tris = S.blob_mesh(200_000, seed=0)
    print(f"case blob200k G=256 solid={solid} pad={pad}", flush=True)
    cpu, cinfo = oracle.voxelize(tris, 256, solid=solid, pad=pad)
    ginfo = _check_paths(tris, 256, cpu, f"blob solid={solid} pad={pad}", solid=solid, pad=pad)
    assert list(ginfo.unit) == list(cinfo.unit)
    assert list(ginfo.bbox_min) == list(cinfo.bbox_min)


@pytest.mark.parametrize("res", [64, 128, 256, 512, 100])
@pytest.mark.parametrize("solid", [False, True])
def test_bunny(oracle, cuda, golden_dir, res, solid):
    tris = np.load(golden_dir / "bunny_tris.npy")
    print(f"case bunny G={res} solid={solid}", flush=True)
    cpu, _ = oracle.voxelize(tris, res, solid=solid)
    _check_paths(tris, res, cpu, f"bunny res={res} solid={solid}", solid=solid)


@pytest.mark.parametrize("solid", [False, True])
def test_morton(oracle, cuda, golden_dir, solid):
    tris = np.load(golden_dir / "bunny_tris.npy")
    cpu, _ = oracle.voxelize(tris, 128, solid=solid, morton=True)
    gpu, _ = _gpu_table(tris, 128, solid=solid, morton=True)
    _assert_same(gpu, cpu, "morton")


def test_closed_shapes(oracle, cuda):
    for tris in (S.box_mesh(), S.sphere_mesh(32, 64)):
        for res in (48, 64, 257):
            for solid in (False, True):
                cpu, _ = oracle.voxelize(tris, res, solid=solid)
                _check_paths(tris, res, cpu, f"closed res={res} solid={solid}", solid=solid)


def test_edge_cases(oracle, cuda):
    rng = np.random.default_rng(3)
    # one triangle; degenerate (zero-area, collinear, repeated vertex) triangles
    one = rng.uniform(0, 1, size=(1, 9)).astype(np.float32)
    degen = np.stack([
        np.array([0.1, 0.1, 0.1, 0.5, 0.5, 0.5, 0.9, 0.9, 0.9], np.float32),  # collinear
        np.array([0.2, 0.3, 0.4, 0.2, 0.3, 0.4, 0.7, 0.1, 0.6], np.float32),  # repeated vertex
        np.array([0.3, 0.3, 0.3] * 3, np.float32),  # point
    ])
    mixed = np.concatenate([rng.uniform(0, 1, size=(300, 9)).astype(np.float32), degen])
    axis_aligned = S.box_mesh((0.25, 0.25, 0.25), (0.75, 0.75, 0.75))  # faces on voxel boundaries
    for name, tris in (("one", one), ("degenerate", mixed), ("axis-aligned", axis_aligned)):
        for res in (16, 64):
            for solid in (False, True):
                for pad in (False, True):
                    cpu, _ = oracle.voxelize(tris, res, solid=solid, pad=pad)
                    _check_paths(tris, res, cpu, f"{name} res={res} solid={solid} pad={pad}", solid=solid,
                                 pad=pad)


@pytest.mark.parametrize("scale", [1e-15, 1e-6, 1e6])
def test_scaled_meshes(oracle, cuda, scale):
    """Tiny and large coordinates (the plane-slab pruning of the surface test
    switches itself off below its underflow-safe range)."""
    tris = (S.blob_mesh(5000, seed=4).astype(np.float64) * scale + 3.0 * scale).astype(np.float32)
    for res in (64, 96):
        for solid in (False, True):
            cpu, _ = oracle.voxelize(tris, res, solid=solid)
            _check_paths(tris, res, cpu, f"scale={scale} res={res} solid={solid}", solid=solid)


def test_non_finite_and_outside_box(oracle, cuda):
    """Explicit voxinfo smaller than the mesh, plus NaN/inf triangles: in-bounds and equal."""
    from neural_lod_amd import voxelizer as V
    rng = np.random.default_rng(9)
    tris = rng.uniform(-0.5, 1.5, size=(2000, 9)).astype(np.float32)
    tris[5, 2] = np.nan
    tris[7, 4] = np.inf
    for solid in (False, True):
        info_c = oracle.voxinfo([0, 0, 0], [1, 1, 1], 32, False, tris.shape[0])
        cpu, _ = oracle.voxelize(tris, 32, solid=solid, info=info_c)
        info_g = V.voxinfo_from_bbox([0, 0, 0], [1, 1, 1], 32)
        _check_paths(tris, 32, cpu, f"outside-box solid={solid}", solid=solid, info=info_g)


@pytest.mark.parametrize("res", [96, 256, 333])
@pytest.mark.parametrize("solid", [False, True])
def test_mixed_triangle_sizes(oracle, cuda, res, solid):
    """Small triangles (tiled) mixed with ones spanning many tiles (direct),
    on aligned (96, 256) and unaligned (333) row lengths."""
    big = np.concatenate([S.box_mesh((0.05, 0.05, 0.05), (0.95, 0.95, 0.95)), S.sphere_mesh(6, 8)])
    tris = np.concatenate([S.blob_mesh(20_000, seed=2), big]).astype(np.float32)
    print(f"case mixed G={res} solid={solid}", flush=True)
    cpu, _ = oracle.voxelize(tris, res, solid=solid)
    _check_paths(tris, res, cpu, f"mixed res={res} solid={solid}", solid=solid)


def test_empty_mesh_and_accumulate(cuda):
    from neural_lod_amd import voxelizer as V
    info = V.voxinfo_from_bbox([0, 0, 0], [1, 1, 1], 64)
    out = torch.full((V.table_words(64),), -1, dtype=torch.int32, device="cuda")
    empty = torch.empty((0, 9), dtype=torch.float32, device="cuda")
    V.voxelize(empty, 64, info=info, out=out)
    torch.cuda.synchronize()
    assert int(out.abs().sum()) == 0
    tri = torch.tensor([[0.1, 0.1, 0.1, 0.9, 0.1, 0.1, 0.1, 0.9, 0.9]], device="cuda")
    a, _ = V.voxelize(tri, 64, info=info)
    tri2 = torch.tensor([[0.5, 0.5, 0.9, 0.9, 0.5, 0.1, 0.5, 0.9, 0.2]], device="cuda")
    c, _ = V.voxelize(tri2, 64, info=info)
    from neural_lod_amd.voxelizer import _flags
    import ctypes as C
    for path in ("direct", "tiled"):
        b = a.clone()
        V._lib.call("nlod_voxelize", C.c_void_p(torch.cuda.current_stream().cuda_stream), C.byref(info),
                    C.c_void_p(tri2.data_ptr()), C.c_void_p(b.data_ptr()), _flags(False, False, False, True, path))
        torch.cuda.synchronize()
        assert torch.equal(b, a | c), path


def test_invalid_arguments(cuda):
    from neural_lod_amd import voxelizer as V
    from neural_lod_amd._lib import NlodError
    tri = torch.rand(4, 9, device="cuda")
    with pytest.raises(NlodError, match="power-of-two"):
        V.voxelize(tri, 100, morton=True)
    with pytest.raises(NlodError):
        V.voxelize(tri, 0)
    with pytest.raises(ValueError):
        V.voxelize(tri, 64, path="fast")


@pytest.mark.parametrize("n_tri,at", [(682, 681), (683, 682), (2048, 2047), (349_526, 0), (349_526, 349_525),
                                      (1_000_000, 700_001)])
def test_mesh_bbox_block_edges(cuda, n_tri, at):
    """The box is found in whichever block holds the extreme triangle: around
    one tile of 6144 floats (682.67 triangles), at three whole tiles, past the
    tiles of one sweep of two blocks per CU (349,525 triangles on 256 CUs), and
    with infinities beside the finite coordinates."""
    from neural_lod_amd import voxelizer as V
    rng = np.random.default_rng(n_tri)
    tris = rng.normal(size=(n_tri, 9)).astype(np.float32)
    tris[at, 1] = -1e4
    tris[at, 3] = np.inf
    tris[at, 8] = 1e4
    print(f"case bbox n_tri={n_tri} at={at}", flush=True)
    mn, mx = V.mesh_bbox(torch.from_numpy(tris).cuda())
    v = tris.reshape(-1, 3)
    np.testing.assert_array_equal(mn, v.min(axis=0))
    np.testing.assert_array_equal(mx, v.max(axis=0))


def test_threads_on_one_stream(cuda):
    """Threads that voxelize different meshes on one stream: the launches of a tiled
    job share scratch with the stream's other jobs, whose launches must not come
    between them; each thread gets the table and box that it gets alone."""
    import threading

    from neural_lod_amd import voxelizer as V
    jobs = [(torch.from_numpy(S.blob_mesh(n, seed=n)).cuda(), res) for n, res in
            ((60_000, 128), (5_000, 96), (30_000, 256))]
    want = [V.voxelize(t, res, solid=True, path="tiled") for t, res in jobs]
    torch.cuda.synchronize()
    print("case voxelize threads", flush=True)
    outs = [[torch.full_like(w[0], -1) for _ in range(20)] for w in want]
    wrong = []

    def work(k):
        for out in outs[k]:
            info = V.voxelize(jobs[k][0], jobs[k][1], solid=True, path="tiled", out=out)[1]
            if list(info.bbox_min) != list(want[k][1].bbox_min):
                wrong.append(k)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(len(jobs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not wrong
    for k, w in enumerate(want):
        assert all(torch.equal(out, w[0]) for out in outs[k]), f"mesh {k}"


def test_mesh_bbox_threads_on_one_stream(cuda):
    """Threads that ask for the boxes of different meshes on one stream: each gets
    its own mesh's box, in whatever order their kernels and copies are enqueued."""
    import threading

    from neural_lod_amd import voxelizer as V
    sizes = (200_000, 700, 40_000, 1)
    meshes = [torch.rand((n, 9), device="cuda") * (k + 1) + 10.0 * k for k, n in enumerate(sizes)]
    want = [(m.view(-1, 3).amin(0).cpu().numpy(), m.view(-1, 3).amax(0).cpu().numpy()) for m in meshes]
    print("case bbox threads", flush=True)
    wrong = []

    def ask(k):
        for _ in range(200):
            mn, mx = V.mesh_bbox(meshes[k])
            if not (np.array_equal(mn, want[k][0]) and np.array_equal(mx, want[k][1])):
                wrong.append(k)

    threads = [threading.Thread(target=ask, args=(k,)) for k in range(len(sizes))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong


@pytest.mark.parametrize("n_tri", [1, 2, 3, 4, 5, 7, 1000, 200_001])
@pytest.mark.parametrize("offset", [0, 1])
def test_mesh_bbox(cuda, n_tri, offset):
    """Device bounding box vs numpy: chunked float4 path (16-byte aligned array),
    float-by-float tail, and a 4-byte offset array (float-by-float throughout);
    NaN coordinates are skipped."""
    from neural_lod_amd import voxelizer as V
    rng = np.random.default_rng(n_tri + offset)
    tris = rng.normal(size=(n_tri, 9)).astype(np.float32) * 3.0 + 1.0
    if n_tri > 2:
        tris[1, 4] = np.nan  # a y coordinate
        tris[-1, 0] = np.nan  # an x coordinate in the tail
    flat = torch.zeros(n_tri * 9 + offset, dtype=torch.float32, device="cuda")
    flat[offset:] = torch.from_numpy(tris.reshape(-1)).cuda()
    t = flat[offset:].view(n_tri, 9)
    assert (t.data_ptr() % 16 == 0) == (offset == 0)
    print(f"case bbox n_tri={n_tri} offset={offset}", flush=True)
    mn, mx = V.mesh_bbox(t)
    v = tris.reshape(-1, 3)
    np.testing.assert_array_equal(mn, np.nanmin(v, axis=0))
    np.testing.assert_array_equal(mx, np.nanmax(v, axis=0))
