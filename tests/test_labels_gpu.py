"""GPU visibility training samples (libnlod nlod_labeler_*) against the CPU
restatement: identical inputs and labels, bit for bit."""
import numpy as np
import pytest
import torch

from neural_lod_amd import synthetic as S

pytestmark = pytest.mark.gpu


def _gpu(tris, res, seed, first, n):
    from neural_lod_amd.labels import VisibilityLabeler
    lb = VisibilityLabeler(torch.from_numpy(np.ascontiguousarray(tris, np.float32)).cuda(), res)
    x, y = lb.sample(n, seed, first)
    torch.cuda.synchronize()
    return lb, x.cpu().numpy(), y.cpu().numpy()


@pytest.mark.parametrize("res", [32, 64])
def test_blob_mesh_matches_oracle(oracle, cuda, res):
    tris = S.blob_mesh(50_000, seed=0)
    print(f"case blob50k res={res}", flush=True)
    lb, x, y = _gpu(tris, res, seed=9, first=12345, n=8192)
    ex, ey, n_occ = oracle.visibility_samples(tris, res, seed=9, first=12345, n=8192)
    assert lb.n_occupied == n_occ
    assert np.array_equal(x, ex), f"{int((x != ex).any(axis=1).sum())} input rows differ"
    assert np.array_equal(y, ey), f"{int((y != ey).sum())} labels differ"
    assert 0 < y.sum() < y.size


def test_bunny_and_grid(oracle, cuda, golden_dir):
    tris = np.load(golden_dir / "bunny_tris.npy")
    lb, x, y = _gpu(tris, 24, seed=1, first=0, n=4096)
    ex, ey, n_occ = oracle.visibility_samples(tris, 24, seed=1, first=0, n=4096)
    assert lb.n_occupied == n_occ
    assert np.array_equal(x, ex) and np.array_equal(y, ey)
    info = oracle.voxinfo(*oracle.mesh_bbox(tris), 24, False, tris.shape[0])
    assert list(lb.grid.bbox_min) == list(info.bbox_min) and list(lb.grid.unit) == list(info.unit)


def test_stream_is_a_function_of_the_index(cuda):
    from neural_lod_amd.labels import VisibilityLabeler
    lb = VisibilityLabeler(torch.from_numpy(S.blob_mesh(10_000, seed=4)).cuda(), 32)
    x, y = lb.sample(3000, seed=77)
    x2, y2 = lb.sample(1000, seed=77, first=1500)
    assert torch.equal(x[1500:2500], x2) and torch.equal(y[1500:2500], y2)
    e = lb.sample(0, seed=77)
    assert e[0].shape == (0, 6)


def test_invalid_arguments(cuda):
    from neural_lod_amd._lib import NlodError
    from neural_lod_amd.labels import VisibilityLabeler
    tris = torch.from_numpy(S.blob_mesh(100, seed=4)).cuda()
    with pytest.raises(NlodError):
        VisibilityLabeler(tris, 0)
    with pytest.raises(NlodError):
        VisibilityLabeler(tris[:0], 16)


@pytest.mark.parametrize("n_lods", [1, 3])
def test_throughput_matches_oracle(oracle, cuda, n_lods):
    from neural_lod_amd.labels import Labeler
    tris = S.blob_mesh(30_000, seed=1)
    print(f"case throughput blob30k res=32 n_lods={n_lods}", flush=True)
    lb = Labeler(torch.from_numpy(tris).cuda(), 32, n_lods)
    x, t, v = lb.throughput(1024, seed=21, first=777, spp=16, max_depth=3, albedo_seed=5)
    torch.cuda.synchronize()
    ex, et, ev, n_occ = oracle.throughput_samples(tris, 32, n_lods, seed=21, first=777, n=1024, spp=16, max_depth=3,
                                                  albedo_seed=5)
    assert [lv["n_occupied"] for lv in lb.levels] == n_occ
    assert np.array_equal(x.cpu().numpy(), ex)
    assert np.array_equal(v.cpu().numpy(), ev)
    assert np.array_equal(t.cpu().numpy(), et), f"{int((t.cpu().numpy() != et).any(axis=1).sum())} targets differ"
    assert 0 < ev.mean() < 1 and et.max() > 0


@pytest.mark.parametrize("n,spp,max_depth", [(1, 5, 3), (5, 1, 1), (63, 3, 9), (4097, 2, 2)])
def test_throughput_block_edges(oracle, cuda, n, spp, max_depth):
    """Blocks that are not full, on lists of every group width: 4 lanes (up to 8
    triangles), 16 (up to 32), 64, and 64 with triangles beyond the 128 kept in
    registers.  The stream, and so every bit, is the oracle's."""
    from neural_lod_amd.labels import Labeler
    tris = S.blob_mesh(20_000, seed=6)
    print(f"case throughput edges n={n} spp={spp} depth={max_depth}", flush=True)
    lb = Labeler(torch.from_numpy(tris).cuda(), 64, 4)
    mean = [lv["n_list_entries"] / lv["n_occupied"] for lv in lb.levels]
    assert mean[0] < 8 and mean[-1] > 32  # of lists of 1 to 427 triangles on the coarsest level
    x, t, v = lb.throughput(n, seed=3, first=10 ** 9, spp=spp, max_depth=max_depth, albedo_seed=8)
    torch.cuda.synchronize()
    ex, et, ev, _ = oracle.throughput_samples(tris, 64, 4, seed=3, first=10 ** 9, n=n, spp=spp, max_depth=max_depth,
                                              albedo_seed=8)
    assert np.array_equal(x.cpu().numpy(), ex)
    assert np.array_equal(v.cpu().numpy(), ev)
    assert np.array_equal(t.cpu().numpy(), et), f"{int((t.cpu().numpy() != et).any(axis=1).sum())} targets differ"


@pytest.mark.parametrize("n", [32769, 70001])
def test_throughput_every_sample_once(cuda, n):
    """The waves of a block take its samples (32 and 64 of them at these sizes on
    256 CUs) from one counter: every row is written, with what calls of 777 samples,
    whose blocks hold 4, write for the same indices.  The last block is not full."""
    from neural_lod_amd.labels import Labeler
    tris = S.blob_mesh(20_000, seed=6)
    print(f"case throughput every sample n={n}", flush=True)
    lb = Labeler(torch.from_numpy(tris).cuda(), 64, 4)
    out = tuple(torch.full(shape, float("nan"), device="cuda") for shape in ((n, 10), (n, 3), (n,)))
    lb.throughput(n, seed=31, first=5, spp=2, max_depth=3, albedo_seed=8, out=out)
    for first in range(0, n, 777):
        m = min(777, n - first)
        part = lb.throughput(m, seed=31, first=5 + first, spp=2, max_depth=3, albedo_seed=8)
        for whole, p in zip(out, part):
            assert torch.equal(whole[first:first + m], p), f"samples {first} .. {first + m}"


def test_throughput_invalid_arguments(cuda):
    from neural_lod_amd._lib import NlodError
    from neural_lod_amd.labels import Labeler
    tris = torch.from_numpy(S.blob_mesh(1000, seed=4)).cuda()
    with pytest.raises(NlodError, match="divisible"):
        Labeler(tris, 30, 3)
    lb = Labeler(tris, 16, 2)
    with pytest.raises(NlodError):
        lb.throughput(8, seed=1, spp=0)
