"""The FP16 encoding's two forms give the same features, bit for bit: large batches
encode the coarse levels from tables in LDS (from 263566 queries of the visibility
network, 183784 of the throughput network, 377778 of the two-point visibility
network), smaller ones take every level row by row."""
import pytest
import torch

from neural_lod_amd import configs, synthetic
from neural_lod_amd.tcnn import FP16, NetworkWithInputEncoding

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,n", [
    *((name, n) for name in ("visibility", "throughput", "reference_visibility") for n in (299999, 300000, 300017)),
    ("visibility", 263565), ("visibility", 263566), ("throughput", 183783), ("throughput", 183784),
    ("reference_visibility", 377777), ("reference_visibility", 377778), ("reference_visibility", 400001)])
def test_large_batch_features_equal_small_batches(cuda, name, n):
    cfg = configs.ALL[name]
    net = NetworkWithInputEncoding(cfg["n_input_dims"], cfg["n_output_dims"], cfg["encoding"], cfg["network"], FP16)
    print(f"case encode {name} n={n}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(3)
    net.set_params(torch.rand(net.n_params, generator=g, device="cuda") - 0.5)
    q = synthetic.throughput_queries(n, seed=1) if name == "throughput" else synthetic.visibility_queries(n, 1)
    x = torch.from_numpy(q).cuda()
    x[:2, :3] = torch.tensor([[0.0, 1.0, 0.0], [1.0, 0.0, 1.0]], device="cuda")  # the grid's corners
    whole = net.encode_fragments(x)
    assert whole.view(torch.float16).isfinite().all()
    row = whole.numel() // ((n + 15) // 16)  # bytes of a 16-query tile
    for first in (0, 131072, n // 16 * 16 - 1600):
        part = x[first:first + 1600 + (n % 16 if first > 131072 else 0)].contiguous()
        got = net.encode_fragments(part)
        assert torch.equal(got, whole[first // 16 * row:first // 16 * row + got.numel()]), f"from {first}"
