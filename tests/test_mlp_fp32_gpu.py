"""FP32 network passes at the edges of their tiles (16 queries per wave, 4
waves per block; 64 columns of the first matrix at a time), against float64.

Every value is a sum of K or W products of FP32 values, layer after layer, so
with L layers of at most 160 terms the error is below
L 160 2^-24 sum |a b| of the last sums; with random signs the sums are about
1/sqrt(160) of that, and rounding errors also add as a random walk: 1e-5 of the
largest value leaves a factor of about ten."""
import numpy as np
import pytest
import torch

from neural_lod_amd.tcnn import FP32, NetworkWithInputEncoding

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width,n_hidden,n_in,n_out", [(16, 1, 3, 1), (32, 2, 40, 3), (64, 1, 64, 16), (64, 4, 66, 5),
                                                       (128, 3, 150, 16)])
@pytest.mark.parametrize("n", [1, 15, 17, 63, 64, 65, 129, 5003, 40001])
def test_passes(cuda, width, n_hidden, n_in, n_out, n):
    print(f"case mlp fp32 width={width} hidden={n_hidden} in={n_in} out={n_out} n={n}", flush=True)
    net = NetworkWithInputEncoding(n_in, n_out, {"otype": "Identity"},
                                   {"otype": "FullyFusedMLP", "activation": "None", "output_activation": "None",
                                    "n_neurons": width, "n_hidden_layers": n_hidden}, FP32)
    rng = np.random.default_rng(width + n)
    p = torch.from_numpy((rng.standard_normal(net.n_params) * (1.5 / np.sqrt(width))).astype(np.float32)).cuda()
    x = torch.from_numpy(rng.uniform(-1, 1, (n, n_in)).astype(np.float32)).cuda()
    d = torch.from_numpy(rng.standard_normal((n, n_out)).astype(np.float32)).cuda()
    net.set_params(p)
    out, ctx = net.forward(x)
    assert torch.equal(out, net.inference(x))
    dx = net.backward(ctx, x, d, input_gradients=True)[1]

    k = net.encoded_width
    xs = x.cpu().double().requires_grad_()
    h = torch.cat([xs, torch.ones(n, k - n_in, dtype=torch.float64)], 1)
    off = 0
    for r, c in [(width, k)] + [(width, width)] * (n_hidden - 1) + [(n_out, width)]:
        h = h @ p[off:off + r * c].cpu().double().reshape(r, c).t()
        off += r * c
    h.backward(d.cpu().double())
    for what, got, ref in (("output", out, h.detach()), ("input gradient", dx, xs.grad)):
        err, scale = (got.cpu().double() - ref).abs().max().item(), ref.abs().max().item()
        assert err <= 1e-5 * scale, f"{what}: error {err:.3e}, largest value {scale:.3e}"
