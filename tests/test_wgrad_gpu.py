"""GPU weight gradients at the sizes where their split over 64 x 64 tiles and
query chunks can go wrong: batches around the 16- and 32-query steps, matrices
narrower than a tile, wider than one, and with a remainder.

FP32: against torch in float64, without a ReLU: a pre-activation within rounding
of 0 (about 1e-6 of them) may take the other side in FP32 and then adds or drops
a whole term |delta h|, which no rounding bound covers.  A weight's gradient is a sum over the batch of
products; with products and sums in FP32 it is off by at most
(N + L W) 2^-23 sum_q |delta h|, here bounded by 1e-5 of the matrix's largest
entry times sqrt(N) (the terms' magnitudes against their sum's).
FP16: the gradient of n queries against that of a longer batch whose further
output gradients are zero, so both sum the same products, in another order."""
import numpy as np
import pytest
import torch

from neural_lod_amd import configs
from neural_lod_amd.tcnn import FP16, FP32, NetworkWithInputEncoding

pytestmark = pytest.mark.gpu


def _net(width, n_hidden, n_in, n_out, precision, activation="ReLU"):
    return NetworkWithInputEncoding(n_in, n_out, {"otype": "Identity"},
                                    {"otype": "FullyFusedMLP", "activation": activation, "output_activation": "None",
                                     "n_neurons": width, "n_hidden_layers": n_hidden}, precision)


def _case(net, n, seed):
    rng = np.random.default_rng(seed)
    p = (rng.standard_normal(net.n_params) * (1.5 / np.sqrt(net.network_width))).astype(np.float32)
    x = rng.uniform(-1, 1, (n, net.n_input_dims)).astype(np.float32)
    d = rng.standard_normal((n, net.n_output_dims)).astype(np.float32)
    return (torch.from_numpy(t).cuda() for t in (p, x, d))


def _gradient(net, x, d):
    out, ctx = net.forward(x)
    return net.backward(ctx, x, d)[0]


@pytest.mark.parametrize("width,n_hidden,n_in,n_out", [(16, 1, 3, 1), (32, 2, 40, 3), (64, 3, 66, 5),
                                                       (128, 2, 150, 16)])
@pytest.mark.parametrize("n", [1, 15, 16, 17, 127, 129, 5003])
def test_fp32(cuda, width, n_hidden, n_in, n_out, n):
    print(f"case wgrad fp32 width={width} hidden={n_hidden} in={n_in} out={n_out} n={n}", flush=True)
    net = _net(width, n_hidden, n_in, n_out, FP32, "None")
    p, x, d = _case(net, n, width + n)
    net.set_params(p)
    got = _gradient(net, x, d).cpu().double()
    k = net.encoded_width
    shapes = [(width, k)] + [(width, width)] * (n_hidden - 1) + [(net.padded_output_width, width)]
    mats, off = [], 0
    for r, c in shapes:
        mats.append(p[off:off + r * c].cpu().double().reshape(r, c).requires_grad_())
        off += r * c
    h = torch.cat([x.cpu().double(), torch.ones(n, k - n_in, dtype=torch.float64)], 1)
    for m in mats[:-1]:
        h = h @ m.t()
    (h @ mats[-1].t())[:, :n_out].backward(d.cpu().double())
    off = 0
    for i, m in enumerate(mats):
        g = got[off:off + m.numel()].reshape(m.shape)
        off += m.numel()
        err, scale = (g - m.grad).abs().max().item(), m.grad.abs().max().item()
        assert err <= 1e-5 * np.sqrt(n) * scale, f"matrix {i}: error {err:.3e}, largest entry {scale:.3e}"


@pytest.mark.parametrize("name", ["visibility", "reference_visibility", "reference_throughput", "width32"])
def test_fp16(cuda, name):
    if name == "width32":
        net = _net(32, 2, 40, 3, FP16)
    else:
        cfg = configs.ALL[name]
        net = NetworkWithInputEncoding(cfg["n_input_dims"], cfg["n_output_dims"], cfg["encoding"], cfg["network"], FP16)
    n_all = 3000
    p, x, d = _case(net, n_all, 5)
    x = (x + 1) / 2
    net.set_params(p)
    n_net = net.n_network_params
    for n in (1, 15, 17, 32, 33, 511, 2999):
        print(f"case wgrad fp16 {name} n={n}", flush=True)
        masked = torch.where(torch.arange(n_all, device="cuda")[:, None] < n, d, torch.zeros_like(d))
        ref = _gradient(net, x, masked)[:n_net].double()
        got = _gradient(net, x[:n].contiguous(), d[:n].contiguous())[:n_net].double()
        assert torch.isfinite(got).all() and ref.norm() > 0
        # sums of n FP32 terms in two orders
        assert (got - ref).norm() <= 1e-6 * np.sqrt(n) * ref.norm(), f"n={n}"
