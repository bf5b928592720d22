"""FP16 network passes at the limits of their blocks: 128-wide networks at the sizes
where the block's shape changes (single tiles while 8 waves a CU cover the batch,
32768 queries on 256 CUs; then pairs of tiles, on 8 waves for 32 inputs and 12 for
more; single tiles on 4 waves for shallow networks, with 1 to 4 chunks of inputs
loaded ahead), and a backward pass whose weights fill the LDS to the last byte.

Against the MLP with FP16 weights and features, rounded to FP16 where the kernels
round and summed in float64: a layer's FP32 sums may round to the next FP16 value
(2^-11 relative), so the outputs, sums of 128 such terms, agree within 2e-3 of
the largest, and gradients within 2e-3 in the 2-norm."""
import numpy as np
import pytest
import torch

from neural_lod_amd.tcnn import FP16, NetworkWithInputEncoding

pytestmark = pytest.mark.gpu


def _net(width, n_hidden, n_in, n_out, activation):
    return NetworkWithInputEncoding(n_in, n_out, {"otype": "Identity"},
                                    {"otype": "FullyFusedMLP", "activation": activation, "output_activation": "None",
                                     "n_neurons": width, "n_hidden_layers": n_hidden}, FP16)


def _h(t):
    return t.half().double()


def _matrices(net, p, width, n_hidden):
    shapes = [(width, net.encoded_width)] + [(width, width)] * (n_hidden - 1) + [(net.padded_output_width, width)]
    mats, off = [], 0
    for r, c in shapes:
        mats.append(_h(p[off:off + r * c].reshape(r, c)))
        off += r * c
    return mats


def _forward(net, mats, x, relu):
    """Activations (features first) and outputs, float64."""
    pad = torch.ones(x.shape[0], net.encoded_width - x.shape[1], device=x.device)
    hs = [_h(torch.cat([x, pad], 1))]
    for m in mats[:-1]:
        z = hs[-1] @ m.t()
        hs.append(_h((z.relu() if relu else z).float()))
    return hs, hs[-1] @ mats[-1].t()


def _inputs(net, n, n_in, width, seed):
    rng = np.random.default_rng(seed)
    p = torch.from_numpy((rng.standard_normal(net.n_params) / np.sqrt(width)).astype(np.float32)).cuda()
    x = torch.from_numpy(rng.uniform(-1, 1, (n, n_in)).astype(np.float32)).cuda()
    return p, x


@pytest.mark.parametrize("n_in,n_hidden,activation", [(30, 4, "None"), (150, 3, "None"), (30, 1, "None"), (30, 1, "ReLU"),
                                                      (50, 2, "ReLU"), (90, 1, "ReLU"), (120, 1, "ReLU")])
@pytest.mark.parametrize("n", [1, 100, 32768, 32769, 40007])
def test_wide_forward(cuda, n_in, n_hidden, activation, n):
    print(f"case mlp fp16 in={n_in} hidden={n_hidden} {activation} n={n}", flush=True)
    net = _net(128, n_hidden, n_in, 5, activation)
    p, x = _inputs(net, n, n_in, 128, n)
    net.set_params(p)
    ref = _forward(net, _matrices(net, p, 128, n_hidden), x, activation == "ReLU")[1][:, :5]
    err, scale = (net.inference(x).double() - ref).abs().max().item(), ref.abs().max().item()
    assert err <= 2e-3 * scale, f"error {err:.3e}, largest value {scale:.3e}"


@pytest.mark.parametrize("width,n_hidden,n_in", [(128, 5, 96), (64, 16, 288)])
def test_backward_weights_fill_the_lds(cuda, width, n_hidden, n_in):
    """Forward weights of 156 and 158 KB, backward weights of 160 KB."""
    print(f"case mlp fp16 backward width={width} hidden={n_hidden} in={n_in}", flush=True)
    net = _net(width, n_hidden, n_in, 5, "None")
    n = 1003
    p, x = _inputs(net, n, n_in, width, 3)
    d = torch.from_numpy(np.random.default_rng(4).standard_normal((n, 5)).astype(np.float32)).cuda()
    net.set_params(p)
    out, ctx = net.forward(x)
    got = net.backward(ctx, x, d)[0].double()
    mats = _matrices(net, p, width, n_hidden)
    hs, _ = _forward(net, mats, x, False)
    delta = torch.zeros(n, net.padded_output_width, dtype=torch.float64, device="cuda")
    delta[:, :5] = _h(d)
    off = got.numel()
    for layer in range(n_hidden, -1, -1):
        ref = delta.t() @ hs[layer]
        off -= ref.numel()
        g = got[off:off + ref.numel()].reshape(ref.shape)
        assert (g - ref).norm() <= 2e-3 * ref.norm(), f"matrix {layer}"
        delta = _h((delta @ mats[layer]).float())
