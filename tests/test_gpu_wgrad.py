"""The weight and bias gradients (k_wgrad_rows, k_conv_wgrad,
k_wgrad_finish) of the output convolution against sums in float64 of the same
bfloat16 operands: its output gradient is the caller's, rounded, and its input
the forward tape, so nothing but the float32 sums differs.  Each sum has at most
5,000 terms of either sign and each rounding is 2^-24 of a partial sum, so the
error stays below 1e-5 of the largest entry.  Grids whose rows fill their last
group of 8 nodes by one node, that have fewer groups than one workgroup's steps,
and unequal axes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("nodes", [(9, 9, 9), (17, 9, 25), (25, 17, 9), (9, 25, 17)])
def test_output_layer_gradient_matches_float64_sums(nodes):
    from alamo_amd.learned import UNet
    net = UNet(nodes, 5, 3, seed=3)
    g = torch.Generator(device="cuda").manual_seed(1)
    shape = net.field_shape
    net.forward(torch.randn((5,) + shape, device="cuda", generator=g))
    dout = torch.randn((3,) + shape, device="cuda", generator=g)
    grad = net.backward(dout)[0].double().cpu().numpy()
    last = len(net.conv_table()) - 1
    x = net.tape(last)[0].double().cpu().numpy()
    dz = dout.bfloat16().double().cpu().numpy()
    xp = np.pad(x, ((0, 0), (1, 1), (1, 1), (1, 1)))
    nz, ny, nx = shape
    want = np.empty((3, 27, x.shape[0]))
    for t in range(27):
        k, j, i = t // 9, t // 3 % 3, t % 3
        want[:, t] = np.einsum("ozyx,czyx->oc", dz, xp[:, k:k + nz, j:j + ny, i:i + nx])
    n = want.size
    got_w, got_b = grad[-n - 3:-3].reshape(want.shape), grad[-3:]
    assert np.abs(got_w - want).max() < 1e-5 * np.abs(want).max()
    bias = dz.sum(axis=(1, 2, 3))
    assert np.abs(got_b - bias).max() < 1e-5 * max(np.abs(bias).max(), np.abs(dz).max())
