"""Weight and bias gradients (k_wgrad_rows, k_conv_wgrad, k_wgrad_finish) of the
five convolutions of the finest level, with up to 192 inputs and many parts of the
nodes, against sums in float64 of the same bfloat16 operands.

The network is set to pass the output gradient through unchanged: every
convolution of that level but the first is the identity on its own channels (the
decoder's first one on the skip channels), those below are zero, and the first
one's bias keeps its ReLU open.  So each of the five has the caller's output
gradient, rounded to bfloat16, in its first three channels and 0 in the others.

An entry is a sum of products that are exact in float32, added up 32 at a time by
the matrix cores, by 4 waves in each part and then over the parts: its roundings
number at most those additions, each at most 2^-24 of the sum of the products'
magnitudes (the bias: 8 nodes a thread and step, 16 threads, then the workgroups)."""
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def center(cout, cin, pairs):
    w = torch.zeros(cout, 27, cin)
    for o, c in pairs:
        w[o, 13, c] = 1.0
    return w


def passing_params(table, gen):
    p = []
    for q, (cin, cout, lev) in enumerate(table):
        w, b = torch.zeros(cout, 27, cin), torch.zeros(cout)
        if q == 0:
            w = 0.02 * torch.randn(cout, 27, cin, generator=gen)
            b = torch.full((cout,), 16.0)
        elif lev == 0:
            w = center(cout, cin, [(o, cin - 16 + o) for o in range(cout)])
        p += [w.reshape(-1), b]
    return torch.cat(p)


@pytest.mark.parametrize("nodes,n_in", [((9, 9, 9), 100), ((33, 33, 33), 51), ((41, 25, 17), 192), ((17, 57, 33), 20)])
def test_finest_level_gradients_match_float64_sums(nodes, n_in):
    from alamo_amd.learned import UNet
    net = UNet(nodes, n_in, 3, seed=None)
    table = net.conv_table()
    gen = torch.Generator().manual_seed(6)
    net.set_params(passing_params(table, gen).cuda())
    shape = net.field_shape
    net.forward(torch.randn((n_in,) + shape, generator=gen).cuda())
    dout = torch.randn((3,) + shape, generator=gen)
    grad = net.backward(dout.cuda())[0].double().cpu()
    dz = dout.bfloat16().double().reshape(3, -1)
    nz, ny, nx = shape
    groups = ny * nz * ((nx + 7) // 8)
    o = 0
    for q, (cin, cout, lev) in enumerate(table):
        g_w, g_b = grad[o:o + 27 * cin * cout].reshape(cout, 27, cin), grad[o + 27 * cin * cout:o + (27 * cin + 1) * cout]
        o += (27 * cin + 1) * cout
        if lev > 0:
            continue
        x, y = net.tape(q)
        if q == 0:
            assert bool((y > 0).all())  # the ReLU is open everywhere
        xp = torch.nn.functional.pad(x.double().cpu(), (1,) * 6)
        total = -(-groups // 4)
        nchunk = max(1, min(256 // (-(-cin // 16) * -(-cout // 16)), total // 4))
        adds = 32 * -(--(-total // nchunk) // 4) + 4 + nchunk
        worst = 0.0
        for t in range(27):
            k, j, i = t // 9, t // 3 % 3, t % 3
            xt = xp[:, k:k + nz, j:j + ny, i:i + nx].reshape(cin, -1)
            want, mag = dz @ xt.T, dz.abs() @ xt.abs().T
            err = (g_w[:3, t] - want).abs()
            worst = max(worst, float((err / (adds * 2.0 ** -24 * mag).clamp(min=1e-30)).max()))
            assert bool((g_w[3:, t] == 0).all()), (q, t)
        blocks = min(256, -(-groups * 16 // 256))
        adds_b = 8 * -(-groups // (16 * blocks)) + 16 + blocks
        err_b = float(((g_b[:3] - dz.sum(1)).abs() / (adds_b * 2.0 ** -24 * dz.abs().sum(1))).max())
        print(f"{nodes} {n_in} conv {q} {cin}->{cout}: error / bound {worst:.3f}, bias {err_b:.3f}")
        assert worst <= 1 and err_b <= 1, q
        assert bool((g_b[3:] == 0).all())
