"""The FP32 isotropic rows (k_stencil_iso, k_stencil_slab): residual and one
Jacobi sweep against the oracle on the same FP32-rounded inputs (2e-6 of the
result's max-norm, the bar of the FP32 kernels), and the diagonal that a sweep
divides by.  On tiled boxes in chunks of 16 planes, the default and 1 plane, on a
per-node box, with and without periodic axes and the uniform flag.

The diagonal: a sweep of x = 0 is w b / D, and D is the FP64 diagonal rounded
once, so with the roundings of w b and of the quotient the sweep is off by at
most 3 2^-24 of itself, to first order (asked: 3.1).  A diagonal summed in FP32
from rounded moduli and spacings exceeds that."""
import numpy as np
import pytest

from alamo_amd import model as M
from oracle import oracle as O

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
from test_oracle_periodic import periodize, rand_case  # noqa: E402

TILED = (70, 52, 46)  # 69 x 51 x 45 interior nodes: 3 x 7 tiles a plane
BY_NODE = (20, 18, 22)


def r32(a):
    return np.asarray(a, dtype=np.float32).astype(np.float64)


def dev32(a):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).cuda()


def operator(n_cell, per, uniform, seed):
    from alamo_amd import elastic as el
    C, bc, u, dx = rand_case(M.ISOTROPIC, n_cell, per, seed)
    if uniform:
        C = np.broadcast_to(C[:, :1, :1, :1], C.shape)
    C = r32(np.ascontiguousarray(C))
    op = el.ElasticOperator(n_cell, dx, M.ISOTROPIC)
    op.SetPeriodic(per)
    op.SetBC(bc)
    op.SetUniform(uniform)
    op.SetModel(torch.from_numpy(C).cuda())
    return op, C, bc, r32(u), dx


@pytest.mark.parametrize("n_cell,target", [(TILED, "1"), (TILED, None), (TILED, "100000"), (BY_NODE, None)])
@pytest.mark.parametrize("per,uniform", [((0, 0, 0), False), ((0, 0, 0), True), ((0, 1, 0), False), ((1, 0, 1), False)])
def test_fp32_residual_and_sweep_match_oracle(per, uniform, n_cell, target, monkeypatch):
    if target:
        monkeypatch.setenv("ALAMO_EL_TILE_TARGET", target)
    op, C, bc, u, dx = operator(n_cell, per, uniform, 7)
    b = r32(periodize(np.random.default_rng(8).standard_normal(u.shape), per))
    with O.periodic(per):
        f = O.fapply(u, C, M.ISOTROPIC, bc, dx, uniform=uniform)
        D = O.diagonal(C, M.ISOTROPIC, bc, dx, u.shape[1:])
    for name, want in (("residual", b - f), ("jacobi", u + 2.0 / 3.0 * (b - f) / D)):
        got = op.level_op32(name, 0, dev32(u), dev32(b)).cpu().numpy()
        err = np.abs(got - want).max() / np.abs(want).max()
        print(f"{n_cell} {per} {uniform} {target} {name}: {err:.2e}")
        assert err < 2e-6, name


@pytest.mark.parametrize("n_cell", [TILED, BY_NODE])
@pytest.mark.parametrize("per", [(0, 0, 0), (0, 1, 0)])
def test_fp32_sweep_divides_by_the_rounded_diagonal(per, n_cell):
    op, C, bc, u, dx = operator(n_cell, per, False, 9)
    b = np.float32(np.random.default_rng(10).uniform(0.5, 1.5, u.shape))
    D = op.Diagonal().cpu().numpy()
    want = float(np.float32(2.0 / 3.0)) * b.astype(np.float64) / D
    got = op.level_op32("jacobi", 0, dev32(np.zeros(u.shape)), dev32(b)).cpu().numpy()
    inner = (slice(None),) + (slice(1, -1),) * 3
    err = np.abs(got / want - 1)[inner].max() * 2.0 ** 24
    print(f"{n_cell} {per}: {err:.2f} 2^-24")
    assert err < 3.1
