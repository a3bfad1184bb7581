"""The tiled isotropic stencil (k_stencil_iso) against the oracle: a box whose
tiles are partial along i and j, in chunks of 16 planes (the longest, with a
shorter last one), the default and 1 plane, with and without periodic axes and
the uniform flag, in FP64 (1e-12, the bar of the operator tests: a few hundred
rounded terms a row) and FP32 (2e-6, the bar of the FP32 kernels')."""
import numpy as np
import pytest

from alamo_amd import model as M
from oracle import oracle as O

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
from test_oracle_periodic import periodize, rand_case  # noqa: E402

N_CELL = (70, 52, 46)  # 69 x 51 x 45 interior nodes: 3 x 7 tiles a plane


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def relerr(a, b):
    torch.cuda.synchronize()
    return np.abs(a.cpu().numpy() - b).max() / np.abs(b).max()


@pytest.mark.parametrize("target", ["1", None, "100000"])
@pytest.mark.parametrize("per,uniform", [((0, 0, 0), False), ((0, 0, 0), True), ((0, 1, 0), False), ((1, 0, 1), False)])
def test_tiled_isotropic_rows_match_oracle(per, uniform, target, monkeypatch):
    from alamo_amd import elastic as el
    if target:
        monkeypatch.setenv("ALAMO_EL_TILE_TARGET", target)
    C, bc, u, dx = rand_case(M.ISOTROPIC, N_CELL, per, 7)
    if uniform:
        C = np.ascontiguousarray(np.broadcast_to(C[:, :1, :1, :1], C.shape))
    b = periodize(np.random.default_rng(8).standard_normal(u.shape), per)
    op = el.ElasticOperator(N_CELL, dx, M.ISOTROPIC)
    op.SetPeriodic(per)
    op.SetBC(bc)
    op.SetUniform(uniform)
    op.SetModel(dev(C))
    op.prepare()
    with O.periodic(per):
        f = O.fapply(u, C, M.ISOTROPIC, bc, dx, uniform=uniform)
        r = O.residual(u, b, C, M.ISOTROPIC, bc, dx, uniform=uniform)
        diag = O.diagonal(C, M.ISOTROPIC, bc, dx, u.shape[1:])
        x = O.fsmooth(u, b, C, M.ISOTROPIC, bc, dx, diag, nsmooth=1, uniform=uniform)
    assert relerr(op.Fapply(dev(u)), f) < 1e-12
    assert relerr(op.residual(dev(u), dev(b)), r) < 1e-12
    assert relerr(op.Fsmooth(dev(u), dev(b)), x) < 1e-12
    u32, b32, C32 = (v.astype(np.float32).astype(np.float64) for v in (u, b, C))
    with O.periodic(per):
        f32 = O.fapply(u32, C32, M.ISOTROPIC, bc, dx, uniform=uniform)
    got = op.level_op32("fapply", 0, dev(u32.astype(np.float32)))
    assert relerr(got, f32) < 2e-6
