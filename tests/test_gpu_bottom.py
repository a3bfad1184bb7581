"""The BiCGStab bottom solve on the assembled rows of the coarsest level
(k_bottom_bicgstab): two V-cycles of the device against the oracle's on
hierarchies of two levels, whose coarsest level runs from one wave of threads
to the largest level that the kernel serves (rows in registers up to 256 nodes,
streamed above)."""
import numpy as np
import pytest

from alamo_amd import bc as B
from alamo_amd import model as M
from oracle import oracle as O

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

# coarsest nodes: 3x3x3 = 27, 5x4x6 = 120, 4x8x8 = 256, 6x8x6 = 288, 8x8x8 = 512
SIZES = [(4, 4, 4), (8, 6, 10), (6, 14, 14), (10, 14, 10), (14, 14, 14)]


# Converged: both sides solve the bottom to 1e-12, so they differ by that times
# the condition of the clamped coarsest operator (a few hundred): 1e-9.  Failed:
# one BiCGStab step, whose result is discarded, then 8 Fsmooth calls: 1e-12
# (rounding of some 40 sweeps).
@pytest.mark.parametrize("ends,kw,bar", [("converged", dict(bottom_tol_rel=1e-12, bottom_max_iter=2000), 1e-9),
                                         ("failed", dict(bottom_tol_rel=1e-12, bottom_max_iter=1), 1e-12)])
@pytest.mark.parametrize("sym", [M.ISOTROPIC, M.MAJORMINOR, M.DIAGONAL])
@pytest.mark.parametrize("cells", SIZES)
def test_bottom_solve_matches_oracle(cells, sym, ends, kw, bar):
    from alamo_amd import elastic as el
    shape = tuple(c + 1 for c in cells[::-1])
    z, y, x = np.meshgrid(*[np.linspace(0.0, 1.0, s) for s in shape], indexing="ij")
    w = 0.5 + 0.3 * np.sin(3.0 * x + 2.0 * y) * np.cos(2.0 * z)
    if sym == M.ISOTROPIC:
        rows = np.array([M.lame_from_E_nu(1.0, 0.3), M.lame_from_E_nu(2.0, 0.25)])
    elif sym == M.MAJORMINOR:
        R = M.haar_rotations(2, 3)
        rows = np.stack([M.cubic(1.7, 1.2, 0.75, R[g], convention="tensor") for g in range(2)])
    else:
        rows = np.array([np.linspace(1.0, 1.8, 9), np.linspace(2.0, 1.2, 9)])
    C = np.ascontiguousarray(M.mix(np.stack([1.0 - w, w]), rows))
    bc = B.Constant()
    dx = (1.0 / 8, 1.0 / 10, 1.0 / 8)
    b = np.zeros((3,) + shape)
    b[:, 1:-1, 1:-1, 1:-1] = np.random.default_rng(5).standard_normal((3,) + tuple(s - 2 for s in shape))
    op = el.ElasticOperator(cells, dx, sym, max_coarsening_level=1)
    assert op.num_levels == 2
    op.SetBC(bc)
    op.SetModel(torch.from_numpy(C).cuda())
    xd = torch.zeros((3,) + shape, dtype=torch.float64, device="cuda")
    s = el.Linear(op, cycle="V", max_iter=2, abort_on_fail=False, **kw)
    s.solve(xd, torch.from_numpy(b).cuda(), 1e-14, 0.0)
    xo, info = O.mlmg_solve(b, C, sym, bc, dx, tol_rel=1e-14, max_iter=2, cycle="V", max_coarsening_level=1, **kw)
    err = np.linalg.norm(xd.cpu().numpy() - xo) / np.linalg.norm(xo)
    print(f"{cells} sym {sym} {ends}: {err:.2e}")
    assert s.info.iters == info["iters"] == 2
    assert err < bar
