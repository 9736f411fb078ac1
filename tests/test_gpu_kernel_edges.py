"""Kernels at the edges of their tiles, splits and dispatch rules, against the
CPU oracle or the general path."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from test_gpu_assembly import T
from test_gpu_fint import FINT_TOL, _mixed_mesh

pytestmark = pytest.mark.gpu
DEV = 'cuda'


@pytest.mark.parametrize('etype', ['quad4', 'quad4r', 'tria3r'])
@pytest.mark.parametrize('n_elem', [1, 63, 64, 65, 129])
def test_element_forces_tiles(etype, n_elem):
    """Element forces of a last block of 1 to 64 elements (one lane each),
    thin and thick records; nothing written past the last element."""
    from pyfe3d_amd import assembly as A
    x, conn, props, u, kw = _mixed_mesh(etype)
    props[3:, 23] = 0.05  # thicker than an element is wide
    sl = slice(0, n_elem)
    conn = conn[sl]
    kw = {k: v[sl] for k, v in kw.items()}
    nn = conn.shape[1]
    ref = np.zeros(u.size)
    O.fint(etype, x, conn, kw['xmat'], kw['pid'], props, u, k6rot=kw['k6rot'], alpha=kw['alpha'],
           hg=kw['hg'], out=ref)
    fe = torch.full((n_elem + 1, nn, 6), -7., dtype=torch.float64, device=DEV)
    A.shell_fe(etype, T(x, torch.float64), T(6 * conn, torch.int64), T(u, torch.float64),
               T(props, torch.float64), pid=T(kw['pid'], torch.int32),
               xmat=T(kw['xmat'], torch.float64), k6rot=T(kw['k6rot'], torch.float64),
               alpha=T(kw['alpha'], torch.float64), hg=T(kw['hg'], torch.float64), fe=fe)
    fe = fe.cpu().numpy()
    assert (fe[n_elem] == -7.).all()
    got = np.zeros((u.size // 6, 6))
    np.add.at(got, conn.ravel(), fe[:n_elem].reshape(-1, 6))
    err = np.abs(got.ravel() - ref).max() / np.abs(ref).max()
    print(etype, n_elem, 'max rel err %.2e' % err)
    assert err <= FINT_TOL


@pytest.mark.parametrize('nx, ny', [(1, 1), (2, 1), (5, 3), (9, 8), (31, 2)])
@pytest.mark.parametrize('etype', ['quad4', 'tria3r'])
def test_static_system_setup(etype, nx, ny):
    """Boundary conditions, FP32 copy and block inverses of systems of 4 to
    96 block rows (one wave a row, 64 rows a wave), 2 to 9 blocks a row,
    random fixed DOFs, against numpy on the same values; block sums with 1
    to 6 sources against the slot plan, bit for bit."""
    from pyfe3d_amd.mesh import PlateMesh
    from pyfe3d_amd.solver import StaticSystem
    from pyfe3d_amd.sparse import BlockPlan, BSRPlan
    m = PlateMesh(nx + 1, ny + 1, 1.0, 0.7)
    conn = m.quads if etype == 'quad4' else m.trias
    E, nn = conn.shape
    rng = np.random.default_rng(nx * 100 + ny)
    # random symmetric positive blocks in place of stiffness values, with
    # diagonals small enough here and there that rows are exchanged
    v = rng.normal(size=(E, 6 * nn, 6 * nn))
    dof = (6 * conn[:, :, None] + np.arange(6)).reshape(E, -1)
    r = np.broadcast_to(dof[:, :, None], v.shape).reshape(-1)
    c = np.broadcast_to(dof[:, None, :], v.shape).reshape(-1)
    tv = T(v.reshape(-1), torch.float64)
    plan = BlockPlan(T(6 * conn, torch.int64), m.n_nodes)
    val = plan.apply(tv)
    slot = BSRPlan(T(r, torch.int64), T(c, torch.int64), m.n_nodes)
    assert torch.equal(val, slot.apply(tv))
    twice = plan.apply(tv, out=val.clone(), accumulate=True)
    assert np.allclose(twice.cpu().numpy(), 2 * val.cpu().numpy(), rtol=1e-13, atol=1e-13)
    fixed = rng.random(m.n_dof) < 0.3
    s = StaticSystem(plan, val, fixed)
    K = plan.to_scipy(val).toarray()
    K[fixed, :] = 0.
    K[:, fixed] = 0.
    K[fixed, fixed] = 1.
    got = plan.to_scipy(s.val).toarray()
    assert (got == K).all()
    assert torch.equal(s.val32, s.val.to(torch.float32))
    for n in range(m.n_nodes):
        blk = K[6 * n:6 * n + 6, 6 * n:6 * n + 6]
        inv = s.dinv.view(-1, 6, 6)[n].cpu().numpy()
        # residual of an inverse by elimination with pivoting: a few n eps cond
        assert np.abs(inv @ blk - np.eye(6)).max() <= 64 * 2.3e-16 * np.linalg.cond(blk)
    assert torch.equal(s.dinv32, s.dinv.to(torch.float32))
