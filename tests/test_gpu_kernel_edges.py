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
