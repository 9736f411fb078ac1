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


def test_static_system_copies_are_flat():
    """Values given as (blocks, 6, 6), with and without some past the pattern:
    kept in that shape, their FP32 copy flat."""
    from types import SimpleNamespace
    from pyfe3d_amd.solver import StaticSystem
    rp, ci, val, _ = _block_system(_graph('3x3'), 1)
    plan = SimpleNamespace(row_ptr=T(rp, torch.int32), col_idx=T(ci, torch.int32), n_nodes=9)
    for more in (0, 2):
        v = T(np.concatenate([val, np.ones((more, 6, 6))]), torch.float64)
        s = StaticSystem(plan, v, np.zeros(54))
        assert s.val.shape == v.shape and torch.equal(s.val, v)
        assert s.val32.dim() == 1 and torch.equal(s.val32, v.reshape(-1).to(torch.float32))


def test_static_system_of_many_rows():
    """Boundary conditions and copies of 6.7e7 block rows with one block each,
    a wave per row: more than 2^32 threads."""
    from pyfe3d_amd import _lib
    if torch.cuda.mem_get_info()[0] < 100e9:
        pytest.skip('needs 100 GB of free memory')
    nb = (1 << 26) + 1001
    rp = torch.arange(nb + 1, dtype=torch.int32, device=DEV)
    src = (torch.arange(36, dtype=torch.float64, device=DEV) + 1.).repeat(nb, 1)
    fixed = torch.zeros(6 * nb, dtype=torch.uint8, device=DEV)
    val = torch.full_like(src, float('nan'))
    val32 = torch.full((nb, 36), float('nan'), dtype=torch.float32, device=DEV)
    _lib.call('pf3d_bsr_system', nb, rp.data_ptr(), rp.data_ptr(), src.data_ptr(),
              fixed.data_ptr(), val.data_ptr(), val32.data_ptr(),
              torch.cuda.current_stream().cuda_stream)
    assert torch.equal(val, src)
    for at in range(0, nb, 1 << 24):
        part = val32[at:at + (1 << 24)]
        assert torch.equal(part, src[:1].to(torch.float32).expand(part.shape))
    del src, val, val32, fixed, rp
    torch.cuda.empty_cache()


def test_mixed_mass_of_many_beams():
    """Lumped mass of more beams (1.3e8, 39 GB of values) than one row of a
    launch holds, all between the same two nodes: every one is written."""
    from pyfe3d_amd import assembly as A
    if torch.cuda.mem_get_info()[0] < 100e9:
        pytest.skip('needs 100 GB of free memory')
    E = (1 << 27) + 4099
    size = A.slot_count('beamc', 'M', 1)
    x = T([[0., 0., 0.], [0.3, 0.1, 0.2]], torch.float64)
    conn = torch.tensor([[0, 6]], device=DEV).repeat(E, 1)
    evec = torch.tensor([[0., 0., 1.]], dtype=torch.float64, device=DEV).repeat(E, 1)
    props = T(np.linspace(1., 2., A.BEAM_STRIDE)[None], torch.float64)
    v = torch.full((E, size), float('nan'), dtype=torch.float64, device=DEV)
    A.mixed_assemble('M', [A.ElementGroup('beamc', conn, props, evec=evec)], x, None, None,
                     v.view(-1), mtype=1, values_only=True, overwrite=True, check=False)
    assert float(v[0].abs().max()) > 0
    for at in range(0, E, 1 << 24):
        part = v[at:at + (1 << 24)]
        assert torch.equal(part, v[:1].expand(part.shape))
    del v, conn, evec
    torch.cuda.empty_cache()


def test_block_sums_past_32_bits():
    """More than 2^32 pairs of entries (69 GB of block values): every block
    is written."""
    from pyfe3d_amd import _lib
    if torch.cuda.mem_get_info()[0] < 100e9:
        pytest.skip('needs 100 GB of free memory')
    nnzb = 2 ** 32 // 18 + 300
    v = torch.arange(2 * 144, dtype=torch.float64, device=DEV)  # two elements' blocks
    src_ptr = torch.arange(nnzb + 1, device=DEV)
    src = 144 * (src_ptr[:-1] % 2)
    out = torch.full((nnzb, 36), -1., dtype=torch.float64, device=DEV)
    _lib.call('pf3d_block_apply', nnzb, src_ptr.data_ptr(), src.data_ptr(), 2, v.data_ptr(),
              out.data_ptr(), 0, torch.cuda.current_stream().cuda_stream)
    want = v.view(2, 12, 12)[:, :6, :6].reshape(2, 36)
    for at in range(0, nnzb, 1 << 24):  # (starts on an even block)
        part = out[at:at + (1 << 24)]
        assert torch.equal(part[0::2], want[:1].expand(part[0::2].shape))
        assert torch.equal(part[1::2], want[1:].expand(part[1::2].shape))
    del out, src, src_ptr
    torch.cuda.empty_cache()


def _graph(name):
    """Block pattern as a list of neighbour sets."""
    rng = np.random.default_rng(len(name))

    def grid(nx, ny, hole=False):
        at, nb = {}, []
        for i in range(nx):
            for j in range(ny):
                if hole and nx // 3 < i < 2 * nx // 3 and ny // 3 < j < 2 * ny // 3:
                    continue
                at[i, j] = len(at)
        nb = [set() for _ in at]
        for (i, j), v in at.items():
            for di in (-1, 0, 1):
                for dj in (-1, 0, 1):
                    if (i + di, j + dj) in at:
                        nb[v].add(at[i + di, j + dj])
        return nb

    if name == 'one':
        return [{0}]
    if name == 'chain':
        return [{j for j in (i - 1, i, i + 1) if 0 <= j < 90} for i in range(90)]
    if name == 'isolated':
        return grid(6, 5) + [{30 + i} for i in range(7)]
    if name == 'two parts':
        a = grid(9, 7)
        return a + [{v + len(a) for v in s} for s in a]
    if name == 'complete':
        return [set(range(40)) for _ in range(40)]
    if name == 'random':
        nb = [{i} for i in range(160)]
        for _ in range(260):
            a, b = rng.integers(0, 160, 2)
            nb[a].add(b)
            nb[b].add(a)
        return nb
    nx, ny = (int(t) for t in name.split(' ')[0].split('x'))
    return grid(nx, ny, 'hole' in name)


def _block_system(nb, seed):
    """(row_ptr, col_idx, values (nnzb, 6, 6), dense) of a random symmetric,
    diagonally dominant matrix on the pattern."""
    rng = np.random.default_rng(seed)
    n = len(nb)
    rp = np.concatenate([[0], np.cumsum([len(s) for s in nb])]).astype(np.int32)
    ci = np.concatenate([sorted(s) for s in nb]).astype(np.int32)
    A = np.zeros((n, 6, n, 6))
    for r in range(n):
        for c in sorted(nb[r]):
            if c <= r:
                A[r, :, c, :] = rng.uniform(-1, 1, (6, 6))
    A = A.reshape(6 * n, 6 * n)
    A = np.tril(A, -1)
    A = A + A.T
    A[np.diag_indices(6 * n)] = np.abs(A).sum(axis=1) + 1.
    rows = np.repeat(np.arange(n), np.diff(rp))
    val = A.reshape(n, 6, n, 6)[rows, :, ci, :]
    return rp, ci, val, A


@pytest.mark.parametrize('leaf', [1, 5, 16])
@pytest.mark.parametrize('name', ['one', 'chain', '2x2', '7x5', '16x16', '40x9', '23x23 hole',
                                  'isolated', 'two parts', 'complete', 'random'])
def test_dissection_against_dense(name, leaf):
    """Nested dissection on patterns with fronts of 6 to 240 own DOFs, panels
    of 6 to 32 columns, more and less than 128 rows, empty separators and
    isolated nodes, two right-hand sides from one factor.  Diagonally
    dominant matrices (condition below 1e3): 1e-12 of numpy's solution."""
    from pyfe3d_amd.direct import DirectPlan
    rp, ci, val, A = _block_system(_graph(name), leaf)
    plan = DirectPlan(rp, ci, DEV, leaf=leaf)
    n = A.shape[0]
    new = lambda m: torch.full((max(1, m),), float('nan'), dtype=torch.float64, device=DEV)
    factor, update, work = new(plan.factor_size), new(plan.update_size), new(plan.work_size)
    bad = torch.zeros(1, dtype=torch.int32, device=DEV)
    tv = T(val.reshape(-1), torch.float64)
    s = torch.cuda.current_stream().cuda_stream
    plan.factor(tv.data_ptr(), factor, update, bad, s)
    rng = np.random.default_rng(7)
    for _ in range(2):
        b = rng.normal(size=n)
        tb, x = T(b, torch.float64), new(n)
        plan.solve(factor, tb.data_ptr(), x.data_ptr(), work, s)
        ref = np.linalg.solve(A, b)
        err = np.linalg.norm(x.cpu().numpy() - ref) / np.linalg.norm(ref)
        # the same right-hand side carried through the factorisation
        y, factor2 = new(n), new(plan.factor_size)
        plan.factor(tv.data_ptr(), factor2, update, bad, s, f=tb.data_ptr())
        plan.solve(factor2, None, y.data_ptr(), work, s)
        err = max(err, np.linalg.norm(y.cpu().numpy() - ref) / np.linalg.norm(ref))
        print(name, leaf, 'err %.2e, %d fronts, widest %d' % (err, plan.n_fronts, plan.widest))
        assert err <= 1e-12
    assert int(bad.item()) == 0
    # not positive definite: reported
    val[rp[:-1] + [sorted(s_).index(i) for i, s_ in enumerate(_graph(name))]] *= -1.
    tv = T(val.reshape(-1), torch.float64)
    plan.factor(tv.data_ptr(), factor, update, bad, s)
    assert int(bad.item()) > 0


@pytest.mark.parametrize('keep', ['lower', 'upper'])
def test_dissection_of_one_sided_blocks(keep):
    """Blocks stored on one side of the diagonal only: the bits of the whole
    matrix."""
    from pyfe3d_amd.direct import DirectPlan
    rp, ci, val, _ = _block_system(_graph('13x10'), 6)
    n = rp.size - 1
    rows = np.repeat(np.arange(n), np.diff(rp))
    s = torch.cuda.current_stream().cuda_stream
    b = T(np.random.default_rng(8).normal(size=6 * n), torch.float64)
    got = []
    for on in (rows >= 0, rows >= ci if keep == 'lower' else rows <= ci):
        orp = np.concatenate([[0], np.cumsum(np.bincount(rows[on], minlength=n))])
        plan = DirectPlan(orp, ci[on], DEV)
        new = lambda m: torch.empty(max(1, m), dtype=torch.float64, device=DEV)
        factor, update, work, x = (new(m) for m in (plan.factor_size, plan.update_size,
                                                    plan.work_size, 6 * n))
        bad = torch.zeros(1, dtype=torch.int32, device=DEV)
        tv = T(val[on].reshape(-1), torch.float64)
        plan.factor(tv.data_ptr(), factor, update, bad, s)
        plan.solve(factor, b.data_ptr(), x.data_ptr(), work, s)
        assert int(bad.item()) == 0
        got.append(x)
    assert torch.equal(*got)


def _duck_plan(nb, seed, make):
    rp, ci, val, _ = _block_system(nb, seed)
    return (make(row_ptr=T(rp, torch.int32), col_idx=T(ci, torch.int32), n_nodes=len(nb)),
            T(val.reshape(-1), torch.float64))


def test_direct_plans_copy_and_pickle():
    """A pattern, a system and a sweep that were solved directly are copied
    and pickled as before, and go on solving; a pattern object without room
    for an analysis is accepted."""
    import copy
    import pickle
    from collections import namedtuple
    from types import SimpleNamespace
    from pyfe3d_amd.solver import StaticSystem
    from pyfe3d_amd.sweep import PlateSweep
    nb = _graph('9x7')
    f = np.random.default_rng(1).normal(size=6 * len(nb))
    plan, val = _duck_plan(nb, 3, SimpleNamespace)
    a = StaticSystem(plan, val, np.zeros(6 * len(nb)))
    u, _ = a.solve(f, method='direct')
    again, _ = a.solve(f, method='direct')
    for b in (copy.deepcopy(a), pickle.loads(pickle.dumps(a))):
        assert torch.equal(b.solve(f, method='direct')[0], again)
        assert torch.equal(b.solve(f, method='direct', refactor=True)[0], u)
        c = StaticSystem(b.plan, val, np.zeros(6 * len(nb)))
        assert torch.equal(c.solve(f, method='direct')[0], u)
    fixed_plan, val = _duck_plan(nb, 3, namedtuple('Pattern', 'row_ptr col_idx n_nodes'))
    d = StaticSystem(fixed_plan, val, np.zeros(6 * len(nb)))
    assert torch.equal(d.solve(f, method='direct')[0], u)
    sw = PlateSweep([(5, 4), (7, 9)])
    h, load = sw.random_designs(2)
    sw.set_thickness(h)
    sw.set_loads(load)
    sw.step(mode='direct')
    u = sw.u.clone()
    for other in (copy.deepcopy(sw), pickle.loads(pickle.dumps(sw))):
        other.u.zero_()
        other.step(mode='direct')
        assert torch.equal(other.u, u)


@pytest.mark.parametrize('in_place', [False, True])
def test_direct_solve_on_a_changed_pattern(in_place):
    """A pattern object whose arrays are replaced or overwritten is analysed
    anew for the next system; the system made before keeps its factor."""
    from types import SimpleNamespace
    from pyfe3d_amd.solver import StaticSystem
    chain = lambda p: [{p[j] for j in (i - 1, i, i + 1) if 0 <= j < 40} for i in range(40)]
    p = np.random.default_rng(2).permutation(40)
    first = chain(np.arange(40))
    mixed = [None] * 40
    for i, nb in enumerate(chain(p)):
        mixed[p[i]] = nb
    second = mixed if in_place else _graph('8x6')
    f = [np.random.default_rng(3).normal(size=6 * len(nb)) for nb in (first, second)]
    alone = []
    for nb, b in zip((first, second), f):
        plan, val = _duck_plan(nb, 5, SimpleNamespace)
        s = StaticSystem(plan, val, np.zeros(b.size))
        alone.append([s.solve(b, method='direct')[0] for _ in range(2)])
    plan, val = _duck_plan(first, 5, SimpleNamespace)
    a = StaticSystem(plan, val, np.zeros(f[0].size))
    assert torch.equal(a.solve(f[0], method='direct')[0], alone[0][0])
    new, val = _duck_plan(second, 5, SimpleNamespace)
    if in_place:
        plan.row_ptr.copy_(new.row_ptr)
        plan.col_idx.copy_(new.col_idx)
    else:
        plan.row_ptr, plan.col_idx, plan.n_nodes = new.row_ptr, new.col_idx, new.n_nodes
    b = StaticSystem(plan, val, np.zeros(f[1].size))
    assert torch.equal(b.solve(f[1], method='direct')[0], alone[1][0])
    x = torch.empty_like(alone[0][1])
    assert torch.equal(a.direct_solve(torch.as_tensor(f[0], device=DEV), x), alone[0][1])


def test_direct_buffers_outlive_a_side_stream():
    """The index maps that systems on one pattern share, and a factor, are not
    handed out again while a factorisation on another stream is enqueued."""
    from types import SimpleNamespace
    from pyfe3d_amd.solver import StaticSystem
    nb = _graph('30x29')
    plan, val = _duck_plan(nb, 5, SimpleNamespace)
    fixed, f = np.zeros(6 * len(nb)), torch.ones(6 * len(nb), dtype=torch.float64, device=DEV)
    a, b = (StaticSystem(plan, val, fixed) for _ in range(2))
    a.factor_direct()
    b.factor_direct()
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        torch.cuda._sleep(1 << 30)
        b.factor_direct(stream=side, b=f)
        b.direct_solve(None, f, stream=side)
    held = [t.data_ptr() for t in (a._factor_plan.image, b._factor)]
    del a, b, plan
    state = {}
    for seg in torch.cuda.memory_snapshot():
        at = seg['address']
        for block in seg['blocks']:
            state.update((p, block['state']) for p in held if at <= p < at + block['size'])
            at += block['size']
    assert not side.query()
    assert [state[p] for p in held] == ['active_pending_free'] * 2
    side.synchronize()


def test_dissection_of_separate_parts():
    """Plates that are not connected, in one system: level by level beside
    each other, each with the bits of its solution alone."""
    from types import SimpleNamespace
    from pyfe3d_amd.solver import StaticSystem
    grid, copies = _graph('14x11'), 9
    rp, ci, val, _ = _block_system(grid, 4)
    f = np.random.default_rng(5).normal(size=6 * len(grid))

    def solve(k):
        plan = SimpleNamespace(
            row_ptr=T(np.concatenate([[0]] + [rp[1:] + s * ci.size for s in range(k)]), torch.int32),
            col_idx=T(np.concatenate([ci + s * len(grid) for s in range(k)]), torch.int32),
            n_nodes=k * len(grid))
        system = StaticSystem(plan, T(np.tile(val.reshape(-1), k), torch.float64),
                              np.zeros(6 * plan.n_nodes))
        u, info = system.solve(np.tile(f, k), method='direct')
        assert info['converged']
        return u.cpu().numpy()

    assert (solve(copies) == np.tile(solve(1), copies)).all()


def test_dissection_sweep_matches_banded(monkeypatch):
    """The sweep's route by nested dissection against the banded kernels
    (an explicit launch shape) on uneven plates: every variant within 1e-9
    and at the same residual level; one group or several, graph replays and
    eager steps: the same bits."""
    import pyfe3d_amd.direct as D
    from pyfe3d_amd.sweep import PlateSweep
    dims = [(41, 50), (10, 12), (2, 40), (20, 30), (8, 64), (3, 3)]
    sw = PlateSweep(dims)
    h, f = sw.random_designs(5)
    sw.set_thickness(h)
    sw.set_loads(f)
    sw.assemble()
    sw.solve_direct(config=(512, 448, 512))
    ref, res = sw.u.clone(), sw.relres.clone()
    sw.u.zero_()
    sw.solve_direct()
    sw.check()
    got = sw.u.clone()
    assert len(sw._batch.groups) == 1
    assert float(sw.relres.max()) <= max(1e-8, 2 * float(res.max()))
    for v in range(sw.n_var):
        nodes, _ = sw.variant(v)
        a, b = ref[6 * nodes.start:6 * nodes.stop], got[6 * nodes.start:6 * nodes.stop]
        assert float((a - b).norm()) <= 1e-9 * float(a.norm()), v
    monkeypatch.setattr(D.DirectBatch, 'GROUP_NODES', 1000)
    sw2 = PlateSweep(dims)
    sw2.set_thickness(h)
    sw2.set_loads(f)
    g = sw2.capture(mode='direct')
    assert len(sw2._batch.groups) > 1
    for seed in (5, 9, 5):
        h, f = sw2.random_designs(seed)
        sw2.set_thickness(h)
        sw2.set_loads(f)
        g.replay()
        torch.cuda.synchronize()
        u = sw2.u.clone()
        sw2.step(mode='direct')
        assert torch.equal(u, sw2.u), seed
    assert torch.equal(u, got)


def test_direct_refuses_wide_bands_and_takes_streams():
    """A star of 240 nodes has no numbering within the widest band: refused
    as before; a plate factorised and solved on a side stream gives the
    current stream's bits; a singular system is reported."""
    from types import SimpleNamespace
    from pyfe3d_amd import _lib
    from pyfe3d_amd.solver import StaticSystem
    nb = [set(range(240))] + [{0, i} for i in range(1, 240)]

    def system(nb, seed, **kw):
        rp, ci, val, A = _block_system(nb, seed)
        plan = SimpleNamespace(row_ptr=T(rp, torch.int32), col_idx=T(ci, torch.int32),
                               n_nodes=len(nb))
        return StaticSystem(plan, T(val.reshape(-1), torch.float64), np.zeros(6 * len(nb)), **kw)

    with pytest.raises(ValueError, match='exceeds'):
        system(nb, 1).factor_direct()
    grid = _graph('12x9')
    f = np.random.default_rng(3).normal(size=6 * len(grid))
    a = system(grid, 2)
    u, info = a.solve(f, method='direct')
    assert info['converged'] and a.bandwidth == 6 * 10 + 5
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        v, _ = system(grid, 2, stream=s).solve(f, method='direct', stream=s)
    s.synchronize()
    assert torch.equal(u, v)
    a.val.neg_()
    with pytest.raises(_lib.Pf3dError):
        a.solve(f, method='direct', refactor=True)


@pytest.mark.parametrize('dims, method', [([(22, 30), (10, 12)], 'banded'),
                                          ([(40, 41), (10, 12)], 'dissection')])
def test_tuning_holds_no_unused_band(tmp_path, monkeypatch, dims, method):
    """Tuning the banded kernels: used by the direct solve up to BANDED_MAX,
    and no band storage left (or made, from the table) where dissection is
    run all the same; one that was there before stays."""
    from pyfe3d_amd.sweep import PlateSweep
    monkeypatch.setenv('PF3D_AUTOTUNE_CACHE', str(tmp_path / 'tune.json'))

    def sweep():
        sw = PlateSweep(dims)
        h, f = sw.random_designs(5)
        sw.set_thickness(h)
        sw.set_loads(f)
        sw.assemble()
        return sw

    for source in ('measured', 'table'):
        sw = sweep()
        assert sw.direct_method == 'dissection'
        assert sw.autotune_direct(repeats=1) and sw.direct_config_source == source
        assert sw.direct_method == method
        if method == 'dissection':
            assert not hasattr(sw, 'band')
        sw.solve_direct()
        sw.check()
        assert float(sw.relres.max()) <= 1e-8
        assert hasattr(sw, '_batch') == (method == 'dissection')
    sw = sweep()
    sw.solve_direct(config=(512, 448, 512))
    band = sw.band
    sw.autotune_direct(repeats=1, use_table=False)
    assert sw.band is band


@pytest.mark.parametrize('rows', [1, 2, 43, 127, 128, 129, 256, 257, 1365, 1366, 2731, 21846])
@pytest.mark.parametrize('method', ['fp64', 'ir'])
def test_pcg_routes(rows, method):
    """Chains of 1 to 21,846 block rows: one and two row slots per thread,
    one and several 256-row blocks, p.q formed in the update (up to 8,192
    entries), by the separate kernel, and the separate kernels throughout
    (above 131,072).  Diagonally dominant (condition below 100), solved to
    1e-12: within 1e-10 of the solution the loads were made from,
    a start at the solution needs no iteration, maxiter is kept."""
    from types import SimpleNamespace
    from pyfe3d_amd.solver import StaticSystem
    rng = np.random.default_rng(rows)
    off = rng.uniform(-1, 1, (rows, 6, 6))        # block (i, i + 1)
    diag = rng.uniform(-1, 1, (rows, 6, 6))
    diag = diag + diag.transpose(0, 2, 1) + 30. * np.eye(6)
    idx = np.arange(rows)
    r = np.concatenate([idx, idx[:-1], idx[1:]])
    c = np.concatenate([idx, idx[1:], idx[:-1]])
    v = np.concatenate([diag, off[:-1], off[:-1].transpose(0, 2, 1)])
    order = np.lexsort((c, r))
    rp = np.concatenate([[0], np.cumsum(np.bincount(r, minlength=rows))])
    plan = SimpleNamespace(row_ptr=T(rp, torch.int32), col_idx=T(c[order], torch.int32),
                           n_nodes=rows)
    s = StaticSystem(plan, T(v[order].reshape(-1), torch.float64), np.zeros(6 * rows))
    u = rng.normal(size=(rows, 6))
    f = np.einsum('nij,nj->ni', diag, u)
    f[:-1] += np.einsum('nij,nj->ni', off[:-1], u[1:])
    f[1:] += np.einsum('nji,nj->ni', off[:-1], u[:-1])
    rtol = 1e-12 if method == 'fp64' else 1e-11
    x, info = s.solve(f.reshape(-1), method=method, rtol=rtol)
    assert info['relres'] <= 2 * rtol and info['iters'] > 0
    assert np.linalg.norm(x.cpu().numpy() - u.ravel()) <= 1e-10 * np.linalg.norm(u)
    if method == 'fp64':
        _, again = s.solve(f.reshape(-1), method=method, rtol=1e-9, x0=x)
        assert again['iters'] == 0
        _, few = s.solve(f.reshape(-1), method=method, rtol=1e-30, maxiter=3)
        assert few['iters'] == 3


@pytest.mark.parametrize('rows', [2, 1366, 21846])
@pytest.mark.parametrize('method', ['fp64', 'mixed'])
def test_pcg_without_a_step(rows, method):
    """Pairs of block rows (I, -I; -I, I) under equal loads: p.q is exactly 0
    with a residual of 1 (a singular matrix).  Reported at once, not after
    maxiter iterations that change nothing."""
    from types import SimpleNamespace
    from pyfe3d_amd.solver import StaticSystem
    pair = np.arange(rows) // 2 * 2
    plan = SimpleNamespace(row_ptr=T(2 * np.arange(rows + 1), torch.int32),
                           col_idx=T((pair[:, None] + [0, 1]).ravel(), torch.int32), n_nodes=rows)
    sign = np.where(np.arange(rows)[:, None] == pair[:, None] + [0, 1], 1., -1.)
    val = sign.reshape(-1, 1, 1) * np.eye(6)
    s = StaticSystem(plan, T(val.reshape(-1), torch.float64), np.zeros(6 * rows))
    f = torch.ones(6 * rows, dtype=torch.float64, device=DEV)
    u, info = s.solve(f, method=method, maxiter=20000)
    assert not info['converged'] and info['iters'] <= 1000
    if method == 'fp64':
        assert info['iters'] == 25


@pytest.mark.parametrize('rows', [40, 2000, 21846])
@pytest.mark.parametrize('method', ['fp64', 'mixed', 'ir'])
def test_pcg_ignores_its_workspace(rows, method):
    """The bits of a solve do not depend on what the workspace held."""
    from types import SimpleNamespace
    from pyfe3d_amd.solver import StaticSystem
    chain = [{j for j in (i - 1, i, i + 1) if 0 <= j < 40} for i in range(40)]
    rp, ci, val, _ = _block_system(chain, 9)
    k = -(-rows // 40)
    plan = SimpleNamespace(
        row_ptr=T(np.concatenate([[0]] + [rp[1:] + s * ci.size for s in range(k)]), torch.int32),
        col_idx=T(np.concatenate([ci + 40 * s for s in range(k)]), torch.int32), n_nodes=40 * k)
    s = StaticSystem(plan, T(np.tile(val.reshape(-1), k), torch.float64), np.zeros(240 * k))
    rng = np.random.default_rng(rows)
    f, x0 = rng.normal(size=240 * k), T(rng.normal(size=240 * k), torch.float64)
    got = []
    for byte in (0, 255):  # (255: every double a NaN)
        s._w64.fill_(byte)
        s._wir.fill_(byte)
        got.append([s.solve(f, method=method, rtol=1e-6, x0=x) for x in (None, x0)])
    for (u, a), (v, b) in zip(*got):
        assert a == b and a['converged'] and torch.equal(u, v)


def _bf16(a):
    return torch.as_tensor(a, dtype=torch.float32).to(torch.bfloat16).to(torch.float64)


@pytest.mark.parametrize('B, H, W, C, N, stride', [
    (1, 1, 1, 32, 32, 1), (1, 1, 1, 32, 64, 2), (2, 3, 5, 64, 32, 1), (3, 8, 8, 32, 96, 2),
    (1, 7, 9, 96, 32, 2), (2, 16, 15, 32, 32, 1), (1, 33, 31, 64, 64, 2), (5, 2, 70, 32, 32, 2),
    (40, 64, 64, 32, 32, 1), (2, 64, 64, 32, 64, 2)])
def test_direct_convolutions(B, H, W, C, N, stride):
    """3x3 convolution, input and weight gradients against float64 sums of
    the same bfloat16 operands: 1 to 163,840 pixels (16 and 32 per wave), odd
    grids (uneven parity classes), rows shorter than a lane's 8 pixels,
    several channel tiles, one and many splits.  A sum of K products in FP32
    is within K eps of the sum of their magnitudes; the order adds at most
    another K.  Weight gradients sum over up to 163,840 pixels, where that
    bound says nothing: operands of whole numbers up to 3, whose sums are
    exact (below 2^24), equal."""
    from pyfe3d_amd import _lib
    import ctypes
    rng = np.random.default_rng(H * W + C)
    Ho, Wo = (H - 1) // stride + 1, (W - 1) // stride + 1
    f32 = lambda *s: torch.as_tensor(rng.normal(size=s), dtype=torch.float32)
    x, w, b, dy, dx0 = (f32(B, H, W, C), f32(N, 9, C), f32(N), f32(B, Ho, Wo, N),
                        f32(B, H, W, C))
    dev = lambda t: t.to(DEV).contiguous()
    xd, wd, bd, dyd = dev(x), dev(w), dev(b), dev(dy)
    wf = torch.empty(N * 9 * C, dtype=torch.bfloat16, device=DEV)
    wb = torch.empty_like(wf)
    st = torch.cuda.current_stream().cuda_stream
    one = lambda t: (ctypes.c_void_p * 1)(t.data_ptr())
    _lib.call('pf3d_nn_pack', 1, (ctypes.c_int * 1)(N), (ctypes.c_int * 1)(C), one(wd), one(wf),
              one(wb), st)
    y = torch.full((B, Ho, Wo, N), float('nan'), device=DEV)
    _lib.call('pf3d_nn_conv', B, H, W, C, stride, xd.data_ptr(), wf.data_ptr(), bd.data_ptr(), 1,
              N, y.data_ptr(), st)
    dx = dev(dx0)
    _lib.call('pf3d_nn_conv_dx', B, H, W, C, stride, dyd.data_ptr(), wb.data_ptr(), N,
              dx.data_ptr(), 1, st)
    n = N * 9 * C
    eps = 2. ** -23
    F = torch.nn.functional
    nchw = lambda t: t.permute(0, 3, 1, 2)
    wk = lambda t: t.reshape(N, 3, 3, C).permute(0, 3, 1, 2)

    def both(fn, *ops):  # value and sum of magnitudes
        return fn(*ops), fn(*[o.abs() for o in ops])

    xb, wbf, dyb = _bf16(x), _bf16(w), _bf16(dy)
    ref, mag = both(lambda p, q: F.conv2d(nchw(p), wk(q), stride=stride, padding=1), xb, wbf)
    got = nchw(y.cpu().double())
    tol = 2 * 9 * C * eps * (mag + b.abs().double()[None, :, None, None])
    assert ((got - (ref + b.double()[None, :, None, None]).clamp(min=0)).abs() <= tol).all()
    ref, mag = both(lambda p, q: torch.nn.grad.conv2d_input((B, C, H, W), wk(q), nchw(p),
                                                            stride=stride, padding=1), dyb, wbf)
    tol = 2 * 9 * N * eps * (mag + nchw(dx0).abs().double())
    assert ((nchw(dx.cpu().double()) - (ref + nchw(dx0).double())).abs() <= tol).all()
    xi, dyi = (torch.as_tensor(rng.integers(-3, 4, t.shape), dtype=torch.float32)
               for t in (x, dy))
    ref = torch.nn.grad.conv2d_weight(nchw(xi.double()), (N, C, 3, 3), nchw(dyi.double()),
                                      stride=stride, padding=1)
    assert float(ref.abs().max()) > 0
    xd, dyd = dev(xi), dev(dyi)
    for floats in (n, 3 * n, 1000 * n):
        if floats * 4 > 1 << 30:
            continue
        dw = torch.full((N, 9, C), float('nan'), device=DEV)
        work = torch.full((floats,), float('nan'), device=DEV)
        _lib.call('pf3d_nn_conv_dw', B, H, W, C, stride, xd.data_ptr(), dyd.data_ptr(), N,
                  dw.data_ptr(), work.data_ptr(), floats, st)
        assert torch.equal(wk(dw.cpu().double()), ref), floats


@pytest.mark.parametrize('B, H, W, C, N, stride', [
    (1, 1, 1, 32, 32, 1), (2, 3, 5, 64, 32, 1), (3, 8, 8, 32, 96, 2), (1, 7, 9, 96, 64, 2),
    (2, 16, 15, 32, 32, 1), (40, 64, 64, 32, 32, 1), (2, 64, 64, 64, 128, 2)])
@pytest.mark.parametrize('accumulate', [0, 1])
def test_direct_convolutions_bits(B, H, W, C, N, stride, accumulate):
    """The forward pass and the input gradient against the products with the
    column matrix, bit for bit: a backward pass rounds each layer's gradient
    to bfloat16, so that a last bit changed in one layer is a change of 1e-3
    some layers on."""
    from pyfe3d_amd import _lib
    import ctypes
    rng = np.random.default_rng(H * W + C)
    Ho, Wo = (H - 1) // stride + 1, (W - 1) // stride + 1
    f32 = lambda *s: T(rng.normal(size=s), torch.float32)
    x, w, dy, dx0 = f32(B, H, W, C), f32(N, 9, C), f32(B, Ho, Wo, N), f32(B, H, W, C)
    wf = torch.empty(N * 9 * C, dtype=torch.bfloat16, device=DEV)
    wb = torch.empty_like(wf)
    st = torch.cuda.current_stream().cuda_stream
    one = lambda t: (ctypes.c_void_p * 1)(t.data_ptr())
    _lib.call('pf3d_nn_pack', 1, (ctypes.c_int * 1)(N), (ctypes.c_int * 1)(C), one(w), one(wf),
              one(wb), st)
    y, y0 = (torch.full((B, Ho, Wo, N), float('nan'), device=DEV) for _ in range(2))
    dx, dxc = dx0.clone(), dx0.clone()
    M, Kd = B * Ho * Wo, 9 * C
    col = torch.empty((M, Kd), device=DEV)
    gemm = lambda n, k, a, sb, o: _lib.call('pf3d_nn_gemm', M, n, k, a.data_ptr(), k, 1,
                                            w.data_ptr(), sb[0], sb[1], o.data_ptr(), n, 0, None,
                                            0, 1, None, st)
    _lib.call('pf3d_nn_conv', B, H, W, C, stride, x.data_ptr(), wf.data_ptr(), None, 0, N,
              y.data_ptr(), st)
    _lib.call('pf3d_nn_im2col', B, H, W, C, stride, x.data_ptr(), col.data_ptr(), st)
    gemm(N, Kd, col, (Kd, 1), y0)
    assert torch.equal(y, y0)
    _lib.call('pf3d_nn_conv_dx', B, H, W, C, stride, dy.data_ptr(), wb.data_ptr(), N,
              dx.data_ptr(), accumulate, st)
    gemm(Kd, N, dy, (1, Kd), col)
    _lib.call('pf3d_nn_col2im', B, H, W, C, stride, col.data_ptr(), dxc.data_ptr(), accumulate, st)
    assert torch.equal(dx, dxc)


@pytest.mark.parametrize('rows, C', [(1, 1), (1, 6), (41, 6), (43, 6), (129, 32), (1000, 128),
                                     (131072, 32), (5, 256), (300, 37), (2500, 3)])
@pytest.mark.parametrize('masked', [True, False])
def test_relu_bias_gradient(rows, C, masked):
    """Mask and column sums for 1 to 256 channels (a multiple of 4 or not,
    dividing 256 or not), less and more rows than row lanes, one and many
    chunks; dy changed only by the mask.  Whole numbers up to 3: the sums are
    exact."""
    from pyfe3d_amd import _lib
    rng = np.random.default_rng(rows + C)
    dy = rng.integers(-3, 4, (rows, C)).astype(np.float32)
    y = rng.normal(size=(rows, C)).astype(np.float32)
    y[rng.random((rows, C)) < 0.1] = 0.
    want = np.where(y > 0, dy, 0.) if masked else dy
    for floats in (C, 4 * C, 1024 * C):
        d, db = T(dy, torch.float32), torch.full((C,), float('nan'), device=DEV)
        work = torch.empty(floats, device=DEV)
        ty = T(y, torch.float32)
        _lib.call('pf3d_nn_relu_bias_grad', rows, C, ty.data_ptr() if masked else None,
                  d.data_ptr(), db.data_ptr(), work.data_ptr(), floats,
                  torch.cuda.current_stream().cuda_stream)
        assert (d.cpu().numpy() == want).all()
        assert (db.cpu().numpy() == want.astype(np.float64).sum(axis=0)).all()


@pytest.mark.parametrize('splits', [2, 15, 16, 17, 300, 1024])
def test_split_products(splits):
    """Thin products divided into many slices (one output tile, slices of
    32 to 131,072 / splits terms).  Whole numbers up to 3: the sums are
    exact."""
    from pyfe3d_amd import _lib
    rng = np.random.default_rng(splits)
    K, M, N = 131072 if splits > 64 else 4096, 32, 18
    a, b = (rng.integers(-3, 4, (K, n)).astype(np.float64) for n in (M, N))
    ta, tb = T(a, torch.float32), T(b, torch.float32)
    c = torch.full((M, N), 2., device=DEV)
    part = torch.full((splits * M * N,), float('nan'), device=DEV)
    _lib.call('pf3d_nn_gemm', M, N, K, ta.data_ptr(), 1, M, tb.data_ptr(), 1, N, c.data_ptr(), N,
              1, None, 0, splits, part.data_ptr(), torch.cuda.current_stream().cuda_stream)
    assert (c.cpu().numpy() == a.T @ b + 2.).all()


@pytest.mark.parametrize('M, N', [(32, 18), (16384, 64), (16385, 64), (4194240, 65)])
def test_split_products_of_many_entries(M, N):
    """Products divided into two slices with few entries, at the line between
    16 threads and one per entry, and with more than 2^28: every entry."""
    from pyfe3d_amd import _lib
    K = 64
    a = torch.ones((M, K), device=DEV)
    a *= (torch.arange(M, device=DEV) % 5).to(torch.float32)[:, None]
    b = (torch.arange(N, device=DEV) % 3).to(torch.float32)[:, None].repeat(1, K)
    c = torch.full((M, N), -1., device=DEV)
    part = torch.empty(2 * M * N, device=DEV)
    _lib.call('pf3d_nn_gemm', M, N, K, a.data_ptr(), K, 1, b.data_ptr(), K, 1, c.data_ptr(), N,
              0, None, 0, 2, part.data_ptr(), torch.cuda.current_stream().cuda_stream)
    assert torch.equal(c, K * a[:, :1] * b[:, 0])


@pytest.mark.parametrize('rows', [1, 3, 4, 5, 12287, 12288, 12301])
def test_product_row_routes(rows):
    """One and four block rows per wave at the line between them and at the
    ends: the product and a smoothing step (with the choices of xacc) against
    float64 sums of the same chain matrix."""
    from pyfe3d_amd import _lib
    rng = np.random.default_rng(rows)
    nb = [[j for j in (i - 1, i, i + 1) if 0 <= j < rows] for i in range(rows)]
    rp = np.concatenate([[0], np.cumsum([len(s) for s in nb])])
    ci = np.concatenate(nb)
    val = rng.normal(size=(ci.size, 6, 6))
    x, b, d, D = (rng.normal(size=s) for s in ((rows, 6), (rows, 6), (rows, 6), (rows, 6, 6)))
    q = np.zeros((rows, 6))
    np.add.at(q, np.repeat(np.arange(rows), np.diff(rp)), np.einsum('nij,nj->ni', val, x[ci]))
    t = lambda a: T(np.ascontiguousarray(a).reshape(-1), torch.float64)
    trp, tci, tv, tx, tb, td, tD = (T(rp, torch.int32), T(ci, torch.int32), t(val), t(x), t(b),
                                    t(d), t(D))
    st = torch.cuda.current_stream().cuda_stream
    y = torch.full((6 * rows,), float('nan'), dtype=torch.float64, device=DEV)
    _lib.call('pf3d_bsr_spmv', rows, trp.data_ptr(), tci.data_ptr(), tv.data_ptr(), tx.data_ptr(),
              y.data_ptr(), st)
    # 18 products of unit size: a few eps of their sum
    assert np.abs(y.cpu().numpy() - q.ravel()).max() <= 1e-13
    r = b - q
    dn = 0.7 * np.einsum('nij,nj->ni', D, r) + 0.3 * d
    for xmode in range(4):
        tr, tn, acc = y.clone(), torch.full_like(y, float('nan')), t(b)
        _lib.call('pf3d_bsr_smooth', rows, trp.data_ptr(), tci.data_ptr(), tv.data_ptr(),
                  tx.data_ptr(), tb.data_ptr(), tr.data_ptr(), tD.data_ptr(), td.data_ptr(),
                  tn.data_ptr(), acc.data_ptr(), 1., -1., 0.7, 0.3, xmode, st)
        want = (0. if xmode & 1 else b) + d + (dn if xmode & 2 else 0.)
        assert np.abs(tr.cpu().numpy() - r.ravel()).max() <= 1e-13
        assert np.abs(tn.cpu().numpy() - dn.ravel()).max() <= 1e-12
        assert np.abs(acc.cpu().numpy() - want.ravel()).max() <= 1e-12


@pytest.mark.parametrize('etype', ['quad4', 'quad4r', 'tria3r'])
@pytest.mark.parametrize('n_elem', [1, 31, 32, 33, 63, 64, 65, 97])
def test_stream_block_edges(etype, n_elem):
    """KG and M of a last block of 1 to 64 elements (32 for M) against the
    oracle, with and without slot offsets, nothing written past the end."""
    from pyfe3d_amd import assembly as A
    from test_gpu_assembly import TOL, element_errors
    x, conn, props, u, kw = _mixed_mesh(etype)
    conn, pid, xmat = conn[:n_elem], kw['pid'][:n_elem], kw['xmat'][:n_elem]
    args = T(x, torch.float64), T(6 * conn, torch.int64)
    gkw = dict(pid=T(pid, torch.int32), xmat=T(xmat, torch.float64))
    rec = T(props, torch.float64)
    for mat, mtype in (('KG', 0), ('M', 0), ('M', 1), ('M', 2)):
        size = O.slot_count(etype, mat, mtype)
        k0 = size * np.arange(n_elem)
        rr = np.zeros(size * n_elem, np.int64); cc = np.zeros_like(rr); vv = np.zeros(rr.size)
        O.assemble(etype, mat, x, conn, k0, xmat, pid, props, rr, cc, vv, mtype=mtype,
                   k6rot=kw['k6rot'][:n_elem], alpha=kw['alpha'][:n_elem],
                   hg=kw['hg'][:n_elem], u=u)
        for init_k in (None, T(k0, torch.int64)):
            r = torch.full((rr.size + 2,), -7, dtype=torch.int64, device=DEV)
            c, v = r.clone(), torch.full((rr.size + 2,), -7., dtype=torch.float64, device=DEV)
            kk = dict(gkw, init_k=init_k, overwrite=True)
            if mat == 'KG':
                A.shell_kg(etype, *args, T(u, torch.float64), r, c, v, rec, **kk)
            else:
                A.shell_m(etype, *args, r, c, v, rec, mtype=mtype, **kk)
            assert (r[-2:] == -7).all() and (c[-2:] == -7).all() and (v[-2:] == -7.).all()
            assert (r[:-2].cpu().numpy() == rr).all() and (c[:-2].cpu().numpy() == cc).all()
            assert element_errors(v[:-2].cpu().numpy(), vv, size, np.arange(n_elem)) <= TOL


@pytest.mark.parametrize('flexible', [0, 1])
@pytest.mark.parametrize('n', [6, 3000, 300006])
def test_cg_updates_two_ways(n, flexible):
    """A conjugate-gradient step with the scalars formed by separate dot
    products (pf3d_cg_update_xr, _beta, _update_p) and left as partial sums
    (pf3d_cg_step_xr, _dots, _step_p): the same bits, and numpy's values."""
    from pyfe3d_amd import _lib
    rng = np.random.default_rng(n)
    st = torch.cuda.current_stream().cuda_stream
    p, q, x, r, z, zold = (rng.normal(size=n) for _ in range(6))
    q = q + 3. * p  # (p.q well away from zero)
    d = {k: T(v, torch.float64) for k, v in dict(p=p, q=q, z=z, zold=zold).items()}
    rz = float(rng.uniform(1, 2))
    got = []
    for fused in (False, True):
        tx, tr, tp = T(x, torch.float64), T(r, torch.float64), T(p, torch.float64)
        s = torch.zeros(8, dtype=torch.float64, device=DEV)
        work = torch.zeros(3 * 1024, dtype=torch.float64, device=DEV)
        at = lambda i: s.data_ptr() + 8 * i
        s[7 if fused else 0] = rz
        if fused:
            _lib.call('pf3d_cg_step_xr', n, at(0), work.data_ptr(), tp.data_ptr(),
                      d['q'].data_ptr(), tx.data_ptr(), tr.data_ptr(), st)
            _lib.call('pf3d_cg_dots', n, tr.data_ptr(), d['z'].data_ptr(),
                      d['zold'].data_ptr() if flexible else None, work.data_ptr(), st)
            _lib.call('pf3d_cg_step_p', n, at(0), work.data_ptr(), flexible, d['z'].data_ptr(),
                      tp.data_ptr(), st)
        else:
            dot = lambda a, b, i: _lib.call('pf3d_dot', n, a.data_ptr(), b.data_ptr(), at(i),
                                            work.data_ptr(), st)
            dot(tp, d['q'], 1)
            _lib.call('pf3d_cg_update_xr', n, at(0), tp.data_ptr(), d['q'].data_ptr(),
                      tx.data_ptr(), tr.data_ptr(), st)
            dot(tr, d['z'], 3)
            dot(tr, d['zold'], 6)
            _lib.call('pf3d_cg_beta', at(0), flexible, st)
            _lib.call('pf3d_cg_update_p', n, at(0), d['z'].data_ptr(), tp.data_ptr(), st)
        got.append((tx, tr, tp))
    assert all(torch.equal(a, b) for a, b in zip(*got))
    alpha = rz / (p @ q)
    r1 = r - alpha * q
    p1 = z + (r1 @ z - (r1 @ zold if flexible else 0.)) / rz * p
    for a, b in zip(got[0], (x + alpha * p, r1, p1)):
        assert np.linalg.norm(a.cpu().numpy() - b) <= 1e-12 * np.linalg.norm(b)


@pytest.mark.parametrize('rows', [5, 12300])
@pytest.mark.parametrize('dt', [torch.float64, torch.float32])
def test_fused_step_is_the_plain_smoothing_step(rows, dt):
    """pf3d_bsr_fused(_f32) and pf3d_bsr_smooth(_f32) without a choice for
    xacc: the same bits."""
    from pyfe3d_amd import _lib
    rng = np.random.default_rng(rows)
    nb = [[j for j in (i - 1, i, i + 1) if 0 <= j < rows] for i in range(rows)]
    rp = T(np.concatenate([[0], np.cumsum([len(k) for k in nb])]), torch.int32)
    ci = T(np.concatenate(nb), torch.int32)
    new = lambda n: T(rng.normal(size=n), dt)
    val, x, b, d, D = new(36 * ci.numel()), new(6 * rows), new(6 * rows), new(6 * rows), new(36 * rows)
    acc0, st = new(6 * rows), torch.cuda.current_stream().cuda_stream
    out = []
    for name, extra in (('pf3d_bsr_fused', ()), ('pf3d_bsr_smooth', (0,))):
        r, dn, acc = torch.zeros_like(x), torch.zeros_like(x), acc0.clone()
        _lib.call(name + ('' if dt == torch.float64 else '_f32'), rows, rp.data_ptr(),
                  ci.data_ptr(), val.data_ptr(), x.data_ptr(), b.data_ptr(), r.data_ptr(),
                  D.data_ptr(), d.data_ptr(), dn.data_ptr(), acc.data_ptr(), 1., -1., 0.7, 0.3,
                  *extra, st)
        out.append((r, dn, acc))
    assert all(torch.equal(a, c) for a, c in zip(*out))
    assert torch.equal(out[0][2], acc0 + d) and float(out[0][1].abs().max()) > 0


@pytest.mark.parametrize('rows, C', [(1, 1), (300, 37), (2500, 64), (5, 300)])
def test_mask_and_column_sums_apart(rows, C):
    """pf3d_nn_relu_bwd and pf3d_nn_bias_grad (any channel count), whole
    numbers up to 3: exact."""
    from pyfe3d_amd import _lib
    rng = np.random.default_rng(rows + C)
    st = torch.cuda.current_stream().cuda_stream
    dy, y = (rng.integers(-3, 4, (rows, C)).astype(np.float32) for _ in range(2))
    d, ty = T(dy, torch.float32), T(y, torch.float32)
    _lib.call('pf3d_nn_relu_bwd', dy.size, ty.data_ptr(), d.data_ptr(), st)
    want = np.where(y > 0, dy, 0.)
    assert (d.cpu().numpy() == want).all()
    db, work = torch.full((C,), float('nan'), device=DEV), torch.empty(4 * C, device=DEV)
    _lib.call('pf3d_nn_bias_grad', rows, C, d.data_ptr(), db.data_ptr(), work.data_ptr(), 4 * C, st)
    assert (db.cpu().numpy() == want.astype(np.float64).sum(axis=0)).all()


@pytest.mark.parametrize('sizes', [(1,), (255, 256, 257, 70000)])
def test_adam_of_several_tensors(sizes):
    """pf3d_nn_adam_many: the bits of pf3d_nn_adam on each tensor."""
    from pyfe3d_amd import _lib
    import ctypes
    rng = np.random.default_rng(len(sizes))
    st = torch.cuda.current_stream().cuda_stream
    make = lambda: [T(np.abs(rng.normal(size=n)), torch.float32) for n in sizes]
    p, g, m, v = make(), make(), make(), make()
    p1, m1, v1 = ([t.clone() for t in ts] for ts in (p, m, v))
    ptrs = lambda ts: (ctypes.c_void_p * len(ts))(*[t.data_ptr() for t in ts])
    _lib.call('pf3d_nn_adam_many', len(sizes), (ctypes.c_int64 * len(sizes))(*sizes), ptrs(p),
              ptrs(g), ptrs(m), ptrs(v), 1e-2, 0.9, 0.99, 1e-8, 3, st)
    for i, n in enumerate(sizes):
        _lib.call('pf3d_nn_adam', n, p1[i].data_ptr(), g[i].data_ptr(), m1[i].data_ptr(),
                  v1[i].data_ptr(), 1e-2, 0.9, 0.99, 1e-8, 3, st)
        assert torch.equal(p[i], p1[i]) and torch.equal(m[i], m1[i]) and torch.equal(v[i], v1[i])
