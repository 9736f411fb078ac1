"""The host analysis of the nested-dissection solver: its elimination trees,
and its index maps carried through a factorisation and a solve in numpy."""
import ctypes

import numpy as np
import pytest

from pyfe3d_amd import _lib

FRONT = np.dtype([(k, np.int64) for k in ('loff', 'uoff', 'doff', 'noff', 'woff')] +
                 [(k, np.int32) for k in ('own0', 'k', 'm', 'c0', 'c1', 'depth')])
LINE = 16


class Plan:
    """The arrays of a plan's device image."""

    def __init__(self, row_ptr, col_idx, node0=None, coord=None, leaf=16):
        rp, ci = np.asarray(row_ptr, np.int32), np.asarray(col_idx, np.int32)
        n = rp.size - 1
        node0 = np.asarray([0, n] if node0 is None else node0, np.int64)
        coord = None if coord is None else np.ascontiguousarray(coord, np.int32)
        plan = ctypes.c_void_p()
        _lib.call('pf3d_nd_create', n, rp.ctypes.data, ci.ctypes.data,
                  None if coord is None else coord.ctypes.data, node0.size - 1, node0.ctypes.data,
                  leaf, ctypes.byref(plan))
        sizes, flops = (ctypes.c_int64 * 6)(), ctypes.c_double()
        _lib.call('pf3d_nd_sizes', plan, sizes, ctypes.byref(flops))
        image = np.empty(sizes[0], np.uint8)
        _lib.call('pf3d_nd_image', plan, image.ctypes.data)
        _lib.load().pf3d_nd_free(plan)
        self.n, self.factor_size = n, sizes[1]
        self.fronts = image[:64 * sizes[4]].view(FRONT)
        lists = int(((self.fronts['k'] + self.fronts['m']) // 6).sum())
        end = sizes[0]
        for name, count, dt in (('rdest', n, np.int64), ('dest', rp[-1], np.int64),
                                ('rld', n, np.int32), ('ld', rp[-1], np.int32),
                                ('pnode', n, np.int32), ('cmap', 2 * lists, np.int32),
                                ('nodes', lists, np.int32)):
            size = int(count) * np.dtype(dt).itemsize
            end -= -(-size // 256) * 256
            setattr(self, name, image[end:end + size].view(dt))
        self.levels = int(self.fronts['depth'].max()) + 1

    def solve(self, val, f):
        """What the kernels do with the plan, a front at a time."""
        L = np.zeros(self.factor_size)
        for b in np.flatnonzero(self.dest >= 0):
            c, r = np.divmod(np.arange(36), 6)
            to = self.dest[b] + c * abs(self.ld[b]) + r
            v = val[b] if self.ld[b] > 0 else val[b].T
            L[to] = v[r, c]
        update, panel = {}, {}
        for i, F in enumerate(self.fronts):  # children before parents
            k, n = int(F['k']), int(F['k'] + F['m'])
            ld = -(-(n + 1) // LINE) * LINE
            A = np.zeros((n, n))
            A[:, :k] = L[F['loff']:F['loff'] + ld * k].reshape(k, ld)[:, :n].T
            A = np.tril(A)
            cmap = self.cmap[2 * F['noff']:2 * F['noff'] + n // 3].reshape(-1, 2)
            for c, kid in enumerate((F['c0'], F['c1'])):
                if kid < 0:
                    continue
                mine = np.flatnonzero(cmap[:, c] >= 0)
                at = (6 * mine[:, None] + np.arange(6)).ravel()
                of = (6 * cmap[mine, c][:, None] + np.arange(6)).ravel()
                assert sorted(of) == list(range(len(update[kid])))
                A[np.ix_(at, at)] += update[kid][np.ix_(of, of)]
            A = np.tril(A) + np.tril(A, -1).T
            L11 = np.linalg.cholesky(A[:k, :k]) if k else np.zeros((0, 0))
            L21 = np.linalg.solve(L11, A[:k, k:]).T if k else np.zeros((n, 0))
            panel[i] = L11, L21
            update[i] = A[k:, k:] - L21 @ L21.T
        y = f.reshape(-1, 6)[self.pnode].ravel().copy()
        dofs = lambda i: (6 * self.nodes[self.fronts[i]['noff']:][:(
            self.fronts[i]['k'] + self.fronts[i]['m']) // 6][:, None] + np.arange(6)).ravel()
        for i, (L11, L21) in panel.items():
            d, k = dofs(i), len(L11)
            y[d[:k]] = np.linalg.solve(L11, y[d[:k]])
            y[d[k:]] -= L21 @ y[d[:k]]
        for i, (L11, L21) in reversed(panel.items()):
            d, k = dofs(i), len(L11)
            y[d[:k]] = np.linalg.solve(L11.T, y[d[:k]] - L21.T @ y[d[k:]])
        x = np.empty((self.n, 6))
        x[self.pnode] = y.reshape(-1, 6)
        return x.ravel()


def _pattern(n, edges):
    """row_ptr, col_idx of a graph (with its diagonal)."""
    e = np.asarray(edges, np.int64).reshape(-1, 2)
    d = np.arange(n)
    r = np.concatenate([e[:, 0], e[:, 1], d])
    c = np.concatenate([e[:, 1], e[:, 0], d])
    r, c = np.unique(r * n + c) // n, np.unique(r * n + c) % n
    return np.concatenate([[0], np.cumsum(np.bincount(r, minlength=n))]), c


def _grid(nx, ny, at=0):
    i, j = np.divmod(np.arange(nx * ny), ny)
    return [(at + a, at + b) for di, dj in ((0, 1), (1, 0), (1, 1), (1, -1))
            for a, b in zip(range(nx * ny), (i + di) * ny + j + dj)
            if i[a] + di < nx and 0 <= j[a] + dj < ny]


def _chain(nodes):
    return list(zip(nodes[:-1], nodes[1:]))


def _comb(spine, tooth):
    e = _chain([tooth * s for s in range(spine)])
    for s in range(spine):
        e += _chain(list(range(tooth * s, tooth * (s + 1))))
    return spine * tooth, e


def _values(n, rp, ci, rng):
    """Random blocks of a symmetric, diagonally dominant matrix, and it."""
    A = np.zeros((n, 6, n, 6))
    rows = np.repeat(np.arange(n), np.diff(rp))
    for r, c in zip(rows, ci):
        if r >= c:
            B = rng.normal(size=(6, 6))
            A[r, :, c] = B
            A[c, :, r] = B.T
    A = A.reshape(6 * n, 6 * n)
    A = (A + A.T) / 2
    A += np.diag(np.abs(A).sum(axis=1))
    return np.array([A.reshape(n, 6, n, 6)[r, :, c] for r, c in zip(rows, ci)]), A


GRAPHS = {
    'grid': (9 * 8, _grid(9, 8)),
    'three parts': (8 * 7 + 40 + 1, _grid(8, 7) + _chain(list(range(56, 96)))),
    'parts of one size': (25 * 6, [e for s in range(6) for e in _grid(5, 5, 25 * s)]),
    'isolated': (40, []),
    'comb': _comb(30, 4),
    # the hub leaves 12 chains, and a grid beside them
    'star': (1 + 12 * 9 + 36, [e for a in range(12) for e in
                               _chain([0] + list(range(1 + 9 * a, 10 + 9 * a)))] +
             _grid(6, 6, 109)),
}


@pytest.mark.parametrize('name', sorted(GRAPHS))
@pytest.mark.parametrize('leaf', [1, 4, 16])
def test_maps_solve(name, leaf):
    """A factorisation and a solve with the plan's own maps against numpy's,
    on connected and separate parts."""
    n, edges = GRAPHS[name]
    rp, ci = _pattern(n, edges)
    rng = np.random.default_rng(n)
    val, A = _values(n, rp, ci, rng)
    f = rng.normal(size=6 * n)
    x = Plan(rp, ci, leaf=leaf).solve(val, f)
    assert np.abs(x - np.linalg.solve(A, f)).max() <= 1e-12


def test_separate_parts_share_the_levels():
    """Parts that are not connected stand beside each other in the tree: as
    many levels as the largest of them has alone, and no recursion as deep
    as there are parts."""
    alone = Plan(*_pattern(169, _grid(13, 13))).levels
    assert Plan(*_pattern(50 * 169, [e for s in range(50) for e in _grid(13, 13, 169 * s)])) \
        .levels == alone
    assert Plan(np.arange(60001), np.arange(60000)).levels == 1
    quads = np.arange(160000).reshape(-1, 4)
    plan = Plan(4 * np.arange(160001), np.repeat(quads, 4, axis=0).ravel())
    assert plan.levels == 1 and plan.fronts.size == 40000


@pytest.mark.parametrize('spine, tooth', [(2000, 10), (20000, 3)])
def test_tree_of_a_comb_is_flat(spine, tooth):
    """A long connected pattern whose smallest separators cut off one tooth:
    no side holds more than 70 % of what is divided, so log(n / leaf) /
    log(1 / 0.7) levels."""
    n, edges = _comb(spine, tooth)
    assert Plan(*_pattern(n, edges)).levels <= np.log(n / 16) / np.log(1 / 0.7) + 2


def _bush(teeth, twigs, length):
    """Branches of a spine that end at the same distance from its start, each
    in a bush."""
    e, n, spine = [], 0, []
    for i in range(teeth):
        tooth = list(range(n, n + teeth - i))
        n += teeth - i
        spine.append(tooth[0])
        e += _chain(tooth)
        for _ in range(twigs):
            twig = list(range(n, n + length))
            n += length
            e += _chain([tooth[-1]] + twig)
    return n, e + _chain(spine)


@pytest.mark.parametrize('teeth, twigs, length', [(20, 20, 3), (30, 30, 2), (32, 31, 2),
                                                  (45, 40, 2)])
def test_wide_levels_are_not_separators(teeth, twigs, length):
    """Levels of up to 1,800 nodes in patterns with a narrow band: no front
    much wider than the band."""
    n, edges = _bush(teeth, twigs, length)
    rp, ci = _pattern(n, edges)
    band = np.abs(np.repeat(np.arange(n), np.diff(rp)) - ci).max()
    plan = Plan(rp, ci)
    # a separator and what it touches of the ones around
    assert (plan.fronts['k'] + plan.fronts['m']).max() <= 3 * 6 * band


@pytest.mark.parametrize('keep', ['lower', 'upper', 'random'])
@pytest.mark.parametrize('name', sorted(GRAPHS))
def test_one_sided_blocks(name, keep):
    """Blocks stored on one side of the diagonal only stand for both: no map
    entry leaves its front, and the solution is the symmetric matrix's."""
    n, edges = GRAPHS[name]
    rp, ci = _pattern(n, edges)
    rng = np.random.default_rng(n)
    val, A = _values(n, rp, ci, rng)
    rows = np.repeat(np.arange(n), np.diff(rp))
    if keep == 'random':  # of every third pair, one block, either one
        pair = {(r, c): rng.integers(3) for r, c in zip(rows, ci) if r > c}
        on = np.array([r == c or pair[max(r, c), min(r, c)] != int(r > c) for r, c in zip(rows, ci)])
    else:
        on = rows >= ci if keep == 'lower' else rows <= ci
    orp = np.concatenate([[0], np.cumsum(np.bincount(rows[on], minlength=n))])
    plan = Plan(orp, ci[on])
    front = np.searchsorted(plan.fronts['loff'], plan.dest, side='right') - 1
    for b in np.flatnonzero(plan.dest >= 0):
        F = plan.fronts[front[b]]
        col, row = divmod(plan.dest[b] - F['loff'], abs(plan.ld[b]))
        assert col + 6 <= F['k'] and row + 6 <= F['k'] + F['m']
    f = rng.normal(size=6 * n)
    assert np.abs(plan.solve(val[on], f) - np.linalg.solve(A, f)).max() <= 1e-12
