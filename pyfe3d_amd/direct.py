"""Direct solves by nested dissection (csrc/dissect.hip): a sparse Cholesky
factor of the Dirichlet-treated stiffness, for one system or for the
independent systems of a design sweep, in place of the reference callers'
``spsolve`` (tests/test_quad4_static_point_load.py:84-102).

A :class:`DirectPlan` is the symbolic part: the elimination tree of a block
pattern, its index maps and launch lists.  It depends on the pattern only and
is kept with it; ``factor`` and ``solve`` launch kernels and neither allocate
nor synchronise, so they can be captured in a graph.
"""
import ctypes

import numpy as np
import torch

from . import _lib

# separators are sought in parts of more nodes than this (measured on the
# 64 x 48 plate and on a sweep of 512 plates)
LEAF_NODES = 16


class DirectPlan:
    """row_ptr, col_idx: host BSR pattern (int32) of n_sys independent
    systems, system s owning block rows [node0[s], node0[s + 1]); coord:
    (n_nodes, 2) integer grid position of every node of structured plates
    (else separators are found from the pattern)."""

    def __init__(self, row_ptr, col_idx, device, coord=None, node0=None, leaf=LEAF_NODES):
        rp = np.ascontiguousarray(row_ptr, dtype=np.int32)
        ci = np.ascontiguousarray(col_idx, dtype=np.int32)
        self.n_nodes = rp.size - 1
        if node0 is None:
            node0 = [0, self.n_nodes]
        node0 = np.ascontiguousarray(node0, dtype=np.int64)
        if coord is not None:
            coord = np.ascontiguousarray(coord, dtype=np.int32)
            if coord.shape != (self.n_nodes, 2):
                raise ValueError('coord must have shape (n_nodes, 2)')
        if ci.size < rp[-1]:
            raise ValueError('col_idx has %d entries, row_ptr says %d' % (ci.size, rp[-1]))
        self.device = torch.device(device)
        self._made = (rp, ci, self.device, coord, node0, int(leaf))  # (for pickling)
        self._plan = ctypes.c_void_p()
        self._free = _lib.load().pf3d_nd_free
        _lib.call('pf3d_nd_create', self.n_nodes, rp.ctypes.data, ci.ctypes.data,
                  None if coord is None else coord.ctypes.data, node0.size - 1,
                  node0.ctypes.data, int(leaf), ctypes.byref(self._plan))
        sizes = (ctypes.c_int64 * 6)()
        flops = ctypes.c_double()
        _lib.call('pf3d_nd_sizes', self._plan, sizes, ctypes.byref(flops))
        self.factor_size, self.update_size, self.work_size = sizes[1], sizes[2], sizes[3]
        self.n_fronts, self.widest, self.flops = sizes[4], sizes[5], flops.value
        image = np.empty(sizes[0], dtype=np.uint8)
        _lib.call('pf3d_nd_image', self._plan, image.ctypes.data)
        self.image = torch.as_tensor(image, device=self.device)
        self.stream = torch.cuda.current_stream(self.device).cuda_stream  # (the image's)

    def __del__(self):
        plan, self._plan = getattr(self, '_plan', None), None
        if plan:
            self._free(plan)

    def __deepcopy__(self, memo):
        return self  # (read-only)

    def __reduce__(self):
        return DirectPlan, self._made

    def factor(self, val, factor, update, bad, stream, f=None):
        """Cholesky factor of the systems with BSR values val (device
        address) into factor (factor_size doubles); update (update_size) is
        scratch; bad counts systems' panels with a non-positive pivot.  f: a
        right-hand side (device address) whose forward substitution is
        carried along; :meth:`solve` with f None then finishes it."""
        _lib.call('pf3d_nd_factor', self._plan, self.image.data_ptr(), val, f, factor.data_ptr(),
                  update.data_ptr(), bad.data_ptr(), stream)

    def solve(self, factor, f, x, work, stream):
        """x = A^-1 f (device addresses; 6 doubles per node); f None: the
        right-hand side given to :meth:`factor`."""
        _lib.call('pf3d_nd_solve', self._plan, self.image.data_ptr(), factor.data_ptr(), f, x,
                  work.data_ptr(), stream)


class DirectBatch:
    """The systems of a block-diagonal BSR matrix (a design sweep) solved in
    groups of consecutive systems that share one factor and scratch storage:
    a group is factorised and solved before the next one."""

    # block rows per group: enough fronts to fill the GPU at every tree
    # level, a bounded factor (about 12 KB per block row)
    GROUP_NODES = 1000000

    def __init__(self, row_ptr, col_idx, device, node0, coord=None):
        rp = np.asarray(row_ptr)
        ci = np.asarray(col_idx)
        node0 = np.asarray(node0, dtype=np.int64)
        self.groups = []
        s = 0
        while s < node0.size - 1:
            e = s + 1
            while e < node0.size - 1 and node0[e + 1] - node0[s] <= self.GROUP_NODES:
                e += 1
            a, b = int(node0[s]), int(node0[e])
            b0, b1 = int(rp[a]), int(rp[b])
            plan = DirectPlan(rp[a:b + 1] - b0, ci[b0:b1] - a, device,
                              coord=None if coord is None else coord[a:b],
                              node0=node0[s:e + 1] - a)
            self.groups.append((plan, 8 * 36 * b0, 8 * 6 * a))  # (byte offsets of val, f and x)
            s = e
        buf = lambda size: torch.empty(max(1, max(size(g[0]) for g in self.groups)),
                                       dtype=torch.float64, device=device)
        self.factor = buf(lambda p: p.factor_size)
        self.update = buf(lambda p: p.update_size)
        self.work = buf(lambda p: p.work_size)
        self.bad = torch.zeros(1, dtype=torch.int32, device=device)

    def solve(self, val, f, x, stream):
        """x = A^-1 f for BSR values val (contiguous FP64 tensors)."""
        for plan, vo, fo in self.groups:
            plan.factor(val.data_ptr() + vo, self.factor, self.update, self.bad, stream,
                        f=f.data_ptr() + fo)
            plan.solve(self.factor, None, x.data_ptr() + fo, self.work, stream)
