"""Rank-local node boxes: Dirichlet rows on every masked dof of the box, those of ghost nodes that no
owned element holds among them (PTQ2_MATMULT: "Dirichlet rows replaced on output"), in every form and
precision of the operators, and the other ghost dofs as the caller left them."""
import ctypes

import numpy as np
import pytest

from oracle import oracle as O
import ptq2
from ptq2 import _lib
from ptq2 import mesh as M

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
DEV = torch.device("cuda:0")

# elements, ghost nodes before and after the elements' along x, y, z
BOXES = [((6, 5, 7), (2, 1, 3), (2, 1, 2)), ((4, 8, 4), (0, 2, 1), (3, 0, 0)), ((1, 2, 9), (1, 1, 0), (0, 9, 1)),
         ((3, 4, 5), (0, 0, 0), (0, 0, 0))]


class GhostBox:
    def __init__(self, dims, lo, hi):
        self.dims, self.lo = dims, lo
        N = [2 * m + 1 + a + b for m, a, b in zip(dims, lo, hi)]
        c = np.stack(np.meshgrid(*[np.linspace(0, 1, n) for n in N], indexing="ij"), axis=-1).transpose(2, 1, 0, 3).copy()
        c += M.uniform(77, c.size, -0.1, 0.1).reshape(c.shape) / max(N)
        self.coords, self.shape = c, c.shape
        self.mask = (M.uniform(78, c.size) < 0.1).astype(np.uint8).reshape(c.shape)
        self.mask[:, :, 0] = 1  # a whole face, of ghost nodes if there are any
        self.own = np.zeros(c.shape, dtype=bool)
        self.own[tuple(slice(a, a + 2 * m + 1) for a, m in zip(lo[::-1], dims[::-1]))] = True
        self.eta = 10.0 ** M.uniform(79, 27 * int(np.prod(dims)), -1, 1)
        self.ctx = ptq2.Context(0)
        h = self.ctx.handle
        _lib.check(_lib.lib().ptq2_setup_mesh_box(h, *dims, *N, *lo, c.ctypes.data, self.mask.ctypes.data),
                   "setup_mesh_box", h)
        self.ctx.nvel, self.ctx.npres = c.size, 4 * int(np.prod(dims))
        self.ctx.set_viscosity(self.eta)

    def sub(self, a):
        return np.ascontiguousarray(a.reshape(self.shape)[self.own])

    def check(self, y, y0, ref_sub, dirichlet, tol):
        """Owned nodes against the oracle, masked dofs bit for bit, the other ghost dofs untouched."""
        y, y0, d = np.asarray(y).reshape(self.shape), np.asarray(y0).reshape(self.shape), self.mask > 0
        want = np.broadcast_to(np.asarray(dirichlet, dtype=y.dtype), y.size).reshape(self.shape)
        assert np.array_equal(y[d], want[d])
        assert np.array_equal(y[~d & ~self.own], y0[~d & ~self.own])
        free = self.sub(self.mask) == 0
        got = self.sub(y).astype(np.float64)
        assert np.linalg.norm((got - ref_sub)[free]) <= tol * np.linalg.norm(ref_sub[free])


@pytest.mark.parametrize("dims,lo,hi", BOXES)
def test_dirichlet_rows_of_ghost_nodes(dims, lo, hi):
    print("case: ghost Dirichlet rows", dims, lo, hi, flush=True)
    B = GhostBox(dims, lo, hi)
    c, L = B.ctx, _lib.lib()
    n, ne = B.coords.size, int(np.prod(dims))
    u, p = M.uniform(3, n, -1, 1), M.uniform(4, 4 * ne, -1, 1)
    y0 = M.uniform(5, n, -1, 1)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(DEV)
    mesh = (*dims, B.sub(B.coords))
    smask = B.sub(B.mask)
    ref = O.matmult_a11(*mesh, B.eta, smask, B.sub(u))
    y32, u32 = y0.astype(np.float32), u.astype(np.float32)
    for f in (0, _lib.ONTHEFLY, _lib.STOREDGEO):
        B.check(c.a11(dev(u), dev(y0), _lib.MATMULT | f).cpu().numpy(), y0, ref, u, 1e-12)
    for f in (0, _lib.MFMA):
        B.check(c.a11(dev(u32), dev(y32), _lib.MATMULT | _lib.FP32 | f).cpu().numpy(), y32, ref, u32, 1e-5)
    # staged host vectors: the ghost dofs without a row are not defined
    yh = c.a11(u, y0.copy(), _lib.MATMULT)
    B.check(np.where(B.own.reshape(-1) | (B.mask.reshape(-1) > 0), yh, y0), y0, ref, u, 1e-12)
    y = dev(y0)
    c._stream(y)
    ud = dev(u)
    _lib.check(L.ptq2_a11_apply_noalloc(c.handle, ud.data_ptr(), y.data_ptr(), _lib.DEVICE | _lib.MATMULT), "noalloc",
               c.handle)
    B.check(y.cpu().numpy(), y0, ref, u, 1e-12)
    B2 = GhostBox(dims, lo, hi)
    for uu, yy, f, tol in ((u, y0, 0, 1e-12), (u32, y32, _lib.FP32, 1e-5)):
        us, ys = [dev(uu), dev(uu)], [dev(yy), dev(yy)]
        ptq2.a11_batch([c, B2.ctx], us, ys, _lib.MATMULT | f)
        for q in ys:
            B.check(q.cpu().numpy(), yy, ref, uu, tol)
    # the other MatMult-like calls
    B.check(c.a12(dev(p), dev(y0), _lib.MATMULT).cpu().numpy(), y0, O.matmult_a12(*mesh, smask, p), 0.0, 1e-12)
    B.check(c.a11_diag(dev(y0), _lib.MATMULT).cpu().numpy(), y0, O.matgetdiag_a11(*mesh, B.eta, smask), 1.0, 1e-12)
    ru, _ = O.matmult_a(*mesh, B.eta, smask, B.sub(u), p)
    B.check(c.stokes(dev(u), dev(p), dev(y0), None, _lib.MATMULT)[0].cpu().numpy(), y0, ru, u, 1e-12)
    B.check(c.stokes(dev(u32), dev(p.astype(np.float32)), dev(y32), None, _lib.MATMULT | _lib.FP32)[0].cpu().numpy(),
            y32, ru, u32, 1e-5)
    B.ctx.destroy()
    B2.ctx.destroy()
