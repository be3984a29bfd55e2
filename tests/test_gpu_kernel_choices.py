"""Kernel forms that ordinary meshes do not reach: the row-split FP32 smoothers on levels of partial bricks, and
64-bit tile addressing (boxes whose tiles span more than 2 GiB)."""
import numpy as np
import pytest

from oracle import oracle as O
import ptq2
from ptq2 import _lib
from ptq2 import mesh as M
from ptq2.solver import ViscousSolver

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
DEV = torch.device("cuda:0")


def brick_mesh(dims, seed=5, mask_share=0.02):
    """Elements of edge 1, jittered, with scattered Dirichlet dofs and a Dirichlet face."""
    c = M.jitter(*dims, M.q2_uniform(*dims), 0.1, 1.0 / (2 * max(dims)), seed).reshape(-1, 3) * np.array(dims, dtype=float)
    eta = 10.0 ** M.uniform(seed + 1, 27 * int(np.prod(dims)), -1.0, 1.0)
    mask = (M.uniform(seed + 2, c.size) < mask_share).astype(np.uint8)
    mask.reshape(-1, 2 * dims[0] + 1, 3)[:, 0, :] = 1
    return c.reshape(-1), eta, mask


@pytest.mark.parametrize("dims,waves", [((14, 14, 32), 9), ((2, 2, 1030), 3)])
def test_row_split_smoother_on_partial_bricks(dims, waves):
    """Nine waves per brick where overlapping blocks would need more than 256 CUs, three beyond 256 bricks: the FP32
    V-cycle against the one-wave kernel's (the autotuner's 1e-5)."""
    print("case: row-split smoother, partial bricks", dims, waves, flush=True)
    bricks = int(np.prod([-(-m // 4) for m in dims]))
    blocks = int(np.prod([1 if m <= 4 else (m - 2) // 3 + 1 for m in dims]))
    assert any(m % 4 for m in dims) and blocks > 256 and (bricks <= 256) == (waves == 9)
    c, eta, mask = brick_mesh(dims)
    r = M.uniform(6, c.size, -1.0, 1.0)
    r[mask > 0] = 0.0
    rd = torch.from_numpy(r).to(DEV)
    z = []
    for at in (0, 2):
        ctx = ptq2.Context(0)
        ctx.setup_mesh(*dims, c, mask)
        ctx.set_viscosity(eta)
        S = ViscousSolver(ctx, nlevels=2, smooth_its=3, fp32=True, galerkin_coarse=False, autotune=at,
                          coarse_max_dofs=30000)
        assert [k for k, _, _, _ in S.tuning()] == [1 if at else 0]
        z.append(S.vcycle(rd).clone())
        assert torch.equal(S.vcycle(rd), z[-1])
        S.destroy()
        ctx.destroy()
    assert (torch.linalg.norm(z[1] - z[0]) / torch.linalg.norm(z[0])).item() <= 1e-5


def test_tiles_beyond_32_bit_offsets():
    """Every operator on a few elements in a node box of 3401 x 3301 x 12: the bits of the same elements in a box
    of their own, whose tiles use 32-bit offsets, and ghost dofs untouched next to the elements."""
    dims, lo = (5, 6, 5), (1200, 3, 1)
    print("case: 64-bit tile offsets", dims, flush=True)
    n = [2 * m + 1 for m in dims]
    N = (3401, 3301, 12)
    assert 8 * (27 + 8 * (3 * N[0] + 3 * N[0] * N[1])) >= 2 ** 31
    c, eta, mask = brick_mesh(dims, mask_share=0.1)
    sl = tuple(slice(a, a + k) for a, k in zip(lo[::-1], n[::-1]))
    shape = (N[2], N[1], N[0], 3)

    def box(a):
        b = np.zeros(shape, dtype=a.dtype)  # pages of the ghost nodes are never written
        b[sl] = a.reshape(n[2], n[1], n[0], 3)
        return b

    small, big = ptq2.Context(0), ptq2.Context(0)
    small.setup_mesh(*dims, c, mask)
    bc, bm = box(c), box(mask)
    _lib.check(_lib.lib().ptq2_setup_mesh_box(big.handle, *dims, *N, *lo, bc.ctypes.data, bm.ctypes.data), "setup_mesh_box",
               big.handle)
    big.nvel, big.npres = bc.size, 4 * int(np.prod(dims))
    del bc, bm
    for ctx in (small, big):
        ctx.set_viscosity(eta)
    ue, pe, fe = M.uniform(3, c.size, -1, 1), M.uniform(4, big.npres, -1, 1), M.uniform(5, 81 * int(np.prod(dims)), -1, 1)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(DEV)

    def vec(a, dt):
        b = torch.zeros(shape, dtype=dt, device=DEV)
        b[sl] = dev(a).to(dt).reshape(n[2], n[1], n[0], 3)
        return b

    wide = tuple(slice(max(0, s.start - 2), s.stop + 2) for s in sl)
    ref = O.matmult_a11(*dims, c, eta, mask, ue)

    def compare(call, dt=torch.float64):
        y0 = torch.full((n[2], n[1], n[0], 3), 0.25, dtype=dt, device=DEV)
        u = dev(ue).to(dt)
        ys, ps = call(small, u, y0.reshape(-1))
        yb = torch.full(shape, 0.25, dtype=dt, device=DEV)
        _, pb = call(big, vec(ue, dt).reshape(-1), yb.reshape(-1))
        assert torch.equal(yb[sl].reshape(-1), ys)
        assert ps is None or torch.equal(pb, ps)
        yb[sl] = 0.25
        assert bool((yb[wide] == 0.25).all())
        return ys

    for f in (0, _lib.ADD, _lib.MATMULT, _lib.MATMULT | _lib.STOREDGEO):
        y = compare(lambda x, u, y: (x.a11(u, y, f), None))
        if f & _lib.MATMULT:
            assert np.linalg.norm(y.cpu().numpy() - ref) <= 1e-12 * np.linalg.norm(ref)
    for f in (0, _lib.MATMULT):
        p = dev(pe)
        compare(lambda x, u, y: x.stokes(u, p, y, None, f))
        compare(lambda x, u, y: (x.a11(u, y, f | _lib.FP32), None), torch.float32)
        p32 = p.to(torch.float32)
        compare(lambda x, u, y: x.stokes(u, p32, y, None, f | _lib.FP32), torch.float32)
        compare(lambda x, u, y: (x.a12(p, y, f), x.a21(u, None, f)))
        compare(lambda x, u, y: (x.a11_diag(y, f), None))
        compare(lambda x, u, y: (x.body_force(dev(fe), y, f), None))
    small.destroy()
    big.destroy()
