"""Element passes on several waves per brick: meshes at the edges of the 4x4x4 bricks, scattered
Dirichlet masks, and the resident coordinate tiles of large meshes, against the oracle.

Tolerance: an output node sums up to 8 elements x 27 points x ~30 rounded products of FP64, whose
errors add like a random walk to well below 1e-14 of the result; 1e-12 (the operators' bar)
leaves room for cancellation between the elements of a stiff inclusion."""
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

EDGES = [(1, 1, 1), (4, 4, 4), (5, 4, 4), (4, 9, 3), (8, 8, 8), (12, 5, 8), (3, 13, 17)]


def problem(dims, seed=5, mask_share=0.05):
    mx, my, mz = dims
    c = M.jitter(mx, my, mz, M.q2_uniform(mx, my, mz), 0.1, 1.0 / (2 * max(dims)), seed)
    eta = 10.0 ** M.uniform(seed + 1, 27 * mx * my * mz, -2.0, 2.0)
    n = 3 * M.nnodes(mx, my, mz)
    # whole Dirichlet faces in x, and single dofs anywhere (inside bricks, on their faces and edges)
    mask = (M.uniform(seed + 2, n) < mask_share).astype(np.uint8)
    mask.reshape(-1, 2 * mx + 1, 3)[:, 0, :] = 1
    return M.Problem(mx, my, mz, M.affine(c, M.SHEAR, [0.0, 0.0, 0.0]), mask, eta)


def rel(a, b):
    return float(np.linalg.norm(np.asarray(a, dtype=np.float64) - b) / np.linalg.norm(b))


@pytest.mark.parametrize("dims", EDGES + [(128, 128, 32)])
def test_a11_fp64(dims):
    """Raw, ADD and MatMult applies; Dirichlet rows are u's bit for bit, ADD adds to what is there."""
    print("case: A11 FP64", dims, flush=True)
    P = problem(dims)
    A = ptq2.MatA11MF("hip")
    A.setup(P)
    u = M.uniform(3, P.nvel, -1.0, 1.0)
    ud = torch.from_numpy(u).to(DEV)
    ref = O.a11_tensor(*dims, P.coords, P.eta, u, threads=8)
    y = A.ctx.a11(ud)
    assert rel(y.cpu().numpy(), ref) <= 1e-12
    y0 = torch.full_like(ud, 0.5)
    assert rel(A.ctx.a11(ud, y0.clone(), _lib.ADD).cpu().numpy(), ref + 0.5) <= 1e-12
    ym = A.mult(ud).cpu().numpy()
    assert rel(ym, O.matmult_a11(*dims, P.coords, P.eta, P.mask, u)) <= 1e-12
    d = P.mask > 0
    assert np.array_equal(ym[d], u[d])


@pytest.mark.parametrize("dims", EDGES)
def test_gradient_divergence_diagonal(dims):
    """A12, A21 and the A11 diagonal, set and ADD; the mesh sits 50 edge lengths from the origin, where
    the pressure basis works with differences of coordinates: a point's position, a sum of 27 rounded
    terms on either side, is off by up to 27 x 50 x 2^-53 against an element's edge of 1 / max(dims)."""
    tol = max(1e-12, 2 * 27 * 50 * max(dims) * 2.0 ** -53)
    print("case: A12, A21, diagonal", dims, flush=True)
    P = problem(dims)
    P = M.Problem(*dims, P.coords + 50.0, P.mask, P.eta)
    A = ptq2.MatA11MF("hip")
    A.setup(P)
    u, p = M.uniform(3, P.nvel, -1.0, 1.0), M.uniform(4, 4 * int(np.prod(dims)), -1.0, 1.0)
    ud, pd = torch.from_numpy(u).to(DEV), torch.from_numpy(p).to(DEV)
    c = A.ctx
    for ref, y, again in (
            (O.a12(*dims, P.coords, p), c.a12(pd), lambda y0: c.a12(pd, y0, _lib.ADD)),
            (O.a21(*dims, P.coords, u), c.a21(ud), lambda y0: c.a21(ud, y0, _lib.ADD)),
            (O.diag_a11(*dims, P.coords, P.eta), c.a11_diag(device=DEV), lambda y0: c.a11_diag(y0, _lib.ADD))):
        assert rel(y.cpu().numpy(), ref) <= tol
        assert rel(again(torch.full_like(y, 0.5)).cpu().numpy(), ref + 0.5) <= tol


@pytest.mark.parametrize("dims,ppe,crowd,rho", [((1, 1, 1), 1, 0, True), ((5, 3, 9), 8, 0, True),
                                                ((8, 4, 1), 56, 0, False), ((4, 4, 3), 57, 0, True),
                                                ((6, 5, 2), 2, 400, True), ((3, 3, 3), 0, 7, False)])
def test_point_buckets(dims, ppe, crowd, rho):
    """Points that fit the elements' slots (up to 56 on average), that do not, and one element
    crowded by `crowd` more: against the oracle at the projection's bars or, if larger, the rounding of
    two weighted means of a node's n points (n 2^-53 each), and away from the crowded element bit for bit
    what the same points give without the crowd."""
    sums = 2 * (8 * ppe + crowd) * 2.0 ** -53
    print("case: point buckets", dims, ppe, crowd, flush=True)
    mx, my, mz = dims
    ne = mx * my * mz
    c = M.q2_uniform(mx, my, mz)
    wil = np.repeat(np.arange(ne), ppe)
    wil = np.concatenate([wil[np.argsort(M.uniform(9, wil.size))], np.full(crowd, ne - 1)]).astype(np.int32)
    xi = M.uniform(10, 3 * wil.size, -1.0, 1.0).reshape(-1, 3)
    eta_p, rho_p = 10.0 ** M.uniform(11, wil.size, -2.0, 3.0), M.uniform(12, wil.size, -1.0, 1.0)
    ctx = ptq2.Context(0)
    ctx.setup_mesh(mx, my, mz, c)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(DEV)

    def run(n):
        out = ctx.project_points(dev(xi[:n]), dev(wil[:n]), dev(eta_p[:n]), dev(rho_p[:n]) if rho else None)
        return [o.cpu().numpy() for o in (out if rho else [out])]

    got = run(wil.size)
    ref = O.project_q1(mx, my, mz, xi, wil, eta_p, rho_p)
    assert np.max(np.abs(got[0] - ref[0]) / np.maximum(np.abs(ref[0]), 1e-300)) <= max(1e-13, sums)
    if rho:
        assert np.max(np.abs(got[1] - ref[1])) <= max(1e-14, sums)
    if crowd and ppe:
        far = np.ones((mz, my, mx), dtype=bool)
        far[-2:, -2:, -2:] = False
        for a, b in zip(got, run(wil.size - crowd)):
            assert np.array_equal(a.reshape(ne, 27)[far.reshape(-1)], b.reshape(ne, 27)[far.reshape(-1)])
    ctx.destroy()


@pytest.mark.parametrize("dims", [(2, 2, 2), (4, 8, 12), (10, 14, 6), (20, 8, 4), (28, 28, 36)])
def test_row_split_smoother(dims):
    """The FP32 V-cycle with the row-split kernels on every level (nine waves per brick up to 256 bricks,
    three beyond) against the one-wave kernel's, on meshes of full and partial bricks with scattered
    Dirichlet dofs.  The smoother amplifies the applies' differing roundings (some 1e-7) by little:
    the autotuner's 1e-5."""
    print("case: row-split smoother", dims, flush=True)
    P = problem(dims, mask_share=0.02)
    r = M.uniform(6, P.nvel, -1.0, 1.0)
    r[P.mask > 0] = 0.0
    rd = torch.from_numpy(r).to(DEV)
    z = []
    for at in (0, 2):
        ctx = ptq2.Context(0)
        ctx.setup_mesh(*dims, P.coords, P.mask)
        ctx.set_viscosity(np.minimum(P.eta, 10.0))
        S = ViscousSolver(ctx, nlevels=3 if max(dims) > 20 else 2, smooth_its=3, fp32=True, galerkin_coarse=False,
                          autotune=at)
        z.append(S.vcycle(rd).clone())
        assert torch.equal(S.vcycle(rd), z[-1])
        S.destroy()
        ctx.destroy()
    assert (torch.linalg.norm(z[1] - z[0]) / torch.linalg.norm(z[0])).item() <= 1e-5


@pytest.mark.parametrize("dims", EDGES)
def test_full_block_and_residual(dims):
    """The full block (set, ADD, MatMult) and the residual with a continuity source, on bricks of all
    fillings, against the oracle at the operators' bar; parts of the residual by superposition."""
    print("case: full block", dims, flush=True)
    P = problem(dims)
    ne = int(np.prod(dims))
    A = ptq2.MatA11MF("hip")
    A.setup(P)
    u, p = M.uniform(3, P.nvel, -1.0, 1.0), M.uniform(4, 4 * ne, -1.0, 1.0)
    ud, pd = torch.from_numpy(u).to(DEV), torch.from_numpy(p).to(DEV)
    ru, rp = O.stokes_a(*dims, P.coords, P.eta, u, p)
    yu, yp = A.ctx.stokes(ud, pd)
    assert rel(yu.cpu().numpy(), ru) <= 1e-12 and rel(yp.cpu().numpy(), rp) <= 1e-12
    au, ap = A.ctx.stokes(ud, pd, torch.full_like(yu, 0.5), torch.full_like(yp, 0.5), _lib.ADD)
    assert rel(au.cpu().numpy(), ru + 0.5) <= 1e-12 and rel(ap.cpu().numpy(), rp + 0.5) <= 1e-12
    d = P.mask > 0
    um = np.where(d, 0.0, u)
    mu, mp = A.ctx.stokes(ud, pd, flags=_lib.MATMULT)
    ru, rp = O.stokes_a(*dims, P.coords, P.eta, um, p)
    assert rel(mu.cpu().numpy(), np.where(d, u, ru)) <= 1e-12 and rel(mp.cpu().numpy(), rp) <= 1e-12
    fu, phi = M.uniform(7, 81 * ne, -1.0, 1.0), M.uniform(8, P.nvel, -1.0, 1.0)
    fp = M.uniform(9, 27 * ne, -1.0, 1.0)
    dev = lambda a: torch.from_numpy(a).to(DEV)
    Fu, Fp = A.ctx.residual(ud, pd, dev(fu), dev(fp), dev(phi))
    ul = np.where(d, phi, u)
    ru, rp = O.stokes_a(*dims, P.coords, P.eta, ul, p)
    ru -= O.body_force(*dims, P.coords, fu)
    assert rel(Fu.cpu().numpy(), np.where(d, u - phi, ru)) <= 1e-12
    # the source alone: fp = 1 integrates the pressure basis
    z, zp = torch.zeros_like(ud), torch.zeros_like(pd)
    F1 = A.ctx.residual(z, zp, dev(0.0 * fu), dev(fp), dev(0.0 * phi))[1]
    F0 = A.ctx.residual(ud, pd, dev(fu), None, dev(phi))[1]
    assert rel(F0.cpu().numpy(), rp) <= 1e-12
    assert rel((F0 + F1).cpu().numpy(), Fp.cpu().numpy()) <= 1e-12


@pytest.mark.parametrize("dims", [(4, 4, 4), (5, 4, 4), (9, 12, 8), (3, 13, 17)])
def test_gradient_diagonal_on_a_second_stream(dims):
    """A12 and the diagonal on a stream other than the one that used the face slots first run coloured:
    set, ADD and MatMult equal to the oracle there too, and to the first stream's to rounding."""
    print("case: A12 and diagonal on a second stream", dims, flush=True)
    P = problem(dims)
    A = ptq2.MatA11MF("hip")
    A.setup(P)
    p = M.uniform(4, 4 * int(np.prod(dims)), -1.0, 1.0)
    pd = torch.from_numpy(p).to(DEV)
    c = A.ctx
    d = P.mask > 0
    side = torch.cuda.Stream(device=DEV)
    for ref, f, bc in ((O.a12(*dims, P.coords, p), lambda y, fl: c.a12(pd, y, fl), 0.0),
                       (O.diag_a11(*dims, P.coords, P.eta), lambda y, fl: c.a11_diag(y, fl), 1.0)):
        first = f(torch.zeros(P.nvel, dtype=torch.float64, device=DEV), 0)
        torch.cuda.synchronize()
        with torch.cuda.stream(side):
            y = [f(torch.full((P.nvel,), 0.5, dtype=torch.float64, device=DEV), fl) for fl in (0, _lib.ADD, _lib.MATMULT)]
        torch.cuda.synchronize()
        for got, want in zip(y, (ref, ref + 0.5, np.where(d, bc, ref))):
            assert rel(got.cpu().numpy(), want) <= 1e-12
        assert rel(first.cpu().numpy(), ref) <= 1e-12
