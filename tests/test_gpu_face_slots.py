"""A12 and the diagonal share face slots between all callers of a context: the same bits on every stream and
with a multigrid hierarchy on the context, overlapping calls on several streams, and calls captured into a graph
whose replays meet eager calls."""
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
OPS = ("a12", "diag")


def problem(dims, seed=3):
    c = M.jitter(*dims, M.q2_uniform(*dims), 0.1, 1.0 / (2 * max(dims)), seed)
    return M.Problem(*dims, c, M.bc_mask(*dims, "freeslip"), 10.0 ** M.uniform(seed, 27 * int(np.prod(dims)), -1, 1))


def context(P):
    ctx = ptq2.Context(0)
    ctx.setup_mesh(P.mx, P.my, P.mz, P.coords, P.mask)
    ctx.set_viscosity(P.eta)
    return ctx


def call(ctx, op, p, y=None):
    if y is None:
        y = torch.empty(ctx.nvel, dtype=torch.float64, device=DEV)
    return ctx.a12(p, y, _lib.MATMULT) if op == "a12" else ctx.a11_diag(y, _lib.MATMULT)


@pytest.mark.parametrize("dims", [(8, 8, 8), (16, 8, 24)])
def test_same_bits_on_every_stream_and_with_a_hierarchy(dims):
    print("case: A12 and diagonal, streams and hierarchy", dims, flush=True)
    P = problem(dims)
    p = torch.from_numpy(M.uniform(4, 4 * int(np.prod(dims)), -1.0, 1.0)).to(DEV)
    ctx = context(P)
    want = {op: call(ctx, op, p) for op in OPS}
    ctx.destroy()
    ctx = context(P)
    S = ViscousSolver(ctx, nlevels=2, smooth_its=2, fp32=True, galerkin_coarse=False, autotune=0)
    r = torch.from_numpy(M.uniform(5, P.nvel, -1.0, 1.0)).to(DEV)
    z = S.vcycle(r).clone()
    for _ in range(2):
        torch.cuda.synchronize()
        for op in OPS:
            assert torch.equal(call(ctx, op, p), want[op])
        for s in (torch.cuda.Stream(device=DEV), torch.cuda.Stream(device=DEV)):
            torch.cuda.synchronize()
            with torch.cuda.stream(s):
                got = {op: call(ctx, op, p) for op in OPS}
            torch.cuda.synchronize()
            for op in OPS:
                assert torch.equal(got[op], want[op])
            del s  # the next user's stream may take its handle
    d = ctx.a11_diag(np.zeros(P.nvel), _lib.MATMULT)  # host vectors, on the stream set last
    assert np.array_equal(d, want["diag"].cpu().numpy())
    torch.cuda.synchronize()
    assert torch.equal(S.vcycle(r), z)
    S.destroy()
    ctx.destroy()


def test_overlapping_streams():
    """Calls with different inputs in flight on the null stream and on two others at once."""
    print("case: A12 and diagonal, overlapping streams", flush=True)
    dims = (24, 20, 28)
    P = problem(dims)
    ps = [torch.from_numpy(M.uniform(20 + i, 4 * int(np.prod(dims)), -1.0, 1.0)).to(DEV) for i in range(3)]
    ctx = context(P)
    want = [call(ctx, "a12", p).clone() for p in ps]
    wd = call(ctx, "diag", ps[0]).clone()
    streams = [torch.cuda.default_stream(DEV), torch.cuda.Stream(device=DEV), torch.cuda.Stream(device=DEV)]
    out = [[torch.empty(P.nvel, dtype=torch.float64, device=DEV) for _ in range(8)] for _ in range(4)]
    torch.cuda.synchronize()
    for k in range(8):
        for i, s in enumerate(streams):
            with torch.cuda.stream(s):
                call(ctx, "a12", ps[i], out[i][k])
                if i == k % 3:
                    call(ctx, "diag", ps[0], out[3][k])
    torch.cuda.synchronize()
    for k in range(8):
        for i in range(3):
            assert torch.equal(out[i][k], want[i])
        assert torch.equal(out[3][k], wd)
    ctx.destroy()


def test_captured_calls_and_eager_ones():
    """A graph captured on one stream, replayed on another while eager calls run on the first: its calls
    share no scratch with them (equal to the oracle), and every replay gives the same bits."""
    print("case: A12 and diagonal under capture", flush=True)
    dims = (20, 16, 12)
    P = problem(dims)
    ref = O.matmult_a12(*dims, P.coords, P.mask, M.uniform(30, 4 * int(np.prod(dims)), -1.0, 1.0))
    p1 = torch.from_numpy(M.uniform(30, 4 * int(np.prod(dims)), -1.0, 1.0)).to(DEV)
    p2 = torch.from_numpy(M.uniform(31, 4 * int(np.prod(dims)), -1.0, 1.0)).to(DEV)
    ctx = context(P)
    cap, other = torch.cuda.Stream(device=DEV), torch.cuda.Stream(device=DEV)
    y = [torch.empty(P.nvel, dtype=torch.float64, device=DEV) for _ in range(2)]
    with torch.cuda.stream(cap):
        want2 = call(ctx, "a12", p2).clone()
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=cap):
            call(ctx, "a12", p1, y[0])
            call(ctx, "diag", p1, y[1])
    torch.cuda.synchronize()
    got = []
    eager = [torch.empty(P.nvel, dtype=torch.float64, device=DEV) for _ in range(12)]
    for _ in range(4):
        torch.cuda.synchronize()
        with torch.cuda.stream(other):
            g.replay()
        with torch.cuda.stream(cap):
            for e in eager:
                call(ctx, "a12", p2, e)
        torch.cuda.synchronize()
        got.append([t.clone() for t in y])
        for e in eager:
            assert torch.equal(e, want2)
    a = got[0][0].cpu().numpy()
    assert np.linalg.norm(a - ref) <= 1e-12 * np.linalg.norm(ref)
    d = O.matgetdiag_a11(*dims, P.coords, P.eta, P.mask)
    assert np.linalg.norm(got[0][1].cpu().numpy() - d) <= 1e-12 * np.linalg.norm(d)
    for g2 in got[1:]:
        assert torch.equal(g2[0], got[0][0]) and torch.equal(g2[1], got[0][1])
    ctx.destroy()
