"""The point projection where the device has no room for its element sums: the nodes sum the points themselves,
to the same bits."""
import ctypes

import numpy as np
import pytest

import ptq2
from ptq2 import _lib
from ptq2 import mesh as M

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
DEV = torch.device("cuda:0")


def project_within(ctx, limit, wil, xi, eta, rho):
    """ptq2_project_points_q1 with at most `limit` bytes of workspace."""
    f = _lib.lib().ptq2_internal_project_points
    f.restype = ctypes.c_int
    f.argtypes = [ctypes.c_void_p, ctypes.c_int64] + [ctypes.c_void_p] * 6 + [ctypes.c_uint, ctypes.c_size_t]
    ptr = lambda t: None if t is None else t.data_ptr()
    out = [torch.full((27 * ctx.nel,), np.nan, dtype=torch.float64, device=DEV) for _ in range(2 if rho is not None else 1)]
    ctx._stream(eta)
    _lib.check(f(ctx.handle, wil.numel(), ptr(xi), ptr(wil), ptr(eta), ptr(rho), ptr(out[0]),
                 ptr(out[1]) if rho is not None else None, _lib.DEVICE, limit), "project", ctx.handle)
    return out


@pytest.mark.parametrize("dims,ppe,crowd,rho", [((5, 3, 9), 8, 0, True), ((8, 4, 1), 3, 500, False), ((4, 4, 3), 60, 0, True),
                                                ((2, 3, 2), 0, 0, False)])
def test_projection_without_element_sums(dims, ppe, crowd, rho):
    print("case: projection without room", dims, ppe, crowd, flush=True)
    ne = int(np.prod(dims))
    wil = np.concatenate([np.repeat(np.arange(ne), ppe), np.full(crowd, ne // 2)]).astype(np.int32)
    wil = wil[np.argsort(M.uniform(9, wil.size))]
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(DEV)
    pts = (dev(wil), dev(M.uniform(10, 3 * wil.size, -1.0, 1.0)), dev(10.0 ** M.uniform(11, wil.size, -2.0, 3.0)),
           dev(M.uniform(12, wil.size, -1.0, 1.0)) if rho else None)
    ctx = ptq2.Context(0)
    ctx.setup_mesh(*dims, M.q2_uniform(*dims))
    want = project_within(ctx, 2 ** 40, *pts)
    nodes = 8 * M.nnodes(*dims) * (2 if rho else 1) + 256
    for limit in (nodes, 2 ** 40, nodes):
        for a, b in zip(project_within(ctx, limit, *pts), want):
            assert torch.equal(a, b)
    with pytest.raises(_lib.PTQ2Error):
        project_within(ctx, nodes - 1, *pts)
    ctx.destroy()
