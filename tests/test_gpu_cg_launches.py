"""The launches of a CG iteration: the gather that also forms p . q, and the
launches that sum the block sums of the one before.

On elements that share no DoF the atomic scatter is exact too (one addition
into a zeroed row), and its CG forms p . q in a pass of its own; so the
deterministic CG, whose gather forms it, has to return the same bits: sizes at
the edges of a block's 256 and 1,024 elements, of a group of 32 blocks, of the
size up to which a solve alone has the gather form it (65,536 DoFs), and past
the largest one of served jobs (1,048,576; both CGs then make the separate
pass).
"""
import numpy as np
import pytest

from amat_amd import BCOP, PREC, SCATTER, Maps, aMatFree, mesh
from amat_amd.amat import IR_RELIABLE
from amat_amd.serve import Server

pytestmark = pytest.mark.gpu

NB = 8  # DoFs per element


def build(gmap, N, K, bc, scatter, precision=PREC.FP64):
    E, n = gmap.shape
    maps = Maps(0, 1)
    maps.set_map(E, gmap.astype(np.uint32), np.full(E, n, np.uint32), N, np.arange(N, dtype=np.uint64), 0, N - 1, N)
    cons = np.arange(0, N, 37, dtype=np.uint64)
    maps.set_bdr_map(cons, np.zeros(len(cons)))
    op = aMatFree(maps)
    op.set_element_matrices(0, K)
    op.set_options(precision, scatter)
    op.set_bc_operator(bc)
    op.set_penalty(1e3)
    op.finalize()
    return op


def spd(E, n, seed):
    """A few symmetric positive matrices, taken in turn."""
    rng = np.random.default_rng(seed)
    A = rng.normal(size=(5, n, n))
    return (A @ A.transpose(0, 2, 1) + n * np.eye(n))[np.arange(E) % 5]


def solve(torch, op, b, method=None, max_it=10000):
    db = torch.from_numpy(b).cuda()
    dx = torch.zeros_like(db)
    s = torch.cuda.current_stream()
    st = (op.cg(db, dx, rtol=1e-10, max_it=max_it, stream=s) if method is None else
          op.ir_cg(method, db, dx, rtol=1e-10, inner_rtol=0.1, max_outer=100, stream=s))
    return dx.cpu().numpy(), st


@pytest.mark.parametrize("E", [1, 32, 33, 128, 129, 4096, 4097, 8192, 8193, 131072, 131073])
def test_gather_forms_the_dot_product(torch_gpu, E):
    N = E * NB
    gmap = np.arange(N).reshape(E, NB)
    K = spd(E, NB, E)
    b = mesh.uniform(E, 3, N, -1.0, 1.0)
    for bc in (BCOP.IDENTITY, BCOP.PENALTY_DIAG):
        x, st = solve(torch_gpu, build(gmap, N, K, bc, SCATTER.DETERMINISTIC), b)
        y, sy = solve(torch_gpu, build(gmap, N, K, bc, SCATTER.ATOMIC), b)
        assert st.converged and st.iterations == sy.iterations and st.rel_residual == sy.rel_residual
        np.testing.assert_array_equal(x, y)


@pytest.mark.parametrize("E", [33, 4097, 8193, 131072, 131073])
def test_served_and_mixed_precision(torch_gpu, E):
    """Reliable updates: the recurrence stops on the device in the launch that
    updates the direction; served and single solves agree bit for bit."""
    N = E * NB
    gmap = np.arange(N).reshape(E, NB)
    op = build(gmap, N, spd(E, NB, E), BCOP.IDENTITY, SCATTER.DETERMINISTIC, PREC.FP64 | PREC.FP32)
    server, want = Server(max_jobs=4), {}
    for k, method in enumerate((None, int(PREC.FP32) | IR_RELIABLE)):
        b = mesh.uniform(k, 4, N, -1.0, 1.0)
        x, st = solve(torch_gpu, op, b, method)
        assert st.converged and st.rel_residual <= 1e-10 * 1.0000001
        want[server.submit(op, int(PREC.FP64) if method is None else method, b, rtol=1e-10, inner_rtol=0.1,
                           max_it=10000, max_outer=100)] = (x, st)
    while want:
        server.step(3)
        for jid in server.poll():
            x, st = want.pop(jid)
            y, sy = server.result(jid, N)
            np.testing.assert_array_equal(x, y)
            assert st.iterations == sy.iterations


def test_long_lists_and_uneven_blocks(torch_gpu):
    """A DoF in 5,000 elements (lists longer than a gather window) beside short
    lists: the solution satisfies the oracle's operator."""
    import oracle as orc
    E, n = 5000, 4
    N = 3 * E // 2 + 1
    rng = np.random.default_rng(2)
    gmap = np.empty((E, n), dtype=np.int64)
    gmap[:, 0] = 700
    for e in range(E):
        rest = rng.choice(N - 1, n - 1, replace=False)
        gmap[e, 1:] = np.where(rest >= 700, rest + 1, rest)
    gmap[: N // 3 + 1, 1:] = np.resize(np.delete(np.arange(N), 700), (N // 3 + 1, 3))
    K = spd(E, n, 1)
    op = build(gmap, N, K, BCOP.IDENTITY, SCATTER.DETERMINISTIC)
    b = mesh.uniform(1, 3, N, -1.0, 1.0)
    x, st = solve(torch_gpu, op, b)
    assert st.converged
    cons = np.arange(0, N, 37, dtype=np.uint64)
    r = b - orc.matmult_mf(gmap, K, x, cons)
    assert np.linalg.norm(r) <= 1.01e-10 * np.linalg.norm(b)


def test_breakdown_is_reported(torch_gpu):
    """An indefinite operator stops the recurrence in the launch that forms alpha."""
    from amat_amd import AmatError
    E = 300
    gmap = np.arange(E * NB).reshape(E, NB)
    K = spd(E, NB, 3)
    K[::2] = 10.0 - 9.0 * np.eye(NB)       # positive diagonal, negative on vectors of zero sum
    op = build(gmap, E * NB, K, BCOP.NONE, SCATTER.DETERMINISTIC)
    b = np.tile([1.0, -1.0], E * NB // 2)  # p . A p < 0 in the first iteration
    with pytest.raises(AmatError, match="breakdown"):
        solve(torch_gpu, op, b)
