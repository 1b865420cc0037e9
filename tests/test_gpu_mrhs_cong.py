"""Multi-RHS products of congruent 60-DoF groups: clusters of 2, 4 and 8
elements (2,048 elements and more form them, in BF16 20,000), columns around the
16 of a wave, elements in any order, offsets past 32 bits.

Bars as for the other multi-RHS products: 2e-6 per column against the rounded
model (K and, for BF16, U as rounded), FP32 accumulation being what differs.
"""
import numpy as np
import pytest

from amat_amd import PREC, SCATTER, Maps, MultiRHS, aMatFree, mesh, problems
from conftest import rel_l2
from test_gpu_mrhs import TOL_MODEL, bf16_round

pytestmark = pytest.mark.gpu


def build(dims, precision, order=None, twice=False):
    p = problems.elasticity_hex20(*dims)
    g = p.gmap if order is None else p.gmap[order]
    if twice:   # every seventh element names DoFs twice, one of them three times
        g = g.copy()
        g[::7, 5] = g[::7, 2]
        g[::7, 40] = g[::7, 41] = g[::7, 17]
    E, N = g.shape[0], p.n_dofs
    maps = Maps(0, 1)
    maps.set_map(E, g.astype(np.uint32), np.full(E, 60, np.uint32), N, np.arange(N, dtype=np.uint64), 0, N - 1, N)
    maps.set_bdr_map(np.zeros(0, np.uint64), np.zeros(0))
    s = mesh.uniform(3, 2, E, 0.5, 2.0)
    op = aMatFree(maps)
    op.set_element_matrices_scaled(p.k_ref, s)
    op.finalize()
    return op, MultiRHS([op], precision), g.astype(np.int64), s, p.k_ref, N


def model(g, s, k_ref, N, U, precision):
    V = np.zeros(U.shape)
    for lo in range(0, len(g), 2048):
        K = (s[lo:lo + 2048, None, None] * k_ref).astype(np.float32)
        if precision == PREC.BF16:
            K = bf16_round(K)
        W = (K.astype(np.float64) @ U[g[lo:lo + 2048]]).reshape(-1, U.shape[1])
        for c in range(U.shape[1]):
            V[:, c] += np.bincount(g[lo:lo + 2048].reshape(-1), weights=W[:, c], minlength=N)
    return V


@pytest.mark.parametrize("dims,shuffled,columns,precision", [
    ((4, 3, 2), True, (2, 50), PREC.FP32), ((13, 13, 13), False, (1, 5, 32), PREC.FP32),
    ((17, 16, 16), True, (3, 16, 17), PREC.FP32), ((20, 20, 21), False, (8, 50), PREC.FP32),
    ((28, 28, 28), False, (1, 16, 18), PREC.BF16), ((30, 29, 23), True, (7, 20), PREC.BF16)])
def test_clusters_and_columns(torch_gpu, dims, shuffled, columns, precision):
    torch = torch_gpu
    E = dims[0] * dims[1] * dims[2]
    op, mr, g, s, k_ref, N = build(dims, precision, np.random.default_rng(1).permutation(E) if shuffled else None)
    for nrhs in columns:
        U = mesh.uniform(7, nrhs, N * nrhs, -1.0, 1.0).astype(np.float32).reshape(N, nrhs)
        dU = torch.from_numpy(U).cuda()
        out = []
        for scatter in (SCATTER.DETERMINISTIC, SCATTER.DETERMINISTIC, SCATTER.ATOMIC):
            mr.set_scatter(scatter)
            dV = torch.full_like(dU, float("nan"))
            mr.apply_dev(nrhs, [dU], [dV], torch.cuda.current_stream())
            out.append(dV.cpu().numpy())
        np.testing.assert_array_equal(out[0], out[1])
        want = model(g, s, k_ref, N, (bf16_round(U) if precision == PREC.BF16 else U).astype(np.float64), precision)
        for V in (out[0], out[2]):
            worst = max(rel_l2(V[:, c].astype(np.float64), want[:, c]) for c in range(nrhs))
            assert worst <= TOL_MODEL, (nrhs, worst)


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("dims,precision", [((13, 13, 13), PREC.FP32), ((28, 28, 28), PREC.BF16)])
def test_many_columns(torch_gpu, dims, precision, wide):
    """A buffer of element rows of more than 2 GiB (the atomic scatter then adds
    into V), and U and V of more than 4 GiB: the columns are those of a product
    of a few columns alone."""
    torch = torch_gpu
    op, mr, g, s, k_ref, N = build(dims, precision)
    nrhs = (2**30 if wide else 2**28) // N + 13
    mr.set_scatter(SCATTER.DETERMINISTIC)
    U = torch.rand(N, nrhs, device="cuda", generator=torch.Generator("cuda").manual_seed(5)) - 0.5
    V = torch.full_like(U, float("nan"))
    pick = torch.tensor([0, 1, 15, 16, nrhs // 2, nrhs - 2, nrhs - 1], device="cuda")
    few = U[:, pick].contiguous()
    want = torch.empty_like(few)
    mr.apply_dev(len(pick), [few], [want], torch.cuda.current_stream())
    mr.apply_dev(nrhs, [U], [V], torch.cuda.current_stream())
    assert torch.equal(V[:, pick], want)
    assert not torch.isnan(V.sum(dim=0)).any()
    mr.set_scatter(SCATTER.ATOMIC)
    V.fill_(float("nan"))
    mr.apply_dev(nrhs, [U], [V], torch.cuda.current_stream())
    assert rel_l2(V[:, pick].cpu().double().numpy(), want.cpu().double().numpy()) <= TOL_MODEL
    assert not torch.isnan(V.sum(dim=0)).any()


def test_atomic_streams_and_capture(torch_gpu):
    """The atomic scatter's row buffer passes between streams; a captured call
    has none."""
    torch = torch_gpu
    op, mr, g, s, k_ref, N = build((13, 13, 13), PREC.FP32)
    mr.set_scatter(SCATTER.ATOMIC)
    nrhs = 100   # 45 MB of rows
    U = [torch.rand(N, nrhs, device="cuda") - 0.5 for _ in range(4)]
    V = [torch.full_like(u, float("nan")) for u in U]
    graph, st = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    W = torch.full_like(U[0], float("nan"))
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=st):   # the first call of all
        mr.apply_dev(nrhs, [U[0]], [W], torch.cuda.current_stream())
    streams = [torch.cuda.Stream() for _ in U]
    for _ in range(3):
        for u, v, q in zip(U, V, streams):
            mr.apply_dev(nrhs, [u], [v], q)
        graph.replay()
    torch.cuda.synchronize()
    mr.set_scatter(SCATTER.DETERMINISTIC)
    for u, v in zip(U, V):
        want = torch.empty_like(u)
        mr.apply_dev(nrhs, [u], [want], torch.cuda.current_stream())
        torch.cuda.synchronize()
        assert torch.equal(v, want)   # the two passes are the deterministic ones
    v0 = V[0].cpu().double().numpy()
    assert rel_l2(W.cpu().double().numpy(), v0) <= TOL_MODEL


def test_dofs_named_twice(torch_gpu):
    torch = torch_gpu
    op, mr, g, s, k_ref, N = build((16, 16, 17), PREC.FP32, twice=True)
    nrhs = 6
    U = mesh.uniform(7, 1, N * nrhs, -1.0, 1.0).astype(np.float32).reshape(N, nrhs)
    want = model(g, s, k_ref, N, U.astype(np.float64), PREC.FP32)
    for scatter in (SCATTER.DETERMINISTIC, SCATTER.ATOMIC):
        mr.set_scatter(scatter)
        dV = torch.full((N, nrhs), float("nan"), device="cuda")
        mr.apply_dev(nrhs, [torch.from_numpy(U).cuda()], [dV], torch.cuda.current_stream())
        V = dV.cpu().numpy().astype(np.float64)
        assert max(rel_l2(V[:, c], want[:, c]) for c in range(nrhs)) <= TOL_MODEL
