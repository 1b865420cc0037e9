"""GPU parity of the congruent-group kernels (operators given as K_e = s_e K_ref).

They rebuild every stored entry (fl(s_e K_ref[r][c]), rounded to FP32 / BF16
for those storages) and keep the stored layouts' products and summation order,
so their results are the bits of whole stored matrices
(set_symmetric_storage(0)) in every storage, BC form and size; the atomic
scatter, whose order is not fixed, agrees to the bars of the other tests.
"""
import numpy as np
import pytest

from amat_amd import BCOP, PREC, SCATTER, Maps, aMatFree, mesh
from amat_amd.amat import IR_RELIABLE
from amat_amd.serve import Server
from conftest import rel_l2

pytestmark = pytest.mark.gpu

ALL = PREC.FP64 | PREC.FP32 | PREC.BF16


def build(n, E, mode, seed, spd=False, bc=BCOP.NONE, scatter=SCATTER.DETERMINISTIC):
    """E elements of n DoFs on random DoF lists, an unsymmetric K_ref (spd: a
    symmetric positive one), factors of either sign and zero (spd: positive)."""
    rng = np.random.default_rng(seed)
    N = max(n, E * n // 3)
    gmap = np.stack([rng.choice(N, n, replace=False) for _ in range(E)])
    gmap[:, 0] = np.arange(E) % N                   # some elements share no order with their neighbours
    for e in range(E):                              # no DoF twice in an element
        rest = np.setdiff1d(np.arange(N), gmap[e, :1])
        gmap[e, 1:] = rng.choice(rest, n - 1, replace=False)
    used = np.unique(gmap)
    gmap = np.searchsorted(used, gmap)
    N = len(used)
    A = rng.normal(size=(n, n))
    kref = A @ A.T + n * np.eye(n) if spd else A
    scale = rng.uniform(0.5, 2.0, E)
    if not spd:
        scale[::3] *= -1.0
        scale[0] = 0.0
    maps = Maps(0, 1)
    maps.set_map(E, gmap.astype(np.uint32), np.full(E, n, np.uint32), N, np.arange(N, dtype=np.uint64), 0, N - 1, N)
    cons = np.sort(rng.choice(N, max(1, N // 7), replace=False)).astype(np.uint64)
    maps.set_bdr_map(cons, np.zeros(len(cons)))
    op = aMatFree(maps)
    op.set_symmetric_storage(mode)
    op.set_element_matrices_scaled(kref, scale)
    op.set_options(ALL, scatter)
    op.set_bc_operator(bc)
    op.set_penalty(1e4)
    op.finalize()
    return op, N


def products(torch, op, N, seed):
    u = mesh.uniform(seed, 1, N, -1.0, 1.0)
    s = torch.cuda.current_stream()
    du, du32 = torch.from_numpy(u).cuda(), torch.from_numpy(u.astype(np.float32)).cuda()
    dv, dv32 = torch.full_like(du, float("nan")), torch.full_like(du32, float("nan"))
    op.matmult_dev(dv, du, s)
    out = [dv.cpu().numpy()]
    for prec in (PREC.FP32, PREC.BF16):
        op.matmult_f32_dev(prec, dv32, du32, s)
        out.append(dv32.cpu().numpy().copy())
    return out


# element counts around a wave (64) and a block of small elements (256), and
# past the size where one block takes all rows of its elements
@pytest.mark.parametrize("n", [8, 20, 24, 60])
@pytest.mark.parametrize("E", [1, 63, 64, 65, 257])
def test_equals_whole_matrices(torch_gpu, n, E):
    for bc in (BCOP.NONE, BCOP.IDENTITY, BCOP.PENALTY_DIAG):
        a, N = build(n, E, 1, 100 * n + E, bc=bc)
        b, _ = build(n, E, 0, 100 * n + E, bc=bc)
        for x, y in zip(products(torch_gpu, a, N, E), products(torch_gpu, b, N, E)):
            np.testing.assert_array_equal(x, y)
        np.testing.assert_array_equal(a.get_diagonal(), b.get_diagonal())
        c, _ = build(n, E, 1, 100 * n + E, bc=bc, scatter=SCATTER.ATOMIC)
        for x, y, tol in zip(products(torch_gpu, c, N, E), products(torch_gpu, b, N, E), (1e-13, 1e-6, 1e-6)):
            assert rel_l2(x, y) <= tol


@pytest.mark.parametrize("n,E", [(8, 70000), (60, 66000)])
def test_large_groups(torch_gpu, n, E):
    """More element groups than blocks in flight: one block per 64 elements,
    a structured chain of elements (neighbours share half their DoFs)."""
    gmap = (np.arange(E)[:, None] * (n // 2) + np.arange(n)[None, :]).astype(np.uint32)
    N = int(gmap.max()) + 1
    rng = np.random.default_rng(n)
    kref, scale = rng.normal(size=(n, n)), rng.uniform(0.5, 2.0, E)
    outs = []
    for mode in (1, 0):
        maps = Maps(0, 1)
        maps.set_map(E, gmap, np.full(E, n, np.uint32), N, np.arange(N, dtype=np.uint64), 0, N - 1, N)
        op = aMatFree(maps)
        op.set_symmetric_storage(mode)
        op.set_element_matrices_scaled(kref, scale)
        op.set_options(ALL)
        op.set_bc_operator(BCOP.NONE)
        op.finalize()
        outs.append(products(torch_gpu, op, N, 3))
    for x, y in zip(*outs):
        np.testing.assert_array_equal(x, y)


@pytest.mark.parametrize("method", [int(PREC.FP64), int(PREC.FP32) | IR_RELIABLE])
def test_served_mix_equals_single_solves(torch_gpu, method):
    """Congruent groups of every supported n, and one with whole matrices, in
    one server: each result is the single solve's."""
    jobs = [build(n, E, mode, 7 + n + E, spd=True, bc=BCOP.IDENTITY)
            for n, E, mode in ((8, 300, 1), (20, 70, 1), (24, 90, 1), (60, 65, 1), (60, 40, 0), (8, 65, 1))]
    server, ids, want = Server(max_jobs=8), {}, {}
    for k, (op, N) in enumerate(jobs):
        b = mesh.uniform(50 + k, 2, N, -1.0, 1.0)
        ids[server.submit(op, method, b, rtol=1e-10, inner_rtol=0.1 if method & IR_RELIABLE else 1e-2,
                          max_outer=200)] = (k, N)
        db = torch_gpu.from_numpy(b).cuda()
        dx = torch_gpu.zeros_like(db)
        s = torch_gpu.cuda.current_stream()
        st = (op.ir_cg(method, db, dx, rtol=1e-10, inner_rtol=0.1, max_outer=200, stream=s)
              if method & IR_RELIABLE else op.cg(db, dx, rtol=1e-10, stream=s))
        assert st.converged
        want[k] = dx.cpu().numpy()
    done = 0
    while done < len(ids):
        server.step(8)
        for jid in server.poll():
            k, N = ids[jid]
            np.testing.assert_array_equal(server.result(jid, N)[0], want[k])
            done += 1
