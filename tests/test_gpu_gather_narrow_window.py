"""The gather's 2,048-entry window (lists of at most 6 entries per DoF in the mean):
256 DoFs whose lists leave a few entries of it empty, fill it, and pass it, beside
DoFs that no element names.  Sums keep the element order: bit for bit the oracle's.
"""
import numpy as np
import pytest

import oracle as orc
from amat_amd import BCOP, PREC, SCATTER, Maps, aMatFree, mesh
from conftest import rel_l2

pytestmark = pytest.mark.gpu

N = 1024


@pytest.mark.parametrize("bc", [BCOP.NONE, BCOP.IDENTITY, BCOP.PENALTY_DIAG])
@pytest.mark.parametrize("E", [255, 256, 257, 511, 512, 513, 640])   # 8 E entries in the first 256 DoFs
def test_narrow_window_edges(torch_gpu, E, bc):
    torch = torch_gpu
    rng = np.random.default_rng(E)
    gmap = np.stack([rng.permutation(256)[:8] for _ in range(E)])
    assert 8 * E <= 6 * N
    K = mesh.uniform(2, E, E * 64, -1.0, 1.0).reshape(E, 8, 8)
    cons = np.arange(0, N, 19, dtype=np.uint64)
    maps = Maps(0, 1)
    maps.set_map(E, gmap.astype(np.uint32), np.full(E, 8, np.uint32), N, np.arange(N, dtype=np.uint64), 0, N - 1, N)
    maps.set_bdr_map(cons, np.zeros(len(cons)))
    op = aMatFree(maps)
    op.set_options(PREC.FP64 | PREC.FP32, SCATTER.DETERMINISTIC)
    op.set_element_matrices(0, K)
    op.set_bc_operator(bc)
    op.set_penalty(1e3)
    op.finalize()
    u = mesh.uniform(5, 1, N, -1.0, 1.0)
    du = torch.from_numpy(u).cuda()
    dv = torch.full_like(du, float("nan"))
    op.matmult_dev(dv, du, torch.cuda.current_stream())
    got = dv.cpu().numpy()
    free = np.ones(N, bool)
    if bc == BCOP.IDENTITY:
        want = orc.matmult_mf(gmap, K, u, cons)
    else:
        want = orc.matvec(gmap, K, u)
        if bc == BCOP.PENALTY_DIAG:
            c = cons.astype(np.int64)
            free[c] = False
            d = orc.get_diagonal(gmap, K, None, 0, N)
            want[c] += (1e3 - d[c]) * u[c]
    np.testing.assert_array_equal(got[free], want[free])
    np.testing.assert_allclose(got, want, rtol=1e-12, atol=1e-12)
    fv = torch.full_like(du.float(), float("nan"))
    op.matmult_f32_dev(PREC.FP32, fv, du.float())
    # some 20 roundings of 6e-8 per entry
    assert rel_l2(fv.cpu().double().numpy(), want) <= 2e-6
