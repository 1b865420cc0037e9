"""The gather's two windows (2,048 entries; 3,072 above a mean of 6 per DoF): 256
DoFs whose lists fill a window to the last entry, pass it by one element, or
leave most of it empty.  Sums keep the element order: bit for bit the oracle's.
"""
import numpy as np
import pytest

import oracle as orc
from amat_amd import PREC, SCATTER, Maps, aMatFree, mesh
from conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [256, 300])
@pytest.mark.parametrize("E", [3, 192, 193, 255, 256, 257, 383, 384, 385, 768, 769])
def test_window_edges(torch_gpu, E, N):
    torch = torch_gpu
    rng = np.random.default_rng(E)
    gmap = np.stack([rng.permutation(256)[:8] for _ in range(E)]) + (np.arange(E)[:, None] % 2) * (N - 256)
    K = mesh.uniform(2, E, E * 64, -1.0, 1.0).reshape(E, 8, 8)
    maps = Maps(0, 1)
    maps.set_map(E, gmap.astype(np.uint32), np.full(E, 8, np.uint32), N, np.arange(N, dtype=np.uint64), 0, N - 1, N)
    maps.set_bdr_map(np.zeros(0, np.uint64), np.zeros(0))
    op = aMatFree(maps)
    op.set_options(PREC.FP64 | PREC.FP32, SCATTER.DETERMINISTIC)
    op.set_element_matrices(0, K)
    op.finalize()
    u = mesh.uniform(5, 1, N, -1.0, 1.0)
    du = torch.from_numpy(u).cuda()
    dv = torch.full_like(du, float("nan"))
    op.matvec_dev(dv, du, torch.cuda.current_stream())
    want = orc.matvec(gmap, K, u)
    np.testing.assert_array_equal(dv.cpu().numpy(), want)
    fu = du.float()
    fv = torch.full_like(fu, float("nan"))
    op.matmult_f32_dev(PREC.FP32, fv, fu)
    # some 8 x 8 roundings of 6e-8 per entry
    assert rel_l2(fv.cpu().double().numpy(), want) <= 1e-6
