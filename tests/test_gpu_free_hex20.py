"""The hex20 kernel of method 2 at its edges: element counts around the 7 (3 at
ngt = 4) elements of a wave, every rule, both scatters, both compute types.

Bars: FP64 1e-13, as for the other forms of the product; FP32 1e-5, some 20
roundings of 6e-8 on differences of coordinates of up to 8 element lengths.
"""
import numpy as np
import pytest

import oracle as orc
from amat_amd import BCOP, PREC, SCATTER, Maps, aMatFree, problems
from conftest import rel_l2
from test_gpu_free import dev, distorted, run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ngt", [1, 2, 3, 4])
@pytest.mark.parametrize("dims", [(1, 1, 1), (2, 1, 1), (3, 1, 1), (2, 2, 1), (3, 2, 1), (7, 1, 1), (2, 2, 2),
                                  (7, 2, 1), (5, 3, 1)])
def test_counts_rules_scatters(torch_gpu, dims, ngt):
    torch = torch_gpu
    p = distorted(problems.elasticity_hex20(*dims, ngt=ngt), 0.1)
    K, u = p.element_matrices(), p.random_u()
    op = p.build_free_operator(aMatFree, Maps, bcop=BCOP.IDENTITY)
    want, masked = orc.matvec(p.gmap, K, u), orc.matmult_mf(p.gmap, K, u, p.constrained)
    assert rel_l2(run(torch, op.matvec_dev, u), want) <= 1e-13
    assert rel_l2(run(torch, op.matmult_dev, u), masked) <= 1e-13
    at = p.build_free_operator(aMatFree, Maps, bcop=BCOP.IDENTITY, scatter=SCATTER.ATOMIC)
    assert rel_l2(run(torch, at.matvec_dev, u), want) <= 1e-13
    assert rel_l2(run(torch, at.matmult_dev, u), masked) <= 1e-13
    du = dev(torch, u.astype(np.float32))
    dv = torch.empty_like(du)
    op.matmult_f32_dev(PREC.FP32, dv, du)
    assert rel_l2(dv.cpu().numpy().astype(np.float64), masked) <= 1e-5
