"""The tet10 kernel of method 2 at its edges: curved elements, rules of 1 to 64
points, element counts around a wave and a block, both scatters and types.

Bars: FP64 1e-13, as for the other forms of the product; FP32 1e-5 (roundings of
6e-8 of coordinates a few element lengths from the origin).
"""
import dataclasses

import numpy as np
import pytest

import oracle as orc
from amat_amd import BCOP, PREC, SCATTER, Maps, aMatFree, fem, mesh, problems
from conftest import rel_l2
from test_gpu_free import dev, run

pytestmark = pytest.mark.gpu


def curved(n_elem, ngt):
    """The first n_elem elements of a mesh whose nodes all moved a little."""
    p = problems.poisson_tet10(4, with_rhs=False)
    m = p.mesh
    c = m.coords + mesh.uniform(3, 1, m.coords.size, -0.008, 0.008).reshape(m.coords.shape)
    nodes = m.elem_nodes[:n_elem]
    K = fem.ke_tet10_batch(c[nodes], ngt)
    m2 = dataclasses.replace(m, coords=c, elem_nodes=nodes)
    return dataclasses.replace(p, mesh=m2, gmap=p.gmap[:n_elem], K=K, k_ref=None, scale=None, free={**p.free, "ngt": ngt})


@pytest.mark.parametrize("ngt", [1, 2, 3, 4])
@pytest.mark.parametrize("n_elem", [1, 63, 64, 65, 255, 257])
def test_counts_rules_scatters(torch_gpu, n_elem, ngt):
    torch = torch_gpu
    p = curved(n_elem, ngt)
    u = p.random_u()
    want, masked = orc.matvec(p.gmap, p.K, u), orc.matmult_mf(p.gmap, p.K, u, p.constrained)
    op = p.build_free_operator(aMatFree, Maps, bcop=BCOP.IDENTITY)
    at = p.build_free_operator(aMatFree, Maps, bcop=BCOP.IDENTITY, scatter=SCATTER.ATOMIC)
    for o in (op, at):
        assert rel_l2(run(torch, o.matvec_dev, u), want) <= 1e-13
        assert rel_l2(run(torch, o.matmult_dev, u), masked) <= 1e-13
    du = dev(torch, u.astype(np.float32))
    dv = torch.empty_like(du)
    op.matmult_f32_dev(PREC.FP32, dv, du)
    assert rel_l2(dv.cpu().numpy().astype(np.float64), masked) <= 1e-5
