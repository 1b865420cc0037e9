"""Error of the multi-RHS products of congruent 60-DoF groups against 64 bits: no
larger than that of the same operator with a stored matrix per element.

The stored entries are s_e K_ref rounded to FP32.  On smooth fields, where the
terms of a row nearly cancel, the rounding of the operands is the error.
"""
import dataclasses

import numpy as np
import pytest

from amat_amd import PREC, SCATTER, Maps, MultiRHS, aMatFree, mesh, problems
from conftest import rel_l2

pytestmark = pytest.mark.gpu


def fields(p, kind, columns):
    x = np.repeat(p.mesh.coords, 3, axis=0)
    rng = np.random.default_rng(3)
    if kind == "random":
        return rng.uniform(-1.0, 1.0, (p.n_dofs, columns))
    comp = np.tile(rng.uniform(-1.0, 1.0, (3, columns)), (len(x) // 3, 1))
    if kind == "quadratic":
        a = rng.uniform(-1.0, 1.0, (3, columns))
        return comp * (1.0 + x @ a + (x * x) @ a[::-1])
    return comp * np.sin(2.0 * np.pi * (x @ rng.uniform(0.5, 2.0, (3, columns))))


def exact(p, U):
    V = np.zeros(U.shape)
    g = p.gmap.astype(np.int64)
    for lo in range(0, p.n_elem, 2048):
        W = (p.element_matrices(lo, min(2048, p.n_elem - lo)) @ U[g[lo:lo + 2048]]).reshape(-1, U.shape[1])
        for c in range(U.shape[1]):
            V[:, c] += np.bincount(g[lo:lo + 2048].reshape(-1), weights=W[:, c], minlength=len(V))
    return V


def pair(p, precision):
    """(operators, products): K_ref and factors; a matrix per element."""
    ops = [q.build_operator(aMatFree, Maps)
           for q in (p, dataclasses.replace(p, K=p.element_matrices(), k_ref=None, scale=None))]
    return ops, [MultiRHS([op], precision) for op in ops]


def product(torch, mr, U, scatter=SCATTER.DETERMINISTIC):
    mr.set_scatter(scatter)
    dU = torch.from_numpy(U).cuda()
    dV = torch.full_like(dU, float("nan"))
    mr.apply_dev(U.shape[1], [dU], [dV], torch.cuda.current_stream())
    return dV.cpu().numpy().astype(np.float64)


@pytest.mark.parametrize("kind", ["random", "quadratic", "sine"])
@pytest.mark.parametrize("n", [14, 20])
def test_fp32_error_not_above_stored(torch_gpu, n, kind):
    p = problems.elasticity_hex20(n)
    ops, mrs = pair(p, PREC.FP32)
    U = fields(p, kind, 8).astype(np.float32)
    want = exact(p, U.astype(np.float64))
    cong, stored = (rel_l2(product(torch_gpu, mr, U), want) for mr in mrs)
    print(f"{kind} {n}^3: congruent {cong:.2e}, stored {stored:.2e}")
    assert cong <= stored
