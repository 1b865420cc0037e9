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


@pytest.mark.parametrize("n,precision", [(14, PREC.FP32), (28, PREC.BF16)])
@pytest.mark.parametrize("factor", [1e-45, 1e45])
def test_factors_beyond_fp32(torch_gpu, factor, n, precision):
    """K_ref or the factors outside FP32's range, their products inside: powers of
    two (exact) change nothing."""
    p = problems.elasticity_hex20(n)
    f = 2.0 ** round(np.log2(factor))
    q = dataclasses.replace(p, k_ref=p.k_ref * f, scale=p.scale / f)
    U = fields(p, "random", 5).astype(np.float32)
    mr, mq = (MultiRHS([r.build_operator(aMatFree, Maps)], precision) for r in (p, q))
    np.testing.assert_array_equal(product(torch_gpu, mq, U), product(torch_gpu, mr, U))


@pytest.mark.parametrize("which", ["entry", "factor"])
def test_values_too_far_apart_for_parts(torch_gpu, which):
    """A K_ref entry or a factor 2^-110 of the largest: the group takes stored
    matrices (FP32 bar of the other multi-RHS products)."""
    p = problems.elasticity_hex20(14)
    k, s = p.k_ref.copy(), p.scale.copy()
    if which == "entry":
        k[3, 7] = k[7, 3] = 2.0 ** -110 * np.abs(k).max()
    else:
        s[5] = 2.0 ** -110
    p = dataclasses.replace(p, k_ref=k, scale=s)
    U = fields(p, "random", 3).astype(np.float32)
    ops, mrs = pair(p, PREC.FP32)
    cong, stored = (product(torch_gpu, mr, U) for mr in mrs)
    np.testing.assert_array_equal(cong, stored)
    assert rel_l2(cong, exact(p, U.astype(np.float64))) <= 2e-7


def test_infinities_as_stored(torch_gpu):
    p = problems.elasticity_hex20(14)
    ops, mrs = pair(p, PREC.FP32)
    U = fields(p, "random", 6).astype(np.float32)
    d = int(p.gmap[1400, 31])
    U[d, :5] = [np.inf, -np.inf, np.nan, np.inf, 3e38]
    U[int(p.gmap[1400, 2]), 3] = np.inf
    cong, stored = (product(torch_gpu, mr, U) for mr in mrs)
    assert np.isinf(stored).any() and np.isnan(stored).any()
    np.testing.assert_array_equal(np.isnan(cong), np.isnan(stored))
    for sign in (np.isposinf, np.isneginf):
        np.testing.assert_array_equal(sign(cong), sign(stored))


@pytest.mark.parametrize("bits", [0x7FC00000, 0x7FFFFFFF, 0xFFFFFFFF])
def test_bf16_nan_stays_nan(torch_gpu, bits):
    """NaN of any payload in U (BF16 rounding in integers carries the largest into
    a zero) reaches every row of its elements."""
    p = problems.elasticity_hex20(28)
    mr = MultiRHS([p.build_operator(aMatFree, Maps)], PREC.BF16)
    U = fields(p, "random", 3).astype(np.float32)
    d = int(p.gmap[11000, 31])
    U.view(np.uint32)[d, 1] = bits
    V = product(torch_gpu, mr, U)
    rows = np.unique(p.gmap[(p.gmap == d).any(axis=1)])
    assert np.isnan(V[rows.astype(np.int64), 1]).all()
    assert not np.isnan(V[:, [0, 2]]).any()


def test_matrix_bytes(torch_gpu):
    """Around the sizes from which congruent groups read no matrices."""
    ops = {n: problems.elasticity_hex20(*n).build_operator(aMatFree, Maps)
           for n in ((12, 12, 14), (13, 13, 13), (27, 27, 27), (28, 28, 28))}
    for (n, op) in ops.items():
        E = n[0] * n[1] * n[2]
        for prec, size, least in ((PREC.FP32, 4, 2048), (PREC.BF16, 2, 20000)):
            b, = MultiRHS([op], prec).matrix_bytes()
            if E < least:
                assert b == E * 3600 * size
            else:   # a factor in two parts per element, one matrix in two parts
                assert 8 * E < b < 8 * E + 40000


@pytest.mark.parametrize("n,precision,bar", [(14, PREC.FP32, 1e-6), (28, PREC.BF16, 1e-2)])
def test_unsymmetric_reference_matrix(torch_gpu, n, precision, bar):
    """Columns are taken in an order of K_ref's own; the bars of the other multi-RHS
    products against the FP64 operator."""
    p = problems.elasticity_hex20(n)
    p = dataclasses.replace(p, k_ref=np.random.default_rng(9).normal(size=(60, 60)))
    U = fields(p, "random", 4).astype(np.float32)
    mr = MultiRHS([p.build_operator(aMatFree, Maps)], precision)
    for scatter in (SCATTER.DETERMINISTIC, SCATTER.ATOMIC):
        assert rel_l2(product(torch_gpu, mr, U, scatter), exact(p, U.astype(np.float64))) <= bar
