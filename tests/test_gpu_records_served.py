"""The record kernels of 60-DoF groups whose elements have matrices of their own
(near-symmetric records in FP64, packed records with exceptions in FP32 / BF16;
groups given as K_ref and factors read neither), single and served, and served
launches of more jobs than one look at the job table takes (64).

Results are the oracle's, those of whole matrices and those of the single solves,
bit for bit.
"""
import dataclasses

import numpy as np
import pytest

import oracle as orc
from amat_amd import BCOP, PREC, SCATTER, Maps, aMatFree, problems
from amat_amd.amat import IR_RELIABLE
from amat_amd.serve import Server, rhs_for
from test_gpu_nsym import check_bitexact, ops_pair, run

pytestmark = pytest.mark.gpu

ALL = PREC.FP64 | PREC.FP32 | PREC.BF16


def own(p):
    """The problem with a matrix per element."""
    return dataclasses.replace(p, K=p.element_matrices(), k_ref=None, scale=None)


def reads(op, p):
    """What an FP64 product reads per element: record, whole matrix or factor."""
    i = op.info()
    b = (i.alg_bytes_fp64 - 16 * p.n_dofs) // p.n_elem - 4 * p.dofs_per_elem
    return "factor" if b == 8 else "record" if i.near_symmetric else "whole"


def test_elasticity_matrices(torch_gpu):
    p = own(problems.elasticity_hex20(5, 4, 3))
    rec, whole = ops_pair(p, precision=ALL)
    assert reads(rec, p) == "record" and reads(whole, p) == "whole"
    assert rec.info().k_bytes_fp64 < 0.62 * whole.info().k_bytes_fp64
    check_bitexact(torch_gpu, p, rec, whole)
    u = p.random_u()
    for prec, kb in ((PREC.FP32, "k_bytes_fp32"), (PREC.BF16, "k_bytes_bf16")):
        assert 0.4 * getattr(whole.info(), kb) < getattr(rec.info(), kb) < 0.56 * getattr(whole.info(), kb)
        a, b = (run(torch_gpu, lambda v, x, s: op.matmult_f32_dev(prec, v, x, s), u, np.float32) for op in (rec, whole))
        np.testing.assert_array_equal(a, b)
    pen, penw = ops_pair(p, bcop=BCOP.PENALTY_DIAG, penalty=1e8)
    np.testing.assert_array_equal(run(torch_gpu, pen.matmult_dev, u), run(torch_gpu, penw.matmult_dev, u))


def test_records_past_4_gib(torch_gpu):
    """64^3 hex20: 4.6 GB of records; the congruent form, which the oracle checks at
    this size, has the same bits."""
    p = problems.elasticity_hex20(64)
    u = p.random_u()
    want = run(torch_gpu, p.build_operator(aMatFree, Maps).matvec_dev, u)
    op = aMatFree(p.build_maps(Maps))
    op.set_matfree_type(3)
    for lo in range(0, p.n_elem, 1 << 14):
        op.set_element_matrices(lo, p.element_matrices(lo, min(1 << 14, p.n_elem - lo)))
    op.set_options(PREC.FP64, SCATTER.DETERMINISTIC)
    op.finalize()
    assert reads(op, p) == "record" and op.info().k_bytes_fp64 > 2 ** 32
    np.testing.assert_array_equal(run(torch_gpu, op.matvec_dev, u), want)


def alone(torch, op, method, b, max_outer, max_it):
    db = torch.from_numpy(b).cuda()
    dx = torch.zeros_like(db)
    if method == PREC.FP64:
        st = op.cg(db, dx, rtol=1e-10, max_it=max_it)
    else:
        st = op.ir_cg(method, db, dx, rtol=1e-10, inner_rtol=1e-2, max_outer=max_outer, max_inner=max_it)
    return dx.cpu().numpy(), st


@pytest.mark.parametrize("bc", [BCOP.IDENTITY, BCOP.PENALTY_DIAG])
@pytest.mark.parametrize("method", [int(PREC.FP64), int(PREC.FP32), int(PREC.FP32) | IR_RELIABLE, int(PREC.BF16)])
def test_records_served(torch_gpu, method, bc):
    """Two record jobs, one of the other BC form and one of a congruent group."""
    other = BCOP.PENALTY_DIAG if bc == BCOP.IDENTITY else BCOP.IDENTITY
    jobs = []
    for p, b in ((own(problems.elasticity_hex20(3, 3, 4)), bc), (own(problems.elasticity_hex20(2, 3, 2)), bc),
                 (own(problems.elasticity_hex20(3)), other), (problems.elasticity_hex20(3, 2, 3), bc)):
        op = p.build_operator(aMatFree, Maps, precision=ALL, bcop=b, penalty=1e8)
        assert reads(op, p) == ("factor" if p.K is None else "record")
        jobs.append((p, op, b, rhs_for(p, 17 + len(jobs))))
    # BF16 refinement under a 1e8 penalty does not converge: three outer steps
    max_outer, max_it = (3, 400) if method == PREC.BF16 else (60, 20000)
    s = Server(max_jobs=8)
    ids = {s.submit(op, method, b, max_it=max_it, max_outer=max_outer): k for k, (p, op, _, b) in enumerate(jobs)}
    while ids:
        s.step(8)
        for jid in s.poll():
            p, op, form, b = jobs[ids.pop(jid)]
            x, st = s.result(jid, p.n_dofs)
            y, sy = alone(torch_gpu, op, method, b, max_outer, max_it)
            np.testing.assert_array_equal(x, y)
            assert st.iterations == sy.iterations and st.converged == sy.converged
            if method != PREC.BF16:
                assert st.converged
                if form == BCOP.IDENTITY:
                    r = b - orc.matmult_mf(p.gmap, p.element_matrices(), x, p.constrained)
                    assert np.linalg.norm(r) <= 1.01e-10 * np.linalg.norm(b)


@pytest.mark.parametrize("copies", [22, 65])
def test_many_jobs(torch_gpu, copies):
    """copies jobs on each of three kinds of element launch (records, packed tiles, a
    congruent group): 66 and 195 jobs in the launches over all, 65 in each of
    the element launches."""
    ops = [own(problems.elasticity_hex20(2, 1, 1)), problems.poisson_tet10(2, with_rhs=False), problems.poisson_hex8(3)]
    ops = [(p, p.build_operator(aMatFree, Maps, bcop=BCOP.IDENTITY)) for p in ops]
    s, want = Server(max_jobs=200), {}
    for k in range(copies):
        for p, op in ops:
            b = rhs_for(p, 1000 + k)
            x, st = alone(torch_gpu, op, PREC.FP64, b, 1, 5000)
            assert st.converged
            want[s.submit(op, PREC.FP64, b, max_it=5000)] = (p, x, st.iterations)
    while want:
        s.step(8)
        for jid in s.poll():
            p, x, iterations = want.pop(jid)
            y, st = s.result(jid, p.n_dofs)
            np.testing.assert_array_equal(y, x)
            assert st.iterations == iterations
