"""amx_op_info.flops of method-2 operators counts the arithmetic of their kernels:
below one multiply-add per node, field and direction for hex20 and tet10, and
linear in the points apart from the set-up per element."""
import dataclasses

import pytest

from amat_amd import Maps, aMatFree, problems

pytestmark = pytest.mark.gpu


def flops(p, ngt):
    p = dataclasses.replace(p, free=dict(p.free, ngt=ngt))
    return p.build_free_operator(aMatFree, Maps).info().flops / p.n_elem


def test_flops_of_the_kernels(torch_gpu):
    hex20, tet10, hex8 = problems.elasticity_hex20(2), problems.poisson_tet10(2, with_rhs=False), problems.poisson_hex8(2)
    for ngt in (2, 3, 4):
        nq = ngt ** 3
        by_nodes = 3 * 2 * 20 * 9 * nq                  # sums over 20 nodes: J, H and the output, 9 values each
        assert 161 * nq < flops(hex20, ngt) < by_nodes
        assert 160 * nq < flops(tet10, ngt) < (30 * 10 + 85) * nq
        assert flops(hex8, ngt) == (30 * 8 + 85) * nq
    assert flops(tet10, 3) - flops(tet10, 2) == 160 * (27 - 8)
    assert flops(hex20, 3) == 9 * (2 * (58 + 14 * 3 + 6 * 9 + 2 * 27) + 58 + 19 * 3 + 8 * 9 + 3 * 27) + 120 + 161 * 27
