"""The row buffer of the multi-RHS products between streams, graphs and calls
with more columns: every product equals the one formed alone, bit for bit (the
two passes sum in a fixed order)."""
import threading

import numpy as np
import pytest

from amat_amd import PREC, SCATTER, Maps, MultiRHS, aMatFree, problems

pytestmark = pytest.mark.gpu


def make(n, scatter):
    p = problems.elasticity_hex20(n)
    mr = MultiRHS([p.build_operator(aMatFree, Maps)], PREC.FP32)
    mr.set_scatter(scatter)
    return p, mr


def rhs(torch, p, nrhs, seed):
    return torch.rand(p.n_dofs, nrhs, device="cuda", generator=torch.Generator("cuda").manual_seed(seed)) - 0.5


def alone(torch, n, U):
    """The deterministic product by a handle of its own."""
    p, mr = make(n, SCATTER.DETERMINISTIC)
    V = torch.full_like(U, float("nan"))
    mr.apply_dev(U.shape[1], [U], [V], torch.cuda.current_stream())
    torch.cuda.synchronize()
    return V


@pytest.mark.parametrize("n", [6, 13])  # stored matrices, clusters
@pytest.mark.parametrize("scatter", [SCATTER.DETERMINISTIC, SCATTER.ATOMIC])
def test_graph_keeps_its_rows(torch_gpu, n, scatter):
    """The handle's graph, replayed after applications with more columns (clusters:
    the atomic scatter's two passes, as in the calls that are not captured)."""
    torch = torch_gpu
    p, mr = make(n, scatter)
    U, st = rhs(torch, p, 5, 1), torch.cuda.Stream()
    V = torch.full_like(U, float("nan"))
    want = alone(torch, n, U)
    torch.cuda.synchronize()
    mr.graph_capture(5, [U], [V], st)
    for nrhs in (64, 200):
        wide = rhs(torch, p, nrhs, 2)
        out = torch.empty_like(wide)
        mr.apply_dev(nrhs, [wide], [out], torch.cuda.current_stream())
        fill = [torch.full((1 << 18,), float("nan"), device="cuda") for _ in range(16)]  # where freed rows would lie
        V.fill_(float("nan"))
        torch.cuda.synchronize()
        mr.graph_launch(st)
        torch.cuda.synchronize()
        if scatter == SCATTER.DETERMINISTIC or n == 13:
            assert torch.equal(V, want)
        else:  # few rows: FP32 atomics, the bar of the other multi-RHS products
            assert float(torch.linalg.norm(V - want) / torch.linalg.norm(want)) <= 2e-6
        assert all(torch.isnan(f).all() for f in fill)


@pytest.mark.parametrize("n", [6, 13])
def test_callers_graph_keeps_its_rows(torch_gpu, n):
    torch = torch_gpu
    p, mr = make(n, SCATTER.DETERMINISTIC)
    U = rhs(torch, p, 5, 1)
    V = torch.full_like(U, float("nan"))
    want = alone(torch, n, U)
    mr.apply_dev(5, [U], [V], torch.cuda.current_stream())  # makes the buffer
    torch.cuda.synchronize()
    graph, st = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    with torch.cuda.graph(graph, stream=st):
        mr.apply_dev(5, [U], [V], torch.cuda.current_stream())
    for nrhs in (64, 200):
        wide = rhs(torch, p, nrhs, 2)
        out = torch.empty_like(wide)
        mr.apply_dev(nrhs, [wide], [out], torch.cuda.current_stream())
        V.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(V, want)


@pytest.mark.parametrize("n", [6, 13])
def test_deterministic_on_several_streams(torch_gpu, n):
    torch = torch_gpu
    p, mr = make(n, SCATTER.DETERMINISTIC)
    U = [rhs(torch, p, 100, k) for k in range(4)]
    V = [torch.full_like(u, float("nan")) for u in U]
    want = [alone(torch, n, u) for u in U]
    streams = [torch.cuda.Stream() for _ in U]
    torch.cuda.synchronize()
    for _ in range(5):
        for u, v, s in zip(U, V, streams):
            mr.apply_dev(100, [u], [v], s)
    torch.cuda.synchronize()
    for v, w in zip(V, want):
        assert torch.equal(v, w)


@pytest.mark.parametrize("scatter", [SCATTER.DETERMINISTIC, SCATTER.ATOMIC])
def test_first_application_beside_a_capture(torch_gpu, scatter):
    """The buffer is allocated while another thread captures (global mode): the
    product is the two-pass one and the capture stays valid."""
    torch = torch_gpu
    p, mr = make(13, scatter)
    U = rhs(torch, p, 32, 1)
    V = torch.full_like(U, float("nan"))
    want = alone(torch, 13, U)
    x = torch.zeros(1000, device="cuda")
    graph, st, other = torch.cuda.CUDAGraph(), torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    errors = []

    def work():
        try:
            mr.apply_dev(32, [U], [V], other)
        except Exception as e:
            errors.append(e)
    with torch.cuda.graph(graph, stream=st):
        x.add_(1.0)
        t = threading.Thread(target=work)
        t.start()
        t.join()
        x.add_(1.0)
    assert not errors
    torch.cuda.synchronize()
    assert torch.equal(V, want)
    for k in range(3):
        graph.replay()
        torch.cuda.synchronize()
        np.testing.assert_array_equal(x.cpu().numpy(), np.full(1000, 2.0 * (k + 1), np.float32))


def test_autotune_of_clusters_times_once(torch_gpu):
    torch = torch_gpu
    p, mr = make(13, SCATTER.DETERMINISTIC)
    U = rhs(torch, p, 40, 1)
    V = torch.empty_like(U)
    res = mr.autotune(40, [U], [V], reps=3)
    assert len(res) == 12 and len(set(res.values())) == 1   # 32 and 64 columns a wave
    assert mr.tiles() == (32, 1, 0)


@pytest.mark.parametrize("scatter", [SCATTER.DETERMINISTIC, SCATTER.ATOMIC])
def test_more_streams_than_buffers(torch_gpu, scatter):
    """Six streams, four with a buffer of their own, one for the others and for the
    products above 128 MiB of rows; sizes in turn on every stream."""
    torch = torch_gpu
    p, mr = make(13, scatter)
    cols = (5, 320, 17)
    want = [alone(torch, 13, rhs(torch, p, c, c)) for c in cols]
    U = [rhs(torch, p, c, c) for c in cols]
    streams = [torch.cuda.Stream() for _ in range(6)]
    V = [[torch.full_like(u, float("nan")) for u in U] for _ in streams]
    torch.cuda.synchronize()
    for k in range(9):
        for i, st in enumerate(streams):
            j = (i + k) % 3
            mr.apply_dev(cols[j], [U[j]], [V[i][j]], st)
    torch.cuda.synchronize()
    for i in range(6):
        for j in range(3):
            assert torch.equal(V[i][j], want[j])


@pytest.mark.parametrize("scatter", [SCATTER.DETERMINISTIC, SCATTER.ATOMIC])
def test_second_stream_beside_a_capture(torch_gpu, scatter):
    """Products above 128 MiB of rows share one buffer: another stream uses it next,
    while another thread's capture runs."""
    torch = torch_gpu
    p, mr = make(13, scatter)
    U = rhs(torch, p, 320, 1)
    want = alone(torch, 13, U)
    V = [torch.full_like(U, float("nan")) for _ in range(2)]
    x = torch.zeros(1000, device="cuda")
    graph, streams = torch.cuda.CUDAGraph(), [torch.cuda.Stream() for _ in range(3)]
    torch.cuda.synchronize()
    mr.apply_dev(320, [U], [V[0]], streams[0])
    errors = []

    def work():
        try:
            for _ in range(3):
                mr.apply_dev(320, [U], [V[1]], streams[1])
                mr.apply_dev(320, [U], [V[0]], streams[0])
        except Exception as e:
            errors.append(e)
    with torch.cuda.graph(graph, stream=streams[2]):
        x.add_(1.0)
        t = threading.Thread(target=work)
        t.start()
        t.join()
        x.add_(1.0)
    assert not errors
    torch.cuda.synchronize()
    assert torch.equal(V[0], want) and torch.equal(V[1], want)
    graph.replay()
    torch.cuda.synchronize()
    np.testing.assert_array_equal(x.cpu().numpy(), np.full(1000, 2.0, np.float32))


@pytest.mark.parametrize("dims", [(6, 7), (13, 14)])   # stored matrices, clusters (and more than 32 MiB of rows)
def test_atomic_operators_add_up_in_a_shared_output(torch_gpu, dims):
    torch = torch_gpu
    ops = [problems.elasticity_hex20(n).build_operator(aMatFree, Maps) for n in dims]
    N = [problems.elasticity_hex20(n).n_dofs for n in dims]
    mr, nrhs = MultiRHS(ops, PREC.FP32), 100
    gen = torch.Generator("cuda").manual_seed(4)
    U = [torch.rand(n, nrhs, device="cuda", generator=gen) - 0.5 for n in N]
    V = [torch.empty_like(u) for u in U]
    mr.set_scatter(SCATTER.DETERMINISTIC)
    mr.apply_dev(nrhs, U, V, torch.cuda.current_stream())
    want = V[1].clone()
    want[:N[0]] += V[0]
    mr.set_scatter(SCATTER.ATOMIC)
    out = torch.full_like(U[1], float("nan"))
    for graph in (False, True):
        out.fill_(float("nan"))
        if graph:
            st = torch.cuda.Stream()
            torch.cuda.synchronize()
            mr.graph_capture(nrhs, U, [out, out], st)
            mr.graph_launch(st)
        else:
            mr.apply_dev(nrhs, U, [out, out], torch.cuda.current_stream())
        torch.cuda.synchronize()
        assert float(torch.linalg.norm(out - want) / torch.linalg.norm(want)) <= 2e-6


@pytest.mark.parametrize("cols", [(5, 64, 200), (320, 400)])   # a stream's buffer, the shared one
@pytest.mark.parametrize("scatter", [SCATTER.DETERMINISTIC, SCATTER.ATOMIC])
def test_buffers_grow_beside_a_capture(torch_gpu, scatter, cols):
    torch = torch_gpu
    p, mr = make(13, scatter)
    U = [rhs(torch, p, c, c) for c in cols]
    want = [alone(torch, 13, u) for u in U]
    V = [torch.full_like(u, float("nan")) for u in U]
    x = torch.zeros(1000, device="cuda")
    graph, st, other = torch.cuda.CUDAGraph(), torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    mr.apply_dev(cols[0], [U[0]], [V[0]], other)
    errors = []

    def work():
        try:
            for c, u, v in list(zip(cols, U, V))[1:]:
                mr.apply_dev(c, [u], [v], other)
        except Exception as e:
            errors.append(e)
    with torch.cuda.graph(graph, stream=st):
        x.add_(1.0)
        t = threading.Thread(target=work)
        t.start()
        t.join()
        x.add_(1.0)
    assert not errors
    torch.cuda.synchronize()
    for v, w in zip(V, want):
        assert torch.equal(v, w)
    graph.replay()
    torch.cuda.synchronize()
    np.testing.assert_array_equal(x.cpu().numpy(), np.full(1000, 2.0, np.float32))
