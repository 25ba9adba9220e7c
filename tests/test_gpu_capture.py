"""Applies captured into a graph: every replay gives what an apply gives at
that time, also after updates of the operator and beside applies on other
streams.

Bars: 1e-13 of the largest result in FP64 and 1e-5 in FP32, the kronmult
parity bars.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

import asgard_amd  # noqa: E402
from asgard_amd import grid  # noqa: E402

TOL = {np.float64: 1e-13, np.float32: 1e-5}


@pytest.fixture(scope="module", autouse=True)
def gpu_present():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


def factors(rng, d, n, level, active):
    size = n << level
    return [rng.uniform(-1, 1, (size, size)) if k in dims else np.eye(size)
            for dims in active for k in range(d)]


def capture(m, x, y, inside=False):
    """A graph of y = A x; the handle is on the null stream again after it.
    `inside`: it moves to the captured stream and back while that is captured."""
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    if not inside:
        m.set_stream(s.cuda_stream)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        m.set_stream(s.cuda_stream)
        m.apply(1.0, x, 0.0, y)
        if inside:
            m.set_stream(0)
    m.set_stream(0)
    return graph


def close(a, b, dtype):
    a, b = (t.double().cpu().numpy() for t in (a, b))
    return np.abs(a - b).max() <= TOL[dtype] * max(np.abs(b).max(), 1e-300)


def check_replays(m, graph, x, y, want, dtype):
    """Eager applies and replays in turn."""
    eager = torch.zeros_like(x)
    for _ in range(3):
        m.apply(1.0, x, 0.0, eager)
        torch.cuda.synchronize()
        assert close(eager, want, dtype)
        y.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert close(y, want, dtype)


# (d, n, level, patterns of non-identity dimensions: the captured one, one it
# covers, and ones it does not)
GRIDS = [
    (4, 2, 5, [[(0,), (1,)], [(0,), ()], [(0,), (1, 2)], [(3,), (0, 1, 2, 3)]]),
    (6, 2, 4, [[(0, 3), (1, 4)], [(0,), (1, 4)], [(0, 3), (2, 4)], [(0, 1, 2), (5,)]]),
]


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("case", GRIDS, ids=lambda c: f"d{c[0]}n{c[1]}L{c[2]}")
def test_sparse_grid_apply_follows_updates(case, dtype):
    d, n, level, patterns = case
    rng = np.random.default_rng(23)
    table, _ = grid.element_table([level] * d)
    T = 2
    ops = factors(rng, d, n, level, patterns[0])
    vA = grid.build_vA(d, n, T, level, ops).astype(dtype)
    m = asgard_amd.KronmultMatrix.sparse_grid(d, n, table, level, T, vA, dtype=dtype)
    x = torch.from_numpy(rng.uniform(-1, 1, m.input_size()).astype(dtype)).cuda()
    y = torch.zeros_like(x)
    graph = capture(m, x, y)  # before any other apply of the handle
    step = 0
    for active in [patterns[0]] + patterns[:3] + [patterns[0], patterns[3]]:
        if step:
            ops = factors(rng, d, n, level, active)
            vA = grid.build_vA(d, n, T, level, ops).astype(dtype)
            if step % 2:
                m.update_stored_coefficients(vA)
            else:
                m.update_operators([torch.from_numpy(np.ascontiguousarray(o.T.astype(dtype))).cuda()
                                    for o in ops])
        step += 1
        ref = asgard_amd.KronmultMatrix.sparse_grid(d, n, table, level, T, vA, dtype=dtype)
        ref.set_tuning(waves_per_row=4)
        want = torch.zeros_like(x)
        ref.apply(1.0, x, 0.0, want)
        check_replays(m, graph, x, y, want, dtype)


def test_replays_beside_applies_on_other_streams():
    """Two graphs and an eager apply of one handle at once."""
    rng = np.random.default_rng(29)
    d, n, level, active = 6, 2, 4, [(0, 3), (1, 4), (2, 5)]
    table, _ = grid.element_table([level] * d)
    vA = grid.build_vA(d, n, 3, level, factors(rng, d, n, level, active))
    m = asgard_amd.KronmultMatrix.sparse_grid(d, n, table, level, 3, vA)
    xs = [torch.from_numpy(rng.uniform(-1, 1, m.input_size())).cuda() for _ in range(3)]
    ys = [torch.zeros_like(x) for x in xs]
    wants = [torch.zeros_like(x) for x in xs]
    m.set_tuning(waves_per_row=4)
    for x, want in zip(xs, wants):
        m.apply(1.0, x, 0.0, want)
    m.set_tuning()
    graphs = [capture(m, x, y, inside) for x, y, inside in zip(xs, ys, (False, True))]
    streams = [torch.cuda.Stream() for _ in graphs]
    own = torch.cuda.Stream()
    m.set_stream(own.cuda_stream)
    torch.cuda.synchronize()
    for _ in range(5):
        for graph, s in zip(graphs, streams):
            with torch.cuda.stream(s):
                graph.replay()
        m.apply(1.0, xs[2], 0.0, ys[2])
    torch.cuda.synchronize()
    assert all(close(y, want, np.float64) for y, want in zip(ys, wants))
    m.set_stream(0)


@pytest.mark.parametrize("inside", [False, True])
@pytest.mark.parametrize("layout", [0, 6, 8])
def test_global_apply_follows_updates(layout, inside):
    rng = np.random.default_rng(31)
    d, n, level, active, T = 3, 2, 5, [(0, 1), (2,)], 2
    table, _ = grid.element_table([level] * d)
    mask = np.array([[int(k in a) for k in range(d)] for a in active], np.int32)

    def make(vA):
        return asgard_amd.KronmultMatrix.global_grid(d, n, table, level, T, vA, active=mask)

    vA = grid.build_vA(d, n, T, level, factors(rng, d, n, level, active))
    m = make(vA)
    m.set_tuning(waves_per_row=layout)
    x = torch.from_numpy(rng.uniform(-1, 1, m.input_size())).cuda()
    y = torch.zeros_like(x)
    graph = capture(m, x, y, inside)
    for step in range(3):
        if step:
            ops = factors(rng, d, n, level, active)
            vA = grid.build_vA(d, n, T, level, ops)
            if step == 1:
                m.update_stored_coefficients(vA)
            else:
                m.update_operators([torch.from_numpy(np.ascontiguousarray(o.T)).cuda()
                                    for o in ops])
        ref = make(vA)
        ref.set_tuning(waves_per_row=1)
        want = torch.zeros_like(x)
        ref.apply(1.0, x, 0.0, want)
        check_replays(m, graph, x, y, want, np.float64)
