"""Sparse-grid operators taken one dimension at a time, against the pair
kernels of the same handle.

A handle whose factors are mostly the identity (or whose grid allows the
split of every product) applies its operator along fibres instead of pair by
pair where that is estimated to be faster.  ``set_tuning`` with a shape selects
the pair kernels, which are the general path here; ``apply_form`` tells which
way an apply goes, and every test looks.  Bars: 1e-13 of the largest result in FP64 and 1e-5 in
FP32, the kronmult parity bars.
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
    """Dense U[-1, 1] factors in each term's listed dimensions, identity in
    the others."""
    size = n << level
    return [rng.uniform(-1, 1, (size, size)) if k in dims else np.eye(size)
            for dims in active for k in range(d)]


def tables(d, level, refine):
    table, _ = grid.element_table([level] * d)
    if refine:
        table = grid.refine(table, 0.3, seed=7)
    return table, int(table[:, :d].max())


def both(m, x, alpha, beta, y0, form=None):
    """The result of the chosen path (`form`, unless None) and of the pair
    kernels."""
    out = []
    for waves in (0, 4):
        m.set_tuning(waves_per_row=waves)
        assert waves == 0 or m.apply_form() == (0, 1)
        assert waves or form is None or m.apply_form() == form
        y = torch.from_numpy(y0.copy()).cuda()
        m.apply(alpha, x, beta, y)
        out.append(y.cpu().numpy().astype(np.float64))
    m.set_tuning()
    return out


def close(a, b, dtype):
    return np.abs(a - b).max() <= TOL[dtype] * max(np.abs(b).max(), 1e-300)


CASES = [
    # (d, n, level, refine, non-identity dimensions per term)
    (1, 2, 7, True, [(0,)] * 24),                   # one table for all terms
    (2, 2, 6, False, [(0,), (1,), (1,)]),           # two terms share a table
    (2, 3, 5, True, [(1,), ()]),                    # an identity term, refined
    (3, 4, 5, False, [(0, 1), (1,)]),               # n = 4, two stages
    (4, 2, 6, False, [(0, 2), (0, 1, 2), ()]),      # three stages
    (4, 3, 5, False, [(0, 1, 2), (1, 2)]),
    (3, 4, 4, True, [(0,), (2,)]),
    (4, 2, 6, True, [(0,), (1,), (2,), (3,)]),
    (4, 3, 4, False, [(3,), (0,)]),                 # 81 lanes: 1024-thread groups
    (4, 4, 3, False, [(1,), (2,), (3,)]),           # 256 lanes
    (5, 3, 3, False, [(0,), (1,), (2,), (3,), (4,)]),  # more dimensions than slots
    (6, 2, 4, False, [(0, 3), (1, 4), (5,)]),
    (6, 3, 2, False, [(0,), (5,)]),                 # 729 lanes: one slot
    (2, 5, 4, False, [(0,), (1,)]),                 # n = 5: a workgroup per cell
    (6, 4, 1, False, [(2,)]),                       # 4096 entries
]


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("case", CASES, ids=str)
def test_matches_pair_kernels(case, dtype):
    d, n, level, refine, active = case
    rng = np.random.default_rng(11)
    table, top = tables(d, level, refine)
    T = len(active)
    vA = grid.build_vA(d, n, T, top, factors(rng, d, n, top, active)).astype(dtype)
    m = asgard_amd.KronmultMatrix.sparse_grid(d, n, table, top, T, vA, dtype=dtype)
    x = torch.from_numpy(rng.uniform(-1, 1, m.input_size()).astype(dtype)).cuda()
    y0 = rng.uniform(-1, 1, m.output_size()).astype(dtype)
    form = (8, max(len(a) for a in active))
    for alpha, beta in ((1.0, 0.0), (-0.7, 0.4), (0.0, 2.0)):
        got, want = both(m, x, alpha, beta, y0, form)
        assert close(got, want, dtype), (alpha, beta)
    if dtype == np.float64:
        out = []
        for waves in (0, 4):
            m.set_tuning(waves_per_row=waves)
            y = torch.from_numpy(y0.copy()).cuda()
            m.apply_euler(0.01, 1.5, x, -0.5, y)
            out.append(y.cpu().numpy())
        assert close(out[0], out[1], dtype)


def test_repeats_bit_for_bit_and_streams():
    rng = np.random.default_rng(3)
    table, top = tables(4, 6, False)
    vA = grid.build_vA(4, 2, 1, top, factors(rng, 4, 2, top, [(0, 1, 2)]))
    m = asgard_amd.KronmultMatrix.sparse_grid(4, 2, table, top, 1, vA)
    assert m.apply_form() == (8, 3)  # its stages share work vectors
    x = torch.from_numpy(rng.uniform(-1, 1, m.input_size())).cuda()
    torch.cuda.synchronize()
    outs = []
    for i in range(6):
        # the handle moves between streams without a wait in between
        s = torch.cuda.Stream()
        m.set_stream(s.cuda_stream)
        y = torch.zeros_like(x)
        torch.cuda.synchronize() if i % 2 else None
        s.wait_stream(torch.cuda.current_stream())
        m.apply(1.0, x, 0.0, y)
        outs.append((s, y))
    torch.cuda.synchronize()
    assert all(torch.equal(y, outs[0][1]) for _, y in outs)
    m.set_stream(0)


@pytest.mark.parametrize("on_device", [False, True])
def test_new_factors_change_the_form(on_device):
    """Updates that keep, add and drop non-identity factors; a form whose
    factors cover the new ones stays (its stages too)."""
    rng = np.random.default_rng(5)
    d, n = 4, 2
    table, top = tables(d, 6, False)
    steps = [([(0,), (1,)], 1), ([(0,), (1, 2)], 2), ([(0,), (1,)], 2), ([(0,), ()], 2),
             ([(3,), (0, 1, 2)], 3), ([(3,), (0, 2)], 3), ([(0, 1, 2), (2,)], 3), ([(), (3,)], 1)]
    ops = factors(rng, d, n, top, steps[0][0])
    m = asgard_amd.KronmultMatrix.sparse_grid(d, n, table, top, 2,
                                              grid.build_vA(d, n, 2, top, ops))
    x = torch.from_numpy(rng.uniform(-1, 1, m.input_size())).cuda()
    y0 = np.zeros(m.output_size())
    for active, stages in steps:
        ops = factors(rng, d, n, top, active)
        vA = grid.build_vA(d, n, 2, top, ops)
        if on_device:
            m.update_operators([torch.from_numpy(np.ascontiguousarray(o.T)).cuda()
                                for o in ops])
        else:
            m.update_stored_coefficients(vA)
        got, want = both(m, x, 1.0, 0.0, y0, (8, stages))
        assert close(got, want, np.float64), active
        fresh = asgard_amd.KronmultMatrix.sparse_grid(d, n, table, top, 2, vA)
        fresh.set_tuning(waves_per_row=4)
        y = torch.zeros_like(x)
        fresh.apply(1.0, x, 0.0, y)
        assert close(got, y.cpu().numpy(), np.float64), active


def test_forms_the_split_does_not_cover():
    """Cells missing from a level, factors that are not finite and repeated
    cells stay with the pair kernels, on a grid whose operators have a form
    otherwise."""
    rng = np.random.default_rng(9)
    d, n = 4, 2
    table, top = tables(d, 6, False)

    def make(cells, vA):
        return asgard_amd.KronmultMatrix.sparse_grid(d, n, cells, top, 2, vA)

    split = grid.build_vA(d, n, 2, top, factors(rng, d, n, top, [(0, 1), (2, 3)]))
    plain = grid.build_vA(d, n, 2, top, factors(rng, d, n, top, [(0,), (2,)]))
    assert make(table, split).apply_form() == (8, 2)
    assert make(table, plain).apply_form() == (8, 1)
    repeated = np.concatenate([table, table[:1]])
    pair = (0, 1)
    for cells, vA, form in ((table[:-1], split, pair), (repeated, split, pair),
                            (table[:-1], plain, (8, 1)), (repeated, plain, pair)):
        m = make(cells, vA)
        x = torch.from_numpy(rng.uniform(-1, 1, m.input_size())).cuda()
        got, want = both(m, x, 1.0, 0.0, np.zeros(m.output_size()), form)
        assert close(got, want, np.float64)
    bad = plain.copy()
    bad[3] = np.inf
    m = make(table, bad)
    x = torch.from_numpy(rng.uniform(-1, 1, m.input_size())).cuda()
    y0 = np.zeros(m.output_size())
    got, want = both(m, x, 1.0, 0.0, y0, pair)
    assert np.array_equal(np.isfinite(got), np.isfinite(want)) and not np.isfinite(got).all()
    m.update_stored_coefficients(plain)
    got, want = both(m, x, 1.0, 0.0, y0, (8, 1))
    assert close(got, want, np.float64)
    m.update_stored_coefficients(bad)
    assert m.apply_form() == pair
    m.update_stored_coefficients(plain)
    got, want = both(m, x, 1.0, 0.0, y0, (8, 1))
    assert close(got, want, np.float64)


def test_autotuned_small_and_large_agree():
    rng = np.random.default_rng(13)
    d, n, level = 6, 2, 5
    table, top = tables(d, level, False)
    active = [(0, 3), (1, 4), (2, 5)]
    vA = grid.build_vA(d, n, 3, top, factors(rng, d, n, top, active))
    m = asgard_amd.KronmultMatrix.sparse_grid(d, n, table, top, 3, vA)
    x = torch.from_numpy(rng.uniform(-1, 1, m.input_size())).cuda()
    assert m.autotune(x, torch.zeros_like(x))[1] == 3
    assert m.apply_form() in ((8, 2), (6, 2))  # whichever was faster
    y = torch.zeros_like(x)
    m.apply(1.0, x, 0.0, y)
    m.set_tuning(waves_per_row=4)
    ref = torch.zeros_like(x)
    m.apply(1.0, x, 0.0, ref)
    assert close(y.cpu().numpy(), ref.cpu().numpy(), np.float64)


def test_batch_mixes_both_ways_of_applying():
    """Systems along fibres (workgroups of 256 and 1024 threads) and pair by
    pair in one batch, across a restart and after new factors."""
    rng = np.random.default_rng(17)
    shapes = [(2, 2, 5, True, [(0,), (1,)]), (4, 3, 3, True, [(0,), (3,)]),
              (5, 3, 2, False, [(4,), (0,)]), (3, 4, 3, False, [(1,)]),
              (3, 2, 4, True, [(0, 2), (1,)]), (2, 3, 4, False, [(0, 1)])]
    mats, problems = [], []
    for d, n, level, refine, active in shapes:
        table, top = tables(d, level, refine)
        ops = [0.05 * o if not np.array_equal(o, np.eye(len(o))) else o
               for o in factors(rng, d, n, top, active)]
        vA = grid.build_vA(d, n, len(active), top, ops)
        mats.append(asgard_amd.KronmultMatrix.sparse_grid(d, n, table, top, len(active), vA))
        problems.append((d, n, table, top, len(active), vA))
    dt = 0.05
    batch = asgard_amd.BatchSolver(mats, [dt] * len(mats), restart=6)
    bs = [torch.from_numpy(rng.uniform(-1, 1, m.output_size())).cuda() for m in mats]
    for step in range(2):
        xs = [torch.zeros_like(b) for b in bs]
        res, its, conv = batch.solve(xs, bs, tol=1e-11)
        assert conv.all() and (res <= 1e-11).all(), res
        for p, x, b in zip(problems, xs, bs):
            m = asgard_amd.KronmultMatrix.sparse_grid(*p)
            m.set_tuning(waves_per_row=4)
            r = b - m.apply_euler(dt, 1.0, x, 0.0, torch.zeros_like(x))
            assert float(torch.linalg.norm(r) / torch.linalg.norm(b)) < 2e-11
        # the first system's second term becomes an identity term and its
        # first a product in both dimensions (pair by pair on these cells)
        d, n, table, top, T, _ = problems[0]
        ops = factors(rng, d, n, top, [(0, 1), ()])
        vA = grid.build_vA(d, n, T, top, [0.1 * o if i < 2 else o for i, o in enumerate(ops)])
        mats[0].update_stored_coefficients(vA)
        problems[0] = (d, n, table, top, T, vA)


def test_tuned_handles_choose_again_with_new_factors():
    """The pair kernels chosen by autotune hold until the form changes; a
    shape asked for holds until it is taken back."""
    rng = np.random.default_rng(19)
    table, top = tables(2, 6, False)
    cells = table[:-1]  # a cell missing: dense factors have no form here
    vA = grid.build_vA(2, 2, 2, top, factors(rng, 2, 2, top, [(0, 1), (1,)]))
    m = asgard_amd.KronmultMatrix.sparse_grid(2, 2, cells, top, 2, vA)
    assert m.apply_form() == (0, 1)
    x = torch.from_numpy(rng.uniform(-1, 1, m.input_size())).cuda()
    m.autotune(x, torch.zeros_like(x))
    assert m.apply_form() == (0, 1)
    m.update_stored_coefficients(
        grid.build_vA(2, 2, 2, top, factors(rng, 2, 2, top, [(0,), (1,)])))
    assert m.apply_form() == (8, 1)
    y0 = np.zeros(m.output_size())
    got, want = both(m, x, 1.0, 0.0, y0)
    assert close(got, want, np.float64)
    m.set_tuning(waves_per_row=2)
    m.update_stored_coefficients(
        grid.build_vA(2, 2, 2, top, factors(rng, 2, 2, top, [(1,), ()])))
    assert m.apply_form() == (0, 1)
    m.set_tuning()
    assert m.apply_form() == (8, 1)


def test_batch_follows_a_request_for_the_pair_kernels():
    rng = np.random.default_rng(37)
    table, top = tables(3, 4, True)
    ops = [0.05 * o if not np.array_equal(o, np.eye(len(o))) else o
           for o in factors(rng, 3, 2, top, [(0,), (2,)])]
    m = asgard_amd.KronmultMatrix.sparse_grid(3, 2, table, top, 2,
                                              grid.build_vA(3, 2, 2, top, ops))
    b = torch.from_numpy(rng.uniform(-1, 1, m.output_size())).cuda()
    batch = asgard_amd.BatchSolver([m], [0.05], restart=20)
    out = []
    for waves in (0, 4, 0):
        m.set_tuning(waves_per_row=waves)
        x = torch.zeros_like(b)
        _, _, conv = batch.solve([x], [b], tol=1e-11)
        assert conv.all()
        out.append(x.cpu().numpy())
    assert np.array_equal(out[0], out[2])  # the walk again
    assert not np.array_equal(out[0], out[1])  # other sums
    assert np.abs(out[0] - out[1]).max() < 1e-9 * np.abs(out[0]).max()


WIDE = [
    # (d, n, level, non-identity dimensions per term)
    (1, 1, 9, [(0,)]),                  # one entry a cell, 512 connections
    (2, 1, 6, [(0,), (0, 1)]),
    (6, 1, 3, [(0, 3), (1, 4), ()]),
    (2, 5, 6, [(0,), (1,)]),            # 25 entries: ten groups, a remainder
    (3, 6, 3, [(0, 1, 2)]),             # 216 entries: one more than half
    (1, 16, 4, [(0,)]),
    (2, 16, 3, [(1,), (0, 1)]),         # 256 entries: the widest single chunk
    (3, 7, 3, [(0,), (2,)]),            # 343: a second, ragged chunk
    (4, 5, 2, [(3,), (0, 2)]),          # 625: three chunks
    (6, 4, 1, [(0, 5)]),                # 4096: sixteen
]


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("case", WIDE, ids=str)
def test_walk_of_single_entries_and_wide_blocks(case, dtype):
    """The fibre walk (a global handle pinned to it) against pair kernels."""
    d, n, level, active = case
    rng = np.random.default_rng(41)
    table, top = tables(d, level, False)
    T = len(active)
    ops = factors(rng, d, n, top, active)
    vA = grid.build_vA(d, n, T, top, ops).astype(dtype)
    pair = asgard_amd.KronmultMatrix.sparse_grid(d, n, table, top, T, vA, dtype=dtype)
    pair.set_tuning(waves_per_row=4)
    walk = asgard_amd.KronmultMatrix.global_grid(d, n, table, top, T, vA, dtype=dtype,
                                                 active=grid.identity_mask(ops, T, d))
    walk.set_tuning(waves_per_row=8)
    assert walk.apply_form() == (8, max(len(a) for a in active))
    x = torch.from_numpy(rng.uniform(-1, 1, pair.input_size()).astype(dtype)).cuda()
    y0 = rng.uniform(-1, 1, pair.output_size()).astype(dtype)
    out = []
    for m in (walk, pair):
        y = torch.from_numpy(y0.copy()).cuda()
        m.apply(-0.7, x, 0.4, y)
        out.append(y.cpu().numpy().astype(np.float64))
    assert close(out[0], out[1], dtype)


@pytest.mark.parametrize("level,active,form", [
    (5, [(0, 3), (1, 4), (2, 5)], (8, 2)),
    (6, [(0, 3), (1, 4), (2, 5)], (6, 2)),          # past 2^23 steps: slabs
    (6, [(0, 3), (1, 4, 2), (5,)], (8, 3)),         # which take no third dimension
    (6, [(k,) for k in range(6)], (8, 1))])
def test_layout_of_untuned_handles(level, active, form):
    """Both sides of the line between the walk and the slabs."""
    rng = np.random.default_rng(43)
    table, top = tables(6, level, False)
    T = len(active)
    vA = grid.build_vA(6, 2, T, top, factors(rng, 6, 2, top, active))
    m = asgard_amd.KronmultMatrix.sparse_grid(6, 2, table, top, T, vA)
    assert m.apply_form() == form
    x = torch.from_numpy(rng.uniform(-1, 1, m.input_size())).cuda()
    got, want = both(m, x, 1.3, -0.4, rng.uniform(-1, 1, m.output_size()))
    assert close(got, want, np.float64)
