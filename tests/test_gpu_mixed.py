"""GPU tests of the mixed-precision / flexible solver (akm_gmres_euler_mixed):
FP64 iterative refinement around FP32-kronmult GMRES cycles, the right
preconditioner path, the plain-FP64 fallback, and the solution against a
dense LU solve (oracle) with the FP64 residual recomputed on the CPU by the
oracle's kronmult."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

import asgard_amd  # noqa: E402
import oracle  # noqa: E402
from asgard_amd import dg, grid  # noqa: E402


@pytest.fixture(scope="module", autouse=True)
def gpu_present():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def host(t):
    torch.cuda.synchronize()
    return t.cpu().numpy()


def operator_case(d, n, L, kind="advdiff", seed=0):
    table, _ = grid.element_table([L] * d)
    if kind == "advdiff":
        ops = dg.operators_advection_diffusion(d, n, L, n_adv=max(1, d // 2), nu=0.1)
        T = d
    else:
        rng = np.random.default_rng(seed)
        T = 2
        s = n << L
        ops = [np.asfortranarray(rng.uniform(-1, 1, (s, s))) for _ in range(T * d)]
    vA = grid.build_vA(d, n, T, L, ops)
    return table, vA, T


def cpu_residual(d, n, L, T, table, vA, dt, x, b):
    pntr, indx, iA = oracle.sparse_pattern(table, n=n, T=T, max_level=L)
    y = np.zeros_like(x)
    oracle.kronmult_sparse(d, n, pntr, indx, T, iA, vA, 1.0, np.ascontiguousarray(x), 0.0, y)
    return np.linalg.norm(b - (x - dt * y)) / np.linalg.norm(b)


def dense_solution(d, n, L, T, table, vA, dt, b):
    pntr, indx, iA = oracle.sparse_pattern(table, n=n, T=T, max_level=L)
    size = b.size
    A = np.zeros((size, size))
    e = np.zeros(size)
    col = np.zeros(size)
    for j in range(size):
        e[:] = 0
        e[j] = 1
        oracle.kronmult_sparse(d, n, pntr, indx, T, iA, vA, 1.0, e, 0.0, col)
        A[:, j] = col
    return oracle.dense_solve(np.eye(size) - dt * A, b)


@pytest.mark.parametrize("d,n,L,dt", [(2, 2, 5, 0.01), (3, 2, 4, 0.005), (2, 3, 4, 0.01)])
def test_fp32_refinement_reaches_fp64_accuracy(d, n, L, dt):
    table, vA, T = operator_case(d, n, L)
    m64 = asgard_amd.KronmultMatrix.sparse_grid(d, n, table, L, T, vA)
    m32 = asgard_amd.KronmultMatrix.sparse_grid(d, n, table, L, T, vA.astype(np.float32),
                                                dtype=np.float32)
    size = m64.output_size()
    rng = np.random.default_rng(1)
    u0 = rng.uniform(-1, 1, size)
    b = host(m64.apply_euler(dt, 1.0, dev(u0), 0.0, dev(np.zeros(size))))
    x = dev(b.copy())
    st = asgard_amd.gmres_euler_mixed(dt, m64, x, dev(b), mat32=m32, restart=30, tol=1e-10)
    assert st.converged == 1 and st.fallback == 0
    assert st.rel_residual <= 1e-10
    # the first cycle's residual uses the FP32 operator, every later one FP64
    # one speculative (discarded) step per cycle when the operator is cheap
    assert st.iterations + 1 <= st.applies_f32 <= st.iterations + 1 + st.cycles
    assert st.iterations > 0
    assert st.applies_f64 == st.cycles
    xs = host(x)
    # the FP64 residual recomputed independently on the CPU
    assert cpu_residual(d, n, L, T, table, vA, dt, xs, b) <= 1.5e-10
    gold = dense_solution(d, n, L, T, table, vA, dt, b)
    assert np.abs(xs - gold).max() < 1e-8 * max(1.0, np.abs(gold).max())
    assert np.abs(xs - u0).max() < 1e-8


def test_fp64_flexible_cycles_match_plain_gmres():
    d, n, L, dt = 3, 2, 4, 0.01
    table, vA, T = operator_case(d, n, L, kind="random", seed=4)
    m64 = asgard_amd.KronmultMatrix.sparse_grid(d, n, table, L, T, vA)
    size = m64.output_size()
    b = np.random.default_rng(5).uniform(-1, 1, size)
    x = dev(np.zeros(size))
    st = asgard_amd.gmres_euler_mixed(dt, m64, x, dev(b), restart=40, tol=1e-11)
    assert st.converged == 1 and st.applies_f32 == 0
    xp = dev(np.zeros(size))
    info = asgard_amd.simple_gmres_euler(dt, m64, xp, dev(b), 40, 100, 1e-11 * np.linalg.norm(b))
    # same Krylov space: same number of Krylov steps up to one
    assert abs(st.iterations - (info.iterations - st.cycles)) <= 1
    assert np.abs(host(x) - host(xp)).max() < 1e-9


def test_fallback_when_a_cycle_does_not_reduce_the_residual():
    # an inner operator a thousand times too large makes the FP32 cycle's
    # correction negligible, so the FP64 residual does not halve; the solver
    # must undo the cycle and finish with plain FP64 GMRES
    d, n, L, dt = 2, 2, 4, 0.01
    table, vA, T = operator_case(d, n, L, kind="random", seed=6)
    m64 = asgard_amd.KronmultMatrix.sparse_grid(d, n, table, L, T, vA)
    wrong = asgard_amd.KronmultMatrix.sparse_grid(d, n, table, L, T,
                                                  (1000.0 * vA).astype(np.float32),
                                                  dtype=np.float32)
    size = m64.output_size()
    b = np.random.default_rng(7).uniform(-1, 1, size)
    x = dev(np.zeros(size))
    st = asgard_amd.gmres_euler_mixed(dt, m64, x, dev(b), mat32=wrong, restart=30, tol=1e-10,
                                      inner_tol=1e-8)
    assert st.fallback == 1 and st.converged == 1
    assert st.fallback_iterations > 0
    assert cpu_residual(d, n, L, T, table, vA, dt, host(x), b) <= 1.5e-10


def test_zero_rhs_and_invalid_arguments():
    d, n, L = 2, 2, 3
    table, vA, T = operator_case(d, n, L, kind="random")
    m64 = asgard_amd.KronmultMatrix.sparse_grid(d, n, table, L, T, vA)
    size = m64.output_size()
    x = dev(np.ones(size))
    st = asgard_amd.gmres_euler_mixed(0.1, m64, x, dev(np.zeros(size)))
    assert st.converged == 1 and not host(x).any()
    small, vs, Ts = operator_case(d, n, L - 1, kind="random")
    m32 = asgard_amd.KronmultMatrix.sparse_grid(d, n, small, L - 1, Ts, vs.astype(np.float32),
                                                dtype=np.float32)
    with pytest.raises(ValueError):
        asgard_amd.gmres_euler_mixed(0.1, m64, x, dev(np.ones(size)), mat32=m32)
    pre = asgard_amd.MlpPreconditioner(d, n, small, L - 1, hidden=16)
    with pytest.raises(ValueError):
        asgard_amd.gmres_euler_mixed(0.1, m64, x, dev(np.ones(size)), precond=pre)
    with pytest.raises(ValueError):
        asgard_amd.gmres_euler_mixed(0.1, m32, x, dev(np.ones(size)))


def test_identity_preconditioner_changes_nothing():
    # the untrained network is the identity: flexible GMRES with it takes the
    # same steps as without it
    d, n, L, dt = 2, 2, 5, 0.01
    table, vA, T = operator_case(d, n, L)
    m64 = asgard_amd.KronmultMatrix.sparse_grid(d, n, table, L, T, vA)
    size = m64.output_size()
    b = np.random.default_rng(8).uniform(-1, 1, size)
    pre = asgard_amd.MlpPreconditioner(d, n, table, L, hidden=32)
    x1, x2 = dev(np.zeros(size)), dev(np.zeros(size))
    s1 = asgard_amd.gmres_euler_mixed(dt, m64, x1, dev(b), restart=30, tol=1e-10)
    s2 = asgard_amd.gmres_euler_mixed(dt, m64, x2, dev(b), precond=pre, restart=30, tol=1e-10)
    assert s1.iterations == s2.iterations and s2.precond_applies == s2.iterations
    assert np.abs(host(x1) - host(x2)).max() < 1e-12


def test_learned_preconditioner_gain():
    """Trains the network on solver pairs of an advection-diffusion step and
    reports the Krylov iterations with and without it (FP64 operator)."""
    from asgard_amd import learned

    d, n, L, dt = 3, 2, 5, 4e-3
    table, vA, T = operator_case(d, n, L)
    m64 = asgard_amd.KronmultMatrix.sparse_grid(d, n, table, L, T, vA)
    size = m64.output_size()
    pre, info = learned.train_preconditioner(m64, table, L, dt, samples=60000, epochs=8,
                                             batch=512, lr=1e-3, hidden=128, seed=11)
    rng = np.random.default_rng(12)
    u0 = rng.uniform(-1, 1, size)
    b = host(m64.apply_euler(dt, 1.0, dev(u0), 0.0, dev(np.zeros(size))))
    x1, x2 = dev(np.zeros(size)), dev(np.zeros(size))
    s1 = asgard_amd.gmres_euler_mixed(dt, m64, x1, dev(b), restart=50, tol=1e-10)
    s2 = asgard_amd.gmres_euler_mixed(dt, m64, x2, dev(b), precond=pre, restart=50, tol=1e-10)
    print(f"\nlearned preconditioner: loss {info['loss_before']:.4f} -> {info['loss_after']:.4f}; "
          f"iterations {s1.iterations} without, {s2.iterations} with")
    assert s1.converged == 1 and s2.converged == 1
    assert np.abs(host(x2) - u0).max() < 1e-7
    assert info["loss_after"] < info["loss_before"]
    assert s2.iterations <= s1.iterations


@pytest.mark.parametrize("guess", [0.0, 1.0])
@pytest.mark.parametrize("layout", [None, "pair"])
@pytest.mark.parametrize("scale", [1e-100, 1e-30, 1e-14, 1e14, 1e60])
def test_fp32_cycles_do_not_depend_on_the_scale(scale, layout, guess):
    """The cycles of a scaled right-hand side are those of the unscaled one:
    as many steps, no fallback, the scaled solution (both residuals are at
    most 1e-10, the operator's condition here is below 10)."""
    d, n, L, dt = 3, 2, 5, 1e-3
    table, vA, T = operator_case(d, n, L)
    m64 = asgard_amd.KronmultMatrix.sparse_grid(d, n, table, L, T, vA)
    m32 = asgard_amd.KronmultMatrix.sparse_grid(d, n, table, L, T, vA.astype(np.float32),
                                                dtype=np.float32)
    if layout == "pair":
        m32.set_tuning(waves_per_row=4)
    b = dev(np.random.default_rng(8).uniform(-1, 1, m64.output_size()))
    out = []
    for f in (1.0, scale):
        x = guess * f * b
        st = asgard_amd.gmres_euler_mixed(dt, m64, x, f * b, mat32=m32, restart=40, tol=1e-10)
        assert st.converged == 1 and st.fallback == 0, (f, st.as_dict())
        out.append((st.iterations, st.cycles, x / f))
    assert out[0][:2] == out[1][:2]
    assert float(torch.linalg.norm(out[1][2] - out[0][2]) / torch.linalg.norm(out[0][2])) < 2e-9
