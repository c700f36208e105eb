"""GPU: the dense route's matrix and lowest eigenpair (H_eff of at most 1000
entries) over its range of sizes, against numpy on the matrix whose columns
are the library's own matvec of the unit vectors.

Both matrices carry the rounding of sums of products, a few eps |H|; the pair
is accepted by the library at a residual of that size, so the energy and the
residual are held to 1e-12 |H|.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _check(H):
    n = H.n
    assert n <= 1000
    M = np.stack([H.apply(c) for c in np.eye(n, dtype=complex)], axis=1)
    M = 0.5 * (M + M.conj().T)
    w = np.linalg.eigvalsh(M)
    E, v, info = H.lowest()
    scale = max(np.abs(w).max(), 1.0)
    assert abs(E - w[0]) <= 1e-12 * scale, (E, w[0])
    assert np.linalg.norm(M @ v - E * v) <= 1e-12 * scale
    assert abs(np.linalg.norm(v) - 1.0) <= 1e-12
    assert info["matvecs_fp64"] == n


@pytest.mark.parametrize("d,chi", [(2, 1), (2, 3), (3, 4), (2, 15), (8, 5), (2, 22), (44, 1)])
def test_dense_sizes(ctx, d, chi):
    print(f"case dense_sizes d={d} chi={chi}", flush=True)
    import chainamps_amd as cam
    from chainamps_amd import workloads
    H = cam.Heff(*workloads.coupled_chain_heff_inputs(ctx, chi=chi, d=d, seed=chi, Jperp=0.3, hermitian=True))
    _check(H)


@pytest.mark.parametrize("field", [0.0, 1.0])
def test_dense_degenerate(ctx, field):
    """An effective Hamiltonian that is zero, or has a many-fold lowest
    level: any vector of the level will do."""
    print(f"case dense_degenerate field={field}", flush=True)
    import chainamps_amd as cam
    from chainamps_amd.capi import IndexDesc
    from chainamps_amd.workloads import tensor_from_dense
    d, chi = 3, 6
    q = lambda n: np.zeros((n, 1), int)  # noqa: E731
    T = np.zeros((d, 2, d, 2), complex)
    T[:, 0, :, 0] = T[:, 1, :, 1] = np.eye(d)
    T[:, 1, :, 0] = field * np.diag([0.0, 0.0, 1.0])
    E = np.zeros((1, chi, 1, 2, 1, chi), complex)
    E[0, :, 0, 1, 0, :] = np.eye(chi)                    # the starting row of the MPO
    F = np.zeros((chi, 1, 2, 1, chi, 1), complex)
    F[:, 0, 0, 0, :, 0] = np.eye(chi)
    up = lambda X, inw, ph, nr: tensor_from_dense(  # noqa: E731
        ctx, [0], [IndexDesc(i, p, q(s)) for s, i, p in zip(X.shape, inw, ph)], nr, X)
    f = [False] * 6
    H = cam.Heff(up(E, [False, True, True, False, True, False], f, 3),
                 up(T, [True, True, False, False], [True, False, True, False], 2),
                 up(F, [False, True, True, False, True, False], f, 2))
    _check(H)
