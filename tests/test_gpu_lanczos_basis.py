"""GPU: the Krylov eigensolver with basis sizes on both sides of the column
groups of its Gram-Schmidt sweep (8, 16, 24 columns, several groups), against
numpy on the matrix of the library's own matvecs.

Convergence is to machine epsilon in the Ritz residual; sums over a few
thousand entries and the matvec itself round at some 10 eps |H|, so energy and
residual are held to 1e-11 |H|.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("ncv", [9, 17, 26, 63])
def test_basis_sizes(ctx, ncv, mixed):
    print(f"case lanczos_basis ncv={ncv} mixed={mixed}", flush=True)
    import chainamps_amd as cam
    from chainamps_amd import workloads
    H = cam.Heff(*workloads.coupled_chain_heff_inputs(ctx, chi=6, d=8, seed=3, Jperp=0.3, hermitian=True))
    n = H.n
    assert 1000 < n <= 2048                                # above the dense route
    M = np.stack([H.apply(c) for c in np.eye(n, dtype=complex)], axis=1)
    M = 0.5 * (M + M.conj().T)
    w = np.linalg.eigvalsh(M)
    E, v, info = H.lowest(converge=True, ncv=ncv, mixed=mixed)
    scale = np.abs(w).max()
    assert abs(E - w[0]) <= 1e-11 * scale, (E, w[0], info)
    assert np.linalg.norm(M @ v - E * v) <= 1e-11 * scale * np.linalg.norm(v), info
