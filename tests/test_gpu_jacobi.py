"""GPU: the Jacobi decompositions behind the blockwise SVD, at the sizes where
they change form (one workgroup in LDS up to 69 square, block Jacobi beyond,
column blocks of 16 with padding, row chunks of 64), against numpy.

A backward-stable SVD of an m x n matrix is off by a small multiple of
eps sqrt(max(m, n)) |A|; with sizes up to 260 that stays below 1e-13 |A| for
the values and the reconstruction, and 1e-12 for the vectors' orthonormality.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _svd(ctx, A):
    import chainamps_amd as cam
    from chainamps_amd.capi import IndexDesc
    from chainamps_amd.workloads import tensor_from_dense
    idx = [IndexDesc(True, False, np.zeros((A.shape[0], 1), int)),
           IndexDesc(False, False, np.zeros((A.shape[1], 1), int))]
    U, s, Vd, disc = cam.svd_truncate(tensor_from_dense(ctx, [0], idx, 1, A), 0, 0.0)

    def dense(T):
        rows, cols, p, i, x = T.to_csc()
        m = np.zeros((rows, cols), complex)
        m[i, np.repeat(np.arange(cols), np.diff(p))] = x
        return m
    return dense(U), s, dense(Vd)


def _check(ctx, A):
    U, s, Vd = _svd(ctx, A)
    ref = np.linalg.svd(A, compute_uv=False)
    nrm = np.linalg.norm(A, 2)
    k = len(ref)
    assert len(s) == k
    assert np.all(np.diff(s) <= 0)
    assert np.abs(s - ref).max() <= 1e-13 * nrm
    assert np.linalg.norm((U * s) @ Vd - A, 2) <= 1e-13 * nrm
    assert np.abs(U.conj().T @ U - np.eye(k)).max() <= 1e-12
    assert np.abs(Vd @ Vd.conj().T - np.eye(k)).max() <= 1e-12


def _rand(rng, *shape):
    return rng.standard_normal(shape) + 1j * rng.standard_normal(shape)


@pytest.mark.parametrize("m,n", [(1, 1), (1, 7), (9, 1), (2, 2), (5, 3), (16, 17), (33, 40), (69, 69), (70, 70), (30, 200),
                                 (200, 30), (64, 65), (129, 96), (97, 130), (80, 300), (192, 192), (260, 257)])
@pytest.mark.parametrize("graded", [False, True])
def test_jacobi_sizes(ctx, m, n, graded):
    print(f"case jacobi m={m} n={n} graded={graded}", flush=True)
    rng = np.random.default_rng(1000 * m + n)
    A = _rand(rng, m, n)
    if graded:      # a decaying spectrum on both sides, as a bond's wavefunction has
        A = (A * np.exp(-rng.permutation(n) * 12.0 / n)) * np.exp(-rng.permutation(m) * 9.0 / m)[:, None]
    _check(ctx, A)


@pytest.mark.parametrize("n", [24, 69, 100])
@pytest.mark.parametrize("rank", [1, 5])
def test_jacobi_rank_deficient(ctx, n, rank):
    """Null directions come back orthonormal too (the first sites of a
    product state)."""
    print(f"case jacobi_rank_deficient n={n} rank={rank}", flush=True)
    rng = np.random.default_rng(n + rank)
    _check(ctx, _rand(rng, n, rank) @ _rand(rng, rank, n))
    # exactly dependent columns: exact zeros appear during the rotations
    _check(ctx, np.tile(_rand(rng, n, 1), (1, n)) * np.where(np.arange(n) % 2, -1.0, 1.0))


# On both sides of the switch from 16 to 8 columns per QR panel (more than 600
# rows of the taller side), trailing columns that start off a multiple of 16,
# and the largest columns and rows the kernels take.  The rounding grows like
# the square root of the longer side: sqrt(1200 / 260) = 2.15 times the bounds
# above, in the Frobenius norm.
def _check_large(ctx, A, monkeypatch, capfd):
    monkeypatch.setenv("CAM_SVD_TRACE", "1")
    capfd.readouterr()
    U, s, Vd = _svd(ctx, A)
    assert "1 of 1 blocks by Jacobi" in capfd.readouterr().err
    ref = np.linalg.svd(A, compute_uv=False)
    k = len(ref)
    assert len(s) == k
    assert np.all(np.diff(s) <= 0)
    assert np.abs(s - ref).max() <= 2.2e-13 * ref[0]
    assert np.linalg.norm((U * s) @ Vd - A) <= 2.2e-13 * np.linalg.norm(A)
    assert np.abs(U.conj().T @ U - np.eye(k)).max() <= 2.2e-12
    assert np.abs(Vd @ Vd.conj().T - np.eye(k)).max() <= 2.2e-12


@pytest.mark.parametrize("m,n", [(600, 70), (601, 70), (70, 601), (1200, 64), (90, 1200), (1200, 9), (640, 600),
                                 (700, 650), (1000, 1024), (1024, 1024)])
def test_jacobi_large(ctx, m, n, monkeypatch, capfd):
    print(f"case jacobi_large m={m} n={n}", flush=True)
    rng = np.random.default_rng(1000 * m + n)
    _check_large(ctx, _rand(rng, m, n), monkeypatch, capfd)


@pytest.mark.parametrize("m,n", [(640, 600), (70, 601), (1024, 1000)])
def test_jacobi_large_rank_deficient(ctx, m, n, monkeypatch, capfd):
    print(f"case jacobi_large_rank_deficient m={m} n={n}", flush=True)
    rng = np.random.default_rng(m + n)
    _check_large(ctx, _rand(rng, m, 7) @ _rand(rng, 7, n), monkeypatch, capfd)
    _check_large(ctx, np.tile(_rand(rng, m, 1), (1, n)) * np.where(np.arange(n) % 2, -1.0, 1.0), monkeypatch, capfd)


@pytest.mark.parametrize("m,n,different", [(100, 96, 48), (96, 130, 24), (130, 300, 70), (768, 768, 384),
                                           (1024, 700, 630), (640, 1024, 160), (512, 512, 40)])
def test_jacobi_repeated_columns(ctx, m, n, different, monkeypatch, capfd):
    """Columns of the shorter side that repeat others once or more: the
    rotations get on with such a block only after a second QR."""
    print(f"case jacobi_repeated_columns m={m} n={n} different={different}", flush=True)
    rng = np.random.default_rng(m + n)
    c = min(m, n)
    A = _rand(rng, max(m, n), different)[:, np.arange(c) % different]
    A = A * np.where(np.arange(c) // different % 2, -1.0, 1.0)
    _check_large(ctx, A if m >= n else A.T, monkeypatch, capfd)


def test_many_blocks(ctx):
    """90000 blocks of one element: three batches."""
    print("case jacobi many_blocks", flush=True)
    import chainamps_amd as cam
    from chainamps_amd.capi import IndexDesc
    n = 300
    q = np.stack(np.meshgrid(np.arange(n), np.arange(n), indexing="ij"), -1).reshape(-1, 2) - 150
    x = np.random.default_rng(9).uniform(0.5, 1.0, n * n) * np.exp(1j * np.arange(n * n))
    t = cam.Tensor.from_csc(ctx, [0, 0], [IndexDesc(True, False, q), IndexDesc(False, False, q)], 1, n * n, n * n,
                            np.arange(n * n + 1), np.arange(n * n), x)
    U, s, Vd, disc = cam.svd_truncate(t, 0, 0.0)
    order = np.argsort(-np.abs(x), kind="stable")
    assert np.abs(s - np.abs(x)[order]).max() <= 1e-15
    rows, cols, p, i, u = U.to_csc()
    assert np.array_equal(i, order) and np.abs(np.abs(u) - 1.0).max() <= 1e-14
    rows, cols, p, i, v = Vd.to_csc()
    k = np.argsort(order)
    assert np.array_equal(i, k) and np.abs(u[k] * s[k] * v - x).max() <= 1e-14


def test_large_blocks_together(ctx):
    """Eighteen blocks of 990 x 1000 (285 MB): each in a buffer of its own."""
    print("case jacobi large_blocks_together", flush=True)
    import chainamps_amd as cam
    from chainamps_amd.capi import IndexDesc
    m, n, k = 990, 1000, 18
    A = _rand(np.random.default_rng(21), m, n)
    scale = np.linspace(1.0, 2.0, k)
    x = (scale[:, None, None] * A.T).reshape(-1)
    rows = (np.arange(k)[:, None, None] * m + np.zeros((n, 1), int) + np.arange(m)).reshape(-1)
    q = lambda s: np.repeat(np.arange(k), s).reshape(-1, 1)  # noqa: E731
    t = cam.Tensor.from_csc(ctx, [0], [IndexDesc(True, False, q(m)), IndexDesc(False, False, q(n))], 1, m * k, n * k,
                            np.arange(n * k + 1) * m, rows, x)
    s = cam.svd_truncate(t, 0, 0.0)[1]
    ref = np.linalg.svd(A, compute_uv=False)
    ref = np.sort(np.outer(scale, ref).reshape(-1))[::-1]
    assert len(s) == m * k and np.abs(s - ref).max() <= 2.2e-13 * ref[0]
