"""GPU: row passes of the grouped GEMM (at most 16 columns per problem, at
most 32 k per segment) at the edges of their 4-wide k steps, 16-column tiles,
16-row strips and items, against numpy in complex128.

Tolerances as for the tiles: a length-K sum of independent entries rounds to
about eps sqrt(K) relative; 1e-13 in FP64 and 2e-5 in FP32 bound it for K up
to a few hundred.
"""
import numpy as np
import pytest

from conftest import rel_err
from test_gpu_gemm_edges import _dense, _env, _rand, _tensor

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (15, 16, 4), (16, 15, 5), (17, 1, 3), (63, 2, 31), (65, 16, 32),
                                   (1023, 7, 8), (1025, 13, 29)])
@pytest.mark.parametrize("conjA,conjB", [(False, False), (True, False), (False, True)])
def test_contract(ctx, m, n, k, conjA, conjB):
    print(f"case row_pass contract m={m} n={n} k={k} conj={conjA},{conjB}", flush=True)
    import chainamps_amd as cam
    rng = np.random.default_rng(m + 1000 * n + k)
    A, B = _rand(rng, m, k), _rand(rng, k, n)
    tB = _tensor(ctx, B, [not conjB, False], 1)
    tBt = _tensor(ctx, np.ascontiguousarray(B.T), [False, not conjB], 1)

    def check(A):
        with np.errstate(invalid="ignore"):
            ref = (A.conj() if conjA else A) @ (B.conj() if conjB else B)
        tA = _tensor(ctx, A, [True, conjA], 1)
        return (_dense(cam.contract(tA, conjA, tB, conjB, [(1, 0)]), (m, n)),
                _dense(cam.contract(tA, conjA, tBt, conjB, [(1, 1)]), (m, n)), ref)

    x, y, ref = check(A)
    assert rel_err(x, ref) <= 1e-13 and rel_err(y, ref) <= 1e-13
    # a row with an infinity leaves the others alone
    A2 = A.copy()
    A2[m // 2, k // 2] = np.inf
    x, y, _ = check(A2)
    keep = np.arange(m) != m // 2
    assert rel_err(x[keep], ref[keep]) <= 1e-13 if m > 1 else not np.isfinite(x).all()


# d * w input and output columns per row: one k step, ragged tiles, outputs
# split over several passes, the most inputs a pass takes, one more (tiles)
@pytest.mark.parametrize("chi,d,w", [(3, 1, 1), (7, 2, 5), (21, 5, 6), (12, 3, 30), (9, 16, 5), (5, 16, 12), (5, 16, 13)])
def test_heff(ctx, chi, d, w):
    print(f"case row_pass heff chi={chi} d={d} w={w}", flush=True)
    import chainamps_amd as cam
    rng = np.random.default_rng(chi)
    (L, W, R), ups = _env(rng, chi, d, w)
    H = cam.Heff(*(u(ctx) for u in ups))
    psi = _rand(rng, d, chi, d, chi)                       # [s1, a0, s2, a2]
    t = np.einsum("xba,iajc->xbijc", L, psi, optimize=True)
    t = np.einsum("pbiq,xbijc->xqpjc", W, t, optimize=True)
    t = np.einsum("rqjs,xqpjc->xsprc", W, t, optimize=True)
    ref = np.einsum("xsprc,ysc->pxry", t, R, optimize=True)
    flat = lambda T: T.transpose(3, 2, 1, 0).reshape(-1)   # noqa: E731  first index fastest
    v, out_ref = flat(psi), flat(ref)
    for prec, tol in ((cam.CAM_FP64, 1e-13), (cam.CAM_FP32, 2e-5)):
        assert rel_err(H.apply(v, prec), out_ref) <= tol, prec
    H.set_slices(2, 2)                                     # accumulating passes
    assert rel_err(H.apply(v), out_ref) <= 1e-13


def test_routes(ctx):
    """The W stages of the cases above run as row passes, past the largest
    number of inputs as something else."""
    import chainamps_amd as cam
    for chi, d, w in [(3, 1, 1), (7, 2, 5), (21, 5, 6), (12, 3, 30), (9, 16, 5), (5, 16, 12), (5, 16, 13)]:
        H = cam.Heff(*(u(ctx) for u in _env(np.random.default_rng(chi), chi, d, w)[1]))
        assert all((r == 2) == (d * w <= 192) for r in H.get_route()[1:3]), (chi, d, w)
