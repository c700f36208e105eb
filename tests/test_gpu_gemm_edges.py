"""GPU: the grouped GEMM kernel at the edges of its tiles and K chunks,
against numpy in complex128.

Charge-free tensors have one block per tensor, so a contraction is one
problem of exactly (M, N, K).  A length-K sum of independent entries rounds
to about eps sqrt(K) relative (three-product form: a few times that);
1e-13 in FP64 and 2e-5 in FP32 bound it for K up to a few hundred.
"""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu


def _tensor(ctx, T, inward, numrows):
    from chainamps_amd.capi import IndexDesc
    from chainamps_amd.workloads import tensor_from_dense
    idx = [IndexDesc(i, False, np.zeros((s, 1), int)) for s, i in zip(T.shape, inward)]
    return tensor_from_dense(ctx, [0], idx, numrows, T)


def _dense(T, shape):
    rows, cols, p, i, x = T.to_csc()
    m = np.zeros((cols, rows), complex)
    m[np.repeat(np.arange(cols), np.diff(p)), i] = x
    return m.reshape(shape[::-1]).transpose(range(len(shape))[::-1])


def _rand(rng, *shape):
    return rng.standard_normal(shape) + 1j * rng.standard_normal(shape)


@pytest.mark.parametrize("m,n,k", [(1, 17, 1), (17, 33, 3), (31, 64, 15), (32, 65, 16), (33, 20, 17), (64, 96, 31),
                                   (65, 63, 33), (129, 130, 100), (200, 18, 257)])
@pytest.mark.parametrize("conjA,conjB", [(False, False), (True, False), (False, True)])
def test_contract_edges(ctx, m, n, k, conjA, conjB):
    print(f"case gemm_edges m={m} n={n} k={k} conj={conjA},{conjB}", flush=True)
    import chainamps_amd as cam
    rng = np.random.default_rng(m + 1000 * n + k)
    A, B = _rand(rng, m, k), _rand(rng, k, n)
    ref = (A.conj() if conjA else A) @ (B.conj() if conjB else B)
    ka = not conjA                      # direction of A's contracted index (out), after conjugation
    tA = _tensor(ctx, A, [True, not ka], 1)
    # B with K contiguous ([k, n]) and with N contiguous ([n, k])
    kb = (not conjB)
    tB = _tensor(ctx, B, [kb, False], 1)
    tBt = _tensor(ctx, np.ascontiguousarray(B.T), [False, kb], 1)
    assert rel_err(_dense(cam.contract(tA, conjA, tB, conjB, [(1, 0)]), (m, n)), ref) <= 1e-13
    assert rel_err(_dense(cam.contract(tA, conjA, tBt, conjB, [(1, 1)]), (m, n)), ref) <= 1e-13


def _env(rng, chi, d, w):
    from chainamps_amd.capi import IndexDesc
    q = lambda s: np.zeros((s, 1), int)  # noqa: E731
    L, W, R = _rand(rng, chi, w, chi), _rand(rng, d, w, d, w), _rand(rng, chi, w, chi)

    def up(T, sizes, inward, physical, numrows):
        from chainamps_amd.workloads import tensor_from_dense
        idx = [IndexDesc(i, p, q(s)) for s, i, p in zip(sizes, inward, physical)]
        return lambda ctx: tensor_from_dense(ctx, [0], idx, numrows, T.reshape(sizes))

    f = [False] * 6
    return (L, W, R), (up(L, (1, chi, 1, w, 1, chi), [False, True, True, False, True, False], f, 3),
                       up(W, (d, w, d, w), [True, True, False, False], [True, False, True, False], 2),
                       up(R, (chi, 1, w, 1, chi, 1), [False, True, True, False, True, False], f, 2))


@pytest.mark.parametrize("chi,d,w", [(131, 3, 2), (66, 33, 2), (129, 17, 1)])
def test_heff_every_launch(ctx, chi, d, w):
    """Every tile policy, product form and chunk length on M, N, K just past
    the tile edges (one charge sector)."""
    print(f"case heff_every_launch chi={chi} d={d} w={w}", flush=True)
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
        for algo in (0, 1):
            for mode in (0, 1, 2, 3):
                for kc in (8, 16):
                    H.set_launch(prec, algo=algo, tile_mode=mode, wg_per_cu=2, kchunk=kc)
                    assert rel_err(H.apply(v, prec), out_ref) <= tol, (prec, algo, mode, kc)


# Blocks that go to the tiles (test_host_rules.py holds the rule to that) with
# several K chunks of 8 and a remainder: conjugated operands through the whole
# pipelined loop.  (Of the sizes above the last two are small plans.)
TILE_SIZES = [(700, 650, 100), (1025, 515, 257), (333, 1500, 129), (513, 700, 75), (97, 1025, 49), (1537, 161, 97)]


@pytest.mark.parametrize("m,n,k", TILE_SIZES)
@pytest.mark.parametrize("conjA,conjB", [(False, False), (True, False), (False, True), (True, True)])
def test_contract_tiles(ctx, m, n, k, conjA, conjB):
    test_contract_edges(ctx, m, n, k, conjA, conjB)


def test_heff_routes(ctx):
    """The launches of test_heff_every_launch run the tiles (its narrow W
    stages row passes)."""
    import chainamps_amd as cam
    for chi, d, w in [(131, 3, 2), (66, 33, 2), (129, 17, 1)]:
        H = cam.Heff(*(u(ctx) for u in _env(np.random.default_rng(chi), chi, d, w)[1]))
        for prec in (cam.CAM_FP64, cam.CAM_FP32):
            H.set_launch(prec, algo=0, tile_mode=1, wg_per_cu=2, kchunk=8)
            assert H.get_route(prec) == ([1, 2, 2, 1] if d == 3 else [1, 1, 1, 1])
