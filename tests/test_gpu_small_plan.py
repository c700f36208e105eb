"""GPU: the one-launch kernel of small plans at the edges of its 16 x 16 tiles
and k shares (one, two, four and eight waves per tile, one step and more than
eight per wave), against numpy in complex128 and against the tile kernels.

Tolerances as for the tiles: a length-K sum of independent entries rounds to
about eps sqrt(K) relative; 1e-13 in FP64 and 2e-5 in FP32 bound it for K up
to a few hundred.
"""
import numpy as np
import pytest

from conftest import rel_err
from test_gpu_gemm_edges import _env, _rand
from test_zz_no_alloc import DevVec, _hip

pytestmark = pytest.mark.gpu


# environments: M = chi, K = chi and w chi; W stages: N = K / w = d
@pytest.mark.parametrize("chi,d,w", [(17, 1, 2), (31, 2, 3), (33, 1, 17), (64, 1, 5), (65, 2, 3), (100, 1, 4),
                                     (9, 17, 2), (2, 40, 3), (1, 65, 2), (200, 1, 2)])
def test_heff(ctx, chi, d, w):
    print(f"case small_plan chi={chi} d={d} w={w}", flush=True)
    import chainamps_amd as cam
    rng = np.random.default_rng(chi)
    (L, W, R), ups = _env(rng, chi, d, w)
    psi = _rand(rng, d, chi, d, chi)                       # [s1, a0, s2, a2]
    t = np.einsum("xba,iajc->xbijc", L, psi, optimize=True)
    t = np.einsum("pbiq,xbijc->xqpjc", W, t, optimize=True)
    t = np.einsum("rqjs,xqpjc->xsprc", W, t, optimize=True)
    ref = np.einsum("xsprc,ysc->pxry", t, R, optimize=True)
    flat = lambda T: T.transpose(3, 2, 1, 0).reshape(-1)   # noqa: E731  first index fastest
    v, out_ref = flat(psi), flat(ref)
    for prec, tol in ((cam.CAM_FP64, 1e-13), (cam.CAM_FP32, 2e-5)):
        H = cam.Heff(*(u(ctx) for u in ups))
        assert rel_err(H.apply(v, prec), out_ref) <= tol, prec
        H.set_launch(prec, algo=0, tile_mode=1, wg_per_cu=4, kchunk=16)
        assert rel_err(H.apply(v, prec), out_ref) <= tol, prec
    H = cam.Heff(*(u(ctx) for u in ups))
    if chi >= 2:
        H.set_slices(2, 2)                                 # accumulates
    assert rel_err(H.apply(v), out_ref) <= 1e-13


@pytest.mark.parametrize("chi", [24, 90, 160])
def test_sectors(ctx, chi):
    """Blocks of many sizes, several segments each: a two-level chain."""
    print(f"case small_plan sectors chi={chi}", flush=True)
    import chainamps_amd as cam
    from chainamps_amd import workloads
    ins = workloads.coupled_chain_heff_inputs(ctx, chi=chi, d=2, seed=chi, Jperp=0.3, hermitian=False)
    H, T = cam.Heff(*ins), cam.Heff(*ins)
    T.set_launch(cam.CAM_FP64, algo=0, tile_mode=1, wg_per_cu=4, kchunk=16)
    rng = np.random.default_rng(chi)
    v = rng.standard_normal(H.n) + 1j * rng.standard_normal(H.n)
    assert rel_err(H.apply(v), T.apply(v)) <= 1e-13


def test_noalloc(ctx):
    """The no-allocation matvec accepts a small plan that has not run yet."""
    print("case small_plan noalloc", flush=True)
    import chainamps_amd as cam
    hip = _hip()
    rng = np.random.default_rng(5)
    _, ups = _env(rng, 100, 1, 4)
    H = cam.Heff(*(u(ctx) for u in ups))
    x, y, z = (DevVec(hip, H.n) for _ in range(3))
    try:
        x.upload(_rand(rng, H.n))
        H.apply_device_noalloc(x.ptr, y.ptr)
        H.apply_device(x.ptr, z.ptr)
        ctx.sync()
        assert np.array_equal(y.download(), z.download())
    finally:
        for b in (x, y, z):
            b.free()


def test_tuned(ctx):
    """A plan of few outputs and a long K is small and yet large enough to be
    tuned (2e10 flops): the one-launch kernel is one of the candidates, and
    both precisions end on a configuration that computes the same."""
    print("case small_plan tuned", flush=True)
    import chainamps_amd as cam
    chi, d, w = 214, 2, 64
    rng = np.random.default_rng(chi)
    (L, W, R), ups = _env(rng, chi, d, w)
    psi = _rand(rng, d, chi, d, chi)                       # [s1, a0, s2, a2]
    t = np.einsum("xba,iajc->xbijc", L, psi, optimize=True)
    t = np.einsum("pbiq,xbijc->xqpjc", W, t, optimize=True)
    t = np.einsum("rqjs,xqpjc->xsprc", W, t, optimize=True)
    ref = np.einsum("xsprc,ysc->pxry", t, R, optimize=True)
    flat = lambda T: T.transpose(3, 2, 1, 0).reshape(-1)   # noqa: E731  first index fastest
    v, out_ref = flat(psi), flat(ref)
    H = cam.Heff(*(u(ctx) for u in ups))
    # K of the last stage is 64 x 214: rounding grows with its square root
    for prec, tol in ((cam.CAM_FP64, 1e-12), (cam.CAM_FP32, 1e-4)):
        assert H.get_route(prec)[3] == 4                   # small until it is tuned
        assert rel_err(H.apply(v, prec), out_ref) <= tol, prec
        print("  launch", H.get_launch(prec), "route", H.get_route(prec), flush=True)
        assert all(r in (1, 2, 3, 4) for r in H.get_route(prec))
        assert rel_err(H.apply(v, prec), out_ref) <= tol, prec
        # the tiles that the tuning left for a plan without the choice
        algo, mode, wg, kc = H.get_launch(prec)[3]
        T = cam.Heff(*(u(ctx) for u in ups))
        T.set_launch(prec, algo, mode, wg, kc)
        assert T.get_route(prec)[3] == 1
        assert rel_err(T.apply(v, prec), out_ref) <= tol, prec
        print("  stage ms tuned", H.profile(prec, 5), "tiles", T.profile(prec, 5), flush=True)


def test_routes(ctx):
    """The cases above run the one-launch kernel before set_launch, and tiles
    or row passes after it."""
    import chainamps_amd as cam
    from chainamps_amd import workloads
    for chi, d, w in [(17, 1, 2), (31, 2, 3), (33, 1, 17), (64, 1, 5), (65, 2, 3), (100, 1, 4), (2, 40, 3), (1, 65, 2),
                      (200, 1, 2)]:
        H = cam.Heff(*(u(ctx) for u in _env(np.random.default_rng(chi), chi, d, w)[1]))
        for prec in (cam.CAM_FP64, cam.CAM_FP32):
            assert 4 in H.get_route(prec), (chi, d, w)
            H.set_launch(prec, algo=0, tile_mode=1, wg_per_cu=4, kchunk=16)
            assert 4 not in H.get_route(prec), (chi, d, w)
    for chi in (90, 160):
        H = cam.Heff(*workloads.coupled_chain_heff_inputs(ctx, chi=chi, d=2, seed=chi, Jperp=0.3, hermitian=False))
        assert 4 in H.get_route(), chi
