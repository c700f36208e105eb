"""CPU: rules the library applies on the host, through a small program linked
against it (tests/host/host_check.cpp)."""
import subprocess
from pathlib import Path

import numpy as np
import pytest

ROOT = Path(__file__).resolve().parents[1]


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    from chainamps_amd import build
    from chainamps_amd.capi import library_path
    lib = library_path()
    if not lib.exists():
        pytest.skip("library not built in this checkout (python -m chainamps_amd.build)")
    exe = tmp_path_factory.mktemp("host") / "host_check"
    subprocess.run([build.hipcc(), "-std=c++17", "-O1", "-x", "c++", "-D__HIP_PLATFORM_AMD__", f"-I{build.ROCM}/include",
                    f"-I{ROOT / 'chainamps_amd/csrc'}", str(ROOT / "tests/host/host_check.cpp"), "-o", str(exe),
                    f"-L{lib.parent}", f"-l:{lib.name}", f"-L{build.ROCM}/lib", "-lamdhip64",
                    f"-Wl,-rpath,{lib.parent}", f"-Wl,-rpath,{build.ROCM}/lib"], check=True)

    def ask(*lines):
        r = subprocess.run([str(exe)], input="\n".join(lines) + "\n", capture_output=True, text=True, check=True)
        return r.stdout.splitlines()
    return ask


def test_svd_batches(check):
    """Blocks decomposed together stay within the memory and the grid that a
    call may use, whatever their number; a block that takes more alone."""
    one = [int(check(f"bytes {v} 1024 1024")[0]) for v in (0, 1)]
    # vectors: U and Vh; work: R with its reflectors, X and V at least
    assert one[0] >= 16 * 3 * 1024 ** 2 and one[1] >= one[0] + 16 * 2 * 1024 ** 2
    for limit, items, blocks in [(3 * one[1], 100, [(1024, 1024)] * 10), (one[1] - 1, 100, [(1024, 1024)] * 3),
                                 (1 << 40, 4, [(8, 5)] * 11), (one[1], 100, [(9, 4), (1024, 1024), (4, 9), (70, 70)]),
                                 (1 << 32, 32768, [(2, 2)] * 70000), (1 << 32, 32768, [(1024, 1100)] * 200),
                                 (1 << 32, 32768, [])]:
        text = " ".join(f"{m} {n}" for m, n in blocks)
        ends = [int(x) for x in check(f"batches {limit} {items} 1 {text}")[0].split()]
        size = {s: int(check(f"bytes 1 {s[0]} {s[1]}")[0]) for s in set(blocks)}
        assert (ends[-1] if ends else 0) == len(blocks)
        first = 0
        for e in ends:
            assert 0 < e - first <= items
            assert e - first == 1 or sum(size[s] for s in blocks[first:e]) <= limit
            first = e
    assert check(f"batches {1 << 32} 32768 1 " + "384 384 " * 30) == ["30 "]


def test_bond_inverse(check):
    """Null values of a charge sector have no inverse; the small values of a
    weak sector, negative and not-finite ones do."""
    def inv(*pairs):
        return [float(x) for x in check("inverse " + " ".join(f"{q} {v!r}" for q, v in pairs))[0].split()]
    assert inv((0, 0.5), (0, 0.25)) == [2.0, 4.0]
    assert inv((0, 1.0), (0, 0.0), (0, 1e-40), (0, 2.2e-16), (0, 2.3e-16)) == [1.0, 0.0, 0.0, 0.0, 1 / 2.3e-16]
    assert inv((0, 1.0), (1, 1e-18), (0, 1e-18), (1, 1e-30), (1, 1e-35)) == [1.0, 1 / 1e-18, 0.0, 1 / 1e-30, 0.0]
    assert inv((0, 0.0), (0, 0.0)) == [0.0, 0.0]
    assert inv((0, -0.5), (0, -1e-20)) == [-2.0, 0.0]
    assert inv((0, float("inf")), (1, 2.0)) == [0.0, 0.5]
    x = inv((0, float("nan")), (1, 2.0))
    assert x[0] != x[0] and x[1] == 0.5


def _problem(m, n, ks, batch=1, beta=0):
    return f"{m} {n} {batch} {beta} {len(ks)} " + " ".join(map(str, ks))


def test_plans_cover_their_outputs(check):
    """Whichever kernels a grouped plan goes to, every output is computed
    once, at sizes around the tiles, the row passes and the k shares."""
    seen = set()
    for ps in [[(1, 1, [1])], [(17, 33, [3])], [(65, 63, [33])], [(200, 18, [257])], [(129, 130, [100])],
               [(1025, 13, [29])], [(16, 16, [32, 32, 7])], [(16, 17, [32])], [(40, 5, [8], 37), (40, 5, [8], 37)],
               [(300, 300, [16]), (300, 300, [700])], [(1000, 700, [200])], [(70, 3, [4, 4]), (70, 130, [9])],
               [(33, 17, [1]), (5, 129, [33]), (31, 15, [65]), (16, 16, [129])], [(64, 20, [300], 3, 1)],
               [(2000, 16, [32]), (1000, 700, [200])], [(7, 9, [])], [(512, 512, [10000])]]:
        probs = [_problem(p[0], p[1], p[2], *p[3:]) for p in ps]
        route, lo, hi = check("plan " + " ".join(probs))[0].split()
        assert (lo, hi) == ("1", "1"), (ps, route, lo, hi)
        seen.add(route)
    assert seen == {"direct", "tiles", "rows", "tiles+rows"}


def test_plan_extended_after_its_lists(check):
    """A problem added to a plan whose lists are built is not left out."""
    a, b = _problem(200, 18, [257]), _problem(100, 40, [300])
    assert check("plan " + a)[0] == "direct 1 1"
    assert check(f"plan {a} + {b}")[0].split()[1:] == ["1", "1"]
    assert check(f"plan {_problem(1000, 700, [200])} + {b}")[0].split()[1:] == ["1", "1"]


def test_tridiagonal_lowest(check):
    """Lowest eigenpair of a symmetric tridiagonal matrix against numpy:
    random, decoupled, degenerate and zero matrices, at scales down to and up
    to those whose squares leave the range of a double."""
    rng = np.random.default_rng(4)
    cases = [(rng.standard_normal(k), rng.standard_normal(max(k - 1, 0))) for k in (1, 2, 3, 20, 63)]
    cases += [(np.array([2.0, 1.0, 3.0]), np.zeros(2)), (np.zeros(4), np.zeros(3)), (np.ones(5), np.zeros(4)),
              (np.full(30, -1.0), np.full(29, 1e-9)), (np.arange(40.0), np.full(39, 1e-3))]
    for scale in (1.0, 1e150, 1e-150, 1e250, 1e-250):
        for a, b in cases:
            k = len(a)
            out = check(f"tridiagonal {k} " + " ".join(repr(float(x) * scale) for x in np.concatenate([a, b])))
            got = np.array([float(x) for x in out[0].split()])
            e, v = got[0] / scale, got[1:]
            T = np.diag(a) + np.diag(b, 1) + np.diag(b, -1)
            nrm = max(np.abs(T).sum(1).max(), 1e-300)
            assert abs(np.linalg.norm(v) - 1.0) <= 1e-14
            assert abs(e - np.linalg.eigvalsh(T)[0]) <= 4e-15 * nrm, (scale, k)
            assert np.linalg.norm(T @ v - e * v) <= 1e-14 * nrm, (scale, k)


def test_routes_of_the_contraction_tests(check):
    """The sizes at which the GPU tests of a kernel contract reach that
    kernel."""
    from test_gpu_gemm_edges import TILE_SIZES
    route = lambda m, n, k: check("plan " + _problem(m, n, [k]))[0].split()[0]  # noqa: E731
    assert {route(*s) for s in TILE_SIZES} == {"tiles"}
    assert {route(*s) for s in [(1, 17, 1), (17, 33, 3), (31, 64, 15), (32, 65, 16), (33, 20, 17), (64, 96, 31),
                                (65, 63, 33)]} == {"tiles"}
    assert {route(*s) for s in [(129, 130, 100), (200, 18, 257)]} == {"direct"}
    assert {route(*s) for s in [(1, 1, 1), (15, 16, 4), (16, 15, 5), (17, 1, 3), (63, 2, 31), (65, 16, 32), (1023, 7, 8),
                                (1025, 13, 29)]} == {"rows"}
