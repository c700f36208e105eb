"""GPU: the CSC form of a tensor read back from the device, sorted there above
a size and on the host below it: exact against the dense array."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _tensor(ctx, sizes, charges, inward, numrows, seed, special=False):
    from chainamps_amd.capi import IndexDesc
    from chainamps_amd.workloads import tensor_from_dense
    rng = np.random.default_rng(seed)
    flux = np.zeros((1,) * len(sizes), int)
    q = []
    for k, (s, m, i) in enumerate(zip(sizes, charges, inward)):
        q.append(rng.integers(0, m, s))                    # sectors interleave in position
        flux = flux + (1 if i else -1) * q[-1].reshape([-1 if j == k else 1 for j in range(len(sizes))])
    T = rng.standard_normal(sizes) + 1j * rng.standard_normal(sizes)
    T[rng.random(sizes) < 0.2] = 0.0                       # exact zeros inside blocks
    if special:
        T.real[rng.random(sizes) < 0.01] = np.nan
        T.imag[rng.random(sizes) < 0.01] = np.inf
    T = np.where(flux == 0, T, 0.0)
    idx = [IndexDesc(i, False, x.reshape(-1, 1)) for x, i in zip(q, inward)]
    return T, tensor_from_dense(ctx, [0], idx, numrows, T)


# class rows around one chunk of 256, several chunks, one sector, columns only
# of size 1, all rows (host), and a tensor below the size line (host)
@pytest.mark.parametrize("sizes,charges,numrows", [
    ((255, 257), (1, 1), 1), ((256, 128), (1, 1), 1), ((700, 90), (3, 2), 1), ((12, 40, 30, 9), (2, 3, 3, 2), 2),
    ((12, 40, 30, 9), (2, 3, 3, 2), 1), ((12, 40, 30, 9), (2, 3, 3, 2), 3), ((130, 1, 300), (2, 1, 2), 1),
    ((150, 200), (1, 1), 2), ((30, 40), (2, 2), 1)])
def test_csc(ctx, sizes, charges, numrows):
    print(f"case csc {sizes} {charges} numrows={numrows}", flush=True)
    inward = [k % 2 == 0 for k in range(len(sizes))]
    for special in (False, True):
        T, t = _tensor(ctx, sizes, charges, inward, numrows, 7, special)
        rows, cols, p, i, x = t.to_csc()
        assert rows == np.prod(sizes[:numrows], dtype=int) and cols == np.prod(sizes[numrows:], dtype=int)
        m = T.reshape(-1, order="F").reshape(cols, rows)   # columns outer, first index fastest
        c, r = np.nonzero(m)
        assert np.array_equal(p, np.concatenate([[0], np.cumsum(np.bincount(c, minlength=cols))]))
        assert np.array_equal(i, r)
        assert np.array_equal(x.view(np.float64), m[c, r].view(np.float64), equal_nan=True)


@pytest.mark.parametrize("sizes,charges", [((2300, 2401), (1, 1)), ((3300, 3400), (2, 2))])
def test_csc_chunks(ctx, sizes, charges):
    """More stored entries than are emitted at a time (2^22)."""
    print(f"case csc chunks {sizes} {charges}", flush=True)
    T, t = _tensor(ctx, sizes, charges, [True, False], 1, 3)
    rows, cols, p, i, x = t.to_csc()
    c, r = np.nonzero(T.T)
    assert len(x) > 1 << 22 and len(c) == len(x)
    assert np.array_equal(p, np.concatenate([[0], np.cumsum(np.bincount(c, minlength=cols))]))
    assert np.array_equal(i, r)
    assert np.array_equal(x.view(np.float64), T.T[c, r].view(np.float64))
