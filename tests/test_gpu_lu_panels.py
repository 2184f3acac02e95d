"""GPU: the LU panels at the edges of what a lane holds -- heights around the 512 lanes and
their multiples, panel widths that are no power of two -- with equal, zero and NaN pivots,
and the triangular solves at every order up to their block of 64.

P A = L U is checked by reconstruction: |L U - P A| <= 2 n u |L||U| entrywise (Higham, ASNA
9.3, twice for the two sums), the solves by their residual against n u |T||X| times 4 for
complex arithmetic.
"""
import numpy as np
import pytest
import torch

import calaman_g_amd as cg

pytestmark = pytest.mark.gpu

NP = {torch.float32: np.float32, torch.float64: np.float64, torch.complex64: np.complex64,
      torch.complex128: np.complex128}


def _matrix(n, dt, seed):
    rng = np.random.default_rng(seed)
    a = rng.standard_normal((n, n))
    if dt.is_complex:
        a = a + 1j * rng.standard_normal((n, n))
    return a.astype(NP[dt])


def _getrf(a, dt, dev):
    n = a.shape[0]
    da = torch.from_numpy(np.ascontiguousarray(a.T)).to(dev)
    ipiv = torch.zeros(n, dtype=torch.int32, device=dev)
    info = torch.full((1,), -1, dtype=torch.int32, device=dev)
    assert cg.getrf_cm(n, da, n, ipiv, info) == 0
    return da, ipiv, int(info.item())


@pytest.mark.parametrize("dt", list(NP))
@pytest.mark.parametrize("n", [3, 31, 63, 511, 513, 530, 1025, 1040, 2049])
def test_panels_reconstruct(dev, dt, n):
    a = _matrix(n, dt, n)
    da, ipiv, info = _getrf(a, dt, dev)
    assert info == 0
    wide = np.complex128 if dt.is_complex else np.float64
    lu = da.cpu().numpy().T.astype(wide)
    lo, up = np.tril(lu, -1) + np.eye(n), np.triu(lu)
    pa = a.astype(wide)
    for k, q in enumerate(ipiv.cpu().numpy()):
        pa[[k, q - 1]] = pa[[q - 1, k]]
    u = np.finfo(NP[dt]).eps / 2
    assert np.all(np.abs(lo @ up - pa) <= 2 * (n + 4) * u * (np.abs(lo) @ np.abs(up)))


@pytest.mark.parametrize("dt,n", [(torch.float64, 4096), (torch.float64, 4097), (torch.complex64, 4097),
                                  (torch.complex128, 2048), (torch.complex128, 2050),
                                  (torch.float32, 4097), (torch.float32, 8193)])
def test_tall_panels_reconstruct(dev, dt, n):
    """the tallest panels in registers (4 columns) and the first that run in memory, the same
    bound; the products in 64 bits on the device"""
    print(f"getrf n={n} {dt}", flush=True)
    a = torch.from_numpy(_matrix(n, dt, n)).to(dev)
    lu = a.t().contiguous()
    ipiv = torch.zeros(n, dtype=torch.int32, device=dev)
    info = torch.full((1,), -1, dtype=torch.int32, device=dev)
    assert cg.getrf_cm(n, lu, n, ipiv, info) == 0 and int(info.item()) == 0
    wide = torch.complex128 if dt.is_complex else torch.float64
    lu = lu.t().to(wide)
    perm = np.arange(n)
    for k, q in enumerate(ipiv.cpu().numpy()):
        perm[[k, q - 1]] = perm[[q - 1, k]]
    lo, up = torch.tril(lu, -1) + torch.eye(n, dtype=wide, device=dev), torch.triu(lu)
    err = (lo @ up - a.to(wide)[torch.from_numpy(perm).to(dev)]).abs()
    u = np.finfo(NP[dt]).eps / 2
    assert bool(torch.all(err <= 2 * (n + 4) * u * (lo.abs() @ up.abs())))


@pytest.mark.parametrize("dt", list(NP))
@pytest.mark.parametrize("rows", [(70, 200, 515), (3, 515), (511, 512), (600, 1112), (64, 63)])
def test_equal_pivots_in_several_waves_take_the_first_row(dev, dt, rows):
    """the largest entry of column 0 in several waves, in two rows of one lane (512 apart)
    and on both sides of a wave's edge"""
    n = 1300
    a = _matrix(n, dt, 9)
    a[:, 0] /= 2 * np.abs(a[:, 0]).max()
    a[list(rows), 0] = 3.0
    _, ipiv, info = _getrf(a, dt, dev)
    assert info == 0 and int(ipiv[0]) == min(rows) + 1


def test_equal_pivots_take_the_first_row(dev):
    n = 40
    a = np.ones((n, n))
    a[1:, 1:] += np.eye(n - 1)  # after column 1 every column has a single non-zero: the diagonal
    _, ipiv, info = _getrf(a, torch.float64, dev)
    assert info == 0 and np.array_equal(ipiv.cpu().numpy(), np.arange(1, n + 1))


def test_a_nan_is_no_pivot(dev):
    n = 20
    a = _matrix(n, torch.float64, 2)
    a[7, 0] = np.nan
    _, ipiv, _ = _getrf(a, torch.float64, dev)
    col = np.abs(a[:, 0])
    assert int(ipiv[0]) == int(np.nanargmax(col)) + 1


@pytest.mark.parametrize("dt", list(NP))
@pytest.mark.parametrize("n,nrhs", [(1, 5), (2, 1), (33, 15), (63, 16), (64, 17), (65, 3), (130, 33)])
def test_solves_leave_a_small_residual(dev, dt, n, nrhs):
    a = _matrix(n, dt, 3 * n) + NP[dt](n ** 0.5) * np.eye(n, dtype=NP[dt])
    b = _matrix(max(n, nrhs), dt, 5 * n)[:n, :nrhs]
    da, ipiv, info = _getrf(a, dt, dev)
    db = torch.from_numpy(np.ascontiguousarray(b.T)).to(dev)
    assert info == 0 and cg.getrs_cm(n, nrhs, da, n, ipiv, db, n) == 0
    wide = np.complex128 if dt.is_complex else np.float64
    x, lu = db.cpu().numpy().T.astype(wide), da.cpu().numpy().T.astype(wide)
    lo, up = np.tril(lu, -1) + np.eye(n), np.triu(lu)
    u = np.finfo(NP[dt]).eps / 2
    bound = 3 * 4 * (n + 4) * u * (np.abs(lo) @ np.abs(up) @ np.abs(x))  # ASNA 9.4: 3 gamma_n
    res = np.abs(a.astype(wide) @ x - b)
    pb = np.empty_like(bound)  # the bound's rows are in pivot order
    p = np.arange(n)
    for k, q in enumerate(ipiv.cpu().numpy()):
        p[[k, q - 1]] = p[[q - 1, k]]
    pb[p] = bound
    assert np.all(res <= pb)
