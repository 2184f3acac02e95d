"""GPU: expm_herm's two routes -- the shifted Taylor exponential up to ||A||_1 = 32, the
Jacobi sweeps beyond it, for diagonal matrices and in a workspace of the sweeps' size --
in the four types, with spectra on one side of zero, of one outlier and degenerate.

Both against numpy's eigh (the oracle). Tolerance: eigh's own normwise error bound
p(n) u ||A||_2 times exp's condition for a Hermitian matrix (1 + ||A||_2), with p(n) = 8 n:
well under the 1e-12 the route is held to elsewhere.
"""
import numpy as np
import pytest
import torch

import calaman_g_amd as cg
import oracle.herm as oh

pytestmark = pytest.mark.gpu


def _spectrum(n, cplx, kind, norm, seed):
    rng = np.random.default_rng(seed)
    g = rng.standard_normal((n, n)) + (1j * rng.standard_normal((n, n)) if cplx else 0)
    if kind == "negative":
        h = -(g @ g.conj().T)
    elif kind == "outlier":
        q, _ = np.linalg.qr(g)
        w = 0.1 * rng.standard_normal(n)
        w[0] = -30.0
        h = (q * w) @ q.conj().T
    else:
        h = g
    h = (h + h.conj().T) / 2
    return h * (norm / np.abs(h).sum(0).max())


def _run(a, uplo, dev, nbytes=None):
    return _call(a, uplo, dev, nbytes)[0]


def _call(a, uplo, dev, nbytes=None, want_info=0):
    n, ld = a.shape[0], a.shape[0] + 1
    buf = np.full((n, ld), np.nan, dtype=a.dtype)
    dt = torch.from_numpy(buf).dtype
    buf[:, :n] = a.T
    other = np.tril(np.ones((n, n), bool), -1) if uplo == "U" else np.triu(np.ones((n, n), bool), 1)
    buf[:, :n].T[other] = np.nan  # never read
    da = torch.from_numpy(buf).to(dev)
    de = torch.full((n, ld), 7.0, dtype=dt, device=dev)
    size = cg.expm_herm_buffer_size(n, dt) if nbytes is None else nbytes
    work = torch.empty(size, dtype=torch.uint8, device=dev)
    info = torch.full((1,), -3, dtype=torch.int32, device=dev)
    assert cg.expm_herm_cm(uplo, n, da, ld, de, ld, work, info) == 0
    assert want_info is None or int(info.item()) == want_info
    out = de.cpu().numpy()
    assert np.all(out[:, n:] == 7.0)
    return out[:, :n].T, int(info.item())


def _jacobi_bytes(n, size):
    """the sweeps' blocks: three of order n rounded up to 64, the rotations and the scalars"""
    up = lambda v: -(-v // 256) * 256
    np_, k = -(-n // 64) * 64, -(-n // 64)
    return 3 * up(np_ * np_ * size) + up(k * 4096 * size) + up(4 * k) + 2 * 256 + up(8 * np_)


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("kind", ["full", "negative", "outlier"])
@pytest.mark.parametrize("n,norm", [(1, 3.0), (2, 31.9), (33, 31.9), (33, 32.1), (130, 8.0),
                                    (130, 60.0)])
def test_routes_agree_with_eigh(dev, cplx, kind, n, norm):
    a = _spectrum(n, cplx, kind, norm, 17 * n + int(norm))
    for uplo, code in (("U", oh.UPPER), ("L", oh.LOWER)):
        ref = oh.expm_herm(a, code)
        err = np.linalg.norm(_run(a, uplo, dev) - ref) / np.linalg.norm(ref)
        assert err <= 8 * n * 1.2e-16 * (1 + np.linalg.norm(a, 2)) + 1e-14


@pytest.mark.parametrize("cplx", [False, True])
def test_a_workspace_of_the_sweeps_size_still_serves(dev, cplx):
    n = 128
    a = _spectrum(n, cplx, "full", 4.0, 5)
    nbytes = _jacobi_bytes(n, 16 if cplx else 8)
    assert nbytes < cg.expm_herm_buffer_size(n, torch.complex128 if cplx else torch.float64)
    ref = oh.expm_herm(a)
    err = np.linalg.norm(_run(a, "U", dev, nbytes) - ref) / np.linalg.norm(ref)
    assert err <= 1e-12


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("n,i,j", [(2, 0, 0), (2, 1, 1), (2, 0, 1), (64, 0, 0), (64, 31, 31),
                                   (64, 5, 40), (512, 0, 0), (512, 255, 255), (512, 511, 511),
                                   (512, 3, 300)])
@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_a_value_that_is_not_finite_goes_to_the_sweeps(dev, cplx, n, i, j, bad):
    """wherever it stands: the same status, info and result as in the sweeps' workspace"""
    a = _spectrum(n, cplx, "full", 4.0, n)
    a[i, j] = a[j, i] = bad
    print(f"expm_herm n={n} cplx={cplx} a[{i},{j}]={bad}", flush=True)
    want, want_info = _call(a, "U", dev, _jacobi_bytes(n, 16 if cplx else 8), None)
    got, info = _call(a, "U", dev, None, None)
    assert info == want_info
    np.testing.assert_array_equal(got, want)  # NaN where it has NaN


def _degenerate(n, cplx, norm):
    """three eigenvalues only: one of multiplicity n - 2"""
    rng = np.random.default_rng(n)
    u = rng.standard_normal((n, 2)) + (1j * rng.standard_normal((n, 2)) if cplx else 0)
    q, _ = np.linalg.qr(u)
    h = 0.5 * np.eye(n) + (q * np.array([2.0, -1.5])) @ q.conj().T
    h = (h + h.conj().T) / 2
    return h * (norm / np.abs(h).sum(0).max())


@pytest.mark.parametrize("dtype", [np.float64, np.complex128, np.float32, np.complex64])
@pytest.mark.parametrize("sweeps", [False, True])
@pytest.mark.parametrize("kind", ["full", "negative", "degenerate"])
@pytest.mark.parametrize("n", [2, 31, 64, 150])
def test_both_routes_on_the_same_matrix(dev, dtype, sweeps, kind, n):
    """the sweeps through their own workspace at norms the Taylor route takes otherwise. The
    single types run in double: one rounding of the result, u |E| entrywise, on top"""
    cplx = np.issubdtype(dtype, np.complexfloating)
    a = _degenerate(n, cplx, 6.0) if kind == "degenerate" else _spectrum(n, cplx, kind, 6.0, n)
    a = a.astype(dtype)
    single = np.finfo(dtype).eps > 1e-10
    wide = a.astype(np.complex128 if cplx else np.float64)
    wide = (wide + wide.conj().T) / 2
    nbytes = _jacobi_bytes(n, 16 if cplx else 8) if sweeps else None
    for uplo, code in (("U", oh.UPPER), ("L", oh.LOWER)):
        ref = oh.expm_herm(wide, code)
        err = np.linalg.norm(_run(a, uplo, dev, nbytes) - ref) / np.linalg.norm(ref)
        bound = 8 * n * 1.2e-16 * (1 + np.linalg.norm(wide, 2)) + 1e-14
        assert err <= bound + (np.finfo(dtype).eps if single else 0)
