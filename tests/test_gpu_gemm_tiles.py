"""GPU: the matrix product at the edges of its workgroup tiles (32, 64 and 128 wide),
of its K slices (16, 32 and 64 deep) and of its 16-byte vectors, for the four element
types: the last tile of a row or column is moved back over its neighbour, so an
accumulating product in place must add every entry exactly once.

Reference: numpy in complex128 / float64. Tolerance per entry, for a k-term sum at unit
roundoff u in any order: 4 (k + 4) u (|alpha| |A||B| + |beta C|), the factor 4 covering
complex arithmetic.
"""
import numpy as np
import pytest
import torch

from calaman_g_amd.expm import Context, gemm_cm

pytestmark = pytest.mark.gpu

SHAPES = [  # small, medium and large tiles; one below, at and above an edge; k down to 1
    (1, 1, 1), (3, 2, 5), (31, 33, 32), (32, 32, 31), (33, 31, 33), (64, 65, 63), (95, 97, 1),
    (257, 33, 130), (33, 511, 70), (999, 1001, 67), (1024, 1000, 64), (1664, 1664, 48),
    (1650, 1687, 37), (1700, 1601, 1), (1921, 1930, 47),
    (2047, 2049, 33), (2048, 2048, 31)]


@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("dtype", [np.float32, np.float64, np.complex64, np.complex128])
@pytest.mark.parametrize("in_place", [False, True])
def test_gemm_tile_edges(dev, m, n, k, dtype, in_place):
    rng = np.random.default_rng(m * 31 + n * 7 + k)
    lda, ldb, ldc = m + 1, k + 2, m + 3

    def mat(rows, cols, ld):
        buf = np.full((cols, ld), np.nan, dtype=dtype)  # padding is never used
        x = rng.standard_normal((cols, rows))
        if np.issubdtype(dtype, np.complexfloating):
            x = x + 1j * rng.standard_normal((cols, rows))
        buf[:, :rows] = x
        return buf

    a, b, c = mat(m, k, lda), mat(k, n, ldb), mat(m, n, ldc)
    alpha, beta = (1.0, 1.0) if in_place else (-0.75, 0.0)
    da, db, dc = (torch.from_numpy(x).to(dev) for x in (a, b, c))
    assert gemm_cm(Context(), m, n, k, alpha, da, lda, db, ldb, beta, dc, ldc) == 0
    got = dc.cpu().numpy()
    wide = np.complex128 if np.issubdtype(dtype, np.complexfloating) else np.float64
    aw, bw, cw = a[:, :m].astype(wide).T, b[:, :k].astype(wide).T, c[:, :m].astype(wide).T
    ref = alpha * (aw @ bw) + beta * cw
    u = np.finfo(dtype).eps / 2
    bound = 4 * (k + 4) * u * (abs(alpha) * (np.abs(aw) @ np.abs(bw)) + beta * np.abs(cw))
    assert np.all(np.abs(got[:, :m].T - ref) <= bound)
    assert np.all(np.isnan(got[:, m:]))
