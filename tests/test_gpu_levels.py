"""Fields stored side by side per cell (x[n, k], field stride 1): the kernel for
that layout against scipy and, for FP64, against one single-field call per
field, bit for bit.  Ragged rows (empty, short, over the block-summed length,
over a tile), field counts around its vector width and chunk size, padded cell
pitches, both directions."""
import numpy as np
import pytest
import scipy.sparse as sp
import torch

from test_gpu_apply import _ragged_matrix

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _lean_matrix(seed=0):
    """About 5 non-zeros a row, some rows of 33 to 200 and one of 1500 next to each other."""
    rng = np.random.default_rng(seed)
    n_dst, n_src = 4001, 3777
    n = rng.integers(0, 10, n_dst)
    n[700:720] = rng.integers(33, 200, 20)
    n[710] = 1500
    row = np.repeat(np.arange(n_dst), n)
    start = np.minimum(np.arange(n_dst) * n_src // n_dst, n_src - n)
    col = np.concatenate([s + np.arange(m) for s, m in zip(start, n)])
    A = sp.csr_matrix((rng.random(row.size) + 0.1, (row, col)), shape=(n_dst, n_src))
    return A, np.asarray(A.sum(1)).ravel() + 0.5, np.asarray(A.sum(0)).ravel() + 0.5


@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize("matrix,k,pad", [
    (_lean_matrix, 6, 0), (_lean_matrix, 7, 9), (_lean_matrix, 9, 1), (_lean_matrix, 50, 0), (_ragged_matrix, 16, 0),
    (_ragged_matrix, 37, 0), (_ragged_matrix, 64, 0), (_ragged_matrix, 129, 3), (_ragged_matrix, 257, 0),
    (_ragged_matrix, 300, 0)])
def test_levels_layout(cr, matrix, k, pad, dtype):
    print(f"[case] levels {matrix.__name__} k={k} pad={pad} {dtype}", flush=True)
    A, a_d, a_s = matrix(2)
    R = cr.Regridder.from_csr(A, a_d, a_s)
    dt = getattr(torch, dtype)
    rng = np.random.default_rng(k)
    for RR, M, area in ((R, A, a_d), (cr.transpose(R), A.T.tocsr(), a_s)):
        n_out, n_in = M.shape
        x = torch.full((n_in, k + pad), float("nan"), dtype=dt, device=DEV)
        x[:, :k] = torch.tensor(rng.random((n_in, k)) - 0.3, dtype=dt, device=DEV)
        y = torch.full((n_out, k + pad), -7.0, dtype=dt, device=DEV)
        cr.regrid_(y[:, :k], RR, x[:, :k])
        assert bool((y[:, k:] == -7.0).all())
        xin = x[:, :k].cpu().numpy().astype(np.float64)
        ref = (M @ xin) / area[:, None]
        scale = (abs(M) @ abs(xin)) / area[:, None] + 1e-300
        # FP32: FP64 sums rounded once (2^-24 of the result); FP64: a sum of at most 3000 products
        tol = 1.01 * 2.0**-24 if dtype == "float32" else 3000 * 2.0**-53
        assert np.max(np.abs(y[:, :k].cpu().numpy() - ref) / scale) <= tol
        if dtype == "float64":
            for f in {0, k // 2, k - 1}:
                yf = torch.zeros(n_out, dtype=dt, device=DEV)
                cr.regrid_(yf, RR, x[:, f].contiguous())
                assert torch.equal(yf, y[:, f]), f
        # unscaled sums
        cr.regrid_(y[:, :k], RR, x[:, :k], normalize=False)
        assert np.max(np.abs(y[:, :k].cpu().numpy() - M @ xin) / (scale * area[:, None])) <= tol
