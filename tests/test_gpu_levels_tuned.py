"""Fields side by side keep their kernel after cr_regrid_tune, on whichever layout it
was tuned; a pinned variant takes its place.  The kernels are told apart by the last
bits of row sums that nearly cancel."""
import numpy as np
import pytest
import scipy.sparse as sp
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _cancelling_matrix():
    """40 non-zeros a row, the second half minus the first but for 1e-12."""
    rng = np.random.default_rng(1)
    n, half = 3000, 20
    v = rng.random((n, half)) + 0.1
    val = np.concatenate([v, -v * (1.0 + 1e-12 * rng.standard_normal((n, half)))], 1)
    col = (np.arange(n)[:, None] + np.arange(2 * half)) % n
    A = sp.csr_matrix((val.ravel(), (np.repeat(np.arange(n), 2 * half), col.ravel())), shape=(n, n))
    return A, np.ones(n), np.ones(n)


@pytest.mark.parametrize("tuned_on", ["cells", "levels"])
@pytest.mark.parametrize("transposed", [False, True])
def test_tuning_leaves_the_side_by_side_kernel(cr, tuned_on, transposed):
    print(f"[case] tuned on {tuned_on}, transposed={transposed}", flush=True)
    R = cr.Regridder.from_csr(*_cancelling_matrix())
    if transposed:
        R = cr.transpose(R)
    n, k = R.shape[0], 24
    x = torch.ones(n, k, dtype=torch.float32, device=DEV)
    before, y = (torch.zeros(n, k, dtype=torch.float32, device=DEV) for _ in range(2))
    cr.regrid_(before, R, x)
    if tuned_on == "levels":
        cr.regrid_tune(y, R, x)
    else:
        cr.regrid_tune(torch.zeros(k, n, dtype=torch.float32, device=DEV), R, x.T.contiguous(), dims=2)
    cr.regrid_(y, R, x)
    assert torch.equal(y, before)
    cr.regrid_set_variant(R, 15)
    cr.regrid_(y, R, x)
    assert not torch.equal(y, before)
    cr.regrid_set_variant(R, -1)
    cr.regrid_(y, R, x)
    assert torch.equal(y, before)
