"""Matrix-core launches by list length: whole, cut into parts, with the K-steps
of a leaf split over the waves, and both."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (dim, n, degree, clustered): few targets (parts), small leaves with long lists
# (split), short lists (neither), long lists of many targets, split tasks
SETS = [(3, 4000, 1, False), (3, 4000, 3, False), (3, 30000, 1, False), (3, 30000, 3, False),
        (2, 30000, 1, False), (2, 30000, 5, False), (1, 9000, 3, False), (2, 30000, 4, True),
        (3, 12000, 4, True)]


@pytest.mark.parametrize("dim,n,deg,clustered", SETS)
@pytest.mark.parametrize("ktype", ["EXPONENTIAL", "MATERN32"])
def test_columns_agree_with_the_vector_forms(dim, n, deg, clustered, ktype):
    """Columns of the matrix-core forms against the same columns one at a time
    (vector forms, other kernels and another order of the sums).  FP64: a sum of
    up to 3e4 terms of both signs, 1e-13; FP32 entries: 1e-5, the repository's
    bar against FP64.  A column's error is bounded by the rounding of |K| |x|,
    which is alike for all columns, while ||K x|| varies between them with the
    cancellation (1-D, the exponential: ten times), so errors are measured
    against the mean norm of the columns, not each column's own."""
    import torch
    import fmca_amd
    print(f"[case] {dim}-D n={n} degree {deg} clustered={clustered} {ktype}", flush=True)
    rng = np.random.default_rng(n + deg)
    P = rng.random((dim, n))
    if clustered:
        P = 0.02 * rng.standard_normal((dim, n)) + rng.random((dim, 16))[:, rng.integers(0, 16, n)]
    P = np.asfortranarray(P)
    H = fmca_amd.H2kernelActor(fmca_amd.CovarianceKernel(ktype, 0.3), P, P, deg, 0.8)
    x = torch.from_numpy(rng.standard_normal((n, 50))).cuda()
    ref = torch.stack([H.action_device(x[:, j].contiguous()) for j in range(50)], 1)
    scale = torch.linalg.norm(ref) / 50 ** 0.5
    for nrhs in (8, 16, 17, 32, 50):
        for prec, tol in ((fmca_amd.FP64, 1e-13), (fmca_amd.FP32, 1e-5), (fmca_amd.FP32_BF16, 2e-5)):
            y = H.action_device(x[:, :nrhs].t().contiguous().t(), precision=prec)
            err = torch.linalg.norm(y - ref[:, :nrhs], dim=0) / scale
            assert err.max().item() <= tol, (nrhs, prec)
