"""The BF16 precision form against FP64: leaves of one to sixteen and more row
tiles (wave groups that share the sources), node counts around the same edges,
passes of 16, 32 and 64 columns with remainders, every distance form.  The
smallest leaves and node sets take the FP32 form's kernels."""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu

# entries and right operands split into two BF16 terms each: the dropped terms
# are 2^-16 of a product, the distances carry FP32 error as in the FP32 form,
# whose bar is 1e-5 (tests/test_gpu_action.py); 2^-16 and that bar together
TOL = 1e-5 + 2.0 ** -16

# (dim, n, degree, interpolation): leaves of 15 to 300 rows, q from 2 to 216
SETS = [
    (1, 700, 3, "tensor_product"), (2, 500, 1, "tensor_product"), (2, 3001, 3, "tensor_product"),
    (2, 5000, 7, "tensor_product"), (2, 9000, 9, "tensor_product"), (3, 900, 1, "tensor_product"),
    (3, 4000, 2, "tensor_product"), (3, 9001, 3, "tensor_product"), (3, 9001, 4, "tensor_product"),
    (3, 9001, 4, "total_degree"), (3, 12000, 5, "tensor_product"),
]


@pytest.mark.parametrize("dim,n,deg,interp", SETS)
def test_tiles_match_fp64(dim, n, deg, interp):
    import torch
    import fmca_amd
    print(f"[case] {dim}-D n={n} deg={deg} {interp}", flush=True)
    rng = np.random.default_rng(n + deg)
    P = np.asfortranarray(rng.random((dim, n)))
    x = torch.from_numpy(np.asfortranarray(rng.standard_normal((n, 97)))).cuda()
    for ktype in ("MATERN32", "EXPONENTIAL", "MATERN52", "GAUSSIAN", "MULTIQUADRIC"):
        H = fmca_amd.H2kernelActor(fmca_amd.CovarianceKernel(ktype, 0.4), P, P, deg, 0.8, interp)
        y = H.action_device(x).cpu().numpy()
        for nrhs in (8, 16, 17, 32, 33, 49, 64, 65, 97):
            yb = H.action_device(x[:, :nrhs].T.contiguous().T,
                                 precision=fmca_amd.FP32_BF16).cpu().numpy()
            assert rel_err(yb, y[:, :nrhs]) <= TOL, (ktype, nrhs)


def test_distances_far_from_the_origin_keep_the_fp32_error():
    """Clusters of a point cloud far off the origin: the squared distances come
    from differences to a nearby centre, so their error does not grow with the
    coordinates' size."""
    import torch
    import fmca_amd
    rng = np.random.default_rng(5)
    P = np.asfortranarray(rng.random((3, 6000)) + np.array([[100.0], [-50.0], [7.0]]))
    x = torch.from_numpy(np.asfortranarray(rng.standard_normal((6000, 40)))).cuda()
    H = fmca_amd.H2kernelActor(fmca_amd.CovarianceKernel("MATERN32", 0.3), P, P, 3, 0.8)
    y = H.action_device(x).cpu().numpy()
    err = [rel_err(H.action_device(x, precision=p).cpu().numpy(), y)
           for p in (fmca_amd.FP32, fmca_amd.FP32_BF16)]
    assert err[1] <= err[0] + 2.0 ** -16
