"""The vector-ALU forms of the entry phases (fewer than 8 right-hand sides) and
the launches cut into parts: leaf and node counts around the workgroup sizes,
every column tile, lists shorter and longer than a staged tile, no far blocks."""
import numpy as np
import pytest

import oracle
from conftest import rel_err

pytestmark = pytest.mark.gpu

# the repository's bar of the FP64 action against the oracle, and of FP32
# against FP64 (tests/test_gpu_action.py)
FP64_TOL = 1e-12
FP32_TOL = 1e-5


# (dim, n, degree, eta): leaf sizes and node counts q around 64, 128 and 256
# lanes, one leaf only, all-dense trees, q above one pass of 256 rows
SETS = [
    (1, 1, 2, 0.8), (1, 700, 3, 0.8), (2, 65, 1, 0.8), (2, 257, 5, 0.8), (2, 3001, 2, 0.8),
    (3, 129, 3, 0.8), (3, 4000, 4, 0.8), (3, 5003, 2, 0.0), (3, 9001, 3, 0.8), (3, 3000, 6, 0.8),
]


@pytest.mark.parametrize("dim,n,deg,eta", SETS)
def test_few_columns_match_the_oracle(dim, n, deg, eta):
    import torch
    import fmca_amd
    print(f"[case] {dim}-D n={n} deg={deg} eta={eta}", flush=True)
    rng = np.random.default_rng(n + deg)
    P = np.asfortranarray(rng.random((dim, n)))
    x = np.asfortranarray(rng.standard_normal((n, 8)))
    K = fmca_amd.CovarianceKernel("MATERN52", 0.4)
    H = fmca_amd.H2kernelActor(K, P, P, deg, eta)
    ref = oracle.OracleH2(P, P, "MATERN52", 0.4, deg, eta).action(x)
    for nrhs in (1, 2, 3, 4, 5, 6, 7, 8):
        xd = torch.from_numpy(np.asfortranarray(x[:, :nrhs])).cuda()
        y = H.action_device(xd).cpu().numpy()
        assert rel_err(y, ref[:, :nrhs]) <= FP64_TOL
        y2 = H.action_device(xd).cpu().numpy()
        assert np.array_equal(y, y2)  # parts are added in order
        y32 = H.action_device(xd, precision=fmca_amd.FP32).cpu().numpy()
        assert rel_err(y32, ref[:, :nrhs]) <= FP32_TOL


@pytest.mark.parametrize("interp", ["tensor_product", "total_degree"])
@pytest.mark.parametrize("nrhs", [1, 6, 8, 16, 40])
def test_parts_on_rectangular_and_transposed_sets(interp, nrhs):
    import torch
    import fmca_amd
    rng = np.random.default_rng(7)
    P, T = (np.asfortranarray(rng.random((3, k))) for k in (6007, 1503))
    K = fmca_amd.CovarianceKernel("EXPONENTIAL", 0.5)
    H = fmca_amd.H2kernelActor(K, T, P, 3, 0.8, interp)
    x = torch.from_numpy(np.asfortranarray(rng.standard_normal((6007, nrhs)))).cuda()
    z = torch.from_numpy(np.asfortranarray(rng.standard_normal((1503, nrhs)))).cuda()
    o = oracle.OracleH2(P, T, "EXPONENTIAL", 0.5, 3, 0.8,
                        scheme="tensor" if interp == "tensor_product" else interp)
    y = o.action(x.cpu().numpy())
    for prec, tol in ((fmca_amd.FP64, FP64_TOL), (fmca_amd.FP32, FP32_TOL),
                      (fmca_amd.FP32_BF16, 2 * FP32_TOL)):
        assert rel_err(H.action_device(x, precision=prec).cpu().numpy(), y) <= tol
        a = H.action_transpose_device(z, precision=prec).cpu().numpy()
        # <K x, z> = <x, K^T z>, to the rounding of the two products
        lhs = float((torch.from_numpy(y).cuda() * z).sum())
        scale = np.linalg.norm(y) * np.linalg.norm(z.cpu().numpy())
        assert abs(float((x.cpu().numpy() * a).sum()) - lhs) <= tol * scale


@pytest.mark.parametrize("ktype,l", [("EXPONENTIAL", 0.3), ("MATERN32", 0.3),
                                     ("MATERN52", 0.05), ("GAUSSIAN", 0.2)])
def test_fp64_entries_are_accurate_to_a_few_ulp(ktype, l):
    """One source at the origin: the outputs are the entries themselves, here
    against 80-bit arithmetic from r = 0 to the underflow of the exponential.
    r carries about 2 ulp (products, sum, root), which the exponential
    multiplies by s r; its own error and the polynomial's are about 2 ulp."""
    import torch
    import fmca_amd
    r = np.concatenate([[0.0, 1e-160, 1e-20], np.geomspace(1e-9, 1.0, 2000),
                        np.linspace(1.0, 800.0, 2000) * l])
    T = np.asfortranarray(np.vstack([r, 0 * r]))
    P = np.zeros((2, 1), order="F")
    H = fmca_amd.H2kernelActor(fmca_amd.CovarianceKernel(ktype, l), T, P, 2, 0.0)
    y = H.action_device(torch.ones((1, 1), dtype=torch.float64, device="cuda")).cpu().numpy()[:, 0]
    q = r.astype(np.longdouble)
    s = {"EXPONENTIAL": np.longdouble(1) / l, "MATERN32": np.sqrt(np.longdouble(3)) / l,
         "MATERN52": np.sqrt(np.longdouble(5)) / l, "GAUSSIAN": np.longdouble(0)}[ktype]
    if ktype == "GAUSSIAN":
        a = q * q / (2 * np.longdouble(l) ** 2)
        k = np.exp(-a)
    else:
        a = s * q
        k = np.exp(-a) * {"EXPONENTIAL": 1, "MATERN32": 1 + a,
                          "MATERN52": 1 + a + a * a / 3}[ktype]
    ok = k > 1e-300
    err = np.abs((y[ok] - k[ok]) / k[ok])
    bound = 2.3e-16 * (2 + 2 * a[ok])
    print(f"  {ktype}: worst error / bound {float((err / bound).max()):.2f}", flush=True)
    assert np.all(err <= bound)
    assert y[0] == 1.0 and np.all(y[~ok] >= 0) and np.all(y[~ok] <= 1e-299)
