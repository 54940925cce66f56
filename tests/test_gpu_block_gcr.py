"""GCR with several right-hand sides: the columns of a block of up to 32 share
one Krylov space."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _setup(n, nrhs, ktype="MATERN32", seed=1):
    import torch
    import fmca_amd
    rng = np.random.default_rng(seed)
    P = np.asfortranarray(rng.random((3, n)))
    H = fmca_amd.H2kernelActor(fmca_amd.CovarianceKernel(ktype, 0.4), P, P, 3, 0.8)
    b = torch.from_numpy(np.asfortranarray(rng.standard_normal((n, nrhs)))).cuda()
    return H, b


def _resid(H, x, b, ridge):
    import torch
    r = b - H.action_device(x) - ridge * x
    return (torch.linalg.norm(r, dim=0) / torch.linalg.norm(b, dim=0)).max().item()


# column counts around one 16-column tile and one and two 32-column blocks; n
# around whole 64-row tiles
@pytest.mark.parametrize("n,nrhs", [(2048, 2), (2049, 16), (3001, 17), (2111, 32), (2500, 33),
                                    (2048, 65)])
@pytest.mark.parametrize("precision", ["FP64", "FP32", "FP32_BF16"])
def test_block_sizes(n, nrhs, precision):
    import torch
    import fmca_amd
    print(f"[case] n={n} nrhs={nrhs} {precision}", flush=True)
    H, b = _setup(n, nrhs)
    ridge = 0.2
    x, info = H.cg(b, x0=torch.zeros_like(b), ridge=ridge, tol=1e-9, method="gcr",
                   precision=getattr(fmca_amd, precision), max_iter=300)
    print("  ", info, flush=True)
    assert info["converged"] and _resid(H, x, b, ridge) <= 1e-9
    x1, i1 = H.cg(b[:, 0].contiguous(), x0=torch.zeros_like(b[:, 0]), ridge=ridge, tol=1e-9,
                  method="gcr", precision=getattr(fmca_amd, precision))
    assert info["iterations"] <= i1["iterations"] + 1
    # both residuals are <= 1e-9: the difference is bounded by cond * 2e-9 in
    # the direction of the smallest eigenvalue, ||dx|| <= 2e-9 ||b|| / ridge
    d = torch.linalg.norm(x[:, 0] - x1).item()
    assert d <= 2e-9 * torch.linalg.norm(b[:, 0]).item() / ridge


def test_dependent_zero_and_non_finite_columns():
    """Equal and linearly dependent columns leave the block with fewer new
    directions than columns; zero columns stay zero; a column of NaN is
    neither solved nor lets its values into the others, which are, and the
    solve reports that not every column reached tol."""
    import torch
    import fmca_amd
    H, b = _setup(3000, 7)
    b[:, 2] = b[:, 0]
    b[:, 3] = b[:, 0] - 2 * b[:, 1]
    b[:, 4] = 0
    b[:, 5] = float("nan")
    good = [0, 1, 2, 3, 6]
    for prec in (fmca_amd.FP64, fmca_amd.FP32_BF16):
        x, info = H.cg(b, x0=torch.zeros_like(b), ridge=0.3, tol=1e-9, method="gcr",
                       precision=prec, max_iter=300)
        assert not info["converged"] and np.isnan(info["rel_residual"])
        assert info["iterations"] < 300
        assert _resid(H, x[:, good].t().contiguous().t(), b[:, good].t().contiguous().t(),
                      0.3) <= 1e-9
        assert torch.all(x[:, 4] == 0) and torch.all(x[:, 5] == 0)


@pytest.mark.parametrize("precision", ["FP64", "FP32_BF16"])
def test_window_that_spans_the_whole_space(precision):
    """32 columns of 90 unknowns: three blocks span the space, after which only
    the replaced residual's projections on the window reduce it."""
    import torch
    import fmca_amd
    H, b = _setup(90, 32, "EXPONENTIAL")
    x, info = H.cg(b, x0=torch.zeros_like(b), ridge=1e-3, tol=1e-10, method="gcr",
                   precision=getattr(fmca_amd, precision), max_iter=60)
    print("  ", info, flush=True)
    assert info["converged"] and _resid(H, x, b, 1e-3) <= 1e-10


def test_start_vector_and_small_window():
    import torch
    import fmca_amd
    H, b = _setup(2500, 5, "EXPONENTIAL")
    x0 = torch.randn_like(b)
    for m in (2, 5):
        x, info = H.cg(b, x0=x0, ridge=0.5, tol=1e-9, method="gcr", precision=fmca_amd.FP32,
                       max_basis=m, max_iter=3000)
        assert info["converged"] and info["iterations"] > m
        assert _resid(H, x, b, 0.5) <= 1e-9


def test_without_room_for_the_shared_space():
    """A memory cap that holds the vectors of one space per column but not the
    block form's partial sums: the solve takes the former."""
    import torch
    import fmca_amd
    H, b = _setup(3000, 8)
    args = dict(ridge=0.5, tol=1e-9, method="gcr", precision=fmca_amd.FP32, max_basis=40)
    x0 = torch.zeros_like(b)
    H.action_device(b, precision=fmca_amd.FP64)
    H.action_device(b, precision=fmca_amd.FP32)
    live = fmca_amd.device_memory()[0]
    # 4 vectors, 40 pairs in chunks of 8, scalars; the block form's sums take 16 MB
    fmca_amd.set_device_memory_limit(live + (4 * 8 + 40 * 8) * 3000 * 8 + (3 << 20))
    try:
        x, info = H.cg(b, x0=x0, **args)
    finally:
        fmca_amd.set_device_memory_limit(0)
    print("  ", info, flush=True)
    assert info["converged"] and _resid(H, x, b, 0.5) <= 1e-9
    y, info2 = H.cg(b, x0=x0, **args)
    assert info2["converged"] and info2["iterations"] < info["iterations"]


@pytest.mark.parametrize("method,nrhs", [("cg", 3), ("gcr", 1), ("gcr", 3)])
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_a_non_finite_column_is_reported(method, nrhs, bad):
    """No solver reports convergence when a column of b (or, as NaN, of the
    start vector) is not finite."""
    import torch
    import fmca_amd
    H, b = _setup(500, nrhs)
    x0 = torch.zeros_like(b)
    for where in (b, x0) if np.isnan(bad) else (b,):
        v = where[7, nrhs - 1].item()
        where[7, nrhs - 1] = bad
        x, info = H.cg(b, x0=x0, ridge=0.5, method=method, precision=fmca_amd.FP64)
        assert not info["converged"] and not np.isfinite(info["rel_residual"])
        where[7, nrhs - 1] = v
    x, info = H.cg(b, x0=x0, ridge=0.5, method=method, precision=fmca_amd.FP64)
    assert info["converged"]


@pytest.mark.parametrize("precision,n,nrhs", [("FP32", 5000, 32), ("FP32", 1000, 2),
                                              ("FP32_BF16", 1000, 8), ("FP32_BF16", 1000, 32)])
def test_a_stalled_recurrence_is_replaced(precision, n, nrhs):
    """Ridge 1e-7 n and a refine_factor below what the stored pairs of lower
    precision reach: the block's recurrence stalls before its columns have
    dropped by the factor, and goes on from the FP64 residual."""
    import torch
    import fmca_amd
    from fmca_amd import workloads as W
    print(f"[case] {precision} n={n} nrhs={nrhs}", flush=True)
    P = W.uniform(n, 3, 1)
    H = fmca_amd.H2kernelActor(fmca_amd.CovarianceKernel("MATERN32", 0.4), P, P, 4, 0.8)
    b = torch.from_numpy(np.random.default_rng(1).standard_normal((n, nrhs))).cuda()
    x, info = H.cg(b, x0=torch.zeros_like(b), ridge=1e-7 * n, tol=1e-8, method="gcr",
                   precision=getattr(fmca_amd, precision), refine_factor=3e-5, max_iter=1000)
    print("  ", info, flush=True)
    assert info["converged"] and info["rel_residual"] <= 1e-8


def test_a_solve_stopped_at_its_cap_is_judged_by_its_residual():
    """The last iteration allowed meets tol: converged, as the FP64 residual
    of the returned x says."""
    import torch
    import fmca_amd
    H, b = _setup(2000, 4)
    args = dict(x0=torch.zeros_like(b), ridge=0.5, tol=1e-8, method="gcr",
                precision=fmca_amd.FP64)
    _, full = H.cg(b, **args)
    for k in (full["iterations"], full["iterations"] - 1):
        _, info = H.cg(b, max_iter=k, **args)
        assert info["converged"] == (info["rel_residual"] <= 1e-8)
