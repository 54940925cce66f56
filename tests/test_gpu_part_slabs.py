"""Slabs of the phases that are cut into parts: one size per column count, kept
in place for the graphs that use them."""
import pytest

pytestmark = pytest.mark.gpu


def _actor(n=60_000, seed=51):
    import fmca_amd
    from fmca_amd import workloads as W
    P = W.uniform(n, 3, seed)
    return fmca_amd.H2kernelActor(fmca_amd.CovarianceKernel("MATERN32", 0.4), P, P, 3, 0.8)


def _columns(n, nrhs, seed=0):
    import torch
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(nrhs, n, generator=g, dtype=torch.float64, device="cuda").t()


@pytest.mark.parametrize("precision", ["FP64", "FP32", "FP32_BF16"])
def test_fewer_columns_allocate_nothing(precision):
    """After an action of 16 columns every action with 16 or fewer, forward or
    transposed, finds its workspaces and slabs in place, although fewer columns
    are cut into more parts."""
    import fmca_amd
    prec = getattr(fmca_amd, precision)
    H = _actor()
    H.action_device(_columns(60_000, 16), precision=prec)
    live, _ = fmca_amd.device_memory(True)
    for nrhs in (16, 8, 7, 5, 3, 1):
        print(f"[case] {precision} {nrhs} columns", flush=True)
        H.action_device(_columns(60_000, nrhs), precision=prec)
        H.action_transpose_device(_columns(60_000, nrhs), precision=prec)
        assert fmca_amd.device_memory() == (live, live)


@pytest.mark.parametrize("precision", ["FP64", "FP32", "FP32_BF16"])
@pytest.mark.parametrize("warm,nrhs", [(16, 16), (32, 5), (16, 1)])
def test_graph_keeps_its_slabs(precision, warm, nrhs):
    """A graph captured after an eager action of `warm` columns allocates
    nothing while it is captured, and eager actions of fewer columns leave its
    memory alone."""
    import torch
    import fmca_amd
    print(f"[case] {precision} warm-up {warm}, captured {nrhs}", flush=True)
    prec = getattr(fmca_amd, precision)
    H = _actor()
    x = _columns(60_000, nrhs, 1)
    y = torch.empty(nrhs, 60_000, dtype=torch.float64, device="cuda").t()
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        H.action_device(_columns(60_000, warm), precision=prec)
    torch.cuda.synchronize()
    live = fmca_amd.device_memory()[0]
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        H.action_device(x, out=y, precision=prec)
    assert fmca_amd.device_memory()[0] == live
    for k in range(3):
        x.mul_(-0.5).add_(0.25 * k)
        for c in (1, 5, 8, 16):
            H.action_device(_columns(60_000, c, 2 + k), precision=prec)
            H.action_transpose_device(_columns(60_000, c, 3 + k), precision=prec)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        ref = H.action_device(x, precision=prec)
        # captured with other parts than the eager call: another order of the sums
        tol = 1e-14 if precision == "FP64" else 4e-6
        assert (torch.linalg.norm(y - ref) / torch.linalg.norm(ref)).item() <= tol


def test_slabs_make_room_for_other_allocations():
    """Under a memory cap that holds the actor's blocks but not its slabs beside
    them, the blocks are stored and the actions go on."""
    import torch
    import fmca_amd
    print("[case] cap without room for slabs", flush=True)
    n = 6000
    x = _columns(n, 16)
    H = _actor(n)
    H.upload()
    live = fmca_amd.device_memory()[0]
    H.assemble(fmca_amd.FP64)
    blocks = fmca_amd.device_memory()[0] - live
    H.action_device(x)
    H = _actor(n)
    H.upload()
    y = H.action_device(x)
    live, _ = fmca_amd.device_memory(True)
    slabs = 16 * n * 16 * 8
    fmca_amd.set_device_memory_limit(live + blocks - slabs // 2)
    try:
        H.assemble(fmca_amd.FP64)
        z = H.action_device(x)
        assert fmca_amd.device_memory()[1] <= live + blocks - slabs // 2
    finally:
        fmca_amd.set_device_memory_limit(0)
    assert (torch.linalg.norm(z - y) / torch.linalg.norm(y)).item() <= 1e-13
