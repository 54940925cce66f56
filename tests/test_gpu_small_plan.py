"""Device trees whose levels are split by one workgroup per node, and block
expansions by one workgroup: node sizes at the edges of its 64, 1024, 4096 and
16384 point tiles, coordinates that differ in few or in all bits of the radix
select, pairs up to and past the small levels; bit-exact against the host
planner, ties handed to it."""
import numpy as np
import pytest

from test_gpu_tree import _points, _same_blocks, _same_tree

pytestmark = pytest.mark.gpu

SIZES = [2, 3, 63, 64, 65, 1023, 1024, 1025, 4095, 4097, 16384, 16385, 32767, 65537]


def _pair(P, deg, eta=0.8):
    import fmca_amd
    ker = fmca_amd.CovarianceKernel("EXPONENTIAL", 0.5)
    return (fmca_amd.H2kernelActor(ker, P, P, deg, eta, planner=p) for p in ("device", "host"))


@pytest.mark.parametrize("kind", ["uniform", "signed", "mixture"])
@pytest.mark.parametrize("n", SIZES)
def test_small_levels_equal_the_host_plan(kind, n):
    print(f"[case] small levels {kind} n={n}", flush=True)
    d = 1 + n % 3
    Hd, Hh = _pair(_points(kind, n, d, n), 1)
    assert Hd.plan_report()["rows_tree"] == "device"
    _same_tree(Hd, Hh, 0)
    _same_blocks(Hd, Hh)


@pytest.mark.parametrize("scale", [2.0 ** -1060, 1e-300, 1.0, 1e300])
def test_keys_that_differ_in_few_bits(scale):
    """Neighbouring doubles (the last bits differ), subnormals, and keys of both
    signs over the whole exponent range (the first bit differs)."""
    rng = np.random.default_rng(2)
    a = np.float64(scale).view(np.int64) + rng.permutation(3000)
    P = np.asfortranarray(a.view(np.float64)[None, :])
    for Q in (P, np.asfortranarray(np.where(rng.random(3000) < 0.5, P, -P))):
        Hd, Hh = _pair(Q, 2, eta=0.0)
        assert Hd.plan_report()["rows_tree"] == "device"
        _same_tree(Hd, Hh, 0)


def test_one_tie_at_the_median_goes_to_the_host():
    rng = np.random.default_rng(3)
    x = np.sort(rng.random(2000))
    x[999] = x[1000]
    Hd, Hh = _pair(np.asfortranarray(rng.permutation(x)[None, :]), 3)
    assert Hd.plan_report()["rows_tree"] == "host-fallback"
    _same_tree(Hd, Hh, 0)
    _same_blocks(Hd, Hh)
