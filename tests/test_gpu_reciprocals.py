"""The Euler plugin's reciprocals taken from a density's square root, and
its three-instruction refinement of the hardware reciprocal, against numpy's
IEEE division and square root where they can go wrong: significands of all
ones and their neighbours (a uniform stream's densities), whose reciprocals
lie next to the midpoint of two numbers, and zero denominators of the
limiter's ratios."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KERNEL = r"""
extern "C" __global__ void ps_recip_check(const double *num, const double *den, double *out, int cnt)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= cnt)
        return;
    const double a = num[i], b = den[i];
    const eu_root w = eu_sqrt_recip(b);
    out[5 * i + 0] = w.s;
    out[5 * i + 1] = eu_quo_pos(a, w.rx);
    /* the Roe density's reciprocal, from two roots */
    const eu_root v = eu_sqrt_recip(b * 1.25);
    const double a0 = w.s * v.s;
    out[5 * i + 2] = a0;
    out[5 * i + 3] = eu_quo_pos(a, eu_recip_from(a0, w.y * v.y));
    out[5 * i + 4] = eu_ratio(a, eu_recip(b));
}
"""


def _run(num, den):
    import ctypes
    from pysweep_amd import compiler, hip, kernels
    from pysweep_amd.equations import path as eq_path
    spec = kernels.standard_spec(eq_path("euler.cu"), 4, 2, 2, 64, 64)
    mod = hip.Module(compiler.compile_cached(spec.source() + KERNEL, "euler_recip_check"))
    n = len(num)
    dn, dd, do = hip.DeviceArray(8 * n), hip.DeviceArray(8 * n), hip.DeviceArray(40 * n)
    dn.upload(np.ascontiguousarray(num))
    dd.upload(np.ascontiguousarray(den))
    hip.launch(mod.get_function("ps_recip_check"), ((n + 255) // 256,), (256,),
               [ctypes.c_void_p(dn.ptr), ctypes.c_void_p(dd.ptr), ctypes.c_void_p(do.ptr), ctypes.c_int(n)])
    hip.synchronize()
    out = do.download(np.empty((n, 5)))
    for a in (dn, dd, do):
        a.close()
    mod.unload()
    return out


def _near(rng, n, centres, ulps):
    v = rng.choice(np.asarray(centres), n).view(np.int64) + rng.integers(-ulps, ulps + 1, n)
    return v.view(np.float64) * 2.0 ** rng.integers(-40, 41, n)


@pytest.mark.parametrize("case", ["stream", "random", "guard"])
def test_reciprocals_from_roots_are_ieee(device, case):
    """Quotients and square roots are the IEEE ones, exactly."""
    rng = np.random.default_rng({"stream": 1, "random": 2, "guard": 3}[case])
    n = 1 << 21
    if case == "stream":
        c = [1.0, 2.0, 1.25, 1.5, 1.4, 1.75, 2.5, 5 / 7, 25 / 14, 4 / 3]
        num, den = _near(rng, n, c, 12), _near(rng, n, c[:4], 12)
    elif case == "random":
        num, den = rng.uniform(1e-3, 10, n), rng.uniform(1e-3, 10, n)
    else:
        num = rng.uniform(1, 2, n) * 2.0 ** rng.integers(-520, 251, n)
        den = rng.uniform(1, 2, n) * 2.0 ** rng.integers(-120, 120, n)
    out = _run(num, den)
    assert np.array_equal(out[:, 0], np.sqrt(den))
    assert np.array_equal(out[:, 1], num / den)
    assert np.array_equal(out[:, 2], np.sqrt(den) * np.sqrt(den * 1.25))
    assert np.array_equal(out[:, 3], num / out[:, 2])


def test_limiter_ratios_are_ieee(device):
    """min(num/den, 1), zeroed when nan, inf, above 1e6 or negative, for
    differences of a few ulps, zeros among them, and at the 1e6 edge."""
    rng = np.random.default_rng(4)
    n = 1 << 20
    num = rng.integers(-6, 7, n) * 2.0 ** -53
    den = rng.integers(-6, 7, n) * 2.0 ** -53
    num[: n // 4] = rng.uniform(-1, 1, n // 4)
    den[n // 8: n // 2] = rng.uniform(-1e-5, 1e-5, n // 2 - n // 8)
    num[-64:] = 1e6 + np.arange(-32, 32) * 2.0 ** -33
    den[-64:] = 1.0
    with np.errstate(all="ignore"):
        pr = num / den
        pr = np.where(np.isnan(pr) | np.isinf(pr) | (pr > 1e6) | (pr < 0), 0.0, pr)
    assert np.array_equal(_run(num, den)[:, 4], np.minimum(pr, 1.0))
