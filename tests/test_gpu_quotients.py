"""The Euler plugin's quotients by a refined hardware reciprocal and by one
taken from square roots, and its inverses, against numpy's IEEE division, on the operands that
are hardest to round: denominators whose significand is all ones or nearly so
(the reciprocal of every second one lies next to a midpoint), and for a
denominator B the numerators A with A * 2**54 or A * 2**53 = +-1 (mod B),
whose quotients lie as close to the midpoint of two numbers as any by B."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KERNEL = r"""
extern "C" __global__ void ps_quotient_check(const double *num, const double *den, double *out, int cnt)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= cnt)
        return;
    const double a = num[i], b = den[i];
    out[4 * i + 0] = eu_quo_pos(a, eu_recip(b));
    out[4 * i + 1] = eu_quo(a, eu_recip(b));
    out[4 * i + 2] = eu_quo_pos(a, eu_sqrt_recip(b).rx);
    out[4 * i + 3] = eu_inverse(b);
}
"""


def _hard_pairs(B):
    """Numerators (integers of 53 bits) that lie hardest for the odd 53-bit
    denominators B, and those denominators."""
    num, den = [], []
    for b in B:
        # quotients in (1/2, 1) have their midpoints at odd multiples of 2**-54, those in (1, 2) at 2**-53
        below, above = pow(1 << 54, -1, b), pow(1 << 53, -1, b)
        for a in (below, b - below, above + b, 2 * b - above):
            if 1 << 52 <= a < 1 << 53:
                num.append(a)
                den.append(b)
    return np.array(num, dtype=np.float64), np.array(den, dtype=np.float64)


def _operands(case):
    rng = np.random.default_rng(11)
    if case == "all_ones":  # every exponent that a density may have, numerators down to a squared momentum's
        e = np.arange(-119, 121)
        den = np.repeat(2.0 ** e * (1 - 2.0 ** -53), 512)
        num = 2.0 ** rng.integers(-800, 241, den.size)
        num[1::2] *= rng.uniform(1, 2, num[1::2].size)
        return num, den
    if case == "near_all_ones":
        k = list(range(1, 1 << 15, 2)) + (2 * rng.integers(1 << 14, 1 << 30, 1 << 15) + 1).tolist()
        num, den = _hard_pairs([(1 << 53) - int(j) for j in k])
    elif case == "near_midpoint":  # (2**53 - k): k*k a whole number of 2**54 puts the reciprocal next to a midpoint
        c = [math.isqrt(m << 54) | 1 for m in range(1, 512)]
        num, den = _hard_pairs([(1 << 53) - k - j for k in c for j in range(-64, 65, 2)])
    elif case == "near_one":
        num, den = _hard_pairs([(1 << 52) + 2 * int(j) + 1 for j in range(1 << 15)])
    else:
        num, den = _hard_pairs([int(b) | 1 for b in rng.integers(1 << 52, 1 << 53, 1 << 16)])
    s = 2.0 ** rng.integers(-110, 60, num.size)
    return num * 2.0 ** -53 * s, den * 2.0 ** -53 * 2.0 ** rng.integers(-100, 100, num.size)


@pytest.mark.parametrize("case", ["all_ones", "near_all_ones", "near_midpoint", "near_one", "any"])
def test_hardest_quotients_are_ieee(device, case):
    import ctypes
    from pysweep_amd import compiler, hip, kernels
    from pysweep_amd.equations import path as eq_path
    num, den = _operands(case)
    n = len(num)
    spec = kernels.standard_spec(eq_path("euler.cu"), 4, 2, 2, 64, 64)
    mod = hip.Module(compiler.compile_cached(spec.source() + KERNEL, "euler_quotient_check"))
    dn, dd, do = hip.DeviceArray(8 * n), hip.DeviceArray(8 * n), hip.DeviceArray(32 * n)
    dn.upload(num)
    dd.upload(den)
    hip.launch(mod.get_function("ps_quotient_check"), ((n + 255) // 256,), (256,),
               [ctypes.c_void_p(dn.ptr), ctypes.c_void_p(dd.ptr), ctypes.c_void_p(do.ptr), ctypes.c_int(n)])
    hip.synchronize()
    out = do.download(np.empty((n, 4)))
    for a in (dn, dd, do):
        a.close()
    mod.unload()
    for j in range(4):
        bad = np.flatnonzero(out[:, j] != (num / den if j < 3 else 1 / den))
        assert not bad.size, (case, j, bad.size, num[bad[0]].hex(), den[bad[0]].hex())
