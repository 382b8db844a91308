/*
 * 2-D compressible Euler equations, conserved variables
 * (rho, rho*u, rho*v, E), finite volume on a periodic grid: minmod
 * pressure-ratio limited reconstruction, central flux plus spectral-radius
 * (Roe-averaged) dissipation, midpoint RK2, radius-2 cross stencil.
 *
 * Device half of the Euler plugin pair (euler.py).  The arithmetic follows
 * the numpy step of the reference plugin operation by operation
 * (pysweep/equations/euler.py:131-313: getFluxInX/Y, evaluateFluxInX/Y,
 * fluxLimiter, evaluateSpectral, getPressure), squares evaluated as a*a, so
 * device results agree bitwise with a numpy evaluation in that order.  The
 * scheme amplifies round-off strongly (the limiter zeroes ratios of
 * round-off-sized pressure differences), so a different operation order
 * would not stay within 1e-12 of the numpy path beyond a few stages.
 *
 * Contract: step(shared_state, idx, globalTimeStep) writes the four
 * variables at shared_state[idx + v*VARS + TIMES]; x neighbours idx +- SY,
 * y neighbours idx +- 1, level one back idx - TIMES.
 */
__device__ __constant__ double DX;
__device__ __constant__ double DY;
__device__ __constant__ double DT;
__device__ __constant__ double GAMMA;
__device__ __constant__ double GAM_M1;
__device__ __constant__ double DTDX;
__device__ __constant__ double DTDY;

struct eu_q {
    double r, m, n, e; /* rho, rho*u, rho*v, E */
};

/*
 * Range of states for which the fast quotients and square roots below are
 * bitwise the IEEE ones: rho, E and the pressure in [2^-120, 2^120], each
 * momentum 0 or of magnitude in [2^-400, 2^120].  Every quotient of the
 * step then has operands at least 2^53 above the subnormal range and fewer
 * than 768 binary orders apart, and every denominator but the limiter's is
 * a positive normal number.  A state outside it sets EU_RANGE_FAULT (a
 * module global the host clears before a solve and reads after it: the
 * solve is then repeated with EU_EXACT_DIVISION, where every quotient and
 * square root is the compiler's IEEE `/` and `sqrt`).
 */
__device__ int EU_RANGE_FAULT;
#ifdef EU_EXACT_DIVISION
#define EU_EXACT 1
#else
#define EU_EXACT 0
#endif

/* (`&` and `|`: short-circuit evaluation compiled to a chain of branches) */
__device__ __forceinline__ bool eu_pos_in_range(double v) { return (v >= 0x1p-120) & (v <= 0x1p120); }

__device__ __forceinline__ bool eu_mom_in_range(double v)
{
    const double a = fabs(v);
    return (a <= 0x1p120) & ((a >= 0x1p-400) | (a == 0.0));
}

__device__ __forceinline__ bool eu_in_range(double r, double m, double n, double e, double p)
{
    return eu_pos_in_range(r) & eu_pos_in_range(e) & eu_pos_in_range(p) & eu_mom_in_range(m) & eu_mom_in_range(n);
}

/* flag a state outside the range (a vector store; a benign race: every
 * writer writes 1) */
__device__ __forceinline__ void eu_range_check(double r, double m, double n, double e, double p)
{
    if (!eu_in_range(r, m, n, e, p))
        *(volatile int *)&EU_RANGE_FAULT = 1;
}

/* state values are read into double whatever the storage type R */
template <class R>
__device__ __forceinline__ eu_q eu_at(const R *s, int i)
{
    eu_q q;
    q.r = s[i];
    q.m = s[i + VARS];
    q.n = s[i + 2 * VARS];
    q.e = s[i + 3 * VARS];
    return q;
}

/* the same from an object indexed like a level slot (s[i]) */
template <class S>
__device__ __forceinline__ eu_q eu_at(const S &s, int i)
{
    eu_q q;
    q.r = s[i];
    q.m = s[i + VARS];
    q.n = s[i + 2 * VARS];
    q.e = s[i + 3 * VARS];
    return q;
}

/*
 * Division.  n/d is formed as a correctly rounded double division without
 * operand scaling: reciprocal estimate, refinement, product, one residual
 * correction, special-case fix-up.  (Scaling changes nothing unless an operand
 * lies within 2^53 of the subnormal range, d is subnormal or the exponents
 * differ by 768 or more: no Euler state comes near.)  The refined reciprocal
 * depends on d alone, so the quotients that share a denominator share it.
 *
 * How good the reciprocal y has to be: the corrected quotient is the
 * correctly rounded one unless y is the wrong neighbour of 1/d (the farther
 * number) and d = 2^j (1 - k 2^-53) with k 2^-53 at most about 1/d's distance
 * to the midpoint of its neighbours, in units of their distance.  For small
 * odd k the reciprocals lie k^2 2^-54 above a midpoint and have to be rounded
 * up; a uniform stream's densities are such numbers.  eu_recip_from sees to it
 * whatever the estimates.  Of what is cheaper, one third-order step from the
 * hardware's estimate, y + y*(e + e*e), left some quotients one ulp off for k
 * around 2^27 sqrt(m), two Newton steps, as the compiler's n / d takes them,
 * for k = 5, 11 and 13 (the numerators hardest to round, found on MI355X, where
 * n / d itself misses those three).  Against the third-order step the two instructions
 * more cost 1.8 % (Euler 1024^2 53.1 -> 54.1 us a step, standard kernel
 * 1000 x 1500 83.6 -> 85.1).
 */
struct eu_rcp {
    double d, y; /* denominator, refined reciprocal */
};

/* The reciprocal of d from an estimate y of it good to 2^-44.3.  One Newton
 * step leaves 1/d less up to 2^-88.6; the 2^-88 added to the residual puts
 * the value above 1/d instead.  A value 2^-88 too large is the wrong
 * neighbour only of reciprocals less than 2^-36 below a midpoint, and of
 * those there are none with k < 2^17, so no quotient is wrong. */
__device__ __forceinline__ eu_rcp eu_recip_from(double d, double y)
{
    eu_rcp q;
    q.d = d;
    q.y = __builtin_fma(y, __builtin_fma(-d, y, 1.0) + 0x1p-88, y);
    return q;
}

/* The hardware's estimate is good to e = 2^-23, a Newton step makes it e^2. */
__device__ __forceinline__ eu_rcp eu_recip(double d)
{
    const double y = __builtin_amdgcn_rcp(d);
    return eu_recip_from(d, __builtin_fma(y, __builtin_fma(-d, y, 1.0), y));
}

/* 1/d, correctly rounded.  The third-order step leaves a neighbour of 1/d and
 * the residual correction 1/d less 2^-106 at most, on the right side of every
 * midpoint but that of k = 1, where the reciprocal instruction returns the
 * upper neighbour itself (tested at every exponent). */
__device__ __forceinline__ double eu_inverse(double d)
{
    if (EU_EXACT)
        return 1.0 / d;
    double y = __builtin_amdgcn_rcp(d);
    const double e = __builtin_fma(-d, y, 1.0);
    y = __builtin_fma(y, __builtin_fma(e, e, e), y);
    return __builtin_fma(y, __builtin_fma(-d, y, 1.0), y);
}

/* the reciprocal of 2d from that of d: doubling d halves every step of
 * eu_recip exactly */
__device__ __forceinline__ eu_rcp eu_twice(const eu_rcp &q)
{
    eu_rcp h;
    h.d = 2 * q.d;
    h.y = q.y * 0.5;
    return h;
}

__device__ __forceinline__ double eu_quo(double n, const eu_rcp &q)
{
    if (EU_EXACT)
        return n / q.d;
    double z = n * q.y;
    const double rem = __builtin_fma(-q.d, z, n);
    z = __builtin_fma(rem, q.y, z);
    return __builtin_amdgcn_div_fixup(z, q.d, n);
}

/* n/d for a positive normal denominator and operands in the range above:
 * the special-case fix-up of eu_quo then changes nothing, and is left out */
__device__ __forceinline__ double eu_quo_pos(double n, const eu_rcp &q)
{
    if (EU_EXACT)
        return n / q.d;
    const double z = n * q.y;
    const double rem = __builtin_fma(-q.d, z, n);
    return __builtin_fma(rem, q.y, z);
}

/* sqrt(x) as the compiler's IEEE double square root forms it -- reciprocal
 * square-root estimate, Goldschmidt refinement, two residual corrections,
 * x itself for +-0 and +inf -- less the scaling of x < 2^-767, which changes
 * nothing for larger x (densities and Roe sound speeds never come near) */
__device__ __forceinline__ double eu_sqrt(double x)
{
    if (EU_EXACT)
        return sqrt(x);
    const double y = __builtin_amdgcn_rsq(x);
    double g = x * y, h = y * 0.5;
    const double r = __builtin_fma(-h, g, 0.5);
    h = __builtin_fma(h, r, h);
    g = __builtin_fma(g, r, g);
    double d = __builtin_fma(-g, g, x);
    g = __builtin_fma(d, h, g);
    d = __builtin_fma(-g, g, x);
    g = __builtin_fma(d, h, g);
    return (x == 0.0 || x == __builtin_inf()) ? x : g;
}

/* sqrt(x) and the reciprocals of x and (an estimate) of sqrt(x), for a density
 * x in the range above.  The square root is eu_sqrt's without its
 * special cases; its refinement also gives 1/sqrt(x), off by 1.5 e^2 for a
 * hardware estimate good to e <= 2^-23.  Its square is the estimate of 1/x and
 * the product of two that of a Roe density's reciprocal (3 e^2 = 2^-44.4, as
 * eu_recip_from wants it), so a density costs one transcendental instruction (a
 * quarter of the issue rate) instead of two. */
struct eu_root {
    double s, y; /* sqrt(x), estimate of 1/sqrt(x) */
    eu_rcp rx;   /* reciprocal of x */
};

__device__ __forceinline__ eu_root eu_sqrt_recip(double x)
{
    eu_root o;
    if (EU_EXACT) {
        o.s = sqrt(x);
        o.y = 1.0 / o.s;
        o.rx = eu_recip(x);
        return o;
    }
    const double y = __builtin_amdgcn_rsq(x);
    double g = x * y, h = y * 0.5;
    const double r = __builtin_fma(-h, g, 0.5);
    h = __builtin_fma(h, r, h);
    g = __builtin_fma(g, r, g);
    double d = __builtin_fma(-g, g, x);
    g = __builtin_fma(d, h, g);
    d = __builtin_fma(-g, g, x);
    o.s = __builtin_fma(d, h, g);
    o.y = h + h;
    o.rx = eu_recip_from(x, o.y * o.y);
    return o;
}

/* gM1*(E - (m*m + n*n)/(2*rho))  (euler.py:284-293); rr is the reciprocal
 * of rho.  Halving is exact, so the quotient by 2*rho is half the one by rho
 * and its subtraction one fused operation; likewise below wherever a
 * product with 0.5 is added (EU_EXACT keeps the written order: its states
 * may be near the subnormal range, where halving rounds). */
__device__ __forceinline__ double eu_pressure(const eu_q &q, const eu_rcp &rr)
{
    const double k = q.m * q.m + q.n * q.n;
    if (EU_EXACT)
        return GAM_M1 * (q.e - eu_quo(k, eu_twice(rr)));
    return GAM_M1 * __builtin_fma(-0.5, eu_quo_pos(k, rr), q.e);
}

__device__ __forceinline__ double eu_pressure(const eu_q &q)
{
    return eu_pressure(q, eu_recip(q.r));
}

/* min(Pr, 1) with Pr = num/den zeroed when nan, inf, >1e6 or <0
 * (euler.py:250-256).  A zero denominator gives NaN here, which the clamp to
 * [0, 1] turns into 0 as it does negative ratios. */
__device__ __forceinline__ double eu_ratio(double num, const eu_rcp &den)
{
    if (EU_EXACT) {
        const double pr = eu_quo(num, den);
        if (isnan(pr) || isinf(pr) || pr > 1e6 || pr < 0) return 0.0;
        return 1.0 < pr ? 1.0 : pr;
    }
    const double pr = eu_quo_pos(num, den);
    const double c = __builtin_fmin(__builtin_fmax(pr, 0.0), 1.0);
    /* above 1e6 c is 1.0, whose low word is zero: only the high word changes */
    const long long b = __double_as_longlong(c);
    const int hi = pr > 1e6 ? 0 : (int)(b >> 32);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)b);
}

/* q + c/2*d and q - c/2*d (the limited states of a face's two sides: d is
 * the difference of its cells, the same for both) */
__device__ __forceinline__ double eu_add_half(double q, double c, double d)
{
    return EU_EXACT ? q + c / 2 * d : __builtin_fma(0.5, c * d, q);
}

__device__ __forceinline__ double eu_sub_half(double q, double c, double d)
{
    return EU_EXACT ? q + c / 2 * -d : __builtin_fma(-0.5, c * d, q);
}

/* one side's part of a face's central flux, along the first (XDIR) or second
 * momentum: a = m*m/rho, p the pressure, c = m*n/rho, e = (E+p)*m/rho */
struct eu_side {
    double a, p, c, e;
};

template <bool XDIR>
__device__ __forceinline__ eu_side eu_flux_side(const eu_q &q, const eu_rcp &rr)
{
    eu_side o;
    const double m = XDIR ? q.m : q.n;
    o.p = eu_pressure(q, rr);
    o.a = eu_quo_pos(m * m, rr);
    o.c = eu_quo_pos(q.m * q.n, rr);
    o.e = eu_quo_pos((q.e + o.p) * m, rr);
    return o;
}

/* Flux f and dissipation d of the face between cells a (low) and b (high),
 * cl and cr the limiter's ratios of its two sides (eu_ratio):
 * states q1 + min(Pr,1)/2*(q2-q1) (euler.py:250-256), central flux in x
 * (euler.py:181-197) or y (225-241), and the spectral radius of the Roe
 * average, zeroed when nan, times (L - R) (euler.py:258-282).
 * Bound by FP64 issue: about 200 instructions, four of them transcendental
 * (three square-root estimates and 1/(sl + sr); the reciprocals of the L, R
 * and Roe densities come from their roots), for 17 quotients.  Against
 * reciprocal instructions for every denominator, separate limiter differences per side and halvings as operations of their
 * own, a band-kernel cell and stage went from 605 to 482 VALU instructions
 * (488 with eu_recip's last step as it is now): Euler 1024^2 72.2 -> 57.2 us a
 * step, 2048^2 FP32 state 223 -> 175, standard kernel 1000 x 1500 108 -> 92.6,
 * bitwise equal. */
template <bool XDIR>
__device__ __forceinline__ void eu_face_vals(const eu_q &a, const eu_q &b, double cl, double cr, eu_q &f, eu_q &d)
{
    eu_q L, R;
    {
        const double dr = b.r - a.r, dm = b.m - a.m, dn = b.n - a.n, de = b.e - a.e;
        L.r = eu_add_half(a.r, cl, dr); R.r = eu_sub_half(b.r, cr, dr);
        L.m = eu_add_half(a.m, cl, dm); R.m = eu_sub_half(b.m, cr, dm);
        L.n = eu_add_half(a.n, cl, dn); R.n = eu_sub_half(b.n, cr, dn);
        L.e = eu_add_half(a.e, cl, de); R.e = eu_sub_half(b.e, cr, de);
    }
    const eu_root wl = eu_sqrt_recip(L.r), wr = eu_sqrt_recip(R.r);
    const eu_rcp &rl = wl.rx, &rr = wr.rx;
    const eu_side l = eu_flux_side<XDIR>(L, rl), r = eu_flux_side<XDIR>(R, rr);
    f.r = XDIR ? L.m + R.m : L.n + R.n;
    (XDIR ? f.m : f.n) = l.a + l.p + r.a + r.p;
    (XDIR ? f.n : f.m) = l.c + r.c;
    f.e = l.e + r.e;
    const double sl = wl.s, sr = wr.s;
    const double den = eu_inverse(sl + sr);
    const double a0 = sl * sr;
    const double a1 = (sl * eu_quo_pos(L.m, rl) + sr * eu_quo_pos(R.m, rr)) * den;
    const double a2 = (sl * eu_quo_pos(L.n, rl) + sr * eu_quo_pos(R.n, rr)) * den;
    const double a3 = (sl * eu_quo_pos(L.e, rl) + sr * eu_quo_pos(R.e, rr)) * den;
    eu_q roe;
    roe.r = a0;
    roe.m = a0 * a1;
    roe.n = a0 * a2;
    roe.e = a0 * a3;
    const eu_rcp ra = eu_recip_from(a0, wl.y * wr.y);
    /* a negative Roe pressure gives NaN, of which fmax takes the 0 */
    const double rad =
        __builtin_fmax(eu_sqrt(eu_quo_pos(GAMMA * eu_pressure(roe, ra), ra)) + fabs(XDIR ? a1 : a2), 0.0);
    d.r = rad * (L.r - R.r);
    d.m = rad * (L.m - R.m);
    d.n = rad * (L.n - R.n);
    d.e = rad * (L.e - R.e);
}

/* b + h*(ax*0.5*dt/dx + ay*0.5*dt/dy), the update of one variable from its
 * two flux sums; h is 1 (final stage) or 0.5 */
template <bool FINAL>
__device__ __forceinline__ double eu_update(double b, double ax, double ay)
{
    if (EU_EXACT) {
        const double s = ax * 0.5 * DTDX + ay * 0.5 * DTDY;
        return FINAL ? b + s : b + 0.5 * s;
    }
    const double s = ax * (0.5 * DTDX) + ay * (0.5 * DTDY);
    return FINAL ? b + s : __builtin_fma(0.5, s, b);
}

template <bool FINAL>
__device__ __forceinline__ eu_q eu_update(const eu_q &b, const eu_q &ax, const eu_q &ay)
{
    eu_q o;
    o.r = eu_update<FINAL>(b.r, ax.r, ay.r);
    o.m = eu_update<FINAL>(b.m, ax.m, ay.m);
    o.n = eu_update<FINAL>(b.n, ax.n, ay.n);
    o.e = eu_update<FINAL>(b.e, ax.e, ay.e);
    return o;
}

/* flux + dissipation of the face on a cell's low side, less those of the
 * face on its high side in turn: (fa + da) - fb - db */
__device__ __forceinline__ eu_q eu_sum(const eu_q &f, const eu_q &d)
{
    eu_q o;
    o.r = f.r + d.r; o.m = f.m + d.m; o.n = f.n + d.n; o.e = f.e + d.e;
    return o;
}

__device__ __forceinline__ eu_q eu_less(const eu_q &a, const eu_q &f, const eu_q &d)
{
    eu_q o;
    o.r = a.r - f.r - d.r; o.m = a.m - f.m - d.m; o.n = a.n - f.n - d.n; o.e = a.e - f.e - d.e;
    return o;
}

/* flux difference along one direction (euler.py:158-179, 202-223): the
 * west face's flux and dissipation added, the east face's subtracted (the
 * factor 0.5 is in eu_update) */
template <bool XDIR, class S>
__device__ __forceinline__ eu_q eu_divergence(const S *s, int idx, int stride)
{
    const eu_q ww = eu_at(s, idx - 2 * stride), w = eu_at(s, idx - stride), c = eu_at(s, idx);
    const eu_q e = eu_at(s, idx + stride), ee = eu_at(s, idx + 2 * stride);
    const double pww = eu_pressure(ww), pw = eu_pressure(w), pc = eu_pressure(c);
    const double pe = eu_pressure(e), pee = eu_pressure(ee);
    eu_range_check(ww.r, ww.m, ww.n, ww.e, pww);
    eu_range_check(w.r, w.m, w.n, w.e, pw);
    eu_range_check(c.r, c.m, c.n, c.e, pc);
    eu_range_check(e.r, e.m, e.n, e.e, pe);
    eu_range_check(ee.r, ee.m, ee.n, ee.e, pee);
    const double dw = pc - pw, de = pe - pc;
    const eu_rcp yw = eu_recip(dw), ye = eu_recip(de);
    eu_q f, d;
    eu_face_vals<XDIR>(w, c, eu_ratio(dw, eu_recip(pw - pww)), eu_ratio(dw, ye), f, d);
    const eu_q acc = eu_sum(f, d);
    eu_face_vals<XDIR>(c, e, eu_ratio(de, yw), eu_ratio(de, eu_recip(pee - pe)), f, d);
    return eu_less(acc, f, d);
}

/* midpoint RK2 (euler.py:131-151): final stages (even globalTimeStep) start
 * from the level one back with the full step, intermediate stages from the
 * current level with half a step.  Arithmetic in double; R is the storage
 * type of the state. */
template <class R>
__device__ __forceinline__ void eu_step(R *shared_state, int idx, int globalTimeStep)
{
    const eu_q fx = eu_divergence<true>(shared_state, idx, SY);
    const eu_q fy = eu_divergence<false>(shared_state, idx, 1);
    R *out = shared_state + idx + TIMES;
    const bool fin = globalTimeStep % 2 == 0;
    const eu_q b = eu_at(shared_state, fin ? idx - TIMES : idx);
    const eu_q v = fin ? eu_update<true>(b, fx, fy) : eu_update<false>(b, fx, fy);
    out[0] = (R)v.r;
    out[VARS] = (R)v.m;
    out[2 * VARS] = (R)v.n;
    out[3 * VARS] = (R)v.e;
}

__device__ void step(double *shared_state, int idx, int globalTimeStep)
{
    eu_step(shared_state, idx, globalTimeStep);
}

/*
 * Optional cooperative level update used by the pysweep_amd kernels when a
 * plugin defines PS_HAS_LEVEL: all lanes of a workgroup evaluate one level
 * of a rectangle of cells S = [x0,x1) x [y0,y1) together.  Each cell's
 * pressure and each face's limited states, flux and dissipation are
 * computed once (the per-cell step evaluates every face from both sides and
 * ten pressures per cell) and shared through LDS; the sums are formed in the
 * per-cell step's order from the same helper functions, so the results are
 * bitwise those of step().
 *
 *   cur    level r-1 in LDS, variable v of cell (x, y) at
 *          cur[v*VARS + x*SY + y];
 *   prev   level r-2 (the base of a final stage), indexed like cur
 *          (prev[v*VARS + x*SY + y]) and read only at the cells of S, by
 *          the lane computing the cell, before that lane writes it: an LDS
 *          slot in the swept kernels, an accessor of the ring in HBM in the
 *          standard kernel;
 *   out    level r in LDS with cur's strides (a slot of its own, so the
 *          caller may keep its window circular; it may be prev's slot), or
 *          null when only emit needs the values;
 *   sc     scratch of PS_LEVEL_SCRATCH(SX * SY, PS_MAXFACES) doubles,
 *          PS_MAXFACES being the most faces of one direction of any
 *          rectangle the harness passes ((x1-x0+1)*(y1-y0) or
 *          (x1-x0)*(y1-y0+1)); the face buffer is component-major so that
 *          consecutive lanes touch consecutive LDS words;
 *   MAXC   upper bound of cells per lane, ceil(|S| / PS_NT);
 *   emit   called as emit(x, y, v) with the tile coordinates and the NV new
 *          values of every cell of S, by the lane that computed it (the
 *          kernels write the cell to HBM from there, without re-reading
 *          LDS).
 */
#define PS_HAS_LEVEL 1
#define PS_LEVEL_SCRATCH(CELLS, FACES) ((CELLS) + 8 * (FACES))
/* prev is read only at the cell being written, by the lane writing it, so
 * out may be prev's own slot (a swept window of ITS levels suffices) */
#define PS_LEVEL_INPLACE 1

/* 1/w for w >= 1 within one ulp: the hardware reciprocal (one instruction
 * where a correctly rounded float division takes ten) */
__device__ __forceinline__ float eu_rcpf(int w) { return __builtin_amdgcn_rcpf((float)w); }

/* t / w for 0 <= t < 2^22, w >= 1, rw within one ulp of 1/w (the hardware
 * reciprocal, eu_rcpf): the float quotient is within one of the true one;
 * one correction makes it exact.  A width known at compile time (the
 * standard tile, unrolled swept levels) divides by the constant instead
 * (measured: Euler 1024^2 Octahedron 88.2 -> 86.0 us, Standard -3 %). */
__device__ __forceinline__ int eu_div(int t, int w, float rw)
{
    if (__builtin_constant_p(w))
        return t / w;
    int q = (int)((float)t * rw);
    const int r = t - q * w;
    if (r < 0)
        q -= 1;
    else if (r >= w)
        q += 1;
    return q;
}

/* exchange the two momentum components */
__device__ __forceinline__ void eu_swap(eu_q &q)
{
    const double t = q.m;
    q.m = q.n;
    q.n = t;
}

/* One face of a level update between the cells at idx - stride and idx:
 * flux in components 0-3 and dissipation in 4-7 of o (component stride
 * PS_MAXFACES), P holding the cells' pressures.  A y face (stride 1) is
 * evaluated as an x face with the momentum components exchanged in its
 * states and exchanged back in its results; the only operations that then
 * run in another order are commutative (m*n as n*m, m*m + n*n as
 * n*n + m*m), so the values are bitwise those of eu_face_vals<false>, and x
 * and y faces share one instruction stream. */
template <class R>
__device__ __forceinline__ void eu_face(const R *cur, const double *P, double *o, int idx, int stride, bool ydir)
{
    constexpr int FS = PS_MAXFACES;
    eu_q wq = eu_at(cur, idx - stride), c = eu_at(cur, idx);
    const double pww = P[idx - 2 * stride], pw = P[idx - stride], pc = P[idx], pe = P[idx + stride];
    if (ydir) {
        eu_swap(wq);
        eu_swap(c);
    }
    eu_q f, d;
    eu_face_vals<true>(wq, c, eu_ratio(pc - pw, eu_recip(pw - pww)), eu_ratio(pc - pw, eu_recip(pe - pc)), f, d);
    if (ydir) {
        eu_swap(f);
        eu_swap(d);
    }
    o[0] = f.r; o[FS] = f.m; o[2 * FS] = f.n; o[3 * FS] = f.e;
    o[4 * FS] = d.r; o[5 * FS] = d.m; o[6 * FS] = d.n; o[7 * FS] = d.e;
}

/* ((flux_a + diss_a) - flux_b) - diss_b per component, face a on the low
 * side of the cell and face b on the high side: the per-cell step's order */
__device__ __forceinline__ eu_q eu_face_diff(const double *fa, const double *fb)
{
    constexpr int FS = PS_MAXFACES;
    eu_q a;
    a.r = fa[0] + fa[4 * FS] - fb[0] - fb[4 * FS];
    a.m = fa[FS] + fa[5 * FS] - fb[FS] - fb[5 * FS];
    a.n = fa[2 * FS] + fa[6 * FS] - fb[2 * FS] - fb[6 * FS];
    a.e = fa[3 * FS] + fa[7 * FS] - fb[3 * FS] - fb[7 * FS];
    return a;
}

template <class R, int MAXC, class Prev, class Emit>
__device__ __forceinline__ void ps_level(const R *cur, const Prev &prev, R *out, int x0, int x1, int y0, int y1,
                                         int globalTimeStep, double *sc, const Emit &emit)
{
    const int h = x1 - x0, w = y1 - y0;
    const float rw = eu_rcpf(w);
    constexpr int FS = PS_MAXFACES;  /* component stride of the face buffer */
    double *P = sc;                  /* pressures, tile-indexed x*SY + y */
    double *F = sc + SX * SY;        /* face f, component c at F[c*FS + f]: flux 0-3, dissipation 4-7 */

    /* 1. pressures on the cross-shaped footprint */
    {
        const int bh = h + 4, bw = w + 4, n = bh * bw;
        const float rbw = eu_rcpf(bw);
        for (int t = threadIdx.x; t < n; t += PS_NT) {
            const int i = eu_div(t, bw, rbw), j = t - i * bw;
            const bool inx = i >= 2 && i < h + 2, iny = j >= 2 && j < w + 2;
            if (!(inx || iny)) continue;
            const int x = x0 - 2 + i, y = y0 - 2 + j;
            const eu_q q = eu_at(cur, x * SY + y);
            const double p = eu_pressure(q);
            P[x * SY + y] = p;
            eu_range_check(q.r, q.m, q.n, q.e, p);
        }
    }
    __syncthreads();

    /* 2. faces.  x face i (0..h) lies west of cell x0+i, at F[i*w + j]; y
     * face j (0..w) lies south of cell y0+j, at Fy[i*(w+1) + j].  When both
     * sets fit the buffer they are evaluated in one pass over one lane space
     * (the small levels then fill whole wavefronts, and the level needs two
     * barriers fewer); otherwise the x divergences are taken first and the
     * y faces overwrite the x faces. */
    const int nfx = (h + 1) * w, nfy = h * (w + 1), wf = w + 1;
    const float rwf = eu_rcpf(wf);
    const bool merged = nfx + nfy <= FS;
    double *Fy = merged ? F + nfx : F;
    {
        const int n = merged ? nfx + nfy : nfx;
        for (int t = threadIdx.x; t < n; t += PS_NT) {
            const bool xf = t < nfx;
            const int u = xf ? t : t - nfx, wd = xf ? w : wf;
            const int i = eu_div(u, wd, xf ? rw : rwf), j = u - i * wd;
            eu_face(cur, P, F + t, (x0 + i) * SY + y0 + j, xf ? SY : 1, !xf);
        }
    }
    __syncthreads();

    eu_q dfx[MAXC];
    if (!merged) {
        /* 3. x divergence of my cells (cell (i, j): west face i, east face i+1) */
#pragma unroll
        for (int m = 0; m < MAXC; ++m) {
            const int t = threadIdx.x + m * PS_NT;
            if (t < h * w) {
                const int i = eu_div(t, w, rw), j = t - i * w;
                dfx[m] = eu_face_diff(F + (i * w + j), F + ((i + 1) * w + j));
            }
        }
        __syncthreads();
        /* 4. y faces over the x faces */
        for (int t = threadIdx.x; t < nfy; t += PS_NT) {
            const int i = eu_div(t, wf, rwf), j = t - i * wf;
            eu_face(cur, P, Fy + t, (x0 + i) * SY + y0 + j, 1, true);
        }
        __syncthreads();
    }

    /* 5. (x and) y divergence and the RK2 update of my cells */
    const bool fin = globalTimeStep % 2 == 0;
#pragma unroll
    for (int m = 0; m < MAXC; ++m) {
        const int t = threadIdx.x + m * PS_NT;
        if (t < h * w) {
            const int i = eu_div(t, w, rw), j = t - i * w;
            const eu_q fx = merged ? eu_face_diff(F + (i * w + j), F + ((i + 1) * w + j)) : dfx[m];
            const double *fs = Fy + (i * wf + j);
            const eu_q a = eu_face_diff(fs, fs + 1);
            const int idx = (x0 + i) * SY + (y0 + j);
            const eu_q b = fin ? eu_at(prev, idx) : eu_at(cur, idx);
            const eu_q u = fin ? eu_update<true>(b, fx, a) : eu_update<false>(b, fx, a);
            const R v[4] = {(R)u.r, (R)u.m, (R)u.n, (R)u.e};
            if (out) {
                R *o = out + idx;
                o[0] = v[0];
                o[VARS] = v[1];
                o[2 * VARS] = v[2];
                o[3 * VARS] = v[3];
            }
            emit(x0 + i, y0 + j, v);
        }
    }
}

#ifdef PS_BAND_COMMON
/*
 * Band sweep (PS_HAS_BAND): the swept solve's kernel with every level of a
 * launch in registers.  One wavefront owns a band of 64 columns, one column
 * per lane, and a segment of rows, and sweeps it along x; a launch of
 * PS_BAND_H = 2 stages (one RK2 step) reads level A over the band and writes
 * level A + 2 over its middle 64 - 4 * PS_BAND_H columns (the radius-2
 * stencil costs two halo columns per level on each side, recomputed by the
 * neighbouring bands instead of exchanged).
 *
 * A segment is sheared along x: the wavefront of rows [a, a + n) computes
 * rows [a + 2, a + n + 2) of level A + 1 and [a + 4, a + n + 4) of level
 * A + 2.  Its first rows then need no halo (level A is in memory), and at its
 * end level A + 2 lacks the first four level A + 1 rows of the segment after
 * it, a + n + 2 .. a + n + 5.  In a chain (PS_HAS_BAND_CHAIN: the wavefronts
 * of one workgroup on consecutive segments of a band) that segment's
 * wavefront computed them at its own start and left them in LDS; the chain's
 * last wavefront, and every wavefront of a launch without chains, computes
 * them itself.  Of the rows a segment recomputed at both ends (two and a
 * face on each side) a chain of four keeps a quarter, which is what small
 * segments are made of: Euler 1024^2 has 19 bands, so that 2048 wavefronts
 * are segments of ten rows.
 *
 * Step tau brings in row a + tau of level A and computes row a + tau - 2 l
 * of level A + l.  Each level keeps the last three rows it produced (states,
 * in the storage type) and their pressure differences: the x face between
 * rows r and r + 1 needs the pressures of rows r - 1 .. r + 2 and the states
 * of r and r + 1.  The x face below a row is the one above the row before,
 * carried from the previous step; the y face east of a column is computed
 * by its lane from the neighbouring lanes' states and pressure differences
 * (DPP), and the west one is the lower lane's east face.  Every face,
 * pressure and update is evaluated by the functions and in the order of
 * ps_level and the per-cell step, so results are bitwise theirs.  Rows and
 * columns that a level cannot yet compute correctly (first steps, the
 * outermost lanes) hold garbage that no valid cell ever reads; only valid
 * cells are range-checked and stored.  Launches start on full steps (the
 * first stage of a launch never reads the level two back).
 */
#define PS_HAS_BAND 1
#define PS_HAS_BAND_CHAIN 1
/* fewest rows of a chain's wavefronts (the rows left in LDS at steps 4..7 are
 * read from step n + 4 on, after the barrier behind step 8), and the rows the
 * last one takes less for computing four level-1 rows more */
#define PS_BAND_MIN_ROWS 5
#define PS_BAND_LAST_LESS 2
/* two wavefronts per SIMD (256 VGPRs): left to itself the compiler takes more
 * registers and one wavefront */
#define PS_BAND_OCC __attribute__((amdgpu_waves_per_eu(2)))
#define EU_BAND_WOUT (64 - 4 * PS_BAND_H)
static_assert(EU_BAND_WOUT >= 8, "PS_BAND_H too deep for a 64-column band");

__device__ __forceinline__ eu_rcp eu_lower(const eu_rcp &q)
{
    eu_rcp o;
    o.d = ps_from_lower(q.d); o.y = ps_from_lower(q.y);
    return o;
}

__device__ __forceinline__ eu_rcp eu_upper(const eu_rcp &q)
{
    eu_rcp o;
    o.d = ps_from_upper(q.d); o.y = ps_from_upper(q.y);
    return o;
}

__device__ __forceinline__ eu_q eu_lower(const eu_q &q)
{
    eu_q o;
    o.r = ps_from_lower(q.r); o.m = ps_from_lower(q.m); o.n = ps_from_lower(q.n); o.e = ps_from_lower(q.e);
    return o;
}

__device__ __forceinline__ eu_q eu_upper(const eu_q &q)
{
    eu_q o;
    o.r = ps_from_upper(q.r); o.m = ps_from_upper(q.m); o.n = ps_from_upper(q.n); o.e = ps_from_upper(q.e);
    return o;
}

template <class R>
struct eu_band_row {
    R v[4];
    __device__ __forceinline__ eu_q q() const
    {
        eu_q o;
        o.r = (double)v[0]; o.m = (double)v[1]; o.n = (double)v[2]; o.e = (double)v[3];
        return o;
    }
};

/* The last three rows a level produced (slot tau % 3 holds the newest, so
 * nothing moves between steps), the newest one's pressure, and each row's
 * pressure difference to the row before it with the reciprocal of that
 * difference: the x face (r | r+1) takes p(r+1) - p(r) over p(r) - p(r-1)
 * and over p(r+2) - p(r+1), so each difference divides twice, two steps
 * apart, and its reciprocal is formed once. */
template <class R>
struct eu_band_win {
    eu_band_row<R> q[3];
    double p[3];
    eu_rcp dp[3];
};

/* Division range of the cells a wavefront met: the extremes of the high
 * words of rho, E and p (as unsigned integers those of positive numbers are
 * in the numbers' order, and negative numbers and NaN lie above them all),
 * and whether a momentum left its range.  The fault flag is written once
 * per wavefront, after the sweep, so the steps hold no branch. */
struct eu_band_range {
    unsigned lo, hi;
    bool mom;
    __device__ __forceinline__ void take(const eu_q &q, double p)
    {
        const unsigned r = (unsigned)(__double_as_longlong(q.r) >> 32);
        const unsigned e = (unsigned)(__double_as_longlong(q.e) >> 32);
        const unsigned k = (unsigned)(__double_as_longlong(p) >> 32);
        lo = min(min(lo, r), min(e, k));
        hi = max(max(hi, r), max(e, k));
        mom |= !(eu_mom_in_range(q.m) & eu_mom_in_range(q.n));
    }
    /* 2^-120 has the high word 0x38700000 and 2^120 0x47700000, both with
     * low word zero; a value in [2^120, 2^120 (1 + 2^-20)) counts as out */
    __device__ __forceinline__ bool fault() const { return mom | (lo < 0x38700000u) | (hi >= 0x47700000u); }
};

template <int PH, class R>
__device__ __forceinline__ void eu_band_push(eu_band_win<R> &w, const eu_band_row<R> &row, bool check,
                                             eu_band_range &rng)
{
    const eu_q q = row.q();
    const double p = eu_pressure(q);
    w.q[PH] = row;
    w.dp[PH] = eu_recip(p - w.p[(PH + 2) % 3]);
    w.p[PH] = p;
    if (check) rng.take(q, p);
}

/* Row r of level l from level l-1's window at step phase PH (its newest
 * row, slot PH, is r + 2): the x face (r | r+1), the y faces of row r, the
 * divergences with the x face below (xc, its flux + dissipation, replaced
 * by the new one's) and the RK2 update from base (the cell itself, or for a
 * final stage the cell two levels back).  A lane forms the pressure
 * difference across its east y face and that difference's reciprocal once
 * and takes its neighbours' for the two limiter ratios. */
template <int PH, bool FINAL, class R>
__device__ __forceinline__ eu_band_row<R> eu_band_cell(const eu_band_win<R> &w, eu_q &xc, const eu_q &base2)
{
    constexpr int pa = (PH + 1) % 3, pb = (PH + 2) % 3;  /* rows r, r + 1 */
    const eu_q a = w.q[pa].q(), b = w.q[pb].q();
    eu_q f, d;
    eu_face_vals<true>(a, b, eu_ratio(w.dp[pb].d, w.dp[pa]), eu_ratio(w.dp[pb].d, w.dp[PH]), f, d);
    const eu_q ax = eu_less(xc, f, d);
    xc = eu_sum(f, d);
    const double pr = w.p[pa];
    const eu_rcp dy = eu_recip(ps_from_upper(pr) - pr);
    eu_face_vals<false>(a, eu_upper(a), eu_ratio(dy.d, eu_lower(dy)), eu_ratio(dy.d, eu_upper(dy)), f, d);
    const eu_q ay = eu_less(eu_lower(eu_sum(f, d)), f, d);
    const eu_q v = eu_update<FINAL>(FINAL ? base2 : a, ax, ay);
    eu_band_row<R> o;
    o.v[0] = (R)v.r;
    o.v[1] = (R)v.m;
    o.v[2] = (R)v.n;
    o.v[3] = (R)v.e;
    return o;
}

/* the x face (r | r+1) alone: the one below a segment's first row */
template <int PH, class R>
__device__ __forceinline__ void eu_band_xface(const eu_band_win<R> &w, eu_q &xc)
{
    constexpr int pa = (PH + 1) % 3, pb = (PH + 2) % 3;
    eu_q f, d;
    eu_face_vals<true>(w.q[pa].q(), w.q[pb].q(), eu_ratio(w.dp[pb].d, w.dp[pa]), eu_ratio(w.dp[pb].d, w.dp[PH]), f,
                       d);
    xc = eu_sum(f, d);
}

#define EU_GLOBAL __attribute__((address_space(1)))

/* byte offset of a column */
#ifdef PS_BAND_WIDE
typedef size_t eu_band_off;
#else
typedef unsigned eu_band_off;
#endif

template <class R>
struct eu_band_ctx {
    /* the ring in the global address space: its accesses compile to global
     * loads and stores also where the pointer was read from memory (an
     * instance table), whose address space the compiler cannot infer */
    EU_GLOBAL R *state;
    const EU_GLOBAL R *in;  /* level A */
    size_t cells;
    int s0, T, nx, ny, wlo, hh;
    int n, e1;         /* rows of the segment; level 1 is computed until step e1 */
    eu_band_off col, oc;  /* this lane's column in bytes; the same unwrapped */
    bool out_col;
};

/* Rows are the same in every lane, so a row's address is scalar and a
 * lane's column a 32-bit offset that the load or store adds by itself.  The
 * empty asm statements keep it so: the compiler would carry the column as a
 * 64-bit number around the loop and add every row to it in vector
 * instructions, 6 a cell. */
__device__ __forceinline__ eu_band_off eu_band_lane(eu_band_off bytes)
{
    eu_band_off o;
    asm volatile("" : "=v"(o) : "0"(bytes));
    return o;
}

template <class T>
__device__ __forceinline__ T *eu_band_at(T *row, eu_band_off bytes)
{
    typedef EU_GLOBAL char B;
    asm("" : "+s"(row));
    return (T *)((B *)(row) + bytes);
}

template <class R>
__device__ __forceinline__ void eu_band_load(const eu_band_ctx<R> &c, int row, eu_band_row<R> &o)
{
    const eu_band_off col = eu_band_lane(c.col);
#pragma unroll
    for (int v = 0; v < 4; ++v) o.v[v] = *eu_band_at(c.in + (v * c.cells + (size_t)row * c.ny), col);
}

template <class R>
__device__ __forceinline__ void eu_band_store(const eu_band_ctx<R> &c, int l, int row, const eu_band_row<R> &o)
{
    const int slot = c.s0 + l >= c.T ? c.s0 + l - c.T : c.s0 + l;
    if (c.out_col) {
        const eu_band_off col = eu_band_lane(c.oc);
#pragma unroll
        for (int v = 0; v < 4; ++v)
            *eu_band_at(c.state + (((size_t)slot * NV + v) * c.cells + (size_t)row * c.ny), col) = o.v[v];
    }
}

/* wrap a row index into [0, nx) (rows stay within one period of the grid
 * around the segment only when nx exceeds the halo, so reduce fully) */
__device__ __forceinline__ int eu_band_wrap(int r, int nx)
{
    r %= nx;
    return r < 0 ? r + nx : r;
}

__device__ __forceinline__ int eu_band_next(int r, int nx) { return r + 1 == nx ? 0 : r + 1; }

/* rows a level reads, loads and stores next (wrapped) */
struct eu_band_rows {
    int load;   /* level A, three steps ahead             */
    int out1;   /* level A + 1's row of this step          */
    int out2;   /* level A + 2's, and its base in level A  */
};

/* One step (phase PH = tau % 3) of a one-step (two-stage) launch.  FULL: a
 * step of the steady state of a two-level launch that writes level 2 only
 * (both levels valid; no test), so that the compiler may interleave the two
 * levels' independent work.  pub: where this wavefront leaves its first four
 * level-1 rows (or null); nxt: where the next segment's lie (or null). */
template <int PH, bool FULL, class R>
__device__ __forceinline__ void eu_band_step(const eu_band_ctx<R> &c, int tau, eu_band_win<R> &w0,
                                             eu_band_win<R> &w1, eu_q (&xc)[2], eu_band_row<R> (&pf)[3],
                                             eu_band_rows &r, eu_band_range &rng, R *pub, const R *nxt)
{
    const int lane = threadIdx.x & 63;
    /* the base of the final stage: level A two rows behind level 1's row,
     * re-read (this wavefront loaded it four steps ago) */
    eu_band_row<R> b2;
    const bool two = FULL || (c.hh >= 2 && tau >= 8 && tau < c.n + 8);
    if (FULL || tau < c.e1) {
        /* level A: this step's row (loaded three steps ago) */
        const eu_band_row<R> in = pf[PH];
        eu_band_load(c, r.load, pf[PH]);
        r.load = eu_band_next(r.load, c.nx);
        if (two) eu_band_load(c, r.out2, b2);
        eu_band_push<PH>(w0, in, true, rng);
        if (!FULL && PH == 0 && tau == 3) {  /* the face below the segment's first row */
            eu_band_xface<PH>(w0, xc[0]);
        } else if (FULL || tau >= 4) {
            /* level 1 (a half stage) */
            const eu_band_row<R> v1 = eu_band_cell<PH, false>(w0, xc[0], eu_q());
            eu_band_push<PH>(w1, v1, true, rng);
            if (!FULL) {
                if (pub && tau < 8)
#pragma unroll
                    for (int v = 0; v < 4; ++v) pub[((tau - 4) * 4 + v) * 64 + lane] = v1.v[v];
                if (c.wlo <= 1 && tau < c.n + 4) eu_band_store(c, 1, r.out1, v1);
            }
        }
    } else {
        if (two) eu_band_load(c, r.out2, b2);
        if (nxt && tau < c.n + 8) {
            eu_band_row<R> v1;
#pragma unroll
            for (int v = 0; v < 4; ++v) v1.v[v] = nxt[((tau - c.n - 4) * 4 + v) * 64 + lane];
            eu_band_push<PH>(w1, v1, false, rng);
        }
    }
    /* level 2 (the final stage) */
    if (!FULL && PH == 1 && tau == 7) {
        eu_band_xface<PH>(w1, xc[1]);
    } else if (two) {
        const eu_band_row<R> v2 = eu_band_cell<PH, true>(w1, xc[1], b2.q());
        eu_band_store(c, 2, r.out2, v2);
    }
    r.out1 = eu_band_next(r.out1, c.nx);
    r.out2 = eu_band_next(r.out2, c.nx);
}

/* The segment of rows [a, a + n) of band `band`; CHAIN: the workgroup's
 * wavefronts are a chain and meet at one barrier (every wavefront of the
 * workgroup passes it). */
template <bool CHAIN, class R>
__device__ __forceinline__ void eu_band_segment(R *state, int A, const ps_band_grid &g, int band, int a, int n,
                                                R *pub, const R *nxt)
{
    static_assert(PS_BAND_H == 2, "the Euler band sweep takes one RK2 step (two stages) per launch");
    constexpr int WOUT = EU_BAND_WOUT;
    const int lane = threadIdx.x & 63;
    eu_band_ctx<R> c;
    c.state = (EU_GLOBAL R *)state;  /* device memory */
    c.cells = (size_t)g.nx * g.ny;
    c.s0 = A % g.T;
    c.T = g.T;
    c.nx = g.nx;
    c.ny = g.ny;
    c.in = c.state + (size_t)c.s0 * NV * c.cells;
    c.hh = g.hh;
    c.wlo = g.wlo;
    c.n = n;
    c.e1 = n + (g.hh >= 2 && !nxt ? 8 : 4);
    const int o = lane - 2 * PS_BAND_H;  /* band-local output column */
    c.out_col = o >= 0 && o < WOUT && band * WOUT + o < g.ny;
    c.oc = (eu_band_off)(band * WOUT + o) * (eu_band_off)sizeof(R);
    c.col = (eu_band_off)eu_band_wrap(band * WOUT + o, g.ny) * (eu_band_off)sizeof(R);
    /* defined values in what the first steps read before any level has
     * produced it (never used by a valid cell) */
    eu_band_win<R> w0, w1;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
#pragma unroll
        for (int v = 0; v < 4; ++v) w0.q[k].v[v] = w1.q[k].v[v] = (R)0;
        w0.p[k] = w1.p[k] = 0.0;
        w0.dp[k].d = w1.dp[k].d = w0.dp[k].y = w1.dp[k].y = 0.0;
    }
    eu_q xc[2];
#pragma unroll
    for (int l = 0; l < 2; ++l) xc[l].r = xc[l].m = xc[l].n = xc[l].e = 0.0;
    eu_band_rows r;
    r.load = eu_band_wrap(a, g.nx);
    r.out1 = eu_band_wrap(a - 2, g.nx);
    r.out2 = eu_band_wrap(a - 4, g.nx);
    eu_band_row<R> pf[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        eu_band_load(c, r.load, pf[k]);
        r.load = eu_band_next(r.load, g.nx);
    }
    const int steps = n + (g.hh >= 2 ? 8 : 4);
    const int full = g.hh == 2 && g.wlo == 2 ? min(c.e1, n + 8) : 0;  /* end of the steady state */
    eu_band_range rng = {~0u, 0u, false};
    int tau = 0;
    for (; tau < 9 || (tau < steps && full == 0); tau += 3) {
        eu_band_step<0, false>(c, tau, w0, w1, xc, pf, r, rng, pub, nxt);
        eu_band_step<1, false>(c, tau + 1, w0, w1, xc, pf, r, rng, pub, nxt);
        eu_band_step<2, false>(c, tau + 2, w0, w1, xc, pf, r, rng, pub, nxt);
        if (CHAIN && tau == 6) __syncthreads();
    }
    for (; tau + 3 <= full; tau += 3) {
        eu_band_step<0, true>(c, tau, w0, w1, xc, pf, r, rng, pub, nxt);
        eu_band_step<1, true>(c, tau + 1, w0, w1, xc, pf, r, rng, pub, nxt);
        eu_band_step<2, true>(c, tau + 2, w0, w1, xc, pf, r, rng, pub, nxt);
    }
    for (; tau < steps; tau += 3) {
        eu_band_step<0, false>(c, tau, w0, w1, xc, pf, r, rng, pub, nxt);
        eu_band_step<1, false>(c, tau + 1, w0, w1, xc, pf, r, rng, pub, nxt);
        eu_band_step<2, false>(c, tau + 2, w0, w1, xc, pf, r, rng, pub, nxt);
    }
    /* a vector store (a benign race: every writer writes 1).  Level 1 is
     * valid in lanes 2..61, and what the outer lanes saw of level A is also
     * seen by the neighbouring bands' inner lanes. */
    if (rng.fault() && lane >= 2 && lane < 62) *(volatile int *)&EU_RANGE_FAULT = 1;
}

/* one wavefront's segment by itself */
template <class R>
__device__ __forceinline__ void ps_band_sweep(R *state, int gts0, int A, const ps_band_grid &g, int band, int seg)
{
    (void)gts0;  /* launches start on full steps: level 1 is a half stage, level 2 a final one */
    const int a = seg * g.rows;
    eu_band_segment<false>(state, A, g, band, a, min(g.rows, g.nx - a), static_cast<R *>(nullptr),
                           static_cast<const R *>(nullptr));
}

/* rows that a chain's wavefronts leave for the one before (PS_BAND_CHAIN
 * wavefronts: each but the first leaves 4 rows of 4 variables) */
#define PS_BAND_CHAIN_WORDS (4 * 4 * 64)

/* wavefront k of a chain: rows [a, a + n), `last` if no wavefront follows */
template <class R>
__device__ __forceinline__ void ps_band_sweep_chain(R *state, int gts0, int A, const ps_band_grid &g, int band,
                                                    int a, int n, R *pub, const R *nxt)
{
    (void)gts0;
    eu_band_segment<true>(state, A, g, band, a, n, pub, nxt);
}
#endif /* PS_BAND_COMMON */
