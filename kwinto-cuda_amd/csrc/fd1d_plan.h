// fd1d_plan.h -- which rows of an option's grid its FD march has to carry.
//
// The mesh spans +-scale sigma sqrt(T) around the strike (50 standard deviations by
// default), and most of its rows have a solution that is known beforehand:
//   * out of the money, beyond a few standard deviations, it is 0: truncating it at
//     distance b from the strike changes the price at a spot by the share of paths that
//     reach b and come back to the payoff, exp(-2 b (b - x*) / (sigma^2 T)) of the price
//     by the reflection principle, whatever the drift (a bridge does not see it);
//   * in the money, past the exercise boundary b(T), every step ends projected onto the
//     payoff, so those rows are constant in time. b(tau) moves away from the strike as tau
//     grows, so rows past b(T) are pinned at every step.
// Rows are counted as positions from the in-the-money edge of the mesh: position i is row
// i of a put's grid and row N - 1 - i of a call's, and xi = log(S/K) for a put, -log(S/K)
// for a call grows with the position. In xi a call is a put with the drift reversed.
//
// The window [lo, end) found here is an estimate of where both start to hold, with
// margins; the march checks the in-the-money cut after its last step and an option whose
// boundary went past it is solved again on its whole grid. Options outside the rule's
// domain keep their whole grid (lo = 0, end = N).
//
// Host and device code; only the C library's mathematics, so that it can be checked on
// the CPU.
#pragma once

#include <math.h>

#include "kwgpu.h"

#ifndef KWGPU_HD
#define KWGPU_HD __host__ __device__ inline
#endif

namespace kwgpu {

struct Window {
    int lo, end;  // positions; lo > 0: the rows before it are pinned to the payoff
};

// Positions of pinned rows eliminated in front of the window in set-up (fd1d_window.h).
constexpr int kPinnedRows = 256;
constexpr int kWindowMinSteps = 64;

// log of the critical spot of an American put with unit strike, rate r > 0 and yield q, in
// Barone-Adesi & Whaley's approximation: the root of
//     f(S) = (1 - S) - E(S) + (1 - e^{-qT} Phi(-d1(S))) S / lambda,
// E the European put. With m2 = 1 - e^{-rT} Phi(-d2) and n1 = 1 - e^{-qT} Phi(-d1) it is that of
//     log m2 - log n1 = x + log(1 - 1 / lambda),   x = log S,
// where nothing cancels at small rates, whose root lies up to five standard deviations from the
// strike. Convex and falling on the root's left, so three Newton steps from a start that lies
// mostly there: to 0.005 sigma sqrt(T) in 99 of 100 options of vol 2-200 %, T 0.005-20 years
// and rates down to 1e-6. (Newton steps in S from the starting value of their paper were off
// by more than 0.5 at a tenth of the rates below 1 %; with the margin of then nearly every cut was
// passed at rates under 1e-4 and half of them under 1e-3: 8192 options of vol 80-150 % and
// rates under 1e-4 at 512 x 512 took 1891 us, on whole grids 685, and so 628.) In FP32: the
// result only places a cut that is checked afterwards. No number where n1 is not positive, as
// it can be at q < 0.
KWGPU_HD float critical_log_spot(float t, float z, float r, float q) {
    const float z2 = z * z, rt = sqrtf(t), st = z * rt, n = 2.0f * (r - q) / z2 - 1.0f;
    const float er1 = -expm1f(-r * t), eq1 = -expm1f(-q * t), er = 1.0f - er1, eq = 1.0f - eq1;
    const float lam = 0.5f * (-n - sqrtf(n * n + 8.0f * r / (z2 * er1)));
    const float perp = 0.5f * (-n - sqrtf(n * n + 8.0f * r / z2));
    const float c = logf(1.0f - 1.0f / lam), drift = (r - q + 0.5f * z2) * t;
    const float top = q > r ? logf(r / q) : 0.0f, gain = q < 0.0f ? r - q : r;
    float x = fmaxf(logf(perp / (perp - 1.0f)), top - st * sqrtf(2.0f * logf(1.0f + 0.3f * z / (gain * rt))));
    for (int it = 0; it < 3; ++it) {
        const float d1 = (x + drift) / st, d2 = d1 - st;
        const float n1 = eq1 + 0.5f * eq * erfcf(-d1 * 0.70710678f);
        const float m2 = er1 + 0.5f * er * erfcf(-d2 * 0.70710678f);
        if (!(n1 > 0.0f)) return NAN;
        const float f = logf(m2 / n1) - x - c;
        const float df = 0.39894228f * (er * expf(-0.5f * d2 * d2) / m2 - eq * expf(-0.5f * d1 * d1) / n1) / st - 1.0f;
        x = fminf(fmaxf(x - f / df, x - 0.7f * st), top);
    }
    return x;
}

// The window of option o on an N-point grid marched `steps` steps at theta = 1/2. `far`:
// the largest xi at which the option's price is asked for (0 or less: at or in the money).
//
// Out of the money the bound is b (b - far) >= 18 sigma^2 T, i.e. a relative truncation
// error of e^-36 = 2e-16. Where the steps are few Crank-Nicolson's tails are heavier than
// the Gaussian's: at 64 steps the exponent 36 loses 2 n (y^3/3 + ...), y = 36 / (2 n), 0.9.
//
// In the money the cut lies 0.18 sigma sqrt(T) / (1 + sqrt(a / 6)), a = r sqrt(T) / sigma, in log S
// and 2 rows past the approximate critical spot. The boundary ends past that spot by more the
// smaller a is: over 5000 marches on 2048 points laid close to the strike (vol 0.3-150 %, T 0.001-20
// years, rates 1e-4 to 90 %) by a row and at most 0.16 sigma sqrt(T) at a < 0.01, 0.12 at 0.2, 0.09
// at 2 and 0.02 beyond 10. A cut that is too near costs a second march after the first, which a
// whole launch may wait for (0.5 ms of 2.2 for one option of 16384); the margin costs about 8
// rows of 1024. The cut needs
//   * kPinnedRows rows to forget the approximate value they are started from: with
//     a = theta dt (sigma^2 / 2) / dx^2 at the cut, an error shrinks by about
//     e^{-1/sqrt(a)} per row, and a <= 150 leaves 1e-9 of an error of O(dt^2);
//   * early exercise to be worth something: while q > r the boundary never comes nearer than
//     log(r / q) to the strike, and past 4.5 sigma sqrt(T) the premium is below about 1e-9 of
//     the price. Such an option keeps the rows its European twin keeps, and with them the
//     same arithmetic, so that rounding cannot price it below the twin (on 32768 options at
//     1024 x 1024 the two had differed by up to 9e-11, the smallest such ratio 5.1). At a < 1e-3 the
//     approximation is off by up to 1.3 sigma sqrt(T) from a ratio of 0.5 on;
//   * the rows past it to be pinned in the scheme too: a payoff falls behind there at r (a call's:
//     at r S) less what waiting earns and what the differences are off by. A put's error is largest
//     near the strike; a call's grows with S and dx, and from xc on, where it reaches r / 2, the
//     rows are not pinned and carry more than the payoff;
//   * those rows of a call, and its unprojected edge row, to be forgotten: their values are
//     e^{x - |xb|} of the cut's, a row with a < 0.1 takes off at least a decade, and 20 more leave
//     nothing. (Without these two, 1 of 2500 cuts of calls in a search over long maturities, coarse
//     grids and yields far below the rate held although they should not have: deep in the money
//     prices were off by up to 2 %. With them 277000 cuts of that search and 565000 windows of a
//     wider one on the CPU are at most 3e-15 of max(K, price) from the whole grid, none passed.)
KWGPU_HD Window window_of(const kwgpu_option& o, int N, int steps, double density, double scale,
                          double far) {
    Window w{0, N};
    const double s = o.z * sqrt(o.t), s2 = s * s;
    const double mu = o.r - o.q - 0.5 * o.z * o.z;
    // the domain: a march long enough to pay for a second set-up, a drift within a few
    // standard deviations, ordinary rates
    if (!(steps >= kWindowMinSteps && N >= 128 && s > 0.0 && scale * s <= 150.0 && scale >= 10.0 &&
          fabs(mu) * o.t <= 3.0 * s && fabs(o.r) <= 1.0 && fabs(o.q) <= 1.0 && far < 1e6))
        return w;
    // ... and no overflow anywhere on the whole mesh, which a march reports and a window that
    // leaves those rows out cannot: a solution starts at up to e^150 (above), grows with the
    // rates by up to e^21 (20 in 64 steps or more), and at a mesh edge, whose one-sided drift may
    // run inward, by e^{1.1 |mu| T / dx} while a step's share is at most 1: e^480 of the e^709 that
    // FP64 holds (largest of 520000 marches: 1e72)
    if (!(fabs(o.r) * o.t <= 20.0 && fabs(o.q) * o.t <= 20.0)) return w;
    const double Y = asinh(scale * s / density), h = 2.0 * Y / (N - 1);  // mesh step in y
    const double per = 1.0 / h;
    {
        const float x = (float)(scale * s), dx = sqrtf(x * x + (float)(density * density)) * (float)h;
        const float drift = (float)(fabs(mu) * o.t) / dx;
        if (!(drift <= (float)steps && drift <= 280.0f)) return w;
    }
    {
        const double u = far > 0.0 ? far : 0.0;
        const double b = 0.5 * (u + sqrt(u * u + 4.0 * 18.0 * s2));
        // the mesh must resolve a standard deviation there
        if (!(sqrt(b * b + density * density) * h <= 0.5 * s)) return w;
        const double at = (asinh(b / density) + Y) * per;
        const int e = (int)ceil(at) + 3;
        if (e < N) w.end = e;
    }
    // the put that the option is in xi
    const double r = o.w < 0 ? o.r : o.q, q = o.w < 0 ? o.q : o.r;
    if (!o.e || !(r > 0.0)) return w;
    const double a0 = r * o.t / s;  // r sqrt(T) / sigma
    if (q > r && log(q / r) > (a0 < 1e-3 ? 0.5 : 4.5) * s) return w;
    const double xb = (double)critical_log_spot((float)o.t, (float)o.z, (float)r, (float)q) -
                      0.18 * s / (1.0 + sqrt(a0 / 6.0));
    if (!(xb > -6.9)) return w;  // nor when it is no number
    const double at = (asinh(xb / density) + Y) * per;
    const int lo = (int)floor(at) - 2;
    if (lo < 16 || lo >= w.end - 8) return w;
    const double dx = sqrt(xb * xb + density * density) * h;
    const double a1 = 0.25 * s2 / steps;  // a at dx = 1
    if (!(a1 <= 150.0 * dx * dx)) return w;
    // the differences of the payoff's exponential, at spacing d = h sqrt(x^2 + density^2) that
    // grows by h^2 |x| a row, are off by c h^2 of it; half as much again for higher orders
    const float xf = (float)xb, rf = (float)r, den = (float)density, d2 = den * den;
    const float up = fmaxf((float)mu, 0.0f), z2 = (float)(o.z * o.z), h2 = 1.5f * (float)(h * h);
    const float idle = fmaxf((float)q, 0.0f);  // what waiting earns of S
    if (o.w < 0) {
        const float u = fmaxf(-xf, 1.0f), v = fmaxf(-xf, 2.0f);  // largest |x| e^x, x^2 e^x past the cut
        const float off = h2 * ((z2 / 6 + up / 2) * u * expf(-u) +
                                fmaxf(-(float)mu, 0.0f) / 6 * (v * v * expf(-v) + d2 * expf(xf)));
        if (!(rf > idle * expf(xf) + off)) return w;
    } else {
        const float a = z2 / 6 + up / 2, b = z2 / 24 + up / 6;  // c = a x + b (x^2 + density^2)
        if (!(rf > idle * expf(xf) + h2 * (b * (xf * xf + d2) - a * xf))) return w;
        const float xc = 0.5f * (sqrtf(fmaxf(0.0f, a * a - 4 * b * (b * d2 - 0.5f * rf / h2))) - a) / b;
        if (!(0.5f * rf > idle * expf(-xc))) return w;
        const float n = (float)per, xa = sqrtf((float)a1 / 0.1f) * n;  // about where a = 0.1
        const float from = asinhf(fmaxf(xa, -xf) / den), edge = (float)(scale * s), end = fminf(xc, edge);
        if (!((asinhf(end / den) - from) * n >= (end + xf) / 2.3f + 20.0f &&
              ((float)Y - from) * n >= (edge + xf) / 2.3f + 20.0f))
            return w;
    }
    w.lo = lo;
    return w;
}

}  // namespace kwgpu
