// The windowed march against the whole-grid one, both serial and on the CPU: options drawn
// over a wide domain, the window from csrc/fd1d_plan.h, the same elimination of the pinned
// rows as the kernels' (fd1d_window.h), the whole grid where the boundary went past the cut.
//   window_test <x points> <t points> <options> <seed>
// prints the counts and the largest difference relative to max(strike, price).
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>

#define KWGPU_HD inline
#include "../../kwinto-cuda_amd/csrc/fd1d_plan.h"

namespace {

struct Result {
    double price;
    bool inside, pinned;
};

struct Grid {
    const kwgpu_option& o;
    int N;
    double sg, den, Y, dt, a0, ax, axx;
    Grid(const kwgpu_option& o_, int N_, int steps, double den_, double scale)
        : o(o_), N(N_), sg(o_.w < 0 ? 1.0 : -1.0), den(den_) {
        const double s = o.z * std::sqrt(o.t);
        Y = std::asinh(scale * s / den);
        dt = o.t / steps;
        a0 = -o.r;
        ax = sg * (o.r - o.q - o.z * o.z / 2);
        axx = o.z * o.z / 2;
    }
    double xi(int i) const { return den * std::sinh(-Y + 2 * Y * i / (N - 1)); }
    double pay(double x) const { return std::max(0.0, o.w < 0 ? 1 - std::exp(x) : std::exp(-x) - 1); }
    void row(int i, double& bl, double& b, double& bu) const {
        const double h = 0.5 * dt;
        if (i == 0 || i == N - 1) {
            const double inv = 1 / (i == 0 ? xi(1) - xi(0) : xi(N - 2) - xi(N - 1));
            b = 1 - h * (a0 - inv * ax);
            bl = i == 0 ? 0 : -h * inv * ax;
            bu = i == 0 ? -h * inv * ax : 0;
            return;
        }
        const double du = xi(i + 1) - xi(i), dd = xi(i) - xi(i - 1), dm = xi(i + 1) - xi(i - 1);
        bl = -h * (-ax / dm + 2 * axx / (dd * dm));
        bu = -h * (ax / dm + 2 * axx / (du * dm));
        b = 1 - h * (a0 - 2 * axx / (dd * du));
    }
};

Result march(const kwgpu_option& o, int N, int steps, double den, double scale, kwgpu::Window w) {
    const Grid g(o, N, steps, den, scale);
    double alpha = 0, beta = 0;  // x_{lo-1} = alpha + beta x_lo
    if (w.lo > 0) {
        const int st = std::max(0, w.lo - kwgpu::kPinnedRows);
        if (st > 0) {
            const double e = std::exp(g.sg * g.xi(st - 1));
            alpha = g.pay(g.xi(st - 1)) + 0.5 * g.dt * (o.w < 0 ? -o.r + o.q * e : o.r - o.q * e);
        }
        for (int i = st; i < w.lo; ++i) {
            double bl, b, bu;
            g.row(i, bl, b, bu);
            const double c = b + bl * beta;
            alpha = (g.pay(g.xi(i)) - bl * alpha) / c;
            beta = -bu / c;
        }
    }
    const int R = w.end - w.lo;
    std::vector<double> l(R), d(R), u(R), V(R), P(R), f(R);
    double k0 = 0;
    for (int i = 0; i < R; ++i) {
        double bl, b;
        g.row(w.lo + i, bl, b, u[i]);
        l[i] = i ? bl / d[i - 1] : 0;
        d[i] = i ? b - l[i] * u[i - 1] : b + bl * beta;
        if (i == 0) k0 = -bl * alpha;
        V[i] = g.pay(g.xi(w.lo + i));
        const int j = o.w < 0 ? w.lo + i : N - 1 - (w.lo + i);
        P[i] = o.e && j < N - 1 ? V[i] : -INFINITY;
    }
    for (int n = 0; n < steps; ++n) {
        f[0] = V[0] + k0;
        for (int i = 1; i < R; ++i) f[i] = V[i] - l[i] * f[i - 1];
        double x = 0;
        for (int i = R - 1; i >= 0; --i) {
            x = (f[i] - u[i] * x) / d[i];
            V[i] = std::max(2 * x - V[i], P[i]);
        }
    }
    Result r{NAN, true, w.lo == 0 || (V[0] == P[0] && V[1] == P[1])};
    const double x = g.sg * std::log(o.s / o.k);
    int i = 0;
    while (i < N && g.xi(i) < x) ++i;
    if (i < 1 || i >= N) return r;
    auto value = [&](int k) {
        if (k >= w.end || (k == 0 && w.lo > 0 && o.w > 0)) r.inside = false;
        return k < w.lo ? g.pay(g.xi(k)) : k < w.end ? V[k - w.lo] : 0.0;
    };
    const double x1 = g.xi(i), x0 = g.xi(i - 1);
    r.price = o.k * ((x1 - x) * value(i - 1) + (x - x0) * value(i)) / (x1 - x0);
    return r;
}

}  // namespace

int main(int, char** v) {
    const int N = std::atoi(v[1]), t_dim = std::atoi(v[2]), n = std::atoi(v[3]);
    std::mt19937_64 rng(std::atoi(v[4]));
    auto U = [&](double a, double b) { return a + (b - a) * (double)(rng() >> 11) * 0x1p-53; };
    int windowed = 0, past = 0, outside = 0;
    double rows = 0, worst = 0;
    for (int k = 0; k < n; ++k) {
        kwgpu_option o{};
        o.k = 100;
        o.z = std::exp(U(std::log(0.01), std::log(2.0)));
        o.t = std::exp(U(std::log(0.005), std::log(30.0)));
        o.r = U(-0.03, 0.25);
        o.q = U(-0.03, 0.3);
        o.s = 100 * std::exp(U(-1.4, 1.4));
        o.e = rng() % 4 != 0;
        o.w = rng() & 1 ? 1 : -1;
        const double x = (o.w < 0 ? 1 : -1) * std::log(o.s / o.k);
        const kwgpu::Window w = kwgpu::window_of(o, N, t_dim - 1, 0.25, 50.0, x);
        rows += (double)(w.end - w.lo) / N;
        if (w.lo == 0 && w.end == N) continue;
        ++windowed;
        const Result a = march(o, N, t_dim - 1, 0.25, 50.0, w);
        if (!a.pinned) {
            ++past;
            continue;
        }
        if (!a.inside) {
            ++outside;
            continue;
        }
        const Result b = march(o, N, t_dim - 1, 0.25, 50.0, {0, N});
        if (std::isnan(a.price) != std::isnan(b.price)) {
            worst = INFINITY;
            continue;
        }
        if (std::isnan(a.price)) continue;
        const double e = std::fabs(a.price - b.price) / std::max(o.k, b.price);
        if (e > worst) {
            worst = e;
            if (e > 1e-13)
                std::fprintf(stderr, "t=%g z=%g r=%g q=%g s=%g e=%d w=%d window %d..%d: %.17g %.17g\n",
                             o.t, o.z, o.r, o.q, o.s, o.e, o.w, w.lo, w.end, a.price, b.price);
        }
    }
    std::printf("%d %d %d %.3f %.3g\n", windowed, past, outside, rows / n, worst);
}
