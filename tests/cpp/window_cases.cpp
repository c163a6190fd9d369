// The window rule and the serial marches of window_test.cpp on options from standard input.
//   window_cases <x points> <t points> [density scale]  < lines "t k z r q s e w"
// prints for each option the window, whether its first two rows were still pinned after the
// last step, whether the price lay inside it, the price on the window as it is (not solved
// again) and the price on the whole grid.
#define main window_test_main
#include "window_test.cpp"
#undef main

int main(int n, char** v) {
    const int N = std::atoi(v[1]), steps = std::atoi(v[2]) - 1;
    const double density = n > 4 ? std::atof(v[3]) : 0.25, scale = n > 4 ? std::atof(v[4]) : 50.0;
    kwgpu_option o{};
    int e, w;
    while (std::scanf("%lf %lf %lf %lf %lf %lf %d %d", &o.t, &o.k, &o.z, &o.r, &o.q, &o.s, &e, &w) == 8) {
        o.e = (uint8_t)e;
        o.w = (int8_t)w;
        const double x = (o.w < 0 ? 1 : -1) * std::log(o.s / o.k);
        const kwgpu::Window win = kwgpu::window_of(o, N, steps, density, scale, x);
        const Result a = march(o, N, steps, density, scale, win);
        const Result b = march(o, N, steps, density, scale, {0, N});
        std::printf("%d %d %d %d %.17g %.17g\n", win.lo, win.end, (int)a.pinned, (int)a.inside, a.price,
                    b.price);
    }
}
