// Which kernels a call launches, against route_mock.cpp (no kernel runs). One request a line
// on standard input, one line of kernel names, comma-separated, out:
//   price|noalloc N X T      a uniform FP64 batch on device buffers
//   uneven|noalloc_uneven N T X,X,..   sizes taken in turn
//   host|control|greeks N X T          host entry points
//   tune FILE | autotune N T X,X,..    (autotune prints its candidates' launches)
//   capture 0|1              whether the caller's stream is being captured
// Test infrastructure only.
#include <cstdio>
#include <iostream>
#include <sstream>
#include <string>
#include <vector>

#include "kwgpu.h"

extern std::vector<std::string> g_launched;
extern bool g_caller_captures;

int main() {
    kwgpu_ctx* c = nullptr;
    if (kwgpu_create(&c, 0)) return 1;
    std::string line;
    while (std::getline(std::cin, line)) {
        std::istringstream in(line);
        std::string what, xs;
        in >> what;
        int rc = KWGPU_OK;
        g_launched.clear();
        kwgpu_fd1d_params p;
        kwgpu_fd1d_params_default(&p);
        if (what == "tune") {
            in >> xs;
            rc = kwgpu_tune_load(c, xs.c_str());
        } else if (what == "save") {
            in >> xs;
            rc = kwgpu_tune_save(c, xs.c_str());
        } else if (what == "capture") {
            in >> g_caller_captures;
        } else {
            size_t n = 0;
            in >> n;
            kwgpu_option one{0.5, 100, 0.3, 0.05, 0.02, 100, 1, -1};
            std::vector<kwgpu_option> o(n, one);
            for (size_t i = 0; i < n; ++i) o[i].t += 1e-4 * (double)i;  // a PDE each
            std::vector<double> v(n);
            std::vector<int32_t> st(n), x, t;
            std::vector<kwgpu_greeks> g(n);
            if (what == "uneven" || what == "noalloc_uneven" || what == "autotune") {
                std::vector<int> sizes;
                int td = 0;
                in >> td >> xs;
                std::istringstream list(xs);
                for (std::string s; std::getline(list, s, ',');) sizes.push_back(std::stoi(s));
                for (size_t i = 0; i < n; ++i) x.push_back(sizes[i % sizes.size()]);
                t.assign(n, td);
                p.x_dims = x.data();
                p.t_dims = t.data();
            } else {
                in >> p.x_dim >> p.t_dim;
            }
            if (what == "price" || what == "uneven")
                rc = kwgpu_fd1d_price_device(c, o.data(), n, &p, v.data(), st.data(), nullptr);
            else if (what == "noalloc" || what == "noalloc_uneven")
                rc = kwgpu_fd1d_price_device_noalloc(c, o.data(), n, &p, v.data(), st.data(), nullptr);
            else if (what == "host")
                rc = kwgpu_fd1d_price(c, o.data(), n, &p, v.data(), st.data());
            else if (what == "control")
                rc = kwgpu_fd1d_bs_price(c, o.data(), n, &p, v.data(), st.data());
            else if (what == "greeks")
                rc = kwgpu_fd1d_greeks(c, o.data(), n, &p, 0.01, g.data(), st.data());
            else if (what == "autotune")
                rc = kwgpu_fd1d_autotune(c, o.data(), n, &p, v.data(), st.data(), nullptr, 0);
            else
                return 2;
        }
        if (rc) {
            std::printf("error %d %s\n", rc, kwgpu_last_error(c));
            continue;
        }
        for (size_t i = 0; i < g_launched.size(); ++i)
            std::printf("%s%s", i ? "," : "", g_launched[i].c_str());
        std::printf("\n");
    }
    kwgpu_destroy(c);
    return 0;
}
