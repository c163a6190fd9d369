// fd1d_window.h -- the FP64 march at theta 1/2 on each option's window of rows
// (fd1d_plan.h) instead of its whole grid. Part of fd1d_wave.hip, whose set-up, scans and
// step loop it uses.
//
// The march is issue-bound on FP64 VALU instructions, and their number is proportional to
// the rows it carries: about 6 per row and step, plus two lane scans per wave and step.
// A window holds 45 % of a grid's rows on average (1024 points, vol 10-60 %, T 1/12-3), so
// most options of a 1024-point grid fit 512 rows, two to a wave. Measured against the
// whole-grid march on one card: 32768 options at 1024 x 1024 9.77 -> 5.44 ms (VALU
// instructions 4.75e9 -> 2.49e9, their issue 90 % busy instead of 98 % at 1.9 GHz), 16384 on
// per-option grids of 256 to 2048 points 3.58 -> 1.76 ms, 3001 at 777 x 301 267 -> 163 us.
//
// Rows run from the in-the-money side (positions in xi), so the rows in front of a window
// are the ones pinned to the payoff: each step's forward elimination runs over constant
// values there and leaves the same relation x_{lo-1} = alpha + beta x_lo at every step,
// computed once. Nothing is approximated on that side. Beyond the window's end x is 0.

// Row counts that a march is built for: class c holds up to M * L * W rows. Class 0 is the
// whole 2048-point grid in two waves and class 1 the two-wave march of 1280 rows (a sixth of
// the windows of a 2048-point grid have 1025 to 1280 rows); of the one-wave classes the
// costliest come first, 64 / L options to a wave. VALU instructions per step and option, scans
// included, from class 2: 129, 105, 93, 64, 52, 30, 24, 18 (the whole-grid march: 137 for 1024
// points, 69 for 512, 33 for 256); classes 0 and 1: 292 and 218.
struct WindowClass {
    int M, L, W;
};
constexpr WindowClass kWindowClasses[] = {{16, 64, 2}, {10, 64, 2}, {16, 64, 1}, {12, 64, 1}, {10, 64, 1},
                                          {16, 32, 1}, {12, 32, 1}, {16, 16, 1}, {12, 16, 1}, {8, 16, 1}};
constexpr int kClasses = sizeof(kWindowClasses) / sizeof(kWindowClasses[0]);
constexpr int kTwoWave = 2;         // classes below are two-wave
constexpr int kAgain = kClasses;    // counter of the PDEs to be solved again in two waves
static_assert(kClasses + 1 <= kWindowCounters / 2, "a count and a cursor per class");

__device__ __forceinline__ int window_class(int rows) {
    int c = 0;
#pragma unroll
    for (int k = 1; k < kClasses; ++k)
        if (rows <= kWindowClasses[k].M * kWindowClasses[k].L * kWindowClasses[k].W) c = k;
    return c;
}

// The relation x_{lo-1} = alpha + beta x_lo left by the pinned rows lo - kPinnedRows .. lo - 1
// (from the mesh's edge when there are fewer): with x_{i-1} = (A + B x_i) / C, row i is
// linear in (A, B, C),
//     A' = V C - bl A,   B' = -bu C,   C' = b C + bl B,
// so each lane composes its rows' maps and the lanes' maps are composed by a scan. Started
// from x = V + (dt / 2) A V on the row before, which is x up to O(dt^2) where V = payoff;
// window_of admits only windows for which that error is forgotten after kPinnedRows rows.
struct PinnedMap {
    double p, q1, q2, a, b, c, d;  // A <- p A + q1 B + q2 C; (B, C) <- [[a, b], [c, d]] (B, C)
};

__device__ __forceinline__ PinnedMap pinned_mul(const PinnedMap& y, const PinnedMap& x) {
    PinnedMap m{y.p * x.p,
                y.p * x.q1 + y.q1 * x.a + y.q2 * x.c,
                y.p * x.q2 + y.q1 * x.b + y.q2 * x.d,
                y.a * x.a + y.b * x.c,
                y.a * x.b + y.b * x.d,
                y.c * x.a + y.d * x.c,
                y.c * x.b + y.d * x.d};
    // a common scale leaves alpha and beta as they are
    const double s = fmax(fmax(fabs(m.a), fabs(m.b)), fmax(fabs(m.c), fabs(m.d)));
    const int e = (s > 0.0 && s < INFINITY) ? -__builtin_amdgcn_frexp_exp(s) : 0;
    return {ldexp(m.p, e), ldexp(m.q1, e), ldexp(m.q2, e), ldexp(m.a, e),
            ldexp(m.b, e), ldexp(m.c, e),  ldexp(m.d, e)};
}

template <int CTRL, int ROWMASK = 0xF>
__device__ __forceinline__ PinnedMap pinned_step(bool take, const PinnedMap& s) {
    const PinnedMap x{dpp<CTRL, ROWMASK>(s.p), dpp<CTRL, ROWMASK>(s.q1), dpp<CTRL, ROWMASK>(s.q2),
                      dpp<CTRL, ROWMASK>(s.a), dpp<CTRL, ROWMASK>(s.b),  dpp<CTRL, ROWMASK>(s.c),
                      dpp<CTRL, ROWMASK>(s.d)};
    const PinnedMap y = pinned_mul(s, x);
    return {take ? y.p : s.p, take ? y.q1 : s.q1, take ? y.q2 : s.q2, take ? y.a : s.a,
            take ? y.b : s.b, take ? y.c : s.c,   take ? y.d : s.d};
}

// In a two-wave group both waves compute it.
template <int L, int W>
__device__ __forceinline__ void pinned_edge(const FdBatch& b, const PdeParams& P,
                                            const kwgpu_option& o, const Lanes& t, double* qp,
                                            Edge& e) {
    constexpr int K = kPinnedRows / L;
    const int l = W == 2 ? t.lane : t.ls;
    const int i0 = e.lo - kPinnedRows + l * K;
    const double yj = (i0 - 1) * P.dy;
    double ey = exp(P.yMin * (1.0 - yj) + P.yMax * yj), ef = rcp(ey);
    const double grow = exp((P.yMax - P.yMin) * P.dy), shrink = rcp(grow);
    auto next = [&]() {
        const double x = b.density * (0.5 * (ey - ef));
        ey *= grow;
        ef *= shrink;
        return x;
    };
    double xm = next(), x0 = next(), rl = rcp(x0 - xm);
    PinnedMap s{1, 0, 0, 1, 0, 0, 1};
    // x on the row before the first, from the first lane's leading node
    const double v = payoff_xi(P, xm);
    const double start = v + 0.5 * P.dt * (P.call ? o.r - o.q * exp(-xm) : o.q * exp(xm) - o.r);
#pragma unroll 1
    for (int k = 0; k < K; ++k) {
        const int i = i0 + k;
        const double xp = next();
        const double ru = rcp(xp - x0), rm = rcp(xp - xm);
        double bl, bb, bu;
        b_row_rcp(P, b.theta, i, rl, ru, rm, bl, bb, bu);
        const double pay = payoff_xi(P, x0);
        const PinnedMap n{-bl * s.p,
                          pay * s.c - bl * s.q1,
                          pay * s.d - bl * s.q2,
                          -bu * s.c,
                          -bu * s.d,
                          bb * s.c + bl * s.a,
                          bb * s.d + bl * s.b};
        if (i >= 0) s = n;  // positions before the mesh's edge take no part
        xm = x0;
        x0 = xp;
        rl = ru;
    }
    s = pinned_step<kRowShr + 1>(t.pr >= 1, s);
    s = pinned_step<kRowShr + 2>(t.pr >= 2, s);
    s = pinned_step<kRowShr + 4>(t.pr >= 4, s);
    s = pinned_step<kRowShr + 8>(t.pr >= 8, s);
    if constexpr (L >= 32) s = pinned_step<kRowBcast15, 0xA>(t.wrow & 1, s);
    if constexpr (L == 64) s = pinned_step<kRowBcast31, 0xC>(t.wrow >= 2, s);
    group_sync<W>();
    if (l == 0) qp[4 * t.seg] = start;
    if (l == L - 1) {
        qp[4 * t.seg + 1] = s.p;
        qp[4 * t.seg + 2] = s.q2;
        qp[4 * t.seg + 3] = s.b;
        qp[16 + t.seg] = s.d;
    }
    group_sync<W>();
    const double inv = 1.0 / qp[16 + t.seg];
    const bool on = e.lo > 0;
    e.alpha = on ? (qp[4 * t.seg + 1] * (e.lo > kPinnedRows ? qp[4 * t.seg] : 0.0) + qp[4 * t.seg + 2]) * inv : 0.0;
    e.beta = on ? qp[4 * t.seg + 3] * inv : 0.0;
    group_sync<W>();
}

// One wave's (W = 2: one workgroup's) work: the options ids[slot] .. (or slot itself without
// ids), at most `slots`, each on its window (from rec[p], or lo_all when rec is null). Bit k
// of the result: segment k's option has to be solved again on its whole grid (what was
// written for it does not stand): its boundary passed the cut, its price is asked for outside
// the window, or a value is not finite.
template <int M, int L, int W = 1>
__device__ __forceinline__ unsigned solve_window(const FdBatch& b, const uint32_t* ids,
                                                 const int* rec, int lo_all, int slot0, int slots,
                                                 double* qp, double* xchg = nullptr) {
    using Gm = Geo<M, L, W>;
    constexpr int NT = Gm::NT, LT = Gm::LT;
    auto pde = [&](const Lanes& t, int s0, int& lo) {
        Pde d;
        const int slot = s0 + t.seg;
        d.live = slot < slots;
        d.p = d.live ? (ids ? (int)ids[slot] : slot) : 0;
        d.oi = d.live ? (b.rep ? b.rep[d.p] : (uint32_t)d.p) : 0u;
        d.opt = b.opts[d.oi];
        const int xd = b.x_dims ? b.x_dims[d.oi] : b.x_dim;
        const int td = b.t_dims ? b.t_dims[d.oi] : b.t_dim;
        d.P = pde_params(d.opt, xd, td, b.density, b.scale);
        d.solve = d.live && d.P.valid;
        d.N = d.solve ? xd : 0;
        d.steps = d.solve ? td - 1 : 0;
        lo = d.solve ? (rec ? (rec[d.p] & 0xffff) : lo_all) : 0;
        d.j0 = lo + t.ls * M;
        if (d.P.call) d.P.ax = -d.P.ax;
        return d;
    };
    // one bit per segment in which any lane says so
    auto segments = [&](bool v) {
        unsigned r = 0;
        if constexpr (W == 2) {
            r = __syncthreads_or(v) ? 1u : 0u;
        } else {
            const uint64_t votes = __ballot(v);
            constexpr uint64_t seg = L == 64 ? ~0ull : ((1ull << (L & 63)) - 1);
#pragma unroll
            for (int k = 0; k < Gm::G; ++k)
                if (votes & (seg << (k * (L & 63)))) r |= 1u << k;
        }
        return r;
    };
    unsigned again = 0;
    double xv[M];
    {
        const Lanes t = lanes_of<M, L, W>(threadIdx.x & (NT - 1));
        Edge edge{};
        const Pde d = pde(t, slot0, edge.lo);
        if (__ballot(edge.lo > 0)) pinned_edge<L, W>(b, d.P, d.opt, t, qp, edge);
        double ap[M], lo[M], up[M], R[M], Q[M], blv[M], buv[M];
        ScanMul<double> sm;
        setup<M, L, W, true>(b, d, t, qp, xv, ap, lo, up, R, Q, blv, buv, sm, &edge);
        int wmin = 0;
        const int wsteps = __builtin_amdgcn_readfirstlane(group_steps<M, L, W>(d, t, qp, &wmin));
        wmin = __builtin_amdgcn_readfirstlane(wmin);
        double aw = 0.0, bw = 0.0;
        sm.TW0 = 0.0;
        if constexpr (W == 2) two_wave_carries(R[0], t, sm, xchg, aw, bw);
        group_sync<W>();
        double2* qpv = reinterpret_cast<double2*>(qp);
#pragma unroll
        for (int i = 0; i < M; ++i) {
            // every row but one is projected. On a whole grid that is row N - 1, a put's last
            // position and a call's first; behind a cut it is the window's last, whose value is
            // about 0 either way: the projection turns a NaN into the payoff, so the row left
            // without it is what carries one on to the end
            const int at = d.j0 + i;
            const bool proj = d.P.american && at < d.N &&
                              at != (d.P.call && edge.lo == 0 ? 0 : min(edge.lo + LT * M, d.N) - 1);
            qpv[i * NT + t.gl] = make_double2(Q[i], proj ? xv[i] : -INFINITY);
        }
        if constexpr (W == 2) qpv[M * NT + t.gl] = make_double2(aw, bw);
        group_sync<W>();
        march_f64<M, L, W, true, true>(xv, ap, lo, up, R, qpv, sm, t, t.ls == 0, t.ls == LT - 1,
                                       xchg, wmin, wsteps, d.steps, 1.0, edge.k0);
        // the cut holds if the window's first two rows are still pinned
        again = segments(t.ls == 0 && edge.lo > 0 &&
                         !(xv[0] == qpv[t.gl].y && xv[1] == qpv[NT + t.gl].y));
    }
    // the option's record and lane indices are derived again rather than kept in registers
    // over the march (as in solve_group_f64)
    int s2 = slot0, tid = threadIdx.x & (NT - 1);
    asm volatile("" : "+v"(s2), "+v"(tid));
    const Lanes t = lanes_of<M, L, W>(tid);
    int lo = 0;
    const Pde d = pde(t, s2, lo);
    bool bad = false;
#pragma unroll
    for (int i = 0; i < M; ++i) bad |= d.j0 + i < d.N && !isfinite(xv[i]);
    const unsigned nonfinite = segments(bad);
    const bool seg_bad = nonfinite >> t.seg & 1;
    again |= nonfinite & segments(lo > 0 || LT * M < d.N);  // the whole grid decides
    group_sync<W>();
#pragma unroll
    for (int i = 0; i < M; ++i) qp[t.seg * LT * M + t.ls * M + i] = xv[i];
    group_sync<W>();
    bool outside = false;
    if (d.live && !(again >> t.seg & 1)) {
        const double* V = qp + t.seg * LT * M;
        const uint32_t beg = b.off ? b.off[d.p] : 0u;
        const uint32_t end = b.off ? b.off[d.p + 1] : 1u;
        for (uint32_t k = beg + t.ls; k < end; k += LT) {
            const uint32_t o2 = b.off ? b.list[k] : d.oi;
            const kwgpu_option q = b.off ? b.opts[o2] : d.opt;
            double price = NAN;
            int st = KWGPU_STATUS_BAD_INPUT;
            if (d.solve && finite_pos(q.s) && finite_pos(q.k)) {
                const double xs = log(q.s / q.k);
                const int j = bracket(d.P, b.density, xs);
                if (j == 0 || j == d.N) {
                    st = KWGPU_STATUS_OUT_OF_GRID;
                } else {
                    const double x1 = grid_x(d.P, b.density, j), x0 = grid_x(d.P, b.density, j - 1);
                    // a pinned row holds the payoff; a row past the window's end, or a call's
                    // unprojected edge row in front of it, needs the whole grid
                    auto value = [&](int jj, double x) {
                        const int at = d.P.call ? d.N - 1 - jj : jj;
                        if (at < lo) {
                            outside |= d.P.call && at == 0;
                            return payoff(d.P, x);
                        }
                        outside |= at >= lo + LT * M;
                        return V[min(at - lo, LT * M - 1)];
                    };
                    const double v0 = value(j - 1, x0), v1 = value(j, x1);
                    if (seg_bad) {
                        st = KWGPU_STATUS_NONFINITE;
                    } else {
                        price = q.k * (((x1 - xs) * v0 + (xs - x0) * v1) / (x1 - x0));
                        st = isfinite(price) ? KWGPU_STATUS_OK : KWGPU_STATUS_NONFINITE;
                    }
                }
            }
            b.prices[o2] = price;
            if (b.status) b.status[o2] = st;
        }
    }
    again |= segments(outside);
    if constexpr (W == 2) group_sync<W>();  // before LDS is used for the next option
    return again;
}

// The largest xi at which PDE p's price is asked for, over its options k0, k0 + step, ...
__device__ __forceinline__ double far_xi(const FdBatch& b, int p, uint32_t oi, uint32_t k0,
                                         uint32_t step) {
    const uint32_t beg = b.off ? b.off[p] : 0u;
    const uint32_t end = b.off ? b.off[p + 1] : 1u;
    double far = -INFINITY;
    for (uint32_t k = beg + k0; k < end; k += step) {
        const kwgpu_option& q = b.opts[b.off ? b.list[k] : oi];
        const double x = log(q.s / q.k);
        far = fmax(far, q.w < 0 ? x : -x);  // a spot that is not a number asks for nothing
    }
    return far;
}

// Planned launch, one thread per slot: each PDE's window and class, and the classes' counts.
// A PDE with over kFarOptions options keeps its whole grid rather than have one thread
// search them for the furthest spot.
constexpr uint32_t kFarOptions = 256;

__global__ __launch_bounds__(256) void plan_windows(FdBatch b, int* rec, int* counts) {
    __shared__ int n[kClasses];
    if (threadIdx.x < kClasses) n[threadIdx.x] = 0;
    __syncthreads();
    const int slot = blockIdx.x * 256 + threadIdx.x;
    if (slot < b.m) {
        const int p = b.order ? (int)b.order[slot] : slot;
        const uint32_t oi = b.rep ? b.rep[p] : (uint32_t)p;
        const int N = b.x_dims ? b.x_dims[oi] : b.x_dim;
        const int td = b.t_dims ? b.t_dims[oi] : b.t_dim;
        Window w{0, N};
        const int pw = b.like ? (int)b.like[p] : p;
        if (!b.off || b.off[pw + 1] - b.off[pw] <= kFarOptions)
            w = window_of(b.opts[b.like ? b.rep[pw] : oi], N, td - 1, b.density, b.scale,
                          far_xi(b, pw, oi, 0, 1));
        const int c = window_class(w.end - w.lo);
        rec[p] = w.lo | c << 16;
        atomicAdd(&n[c], 1);
    }
    __syncthreads();
    if (threadIdx.x < kClasses && n[threadIdx.x]) atomicAdd(&counts[threadIdx.x], n[threadIdx.x]);
}

// ... and the PDEs listed class by class, in slot order within each block of 256 slots (so
// PDEs sorted by march length stay so, and those that share a wave march about as long).
__global__ __launch_bounds__(256) void list_windows(FdBatch b, const int* rec, const int* counts,
                                                    int* cursor, uint32_t* list) {
    constexpr int C = kClasses;
    __shared__ int n[4][C], at[C];
    const int slot = blockIdx.x * 256 + threadIdx.x, w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    int p = 0, c = -1;
    if (slot < b.m) {
        p = b.order ? (int)b.order[slot] : slot;
        c = rec[p] >> 16;
    }
    int rank = 0;
    for (int k = 0; k < C; ++k) {
        const uint64_t v = __ballot(c == k);
        if (c == k) rank = __popcll(v & ((1ull << lane) - 1));
        if (lane == 0) n[w][k] = __popcll(v);
    }
    __syncthreads();
    if (threadIdx.x < C) {
        const int k = threadIdx.x, all = n[0][k] + n[1][k] + n[2][k] + n[3][k];
        int base = 0;
        for (int i = 0; i < k; ++i) base += counts[i];
        at[k] = base + (all ? atomicAdd(&cursor[k], all) : 0);
    }
    __syncthreads();
    if (c >= 0) {
        int i = at[c] + rank;
        for (int q = 0; q < w; ++q) i += n[q][c];
        list[i] = (uint32_t)p;
    }
}

// An option whose boundary went past its window's cut, of a grid too large for one wave: to
// be solved again by fd1d_window_again.
__device__ __forceinline__ void solve_later(uint32_t p, int* counts, uint32_t* later) {
    if ((threadIdx.x & 63) == 0) later[atomicAdd(&counts[kAgain], 1)] = p;
}

// Few options: one to a wave, spread over all 64 lanes with as few rows per lane as its window
// needs, each finding its own window. Nothing is listed, and grids of up to 1024 points take
// no scratch. The step's length is then its chain of dependent instructions -- the lane's two
// substitutions and the lane scans -- rather than their number. Up to kLoneMax options, two
// waves to a SIMD, all are resident at once. 512 x 512, by number of options: 128 in 142 us
// here (238 us on whole grids, 16 rows a lane), 2048 in 199 us; listed by class 2048 take
// about 220 us and 3072 230 us, here 287 us.
struct LoneWindow {
    int lo, rows, N;
};
__device__ __forceinline__ LoneWindow lone_window(const FdBatch& b, int slot) {
    const int p = b.order ? (int)b.order[slot] : slot;
    const uint32_t oi = b.rep ? b.rep[p] : (uint32_t)p;
    const int N = b.x_dims ? b.x_dims[oi] : b.x_dim;
    const int td = b.t_dims ? b.t_dims[oi] : b.t_dim;
    const int pw = b.like ? (int)b.like[p] : p;
    double far = far_xi(b, pw, oi, threadIdx.x & 63, 64);
    for (int k = 32; k > 0; k >>= 1) far = fmax(far, __shfl_xor(far, k));
    const Window w = window_of(b.opts[b.like ? b.rep[pw] : oi], N, td - 1, b.density, b.scale, far);
    return {__builtin_amdgcn_readfirstlane(w.lo), __builtin_amdgcn_readfirstlane(w.end - w.lo), N};
}

__device__ __forceinline__ void lone_wave(const FdBatch& b, int slot, LoneWindow w, double* qp,
                                          int* counts, uint32_t* later) {
    for (;;) {
        unsigned again;
        if (w.rows <= 256)
            again = solve_window<4, 64>(b, b.order, nullptr, w.lo, slot, slot + 1, qp);
        else if (w.rows <= 384)
            again = solve_window<6, 64>(b, b.order, nullptr, w.lo, slot, slot + 1, qp);
        else if (w.rows <= 512)
            again = solve_window<8, 64>(b, b.order, nullptr, w.lo, slot, slot + 1, qp);
        else if (w.rows <= 768)
            again = solve_window<12, 64>(b, b.order, nullptr, w.lo, slot, slot + 1, qp);
        else
            again = solve_window<16, 64>(b, b.order, nullptr, w.lo, slot, slot + 1, qp);
        if (!again) return;
        if (w.N > 1024) return solve_later(b.order ? b.order[slot] : (uint32_t)slot, counts, later);
        w.lo = 0;  // the whole grid: nothing is pinned, nothing lies outside
        w.rows = w.N;
    }
}

__global__ __attribute__((amdgpu_flat_work_group_size(64, 64), amdgpu_waves_per_eu(2, 2)))
void fd1d_lone(FdBatch b) {
    __shared__ double qp[2 * 64 * 16];
    lone_wave(b, blockIdx.x, lone_window(b, blockIdx.x), qp, nullptr, nullptr);
}

// ... and with grids of over 1024 points: a workgroup of two waves an option, for windows of
// over 1024 rows, which march on their whole grids; otherwise the second wave ends at once.
// (The two kinds of march in launches of their own, side by side, kept each other from the
// SIMDs: 1024 options at 2048 x 512 took 705 us.) Up to kLoneMax / 2 options are resident.
__global__ __attribute__((amdgpu_flat_work_group_size(128, 128), amdgpu_waves_per_eu(2, 2)))
void fd1d_lone_big(FdBatch b, int* counts, uint32_t* later) {
    __shared__ double qp[2 * 128 * 17];
    __shared__ double xchg[4];
    const LoneWindow w = lone_window(b, blockIdx.x);
    if (w.rows > 1024)
        solve_group_f64<16, 64, 2, false>(b, blockIdx.x, qp, xchg);
    else if (threadIdx.x < 64)
        lone_wave(b, blockIdx.x, w, qp, counts, later);
}

// Runs one-wave class c's march over the wave starting at slot.
__device__ __forceinline__ unsigned run_class(int c, const FdBatch& b, const uint32_t* ids,
                                              const int* rec, int lo, int slot, int slots,
                                              double* qp) {
    switch (c) {
        case 2: return solve_window<16, 64>(b, ids, rec, lo, slot, slots, qp);
        case 3: return solve_window<12, 64>(b, ids, rec, lo, slot, slots, qp);
        case 4: return solve_window<10, 64>(b, ids, rec, lo, slot, slots, qp);
        case 5: return solve_window<16, 32>(b, ids, rec, lo, slot, slots, qp);
        case 6: return solve_window<12, 32>(b, ids, rec, lo, slot, slots, qp);
        case 7: return solve_window<16, 16>(b, ids, rec, lo, slot, slots, qp);
        case 8: return solve_window<12, 16>(b, ids, rec, lo, slot, slots, qp);
        default: return solve_window<8, 16>(b, ids, rec, lo, slot, slots, qp);
    }
}

// Wave g's share of the one-wave classes, in order; nothing past the last one. An option whose
// boundary passed its cut is solved again on its whole grid by the same wave, or, above 1024
// points, later.
__device__ __forceinline__ void run_wave(const FdBatch& b, int g, const int* rec, int* counts,
                                         const uint32_t* list, uint32_t* later, double* qp) {
    int c = kTwoWave, begin = 0, slots = 0;
#pragma unroll
    for (int k = 0; k < kTwoWave; ++k) begin += counts[k];
    for (;; ++c) {
        if (c == kClasses) return;
        slots = counts[c];
        const int G = 64 / kWindowClasses[c].L, groups = (slots + G - 1) / G;
        if (g < groups) break;
        g -= groups;
        begin += slots;
    }
    const uint32_t* ids = list + begin;
    int slot = g * (64 / kWindowClasses[c].L);
    const int first = slot;
    unsigned pending = 0;
    for (bool whole = false;; whole = true) {
        const unsigned again = run_class(c, b, ids, whole ? nullptr : rec, 0, slot, slots, qp);
        if (!whole) pending = again;
        for (; pending; pending &= pending - 1) {
            slot = first + __ffs(pending) - 1;
            const uint32_t p = ids[slot], oi = b.rep ? b.rep[p] : p;
            if ((b.x_dims ? b.x_dims[oi] : b.x_dim) <= 1024) break;
            solve_later(p, counts, later);
        }
        if (!pending) return;
        pending &= pending - 1;
        c = kTwoWave;
        slots = slot + 1;
    }
}

// All classes in one launch. 16384 options on per-option grids, one call at a time: 2.56 ms
// with the two-wave groups, on whole grids, in a launch after the others (each launch ends
// with idle SIMDs), 2.12 ms with three launches on streams of their own (which keep each other
// from the SIMDs when several contexts are at work), 2.20 ms as one; 65536 8.28, 7.83 and 7.30
// ms. Grids of up to 1024 points: a wave a workgroup.
__global__ __attribute__((amdgpu_flat_work_group_size(64, 64), amdgpu_waves_per_eu(2, 2)))
void fd1d_windowed(FdBatch b, const int* rec, int* counts, const uint32_t* list) {
    __shared__ double qp[2 * 64 * 16];
    run_wave(b, blockIdx.x, rec, counts, list, nullptr, qp);
}

// ... and larger ones: workgroups of two waves, first (they march longest) one option each of
// class 0, on its whole 2048-point grid, and of class 1, then two independent waves of work.
// The whole-grid march has registers that a windowed one of 16 rows a lane does not: there
// every LDS read of the step loop went through one buffer (0.81 instead of 0.58 us a step).
__global__ __attribute__((amdgpu_flat_work_group_size(128, 128), amdgpu_waves_per_eu(2, 2)))
void fd1d_windowed_big(FdBatch b, const int* rec, int* counts, const uint32_t* list, uint32_t* later) {
    __shared__ double qp[2 * 128 * 17];
    __shared__ double xchg[4];
    const int slot = blockIdx.x, whole = counts[0], both = whole + counts[1];
    if (slot >= both) {
        const int w = threadIdx.x >> 6;
        run_wave(b, 2 * (slot - both) + w, rec, counts, list, later, qp + w * (2 * 64 * 16));
        return;
    }
    if (slot >= whole && !solve_window<10, 64, 2>(b, list, rec, 0, slot, both, qp, xchg)) return;
    b.m = both;
    b.order = list;
    solve_group_f64<16, 64, 2, false>(b, slot, qp, xchg);
}

// The PDEs left for later, on their whole grids. Their count is final by now: the launch that
// adds to it has ended.
__global__ __attribute__((amdgpu_flat_work_group_size(128, 128), amdgpu_waves_per_eu(2, 2)))
void fd1d_window_again(FdBatch b, const int* counts, const uint32_t* later) {
    __shared__ double qp[2 * 128 * 17];
    __shared__ double xchg[4];
    b.m = counts[kAgain];
    if ((int)blockIdx.x >= b.m) return;
    b.order = later;
    solve_group_f64<16, 64, 2, false>(b, blockIdx.x, qp, xchg);
}
