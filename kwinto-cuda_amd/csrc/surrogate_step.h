// surrogate_step.h -- one training step of the surrogate's networks in three launches, inside
// namespace kwgpu::sur (included by surrogate.hip only): step_rows (forward and backward of a
// block of rows, the bias and output-layer sums), step_wgrad (the weight gradients) and
// step_update (the sums over blocks, Adam, the BF16 weights).
//
// Every sum is taken in the order of the network's mathematics as first written here, layer by
// layer in a kernel each: training amplifies the last bit (another order of one FP32 sum
// became 4e-5 of the weights in eight Adam steps), and a fit is to stay the same for a seed.
// So each MFMA accumulates the same 32-wide steps of k, the column sums run over rows r,
// r + 4 rs, r + 8 rs .. for rs = n / 64 blocks (at most 128), and the weight gradients over
// n / 512 splits (at most 32) of consecutive rows.
//
// Four networks, 8192 rows each, one step: 444 us as 25 launches (the FP32 pre-activations of
// four layers written and read twice, an FP32 exponential and division per activation and
// direction), 113 us as these three (61, 38 and 14 us); a training step's products take 16 us
// at the dense BF16 rate.

typedef bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef short shortx4 __attribute__((ext_vector_type(4)));
// four floats at any float's address (a member's parameters start at a multiple of kP floats,
// which is odd)
typedef float floatx4u __attribute__((ext_vector_type(4), aligned(4)));

// sigm of four values. The division is one Newton step on v_rcp_f32, which gives the
// correctly rounded 1 / x for every float x in [1, 2^126) (all 1.06e9 of them compared);
// beyond, where the quotient is denormal or x infinite, the four are divided.
__device__ __forceinline__ void sigm4(const float (&z)[4], float (&s)[4]) {
    float x[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) x[e] = 1.0f + __expf(-z[e]);
    if (__builtin_expect(fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3])) < 0x1p126f, 1)) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float r = __builtin_amdgcn_rcpf(x[e]);
            s[e] = fmaf(fmaf(-x[e], r, 1.0f), r, r);
        }
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) s[e] = 1.0f / x[e];
    }
}

// v of the lane N below in its row of 16, around the row.
template <int N>
__device__ __forceinline__ float row_ror(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v),
                                                                 0x120 + N, 0xf, 0xf, true));
}

// The BF16 weights are held in the order in which MFMA 16x16x32 takes them, so that a wave's
// fragment is 1 KB of consecutive addresses: of W[n][k], 16 rows x 32 columns after another,
// each 64 lanes x 8 values, lane n % 16 + 16 ((k / 8) % 4).
__host__ __device__ inline int frag_at(int n, int k) {
    return (((n >> 4) * (H / 32) + (k >> 5)) * 64 + (n & 15) + 16 * ((k >> 3) & 3)) * 8 + (k & 7);
}

// Blocks of the column sums of an n-row batch, of the input layer's gradient, and splits of
// the weight gradients' rows.
inline int sum_blocks(int n) { return std::max(1, std::min(kPartRows, n / 64)); }
inline int l1_blocks(int n) { return std::max(1, std::min(64, n / 128)); }
inline int wgrad_splits(int n) { return std::max(1, std::min(kMaxSplits, n / 512)); }

// Planes of `act`: H1, H2, H3, then dZ1 .. dZ4, each `plane` BF16 values per member.
constexpr int kPlanes = 7, kPlaneDZ = 3;

struct StepArgs {
    const float *feat, *target;  // samples; batch row m of member k is sample idx[k sidx + m]
    const uint32_t* idx;         // ... or sample m (null)
    long sidx;
    int n, rs;                   // rows, blocks of the column sums (gridDim.y)
    const float* p;              // first member's parameters and BF16 weights
    const bf16 *wb, *wbT;
    float* x;                    // the rows' features in batch order (null: not wanted)
    long srow;                   // ... rows per member
    bf16* act;
    long plane;
    float *part_b, *part_o;      // [member][layer][block][H], [member][block][H + 1]
    float* loss;                 // [member], added to
};

// The layer product of a wave: RT x 16 rows of `act` (LDS) by its 32 columns, whose
// fragments W[j][k step] the caller has begun to load (kPre steps of k).
constexpr int kStepLd = H + 8;  // LDS row pitch of BF16 activations: rows 4 banks apart
constexpr int kZ4Ld = H + 4;    // ... of the FP32 last layer
constexpr int kPre = 4;
struct WeightFrags {
    bf16x8 f[2][kPre];
};
__device__ __forceinline__ void load_frags(WeightFrags& wf, const bf16x8* W) {
#pragma unroll
    for (int k = 0; k < kPre; ++k)
#pragma unroll
        for (int j = 0; j < 2; ++j) wf.f[j][k] = W[(j * (H / 32) + k) * 64];
}
template <int RT>
__device__ __forceinline__ void step_mma(floatx4 (&acc)[RT][2], WeightFrags& wf, const bf16x8* W,
                                         const bf16* act, int l) {
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    const bf16* a0 = act + (l & 15) * kStepLd + 8 * (l >> 4);
    const auto rows = [&](int i, int k) {
        return *reinterpret_cast<const bf16x8*>(a0 + 16 * i * kStepLd + 32 * k);
    };
    bf16x8 a[RT];
#pragma unroll
    for (int i = 0; i < RT; ++i) a[i] = rows(i, 0);
#pragma unroll
    for (int k = 0; k < H / 32; ++k) {
        const bf16x8 b0 = wf.f[0][k % kPre], b1 = wf.f[1][k % kPre];
#pragma unroll
        for (int i = 0; i < RT; ++i) {
            acc[i][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b0, a[i], acc[i][0], 0, 0, 0);
            acc[i][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b1, a[i], acc[i][1], 0, 0, 0);
            if (k + 1 < H / 32) a[i] = rows(i, k + 1);
        }
        if (k + kPre < H / 32) {
            wf.f[0][k % kPre] = W[(k + kPre) * 64];
            wf.f[1][k % kPre] = W[(H / 32 + k + kPre) * 64];
        }
        // left alone, the scheduler moves all of a layer's loads to its top and spills
        __builtin_amdgcn_sched_barrier(0);
    }
}

// ... with the loads left to the compiler, for a kernel of enough waves to wait for them
template <int RT>
__device__ __forceinline__ void wave_mma(floatx4 (&acc)[RT][2], const bf16x8* W, const bf16* act,
                                         int l) {
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    const bf16* a0 = act + (l & 15) * kStepLd + 8 * (l >> 4);
#pragma unroll 2
    for (int k = 0; k < H / 32; ++k) {
        const bf16x8 b0 = W[k * 64], b1 = W[(H / 32 + k) * 64];
#pragma unroll
        for (int i = 0; i < RT; ++i) {
            const bf16x8 a = *reinterpret_cast<const bf16x8*>(a0 + 16 * i * kStepLd + 32 * k);
            acc[i][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b0, a, acc[i][0], 0, 0, 0);
            acc[i][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b1, a, acc[i][1], 0, 0, 0);
        }
    }
}

// Forward and backward of the rows of one block `by` of the column sums (rows 4 by + ph +
// 4 rs j, phases ph = 0 .. 3), RT x 16 rows at a time: row 16 i + c of the tile is phase
// c % 4, j = 4 i + c / 4. At n <= 8192 a block is 64 rows, or up to 68 where 64 does not
// divide n: RT = 5 then takes them in one pass instead of two.
//
// One workgroup of eight waves per CU. Activations stay in LDS (two BF16 buffers in turn; the
// last layer's FP32 activations share the second) and wave w computes columns 32 w .. + 31 of
// every row, with the weights as the A operand: a lane then holds four adjacent columns of a
// row. The derivative of SiLU is kept in registers (3 x 8 RT) from the forward pass, so each
// activation costs one exponential. To memory go the rows' H1..H3 and dZ1..dZ4 in BF16 (the
// weight gradients read them), 117 MB for four networks of 8192 rows, instead of 0.6 GB. The
// 512 workgroups of that batch run in two rounds of 65000 cycles: SiLU's VALU and the MFMA of
// the two waves of a SIMD take 40000 of them, the rows' gather and the barriers the rest.
template <int RT>
__global__ __attribute__((amdgpu_flat_work_group_size(512, 512), amdgpu_waves_per_eu(2, 2)))
void step_rows(StepArgs g) {
    constexpr int R = 16 * RT;
    static_assert(H == 256 && R <= 32 * 16, "eight waves of 32 columns; 16 passes of 32 rows");
    static_assert(kZ4Ld * sizeof(float) >= kStepLd * sizeof(bf16), "the buffers' union");
    __shared__ __attribute__((aligned(16))) bf16 act0[R * kStepLd];
    __shared__ __attribute__((aligned(16))) float z4[R * kZ4Ld];
    __shared__ __attribute__((aligned(16))) float xs[R * F];
    __shared__ __attribute__((aligned(16))) float ws[H * F + H];  // W1 | b1
    __shared__ __attribute__((aligned(16))) float bs[4][H];  // b2, b3, b4 and W5
    __shared__ float tg[R], sdy[R], lred[8];
    bf16* const act1 = reinterpret_cast<bf16*>(z4);
    const int t = threadIdx.x, w = t >> 6, l = t & 63;
    const int mem = blockIdx.x, by = blockIdx.y;
    const int c0 = 32 * w + 4 * (l >> 4);  // this lane's columns: c0 + 16 j + 0 .. 3
    const int row = l & 15;                // ... and rows: row + 16 i
    const int wofs = 2 * w * (H / 32) * 64 + l;  // this wave's fragments of a layer
    constexpr int LW = H * H / 8;  // a layer's weights
    const int stride = 4 * g.rs;
    const int cp = t & 127, ph = t >> 7;  // column sums: columns 2 cp, 2 cp + 1 of phase ph
    float so[2] = {}, sb5 = 0.0f, sb[3][2] = {}, loss = 0.0f;
    const auto batch_row = [&](int r, int j0) { return 4 * by + (r & 3) + stride * (j0 + (r >> 2)); };
    // rows of the tile in buffer b to plane q of act, 16 bytes a lane
    const auto copy_out = [&](const bf16* b, int q, int j0) {
        const int m = batch_row(t >> 5, j0);
        bf16* out = g.act + ((long)mem * kPlanes + q) * g.plane + (long)m * H + 8 * (t & 31);
        b += (t >> 5) * kStepLd + 8 * (t & 31);
        bf16x8 v[RT];
#pragma unroll
        for (int i = 0; i < RT; ++i) v[i] = *reinterpret_cast<const bf16x8*>(b + 16 * i * kStepLd);
#pragma unroll
        for (int i = 0; i < RT; ++i)
            if (m + 4 * i * stride < g.n)
                *reinterpret_cast<bf16x8*>(out + (long)(4 * i * stride) * H) = v[i];
    };
    for (int j0 = 0; batch_row(0, j0) < g.n; j0 += 4 * RT) {
        // the parameters' addresses, made new in each pass: kept over the loop, what is loaded
        // from them and the addresses themselves took 160 registers that spilled
        const float* p = g.p + (long)mem * kP;
        const bf16x8* W = reinterpret_cast<const bf16x8*>(g.wb) + (long)mem * 3 * LW;
        const bf16x8* WT = reinterpret_cast<const bf16x8*>(g.wbT) + (long)mem * 3 * LW;
        asm volatile("" : "+s"(p), "+s"(W), "+s"(WT));
        W += wofs;
        WT += wofs;
        // rows of this phase in the tile
        const int m0 = batch_row(ph, j0);
        const int nq = m0 < g.n ? min(4 * RT, (g.n - m0 + stride - 1) / stride) : 0;
        // the rows first: their indices and then their features take a memory latency each
        if (t < R) {
            const int m = batch_row(t, j0);
            floatx4 xa = {0.f, 0.f, 0.f, 0.f}, xb = xa;
            float y = 0.0f;
            if (m < g.n) {
                const size_t s = g.idx ? g.idx[mem * g.sidx + m] : (size_t)m;
                xa = *reinterpret_cast<const floatx4*>(g.feat + s * F);
                xb = *reinterpret_cast<const floatx4*>(g.feat + s * F + 4);
                y = g.target[s];
                if (g.x) {
                    float* q = g.x + ((long)mem * g.srow + m) * F;
                    *reinterpret_cast<floatx4*>(q) = xa;
                    *reinterpret_cast<floatx4*>(q + 4) = xb;
                }
            }
            *reinterpret_cast<floatx4*>(xs + t * F) = xa;
            *reinterpret_cast<floatx4*>(xs + t * F + 4) = xb;
            tg[t] = y;
        } else {
            // W1 | b1, then b2, b3, b4 and W5
            for (int c = t - R; c < kB1 + H; c += 512 - R) ws[c] = p[c];
            for (int c = t - R; c < 4 * H; c += 512 - R) {
                const int k = c / H;
                bs[k][c % H] = p[(k < 3 ? kB2 + k * (H * H + H) : kW5) + c % H];
            }
        }
        WeightFrags wf;
        load_frags(wf, W);
        const float b5 = p[kB5];
        __syncthreads();
        floatx4 acc[RT][2];
        float d1[RT][2][4], d2[RT][2][4], d3[RT][2][4];  // SiLU' of layers 1 .. 3
        // silu of z to row 16 i + row, columns c0 + 16 j, of BF16 buffer b; its derivative to d
        const auto activate = [&](const float (&z)[4], float (&d)[4], bf16* b, int i, int j) {
            float s[4];
            sigm4(z, s);
            bf16x4 h;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                h[e] = (bf16)(z[e] * s[e]);
                d[e] = s[e] * (1.0f + z[e] * (1.0f - s[e]));
                asm volatile("" : "+v"(d[e]));  // here: z and s would live on to its use
            }
            *reinterpret_cast<bf16x4*>(b + (16 * i + row) * kStepLd + c0 + 16 * j) = h;
        };
#pragma unroll
        for (int j = 0; j < 2; ++j) {  // input layer, FP32
            floatx4 w1[4][2], b1 = *reinterpret_cast<const floatx4*>(ws + kB1 + c0 + 16 * j);
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int f = 0; f < 2; ++f)
                    w1[e][f] = *reinterpret_cast<const floatx4*>(ws + (c0 + 16 * j + e) * F + 4 * f);
#pragma unroll
            for (int i = 0; i < RT; ++i) {
                const float* xr = xs + (16 * i + row) * F;
                const floatx4 xa = *reinterpret_cast<const floatx4*>(xr);
                const floatx4 xb = *reinterpret_cast<const floatx4*>(xr + 4);
                float z[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    z[e] = b1[e];
#pragma unroll
                    for (int f = 0; f < 4; ++f) z[e] = fmaf(w1[e][0][f], xa[f], z[e]);
#pragma unroll
                    for (int f = 0; f < 4; ++f) z[e] = fmaf(w1[e][1][f], xb[f], z[e]);
                }
                activate(z, d1[i][j], act0, i, j);
            }
        }
        __syncthreads();
        // hidden layer `layer` (0 .. 2) from buffer in: its sums in acc, biases in bias
        floatx4 bias[2];
        const auto product = [&](int layer, const bf16* in) {
            step_mma<RT>(acc, wf, W + layer * LW, in, l);
            load_frags(wf, layer < 2 ? W + (layer + 1) * LW : WT + 2 * LW);
            copy_out(in, layer, j0);
#pragma unroll
            for (int j = 0; j < 2; ++j)
                bias[j] = *reinterpret_cast<const floatx4*>(&bs[layer][c0 + 16 * j]);
        };
        const auto hidden = [&](int layer, const bf16* in, bf16* out, float (&d)[RT][2][4]) {
            product(layer, in);
#pragma unroll
            for (int i = 0; i < RT; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    float z[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) z[e] = acc[i][j][e] + bias[j][e];
                    activate(z, d[i][j], out, i, j);
                }
            __syncthreads();
        };
        hidden(0, act0, act1, d2);
        hidden(1, act1, act0, d3);
        product(2, act0);
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) {  // silu(Z4) in FP32 to LDS, its derivative to acc
                float z[4], s[4];
                floatx4 h;
#pragma unroll
                for (int e = 0; e < 4; ++e) z[e] = acc[i][j][e] + bias[j][e];
                sigm4(z, s);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    h[e] = z[e] * s[e];
                    float d = s[e] * (1.0f + z[e] * (1.0f - s[e]));
                    asm volatile("" : "+v"(d));
                    acc[i][j][e] = d;
                }
                *reinterpret_cast<floatx4*>(z4 + (16 * i + row) * kZ4Ld + c0 + 16 * j) = h;
            }
        __syncthreads();
        {  // output layer and its error: 16 lanes a row, four rows a wave at a time
            const int c = l & 15;
            float w5[H / 16];
#pragma unroll
            for (int q = 0; q < H / 16; ++q) w5[q] = bs[3][c + 16 * q];
            float y = 0.0f;  // lane c keeps row 32 c + 4 w + l / 16
#pragma unroll
            for (int k = 0; k < RT / 2 + RT % 2; ++k) {
                const int r = 32 * k + 4 * w + (l >> 4);
                const float* z = z4 + min(r, R - 1) * kZ4Ld + c;
                float s[4];  // columns c + 16 a, + 64, + 128, + 192
#pragma unroll
                for (int a = 0; a < 4; ++a) {
                    s[a] = 0.0f;
#pragma unroll
                    for (int q = 0; q < H / 64; ++q)
                        s[a] = fmaf(w5[a + 4 * q], z[16 * a + 64 * q], s[a]);
                }
                float v = (s[0] + s[2]) + (s[1] + s[3]);
                v += row_ror<8>(v);
                v += row_ror<4>(v);
                v += row_ror<2>(v);
                v += row_ror<1>(v);
                y = c == k ? v : y;
            }
            const int r = 32 * c + 4 * w + (l >> 4);
            if (r < R) {
                const float d = y + b5 - tg[r];
                const bool in = batch_row(r, j0) < g.n;
                sdy[r] = in ? 2.0f * d / (float)g.n : 0.0f;
                loss += in ? d * d : 0.0f;
            }
        }
        __syncthreads();
        const auto out_grad = [&](int q) {  // gradient of W5 and b5
            const int r = 4 * q + ph;
            const float dy = sdy[r];
            const float2 h = *reinterpret_cast<const float2*>(z4 + r * kZ4Ld + 2 * cp);
            so[0] = fmaf(dy, h.x, so[0]);
            so[1] = fmaf(dy, h.y, so[1]);
            sb5 += dy;
        };
        if (nq >= 16) {
#pragma unroll
            for (int q = 0; q < 16; ++q) out_grad(q);
            for (int q = 16; q < nq; ++q) out_grad(q);
        } else {
            for (int q = 0; q < nq; ++q) out_grad(q);
        }
        {
            floatx4 w5[2];
#pragma unroll
            for (int j = 0; j < 2; ++j) w5[j] = *reinterpret_cast<const floatx4*>(&bs[3][c0 + 16 * j]);
#pragma unroll
            for (int i = 0; i < RT; ++i) {
                const float dy = sdy[16 * i + row];
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    bf16x4 d;
#pragma unroll
                    for (int e = 0; e < 4; ++e) d[e] = (bf16)(dy * w5[j][e] * acc[i][j][e]);
                    *reinterpret_cast<bf16x4*>(act0 + (16 * i + row) * kStepLd + c0 + 16 * j) = d;
                }
            }
        }
        __syncthreads();
        // dZ of layer + 2 in buffer in: its column sums, its rows to memory, and dZ of the
        // layer below to buffer out
        const auto back = [&](int layer, const bf16* in, bf16* out, const float (&d)[RT][2][4]) {
            step_mma<RT>(acc, wf, WT + layer * LW, in, l);
            if (layer > 0) load_frags(wf, WT + (layer - 1) * LW);
            const bf16* v = in + ph * kStepLd + 2 * cp;
            const auto at = [&](int q) {
                return *reinterpret_cast<const bf16x2*>(v + 4 * q * kStepLd);
            };
            const auto add = [&](bf16x2 x) {
                sb[layer][0] += (float)x[0];
                sb[layer][1] += (float)x[1];
            };
            copy_out(in, kPlaneDZ + 1 + layer, j0);
            if (nq >= 16) {
                bf16x2 x[16];
#pragma unroll
                for (int q = 0; q < 16; ++q) x[q] = at(q);
#pragma unroll
                for (int q = 0; q < 16; ++q) add(x[q]);
                for (int q = 16; q < nq; ++q) add(at(q));
            } else {
                for (int q = 0; q < nq; ++q) add(at(q));
            }
#pragma unroll
            for (int i = 0; i < RT; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    bf16x4 v;
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] = (bf16)(acc[i][j][e] * d[i][j][e]);
                    *reinterpret_cast<bf16x4*>(out + (16 * i + row) * kStepLd + c0 + 16 * j) = v;
                }
            __syncthreads();
        };
        back(2, act0, act1, d3);
        back(1, act1, act0, d2);
        back(0, act0, act1, d1);
        copy_out(act1, kPlaneDZ, j0);
    }
    // the four phases' sums meet in LDS: b2, b3, b4, W5, and b5
    __syncthreads();
#pragma unroll
    for (int e = 0; e < 2; ++e) {
#pragma unroll
        for (int k = 0; k < 3; ++k) z4[(k * 4 + ph) * H + 2 * cp + e] = sb[k][e];
        z4[(12 + ph) * H + 2 * cp + e] = so[e];
    }
    if (cp == 0) sdy[ph] = sb5;
    for (int o = 32; o > 0; o >>= 1) loss += __shfl_xor(loss, o);
    if (l == 0) lred[w] = loss;
    __syncthreads();
    for (int o = t; o < 4 * H; o += 512) {
        const int k = o / H, c = o % H;
        const float* q = z4 + k * 4 * H + c;
        const float v = q[0] + q[H] + q[2 * H] + q[3 * H];
        if (k < 3)
            g.part_b[(((long)mem * 3 + k) * g.rs + by) * H + c] = v;
        else
            g.part_o[((long)mem * g.rs + by) * (H + 1) + c] = v;
    }
    if (t == 0) {
        g.part_o[((long)mem * g.rs + by) * (H + 1) + H] = sdy[0] + sdy[1] + sdy[2] + sdy[3];
        float v = 0.0f;
        for (int k = 0; k < 8; ++k) v += lred[k];
        atomicAdd(g.loss + mem, v);
    }
}

struct WgradArgs {
    const bf16* act;
    long plane;
    int n, members, splits, k_split, l1;  // l1: blocks of the input layer's gradient per member
    const float* x;
    long sx;
    float *part_w, *part_1;  // [member][layer][phase][H H], [member][block][H F + H]
};

// Input layer gradients of one block: part W1[j][f] = sum_m dZ1[m][j] x[m][f], b1[j] = sum_m
// dZ1[m][j] over the block's rows. Each lane owns four adjacent columns, so a wave reads one
// whole 512-byte dZ1 row per iteration and the row's eight inputs once (wave-uniform); the
// four waves' partial sums meet in LDS.
constexpr int kL1V = 4 * (F + 1);
__device__ __forceinline__ void l1_grad(const WgradArgs& g, int mem, int blk, float* lds) {
    static_assert(H == 256, "one wave covers a row as 64 lanes x 4 columns");
    constexpr int V = kL1V;
    const bf16* dZ1 = g.act + ((long)mem * kPlanes + kPlaneDZ) * g.plane;
    const float* x = g.x + mem * g.sx;
    float* part = g.part_1 + ((long)mem * g.l1 + blk) * (H * F + H);  // W1 | b1 order
    const int lane = threadIdx.x & 63, n = g.n;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    float s[V] = {};
    // U rows per wave per pass, all loads issued before any use (one wave per SIMD
    // here, so the loads' latency is hidden only by having several in flight)
    constexpr int U = 8;
    const int stride = 4 * g.l1;
    for (int m0 = blk * 4 + w; m0 < n; m0 += U * stride) {
        bf16x4 d4[U];
        float xf[U][F];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            // rows past the end load the last row (no branch around the loads) and
            // contribute d = 0
            const int m = m0 + u * stride;
            const int mc = min(m, n - 1);
            const bf16x4 v = *(const bf16x4*)(dZ1 + (long)mc * H + 4 * lane);
            d4[u] = m < n ? v : bf16x4{};
#pragma unroll
            for (int f = 0; f < F; ++f) xf[u][f] = x[(long)mc * F + f];
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float d = (float)d4[u][j];
#pragma unroll
                for (int f = 0; f < F; ++f) s[j * (F + 1) + f] = fmaf(d, xf[u][f], s[j * (F + 1) + f]);
                s[j * (F + 1) + F] += d;
            }
    }
#pragma unroll
    for (int v = 0; v < V; ++v) lds[v * 256 + threadIdx.x] = s[v];
    __syncthreads();
    for (int o = threadIdx.x; o < V * 64; o += 256) {
        const int v = o >> 6, l = o & 63;
        const float t = lds[v * 256 + l] + lds[v * 256 + 64 + l] + lds[v * 256 + 128 + l] +
                        lds[v * 256 + 192 + l];
        const int col = 4 * l + v / (F + 1), f = v % (F + 1);
        part[f < F ? col * F + f : H * F + col] = t;
    }
}

// The splits of phase ph in the order of their sum (phase_chain below): chain 0 takes splits
// ph, ph + 16 .. and the tail, chain c of 1 .. 3 takes ph + 4 c, ph + 4 c + 16 ..; within a
// split, rows in steps of 32.
struct SplitRows {
    int ph, nb, m, n0, k_split, n;  // m splits a chain, n0 in chain 0
    int q, chain, k0, ke;           // split number q of the phase: its chain, rows k0 .. ke
    bool end;
    __device__ SplitRows(int ph, int nb, int k_split, int n) : ph(ph), nb(nb), k_split(k_split), n(n) {
        m = nb > ph + 12 ? (nb - ph - 12 + 15) / 16 : 0;
        n0 = m + (nb - ph - 16 * m > 0 ? (nb - ph - 16 * m + 3) / 4 : 0);
        q = -1;
        split();
    }
    __device__ void split() {  // the next one that has rows
        do {
            ++q;
            end = q >= n0 + 3 * m;
            const int r = q - n0;
            chain = r < 0 ? 0 : r < m ? 1 : r < 2 * m ? 2 : 3;
            const int b = r >= 0 ? ph + 4 * chain + 16 * (r - (chain - 1) * m)
                                 : q < m ? ph + 16 * q : ph + 16 * m + 4 * (q - m);
            k0 = b * k_split;
            ke = min(n, k0 + k_split);
        } while (!end && k0 >= ke);
    }
    __device__ void next() {
        k0 += 32;
        if (k0 >= ke) split();
    }
};

// Weight gradients dW[o][i] = sum_m dZ[m][o] H[m][i], summed over splits of consecutive rows
// and those over phases: a workgroup takes the splits of one phase (split % 4) one after
// another for a tile of 64 o x 128 i, 32 x 64 per wave, so that four partial sums go to memory
// instead of one per split. All layers and members in one launch; the last l1 x members
// workgroups take the input layer's gradient. Both operands have the sum's index m across
// rows: 32 rows of each are staged in LDS as they lie and read transposed
// (ds_read_b64_tr_b16: 16 lanes read 4 rows x 16 columns, lane c gets column c). Rows 8 g + r
// and 8 g + 4 + r, r < 4, lie at LDS rows 4 g + r and 16 + 4 g + r, 32 bytes apart mod 256,
// so that the 16 rows of one read spread over all banks. Bound by reading the activations
// (117 MB at four networks of 8192 rows): 43 us
// with a partial sum and a 128 x 128 tile per split, 38 us so, and step_update 19 -> 14 us.
constexpr int kTileO = 64, kTileI = 128, kWgradTiles = (H / kTileO) * (H / kTileI);
__global__ __attribute__((amdgpu_flat_work_group_size(256, 256), amdgpu_waves_per_eu(2, 2)))
void step_wgrad(WgradArgs g) {
    constexpr int BK = 32, LA = kTileO + 16, LB = kTileI + 16;  // LDS row pitches
    constexpr int kStage = BK * (LA + LB);  // BF16 values of one stage: dZ, then H
    constexpr int kLds = std::max<int>(2 * kStage * sizeof(bf16), kL1V * 256 * sizeof(float));
    __shared__ __attribute__((aligned(16))) char raw[kLds];
    const int phases = min(4, g.splits), units = 3 * g.members * phases;
    const int id = blockIdx.x;
    if (id >= kWgradTiles * units) {
        const int b = id - kWgradTiles * units;
        l1_grad(g, b % g.members, b / g.members, reinterpret_cast<float*>(raw));
        return;
    }
    bf16* const lds = reinterpret_cast<bf16*>(raw);
    // the tiles of a unit, which share their rows, are `units` workgroups apart: on the same
    // L2 where 8 divides that
    const int unit = id % units, tile = id / units;
    const int mem = unit % g.members, layer = unit / g.members % 3, ph = unit / g.members / 3;
    const int o0 = tile / (H / kTileI) * kTileO, i0 = tile % (H / kTileI) * kTileI;
    const int t = threadIdx.x, w = t >> 6, l = t & 63;
    // staging: 16 bytes of a row of dZ (8 lanes a row) and of two rows of H (16 lanes a row)
    const int ra = t >> 3, ca = 8 * (t & 7), rb = t >> 4, cb = 8 * (t & 15);
    const bf16* A = g.act + ((long)mem * kPlanes + kPlaneDZ + 1 + layer) * g.plane + o0 + ca;
    const bf16* B = g.act + ((long)mem * kPlanes + layer) * g.plane + i0 + cb;
    struct Stage {
        bf16x8 a, b[2];
    };
    const auto load = [&](Stage& v, const SplitRows& s) {
        v.a = v.b[0] = v.b[1] = bf16x8{};
        if (s.end) return;
        if (s.k0 + ra < s.ke) v.a = *reinterpret_cast<const bf16x8*>(A + (long)(s.k0 + ra) * H);
#pragma unroll
        for (int q = 0; q < 2; ++q)
            if (s.k0 + 16 * q + rb < s.ke)
                v.b[q] = *reinterpret_cast<const bf16x8*>(B + (long)(s.k0 + 16 * q + rb) * H);
    };
    const auto lds_row = [](int m) { return ((m >> 2) & 1) * 16 + (m >> 3) * 4 + (m & 3); };
    const auto store = [&](const Stage& v, bf16* s) {
        *reinterpret_cast<bf16x8*>(s + lds_row(ra) * LA + ca) = v.a;
#pragma unroll
        for (int q = 0; q < 2; ++q)
            *reinterpret_cast<bf16x8*>(s + BK * LA + lds_row(16 * q + rb) * LB + cb) = v.b[q];
    };
    // a fragment: column c0 + l % 16, rows 8 (l / 16) .. + 7 of a stage
    const auto frag = [&](const bf16* s, int ld, int c0) {
        typedef __attribute__((address_space(3))) shortx4 lds_s4;
        const bf16* q = s + (l >> 2) * ld + c0 + 4 * (l & 3);
        const shortx4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)q);
        const shortx4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(q + 16 * ld));
        return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    };
    const int co = 32 * (w >> 1), ci = 64 * (w & 1);
    floatx4 acc[2][4], sum[2][4], s01[2][4], s23[2][4];  // split, chain, chains 0 + 1, 2 + 3
    const auto each = [&](auto f) {
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int b = 0; b < 4; ++b) f(a, b);
    };
    const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
    each([&](int a, int b) { acc[a][b] = sum[a][b] = s01[a][b] = s23[a][b] = zero; });
    const auto product = [&](const bf16* s) {
        bf16x8 fa[2], fb[4];
#pragma unroll
        for (int a = 0; a < 2; ++a) fa[a] = frag(s, LA, co + 16 * a);
#pragma unroll
        for (int b = 0; b < 4; ++b) fb[b] = frag(s + BK * LA, LB, ci + 16 * b);
        each([&](int a, int b) {
            acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[b], fa[a], acc[a][b], 0, 0, 0);
        });
    };
    // four stages on the way to registers, two in LDS in turn
    SplitRows from(ph, g.splits, g.k_split, g.n), at = from;
    constexpr int NS = 4;
    Stage st[NS];
#pragma unroll
    for (int u = 0; u < NS; ++u) {
        load(st[u], from);
        if (!from.end) from.next();
    }
    if (!at.end) store(st[0], lds);
    while (!at.end) {
#pragma unroll
        for (int u = 0; u < NS; ++u) {
            load(st[u], from);
            if (!from.end) from.next();
            __syncthreads();
            product(lds + u % 2 * kStage);
            const int q = at.q, chain = at.chain;
            at.next();
            if (at.q != q) {  // a split is complete
                each([&](int a, int b) {
                    sum[a][b] += acc[a][b];
                    acc[a][b] = zero;
                });
                if (at.end || at.chain != chain) each([&](int a, int b) {
                    (chain < 2 ? s01 : s23)[a][b] += sum[a][b];
                    sum[a][b] = zero;
                });
            }
            if (at.end) break;
            store(st[(u + 1) % NS], lds + (u + 1) % 2 * kStage);
        }
    }
    // lane: column o = l % 16, rows i = 4 (l / 16) + e of each tile
    float* C = g.part_w + (((long)mem * 3 + layer) * 4 + ph) * (H * H);
    each([&](int a, int b) {
        const int o = o0 + co + 16 * a + (l & 15), i = i0 + ci + 16 * b + 4 * (l >> 4);
        *reinterpret_cast<floatx4*>(C + o * H + i) = s01[a][b] + s23[a][b];
    });
}

struct UpdateArgs {
    const float *part_w, *part_b, *part_o, *part_1;
    int splits, rs, l1;
    float *p, *m1, *m2, *grad;
    bf16 *wb, *wbT;
    float lr, b1, b2, eps, c1, c2;
};

// Phase ph of the sum of nb partial sums v[b * width]: those with b % 4 = ph, in four chains
// whose order is fixed (the weight gradients' splits are summed likewise in step_wgrad).
__device__ __forceinline__ float phase_chain(const float* v, long width, int nb, int ph) {
    float s0 = 0.0f, s1 = 0.0f, s2 = 0.0f, s3 = 0.0f;
    int b = ph;
    for (; b + 12 < nb; b += 16) {
        s0 += v[b * width];
        s1 += v[(b + 4) * width];
        s2 += v[(b + 8) * width];
        s3 += v[(b + 12) * width];
    }
    for (; b < nb; b += 4) s0 += v[b * width];
    return (s0 + s1) + (s2 + s3);
}

// Adam on parameter o with gradient g; the new value.
__device__ __forceinline__ float adam_one(const UpdateArgs& u, long o, float gi) {
    const float a = u.b1 * u.m1[o] + (1.0f - u.b1) * gi;
    const float v = u.b2 * u.m2[o] + (1.0f - u.b2) * gi * gi;
    u.m1[o] = a;
    u.m2[o] = v;
    return u.p[o] -= u.lr * (a / u.c1) / (sqrtf(v / u.c2) + u.eps);
}

// Gradients from the partial sums, and Adam on them (or, ADAM false, the gradients alone to
// `grad`). blockIdx.x: 64 tiles of 32 x 32 weights of each hidden layer, then the other
// parameters by 64, four lanes' phases each. A tile's new weights also go out in BF16, as
// they are and transposed through LDS, in the fragments' order.
constexpr int kWTiles = (H / 32) * (H / 32);
constexpr int kL1Blks = (H * F + H) / 64, kBiasBlks = H / 64, kOutBlks = (H + 1 + 63) / 64;
constexpr int kUpdateBlks = 3 * kWTiles + kL1Blks + 3 * kBiasBlks + kOutBlks;
template <bool ADAM>
__global__ __launch_bounds__(256) void step_update(UpdateArgs u) {
    const int t = threadIdx.x, mem = blockIdx.y;
    const long pofs = (long)mem * kP;
    int b = blockIdx.x;
    if (b < 3 * kWTiles) {
        __shared__ bf16 tile[32][36];
        const int layer = b / kWTiles, n0 = b % kWTiles / (H / 32) * 32, k0 = b % (H / 32) * 32;
        const int n = n0 + (t >> 3), k = k0 + 4 * (t & 7);
        const float* v = u.part_w + ((long)mem * 3 + layer) * 4 * (H * H) + n * H + k;
        floatx4 c[4];
#pragma unroll
        for (int ph = 0; ph < 4; ++ph)
            c[ph] = ph < u.splits ? *reinterpret_cast<const floatx4*>(v + ph * (H * H))
                                  : floatx4{0.f, 0.f, 0.f, 0.f};
        const floatx4 s = c[0] + c[1] + c[2] + c[3];
        const long o = pofs + kW2 + layer * (H * H + H) + n * H + k;
        if constexpr (ADAM) {
            bf16x4 h;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                h[e] = (bf16)adam_one(u, o + e, s[e]);
                tile[t >> 3][4 * (t & 7) + e] = h[e];
            }
            const long w0 = ((long)mem * 3 + layer) * (H * H);
            *reinterpret_cast<bf16x4*>(u.wb + w0 + frag_at(n, k)) = h;
            __syncthreads();
#pragma unroll
            for (int e = 0; e < 4; ++e) h[e] = tile[4 * (t & 7) + e][t >> 3];
            *reinterpret_cast<bf16x4*>(u.wbT + w0 + frag_at(k0 + (t >> 3), n0 + 4 * (t & 7))) = h;
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) u.grad[o + e] = s[e];
        }
        return;
    }
    __shared__ float lds[256];
    b -= 3 * kWTiles;
    const float* part;
    int nb, width, ofs;
    if (b < kL1Blks) {
        nb = u.l1;
        width = H * F + H;
        part = u.part_1 + (long)mem * nb * width;
        ofs = kW1;
    } else if (b < kL1Blks + 3 * kBiasBlks) {
        b -= kL1Blks;
        const int layer = b / kBiasBlks;
        b %= kBiasBlks;
        nb = u.rs;
        width = H;
        part = u.part_b + ((long)mem * 3 + layer) * nb * width;
        ofs = kB2 + layer * (H * H + H);
    } else {
        b -= kL1Blks + 3 * kBiasBlks;
        nb = u.rs;
        width = H + 1;
        part = u.part_o + (long)mem * nb * width;
        ofs = kW5;
    }
    const int o = b * 64 + (t & 63);
    lds[t] = phase_chain(part + min(o, width - 1), width, nb, t >> 6);
    __syncthreads();
    if (t >= 64 || o >= width) return;
    const float gi = lds[t] + lds[64 + t] + lds[128 + t] + lds[192 + t];
    if constexpr (ADAM)
        adam_one(u, pofs + ofs + o, gi);
    else
        u.grad[pofs + ofs + o] = gi;
}
