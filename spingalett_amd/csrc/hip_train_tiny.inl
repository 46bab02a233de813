// hip_train_tiny.inl — training of nets that fit one compute unit: any number of steps in one launch.  Part of
// hip_forward.hip's translation unit (included behind hip_train.inl, whose helpers and rules it uses).
//
// A training step of a small net (the reference's exclusive-or example: 2-8-1, four samples, 10,000 epochs) is a chain
// of phases of a few dozen multiplications each.  Launched kernel by kernel it costs 22 launches, about 39 us, whatever
// the sizes; the arithmetic is nothing.  Here one workgroup keeps weights, moments, activations and (where they fit)
// the samples in LDS and walks through the steps; the phases of a step are separated by workgroup barriers, and with 64
// threads (nets whose phases have no more items than that) the barriers cost nothing.  What bounds it is the latency
// of a phase: an LDS read, a short dependent sum, a store, and the branches around them.  2-8-1 with four samples: 39 -> 2.0 us
// per step, 1.5 in sp_train_tiny_one.

namespace {

constexpr uint32_t kTinyLayers = 4;             // weight layers at most
constexpr uint32_t kTinyLds = 156u * 1024u;     // bytes of LDS a workgroup may ask for here

struct TinyArgs {
    uint32_t width[kTinyLayers + 1];
    int act[kTinyLayers];
    uint32_t wofs[kTinyLayers], bofs[kTinyLayers];       // first weight / bias of a layer in the flat arrays
    // LDS offsets (floats): weights, activations (the batch's samples for layer 0, where it is staged), deltas ...
    uint32_t lds_w[kTinyLayers], lds_a[kTinyLayers], lds_d[kTinyLayers];
    uint32_t lds_m, lds_v, lds_g;               // ... moments and gradients, flat: all weights, then all biases
    uint32_t lds_b, lds_z, lds_desc;   // ... biases, logits, what each parameter's gradient reads
    uint32_t lds_x, lds_t, lds_o;               // ... all samples and targets, the sample order of an epoch
    uint32_t lds_tb;                            // ... the batch's targets, where they are staged
    uint32_t ld[kTinyLayers + 1];               // sp_train_tiny_one: floats from row to row of a layer's values and weights
    uint32_t lds_end;                           // ... floats of LDS
    uint32_t total_w, total_b;
    const float *in;                            // weights | biases | mW | mB | vW | vB, flat
    float *out;                                 // the same, then gW | gB (host memory)
    float *dW[kTinyLayers], *dB[kTinyLayers], *dmW, *dvW, *dmB, *dvB, *dgW, *dgB;      // the net's own device arrays
    const float *x, *t;                         // [samples][width]
    const uint32_t *order;                      // [epochs][samples], or nullptr: as they come
    uint32_t samples, batch, epochs;
    OptArgs opt;                                // (its array pointers unused)
    float b1pow, b2pow;                         // beta^t before the first step
    float max_norm;                             // > 0: gradients clipped to this global norm
    int mode;                                   // output deltas: sp_train_out_delta's modes
    int loss_func, sigmoid_out;
    double *loss;                               // sum of the last epoch's per-sample losses, or nullptr
};

// rows are stored with an odd stride: lanes that walk down a column touch different banks
__host__ __device__ constexpr uint32_t tiny_ld(uint32_t w) { return w | 1u; }

// item `i` of a phase over rows of `w` items: quotient and remainder (i < 2^20, w < 2^10: the product is off by less
// than the half that was added)
struct TinyPos {
    uint32_t q, r;
    __device__ TinyPos(uint32_t i, uint32_t w)
    {
        q = (uint32_t)(((float)i + 0.5f) * __builtin_amdgcn_rcpf((float)w));
        r = i - q * w;
    }
};

template <int T>
__device__ __forceinline__ double tiny_block_sum(double v, double *red)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, kWave);
    if constexpr (T > 64) {
        __syncthreads();
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
        __syncthreads();
        v = 0.0;
#pragma unroll
        for (int w = 0; w < T / 64; ++w) v += red[w];
    }
    return v;
}

// Sums over k in the order of the kernels that a batch of up to four samples takes launch by launch, so that small
// problems train to the same bits either way: a layer's sum in chains of four (sp_gemv), two of them in flight ...
__device__ __forceinline__ float tiny_row_dot(const float *w, const float *a, uint32_t K)
{
    float s[2] = {0.0f, 0.0f};
    uint32_t k = 0;
    for (; k + 8u <= K; k += 8u) {
        float wv[8], av[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) { wv[u] = w[k + u]; av[u] = a[k + u]; }
#pragma unroll
        for (int u = 0; u < 8; ++u) s[u >> 2] = fmaf(wv[u], av[u], s[u >> 2]);
    }
    if (K % 4u == 0) {
        for (; k < K; ++k) s[0] = fmaf(w[k], a[k], s[0]);
    } else {
        for (; k < K; ++k) s[k & 1u] = fmaf(w[k], a[k], s[k & 1u]);
    }
    return s[0] + s[1];
}

// ... deltas and gradients in one chain (the matrix instructions)
__device__ __forceinline__ float tiny_chain(const float *a, uint32_t as, const float *b, uint32_t bs, uint32_t K)
{
    float s = 0.0f;
    uint32_t k = 0;
    for (; k + 4u <= K; k += 4u) {
        float av[4], bv[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) { av[u] = a[(k + u) * as]; bv[u] = b[(k + u) * bs]; }
#pragma unroll
        for (int u = 0; u < 4; ++u) s = fmaf(av[u], bv[u], s);
    }
    for (; k < K; ++k) s = fmaf(a[k * as], b[k * bs], s);
    return s;
}

// ... and bias gradients in four (sp_train_colsum_part)
__device__ __forceinline__ float tiny_colsum(const float *d, uint32_t ld, uint32_t n)
{
    float s[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    uint32_t i = 0;
    for (; i + 4u <= n; i += 4u) {
#pragma unroll
        for (int u = 0; u < 4; ++u) s[u] += d[(i + u) * ld];
    }
#pragma unroll
    for (uint32_t u = 0; u < 3u; ++u)
        if (i + u < n) s[u] += d[(i + u) * ld];
    return (s[0] + s[1]) + (s[2] + s[3]);
}

// one output's share of a sample's loss (compute_sample_loss, SIMD.c:522-552)
__device__ __forceinline__ double tiny_loss(const TinyArgs &g, float a, float t)
{
    if (g.loss_func == 0) {
        const float d = a - t;
        return (double)(d * d);
    }
    if (g.sigmoid_out) {
        float c = a < 1e-9f ? 1e-9f : a;
        c = c > 1.0f - 1e-9f ? 1.0f - 1e-9f : c;
        return -(double)(t * logf(c) + (1.0f - t) * logf(1.0f - c));
    }
    return -(double)(t * logf(a < 1e-9f ? 1e-9f : a));
}

// a softmax's output r of n logits, its target, and its delta
__device__ __forceinline__ float tiny_soft_delta(const float *z, const float *tr, uint32_t n, uint32_t r, int mode, float &a, float &t)
{
    float m = z[0];
    for (uint32_t k = 1; k < n; ++k) m = fmaxf(m, z[k]);
    float sum = 0.0f;
    for (uint32_t k = 0; k < n; ++k) sum += expf(z[k] - m);
    const float inv = sum > 0.0f ? 1.0f / sum : 1.0f;
    a = expf(z[r] - m) * inv;
    t = tr[r];
    if (mode != 0) return a - t;
    float c = 0.0f;
    for (uint32_t k = 0; k < n; ++k) { const float ak = expf(z[k] - m) * inv; c += (ak - tr[k]) * ak; }
    return a * ((a - t) - c);
}

// T threads, NL weight layers (compile-time, so that the layers' sizes and offsets live in scalar registers: read from
// the argument block by a layer index they cost a scalar load each, more than the phase itself)
template <int T, int NL>
__global__ __launch_bounds__(T) void sp_train_tiny(const TinyArgs g)
{
    extern __shared__ __attribute__((aligned(16))) float L[];
    __shared__ double red[16];
    const uint32_t tid = threadIdx.x, total = g.total_w + g.total_b;
    const uint32_t n_in = g.width[0], n_out = g.width[NL], ldx = tiny_ld(n_in), ldo = tiny_ld(n_out);
    const bool x_lds = g.lds_x != 0u, staged = g.order || !x_lds;
    uint32_t *Lu = reinterpret_cast<uint32_t *>(L);

    // everything into LDS, and for every parameter what its gradient multiplies: delta column, activation column
    // (weights), where the parameter itself lies, its layer
#pragma unroll
    for (int l = 0; l < NL; ++l) {
        const uint32_t K = g.width[l], N = g.width[l + 1], ld = tiny_ld(K);
        for (uint32_t p = tid; p < K * N; p += T) {
            const TinyPos o(p, K);
            L[g.lds_w[l] + o.q * ld + o.r] = g.in[g.wofs[l] + p];
            Lu[g.lds_desc + 2u * (g.wofs[l] + p)] = (g.lds_d[l] + o.q) | (g.lds_a[l] + o.r) << 16;
            Lu[g.lds_desc + 2u * (g.wofs[l] + p) + 1u] = (g.lds_w[l] + o.q * ld + o.r) | (uint32_t)l << 16;
        }
        for (uint32_t j = tid; j < N; j += T) {
            L[g.lds_b + g.bofs[l] + j] = g.in[g.total_w + g.bofs[l] + j];
            Lu[g.lds_desc + 2u * (g.total_w + g.bofs[l] + j)] = (g.lds_d[l] + j);
            Lu[g.lds_desc + 2u * (g.total_w + g.bofs[l] + j) + 1u] = (g.lds_b + g.bofs[l] + j) | (uint32_t)l << 16 | 1u << 24;
        }
    }
    for (uint32_t p = tid; p < total; p += T) {
        L[g.lds_m + p] = g.in[total + p];
        L[g.lds_v + p] = g.in[2u * total + p];
        L[g.lds_g + p] = 0.0f;
    }
    if (x_lds) {
        for (uint32_t p = tid; p < g.samples * n_in; p += T) {
            const TinyPos o(p, n_in);
            L[g.lds_x + o.q * ldx + o.r] = g.x[p];
        }
        for (uint32_t p = tid; p < g.samples * n_out; p += T) {
            const TinyPos o(p, n_out);
            L[g.lds_t + o.q * ldo + o.r] = g.t[p];
        }
    }

    float b1pow = g.b1pow, b2pow = g.b2pow;
    double loss = 0.0;
    OptArgs opt = g.opt;
    const float decay = g.opt.decay;
    const bool soft = g.act[NL - 1] == A_SOFTMAX, clip = g.max_norm > 0.0f;
    __syncthreads();
    // this thread's first parameter: its record stays in registers
    const uint2 desc0 = tid < total ? *reinterpret_cast<const uint2 *>(Lu + g.lds_desc + 2u * tid) : make_uint2(0u, 0u);

    for (uint32_t epoch = 0; epoch < g.epochs; ++epoch) {
        const bool want_loss = g.loss && epoch + 1u == g.epochs;
        if (g.order) {
            __syncthreads();
            for (uint32_t p = tid; p < g.samples; p += T) Lu[g.lds_o + p] = g.order[(size_t)epoch * g.samples + p];
        }
        for (uint32_t first = 0; first < g.samples; first += g.batch) {
            const uint32_t n = g.samples - first < g.batch ? g.samples - first : g.batch;
            // the batch's samples and targets: where they lie, or gathered
            uint32_t xo = g.lds_x + first * ldx, to = g.lds_t + first * ldo;
            if (staged) {
                xo = g.lds_a[0];
                to = g.lds_tb;
                __syncthreads();
                for (uint32_t p = tid; p < n * n_in; p += T) {
                    const TinyPos o(p, n_in);
                    const uint32_t r = g.order ? Lu[g.lds_o + first + o.q] : first + o.q;
                    L[xo + o.q * ldx + o.r] = x_lds ? L[g.lds_x + r * ldx + o.r] : g.x[(size_t)r * n_in + o.r];
                }
                for (uint32_t p = tid; p < n * n_out; p += T) {
                    const TinyPos o(p, n_out);
                    const uint32_t r = g.order ? Lu[g.lds_o + first + o.q] : first + o.q;
                    L[to + o.q * ldo + o.r] = x_lds ? L[g.lds_t + r * ldo + o.r] : g.t[(size_t)r * n_out + o.r];
                }
            }
            b1pow *= opt.b1;
            b2pow *= opt.b2;
            opt.mf = 1.0f / (1.0f - b1pow);
            opt.vf = 1.0f / (1.0f - b2pow);
            auto add_loss = [&](float a, float t) { loss += tiny_loss(g, a, t); };

            // forward; without a softmax the last layer's threads go straight on to their deltas
#pragma unroll
            for (int l = 0; l < NL; ++l) {
                __syncthreads();
                const uint32_t K = g.width[l], N = g.width[l + 1], ld = tiny_ld(K), ldn = tiny_ld(N);
                const uint32_t ao = l == 0 ? xo : g.lds_a[l];
                for (uint32_t p = tid; p < n * N; p += T) {
                    const TinyPos o(p, N);
                    const float z = tiny_row_dot(L + g.lds_w[l] + o.r * ld, L + ao + o.q * ld, K) + L[g.lds_b + g.bofs[l] + o.r];
                    if (l + 1 < NL) {
                        L[g.lds_a[l + 1 < NL ? l + 1 : 0] + o.q * ldn + o.r] = apply_act(z, g.act[l]);
                    } else if (soft) {
                        L[g.lds_z + o.q * ldn + o.r] = z;
                    } else {
                        const float a = apply_act(z, g.act[l]), t = L[to + o.q * ldo + o.r], diff = a - t;
                        L[g.lds_d[l] + o.q * ldn + o.r] = g.mode == 1 ? diff : diff * act_derivative(a, g.act[l]);
                        if (want_loss) add_loss(a, t);
                    }
                }
            }
            if (soft) {
                __syncthreads();
                for (uint32_t p = tid; p < n * n_out; p += T) {
                    const TinyPos o(p, n_out);
                    float a, t;
                    L[g.lds_d[NL - 1] + o.q * ldo + o.r] = tiny_soft_delta(L + g.lds_z + o.q * ldo, L + to + o.q * ldo, n_out, o.r, g.mode, a, t);
                    if (want_loss) add_loss(a, t);
                }
            }

            // hidden deltas
#pragma unroll
            for (int l = NL - 1; l > 0; --l) {
                __syncthreads();
                const uint32_t K = g.width[l], N = g.width[l + 1], ld = tiny_ld(K), ldn = tiny_ld(N);
                for (uint32_t p = tid; p < n * K; p += T) {
                    const TinyPos o(p, K);
                    const float s = tiny_chain(L + g.lds_d[l] + o.q * ldn, 1u, L + g.lds_w[l] + o.r, ld, N);
                    L[g.lds_d[l - 1] + o.q * ld + o.r] = s * act_derivative(L[g.lds_a[l] + o.q * ld + o.r], g.act[l - 1]);
                }
            }

            // gradients; unless they are clipped first, each thread updates the parameter whose gradient it has formed
            const float gscale = 1.0f / (float)n;
            double sq = 0.0;
            __syncthreads();
            auto finish = [&](uint32_t p, uint32_t at, bool bias, float grad) {
                float w = L[at], m = L[g.lds_m + p], v = L[g.lds_v + p];
                opt.decay = bias ? 0.0f : decay;
                opt_update(opt, w, grad, m, v);
                L[at] = w;
                L[g.lds_m + p] = m;
                L[g.lds_v + p] = v;
                L[g.lds_g + p] = grad;
            };
            uint2 desc = desc0;
            for (uint32_t p = tid; p < total; p += T) {
                if (p != tid) desc = *reinterpret_cast<const uint2 *>(Lu + g.lds_desc + 2u * p);
                const uint32_t layer = desc.y >> 16 & 255u;
                const bool bias = desc.y >> 24 != 0u;
                uint32_t ld_d = tiny_ld(g.width[1]), ld_a = ldx, ao = desc.x >> 16;
#pragma unroll
                for (int l = 1; l < NL; ++l) {
                    ld_d = layer == (uint32_t)l ? tiny_ld(g.width[l + 1]) : ld_d;
                    ld_a = layer == (uint32_t)l ? tiny_ld(g.width[l]) : ld_a;
                }
                if (layer == 0u) ao += xo - g.lds_a[0];
                const float *d = L + (desc.x & 0xFFFFu);
                const float grad = (bias ? tiny_colsum(d, ld_d, n) : tiny_chain(d, ld_d, L + ao, ld_a, n)) * gscale;
                if (clip) {
                    L[g.lds_g + p] = grad;
                    sq += (double)grad * (double)grad;
                } else {
                    finish(p, desc.y & 0xFFFFu, bias, grad);
                }
            }
            if (clip) {
                const float norm = sqrtf((float)tiny_block_sum<T>(sq, red));
                const float f = norm > g.max_norm ? g.max_norm / norm : 1.0f;
                for (uint32_t p = tid; p < total; p += T) {
                    const uint32_t d = Lu[g.lds_desc + 2u * p + 1u];
                    finish(p, d & 0xFFFFu, d >> 24 != 0u, L[g.lds_g + p] * f);
                }
            }
        }
    }

    // results: to the net's device arrays, and flat into host memory
    __syncthreads();
#pragma unroll
    for (int l = 0; l < NL; ++l) {
        const uint32_t K = g.width[l], cnt = K * g.width[l + 1], ld = tiny_ld(K);
        for (uint32_t p = tid; p < cnt; p += T) {
            const TinyPos o(p, K);
            const float w = L[g.lds_w[l] + o.q * ld + o.r];
            g.dW[l][p] = w;
            g.out[g.wofs[l] + p] = w;
        }
        for (uint32_t j = tid; j < g.width[l + 1]; j += T) {
            const float b = L[g.lds_b + g.bofs[l] + j];
            g.dB[l][j] = b;
            g.out[g.total_w + g.bofs[l] + j] = b;
        }
    }
    for (uint32_t p = tid; p < total; p += T) {
        const bool w = p < g.total_w;
        const uint32_t q = w ? p : p - g.total_w;
        const float m = L[g.lds_m + p], v = L[g.lds_v + p], gr = L[g.lds_g + p];
        (w ? g.dmW : g.dmB)[q] = m;
        (w ? g.dvW : g.dvB)[q] = v;
        (w ? g.dgW : g.dgB)[q] = gr;
        g.out[total + p] = m;
        g.out[2u * total + p] = v;
        g.out[3u * total + p] = gr;
    }
    if (g.loss) {
        const double sum = tiny_block_sum<T>(loss, red);
        if (tid == 0) *g.loss = sum;
    }
}

// The same training where every phase has at most one item a thread and every thread at most one parameter.  A step of such a
// net is a few hundred instructions, and what it cost in the kernel above was its branches: the rests of sums term by
// term, each waiting for LDS in turn, loops of one round, places worked out anew in each phase.  Here rows are padded with
// zeros to whole groups of four, which change no sum, every place is a pointer worked out once, a thread's parameter and
// its moments stay in registers, and the corrections of the moments are formed for 64 steps at a time, one a lane.
// A step of 2-8-1 with 4 / 70 samples 2.2 / 6.0 -> 1.5 / 3.2 us, of 7-5-3 with 16 and a softmax 4.3 -> 2.3, of 13-29-17-3
// with 16 9.3 -> 4.0, of 16-16-4 with one 2.7 -> 1.7 (a two-hundredth of a call's 50 us among them).
constexpr uint32_t kTinyOne = 1024u;            // items and parameters at most

// as tiny_row_dot, rows padded with zeros to a multiple of four
__device__ __forceinline__ float tiny_padded_dot(const float *w, const float *a, uint32_t K)
{
    float s0 = 0.0f, s1 = 0.0f;
    uint32_t k = 0;
    for (; k + 8u <= K; k += 8u) {
        float wv[8], av[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) { wv[u] = w[k + u]; av[u] = a[k + u]; }
#pragma unroll
        for (int u = 0; u < 4; ++u) { s0 = fmaf(wv[u], av[u], s0); s1 = fmaf(wv[4 + u], av[4 + u], s1); }
    }
    if (const uint32_t left = K - k) {
        float wv[8], av[8];
#pragma unroll
        for (int u = 0; u < 4; ++u) { wv[u] = w[k + u]; av[u] = a[k + u]; }
        if (left == 4u) {
#pragma unroll
            for (int u = 0; u < 4; ++u) s0 = fmaf(wv[u], av[u], s0);
        } else {
            s0 = fmaf(wv[2], av[2], fmaf(wv[0], av[0], s0));
            s1 = fmaf(wv[3], av[3], fmaf(wv[1], av[1], s1));
            if (left > 4u) {
#pragma unroll
                for (int u = 4; u < 8; ++u) { wv[u] = w[k + u]; av[u] = a[k + u]; }
                s0 = fmaf(wv[6], av[6], fmaf(wv[4], av[4], s0));
                s1 = fmaf(wv[7], av[7], fmaf(wv[5], av[5], s1));
            }
        }
    }
    return s0 + s1;
}

// Gradient of a weight (tiny_chain over the batch) or of a bias (tiny_colsum) side by side: lanes of one wave need either
__device__ __forceinline__ float tiny_gradient(const float *d, uint32_t ds, const float *a, uint32_t as, uint32_t n, bool bias)
{
    float s = 0.0f, c[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    uint32_t i = 0;
    for (; i + 4u <= n; i += 4u) {
        float dv[4], av[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) { dv[u] = *d; av[u] = *a; d += ds; a += as; }
#pragma unroll
        for (int u = 0; u < 4; ++u) { s = fmaf(dv[u], av[u], s); c[u] += dv[u]; }
    }
    if (const uint32_t left = n - i) {
        float dv[3], av[3];
#pragma unroll
        for (uint32_t u = 0; u < 3u; ++u) { const uint32_t at = u < left ? u : 0u; dv[u] = d[at * ds]; av[u] = a[at * as]; }
#pragma unroll
        for (uint32_t u = 0; u < 3u; ++u) { s = u < left ? fmaf(dv[u], av[u], s) : s; c[u] = u < left ? c[u] + dv[u] : c[u]; }
    }
    return bias ? (c[0] + c[1]) + (c[2] + c[3]) : s;
}

// apply_act and act_derivative with the smooth activations, which small nets have, asked for first: each question is a branch
__device__ __forceinline__ float tiny_act(float x, int act)
{
    if (__builtin_expect(act == A_TANH, 1)) return tanh_straight(x);
    if (__builtin_expect(act == A_SIGMOID, 1)) return 1.0f / (1.0f + expf(-x));
    return apply_act(x, act);
}

__device__ __forceinline__ float tiny_derivative(float a, int act)
{
    if (__builtin_expect(act == A_TANH, 1)) return 1.0f - a * a;
    if (__builtin_expect(act == A_SIGMOID, 1)) return a * (1.0f - a);
    return act_derivative(a, act);
}

template <int T, int NL>
__global__ __launch_bounds__(T) void sp_train_tiny_one(const TinyArgs g)
{
    extern __shared__ __attribute__((aligned(16))) float L[];
    __shared__ double red[16];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, total = g.total_w + g.total_b;
    const uint32_t n_in = g.width[0], n_out = g.width[NL], ldx = g.ld[0], ldo = g.ld[NL];
    const bool x_lds = g.lds_x != 0u, staged = g.order || !x_lds;
    const bool soft = g.act[NL - 1] == A_SOFTMAX, clip = g.max_norm > 0.0f;
    uint32_t *Lu = reinterpret_cast<uint32_t *>(L);

    for (uint32_t p = tid; p < g.lds_end; p += T) L[p] = 0.0f;
    __syncthreads();
    if (x_lds) {
        for (uint32_t p = tid; p < g.samples * n_in; p += T) {
            const TinyPos o(p, n_in);
            L[g.lds_x + o.q * ldx + o.r] = g.x[p];
        }
        for (uint32_t p = tid; p < g.samples * n_out; p += T) {
            const TinyPos o(p, n_out);
            L[g.lds_t + o.q * ldo + o.r] = g.t[p];
        }
    }
    // this thread's parameter: where it lies, what its gradient multiplies, its own values
    float *par = L;
    const float *par_d = L, *par_a = L;
    uint32_t par_ld_d = 0, par_ld_a = 0;
    bool bias = false, input = false;
    float w = 0.0f, m = 0.0f, v = 0.0f, grad = 0.0f;
    if (tid < total) {
#pragma unroll
        for (int l = 0; l < NL; ++l) {
            const uint32_t K = g.width[l], N = g.width[l + 1], p = tid - g.wofs[l], j = tid - g.total_w - g.bofs[l];
            if (tid < g.total_w && tid >= g.wofs[l] && p < K * N) {
                const TinyPos o(p, K);
                par = L + g.lds_w[l] + o.q * g.ld[l] + o.r;
                par_d = L + g.lds_d[l] + o.q;
                par_a = l ? L + g.lds_a[l] + o.r : L + o.r;
                par_ld_d = g.ld[l + 1];
                par_ld_a = g.ld[l];
                input = l == 0;
            } else if (tid >= g.total_w + g.bofs[l] && j < N) {
                par = L + g.lds_b + g.bofs[l] + j;
                par_d = par_a = L + g.lds_d[l] + j;
                par_ld_d = par_ld_a = g.ld[l + 1];
                bias = true;
            }
        }
        w = g.in[tid];
        m = g.in[total + tid];
        v = g.in[2u * total + tid];
        *par = w;
    }
    // its items of the phases: forward (row of weights, row of inputs, bias, output), hidden deltas (row of deltas, column of
    // weights, the value, output)
    struct Fwd { const float *w, *a, *b; float *out; uint32_t q; } fwd[NL];
    struct Back { const float *d, *w, *a; float *out; } back[NL];
#pragma unroll
    for (int l = 0; l < NL; ++l) {
        const uint32_t N = g.width[l + 1];
        TinyPos o(tid, N);
        if (tid >= N * g.batch) o.q = o.r = 0u;
        fwd[l].w = L + g.lds_w[l] + o.r * g.ld[l];
        fwd[l].a = L + (l ? g.lds_a[l] : 0u) + o.q * g.ld[l];
        fwd[l].b = L + g.lds_b + g.bofs[l] + o.r;
        fwd[l].out = L + (l + 1 < NL ? g.lds_a[l + 1 < NL ? l + 1 : 0] : g.lds_d[l]) + o.q * g.ld[l + 1] + o.r;
        fwd[l].q = o.q * g.ld[l + 1] + o.r;
        if (l == 0) continue;
        TinyPos i(tid, g.width[l]);
        if (tid >= g.width[l] * g.batch) i.q = i.r = 0u;
        back[l].d = L + g.lds_d[l] + i.q * g.ld[l + 1];
        back[l].w = L + g.lds_w[l] + i.r;
        back[l].a = L + g.lds_a[l] + i.q * g.ld[l] + i.r;
        back[l].out = L + g.lds_d[l - 1] + i.q * g.ld[l] + i.r;
    }

    float b1pow = g.b1pow, b2pow = g.b2pow, mf = 0.0f, vf = 0.0f;
    double loss = 0.0;
    OptArgs opt = g.opt;
    opt.decay = bias ? 0.0f : g.opt.decay;
    const float batch_scale = 1.0f / (float)g.batch;
    uint32_t step = 0;
    for (uint32_t epoch = 0; epoch < g.epochs; ++epoch) {
        const bool want_loss = g.loss && epoch + 1u == g.epochs;
        if (g.order) {
            __syncthreads();
            for (uint32_t p = tid; p < g.samples; p += T) Lu[g.lds_o + p] = g.order[(size_t)epoch * g.samples + p];
        }
        for (uint32_t first = 0; first < g.samples; first += g.batch, ++step) {
            const uint32_t n = g.samples - first < g.batch ? g.samples - first : g.batch;
            uint32_t xo = g.lds_x + first * ldx, to = g.lds_t + first * ldo;
            if (staged) {
                xo = g.lds_a[0];
                to = g.lds_tb;
                __syncthreads();
                for (uint32_t p = tid; p < n * n_in; p += T) {
                    const TinyPos o(p, n_in);
                    const uint32_t r = g.order ? Lu[g.lds_o + first + o.q] : first + o.q;
                    L[xo + o.q * ldx + o.r] = x_lds ? L[g.lds_x + r * ldx + o.r] : g.x[(size_t)r * n_in + o.r];
                }
                for (uint32_t p = tid; p < n * n_out; p += T) {
                    const TinyPos o(p, n_out);
                    const uint32_t r = g.order ? Lu[g.lds_o + first + o.q] : first + o.q;
                    L[to + o.q * ldo + o.r] = x_lds ? L[g.lds_t + r * ldo + o.r] : g.t[(size_t)r * n_out + o.r];
                }
            }
            if (step % 64u == 0u) {
                // beta^t of the next 64 steps, one a lane, each the product of as many factors as the host's
                float p1 = 0.0f, p2 = 0.0f;
                for (uint32_t i = 0; i < 64u; ++i) {
                    b1pow *= opt.b1;
                    b2pow *= opt.b2;
                    p1 = i == lane ? b1pow : p1;
                    p2 = i == lane ? b2pow : p2;
                }
                mf = 1.0f / (1.0f - p1);
                vf = 1.0f / (1.0f - p2);
            }
            opt.mf = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, mf), (int)(step % 64u)));
            opt.vf = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, vf), (int)(step % 64u)));
            auto add_loss = [&](float a, float t) { loss += tiny_loss(g, a, t); };

            // forward; without a softmax the last layer's threads go straight on to their deltas
#pragma unroll
            for (int l = 0; l < NL; ++l) {
                __syncthreads();
                if (tid < n * g.width[l + 1]) {
                    const float z = tiny_padded_dot(fwd[l].w, l ? fwd[l].a : fwd[l].a + xo, g.width[l]) + *fwd[l].b;
                    if (l + 1 < NL) {
                        *fwd[l].out = tiny_act(z, g.act[l]);
                    } else if (soft) {
                        L[g.lds_z + fwd[l].q] = z;
                    } else {
                        const float a = tiny_act(z, g.act[l]), t = L[to + fwd[l].q], diff = a - t;
                        *fwd[l].out = g.mode == 1 ? diff : diff * tiny_derivative(a, g.act[l]);
                        if (want_loss) add_loss(a, t);
                    }
                }
            }
            if (soft) {
                __syncthreads();
                if (tid < n * n_out) {
                    const TinyPos o(tid, n_out);
                    float a, t;
                    *fwd[NL - 1].out = tiny_soft_delta(L + g.lds_z + o.q * ldo, L + to + o.q * ldo, n_out, o.r, g.mode, a, t);
                    if (want_loss) add_loss(a, t);
                }
            }

            // hidden deltas
#pragma unroll
            for (int l = NL - 1; l > 0; --l) {
                __syncthreads();
                if (tid < n * g.width[l]) {
                    const float *wc = back[l].w;
                    float s = 0.0f;
                    for (uint32_t k = 0; k < g.width[l + 1]; k += 4u) {
                        float dv[4], wv[4];
#pragma unroll
                        for (int u = 0; u < 4; ++u) { dv[u] = back[l].d[k + u]; wv[u] = *wc; wc += g.ld[l]; }
#pragma unroll
                        for (int u = 0; u < 4; ++u) s = fmaf(dv[u], wv[u], s);
                    }
                    *back[l].out = s * tiny_derivative(*back[l].a, g.act[l - 1]);
                }
            }

            // gradients and updates
            __syncthreads();
            double sq = 0.0;
            if (tid < total) {
                grad = tiny_gradient(par_d, par_ld_d, input ? par_a + xo : par_a, par_ld_a, n, bias) * (n == g.batch ? batch_scale : 1.0f / (float)n);
                if (clip) sq = (double)grad * (double)grad;
            }
            if (clip) {
                const float norm = sqrtf((float)tiny_block_sum<T>(sq, red));
                grad *= norm > g.max_norm ? g.max_norm / norm : 1.0f;
            }
            if (tid < total) {
                opt_update(opt, w, grad, m, v);
                *par = w;
            }
        }
    }

    // results: to the net's device arrays, and flat into host memory
    if (tid < total) {
        const bool is_w = tid < g.total_w;
        const uint32_t q = is_w ? tid : tid - g.total_w;
#pragma unroll
        for (int l = 0; l < NL; ++l) {
            const uint32_t at = q - (is_w ? g.wofs[l] : g.bofs[l]);
            if (at < (is_w ? g.width[l] : 1u) * g.width[l + 1]) (is_w ? g.dW : g.dB)[l][at] = w;
        }
        (is_w ? g.dmW : g.dmB)[q] = m;
        (is_w ? g.dvW : g.dvB)[q] = v;
        (is_w ? g.dgW : g.dgB)[q] = grad;
        g.out[tid] = w;
        g.out[total + tid] = m;
        g.out[2u * total + tid] = v;
        g.out[3u * total + tid] = grad;
    }
    if (g.loss) {
        const double sum = tiny_block_sum<T>(loss, red);
        if (tid == 0) *g.loss = sum;
    }
}

// LDS layout of a net and batch; false where the net belongs to the launch-by-launch step
struct TinyPlan {
    TinyArgs a;
    uint32_t lds_floats;
    bool x_lds, one;
    uint32_t threads, nl;
};

// one: for sp_train_tiny_one, rows and columns of weights padded to whole groups of four
bool tiny_layout(uint32_t layers, const uint32_t *topo, uint32_t samples, uint32_t batch, bool ordered, bool one, TinyPlan *out)
{
    auto row = [&](uint32_t w) { return one ? ((w + 3u) & ~3u) + 1u : tiny_ld(w); };
    if (layers < 2 || layers - 1u > kTinyLayers || batch == 0 || batch > samples) return false;
    TinyPlan p{};
    TinyArgs &a = p.a;
    p.nl = layers - 1u;
    uint64_t w = 0, b = 0, widest = 0;
    for (uint32_t l = 0; l < layers; ++l) {
        if (topo[l] > 512u) return false;
        a.width[l] = topo[l];
        a.ld[l] = row(topo[l]);
        if (topo[l] > widest) widest = topo[l];
        if (!l) continue;
        a.wofs[l - 1u] = (uint32_t)w;
        a.bofs[l - 1u] = (uint32_t)b;
        w += (uint64_t)topo[l - 1u] * topo[l];
        b += topo[l];
    }
    // One compute unit multiplies and adds about 16 pairs per cycle from LDS, in three products per step: a quarter of
    // a million weight-sample pairs take as long as the launches they replace (48-48-10 with 94 samples 26 against 57 us per
    // step, with 11 samples 8 against 45; 12-12-3 with 1456 samples, few parameters with long sums, 75 against 74).
    if (w * batch > (256u << 10)) return false;
    a.total_w = (uint32_t)w;
    a.total_b = (uint32_t)b;
    uint64_t at = 2;                                      // (offset 0 means "not there")
    auto take = [&](uint64_t floats) { const uint64_t o = at; at += floats; return (uint32_t)o; };
    if (!one) a.lds_desc = take(2u * (w + b));
    const uint64_t x = (uint64_t)samples * row(topo[0]), t = (uint64_t)samples * row(topo[p.nl]);
    const uint64_t xb = (uint64_t)batch * row(topo[0]), tb = (uint64_t)batch * row(topo[p.nl]);
    for (uint32_t l = 0; l < p.nl; ++l) {
        a.lds_w[l] = take((uint64_t)row(topo[l]) * (one ? (topo[l + 1] + 3u) & ~3u : topo[l + 1]));
        a.lds_d[l] = take((uint64_t)batch * row(topo[l + 1]));
        if (l) a.lds_a[l] = take((uint64_t)batch * row(topo[l]));
    }
    a.lds_z = take(tb);
    a.lds_b = take(b);
    if (!one) {
        a.lds_m = take(w + b);
        a.lds_v = take(w + b);
        a.lds_g = take(w + b);
    }
    if (ordered) a.lds_o = take(samples);
    // all samples in LDS where they fit (with room for a gathered batch if there is an order), else batch by batch
    p.x_lds = (at + x + t + (ordered ? xb + tb : 0)) * sizeof(float) <= kTinyLds;
    if (p.x_lds) {
        a.lds_x = take(x);
        a.lds_t = take(t);
    }
    if (p.x_lds && !ordered) a.lds_a[0] = a.lds_x;        // (never written: the base that gradient records are relative to)
    else { a.lds_a[0] = take(xb); a.lds_tb = take(tb); }
    if (at * sizeof(float) > kTinyLds) return false;
    // one wave where the phases hold a round or two of it, sixteen where they hold many
    uint64_t items = widest * batch;
    if (w + b > items) items = w + b;
    if (one && items > kTinyOne) return false;
    p.one = one;
    p.threads = items <= (one ? 64u : 128u) ? 64u : items <= (one ? 256u : 1024u) ? 256u : 1024u;
    a.lds_end = (uint32_t)at;
    p.lds_floats = (uint32_t)at;
    *out = p;
    return true;
}

bool tiny_plan(uint32_t layers, const uint32_t *topo, uint32_t samples, uint32_t batch, bool ordered, TinyPlan *out)
{
    if (!tiny_layout(layers, topo, samples, batch, ordered, false, out)) return false;
    // (the samples in LDS or not as without the padding: trainings are cut into launches by that)
    TinyPlan one;
    if (tiny_layout(layers, topo, samples, batch, ordered, true, &one) && one.x_lds == out->x_lds) *out = one;
    return true;
}

template <int T, int NL>
int launch_tiny_inst(const TinyPlan &p, size_t lds)
{
    if (p.one) {
        auto kern = sp_train_tiny_one<T, NL>;
        static bool once = ((void)hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kTinyLds), true);
        (void)once;
        kern<<<1, T, lds, g_stream>>>(p.a);
        HCHECK(hipGetLastError());
        return 0;
    }
    auto kern = sp_train_tiny<T, NL>;
    static bool once = ((void)hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kTinyLds), true);
    (void)once;
    kern<<<1, T, lds, g_stream>>>(p.a);
    HCHECK(hipGetLastError());
    return 0;
}

template <int T>
int launch_tiny(const TinyPlan &p)
{
    const size_t lds = (size_t)p.lds_floats * sizeof(float);
    switch (p.nl) {
    case 1:  return launch_tiny_inst<T, 1>(p, lds);
    case 2:  return launch_tiny_inst<T, 2>(p, lds);
    case 3:  return launch_tiny_inst<T, 3>(p, lds);
    default: return launch_tiny_inst<T, 4>(p, lds);
    }
}

}  // namespace

extern "C" {

bool sp_train_tiny_fits(uint32_t layers, const uint32_t *topology, uint32_t samples, uint32_t batch, bool ordered)
{
    TinyPlan p;
    return tiny_plan(layers, topology, samples, batch, ordered, &p);
}

int sp_train_tiny_run(sphip_net *net, const sp_tiny_run *r)
{
    if (!net || !net->train) return fail_msg("sp_train_tiny_run: sphip_train_begin was not called for this net");
    sphip_train_state *ts = net->train;
    TinyPlan p;
    if (!tiny_plan(net->layers, net->topo.data(), r->samples, r->batch, r->order != nullptr, &p))
        return fail_msg("sp_train_tiny_run: the net does not fit");
    // (an epoch whose samples fit LDS is never too long for a launch: its steps are a few ten thousand at most)
    if (r->count != r->samples && (p.x_lds || r->epochs != 1u || r->start % r->batch || (uint64_t)r->start + r->count > r->samples))
        return fail_msg("sp_train_tiny_run: not a part of one epoch");
    TinyArgs &a = p.a;
    const uint32_t n_in = net->topo[0], n_out = net->topo[net->layers - 1];
    const uint64_t total = (uint64_t)a.total_w + a.total_b;
    const uint64_t xf = (uint64_t)r->samples * n_in, tf = (uint64_t)r->samples * n_out;
    const uint64_t of = r->order ? (uint64_t)r->epochs * r->count : 0;
    // pinned: loss (two floats) | results (4 arrays) | state (3 arrays) | order | samples | targets
    const uint64_t in_at = 2u + 4u * total, ord_at = in_at + 3u * total, data_at = ord_at + (r->order ? r->order_room : 0u);
    if (of > data_at - ord_at) return fail_msg("sp_train_tiny_run: more sample numbers than announced");
    if (r->first && grow_pinned(&ts->tiny_pin, &ts->tiny_cap, data_at + (p.x_lds ? xf + tf : 0u))) return 1;
    float *pin = ts->tiny_pin;
    if (r->first) {
        float *s = pin + in_at;
        memcpy(s, r->weights, (size_t)a.total_w * 4u);
        memcpy(s + a.total_w, r->biases, (size_t)a.total_b * 4u);
        memcpy(s + total, r->m_weights, (size_t)a.total_w * 4u);
        memcpy(s + total + a.total_w, r->m_biases, (size_t)a.total_b * 4u);
        memcpy(s + 2u * total, r->v_weights, (size_t)a.total_w * 4u);
        memcpy(s + 2u * total + a.total_w, r->v_biases, (size_t)a.total_b * 4u);
        if (p.x_lds) {
            memcpy(pin + data_at, r->x, xf * 4u);
            memcpy(pin + data_at + xf, r->t, tf * 4u);
        } else {
            if (grow(&net->stage_x, &net->stage_x_cap, xf) || grow(&net->stage_y, &net->stage_y_cap, tf)) return 1;
            if (upload_from_host(net->stage_x, r->x, xf * 4u) || upload_from_host(net->stage_y, r->t, tf * 4u)) return 1;
        }
    }
    a.in = r->first ? pin + in_at : pin + 2;
    a.out = pin + 2;
    const uint64_t skip = r->order ? 0u : r->start;          // (an order names samples of the whole set)
    a.x = p.x_lds ? pin + data_at : net->stage_x + skip * n_in;
    a.t = p.x_lds ? pin + data_at + xf : net->stage_y + skip * n_out;
    if (r->order) {
        memcpy(pin + ord_at, r->order, of * 4u);
        a.order = reinterpret_cast<const uint32_t *>(pin + ord_at);
    }
    for (uint32_t l = 0; l < p.nl; ++l) {
        a.act[l] = net->act[l];
        a.dW[l] = reinterpret_cast<float *>(net->W[l].base);
        a.dB[l] = reinterpret_cast<float *>(net->B[l].base);
        net->W[l].cat3_valid = false;
    }
    a.dmW = ts->mW; a.dvW = ts->vW; a.dmB = ts->mB; a.dvB = ts->vB; a.dgW = ts->gW; a.dgB = ts->gB;
    a.samples = r->count;
    a.batch = r->batch;
    a.epochs = r->epochs;
    a.opt = opt_args(*r->args);
    a.opt.decay = r->args->weight_decay;
    a.b1pow = r->args->beta1_pow_t;
    a.b2pow = r->args->beta2_pow_t;
    a.max_norm = r->args->max_grad_norm;
    a.mode = out_delta_mode(r->args->loss_func, a.act[p.nl - 1u]);
    a.loss_func = r->args->loss_func;
    a.sigmoid_out = a.act[p.nl - 1u] == A_SIGMOID;
    a.loss = r->total_loss ? reinterpret_cast<double *>(pin) : nullptr;
    const int rc = p.threads == 64u ? launch_tiny<64>(p) : p.threads == 256u ? launch_tiny<256>(p) : launch_tiny<1024>(p);
    if (rc || wait_for_small_results(net)) return 1;
    const float *o = pin + 2;
    memcpy(r->weights, o, (size_t)a.total_w * 4u);
    memcpy(r->biases, o + a.total_w, (size_t)a.total_b * 4u);
    memcpy(r->m_weights, o + total, (size_t)a.total_w * 4u);
    memcpy(r->m_biases, o + total + a.total_w, (size_t)a.total_b * 4u);
    memcpy(r->v_weights, o + 2u * total, (size_t)a.total_w * 4u);
    memcpy(r->v_biases, o + 2u * total + a.total_w, (size_t)a.total_b * 4u);
    memcpy(r->g_weights, o + 3u * total, (size_t)a.total_w * 4u);
    memcpy(r->g_biases, o + 3u * total + a.total_w, (size_t)a.total_b * 4u);
    if (r->total_loss) memcpy(r->total_loss, pin, sizeof(double));
    return 0;
}

}  // extern "C"
