// hip_train.inl — the batched training step on the device: forward keeping every layer, output and
// hidden deltas, weight and bias gradients, optional clipping by the global norm, one of five
// optimizer updates.  Part of hip_forward.hip's translation unit (included near its end): it uses
// that file's device helpers, launch wrappers and net structure.
//
// What the reference does per step (Src/Spingalett.Training.c): batch_forward :313-345,
// batch_compute_deltas :347-394 (one sgemm NN per hidden layer + apply_derivative_batch),
// batch_accumulate_gradients :396-419 (one sgemm TN + one sgemv T per layer),
// apply_gradients_batch_prescaled :439-507 with the update rules of Src/Spingalett.SIMD.c:279-520.
// Everything stays FP32, as there: products on the FP32 matrix cores, sums in FP32.

namespace {

enum { TR_EPI_DELTA = 0, TR_EPI_SCALE = 1 };

struct TrGemmArgs {
    const float *A, *B;
    float *C;              // [M][N]
    float *ws;             // [splits][M][N] partial sums when the grid splits K, else nullptr
    const float *aux;      // TR_EPI_DELTA: activations [M][N] whose derivative multiplies the product
    uint32_t M, N, K, lda, ldb;
    uint32_t kper;         // k range of one split (multiple of 32)
    int act;               // TR_EPI_DELTA: activation kind of aux
    float scale;           // TR_EPI_SCALE
};

// C[m][n] = sum_k A(m, k) B(n, k) where an operand's rows are not whole 16-byte units (else sp_gemm32_f32 of hip_tile32.inl, with
// the same order of sums), through registers.  Tile 64 x 64 x 32, four waves in a 2 x 2 grid.  Each operand is either
// k-contiguous (element (r, k) at r * ld + k; LDS tile [row][33]) or row-contiguous (element (r, k) at k * ld + r; LDS tile
// [k][96]): the hidden deltas read the weights row-contiguous, the gradients read both operands so.  Both LDS layouts
// are conflict-free for the matrix-core operand reads (lane -> row, half-wave -> k).  Whole pieces are loaded 16 bytes at a time
// from wherever they begin (an epoch of 8000 samples of 785-513-1001-20 803 -> 560 us, a step of 512 180 -> 157 with the same in
// sp_train_grad_update; element by element before).
template <bool AMC, bool BMC, int EPI>
__global__ __launch_bounds__(256) void sp_train_gemm32(const TrGemmArgs g)
{
    constexpr int TM = 1;
    constexpr int BM = 64 * TM, BN = 64 * TM, BK = 32, LDK = BK + 1, LDM = BM + 32;
    constexpr int TILE = BK * LDM > BM * LDK ? BK * LDM : BM * LDK;
    constexpr int PIECES = BM * BK / 4 / 256;            // float4 pieces per thread and operand
    __shared__ __attribute__((aligned(16))) float As[TILE];
    __shared__ __attribute__((aligned(16))) float Bs[TILE];
    const uint32_t M = g.M, N = g.N, K = g.K;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const uint32_t tiles_n = (N + BN - 1) / BN;
    // consecutive workgroups go to different XCDs: give each XCD a contiguous run of tiles, so that the tiles that
    // share a row panel of A meet in one L2
    uint32_t bid = blockIdx.x;
    {
        const uint32_t per = gridDim.x / 8u;
        if (bid < per * 8u) bid = (bid & 7u) * per + (bid >> 3);
    }
    const uint32_t m0 = (bid / tiles_n) * BM, n0 = (bid % tiles_n) * BN;
    const uint32_t kbeg = blockIdx.y * g.kper;
    const uint32_t kend = kbeg + g.kper < K ? kbeg + g.kper : K;

    f32x16 acc[TM][TM];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TM; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

    // four consecutive elements starting at p, of which the first `valid` exist
    auto load4 = [](const float *p, int valid) -> float4 {
        if (valid >= 4) {
            const float4_any x = *reinterpret_cast<const float4_any *>(p);
            return make_float4(x.x, x.y, x.z, x.w);
        }
        float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (e < valid) v[e] = p[e];
        return make_float4(v[0], v[1], v[2], v[3]);
    };
    // piece p of a tile: k-contiguous -> row p / 8, k (p % 8) * 4; row-contiguous -> k p / (BM / 4), row (p % (BM / 4)) * 4
    auto fetch_one = [&](const float *base, uint32_t ld, bool mc, uint32_t r0, uint32_t R, uint32_t k0, int p) -> float4 {
        if (mc) {
            const uint32_t k = k0 + (uint32_t)(p / (BM / 4)), r = r0 + (uint32_t)(p % (BM / 4)) * 4u;
            const int valid = (k < kend && r < R) ? (int)(R - r < 4u ? R - r : 4u) : 0;
            return load4(base + (size_t)(k < K ? k : K - 1) * ld + (r < R ? r : 0u), valid);
        }
        const uint32_t r = r0 + (uint32_t)(p >> 3), k = k0 + (uint32_t)(p & 7) * 4u;
        const int valid = (r < R && k < kend) ? (int)(kend - k < 4u ? kend - k : 4u) : 0;
        return load4(base + (size_t)(r < R ? r : R - 1) * ld + (k < kend ? k : 0u), valid);
    };
    float4 ra[PIECES], rb[PIECES];
    auto fetch = [&](uint32_t k0) {
#pragma unroll
        for (int i = 0; i < PIECES; ++i) {
            ra[i] = fetch_one(g.A, g.lda, AMC, m0, M, k0, t + 256 * i);
            rb[i] = fetch_one(g.B, g.ldb, BMC, n0, N, k0, t + 256 * i);
        }
    };
    auto stash_one = [&](float *tile, bool mc, const float4 &v, int p) {
        if (mc) {
            *reinterpret_cast<float4 *>(tile + (p / (BM / 4)) * LDM + (p % (BM / 4)) * 4) = v;
        } else {
            float *d = tile + (p >> 3) * LDK + (p & 7) * 4;
            d[0] = v.x; d[1] = v.y; d[2] = v.z; d[3] = v.w;
        }
    };
    auto stash = [&]() {
#pragma unroll
        for (int i = 0; i < PIECES; ++i) {
            stash_one(As, AMC, ra[i], t + 256 * i);
            stash_one(Bs, BMC, rb[i], t + 256 * i);
        }
    };

    fetch(kbeg);
    for (uint32_t k0 = kbeg; k0 < kend; k0 += BK) {
        stash();
        __syncthreads();
        if (k0 + BK < kend) fetch(k0 + BK);
#pragma unroll
        for (int ks = 0; ks < BK; ks += 2) {
            const int k = ks + (lane >> 5);
            float a[TM], b[TM];
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                const int ar = (wm * TM + i) * 32 + (lane & 31), br = (wn * TM + i) * 32 + (lane & 31);
                a[i] = AMC ? As[k * LDM + ar] : As[ar * LDK + k];
                b[i] = BMC ? Bs[k * LDM + br] : Bs[br * LDK + k];
            }
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TM; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], b[j], acc[i][j], 0, 0, 0);
        }
        __syncthreads();
    }

    auto emit = [&](auto put) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < TM; ++j) {
            const uint32_t col = n0 + (wn * TM + j) * 32 + (lane & 31);
            if (col >= N) continue;
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const uint32_t row = m0 + (wm * TM + i) * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                    if (row < M) put((size_t)row * N + col, acc[i][j][r]);
                }
        }
    };
    if (g.ws) {
        float *ws = g.ws + (size_t)blockIdx.y * M * N;
        emit([&](size_t o, float v) { ws[o] = v; });
    } else if constexpr (EPI == TR_EPI_DELTA) {
        with_act(g.act, [&](auto act_c) __attribute__((always_inline)) {
            emit([&](size_t o, float v) { g.C[o] = v * act_derivative(g.aux[o], decltype(act_c)::value); });
        });
    } else {
        emit([&](size_t o, float v) { g.C[o] = g.scale * v; });
    }
}

// Weight gradients of a layer of up to 16 outputs: ws[split][m][n] = sum over the split's samples k of d[k][m] a[k][n], in the order
// of sp_gemm32_f32 and sp_train_gemm32, whose tiles of 64 x 64 would be padding for the most part.  A wave owns 16 columns, a
// workgroup's four 64 neighbouring ones (256 bytes of a sample's row); nothing is staged, lane (q, h) loads element q of both
// rows of sample 4 i + h, U steps at once and the next U during their products.  Bound by the inputs' bytes (80 MB of 1000 x 20000).
// An epoch of 20000 samples of 784-512-1000-10 937 -> 917 us, of 500-33-2 171 -> 142, of 8000 of 300-1500-3 299 -> 285.
__global__ __launch_bounds__(256) void sp_train_head_grad(const TrGemmArgs g)
{
    constexpr int U = 16;
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    const uint32_t M = g.M, N = g.N, K = g.K, lane = threadIdx.x & 63u, q = lane & 15u, h = lane >> 4;
    const uint32_t n = blockIdx.x * 64u + (threadIdx.x >> 6) * 16u + q;
    const uint32_t kbeg = blockIdx.y * g.kper, kend = kbeg + g.kper < K ? kbeg + g.kper : K;
    const float *const dp = g.A + (q < M ? q : M - 1u), *const ap = g.B + (n < N ? n : N - 1u);
    struct Round { float d[U], a[U]; } cur, next;
    auto fetch = [&](Round &f, uint32_t k0) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t k = k0 + 4u * u + h, at = k < kend ? k : kend - 1u;
            f.d[u] = dp[(size_t)at * M];
            f.a[u] = ap[(size_t)at * N];
        }
    };
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    fetch(cur, kbeg);
    for (uint32_t k0 = kbeg; k0 < kend; k0 += 4u * U) {
        if (k0 + 4u * U < kend) fetch(next, k0 + 4u * U);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const bool in = k0 + 4u * u + h < kend;                   // (beyond the end: 0 x 0)
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(in ? cur.d[u] : 0.0f, in ? cur.a[u] : 0.0f, acc, 0, 0, 0);
        }
        cur = next;
    }
    if (n >= N) return;
#pragma unroll
    for (uint32_t r = 0; r < 4u; ++r)
        if (4u * h + r < M) g.ws[((size_t)blockIdx.y * M + 4u * h + r) * N + n] = acc[r];
}

// adds the K splits of a hidden-delta product in split order and applies its epilogue
__global__ __launch_bounds__(256) void sp_train_delta_reduce(const TrGemmArgs g, uint32_t splits)
{
    const uint64_t idx = (uint64_t)blockIdx.x * 256u + threadIdx.x;
    const uint64_t total = (uint64_t)g.M * g.N;
    if (idx >= total) return;
    float sum = 0.0f;
    for (uint32_t sp = 0; sp < splits; ++sp) sum += g.ws[(uint64_t)sp * total + idx];
    g.C[idx] = sum * act_derivative(g.aux[idx], g.act);
}

// Hidden deltas of small batches in one launch: C[m][n] = f'(aux[m][n]) sum_k D[m][k] W[k][n].  A workgroup owns 16 samples
// x 16 NJ columns; its eight waves take the segments of K in turn (the tiled kernel's K splits, added in split order: the
// same bits) and meet in LDS; no staging: lane (r, h) loads four k of sample r, and k = 4 i + h of columns NJ r .. for MFMA i.
// The tiled kernel above would need its K split and a second launch to fill the chip: 64 x 512 x 1000 and 64 x 1000 x 10
// together 28 us in three launches, here 11 in two.
template <int NJ>
__global__ __launch_bounds__(512) void sp_train_delta_small(const TrGemmArgs g, uint32_t segments)
{
    constexpr int NW = 8, U = NJ == 4 ? 2 : 4, TN = 16 * NJ;
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    typedef float cols_any __attribute__((ext_vector_type(NJ), aligned(4)));
    extern __shared__ float part[];                               // [segments][16][TN + 1]
    const uint32_t M = g.M, N = g.N, K = g.K;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6, r = lane & 15, h = lane >> 4;
    const uint32_t tiles_n = (N + TN - 1) / TN;
    const uint32_t m0 = (blockIdx.x / tiles_n) * 16u, n0 = (blockIdx.x % tiles_n) * TN;
    const float *ap = g.A + (size_t)(m0 + r < M ? m0 + r : M - 1) * g.lda;
    const uint32_t col0 = n0 + NJ * r;
    const bool whole_cols = n0 + TN <= N;
    for (uint32_t sg = wave; sg < segments; sg += NW) {
        const uint32_t k0 = sg * g.kper, k1 = k0 + g.kper < K ? k0 + g.kper : K;
        f32x4 acc[NJ];
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[j][i] = 0.0f;
        for (uint32_t k = k0; k < k1; k += 16u * U) {
            float a[U][4], b[U][4][NJ];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const uint32_t kb = k + 16u * u;
                if (kb >= k1) break;                              // (uniform)
                load_piece(a[u], ap, kb, h, k1, K);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint32_t kk = kb + 4u * i + h;
                    const float *row = g.B + (size_t)(kk < k1 ? kk : k1 - 1u) * g.ldb;
                    if (whole_cols) {                             // (uniform)
                        const cols_any y = *reinterpret_cast<const cols_any *>(row + col0);
#pragma unroll
                        for (int j = 0; j < NJ; ++j) b[u][i][j] = y[j];
                    } else {
#pragma unroll
                        for (int j = 0; j < NJ; ++j) b[u][i][j] = row[col0 + j < N ? col0 + j : N - 1];
                    }
                    if (kb + 16u > k1) {                          // (uniform; a padded k contributes 0 x 0)
#pragma unroll
                        for (int j = 0; j < NJ; ++j) b[u][i][j] = kk < k1 ? b[u][i][j] : 0.0f;
                    }
                }
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (k + 16u * u >= k1) break;
                chain_order<false>(a[u]);
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int j = 0; j < NJ; ++j) acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u][i], b[u][i][j], acc[j], 0, 0, 0);
            }
        }
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) part[(sg * 16u + 4 * h + i) * (TN + 1) + NJ * r + j] = acc[j][i];
    }
    __syncthreads();
    for (int e = t; e < 16 * TN; e += 512) {
        const int row = e / TN, col = e % TN;
        float v = 0.0f;
        for (uint32_t w = 0; w < segments; ++w) v += part[(w * 16u + row) * (TN + 1) + col];
        if (m0 + row < M && n0 + col < N) {
            const size_t o = (size_t)(m0 + row) * N + n0 + col;
            g.C[o] = v * act_derivative(g.aux[o], g.act);
        }
    }
}

// Deltas of the output layer (Training.c:357-378), one wavefront per sample.
//   mode 0: squared error through a softmax: d_j = a_j ((a_j - t_j) - sum_i (a_i - t_i) a_i)
//   mode 1: cross-entropy through softmax / sigmoid: d = a - t
//   mode 2: every other combination: d = (a - t) f'(a)
__global__ __launch_bounds__(256) void sp_train_out_delta(const float *__restrict__ a, const float *__restrict__ tg,
                                                          float *__restrict__ d, uint32_t n, uint32_t width, int mode, int act)
{
    const int lane = threadIdx.x & 63;
    const uint32_t row = blockIdx.x * 4u + (threadIdx.x >> 6);
    if (row >= n) return;
    const float *ar = a + (size_t)row * width, *tr = tg + (size_t)row * width;
    float *dr = d + (size_t)row * width;
    float sum = 0.0f;
    if (mode == 0) {
        for (uint32_t j = lane; j < width; j += kWave) sum += (ar[j] - tr[j]) * ar[j];
        sum = wave_sum(sum);
    }
    for (uint32_t j = lane; j < width; j += kWave) {
        const float av = ar[j], diff = av - tr[j];
        dr[j] = mode == 0 ? av * (diff - sum) : mode == 1 ? diff : diff * act_derivative(av, act);
    }
}

// Column sums of the deltas [n][width] of all layers (the sgemv against a vector of ones, Training.c:412-417), first pass:
// kColsumRows rows per workgroup into part[chunk][bias]; sp_train_bias_update adds the chunks in order.
constexpr uint32_t kColsumRows = 256;
struct ColsumArgs {
    const float *d[16];
    uint32_t width[16], first_bias[16], first_block[16];       // a layer's first workgroup along x
    uint32_t count, n, total;
    float *part;
};

__global__ __launch_bounds__(256) void sp_train_colsum_part(const ColsumArgs a)
{
    __shared__ float s[4][64];
    uint32_t l = 0;
    while (l + 1u < a.count && blockIdx.x >= a.first_block[l + 1u]) ++l;
    const float *d = a.d[l];
    const uint32_t width = a.width[l], n = a.n;
    const int c = threadIdx.x & 63, rl = threadIdx.x >> 6;
    const uint32_t col = (blockIdx.x - a.first_block[l]) * 64u + c;
    const uint32_t r0 = blockIdx.y * kColsumRows, r1 = r0 + kColsumRows < n ? r0 + kColsumRows : n;
    float sum = 0.0f;
    if (col < width) {
        // four independent partial sums keep four loads in flight per lane
        float p[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        uint32_t r = r0 + rl;
        for (; r + 12u < r1; r += 16u) {
#pragma unroll
            for (int u = 0; u < 4; ++u) p[u] += d[(size_t)(r + 4u * u) * width + col];
        }
        for (; r < r1; r += 4u) p[0] += d[(size_t)r * width + col];
        sum = (p[0] + p[1]) + (p[2] + p[3]);
    }
    s[rl][c] = sum;
    __syncthreads();
    if (rl == 0 && col < width) a.part[(size_t)blockIdx.y * a.total + a.first_bias[l] + col] = (s[0][c] + s[1][c]) + (s[2][c] + s[3][c]);
}

// Sum of squares of one array in FP64, one value per workgroup (first pass of clip_grad_norm, SIMD.c:496-520)
__global__ __launch_bounds__(256) void sp_train_sumsq_part(const float *__restrict__ g, uint64_t cnt, double *__restrict__ part)
{
    __shared__ double s[4];
    double sum = 0.0;
    for (uint64_t i = (uint64_t)blockIdx.x * 256u + threadIdx.x; i < cnt; i += (uint64_t)gridDim.x * 256u) sum += (double)g[i] * (double)g[i];
#pragma unroll
    for (int sft = 32; sft > 0; sft >>= 1) sum += __shfl_xor(sum, sft, kWave);
    if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = sum;
    __syncthreads();
    if (threadIdx.x == 0) part[blockIdx.x] = (s[0] + s[1]) + (s[2] + s[3]);
}

// scal[0] = factor the gradients are multiplied by (max_norm / norm when the norm exceeds max_norm, else 1), scal[1] = norm
__global__ __launch_bounds__(64) void sp_train_clip_fin(const double *__restrict__ part, uint32_t count, float max_norm, float *__restrict__ scal)
{
    double sum = 0.0;
    for (uint32_t i = threadIdx.x; i < count; i += kWave) sum += part[i];
#pragma unroll
    for (int sft = 32; sft > 0; sft >>= 1) sum += __shfl_xor(sum, sft, kWave);
    if (threadIdx.x == 0) {
        const float norm = sqrtf((float)sum);
        scal[0] = norm > max_norm ? max_norm / norm : 1.0f;
        scal[1] = norm;
    }
}

struct OptArgs {
    float *W, *g, *m, *v;
    uint64_t cnt;
    const float *clip;     // device scalar the gradient is multiplied by first, or nullptr
    int opt;               // OptimizerType, Spingalett.h:76-83
    int decay_in_grad;     // RMSprop: decay * W joins the gradient before the second moment (per-sample rule)
    float lr, decay, momentum, b1, b2, omb1, omb2, mf, vf, eps;
};

// One optimizer step of one element: the scalar forms of SIMD.c:279-494 as called from apply_gradients_batch_prescaled
// (Training.c:439-507).  g is left as the reference leaves its gradient (with decay * W added for Adam with weight decay).
__device__ __forceinline__ void opt_update(const OptArgs &a, float &w, float &g, float &m, float &v)
{
    switch (a.opt) {
    case 0:     // SGD
        w -= a.lr * (a.decay > 0.0f ? g + a.decay * w : g);
        break;
    case 1:     // momentum
        m = a.momentum * m + a.decay * w + g;
        w -= a.lr * m;
        break;
    case 2: {   // RMSprop
        const float gd = a.decay_in_grad && a.decay > 0.0f ? g + a.decay * w : g;
        v = a.b2 * v + a.omb2 * (gd * gd);
        w -= a.decay_in_grad ? a.lr * gd / sqrtf(v + a.eps) : a.lr * (a.decay * w + gd / sqrtf(v + a.eps));
        break;
    }
    default: {  // Adam (3): decay joins the gradient; AdamW (4): decay shrinks the weight
        const bool adamw = a.opt == 4;
        if (!adamw && a.decay > 0.0f) g += a.decay * w;
        m = a.b1 * m + a.omb1 * g;
        v = a.b2 * v + a.omb2 * (g * g);
        const float step = a.lr * ((m * a.mf) / sqrtf(v * a.vf + a.eps));
        w = (adamw && a.decay > 0.0f) ? w * (1.0f - a.lr * a.decay) - step : w - step;
        break;
    }
    }
}

// One optimizer step over one array; the gradient array keeps what the reference leaves in it (clipped, and see above)
__global__ __launch_bounds__(256) void sp_train_opt(const OptArgs a)
{
    const uint64_t i = (uint64_t)blockIdx.x * 256u + threadIdx.x;
    if (i >= a.cnt) return;
    const bool has_m = a.opt != 0 && a.opt != 2, has_v = a.opt >= 2;
    const float g0 = a.g[i];
    float w = a.W[i], g = a.clip ? g0 * *a.clip : g0, m = has_m ? a.m[i] : 0.0f, v = has_v ? a.v[i] : 0.0f;
    const bool keep_g = a.clip || (a.opt == 3 && a.decay > 0.0f);
    opt_update(a, w, g, m, v);
    if (keep_g) a.g[i] = g;
    if (has_m) a.m[i] = m;
    if (has_v) a.v[i] = v;
    a.W[i] = w;
}

// One weight layer of a net for the launches that take several at once
struct GradLayer {
    const float *d, *a;    // deltas [n][out], inputs of the layer [n][in]
    float *W, *gW, *mW, *vW, *B, *gB, *mB, *vB;
    uint32_t out, in, tiles_n, first;          // column tiles; first workgroup of the layer
    uint32_t kper;         // samples per segment of the sums (the tiled kernel's K splits, added in split order: the same bits)
};

constexpr uint32_t kGradLayers = 16, kGroupedSamples = 512;

struct GradArgs {
    GradLayer l[kGradLayers];
    uint32_t count, n;
    float scale;           // 1 / n
    int update;            // 0: gradients only
    OptArgs opt;           // (array pointers unused; decay: the weights')
};

// Gradients of several layers in one launch, g = scale delta^T inputs (Training.c:396-419), each workgroup updating the
// weights of its 32 x 64 tile as soon as it has their gradients (unless they are clipped first): no second pass over
// gradients, weights and moments, and small layers share the chip with large ones.  The column tile 0 of a row of tiles
// also adds up its deltas and updates the biases.  For batches whose whole sum over samples one workgroup can walk
// (train_grads_grouped).  Four waves, each 16 x 32; both operands lie row-contiguous, k = sample: LDS tiles [k][width + 16],
// conflict-free for the operand reads; the next tile's loads fly while the matrix cores work, those of weights and moments
// during all of it.  Bound by the 28 bytes per weight of the arrays and by the arithmetic of the update, 8 weights per
// thread (64 samples of 784-512-1000-10, three layers: 13.6 us against 3 x 5.3 + 3 x 2.4 + 3 x 1.8 + 6 x 2.8 for
// products, bias sums and updates one by one; 64 x 64 tiles, 16 weights per thread: 20 us).
__global__ __launch_bounds__(256) void sp_train_grad_update(const GradArgs g)
{
    constexpr int BM = 32, BN = 64, BK = 32, LDA = BM + 16, LDB = BN + 16;
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    __shared__ __attribute__((aligned(16))) float As[BK * LDA];
    __shared__ __attribute__((aligned(16))) float Bs[BK * LDB];
    __shared__ float bias_part[kGroupedSamples / kColsumRows][4][BM];
    uint32_t li = 0;
    while (li + 1u < g.count && blockIdx.x >= g.l[li + 1u].first) ++li;
    const GradLayer &L = g.l[li];
    const uint32_t M = L.out, N = L.in, n = g.n, bid = blockIdx.x - L.first, kper = L.kper;
    const uint32_t m0 = (bid / L.tiles_n) * BM, n0 = (bid % L.tiles_n) * BN;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6, wm = wave >> 1, wn = wave & 1, q = lane & 15, h = lane >> 4;
    const bool has_m = g.update && g.opt.opt != 0 && g.opt.opt != 2, has_v = g.update && g.opt.opt >= 2;

    f32x4 acc[2], sum[2];
    float w[2][4], m[2][4], v[2][4];
    const uint32_t row0 = m0 + wm * 16 + 4 * h, col0 = n0 + wn * 32 + q;
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            acc[j][r] = sum[j][r] = 0.0f;
            const uint32_t row = row0 + r, col = col0 + 16 * j;
            const size_t o = (size_t)(row < M ? row : M - 1) * N + (col < N ? col : N - 1);
            w[j][r] = g.update ? L.W[o] : 0.0f;
            m[j][r] = has_m ? L.mW[o] : 0.0f;
            v[j][r] = has_v ? L.vW[o] : 0.0f;
        }

    // piece p of a tile of width W: sample p / (W / 4), element (p % (W / 4)) * 4; one piece of A, two of B per thread
    auto load4 = [](const float *base, uint32_t ld, uint32_t R, uint32_t r, uint32_t k, bool kin) -> float4 {
        if (!kin || r >= R) return make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        const float *p = base + (size_t)k * ld + r;
        if (r + 4u <= R) {
            const float4_any x = *reinterpret_cast<const float4_any *>(p);
            return make_float4(x.x, x.y, x.z, x.w);
        }
        float e[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (uint32_t i = 0; i < 4u; ++i)
            if (r + i < R) e[i] = p[i];
        return make_float4(e[0], e[1], e[2], e[3]);
    };
    float4 ra, rb[2];
    auto fetch = [&](uint32_t k0) {
        ra = load4(L.d, M, M, m0 + (t & 7) * 4u, k0 + (t >> 3), k0 + (t >> 3) < n);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint32_t p = t + 256u * i, k = k0 + (p >> 4);
            rb[i] = load4(L.a, N, N, n0 + (p & 15u) * 4u, k, k < n);
        }
    };
    // column sums of the deltas, in the order of sp_train_colsum_part: chunks of 256 samples, in a chunk thread (q, c) adds
    // samples q + 4 i of column c in four running sums, the ones that fill no group of 16 in the first
    const bool biases = n0 == 0;
    float bp[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    fetch(0);
    for (uint32_t k0 = 0; k0 < n; k0 += BK) {
        *reinterpret_cast<float4 *>(As + (t >> 3) * LDA + (t & 7) * 4) = ra;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int p = t + 256 * i;
            *reinterpret_cast<float4 *>(Bs + (p >> 4) * LDB + (p & 15) * 4) = rb[i];
        }
        __syncthreads();
        if (k0 + BK < n) fetch(k0 + BK);
#pragma unroll
        for (int ks = 0; ks < BK; ks += 4) {
            const float a = As[(ks + h) * LDA + wm * 16 + q];
#pragma unroll
            for (int j = 0; j < 2; ++j)
                acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, Bs[(ks + h) * LDB + wn * 32 + 16 * j + q], acc[j], 0, 0, 0);
        }
        if (biases && lane < BM) {
            const uint32_t c1 = (k0 / kColsumRows + 1u) * kColsumRows < n ? (k0 / kColsumRows + 1u) * kColsumRows : n;
#pragma unroll
            for (int i = 0; i < BK / 4; ++i) {
                const uint32_t k = k0 + 4u * i + wave, group = (k0 + 16u * (i / 4)) + wave;       // first sample of its group of 16
                if (k < n) {
                    const float d = As[(4 * i + wave) * LDA + lane];
                    if (group + 12u < c1) bp[i & 3] += d;
                    else bp[0] += d;
                }
            }
            if ((k0 + BK) % kColsumRows == 0 || k0 + BK >= n) {
                bias_part[k0 / kColsumRows][wave][lane] = (bp[0] + bp[1]) + (bp[2] + bp[3]);
                bp[0] = bp[1] = bp[2] = bp[3] = 0.0f;
            }
        }
        if ((k0 + BK) % kper == 0 || k0 + BK >= n) {
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                sum[j] += acc[j];
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[j][r] = 0.0f;
            }
        }
        __syncthreads();
    }

    OptArgs opt = g.opt;
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const uint32_t row = row0 + r, col = col0 + 16 * j;
            if (row >= M || col >= N) continue;
            const size_t o = (size_t)row * N + col;
            float grad = g.scale * sum[j][r];
            if (g.update) {
                opt_update(opt, w[j][r], grad, m[j][r], v[j][r]);
                L.W[o] = w[j][r];
                if (has_m) L.mW[o] = m[j][r];
                if (has_v) L.vW[o] = v[j][r];
            }
            L.gW[o] = grad;
        }
    if (!biases) return;                                          // (uniform)
    const uint32_t j = m0 + t;                                    // (the sums are in LDS since the last barrier)
    if (t < BM && j < M) {
        float grad = 0.0f;
        for (uint32_t c = 0; c * kColsumRows < n; ++c) grad += (bias_part[c][0][t] + bias_part[c][1][t]) + (bias_part[c][2][t] + bias_part[c][3][t]);
        grad *= g.scale;
        if (g.update) {
            float b = L.B[j], mb = has_m ? L.mB[j] : 0.0f, vb = has_v ? L.vB[j] : 0.0f;
            opt.decay = 0.0f;
            opt_update(opt, b, grad, mb, vb);
            L.B[j] = b;
            if (has_m) L.mB[j] = mb;
            if (has_v) L.vB[j] = vb;
        }
        L.gB[j] = grad;
    }
}

// The same update behind a product whose K was split over the grid: the splits are added in split order, scaled, and
// applied at once.  Four elements per thread where the array's size and place allow (VEC).
template <bool VEC>
__global__ __launch_bounds__(256) void sp_train_reduce_update(const float *__restrict__ ws, uint32_t splits, uint64_t total, float scale,
                                                              int update, const OptArgs opt)
{
    constexpr uint32_t E = VEC ? 4u : 1u;
    typedef float ve __attribute__((ext_vector_type(E)));
    const uint64_t i = ((uint64_t)blockIdx.x * 256u + threadIdx.x) * E;
    if (i >= total) return;
    const bool has_m = update && opt.opt != 0 && opt.opt != 2, has_v = update && opt.opt >= 2;
    auto at = [&](const float *p) { return *reinterpret_cast<const ve *>(p + i); };
    auto to = [&](float *p, ve x) { *reinterpret_cast<ve *>(p + i) = x; };
    ve w{}, m{}, v{}, sum{};
    if (update) w = at(opt.W);
    if (has_m) m = at(opt.m);
    if (has_v) v = at(opt.v);
    for (uint32_t sp = 0; sp < splits; ++sp) sum += at(ws + (uint64_t)sp * total);
#pragma unroll
    for (uint32_t e = 0; e < E; ++e) {
        float grad = scale * sum[e], we = w[e], me = m[e], ve_ = v[e];
        if (update) opt_update(opt, we, grad, me, ve_);
        sum[e] = grad; w[e] = we; m[e] = me; v[e] = ve_;
    }
    to(opt.g, sum);
    if (update) to(opt.W, w);
    if (has_m) to(opt.m, m);
    if (has_v) to(opt.v, v);
}

// Bias gradients of all layers from the partial column sums (sp_train_colsum_part), and the biases' update
struct BiasArgs {
    const float *part;     // [chunks][total]
    float *B[kGradLayers], *gB, *mB, *vB;      // gradients and moments flat over the layers
    uint32_t first[kGradLayers + 1];           // first bias of a layer; [count]: all of them
    uint32_t count, chunks;
    float scale;
    int update;
    OptArgs opt;           // (decay 0)
};

__global__ __launch_bounds__(256) void sp_train_bias_update(const BiasArgs a)
{
    // eight running sums over the chunks, two to a thread (the chunks that fill no group of eight in the first): a fixed
    // order, and loads enough in flight
    __shared__ float s[4][64];
    const int c = threadIdx.x & 63, q = threadIdx.x >> 6;
    const uint32_t total = a.first[a.count], j = blockIdx.x * 64u + c;
    float sum = 0.0f;
    if (j < total) {
        float p0 = 0.0f, p1 = 0.0f;
        uint32_t ch = 0;
        for (; ch + 8u <= a.chunks; ch += 8u) {
            p0 += a.part[(size_t)(ch + 2u * q) * total + j];
            p1 += a.part[(size_t)(ch + 2u * q + 1u) * total + j];
        }
        for (; q == 0 && ch < a.chunks; ++ch) p0 += a.part[(size_t)ch * total + j];
        sum = p0 + p1;
    }
    s[q][c] = sum;
    __syncthreads();
    if (q || j >= total) return;
    float grad = a.scale * ((s[0][c] + s[1][c]) + (s[2][c] + s[3][c]));
    if (a.update) {
        uint32_t l = 0;
        while (l + 1u < a.count && j >= a.first[l + 1u]) ++l;
        float *B = a.B[l] + (j - a.first[l]);
        const bool has_m = a.opt.opt != 0 && a.opt.opt != 2, has_v = a.opt.opt >= 2;
        float b = *B, m = has_m ? a.mB[j] : 0.0f, v = has_v ? a.vB[j] : 0.0f;
        opt_update(a.opt, b, grad, m, v);
        *B = b;
        if (has_m) a.mB[j] = m;
        if (has_v) a.vB[j] = v;
    }
    a.gB[j] = grad;
}

}  // namespace

// Device state of a net being trained: gradients and optimizer moments laid out like the host net's
// flat arrays (layer l at woff[l] / boff[l]), activations and deltas of every layer for the largest
// batch seen so far.
struct sphip_train_state {
    std::vector<uint64_t> woff, boff;
    uint64_t total_w = 0, total_b = 0;
    float *gW = nullptr, *gB = nullptr, *mW = nullptr, *vW = nullptr, *mB = nullptr, *vB = nullptr;
    uint32_t cap_n = 0;
    std::vector<float *> act, delta;       // [layers]; act[0] stages host inputs, delta[0] is unused
    float *targets = nullptr;              // staged host targets [cap_n][topo[last]]
    uint32_t staged_n = 0;                 // samples of the batch staged last (0: none)
    float *ws = nullptr;                   // split-K partials, column-sum partials
    uint64_t ws_cap = 0;
    double *sq_part = nullptr;             // per-workgroup sums of squares (clipping)
    float *scal = nullptr;                 // clip factor, gradient norm
    float *loss_buf = nullptr;             // per-sample loss / prediction / hit, totals
    uint64_t loss_cap = 0;
    // Host mini-batches travel through a ring of pinned slots and a copy kernel; an event per half of the ring says when
    // its slots may be written again
    float *ring = nullptr;
    uint64_t ring_slot = 0;                // floats per slot
    hipEvent_t ring_ev[2] = {nullptr, nullptr};
    uint32_t ring_next = 0;
    bool ring_full[2] = {false, false};    // the half's event has been recorded
    float *tiny_pin = nullptr;             // pinned host memory of sp_train_tiny: state, results, samples
    uint64_t tiny_cap = 0;
};

namespace {

constexpr uint32_t kSqBlocks = 1024;

void train_free(sphip_net *net)
{
    sphip_train_state *ts = net->train;
    if (!ts) return;
    float *flat[] = {ts->gW, ts->gB, ts->mW, ts->vW, ts->mB, ts->vB, ts->targets, ts->ws, ts->scal, ts->loss_buf};
    for (float *p : flat) if (p) (void)hipFree(p);
    if (ts->sq_part) (void)hipFree(ts->sq_part);
    if (ts->tiny_pin) (void)hipHostFree(ts->tiny_pin);
    if (ts->ring) (void)hipHostFree(ts->ring);
    for (hipEvent_t e : ts->ring_ev) if (e) (void)hipEventDestroy(e);
    for (float *p : ts->act) if (p) (void)hipFree(p);
    for (float *p : ts->delta) if (p) (void)hipFree(p);
    delete ts;
    net->train = nullptr;
}

// Whether the gradients take sp_train_grad_update, one workgroup per 32 x 64 tile: up to 512 samples (16 K tiles);
// more are split over the grid.
bool train_grads_grouped(uint32_t n) { return n <= kGroupedSamples; }

int train_reserve(sphip_net *net, uint32_t n)
{
    sphip_train_state *ts = net->train;
    if (n > ts->cap_n) {
        for (uint32_t l = 0; l < net->layers; ++l) {
            if (ts->act[l]) { HCHECK(hipFree(ts->act[l])); ts->act[l] = nullptr; }
            if (ts->delta[l]) { HCHECK(hipFree(ts->delta[l])); ts->delta[l] = nullptr; }
        }
        if (ts->targets) { HCHECK(hipFree(ts->targets)); ts->targets = nullptr; }
        ts->cap_n = 0;
        ts->staged_n = 0;
        for (uint32_t l = 0; l < net->layers; ++l) {
            HCHECK(hipMalloc((void **)&ts->act[l], (size_t)n * net->topo[l] * sizeof(float) + 16u));
            if (l) HCHECK(hipMalloc((void **)&ts->delta[l], (size_t)n * net->topo[l] * sizeof(float) + 16u));
        }
        HCHECK(hipMalloc((void **)&ts->targets, (size_t)n * net->topo[net->layers - 1] * sizeof(float) + 16u));
        ts->cap_n = n;
    }
    // workspace: K splits of the delta and gradient products, column-sum partials
    uint64_t ws = 0;
    uint32_t kper = 0;
    for (uint32_t l = 1; l + 1 < net->layers; ++l) {
        const uint32_t sp = gemm32_splits(n, net->topo[l], net->topo[l + 1], &kper);
        if (sp > 1 && (uint64_t)sp * n * net->topo[l] > ws) ws = (uint64_t)sp * n * net->topo[l];
    }
    if (!train_grads_grouped(n)) {
        for (uint32_t l = 0; l + 1 < net->layers; ++l) {
            const uint64_t sp = gemm32_splits(net->topo[l + 1], net->topo[l], n, &kper);
            const uint64_t wcnt = (uint64_t)net->topo[l] * net->topo[l + 1];
            if (sp * wcnt > ws) ws = sp * wcnt;
        }
        const uint64_t cs = (uint64_t)((n + kColsumRows - 1) / kColsumRows) * ts->total_b;
        if (cs > ws) ws = cs;
    }
    if (grow(&ts->ws, &ts->ws_cap, ws)) return 1;
    return 0;
}

Tile32Args tile32_args(const TrGemmArgs &g)
{
    return {g.A, g.B, g.C, g.ws, g.aux, nullptr, F32, 1.0f, g.M, g.N, g.K, g.lda, g.ldb, g.kper, g.act, g.scale};
}

// Hidden deltas: one launch of sp_train_delta_small for batches of up to 512 samples and 2048 tiles of 16 x 16 (wider tiles
// as there are more of them than the chip takes at once), else the tiled kernel with its K split.
void launch_train_delta(TrGemmArgs g, float *ws, uint64_t ws_floats)
{
    uint32_t splits = gemm32_splits(g.M, g.N, g.K, &g.kper);
    const uint64_t rows16 = (g.M + 15u) / 16u, tiles = rows16 * ((g.N + 15u) / 16u);
    if (g.M <= 512u && g.K <= 4096u && tiles <= 2048u) {
        const uint32_t nj = tiles <= 512u ? 1u : tiles <= 1024u || splits > 15u ? 2u : 4u;
        const uint32_t grid = (uint32_t)rows16 * ((g.N + 16u * nj - 1u) / (16u * nj));
        const size_t lds = (size_t)splits * 16u * (16u * nj + 1u) * sizeof(float);      // (at most 64 KiB)
        if (nj == 1u) sp_train_delta_small<1><<<grid, 512, lds, g_stream>>>(g, splits);
        else if (nj == 2u) sp_train_delta_small<2><<<grid, 512, lds, g_stream>>>(g, splits);
        else sp_train_delta_small<4><<<grid, 512, lds, g_stream>>>(g, splits);
        return;
    }
    if (splits > 1 && (uint64_t)splits * g.M * g.N > ws_floats) { splits = 1; g.kper = (g.K + 31u) / 32u * 32u; }
    g.ws = splits > 1 ? ws : nullptr;
    if (gemm32_tile_takes(g.A, g.B, g.lda, g.ldb))
        launch_gemm32_tile<T32_DELTA, false, true>(tile32_args(g), splits);
    else
        sp_train_gemm32<false, true, TR_EPI_DELTA><<<dim3(((g.M + 63) / 64) * ((g.N + 63) / 64), splits), 256, 0, g_stream>>>(g);
    if (splits > 1) sp_train_delta_reduce<<<(uint32_t)(((uint64_t)g.M * g.N + 255) / 256), 256, 0, g_stream>>>(g, splits);
}

// the scalars of a step's updates; decay and the arrays are the caller's to set
OptArgs opt_args(const sphip_train_args &a)
{
    OptArgs o{};
    o.opt = a.optimizer;
    o.decay_in_grad = a.decay_in_grad;
    o.lr = a.learning_rate; o.momentum = a.momentum;
    o.b1 = a.beta1; o.b2 = a.beta2;
    // formed in FP32 like the reference's locals (Training.c:447-448, 479-480)
    o.omb1 = 1.0f - a.beta1;
    o.omb2 = 1.0f - a.beta2;
    o.mf = 1.0f / (1.0f - a.beta1_pow_t);
    o.vf = 1.0f / (1.0f - a.beta2_pow_t);
    o.eps = a.epsilon;
    return o;
}

void launch_opt(const sphip_train_args &a, float *W, float *g, float *m, float *v, uint64_t cnt, float decay, const float *clip)
{
    OptArgs o = opt_args(a);
    o.W = W; o.g = g; o.m = m; o.v = v; o.cnt = cnt; o.clip = clip;
    o.decay = decay;
    sp_train_opt<<<(uint32_t)((cnt + 255) / 256), 256, 0, g_stream>>>(o);
}

// which of sp_train_out_delta's rules a loss and an output activation take (Training.c:357-378)
int out_delta_mode(int loss_func, int last_act)
{
    return (loss_func == 0 && last_act == A_SOFTMAX) ? 0
         : (loss_func == 1 && (last_act == A_SOFTMAX || last_act == A_SIGMOID)) ? 1 : 2;
}

// Gradients of every layer for the deltas at hand, with the optimizer's update if asked for
void train_gradients(sphip_net *net, const float *d_x, uint32_t n, const sphip_train_args &args, int update)
{
    sphip_train_state *ts = net->train;
    const uint32_t last = net->layers - 1;
    const float scale = 1.0f / (float)n;
    OptArgs opt = opt_args(args);
    auto aligned = [](const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
    auto inputs = [&](uint32_t l) { return l == 0 ? d_x : (const float *)ts->act[l]; };
    opt.decay = args.weight_decay;
    if (train_grads_grouped(n)) {
        for (uint32_t l0 = 0; l0 < last; l0 += kGradLayers) {
            GradArgs g{};
            g.n = n;
            g.scale = scale;
            g.update = update;
            g.opt = opt;
            uint32_t blocks = 0;
            for (uint32_t l = l0; l < last && g.count < kGradLayers; ++l) {
                GradLayer &q = g.l[g.count++];
                q.d = ts->delta[l + 1]; q.a = inputs(l);
                q.W = reinterpret_cast<float *>(net->W[l].base); q.B = reinterpret_cast<float *>(net->B[l].base);
                q.gW = ts->gW + ts->woff[l]; q.mW = ts->mW + ts->woff[l]; q.vW = ts->vW + ts->woff[l];
                q.gB = ts->gB + ts->boff[l]; q.mB = ts->mB + ts->boff[l]; q.vB = ts->vB + ts->boff[l];
                q.out = net->topo[l + 1]; q.in = net->topo[l];
                (void)gemm32_splits(q.out, q.in, n, &q.kper);
                q.tiles_n = (q.in + 63u) / 64u;
                q.first = blocks;
                blocks += (q.out + 31u) / 32u * q.tiles_n;
            }
            sp_train_grad_update<<<blocks, 256, 0, g_stream>>>(g);
        }
        return;
    }
    // biases: column sums of all layers, 16 at a time, then their update
    const uint32_t chunks = (n + kColsumRows - 1) / kColsumRows;
    for (uint32_t l0 = 0; l0 < last; l0 += kGradLayers) {
        ColsumArgs c{};
        BiasArgs b{};
        uint32_t blocks = 0;
        for (uint32_t l = l0; l < last && c.count < kGradLayers; ++l, ++c.count) {
            c.d[c.count] = ts->delta[l + 1];
            c.width[c.count] = net->topo[l + 1];
            c.first_bias[c.count] = b.first[c.count] = (uint32_t)(ts->boff[l] - ts->boff[l0]);
            c.first_block[c.count] = blocks;
            b.B[c.count] = reinterpret_cast<float *>(net->B[l].base);
            blocks += (net->topo[l + 1] + 63u) / 64u;
            c.total = b.first[c.count + 1u] = c.first_bias[c.count] + net->topo[l + 1];
        }
        c.n = n;
        c.part = ts->ws;
        b.part = ts->ws;
        b.gB = ts->gB + ts->boff[l0]; b.mB = ts->mB + ts->boff[l0]; b.vB = ts->vB + ts->boff[l0];
        b.count = c.count;
        b.chunks = chunks;
        b.scale = scale;
        b.update = update;
        b.opt = opt;
        b.opt.decay = 0.0f;
        sp_train_colsum_part<<<dim3(blocks, chunks), 256, 0, g_stream>>>(c);
        sp_train_bias_update<<<(c.total + 63u) / 64u, 256, 0, g_stream>>>(b);
    }
    for (uint32_t l = 0; l < last; ++l) {
        TrGemmArgs g{};
        g.A = ts->delta[l + 1]; g.lda = net->topo[l + 1];
        g.B = inputs(l); g.ldb = net->topo[l];
        g.M = net->topo[l + 1]; g.N = net->topo[l]; g.K = n;
        g.ws = ts->ws;
        const uint32_t splits = gemm32_splits(g.M, g.N, g.K, &g.kper);
        if (g.M <= 16u)
            sp_train_head_grad<<<dim3((g.N + 63u) / 64u, splits), 256, 0, g_stream>>>(g);
        else if (gemm32_tile_takes(g.A, g.B, g.lda, g.ldb))
            launch_gemm32_tile<T32_SCALE, true, true>(tile32_args(g), splits);
        else
            sp_train_gemm32<true, true, TR_EPI_SCALE><<<dim3(((g.M + 63) / 64) * ((g.N + 63) / 64), splits), 256, 0, g_stream>>>(g);
        opt.W = reinterpret_cast<float *>(net->W[l].base);
        opt.g = ts->gW + ts->woff[l]; opt.m = ts->mW + ts->woff[l]; opt.v = ts->vW + ts->woff[l];
        const uint64_t total = (uint64_t)g.M * g.N;
        const bool vec = total % 4u == 0 && aligned(opt.W) && aligned(opt.g) && aligned(opt.m) && aligned(opt.v);
        if (vec) sp_train_reduce_update<true><<<(uint32_t)((total / 4u + 255) / 256), 256, 0, g_stream>>>(ts->ws, splits, total, scale, update, opt);
        else sp_train_reduce_update<false><<<(uint32_t)((total + 255) / 256), 256, 0, g_stream>>>(ts->ws, splits, total, scale, update, opt);
    }
}

// A host batch of up to this many floats goes through the ring: the runtime's own copies from pageable memory wait for
// the device twice per step.
constexpr uint64_t kRingFloats = 1u << 20;
constexpr uint32_t kRingSlots = 8;

__global__ __launch_bounds__(256) void sp_train_stage(const float4 *__restrict__ src, float4 *__restrict__ x, uint32_t nx, float4 *__restrict__ t,
                                                      uint32_t nt)
{
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i < nx) x[i] = src[i];
    else if (i < nx + nt) t[i - nx] = src[i];
}

// the host batch into act[0] and targets; the caller's arrays have been read when this returns.  A whole set, staged once, does not
// go through the ring beyond kOnceFloats: each call would fill another slot, whose pages are touched for the first time up to
// the eighth call (train() of four epochs of 6469 samples of 121-240-13, mean of calls two to seven 2437 -> 569 us, of three of 314
// of 1529-128-16 1537 -> 488, of three of 300 of 64-100-10 628 -> 180).
constexpr uint64_t kOnceFloats = 32u << 10;
int train_stage(sphip_net *net, const float *x, const float *t, uint32_t n, bool once)
{
    sphip_train_state *ts = net->train;
    const uint64_t cx = (uint64_t)n * net->topo[0], ct = (uint64_t)n * net->topo[net->layers - 1];
    const uint64_t qx = (cx + 3u) / 4u, qt = (ct + 3u) / 4u;
    if (4u * (qx + qt) > (once ? kOnceFloats : kRingFloats)) {
        if (upload_from_host(ts->act[0], x, cx * sizeof(float))) return 1;
        return upload_from_host(ts->targets, t, ct * sizeof(float));
    }
    if (4u * (qx + qt) > ts->ring_slot) {
        HCHECK(hipStreamSynchronize(g_stream));
        if (ts->ring) { HCHECK(hipHostFree(ts->ring)); ts->ring = nullptr; }
        ts->ring_slot = 0;
        HCHECK(hipHostMalloc((void **)&ts->ring, kRingSlots * 4u * (qx + qt) * sizeof(float), hipHostMallocDefault));
        ts->ring_slot = 4u * (qx + qt);
        ts->ring_full[0] = ts->ring_full[1] = false;
        ts->ring_next = 0;
        for (hipEvent_t &e : ts->ring_ev) if (!e) HCHECK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    }
    const uint32_t slot = ts->ring_next++ % kRingSlots, half = slot / (kRingSlots / 2u);
    if (slot % (kRingSlots / 2u) == 0 && ts->ring_full[half]) HCHECK(hipEventSynchronize(ts->ring_ev[half]));
    float *pin = ts->ring + (size_t)slot * ts->ring_slot;
    memcpy(pin, x, cx * sizeof(float));
    memcpy(pin + 4u * qx, t, ct * sizeof(float));
    sp_train_stage<<<(uint32_t)((qx + qt + 255u) / 256u), 256, 0, g_stream>>>(reinterpret_cast<const float4 *>(pin), reinterpret_cast<float4 *>(ts->act[0]),
                                                                            (uint32_t)qx, reinterpret_cast<float4 *>(ts->targets), (uint32_t)qt);
    HCHECK(hipGetLastError());
    if (slot % (kRingSlots / 2u) == kRingSlots / 2u - 1u) {
        HCHECK(hipEventRecord(ts->ring_ev[half], g_stream));
        ts->ring_full[half] = true;
    }
    return 0;
}

}  // namespace

extern "C" {

int sphip_train_begin(sphip_net *net)
{
    if (!net) return fail_msg("sphip_train_begin: invalid argument");
    if (net->prec != F32) return fail_msg("sphip_train_begin: training needs the FP32 arrays on the device (this net holds a packed format)");
    for (uint32_t l = 1; l + 1 < net->layers; ++l)
        if (net->act[l - 1] == A_SOFTMAX) return fail_msg("sphip_train_begin: softmax is not supported in hidden layers");
    if (check_uploaded(net)) return 1;
    if (net->train) return 0;
    sphip_train_state *ts = new (std::nothrow) sphip_train_state;
    if (!ts) return fail_msg("sphip_train_begin: out of host memory");
    net->train = ts;
    ts->act.assign(net->layers, nullptr);
    ts->delta.assign(net->layers, nullptr);
    for (uint32_t l = 0; l + 1 < net->layers; ++l) {
        ts->woff.push_back(ts->total_w);
        ts->boff.push_back(ts->total_b);
        ts->total_w += (uint64_t)net->topo[l] * net->topo[l + 1];
        ts->total_b += net->topo[l + 1];
    }
    float **flat[] = {&ts->gW, &ts->mW, &ts->vW, &ts->gB, &ts->mB, &ts->vB};
    for (int i = 0; i < 6; ++i) {
        const uint64_t cnt = i < 3 ? ts->total_w : ts->total_b;
        hipError_t e = hipMalloc((void **)flat[i], cnt * sizeof(float));
        if (e != hipSuccess) { train_free(net); return fail_hip("sphip_train_begin: device allocation", e); }
        sp_fill0<<<(uint32_t)((cnt + 255) / 256), 256, 0, g_stream>>>(*flat[i], cnt);
    }
    hipError_t e = hipMalloc((void **)&ts->sq_part, 2u * kSqBlocks * sizeof(double));
    if (e == hipSuccess) e = hipMalloc((void **)&ts->scal, 4 * sizeof(float));
    if (e == hipSuccess) e = hipGetLastError();
    if (e == hipSuccess) e = hipStreamSynchronize(g_stream);
    if (e != hipSuccess) { train_free(net); return fail_hip("sphip_train_begin", e); }
    return 0;
}

void sphip_train_end(sphip_net *net)
{
    if (!net || !net->train) return;
    if (g_stream) (void)hipStreamSynchronize(g_stream);
    train_free(net);
}

static float *train_array(sphip_net *net, int which, uint32_t l, uint64_t *cnt)
{
    sphip_train_state *ts = net->train;
    const uint64_t wc = (uint64_t)net->topo[l] * net->topo[l + 1], bc = net->topo[l + 1];
    switch (which) {
    case SPHIP_TRAIN_W:  *cnt = wc; return reinterpret_cast<float *>(net->W[l].base);
    case SPHIP_TRAIN_B:  *cnt = bc; return reinterpret_cast<float *>(net->B[l].base);
    case SPHIP_TRAIN_MW: *cnt = wc; return ts->mW + ts->woff[l];
    case SPHIP_TRAIN_VW: *cnt = wc; return ts->vW + ts->woff[l];
    case SPHIP_TRAIN_MB: *cnt = bc; return ts->mB + ts->boff[l];
    case SPHIP_TRAIN_VB: *cnt = bc; return ts->vB + ts->boff[l];
    case SPHIP_TRAIN_GW: *cnt = wc; return ts->gW + ts->woff[l];
    case SPHIP_TRAIN_GB: *cnt = bc; return ts->gB + ts->boff[l];
    default: *cnt = 0; return nullptr;
    }
}

int sphip_train_set(sphip_net *net, int which, uint32_t l, const float *host)
{
    if (!net || !net->train || l + 1 >= net->layers || !host) return fail_msg("sphip_train_set: invalid argument");
    uint64_t cnt = 0;
    float *dst = train_array(net, which, l, &cnt);
    if (!dst) return fail_msg("sphip_train_set: unknown array");
    HCHECK(hipMemcpyAsync(dst, host, cnt * sizeof(float), hipMemcpyHostToDevice, g_stream));
    HCHECK(hipStreamSynchronize(g_stream));
    if (which == SPHIP_TRAIN_W) net->W[l].cat3_valid = false;      // the FP16 parts describe the old weights
    return 0;
}

int sphip_train_get(sphip_net *net, int which, uint32_t l, float *host)
{
    if (!net || !net->train || l + 1 >= net->layers || !host) return fail_msg("sphip_train_get: invalid argument");
    uint64_t cnt = 0;
    const float *src = train_array(net, which, l, &cnt);
    if (!src) return fail_msg("sphip_train_get: unknown array");
    if (cnt > kSmallOut) return download_to_host(host, src, cnt * sizeof(float));
    if (grow_pinned(&net->pin_out, &net->pin_out_cap, kSmallOut)) return 1;
    sp_copy32<<<(uint32_t)((cnt + 255) / 256), 256, 0, g_stream>>>(src, net->pin_out, cnt);
    if (wait_for_small_results(net)) return 1;
    memcpy(host, net->pin_out, cnt * sizeof(float));
    return 0;
}

int sp_train_arrays(sphip_net *net, const sp_train_host *h, bool to_host)
{
    if (!net || !net->train) return fail_msg("sp_train_arrays: sphip_train_begin was not called for this net");
    sphip_train_state *ts = net->train;
    const std::unique_ptr<Segment[]> seg(new (std::nothrow) Segment[2u * net->layers + 6u]);
    if (!seg) return fail_msg("sp_train_arrays: out of host memory");
    uint32_t count = 0;
    auto add = [&](float *host, void *dev, uint64_t cnt) {
        if (host) seg[count++] = {reinterpret_cast<char *>(host), static_cast<char *>(dev), cnt * sizeof(float)};
    };
    for (uint32_t l = 0; l + 1 < net->layers; ++l) {
        add(h->weights ? h->weights + ts->woff[l] : nullptr, net->W[l].base, net->W[l].count);
        add(h->biases ? h->biases + ts->boff[l] : nullptr, net->B[l].base, net->B[l].count);
        if (!to_host && h->weights) net->W[l].cat3_valid = false;          // the FP16 parts describe the old weights
    }
    add(h->m_weights, ts->mW, ts->total_w);
    add(h->v_weights, ts->vW, ts->total_w);
    add(h->g_weights, ts->gW, ts->total_w);
    add(h->m_biases, ts->mB, ts->total_b);
    add(h->v_biases, ts->vB, ts->total_b);
    add(h->g_biases, ts->gB, ts->total_b);
    return move_arrays(seg.get(), count, to_host);
}

int sphip_train_step(sphip_net *net, const float *x, const float *targets, uint32_t n, const sphip_train_args *args,
                     uint32_t flags, float *total_loss)
{
    const bool restage = (flags & SPHIP_TRAIN_SAME_BATCH) != 0;
    if (!net || ((!x || !targets) && !restage) || n == 0 || !args) return fail_msg("sphip_train_step: invalid argument");
    if (!net->train) return fail_msg("sphip_train_step: sphip_train_begin was not called for this net");
    if (args->optimizer > 4 || (args->loss_func != 0 && args->loss_func != 1)) return fail_msg("sphip_train_step: invalid optimizer or loss");
    sphip_train_state *ts = net->train;
    if (reserve(net, n, false) || train_reserve(net, n)) return 1;
    const uint32_t last = net->layers - 1, width = net->topo[last];
    const bool on_dev = (flags & SPHIP_X_ON_DEVICE) != 0;
    const float *d_x = x, *d_t = targets;
    if (restage) {
        if (ts->staged_n != n) return fail_msg("sphip_train_step: SPHIP_TRAIN_SAME_BATCH without a staged batch of this size");
        d_x = ts->act[0];
        d_t = ts->targets;
    } else if (!on_dev) {
        if (train_stage(net, x, targets, n, (flags & SP_TRAIN_WHOLE_SET) != 0)) return 1;
        d_x = ts->act[0];
        d_t = ts->targets;
        ts->staged_n = n;
    }

    const int last_act = net->act[last - 1], mode = out_delta_mode(args->loss_func, last_act);
    bool have_delta = false;

    // forward, every layer kept (Training.c:313-345); a small last layer forms its deltas too (:357-378)
    const float *in = d_x;
    for (uint32_t l = 1; l <= last; ++l) {
        const LayerArgs L = make_layer_args(net, l);
        const bool softmax = net->act[l - 1] == A_SOFTMAX;
        const bool vec = L.K % 4u == 0 && (reinterpret_cast<uintptr_t>(in) & 15u) == 0;
        KSegments seg;
        const bool vector = n <= kF32VectorMax || f32_thin_vector(L, n);
        const uint32_t tile = l == last && !vector ? gemm32_small_tile(n, L.N, L.K, vec, &seg) : 0u;
        float *main_out = softmax ? net->soft_tmp : ts->act[l];
        if (tile == 16u && (!softmax || L.N <= tile)) {
            const Gemm32Args g{L, in, main_out, nullptr, n, 0};
            launch_gemm32_small(g, tile, seg, softmax ? ts->act[l] : nullptr, DeltaTail{d_t, ts->delta[l], mode, last_act});
            have_delta = true;
            break;
        }
        if (l == last && !vector && !tile && gemm32_head_takes(n, L.N, L.K, true, &seg)) {
            launch_gemm32_head(Gemm32Args{L, in, main_out, nullptr, n, 0}, seg, softmax ? ts->act[l] : nullptr,
                               DeltaTail{d_t, ts->delta[l], mode, last_act});
            have_delta = true;
            break;
        }
        bool soft_done = false;
        if (vector) launch_gemv(net->prec, net->workspace(), L, in, main_out, n, false);
        else soft_done = launch_gemm32(L, in, main_out, n, net->split_ws, net->split_cap, softmax ? ts->act[l] : nullptr, n, true);
        if (softmax && !soft_done) sp_softmax_rows<<<(n + 3) / 4, 256, 0, g_stream>>>(net->soft_tmp, ts->act[l], 0, n, net->topo[l]);
        in = ts->act[l];
    }

    if (total_loss) {
        if (grow(&ts->loss_buf, &ts->loss_cap, 3ull * n + 8u)) return 1;
        float *d_loss = ts->loss_buf;
        uint32_t *d_pred = reinterpret_cast<uint32_t *>(d_loss + n), *d_hit = d_pred + n;
        double *d_tot = reinterpret_cast<double *>((reinterpret_cast<uintptr_t>(d_hit + n) + 7u) & ~(uintptr_t)7u);
        EvalArgs ea{ts->act[last], d_t, d_loss, d_pred, d_hit, n, width, args->loss_func, net->act[last - 1] == A_SIGMOID ? 1 : 0};
        sp_eval_rows<<<(n + 3) / 4, 256, 0, g_stream>>>(ea);
        sp_eval_total<<<1, 1024, 0, g_stream>>>(d_loss, d_hit, n, d_tot, reinterpret_cast<uint32_t *>(d_tot + 1));
        double tot = 0.0;
        HCHECK(hipMemcpyAsync(&tot, d_tot, sizeof(double), hipMemcpyDeviceToHost, g_stream));
        HCHECK(hipStreamSynchronize(g_stream));
        *total_loss = (float)tot;
    }

    // deltas (Training.c:347-394)
    if (!have_delta)
        sp_train_out_delta<<<(n + 3) / 4, 256, 0, g_stream>>>(ts->act[last], d_t, ts->delta[last], n, width, mode, last_act);
    for (uint32_t l = last - 1; l > 0; --l) {
        TrGemmArgs g{};
        g.A = ts->delta[l + 1]; g.lda = net->topo[l + 1];
        g.B = reinterpret_cast<const float *>(net->W[l].base); g.ldb = net->topo[l];
        g.C = ts->delta[l]; g.aux = ts->act[l]; g.act = net->act[l - 1];
        g.M = n; g.N = net->topo[l]; g.K = net->topo[l + 1];
        launch_train_delta(g, ts->ws, ts->ws_cap);
    }

    // gradients (Training.c:396-419) and, unless they are clipped by their common norm first, the update (:439-507)
    const bool clipped = args->optimizer >= 0 && args->max_grad_norm > 0.0f;
    const int update = args->optimizer >= 0 && !clipped;
    for (uint32_t l = 0; l < last && args->optimizer >= 0; ++l) net->W[l].cat3_valid = false;   // FP16 parts of the old weights
    train_gradients(net, d_x, n, *args, update);
    HCHECK(hipGetLastError());
    if (!clipped) return 0;

    {
        uint32_t bw = (uint32_t)((ts->total_w + 255) / 256), bb = (uint32_t)((ts->total_b + 255) / 256);
        if (bw > kSqBlocks) bw = kSqBlocks;
        if (bb > kSqBlocks) bb = kSqBlocks;
        sp_train_sumsq_part<<<bw, 256, 0, g_stream>>>(ts->gW, ts->total_w, ts->sq_part);
        sp_train_sumsq_part<<<bb, 256, 0, g_stream>>>(ts->gB, ts->total_b, ts->sq_part + bw);
        sp_train_clip_fin<<<1, 64, 0, g_stream>>>(ts->sq_part, bw + bb, args->max_grad_norm, ts->scal);
    }
    const float *clip = ts->scal;
    for (uint32_t l = 0; l < last; ++l) {
        const uint64_t wc = (uint64_t)net->topo[l] * net->topo[l + 1], bc = net->topo[l + 1];
        launch_opt(*args, reinterpret_cast<float *>(net->W[l].base), ts->gW + ts->woff[l], ts->mW + ts->woff[l], ts->vW + ts->woff[l],
                   wc, args->weight_decay, clip);
        launch_opt(*args, reinterpret_cast<float *>(net->B[l].base), ts->gB + ts->boff[l], ts->mB + ts->boff[l], ts->vB + ts->boff[l],
                   bc, 0.0f, clip);
    }
    HCHECK(hipGetLastError());
    return 0;
}

// `iters` training steps on device-resident inputs between two HIP events on the library's stream; *ms = total elapsed.
// With args->beta*_pow_t fixed the moments keep their first-step correction; the arithmetic per step is the same.
int sphip_time_train_step(sphip_net *net, const float *d_x, const float *d_targets, uint32_t n, const sphip_train_args *args,
                          int iters, float *ms)
{
    if (!net || !d_x || !d_targets || n == 0 || !args || iters <= 0 || !ms) return fail_msg("sphip_time_train_step: invalid argument");
    if (sphip_train_step(net, d_x, d_targets, n, args, SPHIP_X_ON_DEVICE, nullptr)) return 1;      // sizes every buffer
    TimingEvents ev;
    if (ev.create()) return 1;
    hipEvent_t e0 = ev.e0, e1 = ev.e1;
    int rc = 0;
    HCHECK(hipEventRecord(e0, g_stream));
    for (int it = 0; it < iters && !rc; ++it) rc = sphip_train_step(net, d_x, d_targets, n, args, SPHIP_X_ON_DEVICE, nullptr);
    hipError_t e = hipEventRecord(e1, g_stream);
    if (e == hipSuccess) e = hipEventSynchronize(e1);
    if (e == hipSuccess) e = hipEventElapsedTime(ms, e0, e1);
    if (rc) return rc;
    if (e != hipSuccess) return fail_hip("sphip_time_train_step", e);
    return 0;
}

}  // extern "C"
