// hip_gemm32_parts.inl — FP32 forward products of 2 G multiply-adds and more on the BF16 matrix cores (sp_gemm32_bf16_parts).
// Part of hip_forward.hip's translation unit (included there, inside its unnamed namespace, behind hip_gemm32.inl); not
// compiled on its own.

struct PartsGemm32Args {
    const float *A, *B;    // [M][K], [N][K]
    float *C;              // [M][N]
    float *ws;             // [splits][M][N] partial sums when the grid splits K, else nullptr
    const uint8_t *bias;
    float bscale;
    int bias_fmt, act;
    uint32_t M, N, K;
    uint32_t kper;         // k range of one split (multiple of 32)
};

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// two floats as three BF16 parts each, h + m + l == 2^24 x exactly (8 + 8 + 8 significant bits, each part the nearest one).
// The lowest bit of any FP32 number, 2^-149, is a normal BF16 number (from 2^-126 on) after the scaling: unscaled, operands
// below 2^-110 kept fewer than 24 bits.
constexpr float kPartScale = 0x1p24f, kPartSumScale = 0x1p-48f;
__device__ __forceinline__ void bf16_parts2(float x, float y, uint32_t &h, uint32_t &m, uint32_t &l)
{
    x *= kPartScale;
    y *= kPartScale;
    auto pack = [](float a, float b) {
        const bf16x2 v = {(__bf16)a, (__bf16)b};
        uint32_t u;
        __builtin_memcpy(&u, &v, 4);
        return u;
    };
    auto low = [](uint32_t u) { return bits_to_float(u << 16); };
    auto high = [](uint32_t u) { return bits_to_float(u & 0xFFFF0000u); };
    h = pack(x, y);
    x -= low(h); y -= high(h);
    m = pack(x, y);
    x -= low(m); y -= high(m);
    l = pack(x, y);
}

// C = act(A B^T + bias) with each FP32 operand as three BF16 parts and those six of the nine products of parts that reach
// 2^-24 of the whole: hl + lh + mm + hm + mh + hh, smallest first, in one FP32 accumulator.  v_mfma_f32_32x32x16_bf16 does
// in 6 x 8 passes what v_mfma_f32_32x32x2_f32 does in 8 x 16, and rounds the accumulator 6 times per 16 k instead of 8:
// the error against 64 bits is the smaller one at every size tried (relative, 2-norm, FP32 matrix cores -> here: 20000 x 512
// x 784 5.1e-7 -> 4.3e-7, 4096 x 4096 x 4096 1.15e-6 -> 1.00e-6, 700 x 3000 x 3000 9.9e-7 -> 3.5e-7, 8192 x 16384 x 64 1.4e-7 ->
// 1.1e-7), and so it is for operands down to the smallest subnormal ones, which the splitting scales up.
// Tile (64 TM) x 128 x 32, four waves of (32 TM) x 64; the FP32 elements of the next K tile are loaded while the matrix
// cores work, split in registers on their way into LDS: [operand][part][row][32 k], the 16-byte units of a row XOR-ed with
// row / 4, so that the 16 rows of a read cycle lie in different banks.  48 KB (TM = 2) and one stage: three workgroups
// share a compute unit, and one's splitting runs beside another's products.  Bound by the matrix cores and the splitting's
// vector instructions together: 4096 x 4096 x 4096 1070 -> 732 us (188 TFLOP/s of FP32 products, 1.13 PFLOP/s of BF16),
// 20000 x 1000 x 512 221 -> 124, 2000 x 4096 x 4096 600 -> 353, 512 x 4096 x 4096 (split over K) 178 -> 107.  (Of that the
// scaling of the operands costs between -3 and 4 %: 723, 123, 364 and 110 us without it.)  Rows that are not whole 16-byte
// units are loaded 16 bytes at a time all the same (10000 x 1000 x 1001 278 -> 142 us, 10000 x 1872 x 4650
// 1980 -> 1005; element by element before).
// Infinities and operands from 2^104 on have no such parts, sums from 2^80 on no room for their scale: an element whose sum
// comes out infinite or NaN is formed again as a chain of FP32 products.
template <int TM>
__global__ __launch_bounds__(256) void sp_gemm32_bf16_parts(const PartsGemm32Args g)
{
    constexpr uint32_t BM = 64 * TM, BN = 128, BK = 32;
    constexpr uint32_t PA = BM * BK, PB = BN * BK;        // 16-bit elements of one part of an operand
    __shared__ __attribute__((aligned(16))) uint16_t lds[3 * (PA + PB)];
    const uint32_t M = g.M, N = g.N, K = g.K;
    const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6;
    const uint32_t wm = wave >> 1, wn = wave & 1u, q = lane & 31u, h = lane >> 5;
    // each XCD a contiguous run of tiles, walked in groups of 8 row tiles x all column tiles, the 8 row tiles of a
    // column tile one after the other: the workgroups an XCD holds share few panels
    uint32_t m0, n0;
    {
        constexpr uint32_t GM = 8;
        const uint32_t tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN, per = gridDim.x / 8u;
        uint32_t bid = blockIdx.x;
        if (bid < per * 8u) bid = (bid & 7u) * per + (bid >> 3);
        const uint32_t group = bid / (GM * tiles_n), first = group * GM;
        const uint32_t rows = tiles_m - first < GM ? tiles_m - first : GM;
        const uint32_t in = bid - group * GM * tiles_n;
        m0 = (first + in % rows) * BM;
        n0 = (in / rows) * BN;
    }
    const uint32_t kbeg = blockIdx.y * g.kper;
    const uint32_t kend = kbeg + g.kper < K ? kbeg + g.kper : K;

    f32x16 acc[TM][2];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

    // a thread carries eight k (unit t % 4 of the tile's four) of rows t / 4, t / 4 + 64, ... of each operand; a row past
    // the end repeats the last one, its products are not stored
    const uint32_t row = t >> 2, unit = t & 3u;
    const float *pa[TM], *pb[2];
#pragma unroll
    for (uint32_t i = 0; i < (uint32_t)TM; ++i) pa[i] = g.A + (size_t)(m0 + row + 64u * i < M ? m0 + row + 64u * i : M - 1u) * K;
#pragma unroll
    for (uint32_t i = 0; i < 2u; ++i) pb[i] = g.B + (size_t)(n0 + row + 64u * i < N ? n0 + row + 64u * i : N - 1u) * K;
    float fa[TM][8], fb[2][8];
    auto fetch = [&](float (&f)[8], const float *p, uint32_t k0) {
        const uint32_t k = k0 + unit * 8u;
        if (k0 + BK <= kend) {
            // (rows begin anywhere: the wide loads want no more than the alignment of a float)
            const float4_any v0 = *reinterpret_cast<const float4_any *>(p + k), v1 = *reinterpret_cast<const float4_any *>(p + k + 4u);
            f[0] = v0.x; f[1] = v0.y; f[2] = v0.z; f[3] = v0.w;
            f[4] = v1.x; f[5] = v1.y; f[6] = v1.z; f[7] = v1.w;
        } else {
#pragma unroll
            for (uint32_t e = 0; e < 8u; ++e) {
                const float v = p[k + e < kend ? k + e : kend - 1u];
                f[e] = k + e < kend ? v : 0.0f;
            }
        }
    };
    const uint32_t at = row * BK + (unit ^ (row >> 2 & 3u)) * 8u;      // (64 rows on: the same place of its bank cycle)
    auto stash = [&](const float (&f)[8], uint16_t *op, uint32_t part) {
        u32x4 p[3];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            uint32_t hi, mid, lo;
            bf16_parts2(f[2 * e], f[2 * e + 1], hi, mid, lo);
            p[0][e] = hi; p[1][e] = mid; p[2][e] = lo;
        }
#pragma unroll
        for (uint32_t s = 0; s < 3u; ++s) *reinterpret_cast<u32x4 *>(op + s * part + at) = p[s];
    };
    auto fetch_all = [&](uint32_t k0) {
#pragma unroll
        for (int i = 0; i < TM; ++i) fetch(fa[i], pa[i], k0);
#pragma unroll
        for (int i = 0; i < 2; ++i) fetch(fb[i], pb[i], k0);
    };

    fetch_all(kbeg);
    for (uint32_t k0 = kbeg; k0 < kend; k0 += BK) {
#pragma unroll
        for (int i = 0; i < TM; ++i) stash(fa[i], lds + 64 * i * BK, PA);
#pragma unroll
        for (int i = 0; i < 2; ++i) stash(fb[i], lds + 3 * PA + 64 * i * BK, PB);
        __syncthreads();
        if (k0 + BK < kend) fetch_all(k0 + BK);
#pragma unroll
        for (uint32_t ks = 0; ks < 2u; ++ks) {
            const uint32_t u = 2u * ks + h;
            bf16x8 a[TM][3], b[2][3];
#pragma unroll
            for (uint32_t s = 0; s < 3u; ++s) {
#pragma unroll
                for (uint32_t i = 0; i < (uint32_t)TM; ++i) {
                    const uint32_t r = (wm * TM + i) * 32u + q;
                    a[i][s] = *reinterpret_cast<const bf16x8 *>(lds + s * PA + r * BK + (u ^ (r >> 2 & 3u)) * 8u);
                }
#pragma unroll
                for (uint32_t j = 0; j < 2u; ++j) {
                    const uint32_t r = (wn * 2u + j) * 32u + q;
                    b[j][s] = *reinterpret_cast<const bf16x8 *>(lds + 3 * PA + s * PB + r * BK + (u ^ (r >> 2 & 3u)) * 8u);
                }
            }
            constexpr int sa[6] = {0, 2, 1, 0, 1, 0}, sb[6] = {2, 0, 1, 1, 0, 0};
#pragma unroll
            for (int s = 0; s < 6; ++s)
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i][sa[s]], b[j][sb[s]], acc[i][j], 0, 0, 0);
        }
        __syncthreads();
    }

    auto bias_of = [&](uint32_t n) { return elem_value_rt(g.bias_fmt, g.bias, n) * g.bscale; };
    // element e = 32 j + 16 i + r of a thread
    auto row_of = [&](uint32_t e) { return m0 + (wm * TM + (e >> 4 & 1u)) * 32u + 8u * (e >> 2 & 3u) + 4u * h + (e & 3u); };
    auto col_of = [&](uint32_t e) { return n0 + (wn * 2u + (e >> 5)) * 32u + q; };
    uint64_t again = 0;                                    // the elements whose sum is not finite
    with_act(g.act, [&](auto act_c) __attribute__((always_inline)) {
        constexpr int ACT = decltype(act_c)::value;
#pragma unroll
        for (uint32_t j = 0; j < 2u; ++j) {
            const uint32_t n = col_of(32u * j);
            if (n >= N) continue;
            const float bias = bias_of(n);
#pragma unroll
            for (uint32_t i = 0; i < (uint32_t)TM; ++i)
#pragma unroll
                for (uint32_t r = 0; r < 16u; ++r) {
                    const uint32_t e = 32u * j + 16u * i + r, m = row_of(e);
                    if (m >= M) continue;
                    const float v = acc[i][j][r];
                    if (!(fabsf(v) < __builtin_inff())) again |= 1ull << e;
                    const size_t o = (size_t)m * N + n;
                    if (g.ws) g.ws[(size_t)blockIdx.y * M * N + o] = v * kPartSumScale;
                    else g.C[o] = apply_act(fmaf(v, kPartSumScale, bias), ACT);
                }
        }
    });
    while (again) {
        const uint32_t e = (uint32_t)__builtin_ctzll(again), m = row_of(e), n = col_of(e);
        again &= again - 1u;
        const float *a = g.A + (size_t)m * K, *b = g.B + (size_t)n * K;
        float s = 0.0f;
        for (uint32_t k = kbeg; k < kend && s == s; ++k) s = fmaf(a[k], b[k], s);
        const size_t o = (size_t)m * N + n;
        if (g.ws) g.ws[(size_t)blockIdx.y * M * N + o] = s;
        else g.C[o] = apply_act(s + bias_of(n), g.act);
    }
}
