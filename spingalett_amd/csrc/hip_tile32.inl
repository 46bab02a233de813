// hip_tile32.inl — sp_gemm32_f32: C(m, n) = sum over k of A(m, k) B(n, k) in FP32, for forwards that keep the order of their
// sums and for both products of a training step's backward.  Part of hip_forward.hip's translation unit (included there,
// inside its unnamed namespace); not compiled on its own.

enum { T32_LAYER = 0, T32_DELTA = 1, T32_SCALE = 2 };

struct Tile32Args {
    const float *A, *B;
    float *C;              // [M][N]
    float *ws;             // [splits][M][N] partial sums when the grid splits K, else nullptr
    const float *aux;      // T32_DELTA: activations [M][N] whose derivative multiplies the product
    const uint8_t *bias;   // T32_LAYER
    int bias_fmt;
    float bscale;
    uint32_t M, N, K, lda, ldb;
    uint32_t kper;         // k range of one split (multiple of 32)
    int act;               // T32_LAYER: of the layer, T32_DELTA: of aux
    float scale;           // T32_SCALE
};

template <bool MC, int R>
struct Tile32Side {
    static constexpr int SIZE = 32 * R;                         // floats of a K tile: [k][R] or [row][32]
    static constexpr int PIECES = SIZE / 4 / 256;               // of four floats, per thread
    // What lies at piece p of a K tile: row (the first of four) and k (the first of four).  Odd k of [k][R] have their halves
    // of 32 floats changed over, so that the two k a wave reads at once lie in different banks; two rows of [row][32] are 64
    // banks, their pieces turned by the pair's number.
    static __device__ __forceinline__ void piece(int p, uint32_t &r, uint32_t &k)
    {
        if constexpr (MC) {
            k = (uint32_t)(p / (R / 4));
            r = (uint32_t)(p % (R / 4)) * 4u ^ ((k & 1u) << 5);
        } else {
            r = (uint32_t)p >> 3;
            k = (((uint32_t)p & 7u) ^ (((uint32_t)p >> 4) & 7u)) * 4u;
        }
    }
};

// 64 x (64 TN) x 32 tile, four waves of 32 x (32 TN), the 32 x 32 x 2 MFMAs of an output in ascending order of k.  Each operand is
// k-contiguous (element (r, k) at r * ld + k) or row-contiguous (at k * ld + r): a forward has neither row-contiguous, the
// hidden deltas the weights, the gradients both.
//
// The FP32 matrix instructions leave the vector ALU no room: registers only, one 32 x 32 x 2 MFMA alone takes its 64 cycles
// (153 TFLOP/s), with two vector instructions behind it 75 to 87, with eight 85 to 111.  So the loop has none: K tiles go
// from memory into one of two LDS stages by DMA, behind a scalar base that moves on by scalar adds; every LDS address of
// either stage has a register of its own (b32 reads, as an MFMA wants k = 2 s on its lower and 2 s + 1 on its upper lanes: wider
// ones with an exchange between the halves were slower, 20000 x 512 x 1000 194 us against 187); the outputs leave by a scalar base
// per row.  Against the kernels before, which staged through registers with addresses and conditions computed on the way:
//   20000 x 1000 x 512 forward         214 -> 190 us     20000 x 512 x 1000 deltas              232 -> 186
//   20000 x 512 x 784                  171 -> 151        1000 x 512 x 20000 gradients, 8 splits 207 -> 162 (126 TFLOP/s)
//   20000 x 10 x 1000                   58 -> 39         512 x 784 x 20000, 10 splits           207 -> 171
// Where K is long it is the waits at the barriers that remain, where K is short the first loads and the outputs of tiles that
// all begin and end together.
template <int EPI, bool AMC, bool BMC, int TN>
__global__ __launch_bounds__(256) void sp_gemm32_f32(const Tile32Args g)
{
    constexpr int BM = 64, BN = 64 * TN, BK = 32;
    using SA = Tile32Side<AMC, BM>;
    using SB = Tile32Side<BMC, BN>;
    extern __shared__ __attribute__((aligned(1024))) float smem32[];
    const uint32_t M = g.M, N = g.N, K = g.K;
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int wm = wave >> 1, wn = wave & 1, q = lane & 31, h = lane >> 5;
    const uint32_t tiles_n = (N + BN - 1) / BN;
    uint32_t bid = blockIdx.x;
    {
        const uint32_t per = gridDim.x / 8u;
        if (bid < per * 8u) bid = (bid & 7u) * per + (bid >> 3);
    }
    const uint32_t m0 = (bid / tiles_n) * BM, n0 = (bid % tiles_n) * BN;
    const uint32_t kbeg = blockIdx.y * g.kper;
    const uint32_t kend = kbeg + g.kper < K ? kbeg + g.kper : K;

    // Where a thread's pieces come from (rows beyond the end: the last ones again, never stored), and where it reads its operands
    uint32_t from_a[SA::PIECES], from_b[SB::PIECES];
    uint32_t at_a[2][1][AMC ? 1 : 8], at_b[2][TN][BMC ? 1 : 8];
    auto sources = [&](auto side, auto mc, uint32_t (&from)[decltype(side)::PIECES], uint32_t ld, uint32_t r0, uint32_t R) {
#pragma unroll
        for (int i = 0; i < decltype(side)::PIECES; ++i) {
            uint32_t r, k;
            decltype(side)::piece((wave + 4 * i) * 64 + lane, r, k);
            const uint32_t top = R - r0 - (decltype(mc)::value ? 4u : 1u);
            r = r < top ? r : top;
            from[i] = decltype(mc)::value ? (k * ld + r) * 4u : (r * ld + k) * 4u;
            asm volatile("" : "+v"(from[i]));
        }
    };
    sources(SA{}, std::bool_constant<AMC>{}, from_a, g.lda, m0, M);
    sources(SB{}, std::bool_constant<BMC>{}, from_b, g.ldb, n0, N);
    constexpr int STAGE = SA::SIZE + SB::SIZE;
    // one register per address, whatever the stage: a vector instruction between these MFMAs costs them 10 to 25 cycles
    auto places = [&](auto mc, auto rows, auto &at, int tiles, int first, int base) {
        constexpr int R = decltype(rows)::value;
#pragma unroll
        for (int st = 0; st < 2; ++st)
#pragma unroll
            for (int i = 0; i < tiles; ++i)
#pragma unroll
                for (int p = 0; p < (decltype(mc)::value ? 1 : 8); ++p) {
                    at[st][i][p] = (uint32_t)(base + st * STAGE) +
                                   (decltype(mc)::value ? (uint32_t)(h * R + ((first + i * 32 + q) ^ (h << 5)))
                                                        : (uint32_t)((first + i * 32 + q) * 32 + ((p ^ ((q >> 1) & 7)) * 4) + h));
                    asm volatile("" : "+v"(at[st][i][p]));
                }
    };
    places(std::bool_constant<AMC>{}, std::integral_constant<int, BM>{}, at_a, 1, wm * 32, 0);
    places(std::bool_constant<BMC>{}, std::integral_constant<int, BN>{}, at_b, TN, wn * TN * 32, SA::SIZE);

    const float *pa = AMC ? g.A + (size_t)kbeg * g.lda + m0 : g.A + (size_t)m0 * g.lda + kbeg;
    const float *pb = BMC ? g.B + (size_t)kbeg * g.ldb + n0 : g.B + (size_t)n0 * g.ldb + kbeg;
    const size_t step_a = AMC ? (size_t)BK * g.lda : BK, step_b = BMC ? (size_t)BK * g.ldb : BK;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void *)smem32;
    // the next K tile into a stage; one that is cut short goes through registers, zeros behind its end
    auto side_in = [&](auto side, uint32_t to, const float *p, const uint32_t *from, uint32_t have) __attribute__((always_inline)) {
        if (have == (uint32_t)BK) {
#pragma unroll
            for (int i = 0; i < decltype(side)::PIECES; ++i) lds_dma16(lds0 + to * 4u + (uint32_t)(wave + 4 * i) * 1024u, from[i], p);
        } else {
#pragma unroll
            for (int i = 0; i < decltype(side)::PIECES; ++i) {
                uint32_t r, k;
                decltype(side)::piece((wave + 4 * i) * 64 + lane, r, k);
                float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                if (k < have) v = *reinterpret_cast<const float4 *>(reinterpret_cast<const char *>(p) + from[i]);
                *reinterpret_cast<float4 *>(smem32 + to + ((wave + 4 * i) * 64 + lane) * 4) = v;
            }
        }
    };
    auto next = [&](int stage, uint32_t have) __attribute__((always_inline)) {
        side_in(SA{}, (uint32_t)(stage * STAGE), pa, from_a, have);
        side_in(SB{}, (uint32_t)(stage * STAGE + SA::SIZE), pb, from_b, have);
        pa += step_a;
        pb += step_b;
    };

    f32x16 acc[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[j][r] = 0.0f;
    auto compute = [&](auto stage) __attribute__((always_inline)) {
        constexpr int ST = decltype(stage)::value;
#pragma unroll
        for (int s = 0; s < BK / 2; ++s) {                       // k = 2 s + h
            float b[TN];
            const float a = AMC ? smem32[at_a[ST][0][0] + 2 * s * BM] : smem32[at_a[ST][0][AMC ? 0 : s >> 1] + (2 * s & 2)];
#pragma unroll
            for (int i = 0; i < TN; ++i) b[i] = BMC ? smem32[at_b[ST][i][0] + 2 * s * BN] : smem32[at_b[ST][i][BMC ? 0 : s >> 1] + (2 * s & 2)];
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, b[j], acc[j], 0, 0, 0);
        }
    };
    auto meet = [&]() __attribute__((always_inline)) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
    };

    // the first K tile of an odd number by itself, then pairs; only the very last one can be cut short
    const std::integral_constant<int, 0> even;
    const std::integral_constant<int, 1> odd;
    const uint32_t nk = (kend - kbeg + BK - 1) / BK, last = kend - kbeg - (nk - 1) * BK;
    if (nk & 1u) {
        next(1, nk > 1u ? BK : last);
        meet();
        if (nk > 1u) next(0, BK);
        compute(odd);
    } else {
        next(0, BK);
    }
    meet();
    for (uint32_t pairs = nk / 2u; pairs; --pairs) {
        next(1, pairs > 1u ? BK : last);
        compute(even);
        meet();
        if (pairs > 1u) next(0, BK);
        compute(odd);
        meet();
    }

    // out[row][col] = f(sum, of(col), in[row][col])
    auto emit = [&](float *out, auto of, auto in, auto f) __attribute__((always_inline)) {
        constexpr bool IN = !std::is_same_v<decltype(in), std::nullptr_t>;
        const uint32_t first = m0 + (uint32_t)wm * 32u, have = first < M ? M - first : 0u;
        const uint32_t lane_at = (uint32_t)(4 * h) * N + q;
        auto row = [&](int r) { return (uint32_t)(8 * (r >> 2) + (r & 3)); };        // + 4 h
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const uint32_t col0 = n0 + (wn * TN + j) * 32;
            if (col0 + q >= N) continue;
            const float c = of(col0 + q);
            const size_t at0 = (size_t)first * N + col0;
            float x[16];
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                x[r] = 0.0f;
                if constexpr (IN)
                    if (row(r) + 4u * h < have) x[r] = (in + at0 + (size_t)row(r) * N)[lane_at];
            }
            if (have >= 32u) {
#pragma unroll
                for (int r = 0; r < 16; ++r) (out + at0 + (size_t)row(r) * N)[lane_at] = f(acc[j][r], c, x[r]);
            } else {
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    if (row(r) + 4u * h < have) (out + at0 + (size_t)row(r) * N)[lane_at] = f(acc[j][r], c, x[r]);
            }
        }
    };
    auto nothing = [](uint32_t) { return 0.0f; };
    if (g.ws) {
        emit(g.ws + (size_t)blockIdx.y * M * N, nothing, nullptr, [](float v, float, float) { return v; });
    } else if constexpr (EPI == T32_LAYER) {
        with_act(g.act, [&](auto act_c) __attribute__((always_inline)) {
            emit(g.C, [&](uint32_t col) { return elem_value_rt(g.bias_fmt, g.bias, col) * g.bscale; }, nullptr,
                 [](float v, float bias, float) { return apply_act(v + bias, decltype(act_c)::value); });
        });
    } else if constexpr (EPI == T32_DELTA) {
        with_act(g.act, [&](auto act_c) __attribute__((always_inline)) {
            emit(g.C, nothing, g.aux, [](float v, float, float x) { return v * act_derivative(x, decltype(act_c)::value); });
        });
    } else {
        emit(g.C, nothing, nullptr, [&](float v, float, float) { return g.scale * v; });
    }
}

// One launch of it: both operands at multiples of 16 bytes, rows of multiples of four floats, and byte offsets within a tile, of
// up to 128 rows, that 32 bits hold (gemm32_tile_takes()).  64 x 128 tiles where that leaves four per compute unit: 20000 x 512 x 1000 by the weights
// 185 us against 191 with 64 x 64, 20000 x 512 x 784 forward 151 against 160, but 4096 x 512 x 784 35.4 against 34.0; the gradient
// products, which are cut to about four 64 x 64 tiles per unit, 183 against 173 (512 x 784 x 20000).
// And where the second half of the last tile is not mostly padding: 70000 x 10 x 512 86 us against 54, x 160 x 168 75 / 58, x 320 x 84
// 68 / 58, 20000 x 576 x 164 60 / 52, x 960 x 96 52 / 47, x 1088 x 84 even.
bool gemm32_tile_takes(const void *a, const void *b, uint32_t lda, uint32_t ldb)
{
    auto fits = [](const void *p, uint32_t ld) { return ld % 4u == 0 && ld <= (1u << 23) && (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
    return fits(a, lda) && fits(b, ldb);
}

template <int EPI, bool AMC, bool BMC>
void launch_gemm32_tile(const Tile32Args &g, uint32_t splits)
{
    const uint32_t rows = (g.M + 63u) / 64u, cols = (g.N + 63u) / 64u;
    if constexpr (EPI != T32_SCALE) {
        const uint32_t wide = (cols + 1u) / 2u;
        if ((uint64_t)rows * wide >= 1024u && (cols % 2u == 0 || cols >= 17u)) {
            sp_gemm32_f32<EPI, AMC, BMC, 2><<<dim3(rows * wide, splits), 256, 2u * (64u + 128u) * 32u * sizeof(float), g_stream>>>(g);
            return;
        }
    }
    sp_gemm32_f32<EPI, AMC, BMC, 1><<<dim3(rows * cols, splits), 256, 2u * (64u + 64u) * 32u * sizeof(float), g_stream>>>(g);
}
