// hip_gemm16.inl — the LDS-tiled 16-bit MFMA GEMM for larger batches (sp_gemm16, sp_gemm16_big,
// sp_gemm16_reduce).  Part of hip_kernels.h (included there,
// inside its namespace); not compiled on its own.

// ---------------------------------------------------------------------------
// 16-bit MFMA GEMM (n > 64): C[M][N] = act(bias + scale * A[M][K] . Wq[N][K]^T)
// ---------------------------------------------------------------------------
typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(8 * sizeof(_Float16)))) _Float16 f16x8;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;

struct GemmArgs {
    LayerArgs L;
    const uint16_t *A;     // [M][K] 16-bit activations
    void *C;               // [M][N] 16-bit, or FP32 when out_f32
    uint32_t M;
    int out_f32;
    float *ws;             // [grid y][M][N] partial sums when grid y splits the product, else nullptr
    uint32_t kper;         // k range of one K split, a multiple of 64 (0: all of K)
    // Split activations: the layer input is two 16-bit matrices, hi and (a - hi) 2^11, the second M K elements
    // behind the first; grid y = halves x ksplits, y / ksplits picks the matrix, y % ksplits the K range.
    uint32_t ksplits;      // K splits (>= 1)
    uint32_t halves;       // 1, or 2 with split activations
};

// 2^-11: what the partial sums of the second activation matrix are scaled by
constexpr float kLoScale = 1.0f / 2048.0f;

// hi and lo of a split activation: hi = v rounded to FP16, lo = (v - hi) 2^11 rounded to FP16 (v - hi is exact in FP32)
__device__ __forceinline__ void split_f16(float v, uint16_t &hi, uint16_t &lo)
{
    hi = f32_to_f16_sat(v);
    _Float16 hh;
    __builtin_memcpy(&hh, &hi, 2);
    const float rest = (v - (float)hh) * 2048.0f;
    lo = (rest == rest && fabsf(rest) != __builtin_inff()) ? f32_to_f16_sat(rest) : (uint16_t)0;   // inf / NaN live in hi
}

// (float)q as a 16-bit float; exact for |q| <= 128 in either type
template <bool F16T>
__device__ __forceinline__ uint32_t int_to_t16(int q)
{
    if constexpr (F16T) {
        _Float16 h = (_Float16)q;
        uint16_t r;
        __builtin_memcpy(&r, &h, 2);
        return r;
    } else {
        return __float_as_uint((float)q) >> 16;
    }
}

// packed FP16 subtraction a - c (two lanes at once)
__device__ __forceinline__ uint32_t h2_sub(uint32_t v, uint32_t c)
{
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    h2 a, b;
    __builtin_memcpy(&a, &v, 4);
    __builtin_memcpy(&b, &c, 4);
    a = a - b;
    uint32_t r;
    __builtin_memcpy(&r, &a, 4);
    return r;
}

// unpack one 32-bit word of codes into 16-bit floats, written as packed pairs (codes 0 1, 2 3, ...)
template <int FMT, bool F16T>
__device__ __forceinline__ void unpack_word16(uint32_t w, uint32_t *o)
{
    constexpr int bits = fmt_bits(FMT);
    constexpr int cnt = 32 / bits;
    if constexpr (F16T && (FMT == I8 || FMT == I4 || FMT == I2)) {
        // A field masked in place and XORed onto an FP16 constant whose last mantissa bit weighs as much as
        // the field's lowest bit (the same XOR flips the sign bit: two's complement -> offset binary) reads
        // as constant + offset + code; one packed subtraction leaves the codes of two fields, exactly.  The
        // pairs come out as (code k, code k + cnt/2) and a byte permute puts neighbours together.
        constexpr uint32_t LO = 0x05040100u, HI = 0x07060302u;      // low / high halves of two words
        if constexpr (FMT == I8) {
            const uint32_t t0 = h2_sub((w & 0x00FF00FFu) ^ 0x64806480u, 0x64806480u);            // codes 0, 2
            const uint32_t t1 = h2_sub(((w >> 8) & 0x00FF00FFu) ^ 0x64806480u, 0x64806480u);     // codes 1, 3
            o[0] = __builtin_amdgcn_perm(t1, t0, LO);
            o[1] = __builtin_amdgcn_perm(t1, t0, HI);
        } else if constexpr (FMT == I4) {
            const uint32_t y = w >> 8;
            const uint32_t t0 = h2_sub((w & 0x000F000Fu) ^ 0x64086408u, 0x64086408u);            // codes 0, 4
            const uint32_t t1 = h2_sub((w & 0x00F000F0u) ^ 0x54805480u, 0x54805480u);            // codes 1, 5
            const uint32_t t2 = h2_sub((y & 0x000F000Fu) ^ 0x64086408u, 0x64086408u);            // codes 2, 6
            const uint32_t t3 = h2_sub((y & 0x00F000F0u) ^ 0x54805480u, 0x54805480u);            // codes 3, 7
            o[0] = __builtin_amdgcn_perm(t1, t0, LO);
            o[1] = __builtin_amdgcn_perm(t3, t2, LO);
            o[2] = __builtin_amdgcn_perm(t1, t0, HI);
            o[3] = __builtin_amdgcn_perm(t3, t2, HI);
        } else {
            const uint32_t y = w >> 10;
            uint32_t p[8];                                                                        // codes k, k + 8
            p[0] = h2_sub((w & 0x00030003u) ^ 0x64026402u, 0x64026402u);
            p[1] = h2_sub((w & 0x000C000Cu) ^ 0x5C085C08u, 0x5C085C08u);
            p[2] = h2_sub((w & 0x00300030u) ^ 0x54205420u, 0x54205420u);
            p[3] = h2_sub((w & 0x00C000C0u) ^ 0x4C804C80u, 0x4C804C80u);
            p[4] = h2_sub((w & 0x03000300u) ^ 0x46004600u, 0x46004600u);
            p[5] = h2_sub((y & 0x00030003u) ^ 0x64026402u, 0x64026402u);
            p[6] = h2_sub((y & 0x000C000Cu) ^ 0x5C085C08u, 0x5C085C08u);
            p[7] = h2_sub((y & 0x00300030u) ^ 0x54205420u, 0x54205420u);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                o[q]     = __builtin_amdgcn_perm(p[2 * q + 1], p[2 * q], LO);
                o[4 + q] = __builtin_amdgcn_perm(p[2 * q + 1], p[2 * q], HI);
            }
        }
        return;
    }
#pragma unroll
    for (int j = 0; j < cnt; j += 2) {
        int q0 = (int)(w << (32 - bits - bits * j)) >> (32 - bits);
        int q1 = (int)(w << (32 - bits - bits * (j + 1))) >> (32 - bits);
        o[j / 2] = int_to_t16<F16T>(q0) | (int_to_t16<F16T>(q1) << 16);
    }
}

// Tile: BM x BN x BK (BK = 64, or 128 for a K of 1024 and more), 256 threads = 2 x 2 waves, each wave TM x TN tiles of
// 32x32.  A K split (g.kper) is of whole tiles.
// LDS rows are padded by 8 elements so that 128-bit fragment reads of 32
// consecutive rows spread over the banks.
// W4 (integer codes, ALIGNED activations): the weight rows are whole 32-bit words but not whole 16-byte units
// (784 INT4 codes = 392 bytes): the codes are fetched a word at a time instead of element by element.
template <int FMT, bool F16T, int TM, int TN, bool ALIGNED, bool W4 = false, int BK = 64>
__global__ __launch_bounds__(256) void sp_gemm16(const GemmArgs g)
{
    static_assert(!W4 || (ALIGNED && (FMT == I8 || FMT == I4 || FMT == I2)), "word loads: integer codes, aligned activations");
    constexpr int BM = 64 * TM, BN = 64 * TN, LDK = BK + 8;
    constexpr int KCH = BK / 8;                     // 16-byte pieces of a tile row of activations
    constexpr int bits = fmt_bits(FMT);
    constexpr int EPL = 128 / bits;                 // weight elements per 16-byte load
    constexpr int W_LOADS = (BN * BK / EPL + 255) / 256;
    constexpr int A_LOADS = BM * BK / 8 / 256;
    constexpr int CW = 32 / bits;                   // codes per 32-bit word
    constexpr int W4_LOADS = (BN * BK / CW + 255) / 256;

    __shared__ __attribute__((aligned(16))) uint16_t As[BM * LDK];
    __shared__ __attribute__((aligned(16))) uint16_t Ws[BN * LDK];

    const uint32_t M = g.M, N = g.L.N, K = g.L.K;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    // grid y = halves x K splits: y / ksplits picks the matrix of a split activation, y % ksplits the K range (whole tiles)
    const uint16_t *const A = g.A + (size_t)(blockIdx.y / g.ksplits) * M * K;
    const uint32_t kbeg = g.kper ? (blockIdx.y % g.ksplits) * g.kper : 0u;
    const uint32_t kend = g.kper && kbeg + g.kper < K ? kbeg + g.kper : K;

    // tile index: consecutive workgroups go to different XCDs, so give each XCD a
    // contiguous band of tiles (shared A rows / W rows stay in one L2)
    const uint32_t tiles_n = (N + BN - 1) / BN, tiles_m = (M + BM - 1) / BM;
    const uint32_t ntiles = tiles_m * tiles_n;
    uint32_t bid = blockIdx.x;
    {
        const uint32_t per = ntiles / 8u;
        if (bid < per * 8u) bid = (bid & 7u) * per + (bid >> 3);
    }
    const uint32_t tm = bid / tiles_n, tn = bid % tiles_n;
    const uint32_t m0 = tm * BM, n0 = tn * BN;

    f32x16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

    uint4 ra[A_LOADS], rw[W4 ? 1 : W_LOADS];
    uint32_t rw4[W4 ? W4_LOADS : 1];
    const size_t w_row_bytes = (size_t)K * bits / 8u;

    auto load_tiles = [&](uint32_t k0) {
        if constexpr (ALIGNED) {
#pragma unroll
            for (int i = 0; i < A_LOADS; ++i) {
                const int c = t + 256 * i, row = c / KCH, kc = c % KCH;
                const uint32_t m = m0 + row < M ? m0 + row : M - 1;
                const uint32_t k = k0 + kc * 8;
                ra[i] = k < K ? *reinterpret_cast<const uint4 *>(A + (size_t)m * K + k) : make_uint4(0, 0, 0, 0);
            }
            if constexpr (W4) {
#pragma unroll
                for (int i = 0; i < W4_LOADS; ++i) {
                    const int c = t + 256 * i;
                    constexpr int LPR = BK / CW;        // words per tile row
                    const int row = c / LPR, kc = c % LPR;
                    const uint32_t n = n0 + row < N ? n0 + row : N - 1;
                    const uint32_t k = k0 + kc * CW;
                    const bool ok = (row < BN) && (k < K);      // K is a whole number of words: k < K means k + CW <= K
                    rw4[i] = ok ? *reinterpret_cast<const uint32_t *>(g.L.w + (size_t)n * w_row_bytes + (size_t)k * bits / 8u) : 0u;
                }
            } else {
#pragma unroll
                for (int i = 0; i < W_LOADS; ++i) {
                    const int c = t + 256 * i;
                    constexpr int LPR = BK / EPL;           // loads per tile row
                    const int row = c / LPR, kc = c % LPR;
                    const uint32_t n = n0 + row < N ? n0 + row : N - 1;
                    const uint32_t k = k0 + kc * EPL;
                    const bool ok = (row < BN) && (k < K);
                    rw[i] = ok ? *reinterpret_cast<const uint4 *>(g.L.w + (size_t)n * w_row_bytes + (size_t)k * bits / 8u)
                               : make_uint4(0, 0, 0, 0);
                }
            }
        }
    };

    auto store_tiles = [&](uint32_t k0) {
        if constexpr (ALIGNED) {
#pragma unroll
            for (int i = 0; i < A_LOADS; ++i) {
                const int c = t + 256 * i, row = c / KCH, kc = c % KCH;
                *reinterpret_cast<uint4 *>(&As[row * LDK + kc * 8]) = ra[i];
            }
            if constexpr (W4) {
#pragma unroll
                for (int i = 0; i < W4_LOADS; ++i) {
                    const int c = t + 256 * i;
                    constexpr int LPR = BK / CW;
                    const int row = c / LPR, kc = c % LPR;
                    if (row >= BN) continue;
                    constexpr int PW = 16 / bits;       // packed pairs per 32-bit word: 2, 4 or 8
                    uint32_t o[PW];
                    unpack_word16<FMT, F16T>(rw4[i], o);
                    uint16_t *dst = &Ws[row * LDK + kc * CW];
                    if constexpr (PW == 2) {
                        *reinterpret_cast<uint2 *>(dst) = make_uint2(o[0], o[1]);
                    } else {
#pragma unroll
                        for (int v = 0; v < PW / 4; ++v)
                            *reinterpret_cast<uint4 *>(dst + v * 8) = make_uint4(o[4 * v], o[4 * v + 1], o[4 * v + 2], o[4 * v + 3]);
                    }
                }
            }
#pragma unroll
            for (int i = 0; i < (W4 ? 0 : W_LOADS); ++i) {
                const int c = t + 256 * i;
                constexpr int LPR = BK / EPL;
                const int row = c / LPR, kc = c % LPR;
                if (row >= BN) continue;
                uint16_t *dst = &Ws[row * LDK + kc * EPL];
                if constexpr (FMT == BF16 || FMT == F16) {
                    *reinterpret_cast<uint4 *>(dst) = rw[i];
                } else {
                    const uint32_t w[4] = {rw[i].x, rw[i].y, rw[i].z, rw[i].w};
                    constexpr int PW = 16 / bits;       // packed pairs per 32-bit word
                    uint32_t o[4 * PW];
#pragma unroll
                    for (int q = 0; q < 4; ++q) unpack_word16<FMT, F16T>(w[q], o + q * PW);
#pragma unroll
                    for (int v = 0; v < PW; ++v)
                        *reinterpret_cast<uint4 *>(dst + v * 8) = make_uint4(o[4 * v], o[4 * v + 1], o[4 * v + 2], o[4 * v + 3]);
                }
            }
        } else {
            // element-wise, fully bounds-checked
            for (int e = t; e < BM * BK; e += 256) {
                const int row = e / BK, kk = e % BK;
                const uint32_t m = m0 + row, k = k0 + kk;
                As[row * LDK + kk] = (m < M && k < K) ? A[(size_t)m * K + k] : (uint16_t)0;
            }
            for (int e = t; e < BN * BK; e += 256) {
                const int row = e / BK, kk = e % BK;
                const uint32_t n = n0 + row, k = k0 + kk;
                uint16_t v = 0;
                if (n < N && k < K) {
                    const uint64_t idx = (uint64_t)n * K + k;
                    if constexpr (FMT == BF16 || FMT == F16) v = reinterpret_cast<const uint16_t *>(g.L.w)[idx];
                    else if constexpr (FMT == F32) v = f32_to_t16<F16T>(reinterpret_cast<const float *>(g.L.w)[idx]);
                    else v = (uint16_t)int_to_t16<F16T>(int_code<FMT>(g.L.w, idx));
                }
                Ws[row * LDK + kk] = v;
            }
        }
    };

    const uint32_t ktiles = (kend - kbeg + BK - 1) / BK;
    load_tiles(kbeg);
    for (uint32_t kt = 0; kt < ktiles; ++kt) {
        __syncthreads();                              // previous tile fully consumed
        store_tiles(kbeg + kt * BK);
        __syncthreads();
        if (kt + 1 < ktiles) load_tiles(kbeg + (kt + 1) * BK);

#pragma unroll
        for (int ks = 0; ks < BK; ks += 16) {
            const int koff = ks + 8 * (lane >> 5);
            uint4 fa[TM], fb[TN];
#pragma unroll
            for (int i = 0; i < TM; ++i)
                fa[i] = *reinterpret_cast<const uint4 *>(&As[(wm * TM * 32 + i * 32 + (lane & 31)) * LDK + koff]);
#pragma unroll
            for (int j = 0; j < TN; ++j)
                fb[j] = *reinterpret_cast<const uint4 *>(&Ws[(wn * TN * 32 + j * 32 + (lane & 31)) * LDK + koff]);
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    if constexpr (F16T) {
                        f16x8 a, b;
                        __builtin_memcpy(&a, &fa[i], 16);
                        __builtin_memcpy(&b, &fb[j], 16);
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, acc[i][j], 0, 0, 0);
                    } else {
                        bf16x8 a, b;
                        __builtin_memcpy(&a, &fa[i], 16);
                        __builtin_memcpy(&b, &fb[j], 16);
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc[i][j], 0, 0, 0);
                    }
                }
        }
    }

    if (g.ws) {                                        // partial sums of one activation matrix: a second launch adds them
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const uint32_t col = n0 + wn * TN * 32 + j * 32 + (lane & 31);
            if (col >= N) continue;
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const uint32_t row = m0 + wm * TM * 32 + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                    if (row < M) g.ws[((size_t)blockIdx.y * M + row) * N + col] = acc[i][j][r];
                }
        }
        return;
    }
    // epilogue: scale, bias, activation, store
    const float wscale = g.L.wscale;
    // 16-bit outputs in rows of whole 16-byte units: a wave turns each 32 x 32 block around in LDS (the tiles' memory,
    // free once every wave has read its last fragments) and stores 16 bytes per lane, two store instructions per
    // block instead of sixteen two-byte ones
    const bool rows16 = !g.out_f32 && N % 8u == 0 && (reinterpret_cast<uintptr_t>(g.C) & 15u) == 0;     // (uniform)
    if (rows16) __syncthreads();
    constexpr int SP = 40;                                   // row pitch of a wave's 32 x 32 staging block, elements
    uint16_t *const stage = (wave < 2 ? As : Ws) + (wave & 1) * (32 * SP);
    auto emit = [&](auto act_c) __attribute__((always_inline)) {
        constexpr int ACT = decltype(act_c)::value;
        if (rows16) {
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const uint32_t col = n0 + wn * TN * 32 + j * 32 + (lane & 31);
                const float bias = elem_value_rt(g.L.bias_fmt, g.L.bias, col < N ? col : N - 1) * g.L.bscale;
#pragma unroll
                for (int i = 0; i < TM; ++i) {
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const float pre = fmaf(acc[i][j][r], wscale, bias);
                        const float v = apply_act(pre, ACT);
                        stage[(8 * (r >> 2) + 4 * (lane >> 5) + (r & 3)) * SP + (lane & 31)] = f32_to_t16<F16T>(v);
                    }
                    // padded neurons (layer_sum): only hidden layers of this path have any
                    if (col + g.L.pad >= N) {
#pragma unroll
                        for (int r = 0; r < 16; ++r) stage[(8 * (r >> 2) + 4 * (lane >> 5) + (r & 3)) * SP + (lane & 31)] = 0;
                    }
                    __builtin_amdgcn_wave_barrier();
#pragma unroll
                    for (int p = 0; p < 2; ++p) {
                        const int rr = (lane >> 2) + 16 * p, ch = lane & 3;
                        const uint4 d = *reinterpret_cast<const uint4 *>(&stage[rr * SP + ch * 8]);
                        const uint32_t row = m0 + wm * TM * 32 + i * 32 + rr, c0 = n0 + wn * TN * 32 + j * 32 + ch * 8;
                        if (row < M && c0 < N) *reinterpret_cast<uint4 *>(reinterpret_cast<uint16_t *>(g.C) + (size_t)row * N + c0) = d;
                    }
                    __builtin_amdgcn_wave_barrier();
                }
            }
            return;
        }
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const uint32_t col = n0 + wn * TN * 32 + j * 32 + (lane & 31);
            if (col >= N) continue;
            const float bias = elem_value_rt(g.L.bias_fmt, g.L.bias, col) * g.L.bscale;
#pragma unroll
            for (int i = 0; i < TM; ++i) {
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const uint32_t row = m0 + wm * TM * 32 + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                    if (row >= M) continue;
                    const float pre = fmaf(acc[i][j][r], wscale, bias);
                    const float v = apply_act(pre, ACT);
                    const size_t o = (size_t)row * N + col;
                    if (g.out_f32) reinterpret_cast<float *>(g.C)[o] = v;
                    else reinterpret_cast<uint16_t *>(g.C)[o] = f32_to_t16<F16T>(v);
                }
            }
        }
    };
    with_act(g.L.act, emit);
}

// Small layers in one launch: a workgroup owns a 32 x 32 tile of the output, its eight waves split K in whole steps of
// 32, and their sums meet in LDS.  No operand staging: in step s lane (r, h) loads the sixteen consecutive elements
// k = 32 s + 16 h .. + 15 of row r of both operands straight into registers, as two pieces of eight (K % 8 == 0: a piece
// is inside its row or beyond it), and feeds a piece of each operand to one MFMA (a sum over k in any order).  For
// outputs of a few hundred tiles, where the streaming and the tiled kernels need a K split over the grid and a second
// launch to fill the chip.  XF32: the activations are still the caller's FP32 input, rounded here as sp_cvt16 (or, with
// split activations, sp_cvt16_split) would (g.A then points at floats).  HALVES == 2: split activations, two FP16
// matrices hi and lo = (a - hi) 2^11, M K elements apart; a second accumulator takes the lo products, a wave adds it,
// times 2^-11, to its hi sum, and 16-bit outputs leave as the two matrices of the next layer's input.
// Bound by the latency of its chain (launch, loads, sums through LDS, store): the biases are asked for with the first loads, not
// behind the barrier (four 256 x 256 layers at 64 / 512 samples FP16 17.4 / 17.9 -> 16.2 / 16.8 us).
template <int FMT, bool F16T, bool XF32, int HALVES = 1>
__global__ __launch_bounds__(512) void sp_gemm16_small(const GemmArgs g)
{
    static_assert(HALVES == 1 || F16T, "split activations are FP16");
    constexpr int NW = 8, U = 2;
    constexpr int bits = fmt_bits(FMT);
    constexpr int PB = bits;                           // bytes of a piece of eight weights
    __shared__ float part[NW][32 * 33];
    const uint32_t M = g.M, N = g.L.N, K = g.L.K;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6, q = lane & 31, h = lane >> 5;
    const uint32_t tiles_n = (N + 31u) / 32u;
    const uint32_t m0 = (blockIdx.x / tiles_n) * 32u, n0 = (blockIdx.x % tiles_n) * 32u;
    const uint32_t steps = (K + 31u) / 32u, per = (steps + NW - 1) / NW;
    const uint32_t s0 = wave * per, s1 = s0 + per < steps ? s0 + per : steps;
    const uint32_t am = m0 + q < M ? m0 + q : M - 1, wn = n0 + q < N ? n0 + q : N - 1;
    // (of this thread's two outputs, which are in one column)
    float bias = elem_value_rt(g.L.bias_fmt, g.L.bias, n0 + (t & 31) < N ? n0 + (t & 31) : N - 1) * g.L.bscale;
    const uint16_t *ap16 = g.A + (size_t)am * K + 16 * h;
    const float *ap32 = reinterpret_cast<const float *>(g.A) + (size_t)am * K + 16 * h;
    const uint8_t *wp = g.L.w + (size_t)wn * ((size_t)K * bits / 8u) + (size_t)(2 * h) * PB;

    struct Frag { uint4 a[2], al[HALVES == 2 ? 2 : 1], w[2]; };
    auto ld = [&](uint32_t s) -> Frag {
        Frag f;
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            const bool ok = 32u * s + 16u * h + 8u * p < K;
            if constexpr (XF32) {
                const float4 lo = ok ? *reinterpret_cast<const float4 *>(ap32 + 32u * s + 8 * p) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                const float4 hi = ok ? *reinterpret_cast<const float4 *>(ap32 + 32u * s + 8 * p + 4) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                if constexpr (HALVES == 2) {
                    const float v[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
                    uint16_t eh[8], el[8];
#pragma unroll
                    for (int e = 0; e < 8; ++e) split_f16(v[e], eh[e], el[e]);
                    f.a[p] = make_uint4((uint32_t)eh[0] | ((uint32_t)eh[1] << 16), (uint32_t)eh[2] | ((uint32_t)eh[3] << 16),
                                        (uint32_t)eh[4] | ((uint32_t)eh[5] << 16), (uint32_t)eh[6] | ((uint32_t)eh[7] << 16));
                    f.al[p] = make_uint4((uint32_t)el[0] | ((uint32_t)el[1] << 16), (uint32_t)el[2] | ((uint32_t)el[3] << 16),
                                         (uint32_t)el[4] | ((uint32_t)el[5] << 16), (uint32_t)el[6] | ((uint32_t)el[7] << 16));
                } else {
                    f.a[p].x = (uint32_t)f32_to_t16<F16T>(lo.x) | ((uint32_t)f32_to_t16<F16T>(lo.y) << 16);
                    f.a[p].y = (uint32_t)f32_to_t16<F16T>(lo.z) | ((uint32_t)f32_to_t16<F16T>(lo.w) << 16);
                    f.a[p].z = (uint32_t)f32_to_t16<F16T>(hi.x) | ((uint32_t)f32_to_t16<F16T>(hi.y) << 16);
                    f.a[p].w = (uint32_t)f32_to_t16<F16T>(hi.z) | ((uint32_t)f32_to_t16<F16T>(hi.w) << 16);
                }
            } else {
                f.a[p] = ok ? *reinterpret_cast<const uint4 *>(ap16 + 32u * s + 8 * p) : make_uint4(0, 0, 0, 0);
                if constexpr (HALVES == 2)
                    f.al[p] = ok ? *reinterpret_cast<const uint4 *>(ap16 + (size_t)M * K + 32u * s + 8 * p) : make_uint4(0, 0, 0, 0);
            }
            const uint8_t *src = wp + (size_t)s * (4 * PB) + p * PB;
            if constexpr (FMT == F16 || FMT == BF16) {
                f.w[p] = ok ? *reinterpret_cast<const uint4 *>(src) : make_uint4(0, 0, 0, 0);
            } else if constexpr (FMT == I8) {
                const uint2 c = ok ? *reinterpret_cast<const uint2 *>(src) : make_uint2(0, 0);
                f.w[p].x = c.x; f.w[p].y = c.y;
            } else if constexpr (FMT == I4) {
                f.w[p].x = ok ? *reinterpret_cast<const uint32_t *>(src) : 0u;
            } else {
                f.w[p].x = ok ? (uint32_t)*reinterpret_cast<const uint16_t *>(src) : 0u;
            }
        }
        return f;
    };
    f32x16 acc, accl;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = accl[r] = 0.0f;
    auto fma2 = [&](const Frag &f) {
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            uint4 wv = f.w[p];
            if constexpr (FMT == I8) {
                uint32_t o[4];
                unpack_word16<I8, F16T>(f.w[p].x, o);
                unpack_word16<I8, F16T>(f.w[p].y, o + 2);
                wv = make_uint4(o[0], o[1], o[2], o[3]);
            } else if constexpr (FMT == I4) {
                uint32_t o[4];
                unpack_word16<I4, F16T>(f.w[p].x, o);
                wv = make_uint4(o[0], o[1], o[2], o[3]);
            } else if constexpr (FMT == I2) {
                uint32_t o[8];                          // (the upper eight codes of the word are not there: zeros)
                unpack_word16<I2, F16T>(f.w[p].x, o);
                wv = make_uint4(o[0], o[1], o[2], o[3]);
            }
            if constexpr (F16T) {
                f16x8 a, b;
                __builtin_memcpy(&a, &f.a[p], 16);
                __builtin_memcpy(&b, &wv, 16);
                acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, acc, 0, 0, 0);
                if constexpr (HALVES == 2) {
                    __builtin_memcpy(&a, &f.al[p], 16);
                    accl = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, accl, 0, 0, 0);
                }
            } else {
                bf16x8 a, b;
                __builtin_memcpy(&a, &f.a[p], 16);
                __builtin_memcpy(&b, &wv, 16);
                acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc, 0, 0, 0);
            }
        }
    };
    uint32_t s = s0;
    for (; s + U <= s1; s += U) {
        Frag f[U];
#pragma unroll
        for (int u = 0; u < U; ++u) f[u] = ld(s + u);
#pragma unroll
        for (int u = 0; u < U; ++u) fma2(f[u]);
    }
    for (; s < s1; ++s) fma2(ld(s));
#pragma unroll
    for (int r = 0; r < 16; ++r)
        part[wave][(8 * (r >> 2) + 4 * h + (r & 3)) * 33 + q] = HALVES == 2 ? fmaf(accl[r], kLoScale, acc[r]) : acc[r];
    here(bias);
    __syncthreads();
    // the waves' sums in wave order, scale, bias, activation; 512 threads, two outputs each
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int e = t + 512 * i, row = e >> 5, col = e & 31;
        float v = 0.0f;
#pragma unroll
        for (int w = 0; w < NW; ++w) v += part[w][row * 33 + col];
        if (m0 + row >= M || n0 + col >= N) continue;
        v = apply_act(layer_sum(g.L, v, bias, n0 + col), g.L.act);
        const size_t o = (size_t)(m0 + row) * N + n0 + col;
        if (g.out_f32) reinterpret_cast<float *>(g.C)[o] = v;
        else if constexpr (HALVES == 2) {
            uint16_t eh, el;
            split_f16(v, eh, el);
            reinterpret_cast<uint16_t *>(g.C)[o] = eh;
            reinterpret_cast<uint16_t *>(g.C)[(size_t)M * N + o] = el;
        } else reinterpret_cast<uint16_t *>(g.C)[o] = f32_to_t16<F16T>(v);
    }
}

template <int OFF>
__device__ __forceinline__ void ds_read128(u32x4 &dst, uint32_t addr);

// 16 bytes per lane from global memory straight into LDS (wave-contiguous 1 KiB at lds_addr):
// scalar base + 32-bit lane offset, so issuing it costs no vector-ALU instruction.  The compiler
// does not track these loads: the caller waits with s_waitcnt vmcnt before the data is read.
__device__ __forceinline__ void lds_dma16(uint32_t lds_addr, uint32_t voff, const void *sbase)
{
    // Both are uniform by construction; saying so keeps them in scalar registers where the compiler's own analysis
    // gives up (it folds the intrinsic away where it does not).
    lds_addr = (uint32_t)__builtin_amdgcn_readfirstlane((int)lds_addr);
    const uint64_t b = reinterpret_cast<uint64_t>(sbase);
    sbase = reinterpret_cast<const void *>(((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(b >> 32)) << 32) |
                                           (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)b));
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_addr), "v"(voff), "s"(sbase) : "memory");
}

template <int OFF>
__device__ __forceinline__ void ds_read128(u32x4 &dst, uint32_t addr)
{
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(dst) : "v"(addr), "n"(OFF));
}

// 16 bytes per lane from scalar base + 32-bit lane offset + immediate.  Inline assembly: the compiler's
// wait-count bookkeeping does not see the load, the caller waits with s_waitcnt vmcnt before using dst.
template <int OFF>
__device__ __forceinline__ void load16_async(u32x4 &dst, uint32_t voff, const void *sbase)
{
    asm volatile("global_load_dwordx4 %0, %1, %2 offset:%3" : "=v"(dst) : "v"(voff), "s"(sbase), "n"(OFF) : "memory");
}

// reads CNT fragments 2 KiB apart (16 tile rows of 128 bytes) starting at addr + BASE
template <int BASE, int CNT, int I = 0>
__device__ __forceinline__ void frag_reads(u32x4 *dst, uint32_t addr)
{
    if constexpr (I < CNT) {
        ds_read128<BASE + I * 2048>(dst[I], addr);
        frag_reads<BASE, CNT, I + 1>(dst, addr);
    }
}

// ---------------------------------------------------------------------------
// Large-tile variant of the 16-bit MFMA GEMM (rows 16-byte aligned): 256 x 256 tiles (RM = 8) or 128 x 256 (RM = 4), four
// waves of RM x 8 tiles of 16 x 16, BK = 64.
//
// On this data the part is at its power limit, not at an issue limit: matrix instructions alone, operands in registers, run
// at 1.98 PFLOP/s as v_mfma_f32_16x16x32 and at 1.73 as 32x32x16 (half the accumulator traffic per product), and what LDS
// reads and loads add to the time of 8192 x 8192 x 8192 is nearly additive (0.58 ms without either, 0.18 and 0.14 for
// eight waves of 128 x 64).  So: the small instruction; as much of the tile per wave as the registers hold, which is
// 128 x 128 with one wave per SIMD (128 instead of 192 KiB of fragment reads per K tile); neighbouring products share an
// operand.  8192 x 8192 x 8192 FP16 0.870 -> 0.771 ms (1.43 PFLOP/s; 32 x 32 x 16 in eight waves before, whose 16 x 16 x 32
// form took 0.82), 4096 x 8192 x 8192 INT8 0.465 -> 0.408, INT4 0.449 -> 0.377, INT2 0.395 -> 0.356, 2000 x 4096 x 12288 on
// RM = 4 0.198 -> 0.167 ms.  Sums of a few hundred gain little (8192 x 8192 x 512 98 -> 95 us): a tile's prologue takes 2.4 us,
// its epilogue 8, in which all compute units write at once (4 TB/s).  FP32 outputs of sums of 256, written 4 waves instead
// of 8 at a time, lose 3-5 % (4096 x 4096 x 256 24.6 -> 25.3 us FP16, 25.5 -> 26.8 INT8; x 1024 48.5 -> 45.4).
//
// The accumulators are accumulation registers by number (mfma_acc, acc_read): left to the compiler, 256 of them next to the
// fragments are spilled.  Nothing else here lives in those registers (the first statement claims all of them, and the
// vector registers suffice for the rest; the Makefile refuses a build with a spill in this kernel, which could go there).
//
// One wave per SIMD has nobody to hide behind, so the loop is straight-line code with everything asked for ahead:
//   * A K tile is RM quads of sixteen products (four row tiles x four column tiles).  Consecutive quads share one of their
//     two sets of four fragments, the other was requested a quad earlier.
//   * 16-bit operands (activations always, BF16/FP16 weights) go from global memory straight into LDS
//     (global_load_lds_dwordx4: each wave fills 1 KiB = 8 tile rows per instruction), one instruction behind every fourth
//     product; which global chunk a lane fetches carries the swizzle.  Integer weights come as packed codes, three
//     tiles ahead, and are unpacked through registers a step per product (w_step).
//   * Two LDS stages (RM = 4: three).  The barrier comes when the last fragments of a tile are in registers, two quads (one)
//     before its products end: the next tile's first fragments and the loads that overwrite this tile's stage go
//     out behind those products.
//   * LDS rows hold 64 elements = eight 16-byte chunks, unpadded; chunk c of row r sits at position c ^ ((r >> 1) & 7).  A
//     128-bit fragment read is served 16 lanes (16 consecutive rows, 256 bytes = all 64 banks) per cycle: rows of equal
//     parity share a 128-byte half, and r >> 1 gives those eight rows eight different chunk positions.
// A K that is not a multiple of 64 leaves a partial K tile, which is processed first: its lanes past the end of a row fetch
// the row's element k0 instead (always inside the array) and overwrite what they fetched with zeros once it has landed.
// ---------------------------------------------------------------------------
// accumulation registers ACC .. ACC + 3 += a . b (16 rows of a, 16 columns of b, 32 k)
template <bool F16T, int ACC>
__device__ __forceinline__ void mfma_acc(const u32x4 &a, const u32x4 &b)
{
    if constexpr (F16T) asm volatile("v_mfma_f32_16x16x32_f16 a[%2:%3], %0, %1, a[%2:%3]" ::"v"(a), "v"(b), "n"(ACC), "n"(ACC + 3));
    else asm volatile("v_mfma_f32_16x16x32_bf16 a[%2:%3], %0, %1, a[%2:%3]" ::"v"(a), "v"(b), "n"(ACC), "n"(ACC + 3));
}

template <int R>
__device__ __forceinline__ float acc_read()
{
    float v;
    asm volatile("v_accvgpr_read_b32 %0, a[%1]" : "=v"(v) : "n"(R));
    return v;
}

template <int R>
__device__ __forceinline__ void acc_zero()
{
    asm volatile("v_accvgpr_write_b32 a[%0], 0" ::"n"(R));
}

#define SP_ACC10(d) "a" #d "0", "a" #d "1", "a" #d "2", "a" #d "3", "a" #d "4", "a" #d "5", "a" #d "6", "a" #d "7", "a" #d "8", "a" #d "9"
#define SP_ACC128                                                                                                      \
    "a0", "a1", "a2", "a3", "a4", "a5", "a6", "a7", "a8", "a9", SP_ACC10(1), SP_ACC10(2), SP_ACC10(3), SP_ACC10(4),    \
        SP_ACC10(5), SP_ACC10(6), SP_ACC10(7), SP_ACC10(8), SP_ACC10(9), SP_ACC10(10), SP_ACC10(11), "a120", "a121",   \
        "a122", "a123", "a124", "a125", "a126", "a127"
#define SP_ACC256                                                                                                      \
    SP_ACC128, "a128", "a129", SP_ACC10(13), SP_ACC10(14), SP_ACC10(15), SP_ACC10(16), SP_ACC10(17), SP_ACC10(18),     \
        SP_ACC10(19), SP_ACC10(20), SP_ACC10(21), SP_ACC10(22), SP_ACC10(23), SP_ACC10(24), "a250", "a251", "a252",    \
        "a253", "a254", "a255"

// two FP32 values below 65520 in magnitude (they round to at most 65504), as f32_to_f16_sat converts them
__device__ __forceinline__ uint32_t pack_f16_small(float a, float b)
{
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    const h2 h = {(_Float16)a, (_Float16)b};
    uint32_t r;
    __builtin_memcpy(&r, &h, 4);
    return r;
}

// LDS stages (three where they fit), bytes of packed codes per K tile (integer formats), bytes of LDS
template <int FMT, int RM>
struct BigTile {
    static constexpr int NSTAGE = RM == 8 || FMT == I8 ? 2 : 3;
    static constexpr int W_AT = 32 * RM * 128, STAGE = W_AT + 256 * 128;      // the weights' part of a stage, a stage
    static constexpr int CODES = fmt_bits(FMT) == 16 ? 0 : 256 * 64 * fmt_bits(FMT) / 8;
    static constexpr int TURN = 64 * (128 * 4 + 16);        // of a wave in the epilogue: four row tiles as FP32
    static constexpr int LOOP = NSTAGE * STAGE + 2 * CODES, END = 4 * TURN + 256 * 4, LDS = LOOP > END ? LOOP : END;
};

template <int FMT, bool F16T, int RM>
__global__ __launch_bounds__(256, 1) void sp_gemm16_big(const GemmArgs g)
{
    static_assert(RM == 8 || RM == 4, "");
    constexpr int BM = 32 * RM, BN = 256, BK = 64;
    using B = BigTile<FMT, RM>;
    constexpr int NSTAGE = B::NSTAGE, W_AT = B::W_AT, STAGE = B::STAGE, CODES = B::CODES;
    constexpr int bits = fmt_bits(FMT);
    constexpr bool W_DIRECT = (FMT == BF16 || FMT == F16);
    constexpr int A_DMA = BM / 32, DMA = A_DMA + (W_DIRECT ? BN / 32 : 0);     // load instructions per wave and tile
    constexpr int EPL = 128 / bits;                     // weight elements per 16-byte global load
    constexpr int CPL = EPL / 8;                        // LDS chunks produced per global load
    constexpr int W_LOADS = W_DIRECT ? 1 : BN * BK / EPL / 256;
    constexpr int PW = 16 / bits;                       // packed pairs per 32-bit word of codes (integer formats)

    extern __shared__ __attribute__((aligned(16))) uint16_t smem[];
    if constexpr (RM == 8) asm volatile("" ::: SP_ACC256);
    else asm volatile("" ::: SP_ACC128);

    const uint32_t M = g.M, N = g.L.N, K = g.L.K;
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int wm = wave >> 1, wn = wave & 1;

    // Tile order: each XCD (workgroup id mod 8) gets a contiguous run of tiles; inside the run, 8 row tiles x 4
    // column tiles are consecutive so that the 32 workgroups an XCD runs at once share A rows and W rows in its L2.
    const uint32_t tiles_n = (N + BN - 1) / BN, tiles_m = (M + BM - 1) / BM;
    uint32_t m0, n0;
    {
        const uint32_t ntiles = tiles_m * tiles_n, per = ntiles / 8u;
        uint32_t bid = blockIdx.x;
        if (bid < per * 8u) bid = (bid & 7u) * per + (bid >> 3);
        constexpr uint32_t GM = 8;
        const uint32_t group = bid / (GM * tiles_n);
        const uint32_t first = group * GM;
        const uint32_t rows = tiles_m - first < GM ? tiles_m - first : GM;
        const uint32_t in = bid - group * GM * tiles_n;
        m0 = (first + in % rows) * BM;
        n0 = (in / rows) * BN;
    }

    // grid y splits K for problems with too few tiles to fill the chip
    const uint32_t kbeg = g.kper ? (blockIdx.y % g.ksplits) * g.kper : 0u;
    const uint32_t kend = g.kper && kbeg + g.kper < K ? kbeg + g.kper : K;
    const uint32_t ktiles = (kend - kbeg + BK - 1) / BK;
    const uint32_t tail = (kend - kbeg) % BK;              // only the last K split can have one
    // tile 0 is the partial tile if there is one; tile s >= 1 then starts at kbeg + (s - 1) * BK
    const uint32_t kshift = tail ? (uint32_t)BK : 0u;
    auto k_of = [&](uint32_t s) { return kbeg + s * BK - kshift; };

    // LDS-DMA sources: a uniform base (advanced per K tile on the scalar unit) plus a fixed 32-bit byte offset per lane and
    // load.  A lane fetches the same eight of a tile row's 64 elements in every load: the rows of two of its loads are a
    // multiple of 32 apart.
    const uint32_t kchunk = (uint32_t)((lane & 7) ^ (((wave * 8 + (lane >> 3)) >> 1) & 7)) << 3;
    uint32_t a_voff[A_DMA], w_voff[W_DIRECT ? BN / 32 : W_LOADS];
#pragma unroll
    for (int i = 0; i < A_DMA; ++i) {
        const uint32_t m = m0 + (i * 4 + wave) * 8 + (lane >> 3);
        a_voff[i] = (uint32_t)(((size_t)(m < M ? m : M - 1) * K + kchunk) * 2u);
    }
    if constexpr (W_DIRECT) {
#pragma unroll
        for (int i = 0; i < BN / 32; ++i) {
            const uint32_t n = n0 + (i * 4 + wave) * 8 + (lane >> 3);
            w_voff[i] = (uint32_t)(((size_t)(n < N ? n : N - 1) * K + kchunk) * 2u);
        }
    } else {
#pragma unroll
        for (int i = 0; i < W_LOADS; ++i) {
            constexpr int LPR = BK / EPL;                   // loads per tile row
            const int c = t + 256 * i;
            const uint32_t n = n0 + c / LPR;
            w_voff[i] = (uint32_t)((size_t)(n < N ? n : N - 1) * ((size_t)K * bits / 8u) + (size_t)(c % LPR) * 16u);
        }
    }
    const char *const a_base = reinterpret_cast<const char *>(g.A + (size_t)(blockIdx.y / g.ksplits) * M * K);
    const char *const w_base = reinterpret_cast<const char *>(g.L.w);
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint16_t *)smem;
    // the idx-th load instruction of this wave's share of the tile at k0 (A first, then W); idx is a constant once unrolled
    auto dma_at = [&](uint32_t stage, const char *a_at, const char *w_at, uint32_t back, int idx) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < A_DMA; ++i)
            if (i == idx) lds_dma16(stage + (uint32_t)(i * 4096), a_voff[i] - back, a_at);
        if constexpr (W_DIRECT) {
#pragma unroll
            for (int i = 0; i < BN / 32; ++i)
                if (A_DMA + i == idx) lds_dma16(stage + (uint32_t)(W_AT + i * 4096), w_voff[i] - back, w_at);
        }
    };
    const uint32_t lds_w = lds0 + (uint32_t)wave * 1024u;   // where this wave's share of a stage begins
    auto dma = [&](uint32_t stage, uint32_t k0, uint32_t back, int idx) __attribute__((always_inline)) {
        dma_at(lds_w + stage, a_base + (size_t)k0 * 2u, w_base + (W_DIRECT ? (size_t)k0 * 2u : 0u), back, idx);
    };
    // Integer weights: the packed codes of a tile go to LDS too, a thread's 16-byte pieces to a place of its own, which only
    // that thread reads.  (Loaded into registers two tiles ahead they would be copied while still on their way: the compiler
    // does not see these loads.)
    const uint32_t codes0 = (uint32_t)(NSTAGE * STAGE);
    auto dma_codes = [&](uint32_t buf, uint32_t k0, bool clip) __attribute__((always_inline)) {
        if constexpr (!W_DIRECT) {
#pragma unroll
            for (int i = 0; i < W_LOADS; ++i) {
                constexpr int LPR = BK / EPL;
                const uint32_t piece = (uint32_t)((t + 256 * i) % LPR);
                const uint32_t back = clip && k0 + piece * EPL >= K ? piece * 16u : 0u;      // past its row: the row's start of the tile
                lds_dma16(lds0 + codes0 + buf + (uint32_t)(i * 4 + wave) * 1024u, w_voff[i] - back, w_base + (size_t)k0 * bits / 8u);
            }
        }
    };
    u32x4 rw[W_LOADS];                                      // this thread's codes of the tile that is unpacked
    auto read_codes = [&](uint32_t buf) __attribute__((always_inline)) {
        if constexpr (!W_DIRECT) {
#pragma unroll
            for (int i = 0; i < W_LOADS; ++i) ds_read128<0>(rw[i], lds0 + codes0 + buf + (uint32_t)(t + 256 * i) * 16u);
        }
    };
    auto pin_codes = [&]() __attribute__((always_inline)) {
        if constexpr (!W_DIRECT) {
#pragma unroll
            for (int i = 0; i < W_LOADS; ++i) asm volatile("" : "+v"(rw[i]));
        }
    };
    constexpr int CREADS = W_DIRECT ? 0 : W_LOADS;
    // Step s of 64 that unpack rw into the stage at `stage`: eight chunks of eight codes, eight steps each (INT2: two chunks
    // in sixteen), at most three vector instructions a step, so that a step fits behind a product.
    uint32_t up[8];
    auto w_step = [&](uint32_t stage, int s) __attribute__((always_inline)) {
        if constexpr (!W_DIRECT) {
            constexpr uint32_t LO = 0x05040100u, HI = 0x07060302u;
            constexpr int LPR = BK / EPL;
            const int c = s >> 3, p = s & 7;                 // chunk of this thread, step of it
            const int i = c / CPL, v = c % CPL;              // its load, its chunk of that load
            auto put = [&](int chunk_of_load, uint32_t o0, uint32_t o1, uint32_t o2, uint32_t o3) __attribute__((always_inline)) {
                const int cc = t + 256 * i, row = cc / LPR, chunk = (cc % LPR) * CPL + chunk_of_load;
                char *const at = reinterpret_cast<char *>(smem) + stage + W_AT + row * 128 + ((chunk ^ ((row >> 1) & 7)) << 4);
                *reinterpret_cast<uint4 *>(at) = make_uint4(o0, o1, o2, o3);
            };
            if constexpr (!F16T) {
                (void)LO; (void)HI;
                if (p == 0) {
#pragma unroll
                    for (int q = 0; q < 4 / PW; ++q) unpack_word16<FMT, F16T>(rw[i][v * (4 / PW) + q], up + q * PW);
                    put(v, up[0], up[1], up[2], up[3]);
                }
            } else if constexpr (FMT == I8) {
                if (p < 4) {
                    const uint32_t w = rw[i][2 * v + (p >> 1)];
                    up[p] = h2_sub((((p & 1) ? w >> 8 : w) & 0x00FF00FFu) ^ 0x64806480u, 0x64806480u);
                } else if (p == 4) {
                    up[4] = __builtin_amdgcn_perm(up[1], up[0], LO);
                    up[5] = __builtin_amdgcn_perm(up[1], up[0], HI);
                } else if (p == 5) {
                    up[6] = __builtin_amdgcn_perm(up[3], up[2], LO);
                    up[7] = __builtin_amdgcn_perm(up[3], up[2], HI);
                } else if (p == 6) {
                    put(v, up[4], up[5], up[6], up[7]);
                }
            } else if constexpr (FMT == I4) {
                const uint32_t w = rw[i][v];
                if (p == 0) up[0] = h2_sub((w & 0x000F000Fu) ^ 0x64086408u, 0x64086408u);
                else if (p == 1) up[1] = h2_sub((w & 0x00F000F0u) ^ 0x54805480u, 0x54805480u);
                else if (p == 2) up[2] = h2_sub(((w >> 8) & 0x000F000Fu) ^ 0x64086408u, 0x64086408u);
                else if (p == 3) up[3] = h2_sub(((w >> 8) & 0x00F000F0u) ^ 0x54805480u, 0x54805480u);
                else if (p == 4) {
                    up[4] = __builtin_amdgcn_perm(up[1], up[0], LO);
                    up[5] = __builtin_amdgcn_perm(up[3], up[2], LO);
                } else if (p == 5) {
                    up[6] = __builtin_amdgcn_perm(up[1], up[0], HI);
                    up[7] = __builtin_amdgcn_perm(up[3], up[2], HI);
                } else if (p == 6) {
                    put(v, up[4], up[5], up[6], up[7]);
                }
            } else if constexpr (FMT == I2) {
                const uint32_t w = rw[i][v >> 1], y = w >> 10;
                const int p2 = s & 15;
                if (p2 == 0) up[0] = h2_sub((w & 0x00030003u) ^ 0x64026402u, 0x64026402u);
                else if (p2 == 1) up[1] = h2_sub((w & 0x000C000Cu) ^ 0x5C085C08u, 0x5C085C08u);
                else if (p2 == 2) up[2] = h2_sub((w & 0x00300030u) ^ 0x54205420u, 0x54205420u);
                else if (p2 == 3) up[3] = h2_sub((w & 0x00C000C0u) ^ 0x4C804C80u, 0x4C804C80u);
                else if (p2 == 4) up[4] = h2_sub((w & 0x03000300u) ^ 0x46004600u, 0x46004600u);
                else if (p2 == 5) up[5] = h2_sub((y & 0x00030003u) ^ 0x64026402u, 0x64026402u);
                else if (p2 == 6) up[6] = h2_sub((y & 0x000C000Cu) ^ 0x5C085C08u, 0x5C085C08u);
                else if (p2 == 7) up[7] = h2_sub((y & 0x00300030u) ^ 0x54205420u, 0x54205420u);
                else if (p2 == 9)
                    put(v & ~1, __builtin_amdgcn_perm(up[1], up[0], LO), __builtin_amdgcn_perm(up[3], up[2], LO),
                        __builtin_amdgcn_perm(up[5], up[4], LO), __builtin_amdgcn_perm(up[7], up[6], LO));
                else if (p2 == 11)
                    put(v | 1, __builtin_amdgcn_perm(up[1], up[0], HI), __builtin_amdgcn_perm(up[3], up[2], HI),
                        __builtin_amdgcn_perm(up[5], up[4], HI), __builtin_amdgcn_perm(up[7], up[6], HI));
            }
        }
    };

    // ---- fragments -------------------------------------------------------------
    // Explicit ds_read_b128 with manual lgkmcnt waits: the compiler would otherwise drain every pending LDS-DMA load before
    // the first LDS read of an iteration and serialise load and compute.
    const int q4 = lane >> 4, l15 = lane & 15;
    uint32_t va[2], vw[2];                                  // of k-step 0 and 1 in the current stage
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
        const uint32_t xo = (uint32_t)(((4 * ks + q4) ^ ((lane >> 1) & 7)) << 4);
        va[ks] = lds0 + (uint32_t)((wm * (BM / 2) + l15) * 128) + xo;
        vw[ks] = lds0 + W_AT + (uint32_t)((wn * 128 + l15) * 128) + xo;
    }
    u32x4 alo[4], ahi[4], blo[4], bhi[4];
    auto pin = [&](u32x4 (&d)[4]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; ++i) asm volatile("" : "+v"(d[i]));
    };
    // sixteen products: row tiles AI .. AI + 3, column tiles BJ .. BJ + 3, hook(s) behind product s.  The weights are the
    // first operand, so that a lane ends with four neighbouring outputs of one sample.
    auto quad = [&](const u32x4 (&a)[4], const u32x4 (&b)[4], auto ai_c, auto bj_c, auto &&hook) __attribute__((always_inline)) {
        constexpr int AI = decltype(ai_c)::value, BJ = decltype(bj_c)::value;
        static_for<16>([&](auto s_c) __attribute__((always_inline)) {
            constexpr int s = decltype(s_c)::value, i = s >> 2, j = (i & 1) ? 3 - (s & 3) : (s & 3);
            mfma_acc<F16T, ((AI + i) * 8 + BJ + j) * 4>(b[j], a[i]);
            hook(s);
        });
    };
    using T0 = std::integral_constant<int, 0>;
    using T4 = std::integral_constant<int, 4>;

    // ---- prologue ----------------------------------------------------------------
    const uint32_t bcol = n0 + (uint32_t)t;
    const float my_bias = bcol < N && !g.ws ? elem_value_rt(g.L.bias_fmt, g.L.bias, bcol) * g.L.bscale : 0.0f;
    const uint32_t k0 = tail ? kend - tail : kbeg;
    const bool past = k0 + kchunk >= K && tail;             // this lane's pieces of the partial tile lie past their rows
#pragma unroll
    for (int idx = 0; idx < DMA; ++idx) dma(0, k0, past ? kchunk * 2u : 0u, idx);
    dma_codes(0, k0, true);
    if (1 < ktiles) dma_codes(CODES, k_of(1), false);
    // the loads that the tiles before the first would have issued: of tile 1, and with three stages the first ones of tile 2
    constexpr int AFTER = RM == 8 ? 2 : 1;                  // quads of a tile behind its barrier
    constexpr int FIRST = AFTER * 4 < DMA ? AFTER * 4 : DMA;  // loads that go out there, four a quad
    auto early_loads = [&]() __attribute__((always_inline)) {
        if (1 < ktiles) {
#pragma unroll
            for (int idx = 0; idx < (NSTAGE == 2 ? FIRST : DMA); ++idx) dma(STAGE, k_of(1), 0u, idx);
        }
        if constexpr (NSTAGE == 3) {
            if (2 < ktiles) {
#pragma unroll
                for (int idx = 0; idx < FIRST; ++idx) dma(2 * STAGE, k_of(2), 0u, idx);
            }
        }
    };
    // (three stages of packed codes: only behind the codes of tile 2, which the first barrier waits for)
    constexpr bool EARLY = W_DIRECT || NSTAGE == 2;
    if constexpr (EARLY) early_loads();
    static_for<RM * 32>([&](auto r) __attribute__((always_inline)) { acc_zero<decltype(r)::value>(); });
    if (EARLY && ktiles >= NSTAGE) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NSTAGE == 2 ? FIRST : DMA + FIRST) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (past) {
#pragma unroll
        for (int i = 0; i < A_DMA; ++i)
            *reinterpret_cast<uint4 *>(reinterpret_cast<char *>(smem) + (i * 4 + wave) * 1024 + lane * 16) = make_uint4(0u, 0u, 0u, 0u);
        if constexpr (W_DIRECT) {
#pragma unroll
            for (int i = 0; i < BN / 32; ++i)
                *reinterpret_cast<uint4 *>(reinterpret_cast<char *>(smem) + W_AT + (i * 4 + wave) * 1024 + lane * 16) = make_uint4(0u, 0u, 0u, 0u);
        }
    }
    if constexpr (!W_DIRECT) {
        constexpr int LPR = BK / EPL;
        read_codes(0);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        pin_codes();
        if (2 < ktiles) dma_codes(0, k_of(2), false);
#pragma unroll
        for (int i = 0; i < W_LOADS; ++i)
            if (k0 + ((t + 256 * i) % LPR) * EPL >= K) rw[i] = u32x4{0u, 0u, 0u, 0u};        // (code 0 decodes to 0)
        static_for<64>([&](auto s) __attribute__((always_inline)) { w_step(0, decltype(s)::value); });
    }
    if constexpr (!EARLY) early_loads();
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");

    // ---- main loop -----------------------------------------------------------------
    // Stages as byte offsets: cur (this tile), nxt (the next one), fill (being loaded: NSTAGE - 1 tiles on).
    uint32_t cur = 0, nxt = STAGE, fill = (NSTAGE - 1) * STAGE;
    uint32_t code_buf = CODES;                              // the codes of the next tile
    frag_reads<0, 4>(alo, va[0]);
    frag_reads<0, 4>(blo, vw[0]);
    // the tile whose loads are going out, kt + NSTAGE - 1 before a tile's barrier and kt + NSTAGE behind it
    uint32_t to = lds_w + fill;
    const char *a_at = a_base + (size_t)k_of(NSTAGE - 1) * 2u, *w_at = w_base + (W_DIRECT ? (size_t)k_of(NSTAGE - 1) * 2u : 0u);
    // One tile.  KIND 2: there is a tile kt + NSTAGE, whose loads begin behind the barrier, where this tile's stage is free, and
    // are finished in the next iteration's first quads; 1: the last loads are finished; 0: none are left.  (A branch around
    // each load instead: 0.85 against 0.81 ms on 8192 cubed.)
    auto tile = [&](auto kind_c, uint32_t kt) __attribute__((always_inline)) {
        constexpr int KIND = decltype(kind_c)::value;
        auto finish_loads = [&](int first) __attribute__((always_inline)) {
            return [&, first](int s) __attribute__((always_inline)) {
                if (KIND >= 1 && s % 4 == 3 && first + s / 4 < DMA) dma_at(to, a_at, w_at, 0u, first + s / 4);
            };
        };
        auto begin_loads = [&](int first) __attribute__((always_inline)) {
            return [&, first](int s) __attribute__((always_inline)) {
                if (KIND == 2 && s % 4 == 3 && first + s / 4 < FIRST) dma_at(to, a_at, w_at, 0u, first + s / 4);
            };
        };
        auto unpack = [&](int first) __attribute__((always_inline)) {
            return [&, first](int s) __attribute__((always_inline)) {
                if constexpr (!W_DIRECT && (KIND >= 1 || NSTAGE == 3)) {       // (else there is no next tile)
                    w_step(nxt, first + s);
                    __builtin_amdgcn_sched_barrier(0);
                }
            };
        };
        auto swap_stage = [&]() __attribute__((always_inline)) {
            // this wave's share of the next tile has landed, its fragments of this one are in registers ...
            if constexpr (NSTAGE == 3 && KIND >= 1) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(DMA) : "memory");
            else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();                   // ... and everybody's
            asm volatile("" ::: "memory");
            if constexpr (KIND == 2) {
                if constexpr (!W_DIRECT) dma_codes(code_buf, NSTAGE == 3 || kt + 3 < ktiles ? k_of(kt + 3) : 0u, false);
                to = lds_w + cur;
                a_at = a_base + (size_t)k_of(kt + NSTAGE) * 2u;
                if constexpr (W_DIRECT) w_at = w_base + (size_t)k_of(kt + NSTAGE) * 2u;
            }
            code_buf ^= (uint32_t)CODES;
            const uint32_t step = nxt - cur;                // (wraps around)
            va[0] += step; va[1] += step; vw[0] += step; vw[1] += step;
        };
        if constexpr (RM == 8) {
            frag_reads<8192, 4>(bhi, vw[0]);
            asm volatile("s_waitcnt lgkmcnt(4)");
            pin(alo); pin(blo);
            quad(alo, blo, T0{}, T0{}, finish_loads(FIRST));
            frag_reads<8192, 4>(ahi, va[0]);
            read_codes(code_buf);
            asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(4 + CREADS));
            pin(bhi);
            quad(alo, bhi, T0{}, T4{}, finish_loads(FIRST + 4));
            frag_reads<0, 4>(alo, va[1]);
            asm volatile("s_waitcnt lgkmcnt(4)");
            pin(ahi);
            pin_codes();
            quad(ahi, bhi, T4{}, T4{}, unpack(0));
            frag_reads<8192, 4>(bhi, vw[1]);
            asm volatile("s_waitcnt lgkmcnt(4)");
            pin(alo);
            quad(ahi, blo, T4{}, T0{}, unpack(16));
            frag_reads<0, 4>(blo, vw[1]);
            asm volatile("s_waitcnt lgkmcnt(4)");
            pin(bhi);
            quad(alo, bhi, T0{}, T4{}, unpack(32));
            frag_reads<8192, 4>(ahi, va[1]);
            asm volatile("s_waitcnt lgkmcnt(4)");
            pin(blo);
            quad(alo, blo, T0{}, T0{}, unpack(48));
            swap_stage();
            pin(ahi);
            frag_reads<0, 4>(alo, va[0]);
            quad(ahi, blo, T4{}, T0{}, begin_loads(0));
            frag_reads<0, 4>(blo, vw[0]);
            quad(ahi, bhi, T4{}, T4{}, begin_loads(4));
        } else {
            // (alo: k-step 0, ahi: k-step 1)
            frag_reads<8192, 4>(bhi, vw[0]);
            read_codes(code_buf);
            asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(4 + CREADS));
            pin(alo); pin(blo);
            quad(alo, blo, T0{}, T0{}, finish_loads(FIRST));
            frag_reads<0, 4>(ahi, va[1]);
            frag_reads<0, 4>(blo, vw[1]);
            asm volatile("s_waitcnt lgkmcnt(8)");
            pin(bhi);
            pin_codes();
            quad(alo, bhi, T0{}, T4{}, [&](int s) __attribute__((always_inline)) {
                finish_loads(FIRST + 4)(s);
                unpack(0)(2 * s);
                unpack(1)(2 * s);
            });
            frag_reads<8192, 4>(bhi, vw[1]);
            asm volatile("s_waitcnt lgkmcnt(4)");
            pin(ahi); pin(blo);
            quad(ahi, blo, T0{}, T0{}, [&](int s) __attribute__((always_inline)) {
                unpack(32)(2 * s);
                unpack(33)(2 * s);
            });
            swap_stage();
            pin(bhi);
            frag_reads<0, 4>(alo, va[0]);
            frag_reads<0, 4>(blo, vw[0]);
            quad(ahi, bhi, T0{}, T4{}, begin_loads(0));
        }
        if constexpr (NSTAGE == 2) {
            const uint32_t was = cur;
            cur = nxt;
            nxt = fill = was;
        } else {
            const uint32_t was = cur;
            cur = nxt;
            nxt = fill;
            fill = was;
        }
    };
    uint32_t kt = 0;
    for (; kt + NSTAGE < ktiles; ++kt) tile(std::integral_constant<int, 2>{}, kt);
    if (kt + NSTAGE - 1 < ktiles) tile(std::integral_constant<int, 1>{}, kt++);
    for (; kt < ktiles; ++kt) tile(std::integral_constant<int, 0>{}, kt);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_nop 15\n\ts_nop 15" ::: "memory");      // the last fragments asked for; the last products
    pin(alo); pin(blo);
    __syncthreads();

    // ---- epilogue ------------------------------------------------------------------
    // Lane (l15, q4) holds outputs 4 q4 .. 4 q4 + 3 of each column tile for sample l15 of each row tile.
    const uint32_t mrow = m0 + wm * (BM / 2), ncol = n0 + wn * 128;
    float *const bias_lds = reinterpret_cast<float *>(reinterpret_cast<char *>(smem) + 4 * B::TURN);
    bias_lds[t] = my_bias;
    __syncthreads();
    float4 bias[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) bias[j] = *reinterpret_cast<const float4 *>(bias_lds + wn * 128 + j * 16 + 4 * q4);
    const float wscale = g.L.wscale;
    const uint32_t pad = g.L.pad;
    // A wave turns the 16 x 128 block of each row tile around in LDS (the stages are free after the loop; every wave has a
    // region of its own, so no barrier is needed) and writes whole rows of the block, 16 bytes per lane (rows that are not
    // whole 16-byte units: element by element).  The partial sums of a K split go the same way into the workspace, unscaled,
    // as FP32.
    const bool f32_out = g.ws || g.out_f32;
    char *const out = g.ws ? reinterpret_cast<char *>(g.ws + (size_t)blockIdx.y * M * N) : reinterpret_cast<char *>(g.C);
    const bool rows16 = ((size_t)N * (f32_out ? 4u : 2u)) % 16u == 0 && (reinterpret_cast<uintptr_t>(out) & 15u) == 0;
    // Long K: the outputs bypass the caches' usual retention (they would displace the A and W panels the other
    // tiles of the die are re-reading: 8192 cubed 0.908 against 0.934 ms); short K: the next layer reads them
    // back soon and they are most of the traffic (8192 x 8192 x 1024: 0.162 against 0.175 ms the other way round).
    const bool stream_out = K >= 2048u && !g.ws;
    char *const mine = reinterpret_cast<char *>(smem) + wave * B::TURN;
    // Activations: one uniform branch per row tile to a copy of the code over a lane's 32 outputs.  Sigmoid and tanh are kept
    // out of that unrolled code, where theirs takes longer to fetch than to run: the scaled sums of four row tiles go to LDS
    // as FP32, and one loop, not unrolled, reads them back sixteen a lane, applies the activation and stores whole rows (a loop
    // per row tile, eight copies of it, read and stored in turn: 8192 x 8192 x 448 FP16 and a head with sigmoid 213 -> 185 us, with
    // tanh 239 -> 208, and with tanh_straight, one straight line for the sixteen, as a sigmoid).  150 cycles a value of a lane,
    // what the instructions take.  The same loop does FP16 row tiles with outputs that saturate, infinities or NaNs, which the
    // packed conversion does not know, and rows that are not whole 16-byte units.
    const bool late = !g.ws && (g.L.act == A_SIGMOID || g.L.act == A_TANH);
    // (the lambdas are forced inline: called, they would take what they capture through memory)
    auto turn = [&](auto es_c) __attribute__((always_inline)) {
        constexpr int ES = decltype(es_c)::value;                    // bytes of an element of the output
        constexpr int EPS = 16 / ES;                                 // elements of a 16-byte store
        constexpr int LPR = 128 / EPS, RPP = 64 / LPR;               // lanes that write one row, rows per store instruction
        const int rl0 = lane / LPR, c0 = lane % LPR * EPS;
        auto store = [&](int i, int p, u32x4 vv) __attribute__((always_inline)) {
            const uint32_t row = mrow + i * 16 + p * RPP + rl0, col = ncol + c0;
            if (row >= M || col >= N) return;                        // N is a multiple of EPS: a unit is all in or all out
            u32x4 *dstp = reinterpret_cast<u32x4 *>(out + ((size_t)row * N + col) * ES);
            if (stream_out) __builtin_nontemporal_store(vv, dstp);
            else *dstp = vv;
        };
        constexpr int PUTS = 16 / RPP;
        // the sums of row tile i, scaled and with their bias
        auto sums = [&](auto i_c, float (&v)[32]) __attribute__((always_inline)) {
            static_for<32>([&](auto e_c) __attribute__((always_inline)) {
                constexpr int e = decltype(e_c)::value;
                v[e] = acc_read<decltype(i_c)::value * 32 + e>();
            });
            if (!g.ws) {
#pragma unroll
                for (int e = 0; e < 32; ++e) {
                    const float4 b = bias[e >> 2];
                    v[e] = fmaf(v[e], wscale, (e & 3) == 0 ? b.x : (e & 3) == 1 ? b.y : (e & 3) == 2 ? b.z : b.w);
                }
            }
        };
        uint32_t todo = late || !rows16 ? (1u << RM) - 1u : 0u;      // row tiles for the loop below
        if (!todo) {
            u32x4 held[PUTS];                                        // rows on their way from LDS to memory
            bool pending = false;
            static_for<RM>([&](auto i_c) __attribute__((always_inline)) {
                constexpr int i = decltype(i_c)::value;
                float v[32];
                sums(i_c, v);
                if (!g.ws) {
                    auto each = [&](auto act_c) __attribute__((always_inline)) {
#pragma unroll
                        for (int e = 0; e < 32; ++e) v[e] = decltype(act_c)::value == A_LEAKY ? fmaxf(v[e], 0.01f * v[e]) : apply_act(v[e], decltype(act_c)::value);
                    };
                    if (g.L.act == A_RELU) each(std::integral_constant<int, A_RELU>{});
                    else if (g.L.act == A_LEAKY) each(std::integral_constant<int, A_LEAKY>{});
                    else if (g.L.act == A_FOO52) each(std::integral_constant<int, A_FOO52>{});
                    // padded neurons (only hidden layers of this path have any)
                    if (pad != 0u && ncol + 128u + pad > N) {
#pragma unroll
                        for (int e = 0; e < 32; ++e)
                            if (ncol + (e >> 2) * 16 + 4 * q4 + (e & 3) + pad >= N) v[e] = 0.0f;
                    }
                }
                bool plain = true;
                if constexpr (ES == 2 && F16T) {
                    float top = 0.0f;
#pragma unroll
                    for (int e = 0; e < 32; ++e) top = __builtin_elementwise_maximum(top, __builtin_fabsf(v[e]));
                    plain = __all(top < 65520.0f);
                }
                // the row tile before this one, whose rows were asked for back from LDS before this one's arithmetic
                if (pending) {
#pragma unroll
                    for (int p = 0; p < PUTS; ++p) store(i - 1, p, held[p]);
                }
                pending = plain;
                if (plain) {
                    constexpr int PITCH = 128 * ES + 16;             // rows on different banks
#pragma unroll
                    for (int j = 0; j < 8; ++j) {
                        if constexpr (ES == 4) {
                            *reinterpret_cast<float4 *>(mine + l15 * PITCH + j * 64 + q4 * 16) = make_float4(v[4 * j], v[4 * j + 1], v[4 * j + 2], v[4 * j + 3]);
                        } else {
                            uint2 d;
                            if constexpr (F16T) {
                                d = make_uint2(pack_f16_small(v[4 * j], v[4 * j + 1]), pack_f16_small(v[4 * j + 2], v[4 * j + 3]));
                            } else {
                                d = make_uint2((uint32_t)f32_to_t16<false>(v[4 * j]) | (uint32_t)f32_to_t16<false>(v[4 * j + 1]) << 16,
                                               (uint32_t)f32_to_t16<false>(v[4 * j + 2]) | (uint32_t)f32_to_t16<false>(v[4 * j + 3]) << 16);
                            }
                            *reinterpret_cast<uint2 *>(mine + l15 * PITCH + j * 32 + q4 * 8) = d;
                        }
                    }
                    __builtin_amdgcn_wave_barrier();
#pragma unroll
                    for (int p = 0; p < PUTS; ++p) {
                        const uint4 w = *reinterpret_cast<const uint4 *>(mine + (p * RPP + rl0) * PITCH + c0 * ES);
                        held[p] = u32x4{w.x, w.y, w.z, w.w};
                    }
                    __builtin_amdgcn_wave_barrier();
                } else {
                    todo |= 1u << i;
                }
            });
            if (pending) {
#pragma unroll
                for (int p = 0; p < PUTS; ++p) store(RM - 1, p, held[p]);
            }
        }
        constexpr int PITCH = 128 * 4 + 16;
        constexpr int PASSES = 4 * PUTS, GO = 16 / EPS;              // store instructions of four row tiles, of one turn of the loop
#pragma unroll 1
        for (int four = 0; four < RM; four += 4) {
            if (!(todo >> four & 15u)) continue;
            static_for<RM>([&](auto i_c) __attribute__((always_inline)) {
                constexpr int i = decltype(i_c)::value;
                if (four != (i & ~3)) return;
                float v[32];
                sums(i_c, v);
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    *reinterpret_cast<float4 *>(mine + ((i & 3) * 16 + l15) * PITCH + j * 64 + q4 * 16) = make_float4(v[4 * j], v[4 * j + 1], v[4 * j + 2], v[4 * j + 3]);
            });
            __builtin_amdgcn_wave_barrier();
            // Element x of a lane in the turn at p.  Rows of whole units: of store instruction x / EPS.  Others: 64 neighbouring
            // lanes store 64 neighbouring outputs (16 bytes of a row per lane, stored one element after the other, took
            // 4090 x 4086 x 320 FP16 with FP32 outputs 42 us instead of 34).
            auto row_of = [&](int x) __attribute__((always_inline)) { return rows16 ? x / EPS * RPP + rl0 : x >> 1; };
            auto col_of = [&](int x) __attribute__((always_inline)) { return rows16 ? c0 + x % EPS : (x & 1) * 64 + lane; };
            float next[16];
            auto ask = [&](int p) __attribute__((always_inline)) {
                if (rows16) {
#pragma unroll
                    for (int x = 0; x < 16; x += 4) {
                        const float4 f = *reinterpret_cast<const float4 *>(mine + (p * RPP + row_of(x)) * PITCH + col_of(x) * 4);
                        next[x] = f.x; next[x + 1] = f.y; next[x + 2] = f.z; next[x + 3] = f.w;
                    }
                } else {
#pragma unroll
                    for (int x = 0; x < 16; ++x) next[x] = *reinterpret_cast<const float *>(mine + (p * RPP + row_of(x)) * PITCH + col_of(x) * 4);
                }
            };
            ask(0);
#pragma unroll 1
            for (int p = 0; p < PASSES; p += GO) {
                float e[16];
#pragma unroll
                for (int x = 0; x < 16; ++x) e[x] = next[x];
                if (p + GO < PASSES) ask(p + GO);
                const int i = four + p / PUTS;
                if (!(todo >> i & 1u)) continue;
                // (one branch for all of them: one wave per SIMD hides an exponential only behind another's)
                if (!g.ws) {
                    with_act(g.L.act, [&](auto act_c) __attribute__((always_inline)) {
#pragma unroll
                        for (int x = 0; x < 16; ++x) e[x] = decltype(act_c)::value == A_TANH ? tanh_straight(e[x]) : apply_act(e[x], decltype(act_c)::value);
                    });
                    if (pad != 0u && ncol + 128u + pad > N) {        // padded neurons
#pragma unroll
                        for (int x = 0; x < 16; ++x)
                            if (ncol + col_of(x) + pad >= N) e[x] = 0.0f;
                    }
                }
                if (rows16) {
#pragma unroll
                    for (int k = 0; k < GO; ++k) {
                        const float *const o = e + k * EPS;
                        u32x4 vv;
#pragma unroll
                        for (int x = 0; x < 4; ++x) {
                            if constexpr (ES == 4) vv[x] = __float_as_uint(o[x]);
                            else vv[x] = (uint32_t)f32_to_t16<F16T>(o[2 * x]) | (uint32_t)f32_to_t16<F16T>(o[2 * x + 1]) << 16;
                        }
                        store(i, p % PUTS + k, vv);
                    }
                } else {
#pragma unroll
                    for (int x = 0; x < 16; ++x) {
                        const uint32_t row = mrow + four * 16 + p * RPP + row_of(x), col = ncol + col_of(x);
                        if (row >= M || col >= N) continue;
                        const size_t at = (size_t)row * N + col;
                        if constexpr (ES == 4) reinterpret_cast<float *>(out)[at] = e[x];
                        else reinterpret_cast<uint16_t *>(out)[at] = f32_to_t16<F16T>(e[x]);
                    }
                }
            }
            __builtin_amdgcn_wave_barrier();
        }
    };
    if (f32_out) turn(std::integral_constant<int, 4>{});
    else turn(std::integral_constant<int, 2>{});
}

// The parts of four neighbouring sums, `stride` float4 apart: the first `splits` added in order into sum, the others into low.
// Four are on their way at a time: one after the other, each is a round trip to memory (sixteen parts of 50 x 1000 sums 6.9 ->
// 6.4 us; four of 50 x 8192, which fill the chip, 4.8 / 4.9).
__device__ __forceinline__ void add_parts(const float4 *at, uint64_t stride, uint32_t splits, uint32_t parts, float4 &sum, float4 &low)
{
    sum = low = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    for (uint32_t p0 = 0; p0 < parts; p0 += 4u) {
        float4 v[4];
#pragma unroll
        for (uint32_t i = 0; i < 4u; ++i) v[i] = at[(p0 + i < parts ? p0 + i : p0) * stride];
#pragma unroll
        for (uint32_t i = 0; i < 4u; ++i) {
            if (p0 + i >= parts) continue;
            float4 &to = p0 + i < splits ? sum : low;
            to.x += v[i].x; to.y += v[i].y; to.z += v[i].z; to.w += v[i].w;
        }
    }
}

// adds the partial sums of a split launch (K splits in split order; with split activations the sums of the second
// matrix, scaled by 2^-11, after those of the first) and applies scale, bias and activation; a thread takes four
// neighbouring columns (VEC: N a multiple of four, workspace and C 16-byte aligned) or one.  16-bit outputs of a
// split-activation forward are written as the two matrices of the next layer's input (g.halves == 2).
template <bool F16T, bool VEC>
__global__ __launch_bounds__(256) void sp_gemm16_reduce(const GemmArgs g, uint32_t splits)
{
    const uint64_t total = (uint64_t)g.M * g.L.N;
    const uint32_t parts = splits * g.halves;
    if constexpr (VEC) {
        const uint64_t idx = ((uint64_t)blockIdx.x * 256u + threadIdx.x) * 4u;
        if (idx >= total) return;
        const uint32_t col = (uint32_t)(idx % g.L.N);
        float bias[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) bias[i] = elem_value_rt(g.L.bias_fmt, g.L.bias, col + i) * g.L.bscale;
        float4 sum, low;
        add_parts(reinterpret_cast<const float4 *>(g.ws + idx), total / 4u, splits, parts, sum, low);
        const float in[4] = {fmaf(low.x, kLoScale, sum.x), fmaf(low.y, kLoScale, sum.y), fmaf(low.z, kLoScale, sum.z),
                             fmaf(low.w, kLoScale, sum.w)};
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            v[i] = apply_act(layer_sum(g.L, in[i], bias[i], col + i), g.L.act);
        }
        if (g.out_f32) {
            *reinterpret_cast<float4 *>(reinterpret_cast<float *>(g.C) + idx) = make_float4(v[0], v[1], v[2], v[3]);
        } else if (g.halves == 2) {
            uint16_t hi[4], lo[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) split_f16(v[i], hi[i], lo[i]);
            uint16_t *c = reinterpret_cast<uint16_t *>(g.C);
            *reinterpret_cast<uint2 *>(c + idx) = make_uint2((uint32_t)hi[0] | ((uint32_t)hi[1] << 16), (uint32_t)hi[2] | ((uint32_t)hi[3] << 16));
            *reinterpret_cast<uint2 *>(c + total + idx) = make_uint2((uint32_t)lo[0] | ((uint32_t)lo[1] << 16), (uint32_t)lo[2] | ((uint32_t)lo[3] << 16));
        } else {
            const uint32_t lo = (uint32_t)f32_to_t16<F16T>(v[0]) | ((uint32_t)f32_to_t16<F16T>(v[1]) << 16);
            const uint32_t hi = (uint32_t)f32_to_t16<F16T>(v[2]) | ((uint32_t)f32_to_t16<F16T>(v[3]) << 16);
            *reinterpret_cast<uint2 *>(reinterpret_cast<uint16_t *>(g.C) + idx) = make_uint2(lo, hi);
        }
    } else {
        const uint64_t idx = (uint64_t)blockIdx.x * 256u + threadIdx.x;
        if (idx >= total) return;
        float sum = 0.0f, low = 0.0f;
        for (uint32_t sp = 0; sp < parts; ++sp) {
            const float v = g.ws[(uint64_t)sp * total + idx];
            if (sp < splits) sum += v; else low += v;
        }
        const uint32_t col = (uint32_t)(idx % g.L.N);
        const float bias = elem_value_rt(g.L.bias_fmt, g.L.bias, col) * g.L.bscale;
        const float v = apply_act(layer_sum(g.L, fmaf(low, kLoScale, sum), bias, col), g.L.act);
        if (g.out_f32) reinterpret_cast<float *>(g.C)[idx] = v;
        else if (g.halves == 2) {
            uint16_t hi, lo;
            split_f16(v, hi, lo);
            reinterpret_cast<uint16_t *>(g.C)[idx] = hi;
            reinterpret_cast<uint16_t *>(g.C)[total + idx] = lo;
        } else reinterpret_cast<uint16_t *>(g.C)[idx] = f32_to_t16<F16T>(v);
    }
}
