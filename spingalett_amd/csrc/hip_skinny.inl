// hip_skinny.inl — the streaming MFMA kernels for layers with one thin side (sp_skinny16,
// sp_skinny16_kw, sp_skinny_reduce, sp_codes16).  Part of hip_forward.hip's translation unit (included
// there, inside its unnamed namespace); not compiled on its own.

// ---------------------------------------------------------------------------
// Streaming MFMA kernel for layers with one thin side
// ---------------------------------------------------------------------------
// Few samples (5 .. 256) or few outputs (<= 64): one operand is a tall matrix that is
// read exactly once (the weights, or the 16-bit activations when the layer has few
// outputs), the other a thin 16-bit matrix of at most 64 rows per workgroup.  The tall
// operand never touches LDS: a workgroup has NWV waves (4 or 8), a wave owns RT tiles of 32 streamed rows and loads them
// straight into registers, 16 bytes per lane, one chunk ahead; lanes 0-31 and 32-63 take
// adjacent 16-byte pieces of a row.  The integer codes become FP16 pairs with the
// 0x6400 | code trick (1024 + code, minus the constant, exact), which delivers the codes
// of a step in a format-specific order; the thin operand is written to LDS in that same
// order, so both MFMA operands agree on which k sits where.
// Workgroups split K (grid y) to fill the chip; partial tiles go to a workspace and a
// second launch adds them, otherwise the epilogue is applied here.
struct SkinnyArgs {
    LayerArgs L;
    const uint8_t *stream;   // streamed rows, K codes each
    const uint16_t *thin;    // [NC][K] 16-bit
    void *C;                 // [M][N]
    float *ws;               // [S][NC][R] partial sums when the grid splits K
    uint32_t R, NC;          // streamed rows, thin rows
    uint32_t row_blocks, cblocks;   // workgroups along the streamed rows / blocks of thin rows (grid x covers both)
    uint32_t kper;           // codes per K split (whole chunks)
    int out_f32;
    int mode_b;              // 0: streamed rows are outputs, thin rows samples; 1: the reverse
    // Softmax over a sample's outputs goes here instead of C: by sp_skinny16_kw_head itself where K is not split, by sp_sum_softmax
    // with the addition of the parts behind streamed weights (launch_thin)
    void *soft_out;
    int soft_kind;           // its element type: 0 FP32, 1 BF16, 2 FP16, 3 FP16 in two halves (sp_sum_softmax only)
    // Split activations (GemmArgs has the layout): grid y = halves x ksplits, y / ksplits picks the activation matrix
    // (the thin operand, or the streamed one in mode b), y % ksplits the K range.
    uint32_t ksplits;        // K splits (>= 1)
    uint32_t halves;         // 1, or 2 with split activations
    uint32_t parts;          // partial sums of an output in ws: ksplits x halves, or ksplits where a workgroup adds the halves
    uint64_t half_elems;     // elements between the two activation matrices (samples x K)
};

template <int FMT>
struct SkinnyFmt {
    static constexpr int bits = fmt_bits(FMT);
    static constexpr int EPL = 128 / bits;                                  // codes per 16-byte lane load
    static constexpr int LPC = (FMT == I2) ? 2 : 4;                         // lane loads per chunk and tile
    static constexpr int BKC = 2 * LPC * EPL;                               // codes per chunk: 64 (16-bit), 128, 256, 256
    static constexpr int STEPS = EPL / 8;                                   // MFMA k-steps per lane load
    static constexpr int PITCH = BKC * 2 + 16;                              // LDS row pitch: 16 rows hit 16 different slots
};

// position p of a 16-code group holds code skinny_perm(p) of the group
template <int FMT>
__host__ __device__ constexpr int skinny_perm(int p)
{
    if (FMT == I8) { constexpr int t[8] = {0, 2, 1, 3, 4, 6, 5, 7}; return t[p & 7] + (p & 8); }
    if (FMT == I4) { constexpr int t[8] = {0, 4, 1, 5, 2, 6, 3, 7}; return t[p & 7] + (p & 8); }
    if (FMT == I2) { constexpr int t[16] = {0, 8, 1, 9, 2, 10, 3, 11, 4, 12, 5, 13, 6, 14, 7, 15}; return t[p]; }
    return p;
}

// the 16 codes of a unit of the thin operand (eight 16-bit pairs) in the order skinny_perm gives
template <int FMT>
__device__ __forceinline__ void skinny_permute_unit(const uint32_t (&in)[8], uint32_t (&o)[8])
{
#pragma unroll
    for (int w = 0; w < 8; ++w) {
        const int ea = skinny_perm<FMT>(2 * w), eb = skinny_perm<FMT>(2 * w + 1);
        const uint32_t sel = (uint32_t)(2 * (ea & 1)) | ((uint32_t)(2 * (ea & 1) + 1) << 8) |
                             ((uint32_t)(4 + 2 * (eb & 1)) << 16) | ((uint32_t)(4 + 2 * (eb & 1) + 1) << 24);
        o[w] = __builtin_amdgcn_perm(in[eb >> 1], in[ea >> 1], sel);
    }
}

typedef _Float16 h16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t magic_sub(uint32_t v, uint32_t c)
{
    h16x2 a, b;
    __builtin_memcpy(&a, &v, 4);
    __builtin_memcpy(&b, &c, 4);
    a = a - b;
    uint32_t r;
    __builtin_memcpy(&r, &a, 4);
    return r;
}

// The 8 values of k-step j of one lane load, as four FP16 pairs.  A field of the word is
// masked in place and XORed onto an FP16 constant whose last mantissa bit has the weight of
// the field's lowest bit (1024 for bit 0, 256 for bit 2, 64 for bit 4, ...), the same XOR flips
// the field's sign bit (two's complement -> offset binary); subtracting the constant plus the
// offset leaves the code, exactly.  Only fields above the 10 mantissa bits need a shift first.
template <int FMT>
__device__ __forceinline__ void skinny_frag(const uint4 &v, int j, uint32_t (&f)[4])
{
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
    if constexpr (FMT == I8) {
        // word = codes b0 b1 b2 b3: pairs (b0, b2) and (b1, b3)
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const uint32_t x = w[2 * j + q];
            f[2 * q]     = magic_sub((x & 0x00FF00FFu) ^ 0x64806480u, 0x64806480u);          // 1024 + 128 + q
            f[2 * q + 1] = magic_sub(((x >> 8) & 0x00FF00FFu) ^ 0x64806480u, 0x64806480u);
        }
    } else if constexpr (FMT == I4) {
        // word = nibbles c0 .. c7: pairs (c0, c4), (c1, c5), (c2, c6), (c3, c7)
        const uint32_t x = w[j], y = x >> 8;
        f[0] = magic_sub((x & 0x000F000Fu) ^ 0x64086408u, 0x64086408u);                      // 1024 + 8 + q
        f[1] = magic_sub((x & 0x00F000F0u) ^ 0x54805480u, 0x54805480u);                      // 64 + 8 + q
        f[2] = magic_sub((y & 0x000F000Fu) ^ 0x64086408u, 0x64086408u);
        f[3] = magic_sub((y & 0x00F000F0u) ^ 0x54805480u, 0x54805480u);
    } else if constexpr (FMT == I2) {
        // word = fields c0 .. c15: step 0 pairs (c0, c8) .. (c3, c11), step 1 pairs (c4, c12) .. (c7, c15)
        const uint32_t x = w[j >> 1];
        if ((j & 1) == 0) {
            f[0] = magic_sub((x & 0x00030003u) ^ 0x64026402u, 0x64026402u);                  // 1024 + 2 + q
            f[1] = magic_sub((x & 0x000C000Cu) ^ 0x5C085C08u, 0x5C085C08u);                  // 256 + 2 + q
            f[2] = magic_sub((x & 0x00300030u) ^ 0x54205420u, 0x54205420u);                  // 64 + 2 + q
            f[3] = magic_sub((x & 0x00C000C0u) ^ 0x4C804C80u, 0x4C804C80u);                  // 16 + 2 + q
        } else {
            const uint32_t y = x >> 10;
            f[0] = magic_sub((x & 0x03000300u) ^ 0x46004600u, 0x46004600u);                  // 4 + 2 + q
            f[1] = magic_sub((y & 0x00030003u) ^ 0x64026402u, 0x64026402u);
            f[2] = magic_sub((y & 0x000C000Cu) ^ 0x5C085C08u, 0x5C085C08u);
            f[3] = magic_sub((y & 0x00300030u) ^ 0x54205420u, 0x54205420u);
        }
    } else {
        f[0] = w[0]; f[1] = w[1]; f[2] = w[2]; f[3] = w[3];
    }
}

// ACT: the layer's activation where it is known at compile time (with_act), or -1
template <bool F16T, int ACT = -1>
__device__ __forceinline__ void skinny_emit_biased(const SkinnyArgs &a, uint32_t c, uint32_t r, float accv, float bias)
{
    const uint32_t m = a.mode_b ? r : c, n = a.mode_b ? c : r;
    const float v = apply_act(layer_sum(a.L, accv, bias, n), ACT < 0 ? a.L.act : ACT);
    const size_t o = (size_t)m * a.L.N + n;
    if (a.out_f32) reinterpret_cast<float *>(a.C)[o] = v;
    else reinterpret_cast<uint16_t *>(a.C)[o] = f32_to_t16<F16T>(v);
}

template <bool F16T>
__device__ __forceinline__ void skinny_emit(const SkinnyArgs &a, uint32_t c, uint32_t r, float accv)
{
    const float bias = elem_value_rt(a.L.bias_fmt, a.L.bias, a.mode_b ? c : r) * a.L.bscale;
    skinny_emit_biased<F16T>(a, c, r, accv, bias);
}

template <int FMT, bool F16T, int RT, int CT, int NWV>
__global__ __launch_bounds__(64 * NWV) void sp_skinny16_regs(const SkinnyArgs a)
{
    using F = SkinnyFmt<FMT>;
    constexpr int EPL = F::EPL, LPC = F::LPC, BKC = F::BKC, STEPS = F::STEPS, PITCH = F::PITCH;
    constexpr int UNITS = 32 * CT * (BKC / 16);            // 16-code units of a thin chunk
    constexpr int NT = 64 * NWV;                           // threads of a workgroup
    constexpr int UPT = (UNITS + NT - 1) / NT;
    constexpr int STAGE = 32 * CT * PITCH;
    extern __shared__ __attribute__((aligned(16))) uint8_t sk_lds[];

    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const uint32_t n31 = lane & 31, h = lane >> 5;
    const uint32_t K = a.L.K;
    // Grid x enumerates (row block, thin block).  Consecutive workgroup ids go to consecutive dies (eight of them,
    // each with its own L2): the thin blocks of one row block get ids eight apart, so they run on the same die at
    // about the same time and the second and later ones find the streamed rows in its L2.
    uint32_t rblk = blockIdx.x, cblk = 0;
    if (a.cblocks > 1) {
        const uint32_t per = 8u * a.cblocks, group = blockIdx.x / per, rem = blockIdx.x % per;
        rblk = group * 8u + (rem & 7u);
        cblk = rem >> 3;
        if (rblk >= a.row_blocks) return;                 // padding of the last group
    }
    const uint32_t row0 = (rblk * (uint32_t)NWV + (uint32_t)wave) * (32u * RT);
    const uint32_t cbase = cblk * (32u * CT);
    const uint32_t half = blockIdx.y / a.ksplits;
    const uint8_t *const stream = a.mode_b ? a.stream + (size_t)half * a.half_elems * 2u : a.stream;
    const uint16_t *const thin = a.mode_b ? a.thin : a.thin + (size_t)half * a.half_elems;
    const uint32_t kbeg = (blockIdx.y % a.ksplits) * a.kper;
    const uint32_t kend = kbeg + a.kper < K ? kbeg + a.kper : K;
    const uint32_t nchunks = (kend - kbeg + BKC - 1) / BKC;
    const size_t row_bytes = (size_t)K * F::bits / 8u;

    // per-lane byte offsets (32-bit: the host checks that both operands span less than 4 GiB)
    uint32_t svoff[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        const uint32_t r = row0 + rt * 32u + n31;
        svoff[rt] = (uint32_t)((size_t)(r < a.R ? r : a.R - 1) * row_bytes) + h * 16u;
    }
    uint32_t tvoff[UPT][2];
    bool trow_ok[UPT];
#pragma unroll
    for (int q = 0; q < UPT; ++q) {
        const uint32_t u = (uint32_t)t + (uint32_t)NT * q;
        const uint32_t row = u / (BKC / 16), uc = u % (BKC / 16);
        const uint32_t c = cbase + row;
        trow_ok[q] = u < (uint32_t)UNITS && c < a.NC;
#pragma unroll
        for (int e = 0; e < 2; ++e) tvoff[q][e] = trow_ok[q] ? (uint32_t)(((size_t)c * K + uc * 16u + 8u * e) * 2u) : 0u;
    }

    f32x16 acc[RT][CT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int ct = 0; ct < CT; ++ct)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[rt][ct][r] = 0.0f;

    // Loads are issued two chunks ahead for the streamed rows and one ahead for the thin block.  A chunk past
    // the end is clamped to the last one (a redundant load) so that the number of loads in flight is always the
    // same.  In the last chunk a lane load that would start past the end of its row reads the row's start
    // instead; what it fetched is masked (16-bit values) or meets zeros of the thin operand (integer codes).
    constexpr int S_LOADS = RT * LPC, T_LOADS = UPT * 2;
    const uint32_t last_chunk = nchunks - 1;
    auto issue_stream = [&](uint32_t ch, u32x4 (&dst)[RT][LPC]) {
        if (ch < last_chunk) {
            const uint8_t *sb = stream + (size_t)(kbeg + ch * BKC) * F::bits / 8u;
#pragma unroll
            for (int i = 0; i < LPC; ++i)
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) {
                    if (i == 0) load16_async<0>(dst[rt][i], svoff[rt], sb);
                    else if (i == 1) load16_async<32>(dst[rt][i], svoff[rt], sb);
                    else if (i == 2) load16_async<64>(dst[rt][i], svoff[rt], sb);
                    else load16_async<96>(dst[rt][i], svoff[rt], sb);
                }
        } else {
            const uint32_t kc0 = kbeg + last_chunk * BKC;
#pragma unroll
            for (int i = 0; i < LPC; ++i) {
                const uint32_t k = kc0 + 2u * i * EPL;                 // first code of the h = 0 lane load
                const uint32_t add = k + h * EPL < K ? k * F::bits / 8u : 0u - h * 16u;
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) load16_async<0>(dst[rt][i], svoff[rt] + add, stream);
            }
        }
    };
    u32x4 thin_regs[UPT][2];
    auto issue_thin = [&](uint32_t ch) {
        if (ch < last_chunk) {
            const uint16_t *tb = thin + (kbeg + ch * BKC);
#pragma unroll
            for (int q = 0; q < UPT; ++q)
#pragma unroll
                for (int e = 0; e < 2; ++e) load16_async<0>(thin_regs[q][e], tvoff[q][e], tb);
        } else {
            const uint32_t kc0 = kbeg + last_chunk * BKC;
#pragma unroll
            for (int q = 0; q < UPT; ++q) {
                const uint32_t uc = ((uint32_t)t + (uint32_t)NT * q) % (BKC / 16);
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const bool valid = trow_ok[q] && kc0 + uc * 16u + 8u * e + 8u <= kend;
                    load16_async<0>(thin_regs[q][e], valid ? tvoff[q][e] + kc0 * 2u : 0u, thin);
                }
            }
        }
    };
    // ties the registers to the preceding wait: nothing that reads them is scheduled above it
    auto pin_stream = [&](u32x4 (&r)[RT][LPC]) {
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int i = 0; i < LPC; ++i) asm volatile("" : "+v"(r[rt][i]));
    };
    auto pin_thin = [&]() {
#pragma unroll
        for (int q = 0; q < UPT; ++q)
#pragma unroll
            for (int e = 0; e < 2; ++e) asm volatile("" : "+v"(thin_regs[q][e]));
    };
    auto store_thin = [&](int stage, uint32_t ch) {
        const uint32_t kc0 = kbeg + (ch < last_chunk ? ch : last_chunk) * BKC;
#pragma unroll
        for (int q = 0; q < UPT; ++q) {
            const uint32_t u = (uint32_t)t + (uint32_t)NT * q;
            if (u >= (uint32_t)UNITS) continue;
            const uint32_t row = u / (BKC / 16), uc = u % (BKC / 16);
            const uint32_t k = kc0 + uc * 16u;
            const uint32_t keep0 = (trow_ok[q] && k + 8u <= kend) ? 0xFFFFFFFFu : 0u;
            const uint32_t keep1 = (trow_ok[q] && k + 16u <= kend) ? 0xFFFFFFFFu : 0u;
            const uint32_t in[8] = {thin_regs[q][0].x & keep0, thin_regs[q][0].y & keep0, thin_regs[q][0].z & keep0,
                                    thin_regs[q][0].w & keep0, thin_regs[q][1].x & keep1, thin_regs[q][1].y & keep1,
                                    thin_regs[q][1].z & keep1, thin_regs[q][1].w & keep1};
            uint32_t o[8];
            skinny_permute_unit<FMT>(in, o);
            uint8_t *dst = sk_lds + stage * STAGE + row * PITCH + uc * 32u;
            *reinterpret_cast<uint4 *>(dst) = make_uint4(o[0], o[1], o[2], o[3]);
            *reinterpret_cast<uint4 *>(dst + 16) = make_uint4(o[4], o[5], o[6], o[7]);
        }
    };

    auto compute = [&](int stage, uint32_t ch, const u32x4 (&cur)[RT][LPC]) {
        const uint8_t *sbase = sk_lds + stage * STAGE + n31 * PITCH + h * (EPL * 2);
        const uint32_t kc0 = kbeg + ch * BKC;
#pragma unroll
        for (int i = 0; i < LPC; ++i) {
            // 16-bit values past the end of the row could be NaN or infinite: masked (integer codes need not be)
            const uint32_t keep = (F::bits == 16 && kc0 + (2u * i + h) * EPL >= K) ? 0u : 0xFFFFFFFFu;
#pragma unroll
            for (int j = 0; j < STEPS; ++j) {
                const int koff = (2 * i * EPL + 8 * j) * 2;
                uint4 tf[CT];
#pragma unroll
                for (int ct = 0; ct < CT; ++ct) tf[ct] = *reinterpret_cast<const uint4 *>(sbase + ct * 32 * PITCH + koff);
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) {
                    uint4 v = make_uint4(cur[rt][i].x, cur[rt][i].y, cur[rt][i].z, cur[rt][i].w);
                    if constexpr (F::bits == 16) { v.x &= keep; v.y &= keep; v.z &= keep; v.w &= keep; }
                    uint32_t sf[4];
                    skinny_frag<FMT>(v, j, sf);
#pragma unroll
                    for (int ct = 0; ct < CT; ++ct) {
                        if constexpr (F16T) {
                            f16x8 af, bf;
                            __builtin_memcpy(&af, &tf[ct], 16);
                            __builtin_memcpy(&bf, sf, 16);
                            acc[rt][ct] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af, bf, acc[rt][ct], 0, 0, 0);
                        } else {
                            bf16x8 af, bf;
                            __builtin_memcpy(&af, &tf[ct], 16);
                            __builtin_memcpy(&bf, sf, 16);
                            acc[rt][ct] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af, bf, acc[rt][ct], 0, 0, 0);
                        }
                    }
                }
            }
        }
    };
    // One chunk.  In flight on entry: streamed chunks ch (in `cur`) and ch + 1; issued here: the thin block of
    // ch + 1, then streamed chunk ch + 2 into `far`.  Loads complete in order, so waiting until only the S_LOADS
    // youngest are outstanding means the thin block (and everything older) has arrived.
    auto step = [&](uint32_t ch, u32x4 (&cur)[RT][LPC], u32x4 (&far)[RT][LPC]) {
        const int stage = (int)(ch & 1u);
        issue_thin(ch + 1);
        issue_stream(ch + 2, far);
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * S_LOADS + T_LOADS) : "memory");    // chunk ch is here
        pin_stream(cur);
        compute(stage, ch, cur);
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(S_LOADS) : "memory");
        pin_thin();
        store_thin(stage ^ 1, ch + 1);
        __syncthreads();
    };

    u32x4 ra[RT][LPC], rb[RT][LPC], rc[RT][LPC];
    issue_thin(0);
    issue_stream(0, ra);
    issue_stream(1, rb);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * S_LOADS) : "memory");
    pin_thin();
    store_thin(0, 0);
    __syncthreads();
    for (uint32_t ch = 0; ch < nchunks; ch += 3) {
        step(ch, ra, rc);
        if (ch + 1 < nchunks) step(ch + 1, rb, ra);
        if (ch + 2 < nchunks) step(ch + 2, rc, rb);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // the redundant tail loads

    // accumulator register r of lane (n31, h): thin row 8 (r / 4) + 4 h + r % 4, streamed row n31
    if (a.ws) {
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            const uint32_t r = row0 + rt * 32u + n31;
            if (r >= a.R) continue;
#pragma unroll
            for (int ct = 0; ct < CT; ++ct)
#pragma unroll
                for (int q = 0; q < 16; ++q) {
                    const uint32_t c = cbase + ct * 32u + 8u * (q >> 2) + 4u * h + (q & 3);
                    if (c < a.NC) a.ws[((size_t)blockIdx.y * a.NC + c) * a.R + r] = acc[rt][ct][q];
                }
        }
        return;
    }
    auto emit = [&](auto act_c) __attribute__((always_inline)) {
        constexpr int ACT = decltype(act_c)::value;
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            const uint32_t r = row0 + rt * 32u + n31;
            if (r >= a.R) continue;
            // streamed rows that are outputs have one bias per lane and row tile
            const float bias_r = a.mode_b ? 0.0f : elem_value_rt(a.L.bias_fmt, a.L.bias, r) * a.L.bscale;
#pragma unroll
            for (int ct = 0; ct < CT; ++ct)
#pragma unroll
                for (int q = 0; q < 16; ++q) {
                    const uint32_t c = cbase + ct * 32u + 8u * (q >> 2) + 4u * h + (q & 3);
                    if (c >= a.NC) continue;
                    const float bias = a.mode_b ? elem_value_rt(a.L.bias_fmt, a.L.bias, c) * a.L.bscale : bias_r;
                    skinny_emit_biased<F16T, ACT>(a, c, r, acc[rt][ct][q], bias);
                }
        }
    };
    with_act(a.L.act, emit);
}

// ---------------------------------------------------------------------------
// Layers of 9 .. 256 samples whose weights are streamed: everything through LDS by DMA
// ---------------------------------------------------------------------------
// A workgroup of eight waves owns 128 weight rows x 16 ST samples (ST <= 4) x a share of K (grid y), in chunks of BK.  Wave
// (g, w): rows 32 w .. 32 w + 31, the g-th half of every chunk's k; the halves' sums meet in LDS at the end.
//
// The kernel before spent 1.35 us per chunk of 256 INT2 codes on 64 samples (8192 x 8192: 8 chunks a workgroup) where the matrix
// cores need 0.45: its loads alone take 0.8 (a lane reads 16 bytes of a weight row of its own, so that four lanes touch four
// lines, and half of each line of the samples at a time), its arithmetic alone 0.95 (unpacking and reordering samples
// next to the products of one wave per SIMD), and two waves per SIMD with loads like these gain nothing.  Here
//   * every load is global_load_lds_dwordx4 of whole 64- to 512-byte pieces of rows, NSTAGE - 1 chunks ahead, counted with
//     vmcnt; one barrier per chunk;
//   * samples stay in their own order; the codes are put in order as they are unpacked (unpack_word16);
//   * the two waves of a SIMD work on different halves of the same chunk, so that the second wave costs no loads.
// 8192 x 8192 INT2 at 20 samples 14.5 -> 10.2 us, at 50 15.9 -> 14.2, the reducing launch not counted.
// LDS: a row of a chunk is whole, unpadded, its 16-byte pieces permuted by the row (swz) so that the sixteen rows of a
// fragment read lie on different banks.  Lane (l15, q4) of a wave takes, of row l15 of a tile, the k-quarter q4 of its half
// chunk: which k an operation sums does not matter as long as both operands agree.
template <int FMT>
struct ThinFmt {
    static constexpr int bits = fmt_bits(FMT);
    static constexpr int BK = FMT == I2 || FMT == I4 ? 256 : 128;
    static constexpr int EPL = 128 / bits;                      // codes of a 16-byte piece
    static constexpr int TROW = BK * 2, WROW = BK * bits / 8;   // bytes of a chunk's row
    static constexpr int KQ = BK / 8;                           // k of a lane and chunk: its quarter of its half
    template <int ST>
    struct Tile {
        static constexpr int W_AT = ST * 16 * TROW, STAGE = W_AT + 128 * WROW;
        static constexpr int NSTAGE = 4 * STAGE <= 160 * 1024 ? 4 : 3;
        static constexpr int T_DMA = (ST * 16 * TROW / 1024 + 7) / 8, W_DMA = 128 * WROW / 8192;    // load instructions per wave and chunk
        static constexpr int LDS = NSTAGE * STAGE;
    };
};

// Position of piece p in row r of ROW bytes, and the piece at a position.  A row covers ROW / 256 of the banks' 256 bytes: rows
// that share them get different positions for the same piece, and the lanes of a fragment read that are served together
// (sixteen of them, rows 4 .. 11 of one k-quarter beside rows 0 .. 3 and 12 .. 15 of the one before) too: their pieces may
// differ in the lowest two bits of the sixteen positions only, so that of 512-byte rows, where a quarter is four pieces, they
// trade places with the two above them.
template <int ROW>
__device__ __forceinline__ uint32_t thin_mask(uint32_t r)
{
    return ROW >= 256 ? r & 15u : ROW == 128 ? (r >> 1) & 7u : (r >> 2) & 3u;
}
__device__ __forceinline__ uint32_t thin_trade(uint32_t p) { return (p & ~15u) | (p & 3u) << 2 | ((p >> 2) & 3u); }
template <int ROW>
__device__ __forceinline__ uint32_t thin_pos(uint32_t r, uint32_t p) { return (ROW == 512 ? thin_trade(p) : p) ^ thin_mask<ROW>(r); }
template <int ROW>
__device__ __forceinline__ uint32_t thin_piece(uint32_t r, uint32_t pos)
{
    const uint32_t p = pos ^ thin_mask<ROW>(r);
    return ROW == 512 ? thin_trade(p) : p;
}

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

template <int OFF>
__device__ __forceinline__ void ds_read64(u32x2 &dst, uint32_t addr)
{
    asm volatile("ds_read_b64 %0, %1 offset:%2" : "=v"(dst) : "v"(addr), "n"(OFF));
}

template <int FMT, bool F16T, int ST>
__global__ __launch_bounds__(512) void sp_skinny16(const SkinnyArgs a)
{
    using F = ThinFmt<FMT>;
    using T = typename F::template Tile<ST>;
    constexpr int BK = F::BK, EPL = F::EPL, TROW = F::TROW, WROW = F::WROW, KQ = F::KQ, bits = F::bits;
    constexpr int STAGE = T::STAGE, W_AT = T::W_AT, NSTAGE = T::NSTAGE, T_DMA = T::T_DMA, W_DMA = T::W_DMA;
    constexpr bool W16 = bits == 16;
    extern __shared__ __attribute__((aligned(16))) uint8_t sk_lds[];

    const uint32_t lane = threadIdx.x & 63u, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const uint32_t l15 = lane & 15u, q4 = lane >> 4, w = wave & 3u, g = wave >> 2;
    const uint32_t K = a.L.K;
    // (row block, sample block) as in sp_skinny16_regs
    uint32_t rblk = blockIdx.x, cblk = 0;
    if (a.cblocks > 1) {
        const uint32_t per = 8u * a.cblocks, group = blockIdx.x / per, rem = blockIdx.x % per;
        rblk = group * 8u + (rem & 7u);
        cblk = rem >> 3;
        if (rblk >= a.row_blocks) return;                 // padding of the last group
    }
    const uint32_t row0 = rblk * 128u, cbase = cblk * (16u * ST);
    const uint16_t *const thin = a.thin + (size_t)(blockIdx.y / a.ksplits) * a.half_elems;
    const uint32_t kbeg = (blockIdx.y % a.ksplits) * a.kper;
    const uint32_t kend = kbeg + a.kper < K ? kbeg + a.kper : K;
    const uint32_t nchunks = (kend - kbeg + BK - 1) / BK;
    // Neighbouring row blocks begin at different chunks: where rows are a large power of two of bytes long, the same chunk of
    // all rows lies in a few of the memory's channels, and workgroups that all begin at the first one move over the channels
    // together (cold weights: 16384 x 16384 INT4 at 8 samples 44 -> 33 us, INT8 at 16 76 -> 53, 16384 x 8192 INT8 42 -> 32,
    // 32768 x 8192 FP16 157 -> 92; other rows even).  With several blocks of samples their chunks, of which a die then
    // reads many at once, cost more than that (16384 x 16384 INT8 at 100 samples 88 -> 104 us).
    const uint32_t turn = a.cblocks > 1 ? 0u : rblk % nchunks;
    auto turned = [&](uint32_t c) { return c + turn >= nchunks ? c + turn - nchunks : c + turn; };
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)sk_lds;

    // This wave's load instructions: 1 KiB of LDS each, instruction i of wave v fills bytes 1024 (8 i + v) + 16 lane of the
    // samples' or the weights' part.  Lane offsets (32-bit: the host checks that both operands span less than 4 GiB), and the
    // k of the piece in its chunk.
    uint32_t t_off[T_DMA], w_off[W_DMA], t_k[T_DMA], w_k[W_DMA];
#pragma unroll
    for (int i = 0; i < T_DMA; ++i) {
        const uint32_t at = (8u * i + wave) * 1024u + lane * 16u, r = at / TROW, p = thin_piece<TROW>(r, at % TROW / 16u);
        const uint32_t c = cbase + r < a.NC ? cbase + r : a.NC - 1u;
        t_k[i] = p * 8u;
        t_off[i] = (uint32_t)(((size_t)c * K + t_k[i]) * 2u);
    }
#pragma unroll
    for (int i = 0; i < W_DMA; ++i) {
        const uint32_t at = (8u * i + wave) * 1024u + lane * 16u, r = at / WROW, p = thin_piece<WROW>(r, at % WROW / 16u);
        const uint32_t n = row0 + r < a.R ? row0 + r : a.R - 1u;
        w_k[i] = p * EPL;
        w_off[i] = (uint32_t)((size_t)n * ((size_t)K * bits / 8u) + p * 16u);
    }
    constexpr bool T_FULL = ST * 16 * TROW % 8192 == 0;     // every wave has T_DMA of them (else the later waves have one less)
    const bool t_last = T_FULL || (8u * (T_DMA - 1) + wave) * 1024u < (uint32_t)(ST * 16 * TROW);
    auto load = [&](uint32_t stage, uint32_t ch) __attribute__((always_inline)) {
        const uint32_t k0 = kbeg + ch * BK;
        const uint32_t to = lds0 + stage + wave * 1024u;
        const uint8_t *const tb = reinterpret_cast<const uint8_t *>(thin) + (size_t)k0 * 2u;
        const uint8_t *const wb = a.stream + (size_t)k0 * bits / 8u;
        if (k0 + BK <= kend) {
#pragma unroll
            for (int i = 0; i < W_DMA; ++i) lds_dma16(to + (uint32_t)(W_AT + i * 8192), w_off[i], wb);
#pragma unroll
            for (int i = 0; i < T_DMA; ++i)
                if (i < T_DMA - 1 || t_last) lds_dma16(to + (uint32_t)(i * 8192), t_off[i], tb);
        } else {
            // the partial chunk at the end of K: pieces past the end of their row come from the chunk's start
#pragma unroll
            for (int i = 0; i < W_DMA; ++i) lds_dma16(to + (uint32_t)(W_AT + i * 8192), k0 + w_k[i] < kend ? w_off[i] : w_off[i] - w_k[i] * bits / 8u, wb);
#pragma unroll
            for (int i = 0; i < T_DMA; ++i)
                if (i < T_DMA - 1 || t_last) lds_dma16(to + (uint32_t)(i * 8192), k0 + t_k[i] < kend ? t_off[i] : t_off[i] - t_k[i] * 2u, tb);
        }
    };
    // ... and are cleared once they have landed (packed codes need not be: they meet samples that are zero)
    auto clear_tail = [&](uint32_t stage, uint32_t k0) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < T_DMA; ++i)
            if ((i < T_DMA - 1 || t_last) && k0 + t_k[i] >= kend)
                *reinterpret_cast<uint4 *>(sk_lds + stage + (8u * i + wave) * 1024u + lane * 16u) = make_uint4(0u, 0u, 0u, 0u);
        if constexpr (W16) {
#pragma unroll
            for (int i = 0; i < W_DMA; ++i)
                if (k0 + w_k[i] >= kend)
                    *reinterpret_cast<uint4 *>(sk_lds + stage + W_AT + (8u * i + wave) * 1024u + lane * 16u) = make_uint4(0u, 0u, 0u, 0u);
        }
    };

    f32x4 acc[2][ST];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int s = 0; s < ST; ++s)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[j][s][r] = 0.0f;

    // LDS addresses of this lane in stage 0: its codes, and its samples' pieces of each step of eight k
    constexpr int STEPS = KQ / 8, CW = KQ * bits / 32;      // steps, 32-bit words of codes per row tile
    const uint32_t k_lane = g * (BK / 2) + q4 * KQ;         // first k of this lane in a chunk
    uint32_t c_addr[W16 ? 2 : 1], t_addr[STEPS];
    const uint32_t wr = w * 32u + l15;                      // (row 16 further on: the same position)
#pragma unroll
    for (int p = 0; p < (W16 ? 2 : 1); ++p)
        c_addr[p] = lds0 + W_AT + wr * WROW + thin_pos<WROW>(wr, k_lane / EPL + p) * 16u + (k_lane % EPL) * bits / 8u;
#pragma unroll
    for (int e = 0; e < STEPS; ++e) t_addr[e] = lds0 + l15 * TROW + thin_pos<TROW>(l15, k_lane / 8u + e) * 16u;

    // One chunk.  LDS reads are explicit, with lgkmcnt waits: the samples of a step are asked for a step ahead, while the
    // codes of this one are unpacked (the compiler would ask for them right before the products).
    auto compute = [&](uint32_t stage) __attribute__((always_inline)) {
        u32x4 cw[2][W16 ? 2 : 1];
        u32x2 c2[2];
        u32x4 tf[2][ST];
        auto samples = [&](auto e_c) __attribute__((always_inline)) {
            constexpr int e = decltype(e_c)::value;
            static_for<ST>([&](auto s_c) __attribute__((always_inline)) {
                ds_read128<decltype(s_c)::value * 16 * TROW>(tf[e & 1][decltype(s_c)::value], t_addr[e] + stage);
            });
        };
        if constexpr (FMT == I2) {
            ds_read64<0>(c2[0], c_addr[0] + stage);
            ds_read64<16 * WROW>(c2[1], c_addr[0] + stage);
        } else {
#pragma unroll
            for (int p = 0; p < (W16 ? 2 : 1); ++p) {
                ds_read128<0>(cw[0][p], c_addr[p] + stage);
                ds_read128<16 * WROW>(cw[1][p], c_addr[p] + stage);
            }
        }
        samples(std::integral_constant<int, 0>{});
        asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(ST));
        uint32_t code[2][CW];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            if constexpr (FMT == I2) {
                asm volatile("" : "+v"(c2[j]));
                code[j][0] = c2[j].x;
                code[j][1] = c2[j].y;
            } else {
#pragma unroll
                for (int p = 0; p < (W16 ? 2 : 1); ++p) {
                    asm volatile("" : "+v"(cw[j][p]));
#pragma unroll
                    for (int x = 0; x < 4; ++x) code[j][4 * p + x] = cw[j][p][x];
                }
            }
        }
        // Codes to FP16 (as unpack_word16), in eight pieces a step of at most four vector instructions: piece k of step n takes
        // row tile k / 4.  INT2: a word is two steps, its fields are formed one step ahead.
        u32x4 wf[2][2];                                     // [step & 1][row tile]
        uint32_t fld[2][2][8];                              // [word & 1][row tile]: pairs of fields
        auto piece = [&](auto n_c, auto k_c) __attribute__((always_inline)) {
            constexpr int n = decltype(n_c)::value, j = decltype(k_c)::value >> 2, q = decltype(k_c)::value & 3;
            constexpr uint32_t LO = 0x05040100u, HI = 0x07060302u;
            if constexpr (W16) {
                wf[n & 1][j][q] = code[j][4 * n + q];
            } else if constexpr (FMT == I2) {
                constexpr int word = n >> 1;
                // the first step of a chunk forms all fields of its word, step 2 m + 1 the first half of the next word's,
                // step 2 m + 2 the second
                auto form = [&](auto w_c, auto f_c) __attribute__((always_inline)) {
                    constexpr int w2 = decltype(w_c)::value, f = decltype(f_c)::value;
                    constexpr uint32_t mask = f == 0 || f == 5 ? 0x00030003u : f == 1 || f == 6 ? 0x000C000Cu : f == 2 || f == 7 ? 0x00300030u : f == 3 ? 0x00C000C0u : 0x03000300u;
                    constexpr uint32_t bias = f == 0 || f == 5 ? 0x64026402u : f == 1 || f == 6 ? 0x5C085C08u : f == 2 || f == 7 ? 0x54205420u : f == 3 ? 0x4C804C80u : 0x46004600u;
                    const uint32_t x = f > 4 ? code[j][w2] >> 10 : code[j][w2];
                    fld[w2 & 1][j][f] = h2_sub((x & mask) ^ bias, bias);
                };
                if constexpr (n == 0) {
                    form(std::integral_constant<int, 0>{}, std::integral_constant<int, 2 * q>{});
                    form(std::integral_constant<int, 0>{}, std::integral_constant<int, 2 * q + 1>{});
                } else if constexpr (n % 2 == 0) {
                    form(std::integral_constant<int, word>{}, std::integral_constant<int, 4 + q>{});
                }
                if constexpr (n % 2 == 0) {
                    // (the fields of pair q: 2 q and 2 q + 1, both here by now)
                    constexpr int pq = q;
                    wf[0][j][pq] = __builtin_amdgcn_perm(fld[word & 1][j][2 * pq + 1], fld[word & 1][j][2 * pq], LO);
                } else {
                    wf[1][j][q] = __builtin_amdgcn_perm(fld[word & 1][j][2 * q + 1], fld[word & 1][j][2 * q], HI);
                    if constexpr (n + 1 < STEPS) form(std::integral_constant<int, word + 1>{}, std::integral_constant<int, q>{});
                }
            } else {
                // fields 0 1 | 2 3 of eight codes, then the four pairs in order
                uint32_t(&m)[8] = fld[0][j];
                if constexpr (q < 2) {
                    const uint32_t w = FMT == I8 ? code[j][2 * n + q] : q ? code[j][n] >> 8 : code[j][n];
                    if constexpr (FMT == I8) {
                        m[2 * q] = h2_sub((w & 0x00FF00FFu) ^ 0x64806480u, 0x64806480u);
                        m[2 * q + 1] = h2_sub(((w >> 8) & 0x00FF00FFu) ^ 0x64806480u, 0x64806480u);
                    } else {
                        m[2 * q] = h2_sub((w & 0x000F000Fu) ^ 0x64086408u, 0x64086408u);
                        m[2 * q + 1] = h2_sub((w & 0x00F000F0u) ^ 0x54805480u, 0x54805480u);
                    }
                } else if constexpr (FMT == I8) {
                    wf[n & 1][j][2 * (q - 2)] = __builtin_amdgcn_perm(m[2 * (q - 2) + 1], m[2 * (q - 2)], LO);
                    wf[n & 1][j][2 * (q - 2) + 1] = __builtin_amdgcn_perm(m[2 * (q - 2) + 1], m[2 * (q - 2)], HI);
                } else {
                    wf[n & 1][j][2 * (q - 2)] = __builtin_amdgcn_perm(m[1], m[0], q == 2 ? LO : HI);
                    wf[n & 1][j][2 * (q - 2) + 1] = __builtin_amdgcn_perm(m[3], m[2], q == 2 ? LO : HI);
                }
            }
        };
        static_for<8>([&](auto k_c) __attribute__((always_inline)) { piece(std::integral_constant<int, 0>{}, k_c); });
        static_for<STEPS>([&](auto e_c) __attribute__((always_inline)) {
            constexpr int e = decltype(e_c)::value;
            if constexpr (e + 1 < STEPS) samples(std::integral_constant<int, e + 1>{});
            asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(e + 1 < STEPS ? ST : 0));
#pragma unroll
            for (int s = 0; s < ST; ++s) asm volatile("" : "+v"(tf[e & 1][s]));
            __builtin_amdgcn_sched_barrier(0);
            // The next step's codes are unpacked between this one's products.  (Both waves of a SIMD do the same at the same
            // time: one after the other, the times of unpacking and products add up.)
            static_for<2 * ST>([&](auto x_c) __attribute__((always_inline)) {
                constexpr int x = decltype(x_c)::value, j = x / ST, s = x % ST;
                if constexpr (F16T) {
                    f16x8 av, bv;
                    __builtin_memcpy(&av, &wf[e & 1][j], 16);
                    __builtin_memcpy(&bv, &tf[e & 1][s], 16);
                    acc[j][s] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av, bv, acc[j][s], 0, 0, 0);
                } else {
                    bf16x8 av, bv;
                    __builtin_memcpy(&av, &wf[e & 1][j], 16);
                    __builtin_memcpy(&bv, &tf[e & 1][s], 16);
                    acc[j][s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, bv, acc[j][s], 0, 0, 0);
                }
                if constexpr (e + 1 < STEPS) {
                    constexpr int from = x * 8 / (2 * ST), to = (x + 1) * 8 / (2 * ST);
                    static_for<to - from>([&](auto d_c) __attribute__((always_inline)) {
                        piece(std::integral_constant<int, e + 1>{}, std::integral_constant<int, from + decltype(d_c)::value>{});
                    });
                    if constexpr (!W16) __builtin_amdgcn_sched_barrier(0);
                }
            });
        });
    };

    // ---- chunks ------------------------------------------------------------------
    // The c-th chunk, turned(c), sits in stage c % NSTAGE.  Loads of chunk c + NSTAGE - 1 go out behind the barrier of chunk c, which every wave
    // reaches when it is done with chunk c - 1.
    constexpr int PER = T_DMA + W_DMA;                      // loads of a wave and chunk (one less where !t_last)
#pragma unroll
    for (int c = 0; c < NSTAGE - 1; ++c)
        if ((uint32_t)c < nchunks) {
            if (c) __builtin_amdgcn_s_barrier();            // (every wave's loads of a chunk before anybody's of the next)
            load((uint32_t)(c * STAGE), turned((uint32_t)c));
        }
    uint32_t stage = 0, fill = (NSTAGE - 1) * STAGE;
    for (uint32_t c = 0; c < nchunks; ++c) {
        // chunk c has landed when only the loads of the chunks behind it are on their way (and this wave's
        // fragments of the chunk before are in registers)
        if (c + NSTAGE - 2 < nchunks) {
            if (t_last) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((NSTAGE - 2) * PER) : "memory");
            else asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((NSTAGE - 2) * (PER - 1)) : "memory");
        } else {
            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        }
        if (kbeg + (turned(c) + 1) * BK > kend) {
            clear_tail(stage, kbeg + turned(c) * BK);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        }
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (c + NSTAGE - 1 < nchunks) load(fill, turned(c + NSTAGE - 1));
        compute(stage);
        asm volatile("" ::: "memory");
        fill = stage;
        stage = stage == (NSTAGE - 1) * STAGE ? 0u : stage + STAGE;
    }
    __syncthreads();

    // ---- the two halves meet: a wave keeps row tile g and gives the other away --------
    f32x4 *const ex = reinterpret_cast<f32x4 *>(sk_lds) + (size_t)w * (2 * ST * 64) + lane;
#pragma unroll
    for (int s = 0; s < ST; ++s) ex[((g ^ 1u) * ST + s) * 64u] = g ? acc[0][s] : acc[1][s];
    __syncthreads();
    f32x4 sum[ST];
#pragma unroll
    for (int s = 0; s < ST; ++s) {
        const f32x4 other = ex[(g * ST + s) * 64u];
        sum[s] = g ? other + acc[1][s] : acc[0][s] + other;    // (first half + second half)
    }

    // lane (l15, q4): rows 4 q4 .. 4 q4 + 3 of the tile, samples l15 of each sample tile
    const uint32_t r0 = row0 + w * 32u + g * 16u + 4u * q4;
    if (r0 >= a.R) return;
    if (a.ws) {
        const bool whole = a.R % 4u == 0 && (reinterpret_cast<uintptr_t>(a.ws) & 15u) == 0;
#pragma unroll
        for (int s = 0; s < ST; ++s) {
            const uint32_t c = cbase + s * 16u + l15;
            if (c >= a.NC) continue;
            float *const dst = a.ws + ((size_t)blockIdx.y * a.NC + c) * a.R + r0;
            if (whole) {
                *reinterpret_cast<f32x4 *>(dst) = sum[s];
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (r0 + r < a.R) dst[r] = sum[s][r];
            }
        }
        return;
    }
    float bias[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) bias[r] = elem_value_rt(a.L.bias_fmt, a.L.bias, r0 + r < a.R ? r0 + r : a.R - 1u) * a.L.bscale;
    with_act(a.L.act, [&](auto act_c) __attribute__((always_inline)) {
        constexpr int ACT = decltype(act_c)::value;
#pragma unroll
        for (int s = 0; s < ST; ++s) {
            const uint32_t c = cbase + s * 16u + l15;
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (c < a.NC && r0 + r < a.R) skinny_emit_biased<F16T, ACT>(a, c, r0 + r, sum[s][r], bias[r]);
        }
    });
}

// Variant for a thin operand of at most eight rows: the NW waves of a workgroup share one tile of 32
// streamed rows and split K among themselves (wave w takes chunks w, w + NW, ...), so that a layer with many streamed
// rows needs no K split across workgroups, no partial sums in memory and no second launch.  Each wave stages its own
// thin chunks in its own LDS region (no workgroup barrier in the loop); the NW accumulator tiles meet in LDS at the
// end and are added in wave order.  Loads and their bookkeeping are those of sp_skinny16_regs.
template <int FMT, bool F16T, int NW>
__global__ __launch_bounds__(64 * NW) void sp_skinny16_kw(const SkinnyArgs a)
{
    using F = SkinnyFmt<FMT>;
    constexpr int EPL = F::EPL, LPC = F::LPC, BKC = F::BKC, STEPS = F::STEPS, PITCH = F::PITCH;
    constexpr int NCP = 8;                                 // thin rows held in LDS
    constexpr int UNITS = NCP * (BKC / 16);                // 16-code units of one thin chunk
    constexpr int UPL = (UNITS + 63) / 64;                 // units per lane
    constexpr int STAGE = NCP * PITCH;
    constexpr int NQ = NCP / 2;                            // accumulator registers per lane that belong to thin rows < NCP
    extern __shared__ __attribute__((aligned(16))) uint8_t sk_lds[];

    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);   // uniform: chunk addresses stay in scalar registers
    const uint32_t n31 = lane & 31, h = lane >> 5;
    const uint32_t K = a.L.K;
    const uint32_t r_out = blockIdx.x * 32u + n31;
    const uint32_t half = blockIdx.y / a.ksplits;
    const uint8_t *const stream = a.stream;
    const uint16_t *const thin = a.thin + (size_t)half * a.half_elems;
    const uint32_t kbeg = (blockIdx.y % a.ksplits) * a.kper;
    const uint32_t kend = kbeg + a.kper < K ? kbeg + a.kper : K;
    const uint32_t nchunks = (kend - kbeg + BKC - 1) / BKC;
    const size_t row_bytes = (size_t)K * F::bits / 8u;
    uint8_t *my_lds = sk_lds + wave * (2 * STAGE);

    const uint32_t svoff = (uint32_t)((size_t)(r_out < a.R ? r_out : a.R - 1) * row_bytes) + h * 16u;
    uint32_t tvoff[UPL][2];
    bool trow_ok[UPL];
#pragma unroll
    for (int q = 0; q < UPL; ++q) {
        const uint32_t u = (uint32_t)lane + 64u * q;
        const uint32_t row = u / (BKC / 16), uc = u % (BKC / 16);
        trow_ok[q] = u < (uint32_t)UNITS && row < a.NC;
#pragma unroll
        for (int e = 0; e < 2; ++e) tvoff[q][e] = trow_ok[q] ? (uint32_t)(((size_t)row * K + uc * 16u + 8u * e) * 2u) : 0u;
    }

    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.0f;

    // this wave's chunks: w, w + NW, ...; index i of that sequence past the end is clamped to the last one
    const uint32_t my_n = nchunks > (uint32_t)wave ? (nchunks - (uint32_t)wave + NW - 1) / NW : 0u;
    const uint32_t last_chunk = nchunks - 1;
    auto chunk_of = [&](uint32_t i) { return (uint32_t)wave + (i < my_n ? i : my_n - 1) * NW; };
    constexpr int S_LOADS = LPC, T_LOADS = UPL * 2;
    auto issue_stream = [&](uint32_t i, u32x4 (&dst)[LPC]) {
        const uint32_t ch = chunk_of(i);
        if (ch < last_chunk) {
            const uint8_t *sb = stream + (size_t)(kbeg + ch * BKC) * F::bits / 8u;
#pragma unroll
            for (int j = 0; j < LPC; ++j) {
                if (j == 0) load16_async<0>(dst[j], svoff, sb);
                else if (j == 1) load16_async<32>(dst[j], svoff, sb);
                else if (j == 2) load16_async<64>(dst[j], svoff, sb);
                else load16_async<96>(dst[j], svoff, sb);
            }
        } else {
            const uint32_t kc0 = kbeg + last_chunk * BKC;
#pragma unroll
            for (int j = 0; j < LPC; ++j) {
                const uint32_t k = kc0 + 2u * j * EPL;                 // first code of the h = 0 lane load
                const uint32_t add = k + h * EPL < K ? k * F::bits / 8u : 0u - h * 16u;
                load16_async<0>(dst[j], svoff + add, stream);
            }
        }
    };
    u32x4 thin_regs[UPL][2];
    auto issue_thin = [&](uint32_t i) {
        const uint32_t ch = chunk_of(i);
        if (ch < last_chunk) {
            const uint16_t *tb = thin + (kbeg + ch * BKC);
#pragma unroll
            for (int q = 0; q < UPL; ++q)
#pragma unroll
                for (int e = 0; e < 2; ++e) load16_async<0>(thin_regs[q][e], tvoff[q][e], tb);
        } else {
            const uint32_t kc0 = kbeg + last_chunk * BKC;
#pragma unroll
            for (int q = 0; q < UPL; ++q) {
                const uint32_t uc = ((uint32_t)lane + 64u * q) % (BKC / 16);
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const bool valid = trow_ok[q] && kc0 + uc * 16u + 8u * e + 8u <= kend;
                    load16_async<0>(thin_regs[q][e], valid ? tvoff[q][e] + kc0 * 2u : 0u, thin);
                }
            }
        }
    };
    auto store_thin = [&](int stage, uint32_t i) {
        const uint32_t kc0 = kbeg + chunk_of(i) * BKC;
#pragma unroll
        for (int q = 0; q < UPL; ++q) {
            const uint32_t u = (uint32_t)lane + 64u * q;
            if (u >= (uint32_t)UNITS) continue;
            const uint32_t row = u / (BKC / 16), uc = u % (BKC / 16);
            const uint32_t k = kc0 + uc * 16u;
            const uint32_t keep0 = (trow_ok[q] && k + 8u <= kend) ? 0xFFFFFFFFu : 0u;
            const uint32_t keep1 = (trow_ok[q] && k + 16u <= kend) ? 0xFFFFFFFFu : 0u;
            const uint32_t in[8] = {thin_regs[q][0].x & keep0, thin_regs[q][0].y & keep0, thin_regs[q][0].z & keep0,
                                    thin_regs[q][0].w & keep0, thin_regs[q][1].x & keep1, thin_regs[q][1].y & keep1,
                                    thin_regs[q][1].z & keep1, thin_regs[q][1].w & keep1};
            uint32_t o[8];
            skinny_permute_unit<FMT>(in, o);
            uint8_t *dst = my_lds + stage * STAGE + row * PITCH + uc * 32u;
            *reinterpret_cast<uint4 *>(dst) = make_uint4(o[0], o[1], o[2], o[3]);
            *reinterpret_cast<uint4 *>(dst + 16) = make_uint4(o[4], o[5], o[6], o[7]);
        }
    };
    auto compute = [&](int stage, uint32_t i, const u32x4 (&cur)[LPC]) {
        // lanes of thin rows >= NCP read a row below NCP again: their accumulator rows are never stored
        const uint8_t *sbase = my_lds + stage * STAGE + (n31 & (NCP - 1)) * PITCH + h * (EPL * 2);
        const uint32_t kc0 = kbeg + chunk_of(i) * BKC;
#pragma unroll
        for (int j = 0; j < LPC; ++j) {
            const uint32_t keep = (F::bits == 16 && kc0 + (2u * j + h) * EPL >= K) ? 0u : 0xFFFFFFFFu;
#pragma unroll
            for (int st = 0; st < STEPS; ++st) {
                const uint4 tf = *reinterpret_cast<const uint4 *>(sbase + (2 * j * EPL + 8 * st) * 2);
                uint4 v = make_uint4(cur[j].x, cur[j].y, cur[j].z, cur[j].w);
                if constexpr (F::bits == 16) { v.x &= keep; v.y &= keep; v.z &= keep; v.w &= keep; }
                uint32_t sf[4];
                skinny_frag<FMT>(v, st, sf);
                if constexpr (F16T) {
                    f16x8 af, bf;
                    __builtin_memcpy(&af, &tf, 16);
                    __builtin_memcpy(&bf, sf, 16);
                    acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(af, bf, acc, 0, 0, 0);
                } else {
                    bf16x8 af, bf;
                    __builtin_memcpy(&af, &tf, 16);
                    __builtin_memcpy(&bf, sf, 16);
                    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af, bf, acc, 0, 0, 0);
                }
            }
        }
    };
    auto pin_stream = [&](u32x4 (&r)[LPC]) {
#pragma unroll
        for (int j = 0; j < LPC; ++j) asm volatile("" : "+v"(r[j]));
    };
    auto pin_thin = [&]() {
#pragma unroll
        for (int q = 0; q < UPL; ++q)
#pragma unroll
            for (int e = 0; e < 2; ++e) asm volatile("" : "+v"(thin_regs[q][e]));
    };
    // in flight on entry: streamed chunks i (in `cur`) and i + 1; issued here: thin block i + 1, streamed chunk i + 2
    auto step = [&](uint32_t i, u32x4 (&cur)[LPC], u32x4 (&far)[LPC]) {
        const int stage = (int)(i & 1u);
        issue_thin(i + 1);
        issue_stream(i + 2, far);
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * S_LOADS + T_LOADS) : "memory");
        pin_stream(cur);
        compute(stage, i, cur);
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(S_LOADS) : "memory");
        pin_thin();
        store_thin(stage ^ 1, i + 1);
    };
    if (my_n) {
        u32x4 ra[LPC], rb[LPC], rc[LPC];
        issue_thin(0);
        issue_stream(0, ra);
        issue_stream(1, rb);
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * S_LOADS) : "memory");
        pin_thin();
        store_thin(0, 0);
        for (uint32_t i = 0; i < my_n; i += 3) {
            step(i, ra, rc);
            if (i + 1 < my_n) step(i + 1, rb, ra);
            if (i + 2 < my_n) step(i + 2, rc, rb);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the redundant tail loads
    }

    // accumulator register q of lane (n31, h): thin row 8 (q / 4) + 4 h + q % 4, streamed row n31
    float *red = reinterpret_cast<float *>(sk_lds + NW * 2 * STAGE);
#pragma unroll
    for (int q = 0; q < NQ; ++q) red[(wave * NQ + q) * 64 + lane] = acc[q];
    __syncthreads();
    if (wave != 0 || r_out >= a.R) return;
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        const uint32_t c = 8u * (q >> 2) + 4u * h + (q & 3);
        if (c >= a.NC) continue;
        float sum = 0.0f;
#pragma unroll
        for (int w = 0; w < NW; ++w) sum += red[(w * NQ + q) * 64 + lane];
        if (a.ws) a.ws[((size_t)blockIdx.y * a.NC + c) * a.R + r_out] = sum;
        else skinny_emit<F16T>(a, c, r_out, sum);
    }
}

template <bool F16T>
__device__ __forceinline__ void skinny_store(const SkinnyArgs &a, size_t o, float v)
{
    if (a.out_f32) reinterpret_cast<float *>(a.C)[o] = v;
    else if (a.halves == 2) {
        uint16_t hi, lo;
        split_f16(v, hi, lo);
        uint16_t *c = reinterpret_cast<uint16_t *>(a.C);
        c[o] = hi;
        c[(size_t)a.NC * a.R + o] = lo;               // samples x outputs elements further on
    } else reinterpret_cast<uint16_t *>(a.C)[o] = f32_to_t16<F16T>(v);
}

// Layers of at most 64 outputs (classifier heads, narrow layers): a workgroup owns 16 ST samples and all NT sixteens of outputs,
// its eight waves split K.  Nothing is staged: lane (l15, q4) loads 16 bytes of row l15 of a tile at k = 32 s + 8 q4 straight
// into registers, U steps of both operands at once and the next U while these are multiplied, and the waves' sums meet in
// LDS.  What bounds such a layer below a few thousand samples is the latency of its chain of loads, not their bytes: up to
// K = 1024 there is one round of them.  (The kernels before staged the samples of each chunk of K through LDS, a round trip
// to memory per chunk, and cut K over the grid with a second launch for more than 16 outputs.)  From a few thousand samples on the
// weights' reads from L2 count, so workgroups take more samples (ST).  A layer, conversion of its input included: 1000 x 10 at 16 /
// 256 / 8192 samples 8.3 / 8.8 / 17.0 -> 6.4 / 6.5 / 14.9 us, 4096 x 10 at 256 16.5 -> 11.9; more outputs at plan_thin.
// HALVES == 2: split activations as in sp_gemm16_small.
template <bool F16T, int NT, int ST, int HALVES>
__global__ __launch_bounds__(512) void sp_skinny16_kw_head(const SkinnyArgs a)
{
    static_assert(HALVES == 1 || F16T, "split activations are FP16");
    constexpr int NW = 8, U = NT + ST * HALVES <= 5 ? 4 : 2;
    __shared__ f32x4 part[NW][NT * ST * 64];
    __shared__ float bias_of[NT * 16];
    const uint32_t t = threadIdx.x, lane = t & 63u, l15 = lane & 15u, q4 = lane >> 4;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(t >> 6));
    const uint32_t K = a.L.K, m0 = blockIdx.x * (16u * ST);
    const uint32_t kbeg = blockIdx.y * a.kper, kend = kbeg + a.kper < K ? kbeg + a.kper : K;
    const uint32_t steps = (kend - kbeg + 31u) / 32u, per = (steps + NW - 1) / NW;
    const uint32_t s0 = wave * per, s1 = s0 + per < steps ? s0 + per : steps;

    if (t < NT * 16u && !a.ws) bias_of[t] = t < a.NC ? elem_value_rt(a.L.bias_fmt, a.L.bias, t) * a.L.bscale : 0.0f;
    const uint16_t *wp[NT], *xp[ST];
#pragma unroll
    for (int i = 0; i < NT; ++i) {
        const uint32_t n = 16u * i + l15;
        wp[i] = a.thin + (size_t)(n < a.NC ? n : a.NC - 1u) * K;
    }
#pragma unroll
    for (int j = 0; j < ST; ++j) {
        const uint32_t m = m0 + 16u * j + l15;
        xp[j] = reinterpret_cast<const uint16_t *>(a.stream) + (size_t)(m < a.R ? m : a.R - 1u) * K;
    }
    struct Frag { u32x4 w[NT], x[ST * HALVES]; };
    // (K is a multiple of eight: a piece is inside its row, or beyond K and taken for zeros)
    auto ld = [&](uint32_t s) __attribute__((always_inline)) -> Frag {
        Frag f;
        if (s >= s1) return f;                              // (a wave's last round may be short)
        const uint32_t k = kbeg + 32u * s + 8u * q4, at = k < kend ? k : 0u;
#pragma unroll
        for (int i = 0; i < NT; ++i) f.w[i] = *reinterpret_cast<const u32x4 *>(wp[i] + at);
#pragma unroll
        for (int j = 0; j < ST; ++j) {
            f.x[j] = *reinterpret_cast<const u32x4 *>(xp[j] + at);
            if constexpr (HALVES == 2) f.x[ST + j] = *reinterpret_cast<const u32x4 *>(xp[j] + a.half_elems + at);
        }
        return f;
    };
    f32x4 acc[NT][ST * HALVES];
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int j = 0; j < ST * HALVES; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    auto fma = [&](Frag &f, uint32_t s) __attribute__((always_inline)) {
        if (s >= s1) return;
        const uint32_t keep = kbeg + 32u * s + 8u * q4 < kend ? 0xFFFFFFFFu : 0u;
#pragma unroll
        for (int i = 0; i < NT; ++i) f.w[i] &= keep;
#pragma unroll
        for (int j = 0; j < ST * HALVES; ++j) {
            f.x[j] &= keep;
#pragma unroll
            for (int i = 0; i < NT; ++i) {
                if constexpr (F16T) {
                    f16x8 av, bv;
                    __builtin_memcpy(&av, &f.w[i], 16);
                    __builtin_memcpy(&bv, &f.x[j], 16);
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av, bv, acc[i][j], 0, 0, 0);
                } else {
                    bf16x8 av, bv;
                    __builtin_memcpy(&av, &f.w[i], 16);
                    __builtin_memcpy(&bv, &f.x[j], 16);
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, bv, acc[i][j], 0, 0, 0);
                }
            }
        }
    };
    if (s0 < s1) {
        Frag cur[U];
#pragma unroll
        for (int u = 0; u < U; ++u) cur[u] = ld(s0 + u);
        uint32_t s = s0;
        for (; s + U < s1; s += U) {
            Frag next[U];
#pragma unroll
            for (int u = 0; u < U; ++u) next[u] = ld(s + U + u);
#pragma unroll
            for (int u = 0; u < U; ++u) fma(cur[u], s + u);
#pragma unroll
            for (int u = 0; u < U; ++u) cur[u] = next[u];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) fma(cur[u], s + u);
    }
#pragma unroll
    for (int j = 0; j < ST; ++j)
#pragma unroll
        for (int i = 0; i < NT; ++i) {
            f32x4 v = acc[i][j];
            if constexpr (HALVES == 2)
#pragma unroll
                for (int r = 0; r < 4; ++r) v[r] = fmaf(acc[i][ST + j][r], kLoScale, v[r]);
            part[wave][(j * NT + i) * 64 + lane] = v;
        }
    __syncthreads();

    // lane (l15, q4) of a tile: outputs 16 i + 4 q4 .. + 3 of sample 16 j + l15; the waves' sums in wave order
    for (uint32_t slot = t; slot < NT * ST * 64u; slot += 64u * NW) {
        f32x4 z = part[0][slot];
#pragma unroll
        for (int w = 1; w < NW; ++w) z += part[w][slot];
        if (a.soft_out) {
            part[0][slot] = z;
            continue;
        }
        const uint32_t tile = slot >> 6, m = m0 + 16u * (tile / NT) + l15, n0 = 16u * (tile % NT) + 4u * q4;
        if (m >= a.R) continue;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const uint32_t n = n0 + r;
            if (n >= a.NC) continue;
            if (a.ws) a.ws[((size_t)blockIdx.y * a.NC + n) * a.R + m] = z[r];
            else skinny_store<F16T>(a, (size_t)m * a.L.N + n, apply_act(layer_sum(a.L, z[r], bias_of[n], n), a.L.act));
        }
    }
    if (a.soft_out) {
        // softmax as Activation.c:5-21 (largest logit subtracted, exponentials, one division by their sum), a wave per tile
        __syncthreads();
        if (wave >= (uint32_t)ST) return;
        const uint32_t m = m0 + 16u * wave + l15;
        float v[NT][4], top = -3.402823466e+38f, s = 0.0f;
#pragma unroll
        for (int i = 0; i < NT; ++i) {
            const f32x4 z = part[0][(wave * NT + i) * 64u + lane];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const uint32_t n = 16u * i + 4u * q4 + r;
                v[i][r] = n < a.NC ? fmaf(z[r], a.L.wscale, bias_of[n]) : -3.402823466e+38f;
                top = fmaxf(top, v[i][r]);
            }
        }
        top = fmaxf(top, __shfl_xor(top, 16));
        top = fmaxf(top, __shfl_xor(top, 32));
#pragma unroll
        for (int i = 0; i < NT; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                v[i][r] = 16u * i + 4u * q4 + r < a.NC ? expf(v[i][r] - top) : 0.0f;
                s += v[i][r];
            }
        s += __shfl_xor(s, 16);
        s += __shfl_xor(s, 32);
        const float inv = s > 0.0f ? 1.0f / s : 1.0f;
        if (m >= a.R) return;
#pragma unroll
        for (int i = 0; i < NT; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const uint32_t n = 16u * i + 4u * q4 + r;
                if (n >= a.NC) continue;
                const size_t o = (size_t)m * a.L.N + n;
                const float y = v[i][r] * inv;
                if (a.soft_kind == 0) reinterpret_cast<float *>(a.soft_out)[o] = y;
                else if (a.soft_kind == 1) reinterpret_cast<uint16_t *>(a.soft_out)[o] = f32_to_bf16_rne(y);
                else reinterpret_cast<uint16_t *>(a.soft_out)[o] = f32_to_f16_sat(y);
            }
    }
}

// adds the partial sums of sp_skinny16 (K splits in split order; with split activations the sums of the second matrix,
// scaled by 2^-11, after those of the first) and applies bias and activation; a thread takes four neighbouring
// streamed rows (VEC: R is a multiple of four and the rows are outputs, so they are neighbours in C as well) or one
template <bool F16T, bool VEC>
__global__ __launch_bounds__(256) void sp_skinny_reduce(const SkinnyArgs a, uint32_t splits)
{
    const uint64_t total = (uint64_t)a.NC * a.R;
    const uint32_t parts = a.parts;
    if constexpr (VEC) {
        const uint64_t idx = ((uint64_t)blockIdx.x * 256u + threadIdx.x) * 4u;
        if (idx >= total) return;
        const uint32_t c = (uint32_t)(idx / a.R), r = (uint32_t)(idx % a.R);
        float bias[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) bias[i] = elem_value_rt(a.L.bias_fmt, a.L.bias, r + i) * a.L.bscale;
        float4 sum, low;
        add_parts(reinterpret_cast<const float4 *>(a.ws + idx), total / 4u, splits, parts, sum, low);
        const float in[4] = {fmaf(low.x, kLoScale, sum.x), fmaf(low.y, kLoScale, sum.y), fmaf(low.z, kLoScale, sum.z),
                             fmaf(low.w, kLoScale, sum.w)};
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            v[i] = apply_act(layer_sum(a.L, in[i], bias[i], r + i), a.L.act);
        }
        const size_t o = (size_t)c * a.L.N + r;
        if (a.out_f32) {
            *reinterpret_cast<float4 *>(reinterpret_cast<float *>(a.C) + o) = make_float4(v[0], v[1], v[2], v[3]);
        } else if (a.halves == 2) {
            uint16_t hi[4], lo[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) split_f16(v[i], hi[i], lo[i]);
            uint16_t *cc = reinterpret_cast<uint16_t *>(a.C);
            *reinterpret_cast<uint2 *>(cc + o) = make_uint2((uint32_t)hi[0] | ((uint32_t)hi[1] << 16), (uint32_t)hi[2] | ((uint32_t)hi[3] << 16));
            *reinterpret_cast<uint2 *>(cc + total + o) = make_uint2((uint32_t)lo[0] | ((uint32_t)lo[1] << 16), (uint32_t)lo[2] | ((uint32_t)lo[3] << 16));
        } else {
            const uint32_t lo = (uint32_t)f32_to_t16<F16T>(v[0]) | ((uint32_t)f32_to_t16<F16T>(v[1]) << 16);
            const uint32_t hi = (uint32_t)f32_to_t16<F16T>(v[2]) | ((uint32_t)f32_to_t16<F16T>(v[3]) << 16);
            *reinterpret_cast<uint2 *>(reinterpret_cast<uint16_t *>(a.C) + o) = make_uint2(lo, hi);
        }
    } else {
        const uint64_t idx = (uint64_t)blockIdx.x * 256u + threadIdx.x;
        if (idx >= total) return;
        float sum = 0.0f, low = 0.0f;
        for (uint32_t sp = 0; sp < parts; ++sp) {
            const float v = a.ws[(uint64_t)sp * total + idx];
            if (sp < splits) sum += v; else low += v;
        }
        const uint32_t c = (uint32_t)(idx / a.R), r = (uint32_t)(idx % a.R);
        const uint32_t m = a.mode_b ? r : c, n = a.mode_b ? c : r;
        const float bias = elem_value_rt(a.L.bias_fmt, a.L.bias, n) * a.L.bscale;
        skinny_store<F16T>(a, (size_t)m * a.L.N + n, apply_act(layer_sum(a.L, fmaf(low, kLoScale, sum), bias, n), a.L.act));
    }
}

// unscaled integer codes of a small weight array as FP16 (the thin operand of a layer with few outputs)
template <int FMT>
__global__ __launch_bounds__(256) void sp_codes16(const uint8_t *__restrict__ codes, uint16_t *__restrict__ out, uint64_t n)
{
    const uint64_t i = (uint64_t)blockIdx.x * 256u + threadIdx.x;
    if (i < n) out[i] = f32_to_f16_sat(elem_value<FMT>(codes, i));
}
