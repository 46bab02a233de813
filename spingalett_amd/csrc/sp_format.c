/*
 * sp_format.c — the versioned .nn container: array codecs, load, save.
 *
 * File layout (Serialize.c:348-407, little-endian, no padding):
 *   u16 version=1 | u32 layers | u8 loss | u8 has_optimizer | [u64 time_step]
 *   | u8 precision | u32 topology[L] | u8 activation[L-1]
 *   then per layer:  W [mW vW]  b [mb vb]      (bracketed only with optimizer)
 * Array encodings (Serialize.c:87-193): FP32 raw; FP16/BF16 u16 codes;
 *   INT8 f32 max + i8[n]; INT4 f32 max + packed nibbles (even index low);
 *   INT2 f32 max + packed 2-bit fields (index i at bits 2(i%4)).
 *
 * Unlike the reference loader this one keeps the file's bytes: the device is
 * fed the packed arrays, the public FP32 arrays are filled for API
 * compatibility.  Compile without fast-math: the decode expressions are
 * meant to be evaluated exactly as written.
 */
#define _GNU_SOURCE
#include "sp_internal.h"

#include <fcntl.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <sys/stat.h>
#include <unistd.h>

static inline uint32_t f2u(float x) { uint32_t u; memcpy(&u, &x, 4); return u; }
static inline float    u2f(uint32_t u) { float x; memcpy(&x, &u, 4); return x; }

/* ------------------------------------------------------------------ */
/* array codecs                                                        */
/*                                                                     */
/* A net's arrays are a few megabytes of elementwise work: memory, not */
/* arithmetic, should decide.  Conversions are written without         */
/* branches so that the loops become vector code, each loop exists for */
/* the baseline instruction set and for AVX2 (chosen at run time), and */
/* long arrays are shared out among a few threads.  On an EPYC, saving */
/* 925 K weights as INT8 / INT4 went from 2.8 / 8.8 ms to 0.2 / 0.2    */
/* (half of it the file), loading them from 0.58 / 0.60 to 0.13 / 0.15 */
/* ms; 7 M weights as INT8 18 -> 1.3 and 4.6 -> 1.0 ms.                */
/* ------------------------------------------------------------------ */
#define SP_INLINE static inline __attribute__((always_inline))

/* half -> single, exact; NaNs lose their payload (Serialize.c:45-72) */
SP_INLINE float half_to_float(uint16_t h)
{
    const uint32_t sign = (uint32_t)(h & 0x8000u) << 16, mag = h & 0x7FFFu;
    const uint32_t normal = (mag << 13) + 0x38000000u;                        /* exponent 15 -> 127 */
    const uint32_t tiny = f2u((float)(int32_t)mag * 0x1p-24f);                /* subnormals and zero: exact */
    const uint32_t special = mag > 0x7C00u ? 0x7FC00000u : 0x7F800000u;
    uint32_t r = mag < 0x400u ? tiny : normal;
    r = mag >= 0x7C00u ? special : r;
    return u2f(sign | r);
}

/* single -> half by truncation (Serialize.c:12-43) */
SP_INLINE uint16_t float_to_half_trunc(float x)
{
    const uint32_t u = f2u(x), sign = (u >> 16) & 0x8000u, mag = u & 0x7FFFFFFFu;
    const uint32_t normal = (mag - 0x38000000u) >> 13;                        /* exponent 127 -> 15 */
    /* 2^-24 up to 2^-14: the leading one joins the fraction, shifted by 14 to 23 (other magnitudes take another r) */
    const uint32_t tiny = ((mag & 0x7FFFFFu) | 0x800000u) >> ((126u - (mag >> 23)) & 31u);
    uint32_t r = mag < 0x38800000u ? tiny : normal;
    r = mag < 0x33800000u ? 0u : r;                                           /* below 2^-24, FP32 subnormals */
    r = mag >= 0x47800000u ? 0x7C00u : r;                                     /* 2^16 and above, infinities */
    r = mag > 0x7F800000u ? 0x7E00u : r;
    return (uint16_t)(sign | r);
}

/* roundf() (halves away from zero) of a small magnitude as an integer; a NaN (an infinity over an infinite scale)
 * becomes 0 */
SP_INLINE int32_t round_to_int(float x)
{
    const float v = x == x ? x : 0.0f;
    const int32_t t = (int32_t)v;
    const float rest = v - (float)t;                                          /* exact */
    return t + (rest >= 0.5f ? 1 : 0) - (rest <= -0.5f ? 1 : 0);
}

/* Elements [begin, end) of one array; begin is a multiple of 64 (whole code bytes), max_val > 0 for the integer formats. */
typedef struct {
    const void *src;
    void *dst;
    PrecisionMode p;
    bool release;              /* SPINGALETT_DEQUANT_RELEASE */
    float max_val;
    uint32_t part_max[SP_MAX_THREADS];
} codec_job;

SP_INLINE uint32_t absmax_range(const codec_job *j, size_t begin, size_t end)
{
    const float *src = (const float *)j->src;
    uint32_t top = 0;                                    /* magnitudes order like their bit patterns; NaNs count as 0 */
    for (size_t i = begin; i < end; ++i) {
        const uint32_t mag = f2u(src[i]) & 0x7FFFFFFFu;
        const uint32_t v = mag > 0x7F800000u ? 0u : mag;
        top = v > top ? v : top;
    }
    return top;
}

/* Serialize.c:87-193.  Codes of less than a byte are made one per byte for a block that stays in the first cache, then
 * packed: two vector loops instead of one scalar one. */
#define PACK_BLOCK 1024u
SP_INLINE void encode_range(const codec_job *j, size_t begin, size_t end)
{
    const float *restrict src = (const float *)j->src;
    uint8_t *restrict codes = (uint8_t *)j->dst;
    const float max_val = j->max_val;
    size_t i = begin;
    switch (j->p) {
    case PRECISION_FP16: {
        for (; i < end; ++i) { const uint16_t h = float_to_half_trunc(src[i]); memcpy(codes + 2u * i, &h, 2); }
        break;
    }
    case PRECISION_BFLOAT16:
        for (; i < end; ++i) { const uint16_t h = (uint16_t)(f2u(src[i]) >> 16); memcpy(codes + 2u * i, &h, 2); }
        break;
    case PRECISION_INT8:
        for (; i < end; ++i) codes[i] = (uint8_t)round_to_int(src[i] / max_val * 127.0f);
        break;
    case PRECISION_INT4:                                 /* |ratio| <= 1: the codes are -7 .. 7 as they are */
        while (i < end) {
            uint8_t q[PACK_BLOCK + 1];
            const size_t m = end - i < PACK_BLOCK ? end - i : PACK_BLOCK;
            for (size_t k = 0; k < m; ++k) q[k] = (uint8_t)round_to_int(src[i + k] / max_val * 7.0f);
            q[m] = 0;
            for (size_t k = 0; k < (m + 1u) / 2u; ++k) codes[i / 2u + k] = (uint8_t)((q[2u * k] & 15u) | q[2u * k + 1u] << 4);
            i += m;
        }
        break;
    default:
        while (i < end) {
            uint8_t q[PACK_BLOCK + 3];
            const size_t m = end - i < PACK_BLOCK ? end - i : PACK_BLOCK;
            for (size_t k = 0; k < m; ++k) {
                const float ratio = src[i + k] / max_val;
                q[k] = (uint8_t)((ratio > 0.5f ? 1 : 0) | (ratio < -0.5f ? 3 : 0));
            }
            q[m] = q[m + 1u] = q[m + 2u] = 0;
            for (size_t k = 0; k < (m + 3u) / 4u; ++k)
                codes[i / 4u + k] = (uint8_t)(q[4u * k] | q[4u * k + 1u] << 2 | q[4u * k + 2u] << 4 | q[4u * k + 3u] << 6);
            i += m;
        }
        break;
    }
}

/* Serialize.c:195-297.  The integer formats: strict fl(fl(q / d) max), release fl(q fl(max fl(1/d))). */
SP_INLINE void decode_range(const codec_job *j, size_t begin, size_t end)
{
    const uint8_t *restrict codes = (const uint8_t *)j->src;
    float *restrict dst = (float *)j->dst;
    const size_t whole = begin + (end - begin) / 4u * 4u;
    size_t i = begin;
    if (j->p == PRECISION_FP16) {
        for (; i < end; ++i) { uint16_t h; memcpy(&h, codes + 2u * i, 2); dst[i] = half_to_float(h); }
        return;
    }
    if (j->p == PRECISION_BFLOAT16) {
        for (; i < end; ++i) { uint16_t h; memcpy(&h, codes + 2u * i, 2); dst[i] = u2f((uint32_t)h << 16); }
        return;
    }
    /* q / div * mul covers all of them: div = d, mul = max (strict); div = 1, mul = max fl(1/d) (release; INT2's d is 1) */
    const float d = j->p == PRECISION_INT8 ? 127.0f : j->p == PRECISION_INT4 ? 7.0f : 1.0f;
    const float recip = 1.0f / d;
    const float div = j->release ? 1.0f : d, mul = j->release ? j->max_val * recip : j->max_val;
    if (j->p == PRECISION_INT8) {
        for (; i < end; ++i) dst[i] = (float)(int8_t)codes[i] / div * mul;
    } else if (j->p == PRECISION_INT4) {
        while (i < end) {
            int8_t q[PACK_BLOCK + 1];
            const size_t m = end - i < PACK_BLOCK ? end - i : PACK_BLOCK;
            for (size_t k = 0; k < (m + 1u) / 2u; ++k) {
                const uint8_t c = codes[i / 2u + k];
                q[2u * k] = (int8_t)(((c & 15u) ^ 8u) - 8u);
                q[2u * k + 1u] = (int8_t)(((c >> 4) ^ 8u) - 8u);
            }
            for (size_t k = 0; k < m; ++k) dst[i + k] = (float)q[k] / div * mul;
            i += m;
        }
    } else {
        for (; i < whole; i += 4u) {
            const int32_t c = codes[i / 4u];
            dst[i] = (float)(((c & 3) ^ 2) - 2) * mul;
            dst[i + 1] = (float)(((c >> 2 & 3) ^ 2) - 2) * mul;
            dst[i + 2] = (float)(((c >> 4 & 3) ^ 2) - 2) * mul;
            dst[i + 3] = (float)(((c >> 6 & 3) ^ 2) - 2) * mul;
        }
        for (; i < end; ++i) dst[i] = (float)(((codes[i / 4u] >> 2u * (i & 3u) & 3) ^ 2) - 2) * mul;
    }
}

#if defined(__x86_64__)
__attribute__((target("avx2"))) static uint32_t absmax_avx2(const codec_job *j, size_t b, size_t e) { return absmax_range(j, b, e); }
__attribute__((target("avx2"))) static void encode_avx2(const codec_job *j, size_t b, size_t e) { encode_range(j, b, e); }
__attribute__((target("avx2"))) static void decode_avx2(const codec_job *j, size_t b, size_t e) { decode_range(j, b, e); }
static bool have_avx2(void) { return __builtin_cpu_supports("avx2"); }
#else
#define absmax_avx2 absmax_range
#define encode_avx2 encode_range
#define decode_avx2 decode_range
static bool have_avx2(void) { return false; }
#endif

static void absmax_part(void *ctx, unsigned part, size_t begin, size_t end)
{
    codec_job *j = (codec_job *)ctx;
    j->part_max[part] = have_avx2() ? absmax_avx2(j, begin, end) : absmax_range(j, begin, end);
}

static void encode_part(void *ctx, unsigned part, size_t begin, size_t end)
{
    (void)part;
    if (have_avx2()) encode_avx2((codec_job *)ctx, begin, end); else encode_range((codec_job *)ctx, begin, end);
}

static void decode_part(void *ctx, unsigned part, size_t begin, size_t end)
{
    codec_job *j = (codec_job *)ctx;
    (void)part;
    if (j->p == PRECISION_FLOAT32) memcpy((float *)j->dst + begin, (const uint8_t *)j->src + 4u * begin, 4u * (end - begin));
    else if (j->p >= PRECISION_INT8 && !(j->max_val > 0.0f)) memset((float *)j->dst + begin, 0, 4u * (end - begin));   /* 0, negative or NaN scale */
    else if (have_avx2()) decode_avx2(j, begin, end);
    else decode_range(j, begin, end);
}

size_t sp_array_bytes(uint64_t n, PrecisionMode p)
{
    switch (p) {
    case PRECISION_FLOAT32:  return (size_t)(n * 4u);
    case PRECISION_FP16:
    case PRECISION_BFLOAT16: return (size_t)(n * 2u);
    case PRECISION_INT8:     return (size_t)(4u + n);
    case PRECISION_INT4:     return (size_t)(4u + (n + 1u) / 2u);
    case PRECISION_INT2:     return (size_t)(4u + (n + 3u) / 4u);
    default:                 return 0;
    }
}

bool sp_decode_array(const uint8_t *src, size_t avail, uint32_t n, PrecisionMode p,
                     SpingalettDequantMode mode, float *dst)
{
    if (avail < sp_array_bytes(n, p)) return false;
    codec_job j = {.src = src, .dst = dst, .p = p, .release = mode == SPINGALETT_DEQUANT_RELEASE};
    if (p >= PRECISION_INT8) {
        memcpy(&j.max_val, src, 4);
        j.src = src + 4;
    }
    sp_parallel(n, decode_part, &j);
    return true;
}

/* largest magnitude of an array (the scale of the integer formats, Serialize.c:118-123) */
static float array_absmax(const float *src, uint32_t n)
{
    codec_job j = {.src = src};
    uint32_t top = 0;
    sp_parallel(n, absmax_part, &j);
    for (unsigned t = 0; t < SP_MAX_THREADS; ++t) top = j.part_max[t] > top ? j.part_max[t] : top;
    return u2f(top);
}

/* the codes of n elements (the caller writes the scale); `n` elements starting at a multiple of 64 of the array */
static void encode_codes(const float *src, uint32_t n, PrecisionMode p, float max_val, uint8_t *codes)
{
    codec_job j = {.src = src, .dst = codes, .p = p, .max_val = max_val};
    if (p >= PRECISION_INT8 && !(max_val > 0.0f)) memset(codes, 0, sp_array_bytes(n, p) - 4u);
    else sp_parallel(n, encode_part, &j);
}

void sp_drop_packed(sp_net *sn)
{
    free(sn->file_blob);
    free(sn->packed_w);
    free(sn->packed_b);
    sn->file_blob = NULL;
    sn->file_bytes = 0;
    sn->packed_w = sn->packed_b = NULL;
    sn->packed_precision = PRECISION_FLOAT32;
}

/* ------------------------------------------------------------------ */
/* load                                                                */
/* ------------------------------------------------------------------ */

typedef struct { const uint8_t *p; size_t left; } cursor;

static bool take(cursor *c, void *dst, size_t n)
{
    if (c->left < n) return false;
    memcpy(dst, c->p, n);
    c->p += n;
    c->left -= n;
    return true;
}

/* Reads one array into dst; fills `keep` (may be NULL) with where its codes sit.
 * A short FP32 array keeps its leading whole values (fread semantics at
 * Serialize.c:197); other formats decode nothing when short (:203-208). */
static bool read_array(cursor *c, uint32_t n, PrecisionMode p, SpingalettDequantMode mode,
                       float *dst, sp_packed_array *keep)
{
    const size_t need = sp_array_bytes(n, p);
    if (c->left < need) {
        if (p == PRECISION_FLOAT32) memcpy(dst, c->p, c->left & ~(size_t)3u);
        c->p += c->left;
        c->left = 0;
        return false;
    }
    sp_decode_array(c->p, c->left, n, p, mode, dst);
    if (keep) {
        const bool scaled = p >= PRECISION_INT8;
        keep->codes = c->p + (scaled ? 4 : 0);
        keep->bytes = need - (scaled ? 4u : 0u);
        keep->max_val = 0.0f;
        if (scaled) memcpy(&keep->max_val, c->p, 4);
    }
    c->p += need;
    c->left -= need;
    return true;
}

/* Takes ownership of blob (freed on failure). */
static NeuralNetwork *load_from_blob(uint8_t *blob, size_t bytes, const char *label)
{
    cursor c = {blob, bytes};
#define FAIL(msg) do { sp_set_error(SPINGALETT_ERR_INVALID, msg); free(blob); return NULL; } while (0)
    uint16_t version = 0;
    if (!take(&c, &version, 2)) FAIL("load: failed to read format version");
    if (version != SPINGALETT_FORMAT_VERSION) {
        sp_log(LOG_ERROR, "Unsupported file format version %u (expected %u)", (unsigned)version,
               (unsigned)SPINGALETT_FORMAT_VERSION);
        FAIL("load: unsupported format version");
    }
    uint32_t layers = 0;
    if (!take(&c, &layers, 4)) FAIL("load: failed to read layer count");
    if (layers < 2) FAIL("load: network must have at least 2 layers");
    uint8_t loss = 0, has_opt = 0, prec = 0;
    if (!take(&c, &loss, 1) || loss >= LOSS_COUNT) FAIL("load: invalid loss type");
    if (!take(&c, &has_opt, 1)) FAIL("load: failed to read optimizer flag");
    uint64_t time_step = 0;
    if (has_opt && !take(&c, &time_step, 8)) FAIL("load: failed to read time step");
    if (!take(&c, &prec, 1) || prec >= PRECISION_COUNT) FAIL("load: invalid precision type");
    if (c.left / 4u < layers) FAIL("load: failed to read topology");
    const uint8_t *topo_raw = c.p;                    /* unaligned in the file: copied, never read in place */
    uint32_t *topology = (uint32_t *)malloc((size_t)layers * 4u);
    uint8_t *acts = (uint8_t *)malloc(layers - 1);
    if (!topology || !acts) {
        free(topology); free(acts); free(blob);
        sp_set_error(SPINGALETT_ERR_ALLOC, "load: topology allocation failed");
        return NULL;
    }
    memcpy(topology, topo_raw, (size_t)layers * 4u);
    c.p += (size_t)layers * 4u;
    c.left -= (size_t)layers * 4u;
    bool bad = false;
    for (uint32_t i = 0; i + 1 < layers && !bad; ++i)
        if (!take(&c, &acts[i], 1) || acts[i] >= ACT_COUNT) bad = true;
    for (uint32_t l = 0; l < layers && !bad; ++l) {
        if (topology[l] == 0) bad = true;                /* layer() rejects empty layers (Network.c:53) */
        if (l && (uint64_t)topology[l - 1] * topology[l] > 0xFFFFFFFFull) bad = true;
    }
    if (bad) {
        free(topology); free(acts);
        FAIL("load: invalid activation function or layer size");
    }
#undef FAIL

    /* The reference builds the net with layer() and then tests the sticky error
     * slot without clearing it first (Serialize.c:556): an error left over from
     * an earlier call makes the load fail.  Kept, since callers may rely on it. */
    if (spingalett_last_error_code() != SPINGALETT_OK) {
        free(topology); free(acts); free(blob);
        return NULL;
    }
    NeuralNetwork *net = sp_net_build((LossFunction)loss, layers, topology, acts);
    free(topology);
    free(acts);
    if (!net) {
        free(blob);
        sp_set_error(SPINGALETT_ERR_ALLOC, "load: network creation failed");
        return NULL;
    }
    net->time_step = time_step;
    sp_net *sn = sp_owned(net);           /* sp_net_build() just made it */
    sn->packed_w = (sp_packed_array *)calloc(layers - 1, sizeof(sp_packed_array));
    sn->packed_b = (sp_packed_array *)calloc(layers - 1, sizeof(sp_packed_array));
    if (!sn->packed_w || !sn->packed_b) {
        free(blob);
        free_network(net);
        sp_set_error(SPINGALETT_ERR_ALLOC, "load: descriptor allocation failed");
        return NULL;
    }
    sn->file_blob = blob;
    sn->file_bytes = bytes;
    sn->packed_precision = (PrecisionMode)prec;
    sn->opt_loaded = has_opt != 0;

    const SpingalettDequantMode mode = spingalett_get_dequant_mode();
    const PrecisionMode p = (PrecisionMode)prec;
    bool ok = true;
    for (uint32_t l = 0; l + 1 < layers && ok; ++l) {
        const uint32_t wcount = net->topology[l] * net->topology[l + 1], bcount = net->topology[l + 1];
        const uint64_t wo = net->weight_offsets[l], bo = net->bias_offsets[l];
        ok = read_array(&c, wcount, p, mode, net->weights + wo, &sn->packed_w[l]);
        if (ok && has_opt)
            ok = read_array(&c, wcount, p, mode, net->opt_m_weights + wo, NULL)
              && read_array(&c, wcount, p, mode, net->opt_v_weights + wo, NULL);
        if (ok) ok = read_array(&c, bcount, p, mode, net->biases + bo, &sn->packed_b[l]);
        if (ok && has_opt)
            ok = read_array(&c, bcount, p, mode, net->opt_m_biases + bo, NULL)
              && read_array(&c, bcount, p, mode, net->opt_v_biases + bo, NULL);
    }
    if (!ok) {                                   /* Serialize.c:596-599: the net is still returned */
        sp_set_error(SPINGALETT_ERR_INVALID, "load: file appears truncated or corrupt");
        sp_log(LOG_WARNING, "Network file may be truncated: %s", label);
        sp_drop_packed(sn);                      /* incomplete: the device will be fed the FP32 arrays */
    }
    sp_log(LOG_INFO, "Network loaded from %s", label);
    sp_log(LOG_INFO, "Load info: format=v%u, layers=%u, weights=%llu, biases=%llu, precision=%s, optimizer=%s",
           (unsigned)version, layers, (unsigned long long)net->total_weights, (unsigned long long)net->total_biases,
           sp_precision_names[prec], has_opt ? "ON" : "OFF");
    return net;
}

NeuralNetwork *load_spingalett(const char *filename)
{
    if (!filename) {
        sp_set_error(SPINGALETT_ERR_INVALID, "load: filename is NULL");
        return NULL;
    }
    FILE *fp = fopen(filename, "rb");
    if (!fp) {
        sp_set_error(SPINGALETT_ERR_INVALID, "load: cannot open file for reading");
        return NULL;
    }
    size_t cap = 1u << 16, len = 0;
    if (fseek(fp, 0, SEEK_END) == 0) {
        const long end = ftell(fp);
        if (end > 0) cap = (size_t)end + 1u;                  /* a whole file leaves room: the loop below ends */
        rewind(fp);
    }
    uint8_t *blob = (uint8_t *)malloc(cap ? cap : 1);
    while (blob) {
        const size_t got = fread(blob + len, 1, cap - len, fp);
        len += got;
        if (len < cap || got == 0) break;
        uint8_t *bigger = (uint8_t *)realloc(blob, cap * 2);   /* unseekable stream */
        if (!bigger) { free(blob); blob = NULL; break; }
        blob = bigger;
        cap *= 2;
    }
    fclose(fp);
    if (!blob) {
        sp_set_error(SPINGALETT_ERR_ALLOC, "load: file buffer allocation failed");
        return NULL;
    }
    return load_from_blob(blob, len, filename);
}

NeuralNetwork *load_spingalett_memory(const void *data, size_t bytes)
{
    if (!data) {
        sp_set_error(SPINGALETT_ERR_INVALID, "load: data is NULL");
        return NULL;
    }
    uint8_t *blob = (uint8_t *)malloc(bytes ? bytes : 1);
    if (!blob) {
        sp_set_error(SPINGALETT_ERR_ALLOC, "load: file buffer allocation failed");
        return NULL;
    }
    memcpy(blob, data, bytes);
    return load_from_blob(blob, bytes, "<memory>");
}

/* ------------------------------------------------------------------ */
/* save (Serialize.c:307-424)                                          */
/* ------------------------------------------------------------------ */

/* Codes are made and written in pieces of at most this many elements, so that a piece is still in the caches when it
 * is handed to the file. */
#define WRITE_PIECE (1u << 20)

static bool write_array(FILE *fp, const float *src, uint32_t n, PrecisionMode p, uint8_t **scratch)
{
    if (p == PRECISION_FLOAT32) return fwrite(src, sizeof(float), n, fp) == n;
    if (!*scratch) *scratch = (uint8_t *)malloc(2u * WRITE_PIECE);
    if (!*scratch) { sp_set_error(SPINGALETT_ERR_ALLOC, "save: write buffer allocation failed"); return false; }
    float max_val = 0.0f;
    const size_t scale = p >= PRECISION_INT8 ? 4u : 0u;
    if (scale) {
        max_val = array_absmax(src, n);
        if (fwrite(&max_val, 4, 1, fp) != 1) return false;
    }
    for (size_t i = 0; i < n; i += WRITE_PIECE) {
        const uint32_t m = n - i < WRITE_PIECE ? (uint32_t)(n - i) : WRITE_PIECE;
        const size_t bytes = sp_array_bytes(m, p) - scale;
        encode_codes(src + i, m, p, max_val, *scratch);
        if (fwrite(*scratch, 1, bytes, fp) != bytes) return false;
    }
    return true;
}

/* A file that exists is written over and cut to its new length at the end (also after a failed write), instead of being
 * emptied first: giving up its cached pages, many of them still waiting for the disk, and making as many new ones cost
 * more than writing them (a 3.7 MB file saved again and again: 1.0 ms to empty it, 0.2 ms to write it).  Until it has its
 * length such a file has new arrays in front of old ones, which nothing else would tell from a whole file: its version is
 * zero while it is written, which every loader refuses, and comes last (*held: it does). */
static FILE *open_for_overwrite(const char *name, bool *held)
{
    struct stat st;
    const int fd = open(name, O_WRONLY | O_CREAT | O_CLOEXEC, 0666);
    FILE *fp = fd >= 0 ? fdopen(fd, "wb") : NULL;
    if (fd >= 0 && !fp) close(fd);
    *held = fp && fstat(fd, &st) == 0 && S_ISREG(st.st_mode) && st.st_size > 0;
    return fp;
}

static bool close_at_length(FILE *fp, bool held)
{
    static const uint16_t version = SPINGALETT_FORMAT_VERSION;
    struct stat st;
    bool ok = fflush(fp) == 0;
    if (fstat(fileno(fp), &st) == 0 && S_ISREG(st.st_mode)) {
        const off_t end = ftello(fp);
        bool cut = end >= 0;
        if (cut && end < st.st_size) cut = ftruncate(fileno(fp), end) == 0;
        if (held && (!cut || end < 2 || pwrite(fileno(fp), &version, 2, 0) != 2)) cut = false;
        ok = ok && cut;
    }
    return fclose(fp) == 0 && ok;
}

void save_spingalett_struct_arguments(SaveArgs args)
{
    if (!args.net || !args.filename) {
        sp_set_error(SPINGALETT_ERR_INVALID, "save: net or filename is NULL");
        return;
    }
    if ((unsigned)args.precision >= PRECISION_COUNT) {
        sp_set_error(SPINGALETT_ERR_INVALID, "save: invalid precision mode");
        return;
    }
    /* ".nn" is appended when the last path component has no dot (Serialize.c:321-336) */
    const char *name = args.filename;
    const char *slash = strrchr(name, '/'), *bslash = strrchr(name, '\\');
    const char *sep = (slash && bslash) ? (slash > bslash ? slash : bslash) : (slash ? slash : bslash);
    const char *dot = strrchr(name, '.');
    char *owned = NULL;
    if (!(dot && (!sep || dot > sep))) {
        owned = (char *)malloc(strlen(name) + 4);
        if (!owned) { sp_set_error(SPINGALETT_ERR_ALLOC, "save: filename allocation failed"); return; }
        sprintf(owned, "%s.nn", name);
        name = owned;
    }
    bool held = false;
    FILE *fp = open_for_overwrite(name, &held);
    if (!fp) {
        sp_set_error(SPINGALETT_ERR_INVALID, "save: cannot open file for writing");
        free(owned);
        return;
    }
    const NeuralNetwork *net = args.net;
    const uint8_t has_opt = args.do_not_save_optimizer ? 0 : 1;
    uint8_t head[32];
    size_t h = 0;
    const uint16_t version = held ? 0u : SPINGALETT_FORMAT_VERSION;
    memcpy(head + h, &version, 2); h += 2;
    memcpy(head + h, &net->layers, 4); h += 4;
    head[h++] = (uint8_t)net->loss_func;
    head[h++] = has_opt;
    if (has_opt) { memcpy(head + h, &net->time_step, 8); h += 8; }
    head[h++] = (uint8_t)args.precision;
    bool ok = fwrite(head, 1, h, fp) == h;
    ok = ok && fwrite(net->topology, 4, net->layers, fp) == net->layers;
    for (uint32_t i = 0; i + 1 < net->layers && ok; ++i) {
        const uint8_t a = (uint8_t)net->act_func[i];
        ok = fwrite(&a, 1, 1, fp) == 1;
    }
    if (!ok) {
        sp_set_error(SPINGALETT_ERR_INVALID, "save: failed to write header");
        sp_log(LOG_ERROR, "Failed to write file header to %s", name);
        (void)close_at_length(fp, held);
        free(owned);
        return;
    }
    uint8_t *scratch = NULL;
    const PrecisionMode p = args.precision;
    for (uint32_t l = 0; l + 1 < net->layers && ok; ++l) {
        const uint32_t wcount = net->topology[l] * net->topology[l + 1], bcount = net->topology[l + 1];
        const uint64_t wo = net->weight_offsets[l], bo = net->bias_offsets[l];
        ok = write_array(fp, net->weights + wo, wcount, p, &scratch);
        if (ok && has_opt)
            ok = write_array(fp, net->opt_m_weights + wo, wcount, p, &scratch)
              && write_array(fp, net->opt_v_weights + wo, wcount, p, &scratch);
        if (ok) ok = write_array(fp, net->biases + bo, bcount, p, &scratch);
        if (ok && has_opt)
            ok = write_array(fp, net->opt_m_biases + bo, bcount, p, &scratch)
              && write_array(fp, net->opt_v_biases + bo, bcount, p, &scratch);
    }
    free(scratch);
    if (!close_at_length(fp, held)) ok = false;
    if (!ok) {
        sp_set_error(SPINGALETT_ERR_INVALID, "save: write error (disk full?)");
        sp_log(LOG_ERROR, "Write error saving to %s", name);
    } else {
        sp_log(LOG_INFO, "Network saved to %s", name);
        sp_log(LOG_INFO, "Save info: format=v%u, layers=%u, weights=%llu, biases=%llu, precision=%s, optimizer=%s",
               (unsigned)SPINGALETT_FORMAT_VERSION, net->layers, (unsigned long long)net->total_weights,
               (unsigned long long)net->total_biases, sp_precision_names[p], has_opt ? "ON" : "OFF");
    }
    free(owned);
}
