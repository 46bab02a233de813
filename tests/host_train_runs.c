/* host_train_runs.c — how train() cuts the trainings of small nets into launches (sp_train_tiny_run), on the CPU.
 *
 * Built by `make -C spingalett_amd/csrc train_runs` from the library's own C sources plus the stand-ins below for the
 * kernel translation unit: the device calls succeed, sp_train_tiny_run checks what it is given and counts.  A launch is
 * taken to last 5000 cycles and a quarter of a cycle per weight and sample for every step; none may pass 120 M cycles (50
 * ms) by more than a step.  The places of an epoch come in order, whole batches at a time, each exactly once, so do the
 * samples of a shuffled epoch, and the loss of an epoch is the sum over its parts.
 * Larger nets hand their arrays to sp_train_arrays, which here reads or writes every one at its full length.  Built with
 * NO_ARRAYS it is missing, and train() has to say so.  tests/test_host_sanitizers.py builds and runs both. */
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>

#include "sp_train_tiny.h"
#include "spingalett.h"
#include "spingalett_hip.h"

static char g_device;
int sphip_device_count(void) { return 1; }
const char *sphip_last_error_string(void) { return ""; }
int sphip_create(const sphip_desc *d, sphip_net **o) { (void)d; *o = (sphip_net *)&g_device; return 0; }
void sphip_destroy(sphip_net *n) { (void)n; }
int sphip_upload_array(sphip_net *n, uint32_t l, int w, const void *c, size_t b, float m) { (void)n; (void)l; (void)w; (void)c; (void)b; (void)m; return 0; }
int sphip_forward(sphip_net *n, const float *x, uint32_t k, float *y, uint32_t f) { (void)n; (void)x; (void)k; (void)y; (void)f; return 1; }
int sphip_forward_layers(sphip_net *n, const float *x, float *h) { (void)n; (void)x; (void)h; return 1; }
int sphip_evaluate(sphip_net *n, const float *x, const float *t, uint32_t k, int lf, uint32_t f, float *tl, uint32_t *p, uint32_t *c)
{ (void)n; (void)x; (void)t; (void)k; (void)lf; (void)f; (void)tl; (void)p; (void)c; return 1; }
int sphip_decode(sphip_net *n, uint32_t l, int w, int m, float *o) { (void)n; (void)l; (void)w; (void)m; (void)o; return 1; }
int sphip_synchronize(void) { return 0; }
int sphip_train_begin(sphip_net *n) { (void)n; return 0; }
void sphip_train_end(sphip_net *n) { (void)n; }
int sphip_train_set(sphip_net *n, int w, uint32_t l, const float *h) { (void)n; (void)w; (void)l; (void)h; return 0; }
int sphip_train_get(sphip_net *n, int w, uint32_t l, float *h) { (void)n; (void)w; (void)l; (void)h; return 0; }
int sphip_train_step(sphip_net *n, const float *x, const float *t, uint32_t k, const sphip_train_args *a, uint32_t f, float *tl)
{ (void)n; (void)x; (void)t; (void)k; (void)a; (void)f; if (tl) *tl = 0.0f; return 0; }

static uint64_t g_weights, g_biases;
static bool g_large;                          /* the net does not fit one launch */
static uint32_t g_next, g_runs;
static uint64_t g_places, g_steps;
static int g_bad;
static uint8_t *g_seen;                       /* per sample: how often it came */
static double g_reported;

bool sp_train_tiny_fits(uint32_t layers, const uint32_t *topology, uint32_t samples, uint32_t batch, bool ordered)
{ (void)layers; (void)topology; (void)samples; (void)batch; (void)ordered; return !g_large; }

#define CHECK(c) do { if (!(c)) { fprintf(stderr, "run %u: %s\n", g_runs, #c); ++g_bad; } } while (0)
int sp_train_tiny_run(sphip_net *net, const sp_tiny_run *r)
{
    (void)net;
    const uint64_t steps = ((uint64_t)r->count + r->batch - 1u) / r->batch * r->epochs;
    CHECK(r->start == g_next % r->samples && r->start % r->batch == 0);
    CHECK(r->count <= r->samples - r->start && (r->count == r->samples || r->epochs == 1u));
    CHECK(r->first == (g_runs == 0));
    CHECK((steps - (steps > 0)) * (5000u + g_weights * r->batch / 4u) <= 120000000u);
    if (r->order) {
        CHECK((uint64_t)r->epochs * r->count <= r->order_room);
        for (uint64_t i = 0; i < (uint64_t)r->epochs * r->count; ++i) {
            CHECK(r->order[i] < r->samples);
            if (r->order[i] < r->samples) ++g_seen[r->order[i]];
        }
    }
    g_next = r->start + r->count;
    g_places += (uint64_t)r->count * r->epochs;
    g_steps += steps;
    ++g_runs;
    if (r->total_loss) *r->total_loss = 0.5 * r->count;
    return 0;
}

#ifndef NO_ARRAYS
static uint32_t g_ups, g_downs;
static float g_sum;                           /* of what went up */
int sp_train_arrays(sphip_net *net, const sp_train_host *h, bool to_host)
{
    (void)net;
    float *const arrays[8] = {h->weights, h->m_weights, h->v_weights, h->g_weights, h->biases, h->m_biases, h->v_biases, h->g_biases};
    for (int a = 0; a < 8; ++a) {
        if (!arrays[a]) continue;
        for (uint64_t i = 0; i < (a < 4 ? g_weights : g_biases); ++i) {
            if (to_host) arrays[a][i] = (float)(a + 1);
            else g_sum += arrays[a][i];
        }
    }
    if (to_host) {
        for (int a = 0; a < 8; ++a) CHECK(arrays[a]);
        ++g_downs;
    } else {
        CHECK(h->m_weights && h->m_biases && h->v_weights && h->v_biases);
        CHECK((h->weights != NULL) == (g_ups > 0) && (h->biases != NULL) == (g_ups > 0));      /* (a new device net got them when it was made) */
        ++g_ups;
    }
    return 0;
}
#endif

static bool look(NeuralNetwork *net, size_t epoch, float error)
{
    (void)net; (void)epoch;
    g_reported = (double)error;
    return false;
}

static int one(uint32_t samples, uint32_t hidden, TrainingStrategy strategy, uint32_t batch, size_t epochs)
{
    NeuralNetwork *net = new_spingalett(.loss_func = LOSS_MSE);
    layer(.net = net, .neurons_amount = 2);
    layer(.net = net, .neurons_amount = hidden, .act_func = ACT_TANH, .weight_initialization = WEIGHT_INITIALIZATION_XAVIER);
    layer(.net = net, .neurons_amount = 1, .act_func = ACT_NONE, .weight_initialization = WEIGHT_INITIALIZATION_XAVIER);
    float *x = (float *)calloc((size_t)samples * 2u, sizeof *x), *t = (float *)calloc(samples, sizeof *t);
    g_seen = (uint8_t *)calloc(samples, 1);
    g_weights = net->total_weights;
    g_next = g_runs = 0;
    g_places = g_steps = 0;
    train(.net = net, .inputs = x, .targets = t, .sample_count = samples, .epochs = epochs, .training_strategy = strategy,
          .batch_size = batch, .callback = look, .callback_interval = epochs);
    const uint64_t per = strategy == STRATEGY_SAMPLE ? 1u : strategy == STRATEGY_SMALL_BATCH ? batch : samples;
    CHECK(g_places == (uint64_t)samples * epochs);
    CHECK(g_steps == (samples + per - 1u) / per * epochs && net->time_step == g_steps);
    CHECK(g_reported == 0.5);
    for (uint32_t s = 0; s < samples && strategy == STRATEGY_SMALL_BATCH; ++s) CHECK(g_seen[s] == epochs);
    printf("%u samples, strategy %d, batch %u, %zu epochs: %u launches, %llu steps\n", samples, (int)strategy, batch, epochs, g_runs,
           (unsigned long long)g_steps);
    free(x);
    free(t);
    free(g_seen);
    free_network(net);
    return g_bad;
}

/* a net whose steps are launches of their own, trained twice */
static void large(void)
{
    enum { IN = 33, HIDDEN = 129, OUT = 7, SAMPLES = 50 };
    NeuralNetwork *net = new_spingalett(.loss_func = LOSS_MSE);
    layer(.net = net, .neurons_amount = IN);
    layer(.net = net, .neurons_amount = HIDDEN, .act_func = ACT_TANH, .weight_initialization = WEIGHT_INITIALIZATION_XAVIER);
    layer(.net = net, .neurons_amount = OUT, .act_func = ACT_NONE, .weight_initialization = WEIGHT_INITIALIZATION_XAVIER);
    float *x = (float *)calloc(SAMPLES * IN, sizeof *x), *t = (float *)calloc(SAMPLES * OUT, sizeof *t);
    g_large = true;
    g_weights = net->total_weights;
    g_biases = net->total_biases;
    for (uint32_t run = 0; run < 2u; ++run) {
        const float first = net->weights[0], last = net->biases[g_biases - 1u];
        spingalett_clear_error();
        train(.net = net, .inputs = x, .targets = t, .sample_count = SAMPLES, .epochs = 3, .training_strategy = STRATEGY_FULL_BATCH);
#ifdef NO_ARRAYS
        CHECK(spingalett_last_error_code() != SPINGALETT_OK);
        CHECK(net->weights[0] == first && net->biases[g_biases - 1u] == last && net->time_step == 0);
#else
        (void)first;
        (void)last;
        CHECK(spingalett_last_error_code() == SPINGALETT_OK);
        CHECK(g_ups == run + 1u && g_downs == run + 1u);
        float *const arrays[8] = {net->weights, net->opt_m_weights, net->opt_v_weights, net->grad_weights,
                                  net->biases, net->opt_m_biases, net->opt_v_biases, net->grad_biases};
        for (int a = 0; a < 8; ++a) CHECK(arrays[a][0] == (float)(a + 1) && arrays[a][(a < 4 ? g_weights : g_biases) - 1u] == (float)(a + 1));
#endif
    }
    printf("arrays of a larger net: %s\n", g_bad ? "not as they should be" : "as they should be");
    g_large = false;
    free(x);
    free(t);
    free_network(net);
}

int main(void)
{
    spingalett_set_verbose(false);
    spingalett_set_log_level(LOG_NONE);
    large();
    one(1000000, 8, STRATEGY_SAMPLE, 0, 2);                  /* an epoch of a million steps */
    one(24011, 8, STRATEGY_SAMPLE, 0, 3);                    /* a few steps more than a launch takes */
    one(100, 8, STRATEGY_SAMPLE, 0, 1000);                   /* many epochs to a launch */
    one(30001, 8, STRATEGY_SMALL_BATCH, 1, 2);
    one(300007, 200, STRATEGY_SMALL_BATCH, 7, 2);            /* the last batch and the last launch in part */
    one(4, 8, STRATEGY_FULL_BATCH, 0, 100000);
    return g_bad ? 1 : 0;
}
