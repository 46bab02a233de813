/*
 * sp_train_tiny.h — the training of small nets inside one launch (hip_train_tiny.inl) and the host arrays of any training on
 * their way to the device and back (hip_transfer.inl), as the C side calls them.
 * Internal: not part of the library's interface.
 */
#ifndef SP_TRAIN_TINY_H
#define SP_TRAIN_TINY_H

#include "spingalett_hip.h"

#ifdef __cplusplus
extern "C" {
#else
#include <stdbool.h>
#endif

/* `epochs` passes over the samples in steps of `batch` of them; the arrays are flat like NeuralNetwork's and hold the
 * results when the call returns. */
typedef struct {
    float *weights, *biases, *m_weights, *m_biases, *v_weights, *v_biases, *g_weights, *g_biases;
    const float *x, *t;              /* [samples][width], host memory */
    uint32_t samples, batch, epochs;
    uint32_t start, count;           /* which of an epoch's places this run covers: all of them, or whole batches of one
                                        epoch that is too long for a launch */
    const uint32_t *order;           /* [epochs][count] which sample comes when, or NULL: as they lie */
    uint32_t order_room;             /* entries that any part of this training passes in order at most */
    bool first;                      /* first part of a training: arrays and samples go to the device (later parts go on
                                        from where the last one ended) */
    const sphip_train_args *args;    /* beta*_pow_t: before the first step */
    double *total_loss;              /* sum of the losses of the last epoch's places covered here, or NULL */
} sp_tiny_run;

/* sphip_train_step flag: the batch is the whole training set, which goes to the device once */
#define SP_TRAIN_WHOLE_SET (1u << 30)

/* Arrays of a net, flat like NeuralNetwork's, or NULL for those that stay where they are */
typedef struct {
    float *weights, *biases, *m_weights, *m_biases, *v_weights, *v_biases, *g_weights, *g_biases;
} sp_train_host;

/* A build of the C side alone (the host sanitizer's) has none of these: weak there, checked before use. */
#if defined(__cplusplus)
#define SP_TINY_API __attribute__((visibility("hidden")))
#else
#define SP_TINY_API __attribute__((visibility("hidden"), weak))
#endif
SP_TINY_API bool sp_train_tiny_fits(uint32_t layers, const uint32_t *topology, uint32_t samples, uint32_t batch, bool ordered);
SP_TINY_API int  sp_train_tiny_run(sphip_net *net, const sp_tiny_run *run);
SP_TINY_API int  sp_train_arrays(sphip_net *net, const sp_train_host *arrays, bool to_host);

#ifdef __cplusplus
}
#endif
#endif
