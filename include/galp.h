/*
 * galp.h -- C-ABI of the MI355X (gfx950) label-propagation update.
 *
 * The drop-in boundary for galp's hot path: methods 0 (sort / segmented
 * reduce) and 1 (hash tables) of the `galp [opts] method policy data [test]`
 * program, on one GPU.  Plain C types only; every entry point returns 0 or a
 * negative galp_status (galp_status.h) and never throws.  One galp_ctx per
 * host thread; calls on one ctx (and its graphs) must not overlap.
 *
 * Semantics shared by every method, policy and variant (each a deliberate,
 * documented difference from the reference's GPU kernels, which are
 * asynchronous and resolve ties by atomic order):
 *   - synchronous update: iteration t reads labels(t-1) and writes labels(t);
 *   - tie rule: new(v) = argmax_L (count_v(L), last_v(L)), last_v(L) being the
 *     largest CSR position of v's row holding label L -- the result of the
 *     `if (max_count <= c)` scan of label_propagation/src/common/
 *     hybrid_cpu_worker.cuh:177-186;
 *   - a vertex without neighbours keeps its label;
 *   - updated = #{v : labels(t)[v] != labels(t-1)[v]}; a run stops after an
 *     iteration with updated <= n * 1e-5 (lfht.cuh:97, dpp.cuh:88).
 */
#ifndef GALP_H
#define GALP_H

#include <stdint.h>
#include <stddef.h>
#include "galp_status.h"

#ifdef __cplusplus
extern "C" {
#endif

#ifndef GALP_API
#define GALP_API __attribute__((visibility("default")))
#endif

typedef struct galp_ctx galp_ctx;
typedef struct galp_graph galp_graph;

/* Borrowed host CSR: n+1 offsets (int64 if offsets_are_64, else int32) and m
 * int32 neighbour ids.  The caller keeps the arrays alive for the duration of
 * galp_graph_upload (in-core) or of the graph (out-of-core policies, which
 * stream from them).  Mirrors CSRGraph<V,E>::{offsets, neighbors}
 * (label_propagation/include/graph.h:160-161). */
typedef struct galp_csr_view {
    int64_t n;
    int64_t m;
    const void *offsets;
    const int32_t *neighbors;
    int32_t offsets_are_64;
    int32_t reserved;
} galp_csr_view;

enum { GALP_METHOD_SORT = 0, GALP_METHOD_HASH = 1 };
enum {
    GALP_POLICY_INCORE = 0,     /* main.cu:140-145,169-174 */
    GALP_POLICY_OOC_SYNC = 1,   /* out-of-core, no overlap: main.cu:147-150,176-179 */
    GALP_POLICY_OOC_ASYNC = 2,  /* out-of-core, overlapped: main.cu:152-155,181-184 */
    GALP_POLICY_LI = 4          /* method 0 only, "load-imbalanced": main.cu:162-167 */
};
enum { GALP_DISPATCH_PLAIN = 0, GALP_DISPATCH_LEARNED = 1 };

/* Options of one graph.  Mirrors the CLI state of main.cu:80-116 (method,
 * policy, -b, -l) plus the build's own switches. */
typedef struct galp_opts {
    int32_t method;      /* GALP_METHOD_* */
    int32_t policy;      /* GALP_POLICY_* */
    int32_t variant;     /* -l 0..3 (main.cu:98-100): 0 naive, 1 fused (default),
                            2 small LDS tables + spill, 3 load-balanced tiles */
    int32_t buffer_pow;  /* -b: out-of-core chunk of 2^buffer_pow edges (main.cu:86-88) */
    int32_t dispatch;    /* GALP_DISPATCH_*: degree thresholds, or the MLP */
    int32_t reorder;     /* 1 (default): degree-descending internal renumbering;
                            labels are mapped back on every read-out */
    int32_t profile;     /* 1: time every kernel launch with HIP events */
    int32_t graph_capture; /* 1: galp_lp_run (verbose = 0, in-core, profile = 0)
                              captures its iteration loop in a hipGraph once per
                              niter and replays it */
    int64_t mem_budget;  /* device bytes the graph may allocate; 0 = free memory.
                            Exceeding it fails with GALP_ENOMEM (check_gpu_mem,
                            main.cu:51-64) */
    int32_t offsets64;   /* 1: int64 device offsets even when m < 2^31 (they
                            are int64 whenever m >= 2^31) */
    int32_t reserved;
} galp_opts;

/* Per-iteration result.  Replaces the count returned by iterate()/get_count()
 * (incore.cuh:42-48, lfht.cuh:171-179) and the printed time (lfht.cuh:95). */
typedef struct galp_step_stats {
    int64_t updated;     /* vertices whose label changed */
    int64_t overflowed;  /* vertices re-run on the spill path (learned dispatch) */
    double device_ms;    /* HIP-event time of the iteration on the graph's stream */
    int32_t iteration;   /* 1-based index of the iteration just run */
    int32_t stopped;     /* 1 if the n*1e-5 rule says to stop after it */
} galp_step_stats;

/* Result of a whole run.  f1/f2 keep the meaning of LabelPropagator::run's
 * pair (lfht.cuh:76-111): f1 = main loop including the final label copy,
 * f2 = f1 plus the preprocessing done at upload. */
typedef struct galp_run_result {
    double f1_s;
    double f2_s;
    double device_ms;    /* HIP-event time of the iterations alone */
    int32_t iterations;  /* iterations executed (<= niter) */
    int32_t reserved;
} galp_run_result;

typedef struct galp_graph_info {
    int64_t n;
    int64_t m;
    int32_t offsets_are_64;
    int32_t nbuckets;
    int64_t bucket_vertices[16];
    int64_t bucket_edges[16];
    int64_t device_bytes;
    double preprocess_ms;
} galp_graph_info;

typedef struct galp_device_info {
    char name[64];
    char arch[32];
    int32_t compute_units;
    int32_t wavefront_size;
    int64_t lds_per_block;
    int64_t total_mem;
    int64_t l2_bytes;
} galp_device_info;

/* Per-kernel timing when galp_opts.profile = 1. */
typedef struct galp_kernel_stat {
    char name[48];
    int64_t launches;
    double total_ms;
    double alg_bytes;    /* algorithmic HBM bytes summed over the launches */
} galp_kernel_stat;

/* Fills the reference's defaults: method 1, policy 0, -l 1, -b 24, plain
 * dispatch, reorder on (main.cu:80-83). */
GALP_API void galp_opts_default(galp_opts *o);

/* Opens a device.  Replaces the warm-up cudaSetDevice/cudaFree(0) of
 * main.cu:123-128.  device must be 0 in this one-GPU build's tests, but any
 * visible device is accepted. */
GALP_API int galp_open(int device, galp_ctx **out);
GALP_API int galp_close(galp_ctx *ctx);
GALP_API int galp_device_query(galp_ctx *ctx, galp_device_info *out);

/* Copies the CSR to HBM and prepares the dispatch plan.  Replaces
 * init_gmem + transfer_data (lfht.cuh:182-214, dpp.cuh:154-175,
 * incore.cuh:34-38,59-73) and the propagator constructors selected by
 * main.cu:139-207.  Policies 3 (hybrid), 4 with method 1 and 5 (multi-GPU)
 * return GALP_EUNSUPPORTED, like the one-GPU build's CLI. */
GALP_API int galp_graph_upload(galp_ctx *ctx, const galp_csr_view *csr,
                               const galp_opts *opts, galp_graph **out);
GALP_API int galp_graph_free(galp_graph *g);
GALP_API int galp_graph_query(galp_graph *g, galp_graph_info *out);

/* labels[i] = i.  Replaces initialize_labels (dpp/kernel.cuh:15-22). */
GALP_API int galp_lp_init(galp_graph *g);

/* Sets the current labels from host_labels[n] (original vertex numbering,
 * every value in [0, n)) and marks the graph initialised, so the next step
 * reads them.  No reference counterpart (the reference always starts from
 * labels[i] = i); it lets the tests run an iteration from any label state. */
GALP_API int galp_lp_set_labels(galp_graph *g, const int32_t *host_labels);

/* One synchronous iteration.  Replaces perform_lp + get_count
 * (lfht.cuh:115-179, dpp.cuh:104-150). */
GALP_API int galp_lp_step(galp_graph *g, galp_step_stats *st);

/* init + up to niter iterations with the n*1e-5 stop + final copy to
 * labels_out (n entries, may be NULL).  Replaces LabelPropagator::run
 * (lfht.cuh:73-112, dpp.cuh:64-102).  verbose = 1 prints the reference's
 * per-iteration line "%d: %f (s), updated %d" (lfht.cuh:95) to stdout, which
 * needs a host synchronisation per iteration; verbose = 0 queues all
 * iterations and applies the stop rule on the device. */
GALP_API int galp_lp_run(galp_graph *g, int32_t niter, int32_t verbose,
                         int32_t *labels_out, galp_run_result *res);

/* Copies the current labels (original vertex numbering) to host_out[n].
 * Replaces LabelPropagator::get_labels (label_propagator.h:22-28). */
GALP_API int galp_lp_get_labels(galp_graph *g, int32_t *host_out);

/* Per-kernel timing (profile = 1).  Writes up to max entries; *count gets the
 * number of kernels seen.  galp_profile_reset clears the totals. */
GALP_API int galp_profile_read(galp_graph *g, galp_kernel_stat *out,
                               int32_t max, int32_t *count);
GALP_API int galp_profile_reset(galp_graph *g);

/* Diagnostic, no reference counterpart: the gather ceiling of this graph's
 * access pattern.  One pass reads every neighbour id (sequentially,
 * non-temporal) and gathers that neighbour's current label, as every LP
 * kernel does, with nothing else: no counting, no label writes, only a
 * 64-bit sum of the gathered labels (*checksum, may be NULL).  Runs one pass
 * for the checksum, then `reps` timed ones; *ms_per_pass gets their mean
 * (HIP events on the graph's stream).  In core only. */
GALP_API int galp_graph_gather_probe(galp_graph *g, int32_t reps, double *ms_per_pass,
                                     uint64_t *checksum);

/* ---- learned dispatch: the distinct-label predictor ----------------------
 * A 4 -> H -> H -> 1 MLP (ReLU, ReLU, linear; fp32; H in {8, 16, 32}) with
 * parameters laid out as W1[H][4], b1[H], W2[H][H], b2[H], W3[H], b3.
 * Inputs per vertex: log2(1+degree), log2(1+mean neighbour degree),
 * log2(1+max neighbour degree), log2(1+distinct labels of the previous
 * iteration) or -1 before the first; target log2(1+distinct labels).
 * No reference counterpart (the reference dispatches by -l only,
 * lfht.cuh:127-165).  All computation runs in HIP kernels. */
GALP_API int64_t galp_mlp_num_params(int32_t hidden);
/* He-initialised parameters from a seed (host only). */
GALP_API int galp_mlp_init(int32_t hidden, uint64_t seed, float *params);
/* y_hat[n] for x[n][4] (host arrays). */
GALP_API int galp_mlp_predict(galp_ctx *ctx, int32_t hidden, const float *params,
                              const float *x, int64_t n, float *yhat);
/* Loss (mean of 0.5 (y_hat - y)^2) and its gradient over x[n][4], y[n]. */
GALP_API int galp_mlp_loss_grad(galp_ctx *ctx, int32_t hidden, const float *params,
                                const float *x, const float *y, int64_t n,
                                float *grad, float *loss);
/* galp_mlp_loss_grad on device-resident data, allocating nothing.  No
 * reference counterpart: it is for callers that cannot allocate device
 * memory -- code under HIP graph capture, tight serving loops, harnesses that
 * forbid hipMalloc.  d_params, d_x[n][4], d_y[n], d_grad[P] and d_loss[1]
 * are device pointers on the context's device, which must be current;
 * the kernels are queued on `stream` (a hipStream_t; NULL = the null
 * stream) and the call returns without waiting for them.  The per-block
 * partial gradients live in a fixed device array of the library (2.56 MB per
 * device, held until the process ends), so n is limited to 32768 samples
 * (GALP_EINVAL beyond), and calls that overlap on one device race on it. */
GALP_API int galp_mlp_loss_grad_noalloc(galp_ctx *ctx, int32_t hidden, const float *d_params,
                                        const float *d_x, const float *d_y, int64_t n,
                                        float *d_grad, float *d_loss, void *stream);
/* Adam over `epochs` passes of minibatches of `batch` samples (seeded
 * shuffle); params are updated in place; final_loss = loss over all n. */
GALP_API int galp_mlp_train(galp_ctx *ctx, int32_t hidden, float *params,
                            const float *x, const float *y, int64_t n,
                            int32_t epochs, int32_t batch, float lr,
                            uint64_t seed, float *final_loss);

/* Attaches a trained network to a graph uploaded with dispatch = learned:
 * vertices of degree > 64 whose predicted distinct-label count is <=
 * cand_thresh take the register-candidate path, the others the degree-class
 * kernels; a misprediction falls back to the latter within the iteration. */
GALP_API int galp_graph_set_mlp(galp_graph *g, int32_t hidden, const float *params, float cand_thresh);
/* Logs one training sample per vertex of degree > 64 and iteration (inputs
 * from the previous iteration's distinct count, target this iteration's),
 * up to `capacity` samples; galp_graph_log_read copies them out. */
GALP_API int galp_graph_log_enable(galp_graph *g, int64_t capacity);
GALP_API int galp_graph_log_read(galp_graph *g, float *x, float *y, int64_t max, int64_t *count);
/* Raw static features per vertex (original numbering): degree, mean and max
 * neighbour degree, computed for vertices of degree > 64 (0 otherwise). */
GALP_API int galp_graph_features(galp_graph *g, float *deg, float *mean, float *mx);
/* Counters of the last iteration that learned dispatch was in charge of,
 * zeros where it routed nothing (the first iteration from labels[i] = i in
 * closed form, iterations over the rows that can still change): [0..12) class
 * list sizes, [12..16) candidate tiles per length class (<= 128, 256, 512, 1024
 * edges), [16] candidate overflows, [17] vertices routed to candidates,
 * [18] hubs left to the plain hub path, [19] multi-tile rows routed to
 * candidates, [20..32) sizes of the classes' high-distinct lists ([31], the
 * hub class: hubs of the high-distinct hub launch), [32] big vertices
 * predicted high-distinct on any path. */
GALP_API int galp_graph_dispatch_stats(galp_graph *g, int64_t *out, int32_t max, int32_t *count);

/* ---- autotuner -------------------------------------------------------------
 * Each degree class of either method has kTuneOptions = 3 kernel
 * configurations (0 = default; the others change the workgroup size, slots
 * or keys per lane, the sort algorithm or blocks per CU).
 * galp_graph_autotune runs 10 iterations from labels[i] = i under each
 * option (all untuned classes at once, the graph's own dispatch), `reps`
 * rounds, reads each class's device time from per-kernel events and keeps
 * its fastest option; then, in core, it times such runs with the class
 * kernels on one stream and on three and keeps the size rule's choice
 * unless the other is more than 3 % faster; on a graph small enough to run
 * its row classes in one launch it times that launch against the class
 * kernels so chosen, which have to be more than 3 % faster to replace it;
 * under learned dispatch it then
 * judges the network against the plain classes per iteration
 * (galp_graph_set_learned_iterations) and, when some iterations go to the
 * classes alone, times the class options again under that mask.  It leaves
 * the graph
 * initialised (labels[i] = i) and the per-kernel profile totals as they
 * were.  cache_path (may be NULL) names a text file of earlier
 * choices keyed by device arch, method and the class's log2 sizes; hits are
 * reused without timing and new choices are appended.  chosen (may be NULL)
 * receives 16 entries: the 12 class options as the next run uses them (0 for
 * the classes that run in one launch), then the stream choice of the class
 * kernels (1 or 3; 0 where not timed), then the judge's mask (two halves;
 * zeros without learned dispatch), then 1 where a graph of one-launch size
 * was given the class kernels, else 0.  Labels never depend on the choices.
 * No reference counterpart (fixed block sizes, lfht.cuh:127-165). */
GALP_API int galp_graph_autotune(galp_graph *g, int32_t reps, const char *cache_path, int32_t *chosen);
/* Learned dispatch in core: which iterations route by the network (bit i
 * for iteration i, bit 63 for every later one); the others run the plain
 * degree classes, the dispatcher the network is judged against.
 * galp_graph_autotune sets it by timing both per iteration and keeping the
 * network where it is more than 2 % faster (chosen[13] and chosen[14]
 * receive the mask's low and high halves); the default routes every
 * iteration by the network.  Labels never depend on it.  No reference
 * counterpart. */
GALP_API int galp_graph_set_learned_iterations(galp_graph *g, uint64_t mask);
/* Sets the option of every class directly (12 entries, each 0..2).  An option
 * other than the default 0 for a class that a small or mid-sized graph would
 * run in one launch with others gives it a kernel per class; all such options
 * 0 give back the choice by size. */
GALP_API int galp_graph_set_tuning(galp_graph *g, const int32_t *options);
/* How the next iteration over every row launches its classes: *mode = 0 in one
 * launch for the classes up to 2048 edges (sort: 1024) and a kernel for each
 * longer class; 1 or 3 a kernel per class, on one stream or three. */
GALP_API int galp_graph_row_launches(galp_graph *g, int32_t *mode);

/* ---- batched runs --------------------------------------------------------
 * Declares the uploaded (in-core) CSR to be the disjoint union of ngraphs
 * graphs, graph k owning vertices [vbase[k], vbase[k+1]) of the original
 * numbering (vbase[0] = 0, vbase[ngraphs] = n; an edge joining two graphs is
 * rejected).  Each graph then follows its own stop rule (stop after an
 * iteration with updated_k <= n_k * 1e-5), so graph k's labels equal an
 * independent run of it shifted by vbase[k], while one launch per degree
 * class serves all graphs.  galp_step_stats.updated and the per-iteration
 * counts sum over the graphs still running.  No reference counterpart (the
 * reference runs one graph per process). */
GALP_API int galp_graph_set_batch(galp_graph *g, int64_t ngraphs, const int64_t *vbase);
/* Iterations each graph ran in the last run (ngraphs entries). */
GALP_API int galp_batch_iterations(galp_graph *g, int32_t *iters_out);

/* Message of the last failure on ctx; "" if none. */
GALP_API const char *galp_last_error(galp_ctx *ctx);

#ifdef __cplusplus
}
#endif

#endif /* GALP_H */
