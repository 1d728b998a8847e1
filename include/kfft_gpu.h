/*
 * GPU additions of the MI355X drop-in.  The reference has no counterpart: it
 * has neither a batch API nor device memory.  Everything here is additive;
 * the reference's entry points keep their signatures and semantics.
 *
 * Pointers: every eval entry point of kfft.h accepts host or device memory.
 * Device (or managed) buffers are transformed in place on the GPU; host
 * buffers are staged through device memory (correct but PCIe-bound).
 * The *_async variants take device pointers only and return without
 * synchronising; `stream` is a hipStream_t (NULL: the library's stream).
 */
#pragma once

/* device memory and synchronisation */
KFFT_API void* kfft_gpu_malloc(size_t bytes);
KFFT_API void kfft_gpu_free(void* ptr);
KFFT_API kfft_return_t kfft_gpu_memcpy_h2d(void* dst, const void* src, size_t bytes);
KFFT_API kfft_return_t kfft_gpu_memcpy_d2h(void* dst, const void* src, size_t bytes);
KFFT_API kfft_return_t kfft_gpu_synchronize(void);
KFFT_API void* kfft_gpu_stream(void);
KFFT_API const char* kfft_gpu_last_error(void);
/* non-zero when an asynchronous launch of this complex plan reported a failed
 * dependency wait since the last call (synchronises the library stream) */
KFFT_API int kfft_gpu_plan_error(const kfft_plan_cpx* plan);
/* one line describing how a complex, scalar or 2D plan is executed */
KFFT_API const char* kfft_gpu_plan_describe(const void* plan);

/* `batch` contiguous transforms: complex in/out distance nfft */
KFFT_API kfft_return_t kfft_eval_cpx_batch(kfft_plan_cpx* plan, const kfft_cpx* fin,
                                           kfft_cpx* fout, uint32_t batch);
KFFT_API kfft_return_t kfft_eval_cpx_batch_async(kfft_plan_cpx* plan, const kfft_cpx* fin,
                                                 kfft_cpx* fout, uint32_t batch, void* stream);
/* As kfft_eval_cpx_batch_async, but allocating nothing: no counterpart in the
 * reference; for callers that cannot allocate device memory (code under HIP
 * graph capture, tight serving loops, harnesses that forbid hipMalloc).  The
 * plan's scratch comes from one library-owned device array of 32 MiB per GPU,
 * held until the process ends; batches whose scratch would exceed it return
 * KFFT_RET_BADARGUMENTS (kfft_gpu_last_error() says how much they need; e.g.
 * at most 64 transforms of 65536 points in the float build, 32 in the double
 * build; one-pass lengths need none; Bluestein lengths count their shortest
 * 2,3,5-smooth convolution length).  Every call on one GPU shares that
 * array: calls that overlap on one GPU race.  Device buffers only; not for
 * KFFT_FLAG_GPU_REFINE plans. */
KFFT_API kfft_return_t kfft_eval_cpx_batch_noalloc(kfft_plan_cpx* plan, const kfft_cpx* fin,
                                                   kfft_cpx* fout, uint32_t batch, void* stream);

/* real input: input distance nfft reals; output distance kfft_scalar_out_len(plan) */
KFFT_API uint32_t kfft_scalar_out_len(const kfft_plan_sclr* plan);
KFFT_API kfft_return_t kfft_eval_scalar_batch(kfft_plan_sclr* plan, const kfft_scalar* fin,
                                              kfft_cpx* fout, uint32_t batch);
KFFT_API kfft_return_t kfft_evali_scalar_batch(kfft_plan_sclr* plan, const kfft_cpx* fin,
                                               kfft_scalar* fout, uint32_t batch);
KFFT_API kfft_return_t kfft_eval_scalar_batch_async(kfft_plan_sclr* plan, const kfft_scalar* fin,
                                                    kfft_cpx* fout, uint32_t batch, void* stream);
KFFT_API kfft_return_t kfft_evali_scalar_batch_async(kfft_plan_sclr* plan, const kfft_cpx* fin,
                                                     kfft_scalar* fout, uint32_t batch,
                                                     void* stream);

/* 2D, asynchronous on device pointers */
KFFT_API kfft_return_t kfft_eval2_cpx_async(kfft_plan_c2d* plan, const kfft_cpx* fin,
                                            kfft_cpx* fout, void* stream);

/*
 * Ragged batch (the batching form): `count` transforms of uneven lengths run
 * as one persistent launch fed by device work queues, replayed as a captured
 * hipGraph.  kind[i]: KFFT_RAGGED_COMPLEX (complex, nfft[i] outputs, forward or
 * KFFT_FLAG_INVERSE as for kfft_eval_cpx) or KFFT_RAGGED_REAL (real-input
 * forward: nfft/2+1 outputs for even nfft, nfft for odd, as kfft_eval_scalar).
 * Offsets are in bytes from the base pointers given at evaluation; NULL
 * offsets select the packed layout (transforms in order, each starting on a
 * 256-byte boundary), which kfft_ragged_layout reports.  Data is kfft_cpx /
 * kfft_scalar of the build.  Device pointers only.
 */
#define KFFT_RAGGED_COMPLEX 0
#define KFFT_RAGGED_REAL 1
typedef struct kfft_plan_ragged kfft_plan_ragged;
KFFT_API kfft_plan_ragged* kfft_config_ragged(uint32_t count, const uint32_t* nfft,
                                              const uint8_t* kind, const uint64_t* in_off,
                                              const uint64_t* out_off, uint32_t flags);
/* offsets (count entries each, may be NULL) and the bytes the buffers must span */
KFFT_API kfft_return_t kfft_ragged_layout(const kfft_plan_ragged* plan, uint64_t* in_off,
                                          uint64_t* out_off, uint64_t* in_bytes,
                                          uint64_t* out_bytes);
KFFT_API kfft_return_t kfft_eval_ragged(kfft_plan_ragged* plan, const void* in, void* out);
KFFT_API kfft_return_t kfft_eval_ragged_async(kfft_plan_ragged* plan, const void* in, void* out,
                                              void* stream);
/* non-zero when the last evaluation's dependency waits timed out (synchronises) */
KFFT_API int kfft_ragged_error(kfft_plan_ragged* plan);
KFFT_API const char* kfft_ragged_describe(const kfft_plan_ragged* plan);
KFFT_API void kfft_release_ragged(kfft_plan_ragged* plan);
/* plan shape chosen for each length class (arrays of kfft_ragged_classes'
 * count entries, each may be NULL); returns the number of classes */
KFFT_API uint32_t kfft_ragged_classes(const kfft_plan_ragged* plan, uint32_t* nfft, uint8_t* kind,
                                      uint32_t* count, uint32_t* max_radix, uint32_t* force_four,
                                      uint32_t* ipw_cap);

/*
 * Autotuner and cost model of the batching form.  A choice is (max_radix 16 /
 * 8 / 4: radix-2 levels fused per LDS stage; force_four: bit 0 two-pass
 * four-step where one pass would fit, bit 1 (Bluestein classes) a power-of-two
 * convolution length instead of the shortest 2,3,5-smooth one; ipw_cap: largest
 * transforms per workgroup tile, 0 for as many as fit).  Times are
 * microseconds per batch on this GPU.
 */
/* the candidate choices (arrays may be NULL); returns their number */
KFFT_API uint32_t kfft_tune_candidates(uint32_t* max_radix, uint32_t* force_four,
                                       uint32_t* ipw_cap);
/* time `count` transforms of one class as a ragged batch under one choice, in
 * throughput terms (the class replicated to at least 2^22 points, the time
 * charged per `count` transforms): best of `reps` runs, or a negative value
 * when the choice does not apply */
KFFT_API double kfft_tune_measure(uint32_t nfft, uint8_t kind, uint32_t count, uint32_t max_radix,
                                  uint32_t force_four, uint32_t ipw_cap, uint32_t reps);
/* cost-model inputs of one class and choice (build precision); returns their number */
KFFT_API uint32_t kfft_cost_features(uint32_t nfft, uint8_t kind, uint32_t count,
                                     uint32_t max_radix, uint32_t force_four, uint32_t ipw_cap,
                                     float* out);
/* MLP nin -> hidden -> hidden -> 1 (ReLU, FP32) with GPU training and inference
 * kernels; x, y, t are device pointers ([batch x nin] row-major, [batch]) */
typedef struct kfft_mlp kfft_mlp;
KFFT_API kfft_mlp* kfft_mlp_create(uint32_t nin, uint32_t hidden, uint32_t seed);
KFFT_API uint32_t kfft_mlp_param_count(const kfft_mlp* mlp);
KFFT_API kfft_return_t kfft_mlp_set_params(kfft_mlp* mlp, const float* host);
KFFT_API kfft_return_t kfft_mlp_get_params(const kfft_mlp* mlp, float* host);
KFFT_API kfft_return_t kfft_mlp_forward(kfft_mlp* mlp, const float* x, float* y, uint32_t batch);
/* gradient of the mean squared error into grad_host (param_count floats) */
KFFT_API kfft_return_t kfft_mlp_gradient(kfft_mlp* mlp, const float* x, const float* t,
                                         uint32_t batch, float* grad_host, float* loss);
/* one Adam step (beta 0.9 / 0.999) on the mean squared error */
KFFT_API kfft_return_t kfft_mlp_train_step(kfft_mlp* mlp, const float* x, const float* t,
                                           uint32_t batch, float lr, float* loss);
KFFT_API void kfft_mlp_release(kfft_mlp* mlp);
/* the model KFFT_FLAG_GPU_TUNED ragged configs rank choices with (it predicts
 * ln microseconds); NULL: exhaustive timing of every applicable choice */
KFFT_API kfft_return_t kfft_ragged_set_cost_model(kfft_mlp* mlp);
