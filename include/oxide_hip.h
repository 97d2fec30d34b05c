/*
 * oxide_hip.h -- C ABI of liboxide_hip.so, the MI355X (gfx950) backend for oxide-torch's
 * tensor hot path.
 *
 * This is the surface a Rust `oxide-torch-hip` crate binds with `extern "C"` to replace
 * `oxide-torch-cuda` (tuna2134/oxide-beta) on the hot path: the kernel launchers generated by
 * `#[cuda_module]` in crates/oxide-torch-cuda/src/kernel_module.rs, `load_kernels`
 * (crates/oxide-torch-cuda/src/lib.rs:19-30), the graph wrapper `CudaGraphExec`
 * (crates/oxide-torch-cuda/src/cuda_graph.rs:30-179) and the buffer/stream calls the adapter
 * makes through cuda-core (crates/oxide-torch/src/cuda/runtime.rs:46-105,
 * crates/oxide-torch/src/cuda/jit.rs:25-99).
 *
 * Conventions
 *   - Every function returns an oxh_status; OXH_OK is 0.  On failure a message for the calling
 *     thread is available from oxh_last_error().
 *   - Device pointers are plain `float*` / `void*` from oxh_alloc (or any HIP allocation on the
 *     current device).  Sizes are element counts (uint64_t) unless the name says bytes.
 *   - `stream` is a hipStream_t passed as an opaque pointer; NULL is the device's null stream.
 *     Every launcher only enqueues work; none synchronizes, none allocates.
 *   - The launch configuration is chosen inside the library (the reference's LaunchConfig is an
 *     implementation detail of its launchers).
 *   - Shapes are validated on the host before any launch; a bad shape returns
 *     OXH_INVALID_SHAPE and enqueues nothing.
 *   - Aliasing: elementwise launchers and AdamW may run in place (an output pointer equal to
 *     the matching input pointer); reductions and batch-norm/cross-entropy outputs must not
 *     alias their inputs.
 *   - Reductions that need scratch take a caller-owned device `workspace` of at least the
 *     size returned by the matching *_workspace_size query (16-byte aligned, no initial
 *     contents required).  It carries per-block partial sums from a reduce launch to the launch
 *     that consumes them, so calls sharing one workspace must be ordered on one stream and a
 *     two-phase pair (forward_reduce -> forward_apply, backward_reduce -> backward_input) must
 *     not be interleaved with another user of the same workspace.
 *   - The library is thread-compatible: one host thread issues to a given stream at a time.
 */
#ifndef OXIDE_HIP_H
#define OXIDE_HIP_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* Status codes; the first three mirror crates/oxide-torch/src/error.rs:1-56
 * (Error::InvalidShape, Error::Execution, Error::Cuda -> HIP). */
typedef int oxh_status;
#define OXH_OK 0
#define OXH_INVALID_SHAPE 1 /* Error::InvalidShape: shape / size / argument rejected on host */
#define OXH_EXECUTION 2     /* Error::Execution: runtime condition (e.g. BN with <= 1 sample) */
#define OXH_HIP_ERROR 3     /* Error::Cuda analogue: a HIP runtime call failed */
#define OXH_TRACE 4         /* Error::Trace: plan inputs do not match the compiled plan */

typedef void *oxh_stream; /* hipStream_t */

/* ------------------------------------------------------------------ runtime */

/* Message of the last failure on the calling thread ("" if none). */
const char *oxh_last_error(void);
/* Library version string. */
const char *oxh_version(void);

/* Selects `device` and loads the code object (load_kernels, oxide-torch-cuda/src/lib.rs:19-30:
 * here the gfx950 code object is linked into the library, so this only selects and checks the
 * device). */
oxh_status oxh_init(int device);
oxh_status oxh_device_count(int *count);

/* A non-default stream at the default priority (CudaContext::new_stream, cuda/jit.rs:27-30). */
oxh_status oxh_stream_create(oxh_stream *stream);
oxh_status oxh_stream_destroy(oxh_stream stream);
oxh_status oxh_stream_synchronize(oxh_stream stream);

/* DeviceBuffer::{zeroed, uninitialized_async, from_host, copy_from_host_async_unchecked,
 * to_host_vec} (runtime.rs:83-105, cuda/jit.rs:34-45,93,97). */
oxh_status oxh_alloc(void **ptr, uint64_t bytes);
oxh_status oxh_free(void *ptr);
/* Zeroes `bytes` bytes at any alignment with a fill kernel (no memset node), so it may be
 * recorded into a graph. */
oxh_status oxh_memset0_async(void *ptr, uint64_t bytes, oxh_stream stream);
oxh_status oxh_memcpy_h2d_async(void *dst, const void *src, uint64_t bytes, oxh_stream stream);
/* Synchronous device-to-host copy: returns once `dst` holds the data. */
oxh_status oxh_memcpy_d2h(void *dst, const void *src, uint64_t bytes, oxh_stream stream);
oxh_status oxh_memcpy_d2d_async(void *dst, const void *src, uint64_t bytes, oxh_stream stream);

/* Kernel timing (the reference's MNIST_PROFILE phase timings, mnist_training.rs:159-199, at
 * kernel granularity).  oxh_time_next_launch arms the calling thread's next kernel launch to
 * record `start` when the dispatch begins and `stop` when it ends (hipExtLaunchKernelGGL), the
 * interval a kernel-trace profiler reports; for an entry point that launches several kernels
 * only the first is timed.  Not for use during graph capture. */
typedef void *oxh_event; /* hipEvent_t */
oxh_status oxh_event_create(oxh_event *event);
oxh_status oxh_event_destroy(oxh_event event);
/* Waits for `stop`, then returns the elapsed milliseconds between the two events. */
oxh_status oxh_event_elapsed_ms(oxh_event start, oxh_event stop, float *ms);
oxh_status oxh_time_next_launch(oxh_event start, oxh_event stop);

/* ------------------------------------------------------------------ elementwise
 * kernel_module.rs:8-34 (add, mul, relu), 492-508 (mul_backward, relu_backward),
 * 1052-1059 (accumulate); launched by runtime.rs:140-161,671-749 and cuda/jit.rs:101-194.
 * fp32, bit-exact with the reference CPU path (evaluation.rs:21-34, autograd.rs:94-147). */
oxh_status oxh_add(oxh_stream stream, const float *a, const float *b, float *output, uint64_t n);
oxh_status oxh_mul(oxh_stream stream, const float *a, const float *b, float *output, uint64_t n);
/* output = input > 0 ? input : 0 */
oxh_status oxh_relu(oxh_stream stream, const float *input, float *output, uint64_t n);
/* output = gradient * other (left grad uses the right operand and vice versa) */
oxh_status oxh_mul_backward(oxh_stream stream, const float *gradient, const float *other,
                            float *output, uint64_t n);
/* output = input > 0 ? gradient : 0 */
oxh_status oxh_relu_backward(oxh_stream stream, const float *gradient, const float *input,
                             float *output, uint64_t n);
/* output = a + b (gradient accumulation, runtime.rs:671-692) */
oxh_status oxh_accumulate(oxh_stream stream, const float *a, const float *b, float *output,
                          uint64_t n);

/* Fused extras (no single reference kernel; same per-element results as the reference's
 * add -> mul -> relu plan and its VJPs):
 *   y = relu((a + b) * c)
 *   backward with upstream gradient `gradient` (NULL means ones, the backward of sum(y)):
 *     s = a + b; m = s * c; g = m > 0 ? gradient : 0; da = db = g * c; dc = g * s. */
oxh_status oxh_elementwise_chain_forward(oxh_stream stream, const float *a, const float *b,
                                         const float *c, float *y, uint64_t n);
oxh_status oxh_elementwise_chain_backward(oxh_stream stream, const float *a, const float *b,
                                          const float *c, const float *gradient, float *da,
                                          float *db, float *dc, uint64_t n);

/* ------------------------------------------------------------------ batch norm 2d (NCHW)
 * Reference kernels kernel_module.rs:827-964,1061-1092; driver runtime.rs:526-669 (forward),
 * 1092-1156 (backward); CPU semantics evaluation.rs:448-597, autograd.rs:315-383.
 * Per-channel sums are formed once, with fp64 partials.  The separate statistics and
 * affine-backward entry points take a workspace too (reduce + a per-channel finalize launch). */

/* Bytes of workspace the statistics / affine-backward reductions need for this shape. */
oxh_status oxh_batch_norm_workspace_size(uint64_t batch, uint64_t channels, uint64_t spatial,
                                         uint64_t *bytes);

/* batch_norm_statistics (kernel_module.rs:827-875): per channel mean, 1/sqrt(var + eps) with
 * the biased variance, and the unbiased variance used for the running update.
 * Fails with OXH_EXECUTION when batch * spatial <= 1 (evaluation.rs:498-502). */
oxh_status oxh_batch_norm_statistics(oxh_stream stream, uint64_t batch, uint64_t channels,
                                     uint64_t spatial, float epsilon, const float *input,
                                     float *mean, float *inverse_std, float *unbiased_variance,
                                     void *workspace, uint64_t workspace_bytes);
/* batch_norm_update_running (kernel_module.rs:1074-1092):
 *   new_mean = (1 - momentum) * old_mean + momentum * batch_mean
 *   new_var  = (1 - momentum) * old_var  + momentum * batch_variance
 * new_* may equal old_* (in place). */
oxh_status oxh_batch_norm_update_running(oxh_stream stream, uint64_t channels, float momentum,
                                         const float *batch_mean, const float *batch_variance,
                                         const float *old_mean, const float *old_variance,
                                         float *new_mean, float *new_variance);
/* batch_norm_running_inverse_std (kernel_module.rs:1061-1072): 1 / sqrt(variance + eps). */
oxh_status oxh_batch_norm_running_inverse_std(oxh_stream stream, uint64_t channels,
                                              float epsilon, const float *variance,
                                              float *inverse_std);
/* batch_norm_apply (kernel_module.rs:877-895): y = (x - mean[c]) * inv_std[c] * w[c] + b[c]. */
oxh_status oxh_batch_norm_apply(oxh_stream stream, uint64_t batch, uint64_t channels,
                                uint64_t spatial, const float *input, const float *weight,
                                const float *bias, const float *mean, const float *inverse_std,
                                float *output);
/* batch_norm_affine_backward (kernel_module.rs:929-964): per channel
 *   weight_gradient = sum(g * (x - mean) * inv_std), bias_gradient = sum(g). */
oxh_status oxh_batch_norm_affine_backward(oxh_stream stream, uint64_t batch, uint64_t channels,
                                          uint64_t spatial, const float *gradient,
                                          const float *input, const float *mean,
                                          const float *inverse_std, float *weight_gradient,
                                          float *bias_gradient, void *workspace,
                                          uint64_t workspace_bytes);
/* batch_norm_input_backward (kernel_module.rs:897-927), using the affine gradients as the
 * pre-reduced channel sums (the one-reduction backward):
 *   training: dx = w*inv/M * (M*g - bias_gradient - x_hat*weight_gradient), M = batch*spatial
 *   eval:     dx = g * w * inv */
oxh_status oxh_batch_norm_input_backward(oxh_stream stream, uint64_t batch, uint64_t channels,
                                         uint64_t spatial, int training, const float *gradient,
                                         const float *input, const float *weight,
                                         const float *mean, const float *inverse_std,
                                         const float *weight_gradient,
                                         const float *bias_gradient, float *output);

/* The training forward and backward as two launches each, for callers that schedule (or
 * time) the phases themselves.  The reduce phase writes per-slice fp64 partial sums to the
 * workspace; the second phase finalizes each channel from them (every block sums the same
 * partials in the same order, so all derive identical values) and streams the elementwise pass.
 *   forward_reduce: partial sums of x per channel (reads x once)
 *   forward_apply:  mean, 1/sqrt(var + eps), running update (evaluation.rs:537-558, in place on
 *                   running_*), saved mean / inverse std, and y (reads x, writes y)
 *   backward_reduce: partial sums of g and g * x_hat per channel (reads g, x)
 *   backward_input:  weight / bias gradients and the training-mode input gradient
 *                    (reads g, x, writes dx) */
oxh_status oxh_batch_norm_forward_reduce(oxh_stream stream, uint64_t batch, uint64_t channels,
                                         uint64_t spatial, const float *input, void *workspace,
                                         uint64_t workspace_bytes);
oxh_status oxh_batch_norm_forward_apply(oxh_stream stream, uint64_t batch, uint64_t channels,
                                        uint64_t spatial, float momentum, float epsilon,
                                        const float *input, const float *weight,
                                        const float *bias, float *running_mean,
                                        float *running_variance, float *saved_mean,
                                        float *saved_inverse_std, float *output,
                                        const void *workspace, uint64_t workspace_bytes);
oxh_status oxh_batch_norm_backward_reduce(oxh_stream stream, uint64_t batch, uint64_t channels,
                                          uint64_t spatial, const float *gradient,
                                          const float *input, const float *saved_mean,
                                          const float *saved_inverse_std, void *workspace,
                                          uint64_t workspace_bytes);
oxh_status oxh_batch_norm_backward_input(oxh_stream stream, uint64_t batch, uint64_t channels,
                                         uint64_t spatial, const float *gradient,
                                         const float *input, const float *weight,
                                         const float *saved_mean,
                                         const float *saved_inverse_std, float *input_gradient,
                                         float *weight_gradient, float *bias_gradient,
                                         const void *workspace, uint64_t workspace_bytes);
/* Training forward = forward_reduce + forward_apply: the reference's statistics +
 * update_running + apply sequence of runtime.rs:571-663 in two launches.  running_mean /
 * running_variance are updated in place; the saved mean / inverse std are written for the
 * backward pass. */
oxh_status oxh_batch_norm_forward_train(oxh_stream stream, uint64_t batch, uint64_t channels,
                                        uint64_t spatial, float momentum, float epsilon,
                                        const float *input, const float *weight,
                                        const float *bias, float *running_mean,
                                        float *running_variance, float *saved_mean,
                                        float *saved_inverse_std, float *output, void *workspace,
                                        uint64_t workspace_bytes);
/* No counterpart in the reference: oxh_batch_norm_forward_train without the workspace
 * argument, for callers that cannot allocate (code under hipGraph capture, tight serving loops,
 * harnesses that forbid hipMalloc).  The reduce partials live in a static device array of
 * OXH_BN_NO_ALLOC_SCRATCH_BYTES (1 MiB) per GPU, held until the process ends; that covers every
 * shape the batch-norm entry points accept (at most 65 535 channels, 16 bytes of partials per
 * channel beyond 2048 channels), and a shape needing more is rejected with OXH_INVALID_SHAPE
 * before any launch.  Calls that
 * overlap on one GPU share that array and race; `stream` must belong to the current device.
 * Same kernels, same results as oxh_batch_norm_forward_train. */
#define OXH_BN_NO_ALLOC_SCRATCH_BYTES (1u << 20)
oxh_status oxh_batch_norm_forward_train_no_alloc(oxh_stream stream, uint64_t batch,
                                                 uint64_t channels, uint64_t spatial,
                                                 float momentum, float epsilon,
                                                 const float *input, const float *weight,
                                                 const float *bias, float *running_mean,
                                                 float *running_variance, float *saved_mean,
                                                 float *saved_inverse_std, float *output);
/* Training backward = backward_reduce + backward_input: the channel sums (sum g,
 * sum g * x_hat) are formed once and feed both dweight / dbias and dx. */
oxh_status oxh_batch_norm_backward_train(oxh_stream stream, uint64_t batch, uint64_t channels,
                                         uint64_t spatial, const float *gradient,
                                         const float *input, const float *weight,
                                         const float *saved_mean,
                                         const float *saved_inverse_std, float *input_gradient,
                                         float *weight_gradient, float *bias_gradient,
                                         void *workspace, uint64_t workspace_bytes);

/* BatchNorm2d followed by ReLU, as ConvNormAct composes them (nn.rs:376-385; ReLU
 * kernel_module.rs:26-34), in the launches of the training forward: `output` = relu(batch
 * norm(input)); the batch-norm output itself is not stored. */
oxh_status oxh_batch_norm_relu_forward_train(oxh_stream stream, uint64_t batch,
                                             uint64_t channels, uint64_t spatial, float momentum,
                                             float epsilon, const float *input,
                                             const float *weight, const float *bias,
                                             float *running_mean, float *running_variance,
                                             float *saved_mean, float *saved_inverse_std,
                                             float *output, void *workspace,
                                             uint64_t workspace_bytes);
/* Backward of the above: `gradient` is w.r.t. the ReLU output and `output` is that forward
 * output; the ReLU backward (kernel_module.rs:501-508: gradient where the ReLU input is
 * positive -- exactly where its output is) is applied on the fly, then the training backward. */
oxh_status oxh_batch_norm_relu_backward_train(oxh_stream stream, uint64_t batch,
                                              uint64_t channels, uint64_t spatial,
                                              const float *gradient, const float *output,
                                              const float *input, const float *weight,
                                              const float *saved_mean,
                                              const float *saved_inverse_std,
                                              float *input_gradient, float *weight_gradient,
                                              float *bias_gradient, void *workspace,
                                              uint64_t workspace_bytes);
/* Training forward of a BatchNorm2d followed by a residual add (a MobileNetV4 block's last
 * ConvNormAct plus its shortcut, mobilenet_v4.rs UIB / IB blocks): `output` = batch norm(input)
 * + addend, each element's normalized value rounded to fp32 before the add, as the separate
 * forward and add launches compute it; the batch-norm output itself is not stored (its
 * training backward does not read it).  `addend` must not overlap `output`.  No single
 * counterpart in the reference (batch_norm forward, then add). */
oxh_status oxh_batch_norm_add_forward_train(oxh_stream stream, uint64_t batch, uint64_t channels,
                                            uint64_t spatial, float momentum, float epsilon,
                                            const float *input, const float *weight,
                                            const float *bias, float *running_mean,
                                            float *running_variance, float *saved_mean,
                                            float *saved_inverse_std, const float *addend,
                                            float *output, void *workspace,
                                            uint64_t workspace_bytes);
/* Training backward of a BatchNorm2d whose input is a convolution's output (ConvNormAct,
 * nn.rs:376-385), optionally through the following ReLU (`relu_output` = that forward output,
 * or NULL for none), that also writes `conv_bias_gradient`[c] = sum over (n, y, x) of
 * input_gradient -- the convolution's bias gradient (autograd.rs:412-527's bias term) -- in
 * the same pass when planes are small.  Other outputs as oxh_batch_norm_backward_train /
 * oxh_batch_norm_relu_backward_train.  No single counterpart in the reference: it replaces
 * the BatchNorm backward plus the convolution's separate bias reduction (the
 * conv2d_backward bias sum over the same gradient) for callers that schedule both. */
oxh_status oxh_conv_batch_norm_backward_train(
    oxh_stream stream, uint64_t batch, uint64_t channels, uint64_t spatial,
    const float *gradient, const float *relu_output, const float *input, const float *weight,
    const float *saved_mean, const float *saved_inverse_std, float *input_gradient,
    float *weight_gradient, float *bias_gradient, float *conv_bias_gradient, void *workspace,
    uint64_t workspace_bytes);

/* ------------------------------------------------------------------ cross entropy
 * kernel_module.rs:966-1050; driver runtime.rs:338-357,828-848; CPU evaluation.rs:599-636,
 * autograd.rs:529-554.  Targets are class indices stored as fp32 (tensor/mod.rs:300-307).
 * A target that is not a finite non-negative integer below `classes` makes the loss (forward)
 * or that row of the gradient (backward) NaN, as the reference's kernels do, and sets
 * *error_flag (a device uint32, may be NULL) to 1 so the caller can raise the CPU path's
 * Error::InvalidShape (evaluation.rs:622-636). */
oxh_status oxh_cross_entropy_workspace_size(uint64_t batch, uint64_t classes, uint64_t *bytes);
/* loss[0] = mean over rows of (log(sum exp(x - max)) + max - x[target]) */
oxh_status oxh_cross_entropy_forward(oxh_stream stream, uint64_t batch, uint64_t classes,
                                     const float *logits, const float *targets, float *loss,
                                     uint32_t *error_flag, void *workspace,
                                     uint64_t workspace_bytes);
/* grad = outer_gradient[0] / batch * (softmax(x) - onehot(target)); outer_gradient is a
 * device scalar (runtime.rs:835-844 passes the upstream gradient buffer). */
oxh_status oxh_cross_entropy_backward(oxh_stream stream, uint64_t batch, uint64_t classes,
                                      const float *logits, const float *targets,
                                      const float *outer_gradient, float *grad,
                                      uint32_t *error_flag);
/* Loss and gradient in one read of the logits (the loss is the backward root, so the
 * upstream gradient is already known). */
oxh_status oxh_cross_entropy_forward_backward(oxh_stream stream, uint64_t batch,
                                              uint64_t classes, const float *logits,
                                              const float *targets,
                                              const float *outer_gradient, float *loss,
                                              float *grad, uint32_t *error_flag,
                                              void *workspace, uint64_t workspace_bytes);

/* ------------------------------------------------------------------ AdamW
 * kernel_module.rs:1094-1127; driver runtime.rs:1306-1386; CPU optim.rs:98-125.
 *   m' = b1*m + (1-b1)*g;  v' = b2*v + (1-b2)*g*g
 *   p' = p - lr * ((m'/c1) / (sqrt(v'/c2) + eps) + wd*p)
 * c1 = 1 - b1^t and c2 = 1 - b2^t are passed in, computed by the caller as optim.rs:91-92
 * does (oxh_adamw_corrections gives the reference's powi values).  Outputs may equal the
 * inputs (in-place update).  fp32, bit-exact with the CPU path. */
oxh_status oxh_adamw(oxh_stream stream, float learning_rate, float weight_decay, float beta1,
                     float beta2, float first_correction, float second_correction, float epsilon,
                     const float *parameter, const float *gradient, const float *first_moment,
                     const float *second_moment, float *new_parameter, float *new_first_moment,
                     float *new_second_moment, uint64_t n);
/* c1 = 1 - beta1.powi(step), c2 = 1 - beta2.powi(step) with Rust's powi (binary
 * exponentiation, reciprocal for negative exponents). */
oxh_status oxh_adamw_corrections(float beta1, float beta2, int32_t step, float *first_correction,
                                 float *second_correction);

/* One launch over many parameter tensors (in place), for a training step that updates every
 * parameter of a model (optim.rs:140-152 visits them one by one). */
typedef struct oxh_adamw_tensor {
  float *parameter;
  const float *gradient;
  float *first_moment;
  float *second_moment;
  uint64_t n;
} oxh_adamw_tensor;
oxh_status oxh_adamw_multi_tensor(oxh_stream stream, float learning_rate, float weight_decay,
                                  float beta1, float beta2, float first_correction,
                                  float second_correction, float epsilon,
                                  const oxh_adamw_tensor *tensors, uint32_t count);

/* Step-counting variant for a captured training step: launches a one-thread kernel that
 * increments *step (a device int32, the optimizer step counter of optim.rs:140-152), then the
 * multi-tensor update with c1 = 1 - beta1.powi(*step), c2 = 1 - beta2.powi(*step) formed on the
 * device with the same powi as oxh_adamw_corrections, so every replay of a graph uses the right
 * bias corrections. */
oxh_status oxh_adamw_multi_tensor_step(oxh_stream stream, float learning_rate,
                                       float weight_decay, float beta1, float beta2,
                                       float epsilon, int32_t *step,
                                       const oxh_adamw_tensor *tensors, uint32_t count);

/* The step-counting multi-tensor update for any number of tensors in one update launch (after
 * a one-thread launch that advances the step counter), for callers that keep the tensor table
 * on the device (a captured training step):
 *   oxh_adamw_table_layout fills chunk_starts[0..count] (host memory; the first chunk of each
 *   tensor and the total) for a host copy of the table; the caller copies the table and the
 *   starts to device memory once.
 *   oxh_adamw_multi_tensor_table_step stores t = *step + 1 in *step and updates every tensor
 *   with step t.  Launches sharing a step counter must be ordered (one stream).
 * No single counterpart in the reference (its optimizer loops over parameters, optim.rs:98-152). */
oxh_status oxh_adamw_table_layout(const oxh_adamw_tensor *tensors, uint32_t count,
                                  uint32_t *chunk_starts, uint64_t *total_chunks);
oxh_status oxh_adamw_multi_tensor_table_step(oxh_stream stream, float learning_rate,
                                             float weight_decay, float beta1, float beta2,
                                             float epsilon, int32_t *step,
                                             const oxh_adamw_tensor *device_tensors,
                                             const uint32_t *device_chunk_starts,
                                             uint32_t count, uint64_t total_chunks);

/* ------------------------------------------------------------------ conv2d / avg_pool2d
 * The layers around the hot path that a MobileNetV4-Conv-S training step needs.  Reference
 * kernels kernel_module.rs:359-490,558-825; CPU semantics evaluation.rs:334-445,
 * autograd.rs:412-527.  NCHW fp32, weight OIHW [out, in/groups, kh, kw], square stride and
 * padding (Conv2d::new uses padding = kernel / 2, nn.rs:236-274).  Both pooling directions add
 * their terms in the CPU path's order (bit-identical), and so do the input gradient unless
 * oxh_conv2d_input_backward_serial says otherwise and the forward unless
 * oxh_conv2d_forward_serial says otherwise (where the CPU path skips a tap outside the input,
 * the small-plane K x K kernels add the product of a +0 operand, which for finite operands
 * changes at most the sign of an exactly zero sum).  A forward whose serial grid would leave
 * most of the chip idle (pointwise with at least 256 input channels and fewer than 512 32x32
 * output tiles; ungrouped 3x3 / 5x5 with output planes of at most 64 positions and at least 16
 * input channels), and a pointwise input gradient with at least 256 output channels and fewer
 * than 512 32x32 tiles, sum four contiguous parts of the reduced channels and add the parts in
 * order; ungrouped 1x1, 3x3 and 5x5 layers over larger planes, or of over 2^27 products, sum on
 * the matrix cores where that is the faster kernel (the two queries below tell).  Those sums, and
 * the weight and bias gradients (fixed-order chunks), are deterministic and within a few roundings
 * (1e-5 * sum|terms|) of the serial sum; their products are added by fused multiply-adds (one
 * rounding per term), on the matrix cores (fp32 MFMA) for the split tiles, the 32x32
 * weight-gradient tiles, the large 1x1 and KxK layers and ungrouped KxK weight gradients. */
typedef struct oxh_conv2d_shape {
  uint64_t batch, in_channels, height, width;
  uint64_t out_channels, kernel_h, kernel_w;
  uint64_t stride, padding, groups;
} oxh_conv2d_shape;
/* 1: oxh_conv2d_forward sums each output in the CPU path's order (bit-identical); 0: in another
 * fixed order (four ordered parts over the input channels, or matrix-core sums), within
 * 1e-5 * sum|terms| of the CPU path's; -1: an invalid shape. */
int oxh_conv2d_forward_serial(const oxh_conv2d_shape *shape);
/* The same for the input gradient (oxh_conv2d_input_backward, _accumulate and the input
 * gradient of oxh_conv2d_backward): 0 when it sums four ordered parts over the output channels
 * (pointwise) or on the matrix cores (stride-2 K x K, large layers).  No counterpart in the
 * reference (its CPU path has one order). */
int oxh_conv2d_input_backward_serial(const oxh_conv2d_shape *shape);
oxh_status oxh_conv2d_output_size(const oxh_conv2d_shape *shape, uint64_t *out_h,
                                  uint64_t *out_w);
/* conv2d (kernel_module.rs:359-448) */
oxh_status oxh_conv2d_forward(oxh_stream stream, const oxh_conv2d_shape *shape,
                              const float *input, const float *weight, const float *bias,
                              float *output);
/* conv2d_input_backward (kernel_module.rs:558-658) */
oxh_status oxh_conv2d_input_backward(oxh_stream stream, const oxh_conv2d_shape *shape,
                                     const float *gradient, const float *weight,
                                     float *input_gradient);
/* input_gradient = conv2d_input_backward(gradient, weight) + addend, each element's sum
 * finished before the add: the gradient accumulation of an input with a second consumer
 * (runtime.rs:671-692's a + b) in the same pass.  No single counterpart in the reference (its
 * autograd runs the input backward, then the accumulation).  `addend` may equal
 * `input_gradient` (accumulate in place) but not overlap it partially; `input_gradient` may
 * not overlap `gradient` or `weight` (OXH_INVALID_SHAPE). */
oxh_status oxh_conv2d_input_backward_accumulate(oxh_stream stream,
                                                const oxh_conv2d_shape *shape,
                                                const float *gradient, const float *weight,
                                                const float *addend, float *input_gradient);
/* Workspace for the weight gradient reduction (0 bytes when a single pass suffices). */
oxh_status oxh_conv2d_weight_backward_workspace_size(const oxh_conv2d_shape *shape,
                                                     uint64_t *bytes);
/* conv2d_weight_backward (kernel_module.rs:660-752) */
oxh_status oxh_conv2d_weight_backward(oxh_stream stream, const oxh_conv2d_shape *shape,
                                      const float *gradient, const float *input,
                                      float *weight_gradient, void *workspace,
                                      uint64_t workspace_bytes);
/* conv2d_bias_backward (kernel_module.rs:754-778); single pass: the workspace arguments are
 * accepted for symmetry with the weight gradient and unused (may be null / 0). */
oxh_status oxh_conv2d_bias_backward(oxh_stream stream, const oxh_conv2d_shape *shape,
                                    const float *gradient, float *bias_gradient,
                                    void *workspace, uint64_t workspace_bytes);
/* The whole backward of one convolution (the conv VJP of runtime.rs, which issues
 * conv2d_weight_backward, conv2d_bias_backward and conv2d_input_backward,
 * kernel_module.rs:558-778): weight_gradient and input_gradient as the separate entry points
 * form them, bias_gradient too when not NULL, input_gradient = sum + addend when addend is not
 * NULL (addend may equal input_gradient, as oxh_conv2d_input_backward_accumulate).  Results are
 * bit-identical to the separate calls; for pointwise convolutions whose two products are small
 * both run in one launch, with the bias gradient's reduction.  input_gradient may be NULL (then
 * addend must be NULL): the parameter gradients only, the weight gradient bit-identical to
 * oxh_conv2d_weight_backward; the bias gradient is then summed in the weight gradient's own
 * launches where its per-image kernels take the shape (ungrouped 3x3 / 5x5: the same
 * fixed-order chunks, within 1e-5 * sum|terms| of the serial sum), else as
 * oxh_conv2d_bias_backward.  The workspace is oxh_conv2d_weight_backward_workspace_size bytes.
 * No gradient may overlap the operands or another gradient, and the addend may not overlap
 * weight_gradient, bias_gradient, the workspace or a part of input_gradient
 * (OXH_INVALID_SHAPE). */
oxh_status oxh_conv2d_backward(oxh_stream stream, const oxh_conv2d_shape *shape,
                               const float *gradient, const float *input, const float *weight,
                               const float *addend, float *input_gradient,
                               float *weight_gradient, float *bias_gradient, void *workspace,
                               uint64_t workspace_bytes);

/* A depthwise ConvNormAct (nn.rs:362-395 with groups == channels: conv2d, BatchNorm2d in
 * training mode, optional ReLU) in ONE launch per direction, for small planes.  Output channel
 * c of a depthwise convolution reads only input channel c, and the BatchNorm reduces over
 * channel c only, so one workgroup per channel runs the whole layer.  No single counterpart
 * in the reference: each replaces the separate launches (conv2d, batch_norm_statistics /
 * update_running / apply, relu forward; relu / batch_norm backward, conv2d input, weight and
 * bias backward) with bit-identical results, except that the weight gradient's fixed-order
 * sums use the 256-thread order of oxh_conv2d_weight_backward (its 1024-thread order for at
 * most 128 channels with at least 1024 output values per channel, which such layers run in
 * 1024-thread blocks; those blocks group the BatchNorm's fp64 partial sums differently from
 * the 256-thread channel kernels, the same after rounding to fp32 unless a sum lies within fp64
 * rounding of an fp32 rounding boundary).
 * Eligible shapes (oxh_depthwise_conv_batch_norm_supported returns 1): groups ==
 * in_channels == out_channels, square 3x3 or 5x5 kernel, stride 1 or 2,
 * batch * out_h * out_w <= 2048 and batch * height * width <= 8192; other shapes return
 * OXH_INVALID_SHAPE. */
int oxh_depthwise_conv_batch_norm_supported(const oxh_conv2d_shape *shape);
/* Forward: conv_output = conv2d(input, conv_weight, conv_bias) (stored: the backward reads
 * it); output = relu?(batch_norm(conv_output)) with momentum / epsilon, saved statistics and
 * the running update as oxh_batch_norm_forward_train. */
oxh_status oxh_depthwise_conv_batch_norm_forward_train(
    oxh_stream stream, const oxh_conv2d_shape *shape, int relu, float momentum, float epsilon,
    const float *input, const float *conv_weight, const float *conv_bias, float *conv_output,
    const float *bn_weight, const float *bn_bias, float *running_mean, float *running_variance,
    float *saved_mean, float *saved_inverse_std, float *output);
/* Backward from `gradient` (of the layer output; masked by `relu_output` > 0 when relu_output
 * is not NULL): bn_weight_gradient / bn_bias_gradient as oxh_batch_norm_backward_train; the
 * BatchNorm's input gradient g_c (written to conv_output_gradient unless NULL); from g_c the
 * convolution's bias gradient (per-channel sum), weight gradient and input gradient
 * (input_gradient = conv2d_input_backward(g_c) + addend when addend is not NULL, as
 * oxh_conv2d_input_backward_accumulate; input_gradient NULL: not formed). */
oxh_status oxh_depthwise_conv_batch_norm_backward_train(
    oxh_stream stream, const oxh_conv2d_shape *shape, const float *gradient,
    const float *relu_output, const float *conv_output, const float *bn_weight,
    const float *saved_mean, const float *saved_inverse_std, const float *input,
    const float *conv_weight, const float *addend, float *conv_output_gradient,
    float *bn_weight_gradient, float *bn_bias_gradient, float *conv_bias_gradient,
    float *conv_weight_gradient, float *input_gradient);

/* A BatchNorm2d in training mode (optionally followed by ReLU) whose only consumer is a
 * depthwise ConvNormAct, run inside that layer's launches: channel c of the depthwise input is
 * channel c of the BatchNorm, so one workgroup per channel forms the BatchNorm's statistics,
 * its output (stored: pre_output, the convolution's input) and the depthwise layer, and in the
 * backward the layer's input gradient feeds the BatchNorm's channel backward in registers.
 * Results equal the separate oxh_batch_norm{,_relu}_forward_train /
 * oxh_depthwise_conv_batch_norm_forward_train calls (and their backward counterparts), with the
 * same BatchNorm arithmetic.  pre_residual (may be NULL; not with pre_relu): the BatchNorm's
 * output plus it (a residual add whose first operand is the BatchNorm) is the convolution's
 * input.  In the backward, addend (may be NULL, may equal conv_input_gradient) holds the
 * convolution input's other gradient contributions: the BatchNorm backward runs on the whole
 * gradient, the layer's input gradient + addend, which conv_input_gradient (may be NULL)
 * receives.  pre_input_gradient is the BatchNorm's dx; pre_input_gradient_sum (may be NULL)
 * its per-channel sum, the bias gradient of a convolution feeding the BatchNorm.  Eligible
 * shapes (oxh_batch_norm_depthwise_conv_batch_norm_supported returns 1): those of the
 * depthwise layer with batch * height * width between 2 and 2048. */
int oxh_batch_norm_depthwise_conv_batch_norm_supported(const oxh_conv2d_shape *shape);
oxh_status oxh_batch_norm_depthwise_conv_batch_norm_forward_train(
    oxh_stream stream, const oxh_conv2d_shape *shape, int pre_relu, float pre_momentum,
    float pre_epsilon, const float *pre_input, const float *pre_weight, const float *pre_bias,
    const float *pre_residual, float *pre_running_mean, float *pre_running_variance,
    float *pre_saved_mean, float *pre_saved_inverse_std, float *pre_output, int relu,
    float momentum, float epsilon,
    const float *conv_weight, const float *conv_bias, float *conv_output,
    const float *bn_weight, const float *bn_bias, float *running_mean, float *running_variance,
    float *saved_mean, float *saved_inverse_std, float *output);
oxh_status oxh_batch_norm_depthwise_conv_batch_norm_backward_train(
    oxh_stream stream, const oxh_conv2d_shape *shape, const float *gradient,
    const float *relu_output, const float *conv_output, const float *bn_weight,
    const float *saved_mean, const float *saved_inverse_std, const float *conv_input,
    const float *conv_weight, const float *addend, int pre_relu, const float *pre_input,
    const float *pre_weight, const float *pre_saved_mean, const float *pre_saved_inverse_std,
    float *conv_output_gradient, float *bn_weight_gradient, float *bn_bias_gradient,
    float *conv_bias_gradient, float *conv_weight_gradient, float *conv_input_gradient,
    float *pre_weight_gradient, float *pre_bias_gradient, float *pre_input_gradient,
    float *pre_input_gradient_sum);

typedef struct oxh_pool2d_shape {
  uint64_t batch, channels, height, width;
  uint64_t kernel_h, kernel_w, stride_h, stride_w;
} oxh_pool2d_shape;
/* avg_pool2d (kernel_module.rs:450-490); global_avg_pool2d is kernel = stride = H x W. */
oxh_status oxh_avg_pool2d_forward(oxh_stream stream, const oxh_pool2d_shape *shape,
                                  const float *input, float *output);
/* avg_pool2d_backward (kernel_module.rs:780-825) */
oxh_status oxh_avg_pool2d_backward(oxh_stream stream, const oxh_pool2d_shape *shape,
                                   const float *gradient, float *input_gradient);

/* Host-side deterministic variance-scaled init of an OIHW conv weight (nn.rs:657-674):
 * xorshift64 (13, 7, 17) seeded from the shape, 24-bit uniforms scaled to
 * [-sqrt(2 / fan_in), sqrt(2 / fan_in)). `out` is host memory of shape[0..4] product floats. */
oxh_status oxh_initialized_weights(const uint64_t shape[4], uint64_t input_channels_per_group,
                                   float *out);

/* ------------------------------------------------------------------ argmax
 * mnist_training.rs:201-218 count_correct: per row index of the maximum under total order,
 * the last index winning ties (Iterator::max_by). */
oxh_status oxh_argmax_rows(oxh_stream stream, uint64_t rows, uint64_t classes,
                           const float *logits, uint32_t *indices);

/* ------------------------------------------------------------------ OXTR checkpoints
 * MobileNetV4ConvSmall::save / load_mnist's file format (mobilenet_v4.rs:217-264,386-428):
 * "OXTR\x01", u64 count, then per tensor u64 rank, rank x u64 dims, u64 len, len x f32, all
 * little-endian.  Host memory only; the model's parameters (visit order) then its BatchNorm
 * running mean / variance pairs.  Errors: unreadable / unwritable file, bad magic ("invalid
 * OXTR checkpoint header") or a truncated file -> OXH_EXECUTION, as the reference. */
typedef struct oxh_checkpoint_tensor {
  uint64_t rank;
  const uint64_t *shape;
  uint64_t len;
  const float *data;
} oxh_checkpoint_tensor;
typedef struct oxh_checkpoint oxh_checkpoint;
oxh_status oxh_checkpoint_save(const char *path, const oxh_checkpoint_tensor *tensors,
                               uint64_t count);
oxh_status oxh_checkpoint_load(const char *path, oxh_checkpoint **checkpoint);
oxh_status oxh_checkpoint_count(const oxh_checkpoint *checkpoint, uint64_t *count);
/* Views into the loaded checkpoint, valid until oxh_checkpoint_free. */
oxh_status oxh_checkpoint_entry(const oxh_checkpoint *checkpoint, uint64_t index,
                                 uint64_t *rank, const uint64_t **shape, uint64_t *len,
                                 const float **data);
oxh_status oxh_checkpoint_free(oxh_checkpoint *checkpoint);

/* ------------------------------------------------------------------ MNIST IDX data
 * data/mnist.rs: the four canonical uncompressed IDX files.  Parsing / validation
 * (mnist.rs:145-183) and loading (26-49) fail with OXH_EXECUTION and the reference's messages;
 * oxh_mnist_batch_order is MnistBatches' index order (0..count-1, shuffled by
 * deterministic_shuffle, mnist.rs:191-199, when `shuffle`); oxh_mnist_batch_host builds a
 * batch on the host ((pixel / 255 - 0.1307) / 0.3081 in fp32, labels as fp32,
 * mnist.rs:103-133); oxh_mnist_gather_batch does the same on the device from a split's bytes
 * resident in device memory and device uint32 indices (an index >= count yields a NaN image
 * and label; nothing is read out of bounds). */
typedef struct oxh_mnist oxh_mnist;
oxh_status oxh_idx_parse_images(const uint8_t *bytes, uint64_t len, uint64_t *count);
oxh_status oxh_idx_parse_labels(const uint8_t *bytes, uint64_t len, uint64_t *count);
oxh_status oxh_mnist_load(const char *directory, oxh_mnist **mnist);
oxh_status oxh_mnist_free(oxh_mnist *mnist);
/* Host views of a split (test = 0: train, 1: t10k): `count` images of 784 bytes, labels. */
oxh_status oxh_mnist_split(const oxh_mnist *mnist, int test, const uint8_t **images,
                           const uint8_t **labels, uint64_t *count);
oxh_status oxh_mnist_batch_order(uint64_t count, int shuffle, uint64_t *indices);
oxh_status oxh_mnist_batch_host(const uint8_t *images, const uint8_t *labels, uint64_t count,
                                const uint64_t *indices, uint64_t batch, float *out_images,
                                float *out_labels);
oxh_status oxh_mnist_gather_batch(oxh_stream stream, const uint8_t *images, const uint8_t *labels,
                                  uint64_t count, const uint32_t *indices, uint64_t batch,
                                  float *out_images, float *out_labels);

/* ------------------------------------------------------------------ graphs
 * CudaGraphExec (cuda_graph.rs:47-179): capture on one stream in thread-local mode, end +
 * instantiate, replay, destroy.  A failed capture is ended and discarded so the stream stays
 * usable (cuda_graph.rs:84-97). */
typedef struct oxh_graph oxh_graph;
oxh_status oxh_graph_begin(oxh_stream stream);
oxh_status oxh_graph_end(oxh_stream stream, oxh_graph **graph);
oxh_status oxh_graph_abort(oxh_stream stream);
oxh_status oxh_graph_launch(const oxh_graph *graph, oxh_stream stream);
oxh_status oxh_graph_destroy(oxh_graph *graph);

/* ------------------------------------------------------------------ MobileNetV4-Conv-S
 * The model of mobilenet_v4.rs:84-321 (modules nn.rs:107-655) with its parameters and
 * BatchNorm running statistics resident on the current device, the training step of
 * examples/mnist_training.rs:75-92 as a native executor, and the inference-mode forward.
 *
 * A trainer traces forward + cross entropy + backward + AdamW (betas 0.9 / 0.999, eps 1e-8,
 * optim.rs:54-76) once into a fixed list of launches over buffers carved from one device
 * allocation made at creation, and runs it eagerly (oxh_program_run) or as one captured
 * hipGraph (oxh_program_capture, then oxh_program_replay per step).  The caller fills the
 * images [batch, channels, res, res] and labels [batch] buffers (oxh_trainer_buffers; e.g.
 * with oxh_mnist_gather_batch) on the program's stream before each step.  An evaluator runs the
 * forward with BatchNorm from the running statistics (evaluation.rs:560-575) and argmax
 * predictions (count_correct, mnist_training.rs:201-218).  The model's parameters are shared
 * by its trainers and evaluators; a model must outlive them. */
typedef struct oxh_model oxh_model;
typedef struct oxh_trainer oxh_trainer;
typedef struct oxh_evaluator oxh_evaluator;
typedef struct oxh_program oxh_program;

/* MobileNetV4ConvSmall::build (mobilenet_v4.rs:111-175): MNIST is (10, 1, 28), the
 * supplement's network (num_classes, 3, 224).  Deterministic init as nn.rs:236-274,657-674. */
oxh_status oxh_mnv4_create(uint64_t num_classes, uint64_t input_channels,
                           uint64_t input_resolution, oxh_model **model);
/* Host-only description: parameter tensors / values, BatchNorm layers, and every block's
 * output shape for `batch` images (forward_with_shapes, mobilenet_v4.rs:182-195; the last is
 * the reshaped [batch, classes, 1, 1]); `block_shapes` holds `capacity` x 4 values. */
oxh_status oxh_mnv4_describe(uint64_t num_classes, uint64_t input_channels,
                             uint64_t input_resolution, uint64_t batch, uint64_t *parameters,
                             uint64_t *values, uint64_t *batch_norms, uint64_t *block_shapes,
                             uint64_t capacity, uint64_t *blocks);
oxh_status oxh_model_destroy(oxh_model *model);
oxh_status oxh_model_info(const oxh_model *model, uint64_t *parameters, uint64_t *batch_norms,
                          uint64_t *values, int *training);
/* Parameter `index` in visit order (per conv: weight, bias; per BatchNorm: gamma, beta). */
oxh_status oxh_model_parameter(const oxh_model *model, uint64_t index, uint64_t *rank,
                               uint64_t shape[4], float **device_values);
oxh_status oxh_model_batch_norm(const oxh_model *model, uint64_t index, uint64_t *channels,
                                float **running_mean, float **running_variance);
/* ModuleMode::set_training; a trainer requires a model in training mode. */
oxh_status oxh_model_set_training(oxh_model *model, int training);
/* save (mobilenet_v4.rs:217-264), after copying the device state to the host
 * (sync_batch_norm_state, runtime.rs:1268-1304). */
oxh_status oxh_model_save(oxh_model *model, const char *path);
/* load_mnist (mobilenet_v4.rs:266-321): too few / extra tensors -> OXH_EXECUTION, a tensor of
 * another shape -> OXH_INVALID_SHAPE; the model is returned in inference mode. */
oxh_status oxh_model_load_mnist(const char *path, oxh_model **model);

/* AdamW::new(learning_rate, weight_decay) validation as optim.rs:54-65. */
oxh_status oxh_trainer_create(oxh_model *model, uint64_t batch, float learning_rate,
                              float weight_decay, oxh_trainer **trainer);
oxh_status oxh_trainer_destroy(oxh_trainer *trainer);
oxh_status oxh_trainer_buffers(const oxh_trainer *trainer, float **images, float **labels,
                               float **logits, float **loss);
oxh_status oxh_trainer_program(oxh_trainer *trainer, oxh_program **program);
/* Waits for the step, then the loss; OXH_INVALID_SHAPE if a label was not a class index
 * (evaluation.rs:622-636; the kernels of that step already ran with a NaN row). */
oxh_status oxh_trainer_loss(oxh_trainer *trainer, float *loss);
oxh_status oxh_trainer_steps(oxh_trainer *trainer, int32_t *steps);

oxh_status oxh_evaluator_create(oxh_model *model, uint64_t batch, oxh_evaluator **evaluator);
oxh_status oxh_evaluator_destroy(oxh_evaluator *evaluator);
oxh_status oxh_evaluator_buffers(const oxh_evaluator *evaluator, float **images,
                                 float **logits, uint32_t **predictions);
oxh_status oxh_evaluator_program(oxh_evaluator *evaluator, oxh_program **program);
/* argmax of each logits row into `predictions` (ties to the last index), enqueued. */
oxh_status oxh_evaluator_predict(oxh_evaluator *evaluator);

/* A program's launch list, open to inspection so each launch group can be checked against
 * an independent implementation: a group's kind and name, the tensors it reads (access 0),
 * writes (1) or updates in place (2) with their roles, shapes and types (dtype 0 f32, 1 i32),
 * and its scalar arguments. */
typedef struct oxh_op_tensor {
  const char *role;
  void *data;
  uint64_t shape[4];
  uint32_t rank;
  int access;
  int dtype;
} oxh_op_tensor;
typedef struct oxh_op_attr {
  const char *name;
  double value;
} oxh_op_attr;
typedef struct oxh_op_info {
  const char *kind, *name;
  uint32_t tensor_count;
  const oxh_op_tensor *tensors;
  uint32_t attr_count;
  const oxh_op_attr *attrs;
} oxh_op_info;
oxh_status oxh_program_stream(const oxh_program *program, oxh_stream *stream);
/* Enqueues every launch group once (eager).  The whole program (run, or captured and replayed)
 * may move work between groups without changing any value: a training program ending with
 * AdamW sums its convolutions' weight-gradient chunks in the optimizer group's first launch.
 * oxh_program_run_op launches one group alone, which then forms every output it lists. */
oxh_status oxh_program_run(oxh_program *program);
oxh_status oxh_program_capture(oxh_program *program);
oxh_status oxh_program_replay(oxh_program *program);
oxh_status oxh_program_op_count(const oxh_program *program, uint64_t *count);
oxh_status oxh_program_op(const oxh_program *program, uint64_t index, oxh_op_info *info);
oxh_status oxh_program_run_op(oxh_program *program, uint64_t index);
/* Waits for the program's stream; OXH_INVALID_SHAPE (and the flag cleared) if a cross entropy
 * met a target that is not a class index since the last check (evaluation.rs:622-636). */
oxh_status oxh_program_check(oxh_program *program);
/* The optimizer's device step counter after the enqueued work (0 without AdamW). */
oxh_status oxh_program_steps(oxh_program *program, int32_t *steps);

/* ------------------------------------------------------------------ traced graphs (nets)
 * The lazy graph the reference's Tensor ops build (tensor/graph.rs:70-139 Op; builders
 * tensor/mod.rs:103-389 with their shape rules and error kinds), recorded node by node: node
 * indices are creation order, which is topological.  Leaves: inputs (device buffers owned by
 * the program, written by the caller before each run; an input may require a gradient, as a
 * Data tensor does), trainable parameters and constants (caller-owned device values, ranks
 * 1..4).  A BatchNorm2d holds its running statistics as caller-owned device vectors, updated in
 * place by a training-mode forward (BatchNormState, graph.rs:47-54).
 * Programs built from a net:
 *   forward  -- the eager device evaluation of `output` (runtime.rs:125-379): every ancestor
 *               in creation order; training-mode BatchNorm uses and updates batch statistics,
 *               eval mode the running ones; Reshape aliases its input (jit.rs:345).  This is
 *               what a JIT plan with operations the fused-plan compiler cannot take runs
 *               (CompiledPlan::Eager, jit.rs:205-207,226-243).
 *   training -- the forward, then reverse mode from the one-element `root` (backward,
 *               runtime.rs:1198-1217: reverse topological order over the root's ancestors,
 *               collect_topological 1388-1476, propagate_node 694-860, each value's first
 *               gradient contribution written and later ones accumulated, 671-692), then, with
 *               an AdamW configuration, one AdamW launch over every trainable parameter the
 *               root reaches (optim.rs:78-152; a device step counter keeps the bias
 *               corrections right under graph replay).  A root that is not one element fails
 *               with OXH_EXECUTION (tensor/mod.rs:399-404).
 * Programs own their buffers and stream, are inspected and run with the oxh_program_* calls
 * above, and are released with oxh_program_destroy.  A net may be destroyed once its programs
 * are built; the caller's parameter, constant and running-statistic buffers must outlive them. */
typedef struct oxh_net oxh_net;
typedef struct oxh_adamw_config {
  float learning_rate, weight_decay, beta1, beta2, epsilon;
} oxh_adamw_config;
oxh_status oxh_net_create(oxh_net **net);
oxh_status oxh_net_destroy(oxh_net *net);
oxh_status oxh_net_node_count(const oxh_net *net, uint32_t *count);
oxh_status oxh_net_node_shape(const oxh_net *net, uint32_t node, uint32_t *rank,
                              uint64_t shape[4]);
/* Tensor::placeholder / from_vec leaves (tensor/mod.rs:45-48,520-522). */
oxh_status oxh_net_input(oxh_net *net, uint32_t rank, const uint64_t *shape, int requires_grad,
                         uint32_t *node);
/* nn::Parameter (nn.rs:35-80): trainable, updated in place by the program's AdamW. */
oxh_status oxh_net_parameter(oxh_net *net, uint32_t rank, const uint64_t *shape, float *values,
                             uint32_t *node);
oxh_status oxh_net_constant(oxh_net *net, uint32_t rank, const uint64_t *shape,
                            const float *values, uint32_t *node);
/* Tensor::add / mul (tensor/mod.rs:103-116, equal shapes), relu (118-122), reshape (293-301). */
oxh_status oxh_net_add(oxh_net *net, uint32_t a, uint32_t b, uint32_t *node);
oxh_status oxh_net_mul(oxh_net *net, uint32_t a, uint32_t b, uint32_t *node);
oxh_status oxh_net_relu(oxh_net *net, uint32_t x, uint32_t *node);
oxh_status oxh_net_reshape(oxh_net *net, uint32_t x, uint32_t rank, const uint64_t *shape,
                           uint32_t *node);
/* Tensor::conv2d (tensor/mod.rs:158-237): NCHW x, OIHW weight, [out] bias, square kernel. */
oxh_status oxh_net_conv2d(oxh_net *net, uint32_t x, uint32_t weight, uint32_t bias,
                          uint64_t stride, uint64_t padding, uint64_t groups, uint32_t *node);
/* Tensor::avg_pool2d (tensor/mod.rs:239-272). */
oxh_status oxh_net_avg_pool2d(oxh_net *net, uint32_t x, uint64_t kernel_h, uint64_t kernel_w,
                              uint64_t stride_h, uint64_t stride_w, uint32_t *node);
/* Tensor::batch_norm2d (tensor/mod.rs:331-389): momentum in [0, 1] and epsilon > 0, both
 * finite, else OXH_EXECUTION. */
oxh_status oxh_net_batch_norm2d(oxh_net *net, uint32_t x, uint32_t weight, uint32_t bias,
                                float *running_mean, float *running_variance, int training,
                                float momentum, float epsilon, uint32_t *node);
/* Tensor::cross_entropy (tensor/mod.rs:303-329): [batch, classes] logits, [batch] targets
 * holding class indices as f32; a one-element loss (the batch mean). */
oxh_status oxh_net_cross_entropy(oxh_net *net, uint32_t logits, uint32_t targets,
                                 uint32_t *node);
oxh_status oxh_net_forward_program(const oxh_net *net, uint32_t output, oxh_program **program);
/* adamw NULL: forward + backward only (the gradients stay in the program's buffers). */
oxh_status oxh_net_training_program(const oxh_net *net, uint32_t root,
                                    const oxh_adamw_config *adamw, oxh_program **program);
/* Device buffer of a node's value in the program (inputs: where to write them). */
oxh_status oxh_program_value(const oxh_program *program, uint32_t node, float **device);
/* Device buffer of a node's gradient after a training program ran (Tensor::grad,
 * tensor/mod.rs:429-444); NULL when the node receives none. */
oxh_status oxh_program_gradient(const oxh_program *program, uint32_t node, float **device);
/* Releases a program built by oxh_net_*_program (a trainer's or evaluator's program belongs
 * to it: OXH_INVALID_SHAPE). */
oxh_status oxh_program_destroy(oxh_program *program);

/* ------------------------------------------------------------------ JIT plans
 * CudaJitPlan (cuda/jit.rs:10-99) over the reference's GraphPlan (jit.rs:24-56): buffers are
 * inputs, constants or workspaces; operations read earlier buffers and write one buffer.
 * compile allocates every buffer on the device, uploads constants, captures the operation list
 * into a graph on a dedicated stream and instantiates it; run copies the inputs in, replays
 * and copies the output out; replay only enqueues the graph (device-resident inputs). */
typedef struct oxh_plan oxh_plan;
enum oxh_plan_op {
  OXH_PLAN_ADD = 1,  /* out = in0 + in1          (PlanOperation::Add) */
  OXH_PLAN_MUL = 2,  /* out = in0 * in1          (PlanOperation::Mul) */
  OXH_PLAN_RELU = 3, /* out = relu(in0)          (PlanOperation::Relu) */
  OXH_PLAN_RELU_BACKWARD = 4, /* out = in1 > 0 ? in0 : 0 */
  OXH_PLAN_MUL_BACKWARD = 5,  /* out = in0 * in1 */
  OXH_PLAN_ACCUMULATE = 6     /* out = in0 + in1 */
};
oxh_status oxh_plan_create(int device, oxh_plan **plan);
oxh_status oxh_plan_add_input(oxh_plan *plan, uint64_t elements, uint32_t *slot);
oxh_status oxh_plan_add_constant(oxh_plan *plan, const float *values, uint64_t elements,
                                 uint32_t *slot);
oxh_status oxh_plan_add_workspace(oxh_plan *plan, uint64_t elements, uint32_t *slot);
oxh_status oxh_plan_add_operation(oxh_plan *plan, uint32_t op, const uint32_t *inputs,
                                  uint32_t input_count, uint32_t output);
oxh_status oxh_plan_set_output(oxh_plan *plan, uint32_t slot);
/* Allocates the buffers, records the operations into a graph.  A run of operations each
 * consuming the previous one's result (and reading no buffer an earlier one of the run wrote)
 * becomes one kernel with the same per-element results; a workspace read only inside its run
 * is never written (oxh_plan_buffer then shows its initial zeros). */
oxh_status oxh_plan_compile(oxh_plan *plan);
/* host_inputs[i] holds the elements of the i-th input slot in creation order. */
oxh_status oxh_plan_run(oxh_plan *plan, const float *const *host_inputs, uint32_t input_count,
                        float *host_output, uint64_t output_elements);
/* One hipGraphLaunch of the compiled plan (cuda/jit.rs:86-97 without the copies). */
oxh_status oxh_plan_replay(oxh_plan *plan);
/* No single reference counterpart: the launches the plan's graph holds, issued directly on the
 * plan's stream (a fully fused plan is one kernel launch, without the graph launch's cost). */
oxh_status oxh_plan_launch(oxh_plan *plan);
oxh_status oxh_plan_stream(const oxh_plan *plan, oxh_stream *stream);
oxh_status oxh_plan_buffer(const oxh_plan *plan, uint32_t slot, float **device_pointer,
                           uint64_t *elements);
oxh_status oxh_plan_destroy(oxh_plan *plan);

#ifdef __cplusplus
}
#endif
#endif /* OXIDE_HIP_H */
