// The small passes of a training step around the network.  Each is a handful of kilobytes of
// work: what they cost is their launch, so each is one launch whatever the depth of the network.
#include "../../include/msd_hip.h"
#include "msd_kernels.h"

#include <algorithm>
#include <cmath>

namespace msd {
namespace {

constexpr int kThreads = 256;

// ---------------------------------------------------------------------------
// Adam (Kingma & Ba, without weight decay), all parameters in one launch.  A network has a
// hundred small tensors (9 to a few thousand values each); one workgroup per tensor walks its
// tensor, so the count of updates of that tensor, where it lives on the device, has one
// reader and one writer.  Depth 100 at two values per line: 7 launches of 4 us each and two
// dozen copies and elementwise launches for the recorded form become one launch of 5 us.
// ---------------------------------------------------------------------------
struct AdamEntry {
    void *p;
    const void *g;
    void *m, *v;
    float *step;               // device counter, or null: the two factors below
    double step_size, root2;   // lr / (1 - beta1^t) and sqrt(1 - beta2^t)
    int count;
};
constexpr int kAdamBatch = 60;   // entries of 64 bytes: within the 4 KB of a kernel's arguments
struct AdamBatch {
    AdamEntry e[kAdamBatch];
};

template <typename T>
__global__ __launch_bounds__(kThreads) void adam_kernel(AdamBatch batch, double lr, double beta1, double beta2, T eps)
{
    const AdamEntry &e = batch.e[blockIdx.x];
    T step_size, root2;
    if (e.step) {
        const double t = (double)*e.step + 1.0;
        step_size = (T)(lr / (1.0 - pow(beta1, t)));
        root2 = (T)sqrt(1.0 - pow(beta2, t));
        __syncthreads();                          // every thread has read the counter
        if (threadIdx.x == 0) *e.step = (float)t;
    } else {
        step_size = (T)e.step_size;
        root2 = (T)e.root2;
    }
    T *p = (T *)e.p, *m = (T *)e.m, *v = (T *)e.v;
    const T *g = (const T *)e.g;
    const T a1 = (T)(1.0 - beta1), a2 = (T)(1.0 - beta2), keep2 = (T)beta2;
    for (int i = threadIdx.x; i < e.count; i += kThreads) {
        const T gi = g[i];
        const T mi = m[i] + (gi - m[i]) * a1;
        const T vi = v[i] * keep2 + gi * gi * a2;
        m[i] = mi;
        v[i] = vi;
        p[i] -= step_size * mi / (sqrt(vi) / root2 + eps);
    }
}

template <typename T>
__global__ __launch_bounds__(kThreads) void scale_fold_kernel(int c_out, int c_in, const T *__restrict__ s,
                                                              const T *__restrict__ shift, const T *__restrict__ w,
                                                              const T *__restrict__ b, T *__restrict__ ow,
                                                              T *__restrict__ ob)
{
    // element (o, c) of S.W (or of S^T.W without a shift); c == c_in stands for the bias
    const int i = blockIdx.x * kThreads + threadIdx.x;
    const int o = i / (c_in + 1), c = i % (c_in + 1);
    if (o >= c_out) return;
    T acc = T(0);
    for (int q = 0; q < c_out; q++) acc += (shift ? s[o * c_out + q] : s[q * c_out + o]) * (c < c_in ? w[q * c_in + c] : b[q]);
    if (c < c_in)
        ow[o * c_in + c] = acc;
    else
        ob[o] = shift ? acc + shift[o] : acc;
}

// Bound by the two atomics of each workgroup, which all go to one line (7 ns each): one workgroup of 16
// waves per compute unit and four labels per lane in flight.  Back to back, launch included: 1024 x 1024 labels 180 us
// with the atomics of 4096 waves, 11 us so; 476 523 labels 144 and 11, 65 536 labels 40 and 6.
constexpr int kLabelThreads = 1024, kLabelGroups = 256, kLabelUnroll = 4;
__global__ __launch_bounds__(kLabelThreads) void label_check_kernel(int64_t n, long long num_labels,
                                                                    const int64_t *__restrict__ labels,
                                                                    int64_t *__restrict__ clamped, long long *range)
{
    __shared__ long long ends[2][kLabelThreads / kWave];
    long long lo = INT64_MAX, hi = INT64_MIN;
    const int64_t stride = (int64_t)gridDim.x * kLabelThreads;
    for (int64_t i = (int64_t)blockIdx.x * kLabelThreads + threadIdx.x; i < n; i += kLabelUnroll * stride) {
        long long v[kLabelUnroll];
#pragma unroll
        for (int u = 0; u < kLabelUnroll; u++) v[u] = labels[i + u * stride < n ? i + u * stride : i];
#pragma unroll
        for (int u = 0; u < kLabelUnroll; u++) {
            lo = v[u] < lo ? v[u] : lo;
            hi = v[u] > hi ? v[u] : hi;
            if (i + u * stride < n) clamped[i + u * stride] = v[u] < 0 ? 0 : (v[u] >= num_labels ? num_labels - 1 : v[u]);
        }
    }
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) {
        const long long l2 = __shfl_xor(lo, off, kWave), h2 = __shfl_xor(hi, off, kWave);
        lo = l2 < lo ? l2 : lo;
        hi = h2 > hi ? h2 : hi;
    }
    if (threadIdx.x % kWave == 0) {
        ends[0][threadIdx.x / kWave] = lo;
        ends[1][threadIdx.x / kWave] = hi;
    }
    __syncthreads();
    if (threadIdx.x != 0) return;
    for (int w = 1; w < kLabelThreads / kWave; w++) {
        lo = ends[0][w] < lo ? ends[0][w] : lo;
        hi = ends[1][w] > hi ? ends[1][w] : hi;
    }
    // (read first: after the first few workgroups hardly any has something to add)
    if (lo < range[0]) atomicMin(&range[0], lo);
    if (hi > range[1]) atomicMax(&range[1], hi);
}

}  // namespace

hipError_t adam_step(bool f64, int n, const msd_adam_param *params, double lr, double beta1, double beta2, double eps,
                     hipStream_t s)
{
    for (int i0 = 0; i0 < n; i0 += kAdamBatch) {
        AdamBatch b;
        const int m = std::min(n - i0, kAdamBatch);
        for (int i = 0; i < m; i++) {
            const msd_adam_param &q = params[i0 + i];
            AdamEntry &e = b.e[i];
            if (q.count > INT32_MAX) return hipErrorInvalidValue;
            e.p = q.param;
            e.g = q.grad;
            e.m = q.exp_avg;
            e.v = q.exp_avg_sq;
            e.step = q.device_step;
            e.count = (int)q.count;
            e.step_size = lr / (1.0 - std::pow(beta1, q.step));
            e.root2 = std::sqrt(1.0 - std::pow(beta2, q.step));
        }
        if (f64)
            hipLaunchKernelGGL(adam_kernel<double>, dim3(m), dim3(kThreads), 0, s, b, lr, beta1, beta2, eps);
        else
            hipLaunchKernelGGL(adam_kernel<float>, dim3(m), dim3(kThreads), 0, s, b, lr, beta1, beta2, (float)eps);
        const hipError_t err = hipGetLastError();
        if (err != hipSuccess) return err;
    }
    return hipSuccess;
}

hipError_t scale_fold(bool f64, int c_out, int c_in, const void *scale, const void *shift, const void *weight,
                      const void *bias, void *folded_weight, void *folded_bias, hipStream_t s)
{
    const dim3 grid((unsigned)((c_out * (int64_t)(c_in + 1) + kThreads - 1) / kThreads));
    if (f64)
        hipLaunchKernelGGL(scale_fold_kernel<double>, grid, dim3(kThreads), 0, s, c_out, c_in, (const double *)scale,
                           (const double *)shift, (const double *)weight, (const double *)bias,
                           (double *)folded_weight, (double *)folded_bias);
    else
        hipLaunchKernelGGL(scale_fold_kernel<float>, grid, dim3(kThreads), 0, s, c_out, c_in, (const float *)scale,
                           (const float *)shift, (const float *)weight, (const float *)bias, (float *)folded_weight,
                           (float *)folded_bias);
    return hipGetLastError();
}

hipError_t label_check(int64_t count, int64_t num_labels, const int64_t *labels, int64_t *clamped, int64_t *range,
                       hipStream_t s)
{
    const unsigned blocks = (unsigned)std::min<int64_t>((count + kLabelThreads - 1) / kLabelThreads, kLabelGroups);
    hipLaunchKernelGGL(label_check_kernel, dim3(blocks), dim3(kLabelThreads), 0, s, count, (long long)num_labels, labels,
                       clamped, (long long *)range);
    return hipGetLastError();
}

}  // namespace msd
