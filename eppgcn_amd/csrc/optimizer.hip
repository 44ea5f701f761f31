// Adam for gfx950: the update of all weights of a model in one launch (torch.optim.Adam(lr=0.01) in EPPGCN/gcn_main.py:209).
//
// A weight matrix of this model holds 96 x 16 or 16 x 22 floats, so a step is launches and host work.  As torch's grouped
// operations a step was eleven launches of 2 to 3 us and 90 to 104 us of host time; an epoch without a wait at its end takes, us,
// before -> with this kernel: 2708 vertices 338 -> 225, 19 717 vertices 337 -> 228, there with four layers of 32 (three live
// models) 771 -> 628.
// Every element is rounded as torch's grouped operations round it (a fused multiply-add where one of them multiplies and
// adds), which is needed: the first steps divide a gradient by its own size, so a weight whose gradient is near zero moves by
// what rounding made of it.  What bounds it: the launch; large weights are streamed (28 bytes per element).
#include "common.hpp"

#include <cmath>

namespace eppgcn {

constexpr int kAdamBlock = 256;
constexpr int kAdamTensors = 32;            // weights of a launch: 32 descriptions are 1.5 KB of kernel arguments
constexpr long long kAdamMaxBlocks = 2048;  // per weight; each strides over the rest

struct AdamWeight {
    float* p;
    const float* g;
    float* m;
    float* v;
    long long n;
    float step_size;        // -lr / (1 - beta1^step)
    float root;             // sqrt(1 - beta2^step)
};
struct AdamWeights {
    AdamWeight w[kAdamTensors];
};

__global__ __launch_bounds__(kAdamBlock) void adam_kernel(AdamWeights all, float one_minus_beta1, float beta2,
                                                          float one_minus_beta2, float eps)
{
    const AdamWeight& w = all.w[blockIdx.y];
    const long long stride = static_cast<long long>(gridDim.x) * kAdamBlock;
    for (long long i = static_cast<long long>(blockIdx.x) * kAdamBlock + threadIdx.x; i < w.n; i += stride) {
#pragma clang fp contract(off)
        const float g = w.g[i];
        const float m = __builtin_fmaf(one_minus_beta1, g - w.m[i], w.m[i]);
        const float decayed = w.v[i] * beta2;
        const float v = __builtin_fmaf(one_minus_beta2, g * g, decayed);
        const float denom = __builtin_sqrtf(v) / w.root + eps;
        w.m[i] = m;
        w.v[i] = v;
        w.p[i] = __builtin_fmaf(w.step_size, m / denom, w.p[i]);
    }
}

int launch_adam(int count, float* const* params, const float* const* grads, float* const* exp_avg, float* const* exp_avg_sq,
                const long long* sizes, const double* steps, double lr, double beta1, double beta2, double eps,
                hipStream_t stream)
{
    for (int at = 0; at < count; at += kAdamTensors) {
        AdamWeights all = {};
        const int take = count - at < kAdamTensors ? count - at : kAdamTensors;
        long long largest = 0;
        for (int k = 0; k < take; ++k) {
            const double c1 = 1.0 - std::pow(beta1, steps[at + k]), c2 = 1.0 - std::pow(beta2, steps[at + k]);
            all.w[k] = {params[at + k], grads[at + k], exp_avg[at + k], exp_avg_sq[at + k], sizes[at + k],
                        static_cast<float>(-(lr / c1)), static_cast<float>(std::pow(c2, 0.5))};
            if (sizes[at + k] > largest) largest = sizes[at + k];
        }
        if (largest == 0) continue;
        long long blocks = (largest + kAdamBlock - 1) / kAdamBlock;
        if (blocks > kAdamMaxBlocks) blocks = kAdamMaxBlocks;
        hipLaunchKernelGGL(adam_kernel, dim3(static_cast<unsigned>(blocks), static_cast<unsigned>(take)), dim3(kAdamBlock), 0,
                           stream, all, static_cast<float>(1.0 - beta1), static_cast<float>(beta2),
                           static_cast<float>(1.0 - beta2), static_cast<float>(eps));
        EPPGCN_HIP(hipGetLastError());
    }
    return kOk;
}

}  // namespace eppgcn
