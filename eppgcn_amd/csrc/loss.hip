// Training loss for gfx950: mean negative log-likelihood of the log-softmax over the training rows
// (F.nll_loss(F.log_softmax(out, 1)[mask], y[mask]), EPPGCN/gcn_main.py:252-253) and its gradient.
//
// A row of classes belongs to a team of 16 lanes, 4 rows per wave; its maximum and its sum of exponentials are team
// reductions, the columns are read again from the vector cache instead of being kept (any number of classes).
//   forward    one team per training row; sums per workgroup in double, added in a fixed order by a second kernel
//   backward   one team per row of the gradient: softmax minus the label's one, times d_loss / rows, in training rows,
//              zeros in the others - each element is written once.  The label's element is p * s - s in one fused
//              multiply-add, as torch rounds it: (p - 1) * s rounds twice, a 2-norm error against 64 bits of 5.11e-8 instead
//              of 4.82e-8 (5826 rows of 22 classes), which the first Adam steps, close to a sign, pass on enlarged
// As torch operations the two were 14 launches of 2 to 5 us (log-softmax, gather, mean and negation of the selected rows;
// backward three fills, a scatter and an index_add), most of an epoch on graphs of a few thousand vertices.  What bounds
// them: launches for small graphs, the write of the gradient for large ones.
#include "common.hpp"

namespace eppgcn {

constexpr int kLossBlock = 256;
constexpr int kTeam = 16;
constexpr int kLossTeams = kLossBlock / kTeam;
constexpr int kMaxLossBlocks = 512;

__device__ __forceinline__ float team_max(float v)
{
#pragma unroll
    for (int off = kTeam / 2; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, kTeam));
    return v;
}
__device__ __forceinline__ float team_sum(float v)
{
#pragma unroll
    for (int off = kTeam / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, kTeam);
    return v;
}

// Logarithm as torch rounds it.  Under hipcc's default (contract = fast) logf() expands to a form with 6.3e-8 of relative
// error (2-norm, arguments 1 to 31); without contraction, which has to be said where the builtin is called, it is 5.7e-8.
__device__ __forceinline__ float log_uncontracted(float v)
{
#pragma clang fp contract(off)
    return __builtin_logf(v);
}

// Maximum of a row and logarithm of the sum of its exponentials relative to that maximum.  The sum is the one of 64 lanes
// with a column each (more columns: each lane its own, ascending, first), added in halves - four of them per lane of the
// team.  That keeps the longest chain of additions at dim / 64 + 6 (one running sum per lane of the team: dim / 16 + 4, which
// at 1000 classes gave the gradient a third more error than torch's), and up to 1024 classes it has torch's rounding.
__device__ __forceinline__ void row_norm(const float* __restrict__ x, int dim, int tl, float* top, float* log_sum)
{
    float m = -INFINITY;
    for (int d = tl; d < dim; d += kTeam) m = fmaxf(m, x[d]);
    m = team_max(m);
    float s[4] = {0.f, 0.f, 0.f, 0.f};
    for (int d0 = tl; d0 < dim; d0 += 4 * kTeam) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (d0 + j * kTeam < dim) s[j] += expf(x[d0 + j * kTeam] - m);
    }
    *top = m;
    *log_sum = log_uncontracted(team_sum((s[0] + s[2]) + (s[1] + s[3])));
}

__global__ __launch_bounds__(kLossBlock) void nll_rows_kernel(const float* __restrict__ logits, const long long* __restrict__ rows,
                                                              const int* __restrict__ labels, long long num_rows,
                                                              long long num_nodes, int dim, double* __restrict__ partial)
{
    __shared__ double s_sum[kLossTeams];
    const int tl = threadIdx.x % kTeam, team = threadIdx.x / kTeam;
    double sum = 0.0;
    // the same number of steps for all teams of a wave: the reductions below use all its lanes
    for (long long i0 = static_cast<long long>(blockIdx.x) * kLossTeams; i0 < num_rows;
         i0 += static_cast<long long>(gridDim.x) * kLossTeams) {
        const long long i = i0 + team;
        const long long r = i < num_rows ? rows[i] : -1;
        const bool ok = r >= 0 && r < num_nodes;
        const float* x = logits + (ok ? r : 0) * dim;
        float top, log_sum;
        row_norm(x, dim, tl, &top, &log_sum);
        if (ok && tl == 0) {
            const int label = labels[r];
            sum += label >= 0 && label < dim ? static_cast<double>(log_sum - (x[label] - top)) : static_cast<double>(NAN);
        }
    }
    if (tl == 0) s_sum[team] = sum;
    __syncthreads();
    if (threadIdx.x == 0) {
        double all = 0.0;
        for (int t = 0; t < kLossTeams; ++t) all += s_sum[t];
        partial[blockIdx.x] = all;
    }
}

__global__ __launch_bounds__(kMaxLossBlocks) void nll_mean_kernel(const double* __restrict__ partial, int count,
                                                                  long long num_rows, float* __restrict__ loss)
{
    __shared__ double s_sum[kMaxLossBlocks];
    s_sum[threadIdx.x] = static_cast<int>(threadIdx.x) < count ? partial[threadIdx.x] : 0.0;
    __syncthreads();
    for (int half = kMaxLossBlocks / 2; half > 0; half /= 2) {
        if (static_cast<int>(threadIdx.x) < half) s_sum[threadIdx.x] += s_sum[threadIdx.x + half];
        __syncthreads();
    }
    if (threadIdx.x == 0) *loss = static_cast<float>(s_sum[0] / static_cast<double>(num_rows));   // no rows: NaN, as a mean of nothing is
}

__global__ __launch_bounds__(kLossBlock) void nll_gradient_kernel(float* __restrict__ grad, const float* __restrict__ d_loss,
                                                                  const float* __restrict__ logits, const int* __restrict__ labels,
                                                                  long long num_rows, long long num_nodes, int dim)
{
    const int tl = threadIdx.x % kTeam, team = threadIdx.x / kTeam;
    const float scale = *d_loss / static_cast<float>(num_rows);
    for (long long r0 = static_cast<long long>(blockIdx.x) * kLossTeams; r0 < num_nodes;
         r0 += static_cast<long long>(gridDim.x) * kLossTeams) {
        const long long r = r0 + team;
        const int label = r < num_nodes ? labels[r] : -1;
        const float* x = logits + (r < num_nodes ? r : 0) * dim;
        float top = 0.f, log_sum = 0.f;
        if (__any(label >= 0)) row_norm(x, dim, tl, &top, &log_sum);
        if (r >= num_nodes) continue;
        float* g = grad + r * dim;
        for (int d = tl; d < dim; d += kTeam)
            g[d] = label < 0 ? 0.f : fmaf(expf(x[d] - top - log_sum), scale, d == label ? -scale : 0.f);
    }
}

size_t nll_workspace_bytes() { return kMaxLossBlocks * sizeof(double); }

static unsigned loss_blocks(long long rows, long long most)
{
    const long long blocks = (rows + kLossTeams - 1) / kLossTeams;
    return static_cast<unsigned>(blocks > most ? most : blocks < 1 ? 1 : blocks);
}

int launch_nll_forward(float* loss, const float* logits, const long long* rows, const int* labels, long long num_rows,
                       long long num_nodes, int dim, void* workspace, hipStream_t stream)
{
    double* partial = static_cast<double*>(workspace);
    const unsigned blocks = loss_blocks(num_rows, kMaxLossBlocks);
    hipLaunchKernelGGL(nll_rows_kernel, dim3(blocks), dim3(kLossBlock), 0, stream, logits, rows, labels, num_rows, num_nodes,
                       dim, partial);
    EPPGCN_HIP(hipGetLastError());
    hipLaunchKernelGGL(nll_mean_kernel, dim3(1), dim3(kMaxLossBlocks), 0, stream, partial, static_cast<int>(blocks), num_rows, loss);
    EPPGCN_HIP(hipGetLastError());
    return kOk;
}

int launch_nll_backward(float* grad, const float* d_loss, const float* logits, const int* labels, long long num_rows,
                        long long num_nodes, int dim, hipStream_t stream)
{
    if (num_nodes == 0) return kOk;
    hipLaunchKernelGGL(nll_gradient_kernel, dim3(loss_blocks(num_nodes, 256 * 16)), dim3(kLossBlock), 0, stream, grad, d_loss,
                       logits, labels, num_rows, num_nodes, dim);
    EPPGCN_HIP(hipGetLastError());
    return kOk;
}

}  // namespace eppgcn
