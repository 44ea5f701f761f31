// Training loss for gfx950: mean negative log-likelihood of the log-softmax over the training rows
// (F.nll_loss(F.log_softmax(out, 1)[mask], y[mask]), EPPGCN/gcn_main.py:252-253) and its gradient.
//
// A row of classes belongs to a team of TEAM lanes, 64 / TEAM rows to a step of a wave: 4 lanes up to 16 classes, 16 up to 64,
// else the whole wave.  Each lane keeps its first K columns in registers (4, or 16 from 257 classes on), so that a row of up
// to TEAM * K classes is read once; its maximum and its sum of exponentials are team reductions.
//   forward    a wave takes a stretch of the training rows: their ids and labels in one load each, then a step per 64 / TEAM
//              rows; sums per workgroup in double, added in a fixed order by a second kernel
//   backward   a wave takes a stretch of the rows of the gradient: the rows between training rows are cleared with 16-byte
//              stores, the training rows' elements are softmax minus the label's one, times d_loss / rows - each element is
//              written once.  The label's element is p * s - s in one fused multiply-add, as torch rounds it: (p - 1) * s
//              rounds twice, a 2-norm error against 64 bits of 5.11e-8 instead of 4.82e-8 (5826 rows of 22 classes), which
//              the first Adam steps, close to a sign, pass on enlarged
// As torch operations the two were 14 launches of 2 to 5 us (log-softmax, gather, mean and negation of the selected rows;
// backward three fills, a scatter and an index_add) of a two-layer epoch; now 4 of its 17 (12 us).  What bounds them:
// launches for small graphs, the write of the gradient for large ones (4.1 to 4.8 TB/s).  2^22 rows of 22 classes, a tenth of
// them in training: 31 + 124 us, with torch's operations 260; 2^20 rows of 172, a hundredth: 10 + 150 and 176; 2^20 rows of
// 1000, a tenth: 91 + 1026 and 1721.  (A team per row, one row after another: 114 + 337, 11 + 286 and 667 + 2870.)
#include "common.hpp"

namespace eppgcn {

constexpr int kLossBlock = 256;
constexpr int kLossWaves = kLossBlock / kWave;
constexpr int kMaxLossBlocks = 8192;       // workgroups of the forward pass (its partial sums)
constexpr int kMeanBlock = 512;

template <int TEAM>
__device__ __forceinline__ float team_max(float v)
{
#pragma unroll
    for (int off = TEAM / 2; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, TEAM));
    return v;
}
template <int TEAM>
__device__ __forceinline__ float team_sum(float v)
{
#pragma unroll
    for (int off = TEAM / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, TEAM);
    return v;
}

// Logarithm as torch rounds it.  Under hipcc's default (contract = fast) logf() expands to a form with 6.3e-8 of relative
// error (2-norm, arguments 1 to 31); without contraction, which has to be said where the builtin is called, it is 5.7e-8.
__device__ __forceinline__ float log_uncontracted(float v)
{
#pragma clang fp contract(off)
    return __builtin_logf(v);
}

// Maximum of a row and logarithm of the sum of its exponentials relative to that maximum; v receives the lane's first K
// columns tl, tl + TEAM, ...  The sum is the one of 64 lanes with a column each (more columns: each lane its own, ascending,
// first), added in halves, whatever the team size.  That keeps the longest chain of additions at dim / 64 + 6 (one running sum
// per lane of a team of 16: dim / 16 + 4, which at 1000 classes gave the gradient a third more error than torch's), and up to
// 1024 classes it has torch's rounding.
template <int TEAM, int K>
__device__ __forceinline__ void row_norm(const float* __restrict__ x, int dim, int tl, float (&v)[K], float* top, float* log_sum)
{
    static_assert(TEAM == kWave || K == 4, "smaller teams add their four columns in halves and hold all of a row");
    float m = -INFINITY;
#pragma unroll
    for (int j = 0; j < K; ++j) v[j] = tl + j * TEAM < dim ? x[tl + j * TEAM] : -INFINITY;
#pragma unroll
    for (int j = 0; j < K; ++j) m = fmaxf(m, v[j]);
    if constexpr (TEAM == kWave)
        for (long long d = tl + K * TEAM; d < dim; d += TEAM) m = fmaxf(m, x[d]);
    m = team_max<TEAM>(m);
    float e[K];
#pragma unroll
    for (int j = 0; j < K; ++j) e[j] = tl + j * TEAM < dim ? expf(v[j] - m) : 0.f;
    float s;
    if constexpr (TEAM == kWave) {
        s = e[0];
#pragma unroll
        for (int j = 1; j < K; ++j) s += e[j];
        for (long long d = tl + K * TEAM; d < dim; d += TEAM) s += expf(x[d] - m);
    } else {
        s = (e[0] + e[2]) + (e[1] + e[3]);
    }
    *top = m;
    *log_sum = log_uncontracted(team_sum<TEAM>(s));
}

template <int TEAM, int K>
__global__ __launch_bounds__(kLossBlock) void nll_rows_kernel(const float* __restrict__ logits, const long long* __restrict__ rows,
                                                              const int* __restrict__ labels, long long num_rows,
                                                              long long num_nodes, int dim, int stretch,
                                                              double* __restrict__ partial)
{
    __shared__ double s_sum[kLossWaves];
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x / kWave;
    const int tl = lane % TEAM, team = lane / TEAM;
    double sum = 0.0;
    for (long long i0 = (static_cast<long long>(blockIdx.x) * kLossWaves + wave) * stretch; i0 < num_rows;
         i0 += static_cast<long long>(gridDim.x) * kLossWaves * stretch) {
        long long id = lane < stretch && i0 + lane < num_rows ? rows[i0 + lane] : -1;
        if (id >= num_nodes) id = -1;                             // not a row: it adds nothing
        const int label = id >= 0 ? labels[id] : -1;
        for (int r = 0; r < stretch && i0 + r < num_rows; r += kWave / TEAM) {      // the same for the whole wave
            const long long row = __shfl(id, r + team, kWave);
            const int want = __shfl(label, r + team, kWave);
            const float* x = logits + (row >= 0 ? row : 0) * dim;
            float v[K], top, log_sum;
            row_norm<TEAM, K>(x, dim, tl, v, &top, &log_sum);
            if (row < 0) continue;
            if (want < 0 || want >= dim) {
                if (tl == 0) sum = static_cast<double>(NAN);
            } else if (want % TEAM == tl) {                       // the lane that has the label's column
                float at = want >= K * TEAM ? x[want] : 0.f;
#pragma unroll
                for (int j = 0; j < K; ++j) at = want == tl + j * TEAM ? v[j] : at;
                sum += static_cast<double>(log_sum - (at - top));
            }
        }
    }
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) sum += __shfl_xor(sum, off, kWave);
    if (lane == 0) s_sum[wave] = sum;
    __syncthreads();
    if (threadIdx.x == 0) {
        double all = 0.0;
        for (int w = 0; w < kLossWaves; ++w) all += s_sum[w];
        partial[blockIdx.x] = all;
    }
}

__global__ __launch_bounds__(kMeanBlock) void nll_mean_kernel(const double* __restrict__ partial, int count, long long num_rows,
                                                              float* __restrict__ loss)
{
    __shared__ double s_sum[kMeanBlock];
    double sum = 0.0;
    for (int i = threadIdx.x; i < count; i += kMeanBlock) sum += partial[i];
    s_sum[threadIdx.x] = sum;
    __syncthreads();
    for (int half = kMeanBlock / 2; half > 0; half /= 2) {
        if (static_cast<int>(threadIdx.x) < half) s_sum[threadIdx.x] += s_sum[threadIdx.x + half];
        __syncthreads();
    }
    if (threadIdx.x == 0) *loss = static_cast<float>(s_sum[0] / static_cast<double>(num_rows));   // no rows: NaN, as a mean of nothing is
}

// n zeros from p, by the lanes of a wave: 16-byte stores between the aligned ends
__device__ __forceinline__ void wave_zero(float* __restrict__ p, long long n, int lane)
{
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    const long long head = min(n, static_cast<long long>((16 - reinterpret_cast<uintptr_t>(p) % 16) % 16 / 4));
    const long long vecs = (n - head) / 4;
    f32x4* v = reinterpret_cast<f32x4*>(p + head);
    for (long long i = lane; i < vecs; i += kWave) v[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    const long long tail = head + 4 * vecs;
    if (lane < head) p[lane] = 0.f;
    if (lane < n - tail) p[tail + lane] = 0.f;
}

template <int TEAM, int K>
__global__ __launch_bounds__(kLossBlock) void nll_gradient_kernel(float* __restrict__ grad, const float* __restrict__ d_loss,
                                                                  const float* __restrict__ logits, const int* __restrict__ labels,
                                                                  long long num_rows, long long num_nodes, int dim, int stretch)
{
    const int lane = threadIdx.x & (kWave - 1);
    const int tl = lane % TEAM, team = lane / TEAM;
    const float scale = *d_loss / static_cast<float>(num_rows);
    const long long r0 = (static_cast<long long>(blockIdx.x) * kLossWaves + threadIdx.x / kWave) * stretch;
    if (r0 >= num_nodes) return;
    const int here = static_cast<int>(min(static_cast<long long>(stretch), num_nodes - r0));
    const int label = lane < here ? labels[r0 + lane] : -1;
    const uint64_t marked = __ballot(label >= 0);
    float* g = grad + r0 * dim;
    {   // the rows between the training rows
        uint64_t left = marked;
        for (int a = 0; a < here;) {
            const int b = left ? __builtin_ctzll(left) : here;
            if (b > a) wave_zero(g + static_cast<long long>(a) * dim, static_cast<long long>(b - a) * dim, lane);
            a = b + 1;
            left &= left - 1;
        }
    }
    // lane q gets the q-th training row of the stretch (the lanes behind them the other rows: a permutation)
    const int count = __popcll(marked);
    const int before = ballot_rank(marked);
    const int place = label >= 0 ? before : count + lane - before;
    const int order = __builtin_amdgcn_ds_permute(4 * place, lane);
    for (int q = 0; q < count; q += kWave / TEAM) {               // the same for the whole wave
        const int r = __shfl(order, min(q + team, count - 1), kWave);
        const int want = __shfl(label, r, kWave);
        const float* x = logits + (r0 + r) * dim;
        float v[K], top, log_sum;
        row_norm<TEAM, K>(x, dim, tl, v, &top, &log_sum);
        if (q + team >= count) continue;
        float* out = g + static_cast<long long>(r) * dim;
#pragma unroll
        for (int j = 0; j < K; ++j) {
            const int d = tl + j * TEAM;
            if (d < dim) out[d] = fmaf(expf(v[j] - top - log_sum), scale, d == want ? -scale : 0.f);
        }
        if constexpr (TEAM == kWave)
            for (long long d = tl + K * TEAM; d < dim; d += TEAM)
                out[d] = fmaf(expf(x[d] - top - log_sum), scale, d == want ? -scale : 0.f);
    }
}

size_t nll_workspace_bytes() { return kMaxLossBlocks * sizeof(double); }

// Rows a wave takes: at least a step's, at most one per lane, and as many as leave the chip 8192 waves (32 per CU).
static int loss_stretch(long long rows, int step)
{
    int stretch = step;
    while (stretch < kWave && rows / (2 * stretch) >= 8192) stretch *= 2;
    return stretch;
}

#define EPPGCN_LOSS_BY_CLASSES(LAUNCH_)      \
    do {                                     \
        if (dim <= 16) LAUNCH_(4, 4);        \
        else if (dim <= 64) LAUNCH_(16, 4);  \
        else if (dim <= 256) LAUNCH_(64, 4); \
        else LAUNCH_(64, 16);                \
    } while (0)

int launch_nll_forward(float* loss, const float* logits, const long long* rows, const int* labels, long long num_rows,
                       long long num_nodes, int dim, void* workspace, hipStream_t stream)
{
    double* partial = static_cast<double*>(workspace);
    int blocks = 1;
#define EPPGCN_NLL_ROWS(TEAM_, K_)                                                                                            \
    do {                                                                                                                     \
        const int stretch = loss_stretch(num_rows, kWave / TEAM_);                                                            \
        const long long want = (num_rows + kLossWaves * stretch - 1) / (kLossWaves * stretch);                                \
        blocks = static_cast<int>(want > kMaxLossBlocks ? kMaxLossBlocks : want < 1 ? 1 : want);                              \
        hipLaunchKernelGGL((nll_rows_kernel<TEAM_, K_>), dim3(blocks), dim3(kLossBlock), 0, stream, logits, rows, labels,     \
                           num_rows, num_nodes, dim, stretch, partial);                                                       \
    } while (0)
    EPPGCN_LOSS_BY_CLASSES(EPPGCN_NLL_ROWS);
#undef EPPGCN_NLL_ROWS
    EPPGCN_HIP(hipGetLastError());
    hipLaunchKernelGGL(nll_mean_kernel, dim3(1), dim3(kMeanBlock), 0, stream, partial, blocks, num_rows, loss);
    EPPGCN_HIP(hipGetLastError());
    return kOk;
}

int launch_nll_backward(float* grad, const float* d_loss, const float* logits, const int* labels, long long num_rows,
                        long long num_nodes, int dim, hipStream_t stream)
{
    if (num_nodes == 0) return kOk;
#define EPPGCN_NLL_GRADIENT(TEAM_, K_)                                                                                        \
    do {                                                                                                                     \
        const int stretch = loss_stretch(num_nodes, kWave / TEAM_);                                                           \
        const long long blocks = (num_nodes + kLossWaves * stretch - 1) / (kLossWaves * stretch);                             \
        hipLaunchKernelGGL((nll_gradient_kernel<TEAM_, K_>), dim3(static_cast<unsigned>(blocks)), dim3(kLossBlock), 0, stream, \
                           grad, d_loss, logits, labels, num_rows, num_nodes, dim, stretch);                                  \
    } while (0)
    EPPGCN_LOSS_BY_CLASSES(EPPGCN_NLL_GRADIENT);
#undef EPPGCN_NLL_GRADIENT
    EPPGCN_HIP(hipGetLastError());
    return kOk;
}

}  // namespace eppgcn
