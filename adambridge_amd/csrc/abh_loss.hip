// abh_loss.hip -- cross-entropy of a slice of logits and its gradient, for causal_lm_loss
// (reference adambridge/losses.py:27-70).
//
// A row of logits is one position's vocabulary (152k BF16 values, 304 KB): the work is reading the
// logits once forward, and once more beside writing the gradient backward, so HBM bounds both.  In
// place of the FP32 copy, the FP32 log-probabilities and their FP32 gradient that the composition
// of library operations passes through memory (about 55 bytes per logit and step against 8 here),
// the logits stay BF16 in memory and FP32 in registers, and what the gradient needs beside them is two
// floats per row: the row's maximum and the reciprocal of its sum of exponentials.  Measured on
// MI355X at 1024 x 151936 BF16 logits: forward 54-59 us (5.3-5.8 TB/s of logits read), where the library's
// FP32 copy and softmax took 141 + 464 us; backward 109-111 us (5.6-5.7 TB/s; 92 where the logits have just
// been read), where its zero-fill, softmax gradient and BF16 copy took 57 + 520 + 156 us.  A training
// pass of 4 such slices with a 896-wide head, one box: torch operations 15.32 ms, these kernels in
// checkpointed slices 8.13, and 6.63 in one function (losses.py: _HeadLoss), of which the head's
// products are 5.4.
//
// Rows are spread over workgroups of 256 lanes, 16 bytes a lane and load.  A call of few rows
// splits each row over several workgroups (ce_splits) so that all 256 CUs read; the partial maxima
// and sums are combined in a fixed order by k_ce_finish, so results do not depend on scheduling.

#include <hip/hip_runtime.h>

#include <stdint.h>

#include <algorithm>

#include "../../include/adambridge_hip.h"
#include "abh_device.hpp"
#include "abh_host.hpp"

namespace abh {

constexpr int kCeThreads = 256;
constexpr int kCeWaves = kCeThreads / 64;
constexpr int kFinishThreads = 1024;
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kNegInf = -__builtin_inff();

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// exp(x - m) for x <= m: the difference first (exact or correctly rounded), then one v_exp_f32.
__device__ __forceinline__ float exp_diff(float x, float m) { return __builtin_amdgcn_exp2f((x - m) * kLog2e); }

// A running maximum and the sum of exp(x - m) over what was seen.  m = -inf: nothing above -inf yet.
struct Soft {
    float m, s;
};

// The subtrahend that stands for a maximum: 0 where it is still -inf, so that exp(-inf - 0) = 0
// instead of exp(-inf + inf) = NaN.
__device__ __forceinline__ float shift_of(float m) { return m == kNegInf ? 0.0f : m; }

__device__ __forceinline__ Soft merge(const Soft a, const Soft b)
{
    const float m = __builtin_fmaxf(a.m, b.m), t = shift_of(m);
    return Soft{m, a.s * exp_diff(a.m, t) + b.s * exp_diff(b.m, t)};
}

template <int K>
__device__ __forceinline__ void take(Soft& a, const float (&x)[K])
{
    float m = a.m;
#pragma unroll
    for (int k = 0; k < K; ++k) m = __builtin_fmaxf(m, x[k]);
    const float t = shift_of(m);
    float s = a.s * exp_diff(a.m, t);
#pragma unroll
    for (int k = 0; k < K; ++k) s += exp_diff(x[k], t);
    a = Soft{m, s};
}

// Values per 16-byte access, and their FP32 form.
template <int DT>
constexpr int kPer = DT == DT_BF16 ? 8 : 4;

template <int DT>
__device__ __forceinline__ void unpack(const u32x4 w, float* x)
{
    const uint32_t u[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        if constexpr (DT == DT_BF16) {
            x[2 * k] = bitsf(u[k] << 16);
            x[2 * k + 1] = bitsf(u[k] & 0xffff0000u);
        } else {
            x[k] = bitsf(u[k]);
        }
    }
}

template <int DT>
__device__ __forceinline__ float load_one(const void* row, int64_t i)
{
    if constexpr (DT == DT_BF16) return bitsf((uint32_t)static_cast<const uint16_t*>(row)[i] << 16);
    else return static_cast<const float*>(row)[i];
}

template <int DT>
__device__ __forceinline__ void store_one(void* row, int64_t i, float x)
{
    if constexpr (DT == DT_BF16) static_cast<uint16_t*>(row)[i] = (uint16_t)bf16_rne(x);
    else static_cast<float*>(row)[i] = x;
}

// A row's values before its first 16-byte boundary (a vocabulary of odd size starts its rows off it).
template <int DT>
__device__ __forceinline__ int64_t head_of(const void* row, int64_t vocab)
{
    constexpr int64_t size = DT == DT_BF16 ? 2 : 4;
    const int64_t head = (int64_t)((16 - ((uintptr_t)row & 15)) & 15) / size;
    return head < vocab ? head : vocab;
}

// Workgroup b: split b % splits of row b / splits.  The row's 16-byte vectors are divided evenly;
// the values before and after them go with the first and the last split.
template <int DT>
__global__ __launch_bounds__(kCeThreads) void k_ce_partial(const void* logits, int64_t vocab, int32_t splits,
                                                           Soft* part)
{
    constexpr int64_t size = DT == DT_BF16 ? 2 : 4;
    constexpr int K = kPer<DT>, U = 4;
    const int64_t row = blockIdx.x / (uint32_t)splits;
    const int32_t split = (int32_t)(blockIdx.x % (uint32_t)splits);
    const uint8_t* base = static_cast<const uint8_t*>(logits) + row * vocab * size;
    const int64_t head = head_of<DT>(base, vocab);
    const int64_t nvec = (vocab - head) / K;
    const u32x4* v = reinterpret_cast<const u32x4*>(base + head * size);
    const int64_t lo = nvec * split / splits, hi = nvec * (split + 1) / splits;
    Soft a{kNegInf, 0.0f};
    int64_t i = lo + threadIdx.x;
    for (; i + (U - 1) * kCeThreads < hi; i += U * kCeThreads) {
        u32x4 w[U];
#pragma unroll
        for (int u = 0; u < U; ++u) w[u] = v[i + u * kCeThreads];
        float x[U * K];
#pragma unroll
        for (int u = 0; u < U; ++u) unpack<DT>(w[u], x + u * K);
        take(a, x);
    }
    for (; i < hi; i += kCeThreads) {
        float x[K];
        unpack<DT>(v[i], x);
        take(a, x);
    }
    if (split == 0 && (int64_t)threadIdx.x < head) {
        const float x[1] = {load_one<DT>(base, threadIdx.x)};
        take(a, x);
    }
    const int64_t tail = head + nvec * K;
    if (split == splits - 1 && tail + threadIdx.x < vocab) {   // at most K - 1 values
        const float x[1] = {load_one<DT>(base, tail + threadIdx.x)};
        take(a, x);
    }
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) a = merge(a, Soft{__shfl_xor(a.m, d), __shfl_xor(a.s, d)});
    __shared__ Soft wave[kCeWaves];
    if ((threadIdx.x & 63) == 0) wave[threadIdx.x >> 6] = a;
    __syncthreads();
    if (threadIdx.x == 0) {
        a = wave[0];
#pragma unroll
        for (int k = 1; k < kCeWaves; ++k) a = merge(a, wave[k]);
        part[blockIdx.x] = a;
    }
}

// One workgroup: each row's partials combined in order, its maximum and reciprocal sum kept for
// the backward pass, and the losses m + log(s) - x[target] summed (lane-strided partial sums, then a
// fixed tree).  An ignored row counts zero; a target outside [0, vocab) gives NaN.
template <int DT>
__global__ __launch_bounds__(kFinishThreads) void k_ce_finish(const void* logits, const int64_t* target, int64_t rows,
                                                              int64_t vocab, int64_t ignore, int32_t splits,
                                                              const Soft* part, float* stats, float* loss)
{
    constexpr int64_t size = DT == DT_BF16 ? 2 : 4;
    float sum = 0.0f;
    for (int64_t r = threadIdx.x; r < rows; r += kFinishThreads) {
        Soft a = part[r * splits];
        for (int32_t k = 1; k < splits; ++k) a = merge(a, part[r * splits + k]);
        if (a.m == kNegInf) a.s = __builtin_nanf("");   // every logit -inf: no distribution
        stats[2 * r] = a.m;
        stats[2 * r + 1] = 1.0f / a.s;
        const int64_t t = target[r];
        if (t == ignore) continue;
        if (t < 0 || t >= vocab) {
            sum = __builtin_nanf("");
            continue;
        }
        const float x = load_one<DT>(static_cast<const uint8_t*>(logits) + r * vocab * size, t);
        sum += logf(a.s) - (x - a.m);
    }
    __shared__ float tree[kFinishThreads];
    tree[threadIdx.x] = sum;
    __syncthreads();
#pragma unroll
    for (int d = kFinishThreads / 2; d > 0; d >>= 1) {
        if ((int)threadIdx.x < d) tree[threadIdx.x] += tree[threadIdx.x + d];
        __syncthreads();
    }
    if (threadIdx.x == 0) loss[0] = tree[0];
}

// grad = (exp(x - m) / s - [k == target]) * gout for a row's values, 0 * that for an ignored row (a NaN
// row stays NaN there, as in the composition this replaces), NaN for a row whose target lies outside
// [0, vocab), as its loss is: an update must not follow a gradient that no loss has.  Workgroups as in
// k_ce_partial.
template <int DT>
__global__ __launch_bounds__(kCeThreads) void k_ce_backward(const void* logits, const int64_t* target, int64_t vocab,
                                                            int64_t ignore, int32_t splits, const float* stats,
                                                            const float* gout, void* grad)
{
    constexpr int64_t size = DT == DT_BF16 ? 2 : 4;
    constexpr int K = kPer<DT>, U = 2;
    const int64_t row = blockIdx.x / (uint32_t)splits;
    const int32_t split = (int32_t)(blockIdx.x % (uint32_t)splits);
    const uint8_t* base = static_cast<const uint8_t*>(logits) + row * vocab * size;
    uint8_t* out = static_cast<uint8_t*>(grad) + row * vocab * size;
    const int64_t t = target[row];
    const float m = stats[2 * row], inv = stats[2 * row + 1];
    const float g = t == ignore ? 0.0f : t < 0 || t >= vocab ? __builtin_nanf("") : gout[0];
    const float f = inv * g;
    const int64_t head = head_of<DT>(base, vocab);
    const int64_t nvec = (vocab - head) / K;
    const u32x4* v = reinterpret_cast<const u32x4*>(base + head * size);
    u32x4* o = reinterpret_cast<u32x4*>(out + head * size);
    auto value = [&](float x, int64_t k) {
        const float p = exp_diff(x, m) * f;
        return k == t ? p - g : p;
    };
    auto vector = [&](const u32x4 w, int64_t i) {
        float x[K];
        unpack<DT>(w, x);
        const int64_t k0 = head + i * K;
#pragma unroll
        for (int k = 0; k < K; ++k) x[k] = exp_diff(x[k], m) * f;
        const int64_t at = t - k0;   // the target's place among these, if any
        if (at >= 0 && at < K) {
#pragma unroll
            for (int k = 0; k < K; ++k) x[k] = k == at ? x[k] - g : x[k];
        }
        u32x4 r;
        if constexpr (DT == DT_BF16)
            r = u32x4{bf16x2_rne(x[0], x[1]), bf16x2_rne(x[2], x[3]), bf16x2_rne(x[4], x[5]), bf16x2_rne(x[6], x[7])};
        else
            r = u32x4{fbits(x[0]), fbits(x[1]), fbits(x[2]), fbits(x[3])};
        __builtin_nontemporal_store(r, o + i);
    };
    const int64_t lo = nvec * split / splits, hi = nvec * (split + 1) / splits;
    int64_t i = lo + threadIdx.x;
    for (; i + (U - 1) * kCeThreads < hi; i += U * kCeThreads) {
        u32x4 w[U];
#pragma unroll
        for (int u = 0; u < U; ++u) w[u] = v[i + u * kCeThreads];
#pragma unroll
        for (int u = 0; u < U; ++u) vector(w[u], i + u * kCeThreads);
    }
    for (; i < hi; i += kCeThreads) vector(v[i], i);
    if (split == 0 && (int64_t)threadIdx.x < head)
        store_one<DT>(out, threadIdx.x, value(load_one<DT>(base, threadIdx.x), threadIdx.x));
    const int64_t tail = head + nvec * K;
    if (split == splits - 1 && tail + threadIdx.x < vocab)
        store_one<DT>(out, tail + threadIdx.x, value(load_one<DT>(base, tail + threadIdx.x), tail + threadIdx.x));
}

// Workgroups per row: enough for 8 of them on each of the 256 CUs, while each still has 4 loads a
// lane (8192 BF16 values); one once the rows alone give that many.
static int32_t ce_splits(int64_t rows, int64_t vocab)
{
    const int64_t want = (2048 + rows - 1) / rows, most = std::max<int64_t>(1, vocab / 8192);
    return (int32_t)std::min<int64_t>(std::min(want, most), 64);
}

// rows * splits workgroups of 256 lanes stay within one dispatch's 2^32 - 1 work-items.
constexpr int64_t kCeMaxRows = (int64_t)1 << 23;

static int ce_check(const void* logits, int32_t dtype, const void* target, int64_t rows, int64_t vocab,
                    const void* grad)
{
    if (rows < 1 || vocab < 1 || rows > kCeMaxRows) return ADAMBRIDGE_EBADN;
    if (dtype != DT_F32 && dtype != DT_BF16) return ADAMBRIDGE_EMVDTYPE;
    if (!logits || !target) return ADAMBRIDGE_ENULL;
    const uintptr_t size = dtype == DT_F32 ? 4 : 2;
    if ((uintptr_t)logits % size || ((uintptr_t)grad - (uintptr_t)logits) % 16) return ADAMBRIDGE_EALIGN;
    return 0;
}

}  // namespace abh

using namespace abh;

extern "C" {

ADAMBRIDGE_API int64_t adambridge_cross_entropy_work(int64_t rows, int64_t vocab)
{
    if (rows < 1 || vocab < 1 || rows > kCeMaxRows) return ADAMBRIDGE_EBADN;
    return rows * ce_splits(rows, vocab) * (int64_t)sizeof(Soft);
}

ADAMBRIDGE_API int adambridge_cross_entropy(const void* logits, int32_t dtype, const int64_t* target, int64_t rows,
                                            int64_t vocab, int64_t ignore_index, void* work, float* stats,
                                            float* loss)
{
    const int rc = ce_check(logits, dtype, target, rows, vocab, logits);
    if (rc) return rc;
    if (!work || !stats || !loss) return ADAMBRIDGE_ENULL;
    const int32_t splits = ce_splits(rows, vocab);
    Soft* part = static_cast<Soft*>(work);
    const dim3 grid((unsigned)(rows * splits));
    if (dtype == DT_BF16) {
        hipLaunchKernelGGL(k_ce_partial<DT_BF16>, grid, dim3(kCeThreads), 0, t_stream, logits, vocab, splits, part);
        hipLaunchKernelGGL(k_ce_finish<DT_BF16>, dim3(1), dim3(kFinishThreads), 0, t_stream, logits, target, rows, vocab,
                           ignore_index, splits, part, stats, loss);
    } else {
        hipLaunchKernelGGL(k_ce_partial<DT_F32>, grid, dim3(kCeThreads), 0, t_stream, logits, vocab, splits, part);
        hipLaunchKernelGGL(k_ce_finish<DT_F32>, dim3(1), dim3(kFinishThreads), 0, t_stream, logits, target, rows, vocab,
                           ignore_index, splits, part, stats, loss);
    }
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : hip_fail(e, "hipLaunchKernelGGL (cross entropy)");
}

ADAMBRIDGE_API int adambridge_cross_entropy_backward(const void* logits, int32_t dtype, const int64_t* target,
                                                     int64_t rows, int64_t vocab, int64_t ignore_index,
                                                     const float* stats, const float* gout, void* grad)
{
    const int rc = ce_check(logits, dtype, target, rows, vocab, grad);
    if (rc) return rc;
    if (!stats || !gout || !grad) return ADAMBRIDGE_ENULL;
    const int32_t splits = ce_splits(rows, vocab);
    const dim3 grid((unsigned)(rows * splits));
    if (dtype == DT_BF16)
        hipLaunchKernelGGL(k_ce_backward<DT_BF16>, grid, dim3(kCeThreads), 0, t_stream, logits, target, vocab,
                           ignore_index, splits, stats, gout, grad);
    else
        hipLaunchKernelGGL(k_ce_backward<DT_F32>, grid, dim3(kCeThreads), 0, t_stream, logits, target, vocab,
                           ignore_index, splits, stats, gout, grad);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : hip_fail(e, "hipLaunchKernelGGL (cross entropy backward)");
}

}  // extern "C"
