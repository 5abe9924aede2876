// abh_gemm.hip -- C = A B for a long inner dimension and a small result: the hidden states' gradient of a
// language-model head, [positions x vocabulary] times [vocabulary x hidden] (BF16, FP32 sums).
//
// A result of 1024 x 896 is 28 tiles for 256 CUs while the inner dimension has 152k terms, so the work is
// split there: tiles x splits fill the chip's 512 places (two workgroups a CU), each split's FP32 sums
// go to memory and are added in order and rounded once.  The splits follow each other through the
// XCDs' workgroups, so the tiles that share a split's slices of A and B run on one XCD at a time and
// find them in its L2.  Bound by the matrix cores and the LDS reads that feed them.
//
// Tile 256 x 128 of 4 wavefronts, each 128 x 64 in 4 x 2 MFMAs of 32 x 32 x 16 (6 KB of LDS reads for
// 8 of them; 64 x 64 a wavefront would read 8 KB for 4 and be bound by the LDS).  A step of 64 terms is
// loaded to registers while the one before is multiplied.  B's rows are turned on the way to the
// LDS: a lane's 8 rows x 4 columns become 4 entries of 8 terms by 16 byte permutes, and column n goes to
// slot n / 4 + 32 (n mod 4), so that both the writes and the reads of 32 lanes are contiguous (the MFMA's
// column i of tile t is column 4 i + t of the result).
//
// Measured on MI355X, us, the library's product beside it: 1024 x 896 over 151936 terms 346-359 (777-805
// TFLOP/s; 318 within a training pass) against 619; 333 x 896 196 / 451; 1024 x 4096 1346 / 1793; over 50264 terms 1024 x 2048 283 /
// 484.  512 places are best (256: 508, 1024: 440); fragments read one step ahead, a raised wave priority
// and the other order of tiles changed nothing (345-354).  The caller's rule (losses.py: _matmul_into): 2^14
// terms or more, at most 4096 rows and 2^22 results (below 2^15 terms 2^21); beyond, the library is as fast
// or faster (4096 x 2048: 2635 / 1865, 8192 x 512: 1460 / 1354, over 8192 terms 1024 x 896 39 / 44).

#include <hip/hip_runtime.h>

#include <stdint.h>

#include <algorithm>

#include "../../include/adambridge_hip.h"
#include "abh_device.hpp"
#include "abh_host.hpp"

namespace abh {

constexpr int kMmThreads = 256;
constexpr int kBM = 256, kBN = 128, kBK = 64;
constexpr int kRowPad = 2;
constexpr int kXcdCount = 8;

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

struct MmArgs {
    const uint16_t* a;   // m x k
    const uint16_t* b;   // k x n
    float* part;         // splits x m x n
    int64_t k;
    int32_t m, n;
    int32_t tiles_m, tiles_n, splits, ksteps;
};

__global__ __launch_bounds__(kMmThreads, 2) void k_mm_split(MmArgs A)
{
    __shared__ u32x4 la[8 * (kBM + kRowPad)];   // [k / 8][row], 8 values of k each
    __shared__ u32x4 lb[8 * kBN];               // [k / 8][slot]: column n at slot n / 4 + 32 (n mod 4)
    const int total = A.tiles_m * A.tiles_n * A.splits;
    const int per = (total + kXcdCount - 1) / kXcdCount;
    const int idx = (int)(blockIdx.x % kXcdCount) * per + (int)(blockIdx.x / kXcdCount);
    if ((int)(blockIdx.x / kXcdCount) >= per || idx >= total) return;
    const int tiles = A.tiles_m * A.tiles_n;
    const int split = idx / tiles, tile = idx % tiles;
    const int m0 = (tile % A.tiles_m) * kBM, n0 = (tile / A.tiles_m) * kBN;
    const int s0 = (int)((int64_t)A.ksteps * split / A.splits), s1 = (int)((int64_t)A.ksteps * (split + 1) / A.splits);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int half = lane >> 5, col = lane & 31;
    const int wm = wave & 1, wn = wave >> 1;

    // this thread's loads: A rows tid / 8 + 32 r, values 8 (tid mod 8) on; B rows 8 (tid / 32) + j, columns
    // 4 (tid mod 32) on
    const int ar = tid >> 3, ac = tid & 7, bk = tid >> 5, bn = (tid & 31) * 4;
    const int nb = n0 + bn <= A.n - 4 ? n0 + bn : A.n - 4;   // past the end: any valid columns, not stored
    const uint16_t* pa = A.a + (int64_t)m0 * A.k;
    int32_t ao[8];   // rows past the end: the last one again, not stored
#pragma unroll
    for (int r = 0; r < 8; ++r) {
        const int row = m0 + ar + 32 * r < A.m ? ar + 32 * r : A.m - 1 - m0;
        ao[r] = row * (int32_t)A.k + ac * 8;
    }
    const uint16_t* pb = A.b + (int64_t)(bk * 8) * A.n + nb;
    u32x4 ga[8];
    u32x2 gb[8];
    auto fetch = [&](int s) {
        const int64_t k0 = (int64_t)s * kBK;
        if (k0 + kBK <= A.k) {
#pragma unroll
            for (int r = 0; r < 8; ++r) ga[r] = *reinterpret_cast<const u32x4*>(pa + k0 + ao[r]);
#pragma unroll
            for (int j = 0; j < 8; ++j) gb[j] = *reinterpret_cast<const u32x2*>(pb + (k0 + j) * A.n);
        } else {   // the last step: zeros past k
#pragma unroll
            for (int r = 0; r < 8; ++r)
                ga[r] = k0 + ac * 8 + 8 <= A.k ? *reinterpret_cast<const u32x4*>(pa + k0 + ao[r]) : u32x4{0u, 0u, 0u, 0u};
#pragma unroll
            for (int j = 0; j < 8; ++j)
                gb[j] = k0 + bk * 8 + j < A.k ? *reinterpret_cast<const u32x2*>(pb + (k0 + j) * A.n) : u32x2{0u, 0u};
        }
    };
    f32x16 acc[4][2];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

    if (s0 < s1) fetch(s0);
    for (int s = s0; s < s1; ++s) {
#pragma unroll
        for (int r = 0; r < 8; ++r) la[ac * (kBM + kRowPad) + ar + 32 * r] = ga[r];
        // 8 rows x 4 columns of B turned: column c's 8 values of k, pairs of rows by byte permutes
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const uint32_t sel = (c & 1) ? 0x07060302u : 0x05040100u;
            u32x4 w;
            w.x = __builtin_amdgcn_perm(c < 2 ? gb[1].x : gb[1].y, c < 2 ? gb[0].x : gb[0].y, sel);
            w.y = __builtin_amdgcn_perm(c < 2 ? gb[3].x : gb[3].y, c < 2 ? gb[2].x : gb[2].y, sel);
            w.z = __builtin_amdgcn_perm(c < 2 ? gb[5].x : gb[5].y, c < 2 ? gb[4].x : gb[4].y, sel);
            w.w = __builtin_amdgcn_perm(c < 2 ? gb[7].x : gb[7].y, c < 2 ? gb[6].x : gb[6].y, sel);
            lb[bk * kBN + 32 * c + (tid & 31)] = w;
        }
        __syncthreads();
        if (s + 1 < s1) fetch(s + 1);
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) {
            const int k8 = 2 * kk + half;
            bf16x8 fa[4], fb[2];
#pragma unroll
            for (int i = 0; i < 4; ++i)
                fa[i] = __builtin_bit_cast(bf16x8, la[k8 * (kBM + kRowPad) + wm * 128 + 32 * i + col]);
#pragma unroll
            for (int j = 0; j < 2; ++j) fb[j] = __builtin_bit_cast(bf16x8, lb[k8 * kBN + 32 * (2 * wn + j) + col]);
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i], fb[j], acc[i][j], 0, 0, 0);
        }
        __syncthreads();
    }
    // the two columns 4 col + 2 wn, + 1 of each row
    const int n = n0 + 4 * col + 2 * wn;
    float* out = A.part + (int64_t)split * A.m * A.n;
    if (n < A.n) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int row = m0 + wm * 128 + 32 * i + (r & 3) + 8 * (r >> 2) + 4 * half;
                if (row < A.m) *reinterpret_cast<f32x2*>(out + (int64_t)row * A.n + n) = f32x2{acc[i][0][r], acc[i][1][r]};
            }
        }
    }
}

// c = the sum of the splits' partial results, in order, rounded to BF16 once; 4 values a lane.
__global__ __launch_bounds__(256) void k_mm_sum(const float* part, int64_t size, int32_t splits, uint16_t* c)
{
    const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (i >= size) return;
    f32x4 x = *reinterpret_cast<const f32x4*>(part + i);
    for (int s = 1; s < splits; ++s) x += *reinterpret_cast<const f32x4*>(part + s * size + i);
    *reinterpret_cast<u32x2*>(c + i) = u32x2{bf16x2_rne(x.x, x.y), bf16x2_rne(x.z, x.w)};
}

constexpr int64_t kMmMost = (int64_t)1 << 22;   // rows, columns, inner: a tile's 256 rows at 32-bit offsets

static int mm_splits(int64_t m, int64_t n, int64_t k)
{
    const int64_t tiles = ((m + kBM - 1) / kBM) * ((n + kBN - 1) / kBN), ksteps = (k + kBK - 1) / kBK;
    return (int)std::max<int64_t>(1, std::min<int64_t>(512 / tiles, ksteps / 16));
}

}  // namespace abh

using namespace abh;

extern "C" {

ADAMBRIDGE_API int64_t adambridge_matmul_work(int64_t m, int64_t n, int64_t k)
{
    if (m < 1 || n < 1 || k < 1 || m > kMmMost || n > kMmMost || k > kMmMost) return ADAMBRIDGE_EBADN;
    return (int64_t)mm_splits(m, n, k) * m * n * 4;
}

ADAMBRIDGE_API int adambridge_matmul(const void* a, const void* b, void* c, int64_t m, int64_t n, int64_t k, void* work)
{
    if (m < 1 || n < 4 || k < 8 || m > kMmMost || n > kMmMost || k > kMmMost || n % 4 || k % 8) return ADAMBRIDGE_EBADN;
    if (!a || !b || !c || !work) return ADAMBRIDGE_ENULL;
    if ((uintptr_t)a % 16 || (uintptr_t)b % 8 || (uintptr_t)c % 8 || (uintptr_t)work % 16) return ADAMBRIDGE_EALIGN;
    MmArgs A;
    A.a = static_cast<const uint16_t*>(a);
    A.b = static_cast<const uint16_t*>(b);
    A.part = static_cast<float*>(work);
    A.k = k;
    A.m = (int32_t)m;
    A.n = (int32_t)n;
    A.tiles_m = (int32_t)((m + kBM - 1) / kBM);
    A.tiles_n = (int32_t)((n + kBN - 1) / kBN);
    A.splits = mm_splits(m, n, k);
    A.ksteps = (int32_t)((k + kBK - 1) / kBK);
    const int64_t total = (int64_t)A.tiles_m * A.tiles_n * A.splits;
    const int64_t per = (total + kXcdCount - 1) / kXcdCount;
    hipLaunchKernelGGL(k_mm_split, dim3((unsigned)(per * kXcdCount)), dim3(kMmThreads), 0, t_stream, A);
    hipLaunchKernelGGL(k_mm_sum, dim3((unsigned)((m * n / 4 + 255) / 256)), dim3(256), 0, t_stream, A.part, m * n,
                       A.splits, static_cast<uint16_t*>(c));
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : hip_fail(e, "hipLaunchKernelGGL (matmul)");
}

}  // extern "C"
