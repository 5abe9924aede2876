// abh_state.hip -- one parameter's interleaved state to and from the reference's separate arrays
// (checkpoints and precision changes; reference optimizer.py:525-602, engine.py:1030-1043).
//
// Bound by HBM: each call reads its source once and writes its destination once, all columns of
// the state in one pass.  A lane takes 4 consecutive elements (2 in the pairs; 8 in the FP8 block
// records, 16 lanes to a 128-element block), as the update kernels do, so every column access of a
// wavefront is one contiguous span.  Before, a checkpoint went column by column through strided
// copies, zeroed stores and whole-tensor temporaries: 4 to 9 passes over the state.
//
// Measured on MI355X, one tensor of 136M elements, us and TB/s of source read plus destination
// written: pairs packed 358 (6.09), unpacked 342 (6.37); FP8 records packed 281 (5.82), unpacked 277
// (5.91), packed from FP32 moments 436 (5.62); FP32 records 539 (6.06) and 573 (5.71); FP24 records
// 327 (5.83) both ways; Lion records 260 (6.27) and 261 (6.25).  A 2 GB copy here runs at 6.58.
// Fewer workgroups a CU (24 to 40 KiB of dynamic LDS) were slower for all but FP8 packing (281 -> 267).

#include <hip/hip_runtime.h>

#include <stdint.h>

#include <algorithm>

#include "../../include/adambridge_hip.h"
#include "abh_device.hpp"
#include "abh_host.hpp"

namespace abh {

constexpr int kStateThreads = 256;
constexpr int kStateXcds = 8;

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

#define ABH_GLOBAL __attribute__((address_space(1)))

template <typename T>
__device__ __forceinline__ T get(const void* p) { return *(const ABH_GLOBAL T*)p; }
template <typename T>
__device__ __forceinline__ void put(void* p, T v) { *(ABH_GLOBAL T*)p = v; }

// Streaming accesses (every byte is touched once), for runs that a wavefront's lanes cover without gaps.
template <typename T>
__device__ __forceinline__ T ld(const void* p) { return __builtin_nontemporal_load((const ABH_GLOBAL T*)p); }
template <typename T>
__device__ __forceinline__ void st(void* p, T v) { __builtin_nontemporal_store(v, (ABH_GLOBAL T*)p); }

// Where a layout keeps things: elements and bytes per record, and the byte offsets of the columns
// in a record (include/adambridge_hip.h).  kMv: moment storage; kF24: FP24 master planes.
template <int L>
struct Layout;

template <int RECORD_ELEMS, int RECORD_BYTES, int MV, bool F24, bool V, int M, int VAT>
struct RecordLayout {
    static constexpr int64_t kElems = RECORD_ELEMS, kBytes = RECORD_BYTES;
    static constexpr int kMv = MV;
    static constexpr bool kF24 = F24, kV = V;
    static constexpr int64_t kLo = F24 ? RECORD_ELEMS * 2 : 0, kM = M, kVAt = VAT;
};

template <> struct Layout<DT_PACKED_LION> : RecordLayout<256, 1536, DT_BF16, false, false, 1024, 0> {};
template <> struct Layout<DT_PACKED_LION_F32> : RecordLayout<256, 2048, DT_F32, false, false, 1024, 0> {};
template <> struct Layout<DT_PACKED_F32> : RecordLayout<256, 3072, DT_F32, false, true, 1024, 2048> {};
template <> struct Layout<DT_PACKED_F24> : RecordLayout<256, 1792, DT_BF16, true, true, 768, 1280> {};
template <> struct Layout<DT_PACKED_F24_F32> : RecordLayout<256, 2816, DT_F32, true, true, 768, 1792> {};
template <> struct Layout<DT_PACKED_LION_F24> : RecordLayout<256, 1280, DT_BF16, true, false, 768, 0> {};
template <> struct Layout<DT_PACKED_LION_F24_F32> : RecordLayout<256, 1792, DT_F32, true, false, 768, 0> {};
template <> struct Layout<DT_PACKED8> : RecordLayout<128, 768, DT_FP8, false, true, 512, 520> {};
template <> struct Layout<DT_PACKED8_F24> : RecordLayout<128, 640, DT_FP8, true, true, 384, 392> {};
template <> struct Layout<DT_PACKED8_LION> : RecordLayout<128, 640, DT_FP8, false, false, 512, 0> {};
template <> struct Layout<DT_PACKED8_LION_F24> : RecordLayout<128, 512, DT_FP8, true, false, 384, 0> {};
template <> struct Layout<DT_PACKED> : RecordLayout<2, 16, DT_BF16, false, true, 8, 12> {};   // the pairs

// Byte offsets of element e's master (or its high half), low byte and moments.
template <int L>
__device__ __forceinline__ int64_t at_p(int64_t e)
{
    using T = Layout<L>;
    const int64_t rec = e / T::kElems * T::kBytes, j = e % T::kElems;
    if constexpr (T::kF24) return rec + 2 * j;
    else if constexpr (T::kMv == DT_FP8) return rec + ((j & 4) ? 256 : 0) + (j >> 3) * 16 + (j & 3) * 4;
    else return rec + 4 * j;
}
template <int L>
__device__ __forceinline__ int64_t at_lo(int64_t e)
{
    using T = Layout<L>;
    return e / T::kElems * T::kBytes + T::kLo + e % T::kElems;
}
template <int L, bool SECOND>
__device__ __forceinline__ int64_t at_mv(int64_t e)
{
    using T = Layout<L>;
    const int64_t rec = e / T::kElems * T::kBytes, j = e % T::kElems, col = SECOND ? T::kVAt : T::kM;
    if constexpr (T::kMv == DT_FP8) return rec + col + (T::kV ? (j >> 3) * 16 + (j & 7) : j);
    else return rec + col + j * (T::kMv == DT_F32 ? 4 : 2);
}

// A separate array of moments: FP32, BF16, or FP8 codes with a scale per 128.  dtype 0: none.
struct Moments {
    uint8_t* data;
    float* scale;
    int32_t dtype;
    int32_t pad;
};

struct StateArgs {
    uint8_t* state;
    float* m_scale;    // the state's own block scales (FP8 layouts)
    float* v_scale;
    uint8_t* p;        // separate master: FP32, BF16 (pack only), or the FP24 high halves
    uint8_t* p_lo;
    Moments m, v;
    int64_t n;
    int64_t first;     // lane groups of the state that earlier launches took, and this launch's
    int64_t groups;
    int32_t p_dtype;   // 0: none
    int32_t vec;       // every array allows a lane's vector accesses
};

// ------------------------------------------------------------ a lane's values

// E consecutive values of SIZE bytes as the low bits of words: one access of 2 to 16 bytes, or (8
// FP32 values, the ends of FP8 blocks) two of 16.  Those two are ordinary accesses: each covers half
// of every cache line it touches, and the second finds the line the first brought in.
template <int SIZE, int E>
__device__ __forceinline__ void load_run(const uint8_t* p, uint32_t (&x)[E])
{
    constexpr int kBytes = SIZE * E;
    uint32_t w[(kBytes + 3) / 4];
    if constexpr (kBytes == 2) {
        w[0] = ld<uint16_t>(p);
    } else if constexpr (kBytes == 4) {
        w[0] = ld<uint32_t>(p);
    } else if constexpr (kBytes == 8) {
        const u32x2 a = ld<u32x2>(p);
        w[0] = a.x; w[1] = a.y;
    } else {
#pragma unroll
        for (int k = 0; k < kBytes / 4; k += 4) {
            const u32x4 a = kBytes == 16 ? ld<u32x4>(p) : get<u32x4>(p + 4 * k);
            w[k] = a.x; w[k + 1] = a.y; w[k + 2] = a.z; w[k + 3] = a.w;
        }
    }
#pragma unroll
    for (int k = 0; k < E; ++k) {
        if constexpr (SIZE == 4) x[k] = w[k];
        else if constexpr (SIZE == 2) x[k] = (w[k / 2] >> (16 * (k & 1))) & 0xffffu;
        else x[k] = (w[k / 4] >> (8 * (k & 3))) & 0xffu;
    }
}

template <int SIZE, int E>
__device__ __forceinline__ void store_run(uint8_t* p, const uint32_t (&x)[E])
{
    constexpr int kBytes = SIZE * E;
    uint32_t w[(kBytes + 3) / 4] = {};
#pragma unroll
    for (int k = 0; k < E; ++k) {
        if constexpr (SIZE == 4) w[k] = x[k];
        else if constexpr (SIZE == 2) w[k / 2] |= x[k] << (16 * (k & 1));
        else w[k / 4] |= x[k] << (8 * (k & 3));
    }
    if constexpr (kBytes == 2) {
        st(p, (uint16_t)w[0]);
    } else if constexpr (kBytes == 4) {
        st(p, w[0]);
    } else if constexpr (kBytes == 8) {
        st(p, u32x2{w[0], w[1]});
    } else if constexpr (kBytes == 16) {
        st(p, u32x4{w[0], w[1], w[2], w[3]});
    } else {
        put(p, u32x4{w[0], w[1], w[2], w[3]});
        put(p + 16, u32x4{w[4], w[5], w[6], w[7]});
    }
}

template <int SIZE>
__device__ __forceinline__ uint32_t load_value(const uint8_t* p)
{
    if constexpr (SIZE == 4) return get<uint32_t>(p);
    else if constexpr (SIZE == 2) return get<uint16_t>(p);
    else return get<uint8_t>(p);
}

template <int SIZE>
__device__ __forceinline__ void store_value(uint8_t* p, uint32_t x)
{
    if constexpr (SIZE == 4) put(p, x);
    else if constexpr (SIZE == 2) put(p, (uint16_t)x);
    else put(p, (uint8_t)x);
}

// Elements e .. e + E - 1 of a separate array (those below n), vector accesses where `whole`.
template <int SIZE, int E>
__device__ __forceinline__ void load_array(const uint8_t* base, int64_t e, int64_t n, bool whole, uint32_t (&x)[E])
{
    if (whole) {
        load_run<SIZE>(base + e * SIZE, x);
        return;
    }
#pragma unroll
    for (int k = 0; k < E; ++k) x[k] = e + k < n ? load_value<SIZE>(base + (e + k) * SIZE) : 0u;
}

template <int SIZE, int E>
__device__ __forceinline__ void store_array(uint8_t* base, int64_t e, int64_t n, bool whole, const uint32_t (&x)[E])
{
    if (whole) {
        store_run<SIZE>(base + e * SIZE, x);
        return;
    }
#pragma unroll
    for (int k = 0; k < E; ++k)
        if (e + k < n) store_value<SIZE>(base + (e + k) * SIZE, x[k]);
}

template <int MV>
constexpr int mv_size = MV == DT_F32 ? 4 : MV == DT_BF16 ? 2 : 1;

// Elements a lane takes: that many consecutive moments, and masters in runs of kRun.  In the FP8
// records with an FP32 master, 8 FP32 values a lane would lie at a 32-byte stride in the separate
// array (each access half of its cache lines), so lane l of a block's 16 takes the masters 4l ..
// 4l + 3 and 64 + 4l .. 64 + 4l + 3 instead, and FP32 source moments likewise: every access of the 16
// lanes then covers whole lines on both sides (136M elements from FP32 moments: 451 -> 434 us).
template <int L>
constexpr int lane_elems = Layout<L>::kMv == DT_FP8 ? 8 : L == DT_PACKED ? 2 : 4;

template <int L>
constexpr int kRun = Layout<L>::kMv == DT_FP8 && !Layout<L>::kF24 ? 4 : lane_elems<L>;
template <int L>
constexpr int kRuns = lane_elems<L> / kRun<L>;

// The first element of a lane's run r of masters, its moments starting at element e.
template <int L>
__device__ __forceinline__ int64_t run_at(int64_t e, int r)
{
    if constexpr (kRuns<L> == 1) return e;
    else return (e & ~(int64_t)(kFp8Block - 1)) + 64 * r + ((e >> 1) & 60);
}

// The state is 16-byte aligned (checked) and a lane's group never crosses a record, so its column
// accesses are vectors wherever the group lies below n.  The pairs are handled apart.

// The FP32 bits of a lane's masters in the state (FP24: high half << 16 | low byte << 8).
template <int L, int E>
__device__ __forceinline__ void load_state_p(const uint8_t* s, int64_t e, int64_t n, uint32_t (&x)[E])
{
    using T = Layout<L>;
    if constexpr (T::kF24) {
        uint32_t h[E], l[E];
        if (e + E <= n) {
            load_run<2>(s + at_p<L>(e), h);
            load_run<1>(s + at_lo<L>(e), l);
        } else {
#pragma unroll
            for (int k = 0; k < E; ++k) {
                h[k] = e + k < n ? load_value<2>(s + at_p<L>(e + k)) : 0u;
                l[k] = e + k < n ? load_value<1>(s + at_lo<L>(e + k)) : 0u;
            }
        }
#pragma unroll
        for (int k = 0; k < E; ++k) x[k] = (h[k] << 16) | (l[k] << 8);
    } else if (e + E <= n) {
#pragma unroll
        for (int k = 0; k < E; k += 4) {
            const u32x4 w = ld<u32x4>(s + at_p<L>(e + k));
            x[k] = w.x; x[k + 1] = w.y; x[k + 2] = w.z; x[k + 3] = w.w;
        }
    } else {
#pragma unroll
        for (int k = 0; k < E; ++k) x[k] = e + k < n ? load_value<4>(s + at_p<L>(e + k)) : 0u;
    }
}

template <int L, int E>
__device__ __forceinline__ void store_state_p(uint8_t* s, int64_t e, int64_t n, const uint32_t (&x)[E])
{
    using T = Layout<L>;
    if constexpr (T::kF24) {
        uint32_t h[E], l[E];
#pragma unroll
        for (int k = 0; k < E; ++k) {
            h[k] = x[k] >> 16;
            l[k] = (x[k] >> 8) & 0xffu;
        }
        if (e + E <= n) {
            store_run<2>(s + at_p<L>(e), h);
            store_run<1>(s + at_lo<L>(e), l);
        } else {
#pragma unroll
            for (int k = 0; k < E; ++k) {
                if (e + k >= n) continue;
                store_value<2>(s + at_p<L>(e + k), h[k]);
                store_value<1>(s + at_lo<L>(e + k), l[k]);
            }
        }
    } else if (e + E <= n) {
#pragma unroll
        for (int k = 0; k < E; k += 4) st(s + at_p<L>(e + k), u32x4{x[k], x[k + 1], x[k + 2], x[k + 3]});
    } else {
#pragma unroll
        for (int k = 0; k < E; ++k)
            if (e + k < n) store_value<4>(s + at_p<L>(e + k), x[k]);
    }
}

// The lane's group among the launch's, XCD by XCD (adambridge_hip.hip: block_tile).
__device__ __forceinline__ int64_t lane_group(int64_t groups)
{
    const int64_t tiles = (groups + kStateThreads - 1) / kStateThreads;
    const int64_t per = (tiles + kStateXcds - 1) / kStateXcds, b = blockIdx.x;
    return ((b % kStateXcds) * per + b / kStateXcds) * kStateThreads + threadIdx.x;
}

// NATIVE: every column is given, in the layout's own formats, and the arrays allow vector accesses
// -- the checkpoint's case.  Its kernels are straight-line, all loads before the first store: with
// the formats tested at run time each column's load waits for the one before it (136M elements,
// pairs, packed: 434 us tested at run time).
template <int L>
constexpr int own_master = Layout<L>::kF24 ? DT_F24 : DT_F32;

// ---------------------------------------------------------------- state -> arrays

template <int L, int E, bool SECOND>
__device__ __forceinline__ void load_state_mv(const StateArgs& a, int64_t e, uint32_t (&x)[E])
{
    constexpr int S = mv_size<Layout<L>::kMv>;
    if (e + E <= a.n) {
        load_run<S>(a.state + at_mv<L, SECOND>(e), x);
    } else {
#pragma unroll
        for (int k = 0; k < E; ++k) x[k] = e + k < a.n ? load_value<S>(a.state + at_mv<L, SECOND>(e + k)) : 0u;
    }
}

// A lane's 8 codes (two words) and, on the block's first lane, the block's scale into separate arrays.
__device__ __forceinline__ void unpack_codes(const StateArgs& a, const Moments& to, const float* scales, int64_t e,
                                             const u32x2 w, bool vec)
{
    if (vec) {
        put(to.data + e, w);   // 8-byte streaming stores were slower (136M elements: 329 against 277 us)
    } else {
#pragma unroll
        for (int k = 0; k < 8; ++k) put(to.data + e + k, (uint8_t)((k < 4 ? w.x : w.y) >> (8 * (k & 3))));
    }
    if ((e & (kFp8Block - 1)) == 0) put(to.scale + e / kFp8Block, get<float>(scales + e / kFp8Block));
}

template <int L, bool NATIVE>
__global__ __launch_bounds__(kStateThreads) void k_unpack_state(StateArgs a)
{
    using T = Layout<L>;
    constexpr int E = lane_elems<L>;
    const int64_t g = lane_group(a.groups);
    if (g >= a.groups) return;
    const int64_t e = (a.first + g) * E;
    const bool p = NATIVE || a.p_dtype, m = NATIVE || a.m.dtype, v = T::kV && (NATIVE || a.v.dtype);
    const bool vec = NATIVE || a.vec, whole = vec && e + E <= a.n;
    constexpr int R = kRun<L>, N = kRuns<L>;
    uint32_t xp[N][R], xm[E], xv[E];
    u32x4 codes{0u, 0u, 0u, 0u};
    if constexpr (L == DT_PACKED) {
        // one pair: 16 bytes {p, p, m | m << 16, v | v << 16}; an odd n's last pair is there whole
        const u32x4 x = ld<u32x4>(a.state + e * 8);
        xp[0][0] = x.x; xp[0][1] = x.y;
        xm[0] = x.z & 0xffffu; xm[1] = x.z >> 16;
        xv[0] = x.w & 0xffffu; xv[1] = x.w >> 16;
    } else {
        if (p) {
#pragma unroll
            for (int r = 0; r < N; ++r) load_state_p<L>(a.state, run_at<L>(e, r), a.n, xp[r]);
        }
        if constexpr (T::kMv != DT_FP8) {
            if (m) load_state_mv<L, E, false>(a, e, xm);
            if constexpr (T::kV) {
                if (v) load_state_mv<L, E, true>(a, e, xv);
            }
        }
    }
    if (p) {
#pragma unroll
        for (int r = 0; r < N; ++r) {
            const int64_t at = run_at<L>(e, r);
            const bool in = vec && at + R <= a.n;
            if constexpr (T::kF24) {
                uint32_t h[R], l[R];
#pragma unroll
                for (int k = 0; k < R; ++k) {
                    h[k] = xp[r][k] >> 16;
                    l[k] = (xp[r][k] >> 8) & 0xffu;
                }
                store_array<2>(a.p, at, a.n, in, h);
                store_array<1>(a.p_lo, at, a.n, in, l);
            } else {
                store_array<4>(a.p, at, a.n, in, xp[r]);
            }
        }
    }
    if constexpr (T::kMv == DT_FP8) {
        // whole blocks of codes on both sides, m's and v's of a lane in one 16-byte load
        if constexpr (T::kV) {
            if (m || v) codes = ld<u32x4>(a.state + at_mv<L, false>(e));
        } else if (m) {
            const u32x2 w = ld<u32x2>(a.state + at_mv<L, false>(e));
            codes = u32x4{w.x, w.y, 0u, 0u};
        }
        if (m) unpack_codes(a, a.m, a.m_scale, e, u32x2{codes.x, codes.y}, vec);
        if (v) unpack_codes(a, a.v, a.v_scale, e, u32x2{codes.z, codes.w}, vec);
    } else {
        if (m) store_array<mv_size<T::kMv>>(a.m.data, e, a.n, whole, xm);
        if constexpr (T::kV) {
            if (v) store_array<mv_size<T::kMv>>(a.v.data, e, a.n, whole, xv);
        }
    }
}

// ---------------------------------------------------------------- arrays -> state

// A lane's source masters as FP32 bits, rounded to FP24 where the layout's master is one and the
// source is FP32 (to nearest, a NaN quietened: adambridge_convert_plane's rule).
template <int L, bool NATIVE, int E>
__device__ __forceinline__ void load_master(const StateArgs& a, int64_t e, uint32_t (&x)[E])
{
    const bool whole = (NATIVE || a.vec) && e + E <= a.n;
    const int dt = NATIVE ? own_master<L> : a.p_dtype;
    if (dt == DT_F32) {
        load_array<4>(a.p, e, a.n, whole, x);
        if constexpr (Layout<L>::kF24) {
#pragma unroll
            for (int k = 0; k < E; ++k) x[k] = f24_round<false>(bitsf(x[k]), 0u);
        }
        return;
    }
    load_array<2>(a.p, e, a.n, whole, x);
#pragma unroll
    for (int k = 0; k < E; ++k) x[k] <<= 16;
    if (dt == DT_F24) {
        uint32_t l[E];
        load_array<1>(a.p_lo, e, a.n, whole, l);
#pragma unroll
        for (int k = 0; k < E; ++k) x[k] |= l[k] << 8;
    }
}

// A lane's source moments as FP32 values, decoded exactly (k_convert's rules); zero past the end.
template <bool V, int E>
__device__ __forceinline__ void load_moment(const StateArgs& a, const Moments& from, int64_t e, float (&x)[E])
{
    const bool whole = a.vec && e + E <= a.n;
    uint32_t w[E];
    if (from.dtype == DT_F32) {
        load_array<4>(from.data, e, a.n, whole, w);
#pragma unroll
        for (int k = 0; k < E; ++k) x[k] = bitsf(w[k]);
    } else if (from.dtype == DT_BF16) {
        load_array<2>(from.data, e, a.n, whole, w);
#pragma unroll
        for (int k = 0; k < E; ++k) x[k] = bitsf(w[k] << 16);
    } else {
        load_array<1>(from.data, e, a.n, whole, w);
        const float s = e < a.n ? get<float>(from.scale + e / kFp8Block) : 0.0f;
#pragma unroll
        for (int k = 0; k < E; ++k) {
            const float u = (V ? e5m2_decode<0>(w[k]) : e4m3_decode<0>(w[k])) * s;
            x[k] = e + k < a.n ? (V ? u * u : u) : 0.0f;
        }
    }
}

// Storage bits of an FP32 value in an FP32 or BF16 column: BF16 to nearest with torch's NaN (0x7fc0).
template <int MV>
__device__ __forceinline__ uint32_t encode_value(float x)
{
    if constexpr (MV == DT_F32) return fbits(x);
    else return x != x ? 0x7fc0u : bf16_rne(x);
}

// A lane's source moments in the storage bits of an FP32 or BF16 column; the same format as it is.
template <int MV, bool V, bool NATIVE, int E>
__device__ __forceinline__ void load_encoded(const StateArgs& a, const Moments& from, int64_t e, uint32_t (&w)[E])
{
    if (NATIVE || from.dtype == MV) {
        load_array<mv_size<MV>>(from.data, e, a.n, (NATIVE || a.vec) && e + E <= a.n, w);
        return;
    }
    float x[E];
    load_moment<V>(a, from, e, x);
#pragma unroll
    for (int k = 0; k < E; ++k) w[k] = encode_value<MV>(x[k]);
}

// FP8 codes and scale of one block, 8 elements a lane of 16: k_convert's encoding to nearest.
template <bool V>
__device__ __forceinline__ float encode_block(float (&x)[8], uint32_t (&code)[8])
{
    constexpr float kMax = V ? 57344.0f : 448.0f;
    float amax = 0.0f;
    int nan = 0;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        if constexpr (V) x[k] = __builtin_sqrtf(x[k] < 0.0f ? 0.0f : x[k]);   // NaN and -0 pass through
        const float b = fabsf(x[k]);
        nan |= b != b;
        amax = b > amax ? b : amax;
    }
#pragma unroll
    for (int d = 1; d < 16; d <<= 1) {
        amax = fmaxf(amax, __shfl_xor(amax, d, 16));
        nan |= __shfl_xor(nan, d, 16);
    }
    const float scale = (!nan && amax > 0.0f) ? amax / kMax : 1.0f;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        float y = x[k] / scale;
        y = y > kMax ? kMax : (y < -kMax ? -kMax : y);   // NaN passes
        code[k] = y != y ? ((fbits(y) >> 24) & 0x80u) | 0x7fu : V ? e5m2_encode<false>(y, 0u) : e4m3_encode<false>(y, 0u);
    }
    return scale;
}

// A lane's 8 codes of an FP8 layout (two words) and, on the block's first lane, the block's scale.
template <bool V, bool NATIVE>
__device__ __forceinline__ u32x2 block_codes(const StateArgs& a, const Moments& from, int64_t e, float& scale)
{
    if (NATIVE || (from.dtype == DT_FP8 && a.vec)) {   // whole blocks of codes on both sides
        if ((e & (kFp8Block - 1)) == 0) scale = get<float>(from.scale + e / kFp8Block);
        return ld<u32x2>(from.data + e);
    }
    uint32_t w[8];
    const int64_t b0 = e & ~(int64_t)(kFp8Block - 1);
    if (from.dtype == DT_F32 && a.vec && b0 + kFp8Block <= a.n) {
        // FP32 values in the masters' runs (whole lines), encoded there; the codes, a word a run, then
        // go to the lanes that hold them: run 2l and 2l + 1 to lane l, runs 0-15 first, 16-31 second
        uint32_t lo[4], hi[4];
        const int l = (int)(e >> 3) & 15;
        load_run<4>(from.data + (b0 + 4 * l) * 4, lo);
        load_run<4>(from.data + (b0 + 64 + 4 * l) * 4, hi);
        float x[8];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            x[k] = bitsf(lo[k]);
            x[4 + k] = bitsf(hi[k]);
        }
        scale = encode_block<V>(x, w);
        const uint32_t first = w[0] | (w[1] << 8) | (w[2] << 16) | (w[3] << 24);
        const uint32_t second = w[4] | (w[5] << 8) | (w[6] << 16) | (w[7] << 24);
        const int src = (2 * l) & 15;
        const uint32_t a0 = __shfl(first, src, 16), a1 = __shfl(first, src + 1, 16);
        const uint32_t b0w = __shfl(second, src, 16), b1w = __shfl(second, src + 1, 16);
        return l < 8 ? u32x2{a0, a1} : u32x2{b0w, b1w};
    }
    if (from.dtype == DT_FP8) {
        load_array<1>(from.data, e, INT64_MAX, false, w);
        if ((e & (kFp8Block - 1)) == 0) scale = get<float>(from.scale + e / kFp8Block);
    } else {
        float x[8];
        load_moment<V>(a, from, e, x);
        scale = encode_block<V>(x, w);
    }
    return u32x2{w[0] | (w[1] << 8) | (w[2] << 16) | (w[3] << 24), w[4] | (w[5] << 8) | (w[6] << 16) | (w[7] << 24)};
}

template <int L, bool SECOND, int E>
__device__ __forceinline__ void store_state_mv(const StateArgs& a, int64_t e, const uint32_t (&w)[E])
{
    constexpr int S = mv_size<Layout<L>::kMv>;
    if (e + E <= a.n) {
        store_run<S>(a.state + at_mv<L, SECOND>(e), w);
    } else {
#pragma unroll
        for (int k = 0; k < E; ++k)
            if (e + k < a.n) store_value<S>(a.state + at_mv<L, SECOND>(e + k), w[k]);
    }
}

template <int L, bool NATIVE>
__global__ __launch_bounds__(kStateThreads) void k_pack_state(StateArgs a)
{
    using T = Layout<L>;
    constexpr int E = lane_elems<L>;
    const int64_t g = lane_group(a.groups);
    if (g >= a.groups) return;   // FP8: 16-lane groups leave whole (their shuffles stay within live lanes)
    const int64_t e = (a.first + g) * E;
    const bool p = NATIVE || a.p_dtype, m = NATIVE || a.m.dtype, v = T::kV && (NATIVE || a.v.dtype);
    constexpr int R = kRun<L>, N = kRuns<L>;
    uint32_t xp[N][R], xm[E], xv[E];
    u32x2 cm{0u, 0u}, cv{0u, 0u};
    float sm = 0.0f, sv = 0.0f;
    u32x4 kept{0u, 0u, 0u, 0u};
    if constexpr (L == DT_PACKED) {   // what is not given, and the slot past an odd n, is kept
        if (!(p && m && v && e + 2 <= a.n)) kept = ld<u32x4>(a.state + e * 8);
    }
    if (p) {
#pragma unroll
        for (int r = 0; r < N; ++r) load_master<L, NATIVE>(a, run_at<L>(e, r), xp[r]);
    }
    if constexpr (T::kMv == DT_FP8) {
        if (m) cm = block_codes<false, NATIVE>(a, a.m, e, sm);
        if constexpr (T::kV) {
            if (v) cv = block_codes<true, NATIVE>(a, a.v, e, sv);
        }
    } else {
        if (m) load_encoded<T::kMv, false, NATIVE>(a, a.m, e, xm);
        if constexpr (T::kV) {
            if (v) load_encoded<T::kMv, true, NATIVE>(a, a.v, e, xv);
        }
    }
    if constexpr (L == DT_PACKED) {   // one pair, its 16 bytes whole
        const bool both = e + 1 < a.n;
        const uint32_t p1 = p && both ? xp[0][1] : kept.y;
        const uint32_t m0 = m ? xm[0] : kept.z & 0xffffu, m1 = m && both ? xm[1] : kept.z >> 16;
        const uint32_t v0 = v ? xv[0] : kept.w & 0xffffu, v1 = v && both ? xv[1] : kept.w >> 16;
        st(a.state + e * 8, u32x4{p ? xp[0][0] : kept.x, p1, m0 | (m1 << 16), v0 | (v1 << 16)});
        return;
    }
    if (p) {
#pragma unroll
        for (int r = 0; r < N; ++r) store_state_p<L>(a.state, run_at<L>(e, r), a.n, xp[r]);
    }
    if constexpr (T::kMv == DT_FP8) {
        // the codes of m and v in one 16-byte store: 8 bytes at a 16-byte stride would leave every
        // line half written
        uint8_t* const at = a.state + at_mv<L, false>(e);
        if constexpr (T::kV) {
            if (m && v) st(at, u32x4{cm.x, cm.y, cv.x, cv.y});
            else if (m) put(at, cm);
            else if (v) put(at + 8, cv);
        } else if (m) {
            st(at, cm);
        }
        if ((e & (kFp8Block - 1)) == 0) {
            if (m) put(a.m_scale + e / kFp8Block, sm);
            if (v) put(a.v_scale + e / kFp8Block, sv);
        }
    } else {
        if (m) store_state_mv<L, false>(a, e, xm);
        if constexpr (T::kV) {
            if (v) store_state_mv<L, true>(a, e, xv);
        }
    }
}

// ------------------------------------------------------------------------- host

using StateFn = void (*)(StateArgs);

struct StateKernels {
    StateFn unpack[2], pack[2];   // any arrays; every column in the layout's own formats, aligned
    int mv, lane, run;   // moment storage; elements a lane takes, and masters in one run of them
    bool f24, v;
};

template <int L>
static StateKernels kernels_of()
{
    return {{&k_unpack_state<L, false>, &k_unpack_state<L, true>}, {&k_pack_state<L, false>, &k_pack_state<L, true>},
            Layout<L>::kMv, lane_elems<L>, kRun<L>, Layout<L>::kF24, Layout<L>::kV};
}

static bool state_kernels(int layout, StateKernels* k)
{
    switch (layout) {
    case DT_PACKED: *k = kernels_of<DT_PACKED>(); return true;
    case DT_PACKED8: *k = kernels_of<DT_PACKED8>(); return true;
    case DT_PACKED_LION: *k = kernels_of<DT_PACKED_LION>(); return true;
    case DT_PACKED_F32: *k = kernels_of<DT_PACKED_F32>(); return true;
    case DT_PACKED_F24: *k = kernels_of<DT_PACKED_F24>(); return true;
    case DT_PACKED_LION_F24: *k = kernels_of<DT_PACKED_LION_F24>(); return true;
    case DT_PACKED8_F24: *k = kernels_of<DT_PACKED8_F24>(); return true;
    case DT_PACKED_LION_F32: *k = kernels_of<DT_PACKED_LION_F32>(); return true;
    case DT_PACKED8_LION: *k = kernels_of<DT_PACKED8_LION>(); return true;
    case DT_PACKED_F24_F32: *k = kernels_of<DT_PACKED_F24_F32>(); return true;
    case DT_PACKED_LION_F24_F32: *k = kernels_of<DT_PACKED_LION_F24_F32>(); return true;
    case DT_PACKED8_LION_F24: *k = kernels_of<DT_PACKED8_LION_F24>(); return true;
    default: return false;
    }
}

static bool aligned_to(const void* p, uintptr_t a) { return ((uintptr_t)p % a) == 0; }

// The arrays of a call checked against the layout, and the kernel's arguments filled: 0 or a code.
static int state_args(const adambridge_state* s, const adambridge_arrays* q, bool pack, StateKernels* k, StateArgs* a)
{
    if (!s || !q) return ADAMBRIDGE_ENULL;
    if (s->n < 0) return ADAMBRIDGE_EBADN;
    if (!state_kernels(s->layout, k)) return ADAMBRIDGE_EPDTYPE;
    if (s->n == 0) return 0;
    if (!s->data) return ADAMBRIDGE_ENULL;
    if (!aligned_to(s->data, 16)) return ADAMBRIDGE_EALIGN;
    const bool fp8 = k->mv == DT_FP8;
    if (fp8 && ((q->m && !s->m_scale) || (q->v && !s->v_scale))) return ADAMBRIDGE_ESCALES;
    if (q->v && !k->v) return ADAMBRIDGE_EMVDTYPE;
    *a = StateArgs{};
    a->state = static_cast<uint8_t*>(s->data);
    a->m_scale = s->m_scale;
    a->v_scale = s->v_scale;
    a->n = s->n;
    bool vec = true, natural = true;   // a lane's vector accesses; each value at its own alignment
    const uintptr_t lane = (uintptr_t)k->lane;
    if (q->p) {
        const int own = k->f24 ? DT_F24 : DT_F32;
        if (pack ? (q->p_dtype != DT_F32 && q->p_dtype != DT_BF16 && q->p_dtype != DT_F24) : q->p_dtype != own)
            return ADAMBRIDGE_EPDTYPE;
        if (q->p_dtype == DT_F24 && !q->p_lo) return ADAMBRIDGE_ENULL;
        a->p = static_cast<uint8_t*>(q->p);
        a->p_lo = q->p_dtype == DT_F24 ? q->p_lo : nullptr;
        a->p_dtype = q->p_dtype;
        const uintptr_t size = q->p_dtype == DT_F32 ? 4 : 2;
        natural = aligned_to(a->p, size);
        const uintptr_t run = (uintptr_t)k->run;
        vec = aligned_to(a->p, std::min<uintptr_t>(16, size * run)) && aligned_to(a->p_lo, run);
    }
    const struct { void* data; float* scale; Moments* to; } mv[2] = {{q->m, q->m_scale, &a->m}, {q->v, q->v_scale, &a->v}};
    for (const auto& x : mv) {
        if (!x.data) continue;
        const int dt = q->mv_dtype;
        if (pack ? (dt != DT_F32 && dt != DT_BF16 && dt != DT_FP8) : dt != k->mv) return ADAMBRIDGE_EMVDTYPE;
        if (dt == DT_FP8 && !x.scale) return ADAMBRIDGE_ESCALES;
        *x.to = Moments{static_cast<uint8_t*>(x.data), x.scale, dt, 0};
        const uintptr_t size = dt == DT_F32 ? 4 : dt == DT_BF16 ? 2 : 1;
        natural = natural && aligned_to(x.data, size) && aligned_to(x.scale, 4);
        vec = vec && aligned_to(x.data, std::min<uintptr_t>(16, size * lane));
    }
    if (!natural) return ADAMBRIDGE_EALIGN;
    a->vec = vec ? 1 : 0;
    return 0;
}

// The launches of one call, each within a dispatch's 2^32 - 1 work-items.
static int run_state(const StateKernels& k, StateArgs a, bool pack)
{
    constexpr int64_t kMost = (int64_t)(0xffffffffu / kStateThreads) / kStateXcds * kStateXcds * kStateThreads;
    // FP8 records to the end of their last block (its codes exist), 16 groups of 8 to a block
    const int64_t whole = k.mv == DT_FP8 ? kFp8Block : k.lane, total = (a.n + whole - 1) / whole * (whole / k.lane);
    const bool native = a.vec && a.p_dtype == (k.f24 ? DT_F24 : DT_F32) && a.m.dtype == k.mv && (!k.v || a.v.dtype == k.mv);
    for (a.first = 0; a.first < total; a.first += a.groups) {
        a.groups = std::min(total - a.first, kMost);
        const int64_t tiles = (a.groups + kStateThreads - 1) / kStateThreads;
        const int64_t grid = (tiles + kStateXcds - 1) / kStateXcds * kStateXcds;
        hipLaunchKernelGGL(pack ? k.pack[native] : k.unpack[native], dim3((unsigned)grid), dim3(kStateThreads), 0, t_stream, a);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return hip_fail(e, pack ? "hipLaunchKernelGGL (pack)" : "hipLaunchKernelGGL (unpack)");
    }
    return 0;
}

}  // namespace abh

using namespace abh;

extern "C" {

ADAMBRIDGE_API int adambridge_unpack_state(const adambridge_state* state, const adambridge_arrays* to)
{
    StateKernels k;
    StateArgs a;
    const int rc = state_args(state, to, false, &k, &a);
    return rc || state->n == 0 || (!to->p && !to->m && !to->v) ? rc : run_state(k, a, false);
}

ADAMBRIDGE_API int adambridge_pack_state(const adambridge_state* state, const adambridge_arrays* from)
{
    StateKernels k;
    StateArgs a;
    const int rc = state_args(state, from, true, &k, &a);
    return rc || state->n == 0 || (!from->p && !from->m && !from->v) ? rc : run_state(k, a, true);
}

}  // extern "C"
