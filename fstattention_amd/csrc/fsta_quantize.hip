// K and V -> the 8-bit storage of fsta_attention_fwd_kv8: OCP e4m3 bytes and one float32 scale per slice, chosen so
// that the slice's largest magnitude maps to the format's largest value (448).
//
// HBM-bound: 2 (or 4) bytes read and 1 written per element, and the scale needs the whole slice before the first byte
// can be written.  A slice of up to kOneWg bytes is kept in the registers of one workgroup: one launch, every element
// read once.  Larger slices take two launches: the first reads them for the maxima of 16 KB pieces, the second reads
// them again (what the 256 MB Infinity Cache still holds does not come from HBM a second time), joins the maxima of its
// slice (at most a few hundred words) and writes the bytes.  The second reading and the bytes go past the caches, so that
// they do not drive out what is still to be read (K and V of 32 heads x 8192 keys x 128, bf16: 58.0 -> 53.0 us by the
// stores, 50.8 with the loads and pieces of half the size).  Pieces are 16 KB, one unit of 16 elements for each of 512
// threads: 48.6 us (256 threads with two units 50.6, 512 with two 50.4, 256 with one 49.6, 1024 with one 51.8).  Both launches
// deal the same pieces to the same workgroup numbers, hence XCDs: with pieces of another size in the second one its reading
// misses what the first left in the XCD's L2 (8 heads, 33 MB: 12.7 us against 16.1).  Several pieces per workgroup with the
// next one's loads in flight: 53 to 57 us (half the waves by their registers).
#include "fsta_common.h"

namespace fsta {
namespace {

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

constexpr float kFp8Max = 448.f;
constexpr int kThreads = 512;            // two launches: threads per piece, a unit of 16 elements each
constexpr int kOneThreads = 1024;        // one launch: threads per slice
constexpr int kUnitElems = 16;
constexpr double kGridThreads = 4294967296.0;      // a grid ends before 2^32 threads

template <typename T> struct Unit {      // 16 elements as they lie in memory
    static constexpr int kWords = kUnitElems * (int)sizeof(T) / 16;
    u32x4 w[kWords];
};

// LAST: nobody reads these elements again (past the caches)
template <bool LAST, typename T> __device__ __forceinline__ Unit<T> load_unit(const T* src) {
    Unit<T> u;
#pragma unroll
    for (int i = 0; i < Unit<T>::kWords; ++i) {
        const u32x4* word = reinterpret_cast<const u32x4*>(src) + i;
        if constexpr (LAST) u.w[i] = __builtin_nontemporal_load(word);
        else u.w[i] = *word;
    }
    return u;
}

// Magnitudes compare like the integers their bits are; a NaN is above infinity, so it comes out on top as it does in a
// maximum that propagates NaN.
template <typename T> __device__ __forceinline__ uint32_t unit_max(const Unit<T>& u) {
    uint32_t mx = 0;
#pragma unroll
    for (int i = 0; i < Unit<T>::kWords; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const uint32_t x = u.w[i][e];
            if constexpr (sizeof(T) == 4) {
                mx = max(mx, x & 0x7fffffffu);
            } else {
                mx = max(mx, max(x & 0x7fffu, (x >> 16) & 0x7fffu));
            }
        }
    return mx;
}
template <typename T> __device__ __forceinline__ float from_bits(uint32_t bits);
template <> __device__ __forceinline__ float from_bits<float>(uint32_t bits) { return __builtin_bit_cast(float, bits); }
template <> __device__ __forceinline__ float from_bits<__half>(uint32_t bits) {
    return (float)__builtin_bit_cast(_Float16, (unsigned short)bits);
}
template <> __device__ __forceinline__ float from_bits<__hip_bfloat16>(uint32_t bits) {
    return __builtin_bit_cast(float, bits << 16);
}
template <typename T> __device__ __forceinline__ float unit_value(const Unit<T>& u, int i) {
    if constexpr (sizeof(T) == 4) {
        const uint32_t x = u.w[i / 4][i % 4];
        return __builtin_bit_cast(float, x);
    } else {
        const uint32_t x = u.w[i / 8][(i / 2) % 4];
        return from_bits<T>((i & 1) ? x >> 16 : x & 0xffffu);
    }
}

// Scales at the ends of the range, and slices with an infinity or a NaN (`plain` = false): divisor and values are brought to the
// middle of the range by a power of two, where the short division below is as exact as elsewhere (what is lost of a value
// underneath rounds to zero either way).  Denormal scales are coarse, so quotients past 448 have to be looked for.
struct Scale {
    float s;             // as stored
    float div, inv, pre; // the quotient is (x * pre) / div, inv = 1 / div
    bool plain;          // pre = 1, and no quotient exceeds 448 by more than a rounding
};
__device__ __forceinline__ Scale make_scale(float amax) {
    Scale sc;
    sc.s = amax > 0.f ? amax * (1.f / kFp8Max) : 1.f;                // (NaN: 1)
    sc.plain = amax >= 0.f && sc.s > 0x1p-60f && sc.s < 0x1p60f;
    sc.pre = sc.plain || !(amax >= 0.f) ? 1.f : sc.s < 1.f ? 0x1p100f : 0x1p-100f;
    sc.div = sc.s * sc.pre;
    sc.inv = 1.f / sc.div;
    if (sc.s == INFINITY) sc.div = sc.inv = 0.f;                      // finite values: x * 0 = 0, infinities: NaN
    return sc;
}
// x / s, correctly rounded: with inv = 1/s correctly rounded, one residual step on x * inv gives the rounded quotient
// (Markstein); 3 instructions in place of the ten of a full division.  A zero loses its sign.
__device__ __forceinline__ float divide(float x, const Scale& sc) {
    const float q0 = x * sc.inv;
    return __builtin_fmaf(__builtin_fmaf(-q0, sc.div, x), sc.inv, q0);
}
// The same for any scale; magnitudes that round beyond 448 become NaN, as the format has no infinity (464 is a tie, to 448).
__device__ __forceinline__ float divide_any(float x, const Scale& sc) {
    const float q = fabsf(divide(x * sc.pre, sc));
    return q <= 464.f ? fminf(q, kFp8Max) : __builtin_nanf("");
}
// The signs of elements 4w .. 4w+3 in bit 7 of their bytes (the scale is positive: they are the bytes' signs, zeros' and
// NaNs' too; two instructions for four elements instead of one each).
template <typename T> __device__ __forceinline__ uint32_t signs(const Unit<T>& u, int w) {
    if constexpr (sizeof(T) == 4) {
        const uint32_t a = u.w[w][0], b = u.w[w][1], c = u.w[w][2], d = u.w[w][3];
        return __builtin_amdgcn_perm(__builtin_amdgcn_perm(d, c, 0x07030c0cu), __builtin_amdgcn_perm(b, a, 0x0c0c0703u), 0x07060100u) &
               0x80808080u;
    } else {
        const uint32_t a = u.w[w / 2][2 * (w % 2)], b = u.w[w / 2][2 * (w % 2) + 1];
        return __builtin_amdgcn_perm(b, a, 0x07050301u) & 0x80808080u;
    }
}
// PAST: around the caches
template <bool PAST, typename T> __device__ __forceinline__ void store_unit(const Unit<T>& u, const Scale& sc, uint8_t* dst) {
    u32x4 out;
    auto bytes = [&](auto quotient) {
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            int pk = __builtin_amdgcn_cvt_pk_fp8_f32(quotient(unit_value(u, 4 * w), sc), quotient(unit_value(u, 4 * w + 1), sc), 0, false);
            pk = __builtin_amdgcn_cvt_pk_fp8_f32(quotient(unit_value(u, 4 * w + 2), sc), quotient(unit_value(u, 4 * w + 3), sc), pk, true);
            out[w] = ((uint32_t)pk & 0x7f7f7f7fu) | signs(u, w);
        }
    };
    if (sc.plain) bytes([](float x, const Scale& c) { return divide(x, c); });
    else bytes([](float x, const Scale& c) { return divide_any(x, c); });
    if constexpr (PAST) __builtin_nontemporal_store(out, reinterpret_cast<u32x4*>(dst));
    else *reinterpret_cast<u32x4*>(dst) = out;
}

__device__ __forceinline__ uint32_t wave_max(uint32_t x) {
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) x = max(x, (uint32_t)__shfl_xor((int)x, d));
    return x;
}

struct QuantArgs {
    const void* src[2];
    uint8_t* dst[2];
    float* scale[2];
    uint32_t* part;        // two launches: [tensor][slice][piece] maxima
    int64_t elems;         // per slice
    int32_t slices, pieces;
};

template <typename T, int N>
__global__ __launch_bounds__(kOneThreads) void quantize_slice_kernel(QuantArgs a) {
    __shared__ uint32_t wave_mx[kOneThreads / 64];
    const int tensor = blockIdx.x >= (unsigned)a.slices;
    const int slice = (int)blockIdx.x - tensor * a.slices;
    const T* src = static_cast<const T*>(tensor ? a.src[1] : a.src[0]) + (size_t)slice * a.elems;
    const int units = (int)(a.elems / kUnitElems), tid = threadIdx.x;
    Unit<T> u[N];
    uint32_t mx = 0;
#pragma unroll
    for (int i = 0; i < N; ++i)
        if (tid + i * kOneThreads < units) u[i] = load_unit<false>(src + (size_t)(tid + i * kOneThreads) * kUnitElems);
#pragma unroll
    for (int i = 0; i < N; ++i)
        if (tid + i * kOneThreads < units) mx = max(mx, unit_max(u[i]));
    mx = wave_max(mx);
    if ((tid & 63) == 0) wave_mx[tid >> 6] = mx;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kOneThreads / 64; ++i) mx = max(mx, wave_mx[i]);
    const Scale sc = make_scale(from_bits<T>(mx));
    uint8_t* dst = (tensor ? a.dst[1] : a.dst[0]) + (size_t)slice * a.elems;
#pragma unroll
    for (int i = 0; i < N; ++i)
        if (tid + i * kOneThreads < units) {
            const size_t at = (size_t)(tid + i * kOneThreads) * kUnitElems;
            store_unit<false>(u[i], sc, dst + at);
        }
    if (tid == 0) (tensor ? a.scale[1] : a.scale[0])[slice] = sc.s;
}

// Workgroup -> (tensor, slice, piece), thread -> unit.
template <typename T, bool WRITE>
__global__ __launch_bounds__(kThreads) void quantize_pieces_kernel(QuantArgs a) {
    __shared__ uint32_t wave_mx[kThreads / 64];
    const unsigned row = blockIdx.x / (unsigned)a.pieces;      // tensor * slices + slice
    const int piece = (int)(blockIdx.x - row * (unsigned)a.pieces);
    const int tensor = row >= (unsigned)a.slices;
    const int slice = (int)row - tensor * a.slices, tid = threadIdx.x;
    const T* src = static_cast<const T*>(tensor ? a.src[1] : a.src[0]) + (size_t)slice * a.elems;
    const int64_t at = ((int64_t)piece * kThreads + tid) * kUnitElems;
    Unit<T> u;
    uint32_t mx = 0;
    if (at < a.elems) {
        u = load_unit<WRITE>(src + at);
        if constexpr (!WRITE) mx = unit_max(u);
    }
    if constexpr (WRITE)
        for (int i = tid; i < a.pieces; i += kThreads) mx = max(mx, a.part[(size_t)row * a.pieces + i]);
    mx = wave_max(mx);
    if ((tid & 63) == 0) wave_mx[tid >> 6] = mx;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kThreads / 64; ++i) mx = max(mx, wave_mx[i]);
    if constexpr (!WRITE) {
        if (tid == 0) a.part[(size_t)row * a.pieces + piece] = mx;
    } else {
        const Scale sc = make_scale(from_bits<T>(mx));
        uint8_t* dst = (tensor ? a.dst[1] : a.dst[0]) + (size_t)slice * a.elems;
        if (at < a.elems) store_unit<true>(u, sc, dst + at);
        if (tid == 0 && piece == 0) (tensor ? a.scale[1] : a.scale[0])[slice] = sc.s;
    }
}

// Units a thread of the one-launch kernel may hold: 64 registers of data.  Above that two launches are faster as well: a
// workgroup alone draws at most ~50 GB/s per CU, and there are few slices.
template <typename T> constexpr int one_launch_units() { return 64 / (4 * Unit<T>::kWords) < 4 ? 64 / (4 * Unit<T>::kWords) : 4; }

int64_t pieces_of(int64_t elems) {
    const int64_t per = (int64_t)kThreads * kUnitElems;
    return (elems + per - 1) / per;
}

bool one_launch(int64_t elems, int dtype) {
    const int n = dtype == FSTA_F32 ? one_launch_units<float>() : one_launch_units<__half>();
    return elems <= (int64_t)n * kOneThreads * kUnitElems;
}

template <typename T> int launch_quantize(QuantArgs a, int tensors, int dtype, double grid_threads, hipStream_t stream) {
    if (one_launch(a.elems, dtype)) {
        const dim3 grid((unsigned)(tensors * a.slices)), block(kOneThreads);
        constexpr int kMost = one_launch_units<T>();
        if (a.elems <= (int64_t)kOneThreads * kUnitElems)
            hipLaunchKernelGGL((quantize_slice_kernel<T, 1>), grid, block, 0, stream, a);
        else
            hipLaunchKernelGGL((quantize_slice_kernel<T, kMost>), grid, block, 0, stream, a);
    } else {
        // (both tensors in a grid, or one after the other where that would be more threads than a grid has)
        const int64_t each = (int64_t)a.slices * a.pieces;
        const int in_grid = (double)tensors * (double)each * kThreads < grid_threads ? tensors : 1;
        for (int t = 0; t < tensors; t += in_grid) {
            if (t > 0) {
                a.src[0] = a.src[1];
                a.dst[0] = a.dst[1];
                a.scale[0] = a.scale[1];
            }
            const dim3 grid((unsigned)(in_grid * each)), block(kThreads);
            hipLaunchKernelGGL((quantize_pieces_kernel<T, false>), grid, block, 0, stream, a);
            FSTA_HIP_OK(hipGetLastError());
            hipLaunchKernelGGL((quantize_pieces_kernel<T, true>), grid, block, 0, stream, a);
            FSTA_HIP_OK(hipGetLastError());
        }
    }
    FSTA_HIP_OK(hipGetLastError());
    return FSTA_OK;
}

}  // namespace
}  // namespace fsta

using namespace fsta;

extern "C" size_t fsta_quantize_workspace_bytes(int64_t slices, int64_t elements, int32_t dtype) {
    if (slices <= 0 || elements <= 0 || one_launch(elements, dtype)) return 0;
    return (size_t)(2 * slices * pieces_of(elements)) * sizeof(uint32_t);
}

// fsta_quantize_fp8 for a grid that ends before `grid_threads` threads: tests reach the way of two launches per tensor with
// tensors of ordinary size.  Not part of the interface.
extern "C" int fsta_internal_quantize_fp8(const void* a, const void* b, void* a8, void* b8, float* a_scale, float* b_scale,
                                          int64_t slices, int64_t elements, int32_t dtype, void* workspace,
                                          size_t workspace_bytes, double grid_threads, void* stream) {
    if (slices < 0 || elements < 0 || elements % kUnitElems != 0)
        return fail(FSTA_EINVAL, "fsta_quantize_fp8: slices=%lld elements=%lld (need a multiple of 16)", (long long)slices,
                    (long long)elements);
    if (dtype != FSTA_F32 && dtype != FSTA_F16 && dtype != FSTA_BF16) return fail(FSTA_EINVAL, "fsta_quantize_fp8: dtype=%d", dtype);
    if (slices == 0 || elements == 0) return FSTA_OK;
    if (!a || !a8 || !a_scale || (b && (!b8 || !b_scale))) return fail(FSTA_EINVAL, "fsta_quantize_fp8: null pointer");
    if (misaligned(a, 16) || misaligned(b, 16) || misaligned(a8, 16) || misaligned(b8, 16))
        return fail(FSTA_EINVAL, "fsta_quantize_fp8: tensors must be 16-byte aligned");
    if (misaligned(a_scale, 4) || misaligned(b_scale, 4) || misaligned(workspace, 4))
        return fail(FSTA_EINVAL, "fsta_quantize_fp8: scales and workspace must be 4-byte aligned");
    const int64_t pieces = pieces_of(elements);
    if (slices > 0x7fffffff || pieces > 0x7fffffff ||
        (double)slices * (one_launch(elements, dtype) ? 2.0 * kOneThreads : (double)pieces * kThreads) >= kGridThreads)
        return fail(FSTA_EUNSUPPORTED, "fsta_quantize_fp8: %lld slices of %lld elements", (long long)slices, (long long)elements);
    const size_t need = fsta_quantize_workspace_bytes(slices, elements, dtype);
    if (need && (!workspace || workspace_bytes < need))
        return fail(FSTA_EINVAL, "fsta_quantize_fp8: needs %zu bytes of workspace, got %zu", need, workspace_bytes);
    QuantArgs args;
    args.src[0] = a; args.src[1] = b;
    args.dst[0] = static_cast<uint8_t*>(a8); args.dst[1] = static_cast<uint8_t*>(b8);
    args.scale[0] = a_scale; args.scale[1] = b_scale;
    args.part = static_cast<uint32_t*>(workspace);
    args.elems = elements; args.slices = (int32_t)slices; args.pieces = (int32_t)pieces;
    const int tensors = b ? 2 : 1;
    hipStream_t s = static_cast<hipStream_t>(stream);
    switch (dtype) {
        case FSTA_F32: return launch_quantize<float>(args, tensors, dtype, grid_threads, s);
        case FSTA_F16: return launch_quantize<__half>(args, tensors, dtype, grid_threads, s);
        default: return launch_quantize<__hip_bfloat16>(args, tensors, dtype, grid_threads, s);
    }
}

extern "C" int fsta_quantize_fp8(const void* a, const void* b, void* a8, void* b8, float* a_scale, float* b_scale,
                                 int64_t slices, int64_t elements, int32_t dtype, void* workspace, size_t workspace_bytes,
                                 void* stream) {
    return fsta_internal_quantize_fp8(a, b, a8, b8, a_scale, b_scale, slices, elements, dtype, workspace, workspace_bytes,
                                      kGridThreads, stream);
}
