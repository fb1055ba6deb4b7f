// Auxiliary device kernels of the linear path: the per-channel quantizer,
// dtype conversion, and a counter-based normal generator for synthetic data.
#include <hip/hip_runtime.h>

#include "common.h"

namespace vvh {

typedef _Float16 f16;

// ---------------------------------------------------------------------------
// quantize_per_channel on the device (src/quantize/quantize.cc:9-48).
// One block per row.  The absmax uses the reference's comparison
// `std::max(absmax, |w|)` == (absmax < |w|) ? |w| : absmax, which ignores NaN;
// max is exact, so the reduction order cannot change the result.  The scale
// and its reciprocal are IEEE-correct fp32 divisions (this file is compiled
// with -fhip-fp32-correctly-rounded-divide-sqrt and without fast-math), the
// code is round-half-away-from-zero (roundf) of w * (1/scale), clamped with
// the reference's argument order so NaN becomes +127.
// ---------------------------------------------------------------------------
__device__ __forceinline__ float ref_max(float a, float b) { return (a < b) ? b : a; }
__device__ __forceinline__ float ref_min(float a, float b) { return (b < a) ? b : a; }

// Source elements: fp32, or BF16 bits widened exactly to fp32 (the bits
// become the high half of the fp32 word, as the reference's loader does,
// src/safetensors/safetensors.cc:135-141).
__device__ __forceinline__ float src_f32(const float* w, int64_t i) { return w[i]; }
__device__ __forceinline__ float src_f32(const uint16_t* w, int64_t i)
{
    return __builtin_bit_cast(float, (uint32_t)w[i] << 16);
}

template <typename ST>
__global__ __launch_bounds__(256) void k_quantize(const ST* __restrict__ w, int64_t N, int64_t K,
                                                  int8_t* __restrict__ q, float* __restrict__ scales)
{
    __shared__ float part[4];
    __shared__ float row_scale;
    for (int64_t row = blockIdx.x; row < N; row += gridDim.x) {
        const ST* wr = w + row * K;
        float mx = 0.0f;
        for (int64_t k = threadIdx.x; k < K; k += 256) mx = ref_max(mx, __builtin_fabsf(src_f32(wr, k)));
        for (int off = 32; off > 0; off >>= 1) mx = ref_max(mx, __shfl_xor(mx, off));
        if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = mx;
        __syncthreads();
        if (threadIdx.x == 0) {
            float absmax = ref_max(ref_max(part[0], part[1]), ref_max(part[2], part[3]));
            const float scale = absmax / 127.0f;
            scales[row] = scale;
            row_scale = scale;
        }
        __syncthreads();
        const float scale = row_scale;
        int8_t* qr = q + row * K;
        if (scale == 0.0f) {
            for (int64_t k = threadIdx.x; k < K; k += 256) qr[k] = 0;
        } else {
            const float inv_scale = 1.0f / scale;
            for (int64_t k = threadIdx.x; k < K; k += 256) {
                float val = src_f32(wr, k) * inv_scale;
                val = ref_max(-128.0f, ref_min(127.0f, roundf(val)));
                qr[k] = (int8_t)val;
            }
        }
        __syncthreads();
    }
}

int launch_quantize(const void* w, int src_dtype, int64_t N, int64_t K, int8_t* q, float* scales, void* stream)
{
    const int64_t grid = N < 65536 ? N : 65536;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (src_dtype == VVH_BF16)
        hipLaunchKernelGGL(k_quantize<uint16_t>, dim3((unsigned)grid), dim3(256), 0, s,
                           static_cast<const uint16_t*>(w), N, K, q, scales);
    else
        hipLaunchKernelGGL(k_quantize<float>, dim3((unsigned)grid), dim3(256), 0, s,
                           static_cast<const float*>(w), N, K, q, scales);
    return (int)hipGetLastError();
}

// ---------------------------------------------------------------------------
// dtype conversion (round to nearest even), grid-stride.
// ---------------------------------------------------------------------------
template <typename DT, typename ST>
__global__ __launch_bounds__(256) void k_convert(DT* __restrict__ d, const ST* __restrict__ s, int64_t n)
{
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256)
        d[i] = (DT)(float)s[i];
}

// The same, 8 elements a thread in 16-byte accesses, for 32-byte aligned rows; the
// thread after the whole chunks takes the remainder.
template <typename DT, typename ST>
__global__ __launch_bounds__(256) void k_convert_vec(DT* __restrict__ d, const ST* __restrict__ s, int64_t n)
{
    typedef DT d8 __attribute__((ext_vector_type(8)));
    typedef ST s8 __attribute__((ext_vector_type(8)));
    const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 8;
    if (i + 8 <= n) {
        const s8 v = *reinterpret_cast<const s8*>(s + i);
        d8 o;
#pragma unroll
        for (int e = 0; e < 8; e++) o[e] = (DT)(float)v[e];
        *reinterpret_cast<d8*>(d + i) = o;
    } else {
        for (int64_t e = i; e < n; e++) d[e] = (DT)(float)s[e];
    }
}

template <typename DT, typename ST>
static void convert_go(DT* d, const ST* src, int64_t n, hipStream_t s)
{
    const int64_t want = (n + 255) / 256;
    if (((reinterpret_cast<uintptr_t>(d) | reinterpret_cast<uintptr_t>(src)) & 31) == 0 && (n + 2047) / 2048 <= (1 << 22))
        hipLaunchKernelGGL((k_convert_vec<DT, ST>), dim3((unsigned)(n > 0 ? (n + 2047) / 2048 : 1)), dim3(256), 0, s, d, src, n);
    else
        hipLaunchKernelGGL((k_convert<DT, ST>), dim3((unsigned)(want < 16384 ? (want > 0 ? want : 1) : 16384)), dim3(256), 0,
                           s, d, src, n);
}

int launch_convert(void* dst, int dst_dtype, const void* src, int src_dtype, int64_t n, void* stream)
{
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (dst_dtype == VVH_F16 && src_dtype == VVH_F32) convert_go((f16*)dst, (const float*)src, n, s);
    else if (dst_dtype == VVH_F32 && src_dtype == VVH_F16) convert_go((float*)dst, (const f16*)src, n, s);
    else if (dst_dtype == VVH_F32) convert_go((float*)dst, (const float*)src, n, s);
    else convert_go((f16*)dst, (const f16*)src, n, s);
    return (int)hipGetLastError();
}

// ---------------------------------------------------------------------------
// Synthetic N(mean, std) data: element i draws h = splitmix64(seed ^ i*phi),
// u1 = (top 24 bits + 0.5) / 2^24 in (0, 1), u2 = next 24 bits / 2^24, and
// takes the Box-Muller cosine branch in fp32.
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint64_t splitmix64(uint64_t z)
{
    z += 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

template <typename T>
__global__ __launch_bounds__(256) void k_fill_normal(T* __restrict__ d, int64_t n, uint64_t seed, float mean,
                                                     float std)
{
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
        const uint64_t h = splitmix64(seed ^ ((uint64_t)i * 0x9E3779B97F4A7C15ull));
        const float u1 = ((float)(h >> 40) + 0.5f) * (1.0f / 16777216.0f);
        const float u2 = (float)((h >> 16) & 0xFFFFFFull) * (1.0f / 16777216.0f);
        const float z = sqrtf(-2.0f * logf(u1)) * cosf(6.283185307179586f * u2);
        d[i] = (T)(mean + std * z);
    }
}

// ---------------------------------------------------------------------------
// fp32 activations for the fp16 MFMA GEMM: row m of x [M, K] becomes row m of
// xs [M, 2K] fp16, the low parts lo_k = fp16(x_k * s - hi_k) followed by the high
// parts hi_k = fp16(x_k * s), with s = 2^p chosen per row so that the
// row's largest |x| * s lies in [2^14, 2^15) (in range for fp16 with room for
// its 11-bit significand), and rs[m] = 1/s.  x_k * s is exact (a power of
// two), x_k * s - hi_k is exact (Sterbenz), so hi + lo carries x_k * s to
// about 22 bits (or to the fp16 subnormal step 2^-24 of the scaled row); the
// int8 x fp16 products of both parts are exact in the GEMM's fp32
// accumulation.  The low parts come first: while their sum grows it is small,
// and so are its roundings; after the high parts each would round the whole
// sum (error against 64 bits of unsplit calls: K = 896 3.1e-7 -> 1.6e-7).
// A row without a finite nonzero maximum (all zeros, or
// containing Inf or NaN) keeps s = 1, so Inf and NaN reach the sums as such.
// One block per row, read once: C chunks of 4 values per thread (K % 4 == 0,
// 16-byte aligned rows), or two passes.
// ---------------------------------------------------------------------------
__device__ __forceinline__ float split_max(float mx, float x)
{
    // an Inf or NaN anywhere in the row makes the row maximum Inf
    const float v = __builtin_fabsf(x);
    return __builtin_isfinite(v) ? fmaxf(mx, v) : __builtin_inff();
}

// The row's scale s = 2^p from the threads' maxima; rs = 1/s.
__device__ __forceinline__ float split_scale(float mx, float* part, float* rs)
{
    for (int off = 32; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off));
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(part[0], part[1]), fmaxf(part[2], part[3]));
    int p = 0;
    if (mx > 0.0f && __builtin_isfinite(mx)) {
        int e;
        (void)frexpf(mx, &e);          // mx = f * 2^e, f in [0.5, 1)
        p = 15 - e;                    // mx * 2^p in [2^14, 2^15)
        p = p < -126 ? -126 : (p > 126 ? 126 : p);
    }
    if (threadIdx.x == 0) *rs = ldexpf(1.0f, -p);
    return ldexpf(1.0f, p);
}

__device__ __forceinline__ void split_parts(float v, f16& hi, f16& lo)
{
    hi = (f16)v;
    lo = __builtin_isfinite((float)hi) ? (f16)(v - (float)hi) : (f16)0.0f;
}

__global__ __launch_bounds__(256) void k_split_f32(const float* __restrict__ x, int64_t K, f16* __restrict__ xs,
                                                   float* __restrict__ rs)
{
    __shared__ float part[4];
    const int64_t m = blockIdx.x;
    const float* xr = x + m * K;
    float mx = 0.0f;
    for (int64_t k = threadIdx.x; k < K; k += 256) mx = split_max(mx, xr[k]);
    const float s = split_scale(mx, part, rs + m);
    f16* lr = xs + m * 2 * K;
    for (int64_t k = threadIdx.x; k < K; k += 256) split_parts(xr[k] * s, lr[K + k], lr[k]);
}

template <int C>
__global__ __launch_bounds__(256) void k_split_f32_rows(const float* __restrict__ x, int32_t K, f16* __restrict__ xs,
                                                        float* __restrict__ rs)
{
    typedef float f4 __attribute__((ext_vector_type(4)));
    typedef _Float16 h4 __attribute__((ext_vector_type(4)));
    __shared__ float part[4];
    const int64_t m = blockIdx.x;
    const f4* xr = reinterpret_cast<const f4*>(x + m * K);
    const int kc = K / 4;
    f4 v[C];
#pragma unroll
    for (int c = 0; c < C; c++) {
        const int i = threadIdx.x + 256 * c;
        v[c] = xr[i < kc ? i : kc - 1];  // past the row: its last chunk again
    }
    float mx = 0.0f;
#pragma unroll
    for (int c = 0; c < C; c++)
#pragma unroll
        for (int e = 0; e < 4; e++) mx = split_max(mx, v[c][e]);
    const float s = split_scale(mx, part, rs + m);
    f16* lr = xs + m * 2 * K;
#pragma unroll
    for (int c = 0; c < C; c++) {
        const int i = threadIdx.x + 256 * c;
        if (i >= kc) continue;
        h4 hi, lo;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            f16 h, l;
            split_parts(v[c][e] * s, h, l);
            hi[e] = h;
            lo[e] = l;
        }
        *reinterpret_cast<h4*>(lr + 4 * i) = lo;
        *reinterpret_cast<h4*>(lr + K + 4 * i) = hi;
    }
}

int launch_split_f32(const float* x, int64_t M, int64_t K, void* xs, float* rs, void* stream)
{
    if (M <= 0) return 0;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const dim3 grid((unsigned)M);
    f16* o = static_cast<f16*>(xs);
    const bool rows = K % 4 == 0 && reinterpret_cast<uintptr_t>(x) % 16 == 0 && reinterpret_cast<uintptr_t>(xs) % 8 == 0;
    if (rows && K <= 1024) hipLaunchKernelGGL(k_split_f32_rows<1>, grid, dim3(256), 0, s, x, (int32_t)K, o, rs);
    else if (rows && K <= 2048) hipLaunchKernelGGL(k_split_f32_rows<2>, grid, dim3(256), 0, s, x, (int32_t)K, o, rs);
    else if (rows && K <= 5120) hipLaunchKernelGGL(k_split_f32_rows<5>, grid, dim3(256), 0, s, x, (int32_t)K, o, rs);
    else if (rows && K <= 9216) hipLaunchKernelGGL(k_split_f32_rows<9>, grid, dim3(256), 0, s, x, (int32_t)K, o, rs);
    else hipLaunchKernelGGL(k_split_f32, grid, dim3(256), 0, s, x, K, o, rs);
    return (int)hipGetLastError();
}

int launch_fill_normal(void* dst, int dtype, int64_t n, uint64_t seed, float mean, float std, void* stream)
{
    const int64_t want = (n + 255) / 256;
    const dim3 grid((unsigned)(want < 16384 ? (want > 0 ? want : 1) : 16384));
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (dtype == VVH_F32)
        hipLaunchKernelGGL((k_fill_normal<float>), grid, dim3(256), 0, s, (float*)dst, n, seed, mean, std);
    else
        hipLaunchKernelGGL((k_fill_normal<f16>), grid, dim3(256), 0, s, (f16*)dst, n, seed, mean, std);
    return (int)hipGetLastError();
}

}  // namespace vvh
