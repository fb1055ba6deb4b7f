// Dense linear of several rows on the matrix cores (Backend::linear /
// linear_add, backend_naive.cc:139-156, :302-320; the model run without
// quantization): out[m][n] = sum_k x[m][k] W[n][k] + bias[n] (+ res[m][n]),
// activations and weights both fp16 or both fp32.  The forms for up to 4 rows,
// mixed types and odd K are in model_kernels.hip.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "common.h"
#include "device.h"

namespace vvh {

namespace {

template <typename T>
struct DenseVec;
template <>
struct DenseVec<f16> {
    typedef h8 chunk;                                          // 16 bytes of a row
    typedef _Float16 out4 __attribute__((ext_vector_type(4)));
};
template <>
struct DenseVec<float> {
    typedef f4 chunk;
    typedef f4 out4;
};

// One 16-byte chunk of a W row (A) and of an x row (B) per lane: fp16, one
// 32x32x16 MFMA; fp32, four 32x32x2 with an accumulator each.  The k of a
// slot is the same in both.
__device__ __forceinline__ void dense_mma(const h8 a, const h8 b, f16v (&c)[1])
{
    c[0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c[0], 0, 0, 0);
}
__device__ __forceinline__ void dense_mma(const f4 a, const f4 b, f16v (&c)[4])
{
#pragma unroll
    for (int w = 0; w < 4; w++) c[w] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[w], b[w], c[w], 0, 0, 0);
}

// 16 bytes per lane at byte offset off of r to LDS, lane i's at dst + 16 i
__device__ __forceinline__ void load_lds16(__amdgpu_buffer_rsrc_t r, char* dst, uint32_t off)
{
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, dst, 16, off, 0, 0, 0);
}

// out = acc + bias (+ res) of 4 consecutive columns, one rounding
template <typename T>
__device__ __forceinline__ void dense_store4(T* out, const T* res, const float* bias, int64_t o, int64_t n, int64_t N,
                                             bool vec, f4 y)
{
    typedef typename DenseVec<T>::out4 V;
    if (vec) {
        if (bias) y += *reinterpret_cast<const f4*>(bias + n);
        if (res) {
            const V r = *reinterpret_cast<const V*>(res + o);
#pragma unroll
            for (int e = 0; e < 4; e++) y[e] += (float)r[e];
        }
        V v;
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = (T)y[e];
        *reinterpret_cast<V*>(out + o) = v;
    } else {
        for (int e = 0; e < 4 && n + e < N; e++) {
            float t = y[e] + (bias ? bias[n + e] : 0.0f);
            if (res) t += (float)res[o + e];
            out[o + e] = (T)t;
        }
    }
}

}  // namespace

// ---------------------------------------------------------------------------
// Block tile BM x 64 (x rows by W rows), k stages of 128 bytes per row (64 fp16
// or 32 fp32 values) in a ring of 4, filled straight from memory.  The 4 waves
// share the tile and take two of every stage's eight 16-byte chunks each; their
// sums are added through LDS at the end.  The products are computed transposed
// (W rows as the A operand), so a lane holds 4 consecutive columns of one
// output row per accumulator group.
//
// fp32: v_mfma_f32_32x32x2_f32, exact products, fp32 sums.  Four accumulators
// take turns, and every 4 stages they are added to a fifth, so a chain runs over
// 4 products' additions and then K / 128; the four waves' sums are added in 64
// bits.  That is closer to 64 bits than the vector form's 64 lanes and their
// butterfly at every K (relative error, 2-norm: K = 256 7.7e-8 against 8.1e-8, 512
// 8.2e-8 against 8.5e-8, 896 8.9e-8 against 9.8e-8, 4864 1.0e-7 against 1.7e-7; with
// the waves' sums added in 32 bits 8.2e-8 and 8.7e-8 at K = 256 and 512, in the
// same time; two accumulators, folded every 4 or 2 stages, 1.0e-7 at K = 896).
// Bound by the fp32 matrix rate (256 flop per clock and CU) where the tiles fill
// the chip.
// fp16: v_mfma_f32_32x32x16_f16; bound by the fill of LDS.
// Against k_dense_vec (graph replay, us): fp32 128 x 4864 x 896 108 -> 27, 128 x 896 x
// 4864 389 -> 22, 512 x 4864 x 896 435 -> 62; fp16 109 -> 9.8, 267 -> 12.6, 572 -> 19.4.
//
// Split-K (gridDim.y > 1, few tiles over a long K): block (tile, s) takes the
// stages [s per, (s + 1) per) and writes its sums to plane s of ws [s][M][N];
// k_dense_reduce adds the planes in order and applies the epilogue.
// ---------------------------------------------------------------------------
template <typename T, int BM>
__global__ __launch_bounds__(256, 2) void k_dense_mfma(const T* __restrict__ x, const T* __restrict__ w, int32_t M,
                                                       int32_t N, int32_t K, const float* __restrict__ bias, const T* res,
                                                       T* out, float* __restrict__ ws)
{
    constexpr int D = 4;                       // stages in the ring
    constexpr int E = 16 / (int)sizeof(T);     // values per chunk
    constexpr int SK = 8 * E;                  // k per stage
    constexpr int BN = 64, TI = BM / 32, TJ = BN / 32;  // 32 x 32 tiles: x rows, W rows
    constexpr int LA = BM / 32, LB = BN / 32;  // 1 KB loads (8 rows) per wave and stage
    constexpr int LPS = LA + LB;
    constexpr bool TWO = sizeof(T) == 4;       // sums of the accumulators
    constexpr int NA = TWO ? 4 : 1;            // accumulators per tile
    typedef typename DenseVec<T>::chunk C;
    constexpr int kStage = (BM + BN) * SK;     // values: x rows, then W rows
    static_assert(kStage * (int)sizeof(T) >= BM * BN * 4, "a wave's sums in each stage");
    __shared__ __align__(1024) T st0[kStage], st1[kStage], st2[kStage], st3[kStage];

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ln = lane & 31, hb = lane >> 5;
    const int nbm = (M + BM - 1) / BM;
    // row blocks fastest: the blocks of a column of tiles share its W rows in one XCD's L2
    const int tile = (int)xcd_remap(blockIdx.x, gridDim.x);
    const int mb = tile % nbm, nb = tile / nbm;
    const int m0 = mb * BM, n0 = nb * BN;
    const int stages = (K + SK - 1) / SK, per = (stages + (int)gridDim.y - 1) / (int)gridDim.y;
    const int s0 = (int)blockIdx.y * per, s1 = s0 + per < stages ? s0 + per : stages;

    // rows past M or N read the last valid row (their results are not stored),
    // chunks past K the row's last chunk (zeroed where they are used)
    const int64_t xb = ((int64_t)M - m0) * K * sizeof(T), wb = ((int64_t)N - n0) * K * sizeof(T);
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<T*>(x + (int64_t)m0 * K), 0, (int)(uint32_t)(xb < 0xFFFFFFFFll ? xb : 0xFFFFFFFFll), 0x00020000);
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<T*>(w + (int64_t)n0 * K), 0, (int)(uint32_t)(wb < 0xFFFFFFFFll ? wb : 0xFFFFFFFFll), 0x00020000);
    uint32_t ao[LA], bo[LB];  // byte offset of the lane's row
    int ac[LA], bc[LB];       // the lane's chunk of a stage
#pragma unroll
    for (int i = 0; i < LA; i++) {
        const int r = (wave * LA + i) * 8 + (lane >> 3);
        ao[i] = (uint32_t)(m0 + r < M ? r : M - 1 - m0) * (uint32_t)K * (uint32_t)sizeof(T);
        ac[i] = swz_a(r, lane & 7);
    }
#pragma unroll
    for (int i = 0; i < LB; i++) {
        const int r = (wave * LB + i) * 8 + (lane >> 3);
        bo[i] = (uint32_t)(n0 + r < N ? r : N - 1 - n0) * (uint32_t)K * (uint32_t)sizeof(T);
        bc[i] = swz_a(r, lane & 7);
    }
    auto ring = [&](auto S) -> T* {
        constexpr int s = decltype(S)::value % D;
        if constexpr (s == 0) return st0;
        else if constexpr (s == 1) return st1;
        else if constexpr (s == 2) return st2;
        else return st3;
    };
    const int kc = K / E;  // chunks per row
    auto issue = [&](auto S, int s) {
        char* a = reinterpret_cast<char*>(ring(S));
        char* b = a + BM * 128;
        s = s < stages ? s : stages - 1;  // past the end: a stage again, never used (keeps the waits' counts)
#pragma unroll
        for (int i = 0; i < LA; i++) {
            const int c = s * 8 + ac[i] < kc ? s * 8 + ac[i] : kc - 1;
            load_lds16(rx, a + (wave * LA + i) * 1024, ao[i] + (uint32_t)c * 16);
        }
#pragma unroll
        for (int i = 0; i < LB; i++) {
            const int c = s * 8 + bc[i] < kc ? s * 8 + bc[i] : kc - 1;
            load_lds16(rw, b + (wave * LB + i) * 1024, bo[i] + (uint32_t)c * 16);
        }
    };

    f16v acc[TJ][TI][NA], sum[TWO ? TJ : 1][TWO ? TI : 1];
#pragma unroll
    for (int j = 0; j < TJ; j++)
#pragma unroll
        for (int i = 0; i < TI; i++) {
#pragma unroll
            for (int c = 0; c < NA; c++) acc[j][i][c] = f16v{};
            if constexpr (TWO) sum[j][i] = f16v{};
        }
    auto step = [&](auto S, int s) {
        constexpr auto SN = std::integral_constant<int, decltype(S)::value + D - 1>{};
        wait_vmcnt<(D - 2) * LPS>();
        lds_barrier();  // stage s in LDS for every wave; every wave is done with stage s - 1
        issue(SN, s + D - 1);
        const T* a = ring(S);
        const T* b = a + BM * SK;
        const bool tail = s * 8 + 8 > kc;
        const int c = 2 * wave + hb;  // the half-wave's chunk
        C xa[TI], wa[TJ];
#pragma unroll
        for (int i = 0; i < TI; i++)
            xa[i] = *reinterpret_cast<const C*>(a + (32 * i + ln) * SK + swz_a(ln, c) * E);
#pragma unroll
        for (int j = 0; j < TJ; j++)
            wa[j] = *reinterpret_cast<const C*>(b + (32 * j + ln) * SK + swz_a(ln, c) * E);
        if (tail) {
            const bool on = s * 8 + c < kc;
#pragma unroll
            for (int i = 0; i < TI; i++) xa[i] = on ? xa[i] : C{};
#pragma unroll
            for (int j = 0; j < TJ; j++) wa[j] = on ? wa[j] : C{};
        }
#pragma unroll
        for (int j = 0; j < TJ; j++)
#pragma unroll
            for (int i = 0; i < TI; i++) dense_mma(wa[j], xa[i], acc[j][i]);
    };
    auto fold = [&] {
        if constexpr (TWO) {
#pragma unroll
            for (int j = 0; j < TJ; j++)
#pragma unroll
                for (int i = 0; i < TI; i++) {
                    sum[j][i] += (acc[j][i][0] + acc[j][i][1]) + (acc[j][i][2] + acc[j][i][3]);
#pragma unroll
                    for (int c = 0; c < NA; c++) acc[j][i][c] = f16v{};
                }
        }
    };
    if (s0 < s1) {
        issue(std::integral_constant<int, 0>{}, s0);
        issue(std::integral_constant<int, 1>{}, s0 + 1);
        issue(std::integral_constant<int, 2>{}, s0 + 2);
        for (int s = s0; s < s1; s += D) {
            step(std::integral_constant<int, 0>{}, s);
            if (s + 1 < s1) step(std::integral_constant<int, 1>{}, s + 1);
            if (s + 2 < s1) step(std::integral_constant<int, 2>{}, s + 2);
            if (s + 3 < s1) step(std::integral_constant<int, 3>{}, s + 3);
            fold();
        }
        if constexpr (TWO) {
#pragma unroll
            for (int j = 0; j < TJ; j++)
#pragma unroll
                for (int i = 0; i < TI; i++) acc[j][i][0] = sum[j][i];
        }
    }
    wait_vmcnt<0>();
    lds_barrier();  // the ring is free

    const bool split = gridDim.y > 1;
    float* plane = ws + (int64_t)blockIdx.y * M * N;
    const bool vec = N % 4 == 0 && (split || ((reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(res)) %
                                                  (4 * sizeof(T)) == 0 && reinterpret_cast<uintptr_t>(bias) % 16 == 0));
    auto store = [&](int m, int n, f4 y) {
        if (m >= M || n >= N) return;
        const int64_t o = (int64_t)m * N + n;
        if (split) dense_store4<float>(plane, nullptr, nullptr, o, n, N, vec, y);
        else dense_store4<T>(out, res, bias, o, n, N, vec, y);
    };
    // wave g's sums in stage buffer g: row m of BN floats, 16-byte chunk q at slot q ^ (m % 8)
    auto at = [&](int g, int m, int q) {
        T* b = g == 0 ? st0 : g == 1 ? st1 : g == 2 ? st2 : st3;
        return reinterpret_cast<f4*>(b) + m * (BN / 4) + (q ^ (m & 7));
    };
#pragma unroll
    for (int j = 0; j < TJ; j++)
#pragma unroll
        for (int i = 0; i < TI; i++)
#pragma unroll
            for (int g = 0; g < 4; g++)
                *at(wave, 32 * i + ln, 8 * j + 2 * g + hb) = f4{acc[j][i][0][4 * g], acc[j][i][0][4 * g + 1],
                                                                acc[j][i][0][4 * g + 2], acc[j][i][0][4 * g + 3]};
    lds_barrier();
    for (int idx = tid; idx < BM * BN / 4; idx += 256) {
        const int m = idx / (BN / 4), q = idx % (BN / 4);
        const f4 y0 = *at(0, m, q), y1 = *at(1, m, q), y2 = *at(2, m, q), y3 = *at(3, m, q);
        f4 y;
#pragma unroll
        for (int e = 0; e < 4; e++) y[e] = (float)(((double)y0[e] + y1[e]) + ((double)y2[e] + y3[e]));
        store(m0 + m, n0 + 4 * q, y);
    }
}

// The planes of a split call added in order, and the epilogue; 4 columns per thread.
template <typename T>
__global__ __launch_bounds__(256) void k_dense_reduce(const float* __restrict__ ws, int32_t splits, int32_t M, int32_t N,
                                                      const float* __restrict__ bias, const T* res, T* out)
{
    const int64_t nq = (N + 3) / 4, i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= nq * M) return;
    const int64_t m = i / nq, n = (i - m * nq) * 4, o = m * N + n, mn = (int64_t)M * N;
    f4 y = f4{};
    if (N % 4 == 0) {
#pragma unroll 4
        for (int s = 0; s < splits; s++) y += *reinterpret_cast<const f4*>(ws + s * mn + o);
    } else {
        for (int s = 0; s < splits; s++)
            for (int e = 0; e < 4 && n + e < N; e++) y[e] += ws[s * mn + o + e];
    }
    const bool vec = N % 4 == 0 && (reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(res)) % (4 * sizeof(T)) == 0 &&
                     reinterpret_cast<uintptr_t>(bias) % 16 == 0;
    dense_store4<T>(out, res, bias, o, n, N, vec, y);
}

// Calls the MFMA form takes: both types alike, 5 rows or more, rows of whole
// 16-byte chunks, aligned, and sizes in 31 bits (rows and byte offsets within a
// tile of 64 rows).  Few rows over short ones keep the vector form, two or
// three passes over the weights, where that is faster (graph replay, us, against
// this form): fp32 calls of 5 to 8 rows over up to 2048 values (5 x 4864 x 896 9.2
// against 10.8, 8 x 896 x 896 7.6 against 8.3) and of 9 and 10 over small weights (9
// x 512 x 512 6.2 against 6.9, 9 / 10 x 896 x 896 7.4 / 7.8 against 7.9; 9 x 1200 x 1024
// 8.0 against 7.5) or of 11 over about 512 (11 x 1000 x 512 6.8 against 7.0); fp16
// calls of 5 to 8 rows over 769 to 1024 values (5 / 8 x 896 x 896 5.7 / 6.9 against 7.2, 6
// x 3000 x 1024 6.9 against 7.8, 8 x 2000 x 1000 7.4 against 7.8; 8 x 2400 x 896 7.6
// against 7.2), and over small weights of 5 and 6 rows from 512 on (5 x 512 x 512 4.8
// against 5.3) and of 5 up to 1536 (512 x 1536 6.5 against 6.8).
bool dense_mfma_ok(const void* x, const void* w, int wdtype, int64_t M, int64_t N, int64_t K, int dtype)
{
    const int64_t es = dtype == VVH_F16 ? 2 : 4;
    const int64_t nk = N * K;
    if (dtype == VVH_F32 && ((M <= 8 && K <= 2048) || (M <= 10 && K <= 1024 && nk <= 900000) ||
                             (M <= 11 && K > 384 && K <= 512 && nk <= 600000)))
        return false;
    if (dtype == VVH_F16 && ((M <= 8 && K > 768 && K <= 1024 && nk <= (M <= 6 ? 3300000 : M == 7 ? 3100000 : 2100000)) ||
                             (M <= 6 && K >= 512 && K <= (M == 5 ? 1536 : 768) && nk <= (1 << 20))))
        return false;
    return dtype == wdtype && M > 4 && K > 0 && K % (16 / es) == 0 &&
           ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w)) & 15) == 0 && M <= (1 << 30) &&
           N <= (1 << 30) && K * es * 64 < ((int64_t)1 << 31) && (M + 31) / 32 * ((N + 63) / 64) <= (1 << 30);
}

// fp32 tiles have 32 rows (on 64, with twice the registers and half the blocks,
// 512 x 896 x 896 takes 25.0 us instead of 16.3, 80 x 8960 x 1536 69 instead of 42), fp16
// ones 64 from 33 rows on (less LDS fill per product: 512 x 4864 x 896 20.6 -> 19.0).
// The k splits minimise a model fitted to forced counts (graph replay): a stage
// costs a CU with b blocks 0.1 + 0.39 b us (fp16: 0.1 + 0.24 b), a split call adds
// the reduction's launch and its planes.
DensePlan dense_plan(int64_t M, int64_t N, int64_t K, int dtype, int64_t cus)
{
    const bool f16 = dtype == VVH_F16;
    const int64_t sk = f16 ? 64 : 32, stages = (K + sk - 1) / sk;
    DensePlan p{f16 && M > 32 ? 64 : 32, 1};
    const int64_t t = (M + p.bm - 1) / p.bm * ((N + 63) / 64);
    double best = INFINITY;
    for (int64_t s = 1; s <= std::min<int64_t>(32, std::max<int64_t>(1, stages / 4)); s++) {
        const int64_t per = (stages + s - 1) / s, ce = (stages + per - 1) / per;  // no empty split
        const double b = (double)((t * ce + cus - 1) / cus);
        double us = (double)per * (0.1 + (f16 ? 0.24 : 0.39) * b);
        if (ce > 1) us += 4.0 + (double)(ce * M * N * 4) / 1e6;
        if (us < best) {
            best = us;
            p.splits = ce;
        }
    }
    return p;
}

// Whether a call that would split k is worth the reduction's launch, whose host
// time a program that issues its calls one by one pays too: two launches take it
// 9.3 to 10.6 us.  Not where the vector form is done before (issued in a row, us,
// vector / split: fp16 8 / 10 x 1536 x 1536 8.1 / 10.2 against 9.4 / 11.4, 10 x 256 x 1536
// 9.4 against 11.1, 7 x 3000 x 2048 9.1 against 10.7; fp32 16 x 512 x 512 8.0 against 9.3,
// 12 x 896 x 896 8.0 against 9.3, 10 x 1536 x 1536 9.5 against 11.0): its time fitted to
// these, passes of 4 rows over the weights and the products of a row and a value.
bool dense_split_pays(int64_t M, int64_t N, int64_t K, int dtype)
{
    const double pass = 0.8 + 0.45 * std::max(0.0, (double)(N - 2000) / 1000.0), mk = (double)M * (double)K;
    const double us = (double)((M + 3) / 4) * pass + (dtype == VVH_F32 ? 2.4 + 2.7e-4 * mk : 3.5 + 2.1e-4 * mk);
    return us > 9.6;
}

// Whether a call that would split k and has no workspace for the planes takes a
// tile's whole k in one block, or the vector form: its passes over the weights
// (2.5 us and 0.42 ns per row and value, on 2200 weight rows and more in
// proportion) against the chain of stages.  Graph replay, us, vector / unsplit:
// fp32 896 x 4864, 5 rows 16.6 / 70, 24 47.7 / 70.6, 32 67 / 70.6; fp16 5 13.4 / 26.0, 10 23.0 /
// 25.9, 12 27 / 26; 4864 x 896 fp32 12 rows 13.3 / 15.5.
bool dense_unsplit_pays(const DensePlan& p, int64_t M, int64_t N, int64_t K, int dtype, int64_t cus)
{
    const bool f16 = dtype == VVH_F16;
    const int64_t stages = (K + (f16 ? 63 : 31)) / (f16 ? 64 : 32), t = (M + p.bm - 1) / p.bm * ((N + 63) / 64);
    const double b = (double)((t + cus - 1) / cus);
    return (double)stages * (0.1 + (f16 ? 0.24 : 0.39) * b) <=
           2.5 + 4.2e-4 * (double)M * (double)K * std::max(1.0, (double)N / 2200.0);
}

int64_t dense_ws_floats(const DensePlan& p, int64_t M, int64_t N) { return p.splits > 1 ? p.splits * M * N : 0; }

template <typename T, int BM>
static void dense_go(const DensePlan& p, void* out, const void* x, const void* w, const float* bias, const void* res,
                     int64_t M, int64_t N, int64_t K, float* ws, hipStream_t s)
{
    const dim3 grid((unsigned)((M + BM - 1) / BM * ((N + 63) / 64)), (unsigned)p.splits);
    hipLaunchKernelGGL((k_dense_mfma<T, BM>), grid, dim3(256), 0, s, (const T*)x, (const T*)w, (int32_t)M, (int32_t)N,
                       (int32_t)K, bias, (const T*)res, (T*)out, ws);
    if (p.splits > 1)
        hipLaunchKernelGGL(k_dense_reduce<T>, dim3((unsigned)(((N + 3) / 4 * M + 255) / 256)), dim3(256), 0, s, ws,
                           (int32_t)p.splits, (int32_t)M, (int32_t)N, bias, (const T*)res, (T*)out);
}

int launch_dense_mfma(const DensePlan& p, void* out, const void* x, const void* w, const float* bias, const void* res,
                      int64_t M, int64_t N, int64_t K, int dtype, float* ws, void* stream)
{
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (dtype == VVH_F32) dense_go<float, 32>(p, out, x, w, bias, res, M, N, K, ws, s);
    else if (p.bm == 64) dense_go<f16, 64>(p, out, x, w, bias, res, M, N, K, ws, s);
    else dense_go<f16, 32>(p, out, x, w, bias, res, M, N, K, ws, s);
    return (int)hipGetLastError();
}

}  // namespace vvh
