// k_gemv_f32: the int8 linear of fp32 activations below the GEMM's rows (the
// reference's default mode, one token or a few), exact int8 -> fp32 conversion
// and fp32 FMAs (Backend::linear_q8 / linear_q8_add,
// include/vvllm/backend/backend.h:62-65, 75-78).
#include <algorithm>

#include "common.h"
#include "device.h"

namespace vvh {

namespace {

// Sixteen codes as fp32.
__device__ __forceinline__ void codes_f32(const u4 w, float (&f)[16])
{
#pragma unroll
    for (int j = 0; j < 4; j++)
#pragma unroll
        for (int b = 0; b < 4; b++) f[4 * j + b] = (float)(int8_t)((w[j] >> (8 * b)) & 0xff);
}

}  // namespace

// ---------------------------------------------------------------------------
// A wave owns a tile of 16 output channels (ksplit waves of a block share one,
// each a contiguous range of its 128-wide k steps).  Lane l reads the 16-byte
// chunk l % 8 of one 128-byte line of rows l / 8 and 8 + l / 8, so a load covers 8
// rows x one whole line; D steps are in flight, the slot consumed refilled with
// the step D ahead (past the range: its last step again, never used).  The 8
// chunk lanes of a row are added at the end, then the ksplit waves through LDS,
// so no sum runs over more than K / 32 products in one chain at ksplit 4.  Up to 2
// activation rows travel in the ring with the weights; more are read where they
// are used.  Scales, biases and residuals are requested before the weights.
//
// Bound by latency for one 0.5B projection and by the weight stream for the
// larger ones.  Against 16 rows x 64 bytes per load with two in flight and the
// epilogue's operands loaded last (graph replay, us, M = 1): 896 x 896 3.56 -> 3.21,
// 9728 x 896 5.1 -> 4.5, 896 x 4864 12.8 -> 6.0, 17920 x 1536 12.6 -> 10.6, 1536 x 8960 22.0 ->
// 8.3; M = 8 9728 x 896 18.8 -> 15.8.
// ---------------------------------------------------------------------------
template <int MT, typename OT, int D>
__device__ __forceinline__ void gemv_f32_body(const int8_t* __restrict__ w, const float* __restrict__ x, int64_t N,
                                              int64_t K, int32_t ksplit, int64_t M, const LinArgs& a, int64_t block,
                                              int64_t mbase)
{
    constexpr bool XR = MT <= 2;  // activations in the ring
    __shared__ float red[4][MT][16];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane >> 3, c = lane & 7;
    const int ks = wave % ksplit;
    const int64_t n0 = (block * (4 / ksplit) + wave / ksplit) * kDecodeTileN;
    const bool active = n0 < N;
    const int64_t nA = n0 + r < N ? n0 + r : N - 1, nB = n0 + 8 + r < N ? n0 + 8 + r : N - 1;
    const int8_t* wa = w + nA * K;
    const int8_t* wb = w + nB * K;
    const int32_t steps = (int32_t)((K + 127) / 128), per = (steps + ksplit - 1) / ksplit;
    const int32_t s0 = ks * per, s1 = s0 + per < steps ? s0 + per : steps;
    const float* xr[MT];
#pragma unroll
    for (int m = 0; m < MT; m++) xr[m] = x + (mbase + m < M ? mbase + m : M - 1) * K;

    struct Slot {
        u4 wA, wB;
        f4 xv[XR ? MT : 1][4];
    };
    Slot ring[D];
    auto chunk = [&](int32_t s) {  // the lane's first k of step s, clamped into the row
        s = s < s1 ? s : s1 - 1;
        const int64_t k = (int64_t)s * 128 + c * 16;
        return k < K ? k : K - 16;
    };
    auto issue = [&](int u, int32_t s) {
        const int64_t k = chunk(s);
        ring[u].wA = __builtin_nontemporal_load(reinterpret_cast<const u4*>(wa + k));
        ring[u].wB = __builtin_nontemporal_load(reinterpret_cast<const u4*>(wb + k));
        if constexpr (XR) {
#pragma unroll
            for (int m = 0; m < MT; m++)
#pragma unroll
                for (int q = 0; q < 4; q++) ring[u].xv[m][q] = *reinterpret_cast<const f4*>(xr[m] + k + 4 * q);
        }
    };
    float accA[MT], accB[MT];
#pragma unroll
    for (int m = 0; m < MT; m++) accA[m] = accB[m] = 0.0f;
    auto consume = [&](int u, int32_t s) {
        const int64_t k = chunk(s);
        const bool on = (int64_t)s * 128 + c * 16 < K;
        float fa[16], fb[16];
        codes_f32(ring[u].wA, fa);
        codes_f32(ring[u].wB, fb);
#pragma unroll
        for (int m = 0; m < MT; m++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                f4 v;
                if constexpr (XR) v = ring[u].xv[m][q];
                else v = *reinterpret_cast<const f4*>(xr[m] + k + 4 * q);
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const float t = on ? v[e] : 0.0f;
                    accA[m] = __builtin_fmaf(t, fa[4 * q + e], accA[m]);
                    accB[m] = __builtin_fmaf(t, fb[4 * q + e], accB[m]);
                }
            }
    };

    // epilogue operands of the storing lanes: lane c == 0 of the tile's first
    // wave stores rows nA and nB of every activation row
    const bool st = active && ks == 0 && c == 0;
    const bool okA = st && n0 + r < N, okB = st && n0 + 8 + r < N;
    float sA = 0.0f, sB = 0.0f, bA = 0.0f, bB = 0.0f, rA[MT], rB[MT];
    if (st) {
        sA = a.scales[nA];
        sB = a.scales[nB];
        if (a.bias) {
            bA = a.bias[nA];
            bB = a.bias[nB];
        }
    }
#pragma unroll
    for (int m = 0; m < MT; m++) {
        rA[m] = rB[m] = 0.0f;
        if (st && a.res && mbase + m < M) {
            rA[m] = ld_f(static_cast<const OT*>(a.res) + (mbase + m) * N + nA);
            rB[m] = ld_f(static_cast<const OT*>(a.res) + (mbase + m) * N + nB);
        }
    }
    if (active && s0 < s1) {
#pragma unroll
        for (int u = 0; u < D; u++) issue(u, s0 + u);
        int32_t s = s0;
        for (; s + D < s1; s += D) {
#pragma unroll
            for (int u = 0; u < D; u++) {
                consume(u, s + u);
                __builtin_amdgcn_sched_barrier(0);
                issue(u, s + u + D);
            }
        }
#pragma unroll
        for (int u = 0; u < D; u++)
            if (s + u < s1) consume(u, s + u);
    }
#pragma unroll
    for (int m = 0; m < MT; m++) {
        accA[m] = group_sum(accA[m], 8);
        accB[m] = group_sum(accB[m], 8);
    }
    if (ksplit > 1) {
        if (c == 0) {
#pragma unroll
            for (int m = 0; m < MT; m++) {
                red[wave][m][r] = accA[m];
                red[wave][m][8 + r] = accB[m];
            }
        }
        __syncthreads();
        if (st) {
#pragma unroll
            for (int m = 0; m < MT; m++)
                for (int j = 1; j < ksplit; j++) {
                    accA[m] += red[wave + j][m][r];
                    accB[m] += red[wave + j][m][8 + r];
                }
        }
    }
#pragma unroll
    for (int m = 0; m < MT; m++) {
        if (mbase + m >= M) continue;
        OT* o = static_cast<OT*>(a.out) + (mbase + m) * N;
        float yA = accA[m] * sA, yB = accB[m] * sB;
        if (a.bias) {
            yA += bA;
            yB += bB;
        }
        if (a.res) {
            yA += rA[m];
            yB += rB[m];
        }
        if (okA) st_f(o + nA, yA);
        if (okB) st_f(o + nB, yB);
    }
}

// The grid row's pass of up to MT activation rows.  The rows past M of the last
// one would cost what the others do, so it runs a body of 1, 2, 4, 6 or 8 rows
// (graph replay, us, all passes of 8 -> these: M = 9 9728 x 896 23.6 -> 14.6, 17920 x
// 1536 58.6 -> 42.4; M = 5 17920 x 1536 37.3 -> 29.7).
template <int MT, typename OT, int D>
__device__ __forceinline__ void gemv_f32_pass(const int8_t* __restrict__ w, const float* __restrict__ x, int64_t N,
                                              int64_t K, int32_t ksplit, int64_t M, const LinArgs& a, int64_t block)
{
    const int64_t mbase = (int64_t)blockIdx.y * MT;
    if constexpr (MT == 8) {
        const int64_t rows = M - mbase;
        if (rows == 1) return gemv_f32_body<1, OT, D>(w, x, N, K, ksplit, M, a, block, mbase);
        if (rows == 2) return gemv_f32_body<2, OT, D>(w, x, N, K, ksplit, M, a, block, mbase);
        if (rows <= 4) return gemv_f32_body<4, OT, D>(w, x, N, K, ksplit, M, a, block, mbase);
        if (rows <= 6) return gemv_f32_body<6, OT, D>(w, x, N, K, ksplit, M, a, block, mbase);
    }
    gemv_f32_body<MT, OT, D>(w, x, N, K, ksplit, M, a, block, mbase);
}

// What the first loads depend on comes first (10 dwords, preloaded into
// registers at dispatch).
template <int MT, typename OT, int D>
__global__ __launch_bounds__(256) void k_gemv_f32(const int8_t* __restrict__ w, const float* __restrict__ x, int64_t N,
                                                  int64_t K, int32_t ksplit, int32_t M, LinArgs a)
{
    gemv_f32_pass<MT, OT, D>(w, x, N, K, ksplit, M, a, blockIdx.x);
}

// The problems of a plan (q, k and v of a decode layer) in one launch.
template <int MT, typename OT, int D>
__global__ __launch_bounds__(256) void k_gemv_f32_group(LinGroup l)
{
    const int b = blockIdx.x;
    const LinArgs a = l.g.p[(b >= l.b[0]) + (b >= l.b[1]) + (b >= l.b[2])];
    gemv_f32_pass<MT, OT, D>(a.w, static_cast<const float*>(a.inp), a.N, a.K, a.ksplit, a.M, a, b - a.block_begin);
}

namespace {

// Rows of a pass: the fewest that take the call's, up to 8.
int gemv_rows(int64_t M) { return M <= 2 ? (int)std::max<int64_t>(M, 1) : M <= 4 ? 4 : M <= 6 ? 6 : 8; }

// Steps in flight: the wave's whole range where it is short (2, or 5 to 7 steps),
// else 4 (see dot_depth).
int gemv_depth(int64_t K, int32_t ksplit, int mt)
{
    const int64_t per = dot_wave_steps(K, ksplit);
    return per <= 2 ? 2 : mt == 1 && per >= 5 && per <= 7 ? 7 : 4;
}

template <int MT, typename OT>
void gemv_go(const LinArgs& a, int d, hipStream_t s)
{
    const dim3 grid((unsigned)decode_blocks(a), (unsigned)((a.M + MT - 1) / MT));
    const float* x = static_cast<const float*>(a.inp);
#define VVH_GEMV(D) \
    hipLaunchKernelGGL((k_gemv_f32<MT, OT, D>), grid, dim3(256), 0, s, a.w, x, a.N, a.K, a.ksplit, (int32_t)a.M, a)
    if (MT == 1 && d == 7) VVH_GEMV((MT == 1 ? 7 : 4));
    else if (d == 2) VVH_GEMV(2);
    else VVH_GEMV(4);
#undef VVH_GEMV
}

template <int MT, typename OT>
void gemv_group_go(const LinGroup& l, int d, hipStream_t s)
{
    const dim3 grid((unsigned)l.blocks, (unsigned)((l.g.p[0].M + MT - 1) / MT));
    if (d == 2) hipLaunchKernelGGL((k_gemv_f32_group<MT, OT, 2>), grid, dim3(256), 0, s, l);
    else hipLaunchKernelGGL((k_gemv_f32_group<MT, OT, 4>), grid, dim3(256), 0, s, l);
}

}  // namespace

int launch_gemv_f32(const LinArgs& a, int out, void* stream)
{
    hipStream_t s = static_cast<hipStream_t>(stream);
    const int mt = gemv_rows(a.M);
    const int d = gemv_depth(a.K, a.ksplit, mt);
    auto go = [&]<typename OT>(OT*) {
        switch (mt) {
            case 1: gemv_go<1, OT>(a, d, s); break;
            case 2: gemv_go<2, OT>(a, d, s); break;
            case 4: gemv_go<4, OT>(a, d, s); break;
            case 6: gemv_go<6, OT>(a, d, s); break;
            default: gemv_go<8, OT>(a, d, s); break;
        }
    };
    if (out == VVH_F32) go(static_cast<float*>(nullptr));
    else go(static_cast<f16*>(nullptr));
    return (int)hipGetLastError();
}

int launch_gemv_f32_group(const LinGroup& l, int count, int out, void* stream)
{
    hipStream_t s = static_cast<hipStream_t>(stream);
    const int64_t M = l.g.p[0].M;
    const int mt = gemv_rows(M);
    int d = 2;
    for (int i = 0; i < count; i++) d = std::max(d, gemv_depth(l.g.p[i].K, l.g.p[i].ksplit, 2));
    auto go = [&]<typename OT>(OT*) {
        switch (mt) {
            case 1: gemv_group_go<1, OT>(l, d, s); break;
            case 2: gemv_group_go<2, OT>(l, d, s); break;
            case 4: gemv_group_go<4, OT>(l, d, s); break;
            case 6: gemv_group_go<6, OT>(l, d, s); break;
            default: gemv_group_go<8, OT>(l, d, s); break;
        }
    };
    if (out == VVH_F32) go(static_cast<float*>(nullptr));
    else go(static_cast<f16*>(nullptr));
    return (int)hipGetLastError();
}

}  // namespace vvh
