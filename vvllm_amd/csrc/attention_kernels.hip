// Causal attention of several queries (the prompt, or a piece of it against
// the cache; backend_naive.cc:344-378) on the matrix cores.  The one-query
// decode forms and the general kernel are in model_kernels.hip.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "common.h"
#include "device.h"

namespace vvh {

namespace {

typedef _Float16 h4v __attribute__((ext_vector_type(4)));

__device__ __forceinline__ h4v lds_read_tr16(const f16* p)
{
    typedef short s4v __attribute__((ext_vector_type(4)));
    const s4v v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s4v*)(p));
    return __builtin_bit_cast(h4v, v);
}

// LDS slot of 16-byte chunk c of row r in a tile of D-wide fp16 rows.  Two
// kinds of reads meet no bank twice: 16 consecutive rows of one chunk (the K
// operand), and 4 consecutive rows of 4 consecutive chunks (the transposed V
// operand, whose rows must fall in different 64-byte groups).
template <int D>
__device__ __forceinline__ int attn_swz(int r)
{
    return D == 128 ? ((r & 3) << 2) | ((r >> 2) & 3) : (((r >> 1) & 1) << 2) | ((r >> 2) & 3);
}

// One row of the general kernel's arithmetic by a wave, over the `len` visible
// keys only: scores, their maximum and the sum of the exponentials, then the
// scores again and the weighted values.  For rows whose result from the tiles is
// not finite: a key past a row's last visible one has weight 0 in the tiles, and
// 0 times an infinity or NaN of its V row would reach the sums, as would an
// infinity times the 0 of a weight's low part.  A key row is shared by L lanes of
// 16 bytes, U keys of each group of lanes in flight.  M and den: the maximum (in
// log2 units, or a little less) and the sum of the weights under it that the tiles
// found, which no V row reaches; where they are not finite, or no weight is left,
// they are worked out as the general kernel does.  With an infinity in a V row
// that every query sees, us, one block per head and query (k_attention) / a wave
// per row and one key at a time / here: 512 queries, 14 heads of 64, 72 / 2390 /
// 93, fp32 92 / 2390 / 159; 2048, 12 of 128, 1820 / 9960 / 895, fp32 2030 / 20200 / 2390; 7
// after 4000 242 / 2540 / 206; a NaN or infinite key 73 / 2390 / 13 at 512 (attn_redo).
template <typename T, int D>
__device__ void attn_row_general(const T* __restrict__ qr, const T* __restrict__ kh, const T* __restrict__ vh,
                                 int64_t kvs, int len, float scale, float M, float den, T* __restrict__ orow, int lane)
{
    constexpr int E = 16 / (int)sizeof(T), L = D / E, G = 64 / L, U = (int)sizeof(T) * 2;
    typedef T te __attribute__((ext_vector_type(E)));
    const int c = lane % L, g = lane / L;
    const te qv = *reinterpret_cast<const te*>(qr + c * E);
    auto load = [&](const T* base, int t0, te (&r)[U]) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int t = t0 + u * G < len ? t0 + u * G : len - 1;
            r[u] = *reinterpret_cast<const te*>(base + t * kvs + c * E);
        }
    };
    auto score = [&](const te k) {
        float d = 0.0f;
#pragma unroll
        for (int e = 0; e < E; e++) d = __builtin_fmaf((float)qv[e], (float)k[e], d);
        return group_sum(d, L);
    };
    const bool known = __builtin_fabsf(M) < 1.0e30f && den > 0.0f && den < INFINITY;
    float m = -INFINITY, l = 0.0f;  // a key at -inf adds nothing, unless all are
    for (int t0 = g; !known && t0 < len; t0 += U * G) {
        te k[U];
        load(kh, t0, k);
#pragma unroll
        for (int u = 0; u < U; u++) {
            const float s = score(k[u]) * scale;
            if (t0 + u * G >= len || s == -INFINITY) continue;
            if (s > m) {
                l = l * expf(m - s) + 1.0f;
                m = s;
            } else {
                l += expf(s - m);
            }
        }
    }
    for (int off = L; off < 64; off <<= 1) {
        const float m2 = __shfl_xor(m, off), l2 = __shfl_xor(l, off), mx = fmaxf(m, m2);
        l = mx == -INFINITY ? l + l2 : l * expf(m - mx) + l2 * expf(m2 - mx);
        m = mx;
    }
    if (known) {
        m = M;
        l = den;
    } else if (!(__builtin_fabsf(m) < INFINITY)) {
        l = __builtin_nanf("");  // exp(inf - inf)
    }
    // exp2(score sl + score slo - m) / l, or exp(score scale - m) / l
    const double sd = known ? (double)scale * 1.4426950408889634 : 0.0;
    const float sl = (float)sd, slo = (float)(sd - (double)sl), rl = 1.0f / l;
    float o[E];
#pragma unroll
    for (int e = 0; e < E; e++) o[e] = l == l ? 0.0f : l;
    if (l == l) {
        for (int t0 = g; t0 < len; t0 += U * G) {
            te k[U], v[U];
            load(kh, t0, k);
            load(vh, t0, v);
#pragma unroll
            for (int u = 0; u < U; u++) {
                const float s = score(k[u]);
                if (t0 + u * G >= len) continue;
                float p;
                if (known) {
                    const float x = __builtin_fmaf(s, sl, -m);
                    p = __builtin_amdgcn_exp2f(s > -INFINITY ? __builtin_fmaf(s, slo, x) : x) * rl;
                } else {
                    p = expf(s * scale - m) / l;
                }
#pragma unroll
                for (int e = 0; e < E; e++) o[e] = __builtin_fmaf(p, (float)v[u][e], o[e]);
            }
        }
    }
    T y[E];
#pragma unroll
    for (int e = 0; e < E; e++) {
        for (int off = L; off < 64; off <<= 1) o[e] += __shfl_xor(o[e], off);
        y[e] = (T)o[e];
    }
    if (g == 0)
#pragma unroll
        for (int e = 0; e < E; e++) orow[c * E + e] = y[e];
}

// Whether a row of numerators and denominator den under the maximum M is to be
// done again by attn_row_general: some quotient is not finite, but not because a
// visible score is NaN, which makes the whole row NaN there too.
__device__ __forceinline__ bool attn_redo(const f4 y, float den, float M)
{
    bool nf = false;
#pragma unroll
    for (int j = 0; j < 4; j++) nf = nf || !(__builtin_fabsf(y[j]) <= 3.0e38f);
    return nf && !(den != den && __builtin_fabsf(M) < INFINITY);
}

}  // namespace

// ---------------------------------------------------------------------------
// fp16 q, K and V, head_dim 64 or 128.  The G = H / KVH query heads of a kv
// head read the same keys, so the rows of a kv head's problem are the pairs
// (query s, head h of the group), row r = s G + h: a tile of consecutive rows
// covers few queries, which keeps its causal edge short, and a call of a few
// queries still fills tiles.
//
// A block of 4 RG waves takes 32 RG rows; wave (rg, kg) takes rows 32 rg .. + 31
// and, of every stage of 128 keys, the 32 keys of group kg.  K and V stages go
// straight from memory to LDS, two stages deep, one barrier per stage.  Per
// stage a wave:
//   S^T = K q^T    v_mfma_f32_32x32x16_f16, A = K rows, B = the 32 query rows
//                  (kept in registers): lane l gets row l % 32's scores of 16
//                  keys, 8 (i / 4) + 4 (l / 32) + i % 4 for i < 16;
//   softmax        p = exp2(score scale log2 e - b), b the row's running
//                  maximum in log2 units less 10, moved (and O, l rescaled) only
//                  when a score exceeds that maximum by more than 5: p stays
//                  below 2^15, and the largest is 2^10 or more;
//   O^T += V^T p   A = V^T by LDS transpose reads, B = the lane's own p: the
//                  order of keys inside an MFMA is free as long as A and B
//                  share it, so p needs no shuffles.  p goes in as fp16 high
//                  and low parts (two products): about 22 bits, and steps of
//                  2^-24, fp16's smallest, 2^-34 of the largest weight.  (With
//                  weights from 2^0 to 2^8 those of 2^-25 of the largest were
//                  lost while l counted them: 4000 keys under one of 2^22 times
//                  their weight whose V is 0, 3e-2 off.  2^13 to 2^15 would
//                  keep three bits more, but moves b, and with it O, in nearly
//                  every stage: 500 queries after 3500 positions 32.2 us with
//                  2^0 or 2^7 .. 2^15, 31.4 to 33.3 here, 35.4 with 2^13.)
// The groups' (b, l, O) are merged through LDS at the end; blocks that share a
// row block's keys (gridDim.y of them) leave theirs to k_attention_prefill_merge.
//
// A stage costs about 3400 clocks with one wave per SIMD or two (8 waves): the
// chain of a wave's products, softmax and products (24 MFMAs of 32 clocks and
// about 190 vector operations at head_dim 128), not the loads (the same with
// them left out).  Measured against one block per (head, query) with the dot
// products on the vector unit (k_attention): 512 queries, 14 heads on 2 of 64,
// 78 -> 7.7 us; 2048, 12 on 2 of 128, 1740 -> 34; 500 after 3500 positions, 1840
// -> 34.  Two 32-key tiles per wave and stage (half as many stages of twice the
// length), 128 rows per block, and the next stage's scores computed during
// this one's softmax all measured the same or slower.
// ---------------------------------------------------------------------------
template <int D, int RG>
__global__ __launch_bounds__(256 * RG) void k_attention_prefill(
    const f16* __restrict__ q, const f16* __restrict__ k, const f16* __restrict__ v, int32_t n_q, int32_t len0,
    int32_t KVH, int32_t G, float scale, float scale_log2, f16* __restrict__ out, float* __restrict__ ws)
{
    constexpr int KG = 4;  // key groups
    constexpr int NW = RG * KG, NT = 64 * NW, ROWS = 32 * RG;
    constexpr int KS = 32 * KG;           // keys per stage
    constexpr int CPR = D / 8;            // 16-byte chunks per row
    constexpr int RPP = 64 / CPR;         // rows per 1 KB load
    constexpr int LP = KS / RPP / NW;     // loads of K (and of V) per wave and stage
    constexpr int DT = D / 16, DE = D / 32;
    constexpr float kTopLog2 = 10.0f;     // log2 of a row's largest weight when b moves
    static_assert(KS / RPP % NW == 0, "whole loads per wave");
    constexpr int kStage = 2 * KS * D;    // halves: K rows, then V rows
    static_assert(kStage * 2 >= NW / 2 * 32 * D * 4, "half of the waves' O in each stage");
    __shared__ __align__(1024) f16 sm0[kStage], sm1[kStage];
    __shared__ float wm[NW][32], wl[NW][32];
    __shared__ int32_t bad[ROWS];

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int rg = wave % RG, kg = wave / RG;
    const int ln = lane & 31, hb = lane >> 5, gl = lane & 15;
    const int H = G * KVH;
    const int R = n_q * G, nrb = (R + ROWS - 1) / ROWS;
    // longest rows first, so the last blocks to start are the short ones
    const int kvh = blockIdx.x % KVH, rb = nrb - 1 - (int)(blockIdx.x / KVH);
    const int r0 = rb * ROWS, wr0 = r0 + rg * 32;
    const int total = len0 + n_q - 1;
    const int blk_last = (r0 + ROWS < R ? r0 + ROWS : R) - 1;
    const int all_stages = (len0 + blk_last / G + KS - 1) / KS;
    // split z of the block's keys: stages [st0, st1)
    const int ns = (int)gridDim.y, per = (all_stages + ns - 1) / ns;
    const int st0 = (int)blockIdx.y * per, st1 = st0 + per < all_stages ? st0 + per : all_stages;
    const bool active = wr0 < R;
    const int wlast = wr0 + 31 < R ? wr0 + 31 : R - 1;
    const int row = wr0 + ln < R ? wr0 + ln : R - 1;
    const int qs = row / G;
    const int lim = len0 + qs;                                     // keys the lane's row sees
    const int wmin = active ? len0 + wr0 / G : 0, wmax = active ? len0 + wlast / G : 0;
    const int64_t kvs = (int64_t)KVH * D;
    const f16* kh = k + (int64_t)kvh * D;
    const f16* vh = v + (int64_t)kvh * D;
    const int64_t q_off = ((int64_t)qs * H + (int64_t)kvh * G + (row - qs * G)) * D;

    const uint32_t kv_bytes = (uint32_t)(((int64_t)total * kvs - (int64_t)kvh * D) * 2);
    const __amdgpu_buffer_rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc(const_cast<f16*>(kh), 0, (int)kv_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc(const_cast<f16*>(vh), 0, (int)kv_bytes, 0x00020000);
    const uint32_t stride = (uint32_t)(kvs * 2);
    // a lane's 16 bytes of a load: row r of the stage, the chunk that belongs in its slot
    auto stage = [&](auto P) -> f16* {
        if constexpr (decltype(P)::value == 0) return sm0;
        else return sm1;
    };
    auto issue = [&](auto P, int st) {
        f16* sk = stage(P);
        f16* sv = sk + KS * D;
#pragma unroll
        for (int i = 0; i < LP; i++) {
            const int p = wave * LP + i, r = p * RPP + lane / CPR;
            const int c = (lane % CPR) ^ attn_swz<D>(r);
            const int key = st * KS + r < total ? st * KS + r : total - 1;
            const uint32_t off = (uint32_t)key * stride + (uint32_t)c * 16;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rk, sk + p * 512, 16, off, 0, 0, 0);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rv, sv + p * 512, 16, off, 0, 0, 0);
        }
    };

    constexpr auto P0 = std::integral_constant<int, 0>{};
    constexpr auto P1 = std::integral_constant<int, 1>{};
    if (st0 < st1) issue(P0, st0);
    h8 qf[DT];
#pragma unroll
    for (int d = 0; d < DT; d++) qf[d] = *reinterpret_cast<const h8*>(q + q_off + 16 * d + 8 * hb);
    float b = -1e30f, l = 0.0f;
    f16v o[DE];
#pragma unroll
    for (int e = 0; e < DE; e++) o[e] = f16v{};

    auto step = [&](auto P, auto PN, int st) {
        wait_vmcnt<0>();
        lds_barrier();  // stage st in LDS for every wave; every wave is done with stage st - 1
        if (st + 1 < st1) issue(PN, st + 1);
        const int k0 = st * KS + kg * 32;  // the wave's first key of the stage
        if (k0 >= wmax) return;
        const f16* sk = stage(P) + kg * 32 * D;
        const f16* sv = sk + KS * D;
        f16v s = f16v{};
#pragma unroll
        for (int d = 0; d < DT; d++) {
            const h8 kf = *reinterpret_cast<const h8*>(sk + ln * D + (((2 * d + hb) ^ attn_swz<D>(ln)) * 8));
            s = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf, qf[d], s, 0, 0, 0);
        }
        if (k0 + 32 > wmin) {  // keys past some row's last visible one
#pragma unroll
            for (int i = 0; i < 16; i++)
                if (k0 + 8 * (i / 4) + 4 * hb + i % 4 >= lim) s[i] = -INFINITY;
        }
        float mx = s[0];
#pragma unroll
        for (int i = 1; i < 16; i++) mx = fmaxf(mx, s[i]);
        mx = max_x32(mx) * scale_log2;
        const bool up = mx > b + (kTopLog2 + 5.0f);
        if (__any(up)) {
            const float bn = fmaxf(mx - kTopLog2, b), corr = __builtin_amdgcn_exp2f(b - bn);
            b = bn;
            l *= corr;
#pragma unroll
            for (int e = 0; e < DE; e++) o[e] *= corr;
        }
#pragma unroll
        for (int u = 0; u < 2; u++) {
            h8 ph, pl;
#pragma unroll
            for (int j = 0; j < 8; j += 2) {
                float p[2];
#pragma unroll
                for (int w = 0; w < 2; w++) {
                    p[w] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[8 * u + j + w], scale_log2, -b));
                    l += p[w];
                }
                const h2 hi = __builtin_convertvector(f2{p[0], p[1]}, h2);
                // the remainders, exact, by one mixed-precision FMA each
                const h2 lo = __builtin_convertvector(
                    f2{__builtin_fmaf((float)hi[0], -1.0f, p[0]), __builtin_fmaf((float)hi[1], -1.0f, p[1])}, h2);
                ph[j] = hi[0];
                ph[j + 1] = hi[1];
                pl[j] = lo[0];
                pl[j + 1] = lo[1];
            }
            // V^T: lane (dim 32 e + ln) of keys 16 u + 8 jj + 4 hb + 0..3, jj = 0, 1,
            // one transpose read each (16 lanes: 4 keys x 16 dims)
            h8 va[DE];
#pragma unroll
            for (int e = 0; e < DE; e++) {
                h4v a[2];
#pragma unroll
                for (int jj = 0; jj < 2; jj++) {
                    const int r = 16 * u + 8 * jj + 4 * hb + (gl >> 2);
                    const int c = 4 * e + 2 * ((lane >> 4) & 1) + ((gl & 3) >> 1);
                    a[jj] = lds_read_tr16(sv + r * D + (c ^ attn_swz<D>(r)) * 8 + 4 * (gl & 1));
                }
                va[e] = h8{a[0][0], a[0][1], a[0][2], a[0][3], a[1][0], a[1][1], a[1][2], a[1][3]};
            }
            // every dim tile's high product before the low ones: no product waits on the one before it
#pragma unroll
            for (int e = 0; e < DE; e++) o[e] = __builtin_amdgcn_mfma_f32_32x32x16_f16(va[e], ph, o[e], 0, 0, 0);
#pragma unroll
            for (int e = 0; e < DE; e++) o[e] = __builtin_amdgcn_mfma_f32_32x32x16_f16(va[e], pl, o[e], 0, 0, 0);
        }
    };
    for (int st = st0; st < st1; st += 2) {
        step(P0, P1, st);
        if (st + 1 < st1) step(P1, P0, st + 1);
    }
    l = sum_x32(l);

    lds_barrier();  // every wave is done with the stages
    // wave w's O rows of D floats (half of the waves per stage), 16-byte chunk c of row r at slot c ^ r
    auto os = [&](int w, int r, int c) {
        return reinterpret_cast<f4*>((w < NW / 2 ? sm0 : sm1) + w % (NW / 2) * 64 * D) + r * (D / 4) + (c ^ (r & 15));
    };
    if (hb == 0) {
        wm[wave][ln] = b;
        wl[wave][ln] = l;
    }
    if (tid < ROWS) bad[tid] = 0;
#pragma unroll
    for (int e = 0; e < DE; e++)
#pragma unroll
        for (int g = 0; g < 4; g++)
            *os(wave, ln, 8 * e + 2 * g + hb) =
                f4{o[e][4 * g], o[e][4 * g + 1], o[e][4 * g + 2], o[e][4 * g + 3]};
    __syncthreads();
    auto row_off = [&](int r) {
        const int s_ = r / G;
        return ((int64_t)s_ * H + (int64_t)kvh * G + (r - s_ * G)) * D;
    };
    // the maximum and the sum of the weights of row rr, over its key groups
    auto row_sums = [&](int rr, float& M, float& den) {
        const int w0 = rr / 32, ri = rr & 31;  // wave of key group g: w0 + g RG
        M = wm[w0][ri];
#pragma unroll
        for (int g = 1; g < KG; g++) M = fmaxf(M, wm[w0 + g * RG][ri]);
        den = 0.0f;
#pragma unroll
        for (int g = 0; g < KG; g++) den += __builtin_amdgcn_exp2f(wm[w0 + g * RG][ri] - M) * wl[w0 + g * RG][ri];
    };
    // partials of split z of row r: D floats at row z KVH R + kvh R + r, and (m, l) after all rows
    const int64_t pr0 = ((int64_t)blockIdx.y * KVH + kvh) * R + r0;
    f4* wo = reinterpret_cast<f4*>(ws);
    float2* wml = reinterpret_cast<float2*>(ws + (int64_t)ns * KVH * R * D);
    for (int idx = tid; idx < ROWS * (D / 4); idx += NT) {
        const int rr = idx / (D / 4), c = idx % (D / 4);
        if (r0 + rr >= R) break;
        const int w0 = rr / 32, ri = rr & 31;  // wave of key group g: w0 + g RG
        float M = wm[w0][ri];
#pragma unroll
        for (int g = 1; g < KG; g++) M = fmaxf(M, wm[w0 + g * RG][ri]);
        f4 num = f4{0.0f, 0.0f, 0.0f, 0.0f};
        float den = 0.0f;
#pragma unroll
        for (int g = 0; g < KG; g++) {
            const float f = __builtin_amdgcn_exp2f(wm[w0 + g * RG][ri] - M);
            num += f * *os(w0 + g * RG, ri, c);
            den += f * wl[w0 + g * RG][ri];
        }
        if (ns == 1) {
            const f4 y = num / den;
            // the row's D / 4 lanes agree before any stores (out may be q, which a redone row reads)
            const uint64_t redo = __ballot(attn_redo(y, den, M)) >> (lane & (64 - D / 4)) & (((uint64_t)1 << (D / 4)) - 1);
            if (redo) bad[rr] = 1;
            else *reinterpret_cast<h4v*>(out + row_off(r0 + rr) + 4 * c) = __builtin_convertvector(y, h4v);
        } else {
            wo[(pr0 + rr) * (D / 4) + c] = num;
            if (c == 0) wml[pr0 + rr] = make_float2(M, den);
        }
    }
    if (ns > 1) return;  // k_attention_prefill_merge finishes the rows
    __syncthreads();
    // rows to be done again, a wave each: none, with finite inputs
    int turn = 0;
    for (uint64_t rows = __ballot(lane < ROWS && bad[lane % ROWS]); rows; rows &= rows - 1) {
        if (turn++ % NW != wave) continue;
        const int rr = __builtin_ctzll(rows);
        const int64_t off = row_off(r0 + rr);
        float M, den;
        row_sums(rr, M, den);
        attn_row_general<f16, D>(q + off, kh, vh, kvs, len0 + (r0 + rr) / G, scale, M, den, out + off, lane);
    }
}

// ---------------------------------------------------------------------------
// fp32 q, K and V, head_dim 64 or 128, on v_mfma_f32_32x32x2_f32: the same
// rows, tiles, softmax and merge, with exact fp32 products and sums throughout
// (no operand is split or rounded).  A stage holds 8192 / D keys (64 KB of K
// and V); KG waves share them, RG row groups, 4 waves in all, one block per CU.
// The assignment of dims (K q^T) and keys (V^T p) to an MFMA's two k slots is
// free as long as both operands share it:
//   K q^T   slot hb = lane / 32 takes dims hb D / 2 + j, so a 16-byte read of a
//           K row feeds 4 MFMAs, and a lane keeps D / 2 dims of its query row;
//   V^T p   slot hb takes the lane's own keys 8 (i / 4) + 4 hb + i % 4; row r of
//           dim tile e is dim DE r + e, so a read of DE consecutive values of a V
//           row feeds the DE tiles.
// The exponent adds the low half of scale log2 e (scale_lo), which fp32 rounds
// off, and the running maximum follows every new one, so that the largest
// weights have the smallest exponents to round.  A score is summed in two chains
// of D / 2 products and a stage's weights four at a time, which one block per head
// and query did in one of D and in a butterfly (error against 64 bits, that form /
// one chain each here / now: 333 queries, 14 heads of 64, 4.28e-7 / 4.35e-7 / 2.86e-7,
// 14.4 -> 14.8 us; 1000, 12 of 128, 7.6e-7 / 7.6e-7 / 4.7e-7, 84 -> 86 us).
// Bound by the fp32 matrix rate (64 clocks per MFMA, D / 2 + 16 DE of them per
// 32 x 32 scores).
// ---------------------------------------------------------------------------
template <int D, int RG, int KG>
__global__ __launch_bounds__(256) void k_attention_prefill_f32(
    const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v, int32_t n_q, int32_t len0,
    int32_t KVH, int32_t G, float scale, float scale_log2, float scale_lo, float* __restrict__ out,
    float* __restrict__ ws)
{
    static_assert(RG * KG == 4, "4 waves");
    constexpr int ROWS = 32 * RG;
    constexpr int KS = 32 * KG;           // keys per stage
    constexpr int CPR = D / 4;            // 16-byte chunks per row
    constexpr int RPP = 64 / CPR;         // rows per 1 KB load
    constexpr int LP = KS / RPP / 4;      // loads of K (and of V) per wave and stage
    constexpr int DE = D / 32;
    constexpr int kStage = 2 * KS * D;    // floats: K rows, then V rows
    static_assert(kStage >= 2 * 32 * D, "two waves' O in each stage");
    typedef float fe __attribute__((ext_vector_type(DE)));
    __shared__ __align__(1024) float sm0[kStage], sm1[kStage];
    __shared__ float wm[4][32], wl[4][32];
    __shared__ int32_t bad[ROWS];

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int rg = wave % RG, kg = wave / RG;
    const int ln = lane & 31, hb = lane >> 5;
    const int H = G * KVH;
    const int R = n_q * G, nrb = (R + ROWS - 1) / ROWS;
    const int kvh = blockIdx.x % KVH, rb = nrb - 1 - (int)(blockIdx.x / KVH);  // longest rows first
    const int r0 = rb * ROWS, wr0 = r0 + rg * 32;
    const int total = len0 + n_q - 1;
    const int blk_last = (r0 + ROWS < R ? r0 + ROWS : R) - 1;
    const int all_stages = (len0 + blk_last / G + KS - 1) / KS;
    const int ns = (int)gridDim.y, per = (all_stages + ns - 1) / ns;
    const int st0 = (int)blockIdx.y * per, st1 = st0 + per < all_stages ? st0 + per : all_stages;
    const bool active = wr0 < R;
    const int wlast = wr0 + 31 < R ? wr0 + 31 : R - 1;
    const int row = wr0 + ln < R ? wr0 + ln : R - 1;
    const int qs = row / G;
    const int lim = len0 + qs;
    const int wmin = active ? len0 + wr0 / G : 0, wmax = active ? len0 + wlast / G : 0;
    const int64_t kvs = (int64_t)KVH * D;
    const float* kh = k + (int64_t)kvh * D;
    const float* vh = v + (int64_t)kvh * D;
    const int64_t q_off = ((int64_t)qs * H + (int64_t)kvh * G + (row - qs * G)) * D;

    const uint32_t kv_bytes = (uint32_t)(((int64_t)total * kvs - (int64_t)kvh * D) * 4);
    const __amdgpu_buffer_rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(kh), 0, (int)kv_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(vh), 0, (int)kv_bytes, 0x00020000);
    const uint32_t stride = (uint32_t)(kvs * 4);
    auto stage = [&](auto P) -> float* {
        if constexpr (decltype(P)::value == 0) return sm0;
        else return sm1;
    };
    // LDS slot of chunk c of row r: c ^ (r % 16) (16 rows of one chunk in 16 bank groups)
    auto issue = [&](auto P, int st) {
        float* sk = stage(P);
        float* sv = sk + KS * D;
#pragma unroll
        for (int i = 0; i < LP; i++) {
            const int p = wave * LP + i, r = p * RPP + lane / CPR;
            const int c = (lane % CPR) ^ (r & 15);
            const int key = st * KS + r < total ? st * KS + r : total - 1;
            const uint32_t off = (uint32_t)key * stride + (uint32_t)c * 16;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rk, sk + p * 256, 16, off, 0, 0, 0);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rv, sv + p * 256, 16, off, 0, 0, 0);
        }
    };

    constexpr auto P0 = std::integral_constant<int, 0>{};
    constexpr auto P1 = std::integral_constant<int, 1>{};
    if (st0 < st1) issue(P0, st0);
    f4 qf[D / 8];
#pragma unroll
    for (int j = 0; j < D / 8; j++) qf[j] = *reinterpret_cast<const f4*>(q + q_off + hb * (D / 2) + 4 * j);
    float m = -1e30f, l = 0.0f;
    f16v o[DE];
#pragma unroll
    for (int e = 0; e < DE; e++) o[e] = f16v{};

    auto step = [&](auto P, auto PN, int st) {
        wait_vmcnt<0>();
        lds_barrier();  // stage st in LDS for every wave; every wave is done with stage st - 1
        if (st + 1 < st1) issue(PN, st + 1);
        const int k0 = st * KS + kg * 32;
        if (k0 >= wmax) return;
        const float* sk = stage(P) + kg * 32 * D;
        const float* sv = sk + KS * D;
        f16v s2[2] = {f16v{}, f16v{}};
#pragma unroll
        for (int j = 0; j < D / 8; j++) {
            const f4 kf = *reinterpret_cast<const f4*>(sk + ln * D + (((hb * (CPR / 2) + j) ^ (ln & 15)) * 4));
#pragma unroll
            for (int w = 0; w < 4; w++) s2[w & 1] = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[w], qf[j][w], s2[w & 1], 0, 0, 0);
        }
        f16v s = s2[0] + s2[1];
        if (k0 + 32 > wmin) {  // keys past some row's last visible one
#pragma unroll
            for (int i = 0; i < 16; i++)
                if (k0 + 8 * (i / 4) + 4 * hb + i % 4 >= lim) s[i] = -INFINITY;
        }
        float mx = s[0];
#pragma unroll
        for (int i = 1; i < 16; i++) mx = fmaxf(mx, s[i]);
        mx = max_x32(mx) * scale_log2;
        const bool up = mx > m;
        if (__any(up)) {
            const float mn = up ? mx : m, corr = __builtin_amdgcn_exp2f(m - mn);
            m = mn;
            l *= corr;
#pragma unroll
            for (int e = 0; e < DE; e++) o[e] *= corr;
        }
        float lp[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int i = 0; i < 16; i++) {
            // a masked score is -inf; its low part would make it NaN (-inf + inf) when scale_lo < 0
            const float x = __builtin_fmaf(s[i], scale_log2, -m);
            const float p = __builtin_amdgcn_exp2f(s[i] > -INFINITY ? __builtin_fmaf(s[i], scale_lo, x) : x);
            lp[i % 4] += p;
            const int r = 8 * (i / 4) + 4 * hb + i % 4;
            // dims DE ln .. + DE - 1 of V row r
            const fe vf = *reinterpret_cast<const fe*>(sv + r * D + ((ln * DE / 4) ^ (r & 15)) * 4 + (ln * DE) % 4);
#pragma unroll
            for (int e = 0; e < DE; e++) o[e] = __builtin_amdgcn_mfma_f32_32x32x2f32(vf[e], p, o[e], 0, 0, 0);
        }
        l += (lp[0] + lp[1]) + (lp[2] + lp[3]);
    };
    for (int st = st0; st < st1; st += 2) {
        step(P0, P1, st);
        if (st + 1 < st1) step(P1, P0, st + 1);
    }
    l = sum_x32(l);

    lds_barrier();  // every wave is done with the stages
    // wave w's O rows of D floats, two waves per stage, 16-byte chunk c of row r at slot c ^ (r % 16)
    auto os = [&](int w, int r, int c) {
        return reinterpret_cast<f4*>((w < 2 ? sm0 : sm1) + (w & 1) * 32 * D) + r * (D / 4) + (c ^ (r & 15));
    };
    if (hb == 0) {
        wm[wave][ln] = m;
        wl[wave][ln] = l;
    }
    if (tid < ROWS) bad[tid] = 0;
#pragma unroll
    for (int i = 0; i < 16; i += 4 / DE) {
        // DE consecutive dims per accumulator index: 4 / DE indices make a chunk
        const int d = DE * (8 * (i / 4) + 4 * hb + i % 4);
        f4 w;
#pragma unroll
        for (int j = 0; j < 4 / DE; j++)
#pragma unroll
            for (int e = 0; e < DE; e++) w[DE * j + e] = o[e][i + j];
        *os(wave, ln, d / 4) = w;
    }
    __syncthreads();
    auto row_off = [&](int r) {
        const int s_ = r / G;
        return ((int64_t)s_ * H + (int64_t)kvh * G + (r - s_ * G)) * D;
    };
    // the maximum and the sum of the weights of row rr, over its key groups
    auto row_sums = [&](int rr, float& M, float& den) {
        const int w0 = rr / 32, ri = rr & 31;  // wave of key group g: w0 + g RG
        M = wm[w0][ri];
#pragma unroll
        for (int g = 1; g < KG; g++) M = fmaxf(M, wm[w0 + g * RG][ri]);
        den = 0.0f;
#pragma unroll
        for (int g = 0; g < KG; g++) den += __builtin_amdgcn_exp2f(wm[w0 + g * RG][ri] - M) * wl[w0 + g * RG][ri];
    };
    const int64_t pr0 = ((int64_t)blockIdx.y * KVH + kvh) * R + r0;
    f4* wo = reinterpret_cast<f4*>(ws);
    float2* wml = reinterpret_cast<float2*>(ws + (int64_t)ns * KVH * R * D);
    for (int idx = tid; idx < ROWS * (D / 4); idx += 256) {
        const int rr = idx / (D / 4), c = idx % (D / 4);
        if (r0 + rr >= R) break;
        const int w0 = rr / 32, ri = rr & 31;
        float M = wm[w0][ri];
#pragma unroll
        for (int g = 1; g < KG; g++) M = fmaxf(M, wm[w0 + g * RG][ri]);
        f4 num = f4{0.0f, 0.0f, 0.0f, 0.0f};
        float den = 0.0f;
#pragma unroll
        for (int g = 0; g < KG; g++) {
            const float f = __builtin_amdgcn_exp2f(wm[w0 + g * RG][ri] - M);
            num += f * *os(w0 + g * RG, ri, c);
            den += f * wl[w0 + g * RG][ri];
        }
        if (ns == 1) {
            const f4 y = num / den;
            // the row's D / 4 lanes agree before any stores (out may be q, which a redone row reads)
            const uint64_t redo = __ballot(attn_redo(y, den, M)) >> (lane & (64 - D / 4)) & (((uint64_t)1 << (D / 4)) - 1);
            if (redo) bad[rr] = 1;
            else *reinterpret_cast<f4*>(out + row_off(r0 + rr) + 4 * c) = y;
        } else {
            wo[(pr0 + rr) * (D / 4) + c] = num;
            if (c == 0) wml[pr0 + rr] = make_float2(M, den);
        }
    }
    if (ns > 1) return;  // k_attention_prefill_merge finishes the rows
    __syncthreads();
    // rows to be done again, a wave each: none, with finite inputs
    int turn = 0;
    for (uint64_t rows = __ballot(lane < ROWS && bad[lane % ROWS]); rows; rows &= rows - 1) {
        if (turn++ % 4 != wave) continue;
        const int rr = __builtin_ctzll(rows);
        const int64_t off = row_off(r0 + rr);
        float M, den;
        row_sums(rr, M, den);
        attn_row_general<float, D>(q + off, kh, vh, kvs, len0 + (r0 + rr) / G, scale, M, den, out + off, lane);
    }
}

// The rows of a call whose keys were split over ns blocks: a wave per row sums
// the splits' numerators and denominators under their common maximum, in order.
template <typename T, int D>
__global__ __launch_bounds__(256) void k_attention_prefill_merge(const T* __restrict__ q, const T* __restrict__ k,
                                                                 const T* __restrict__ v, int32_t n_q, int32_t len0,
                                                                 int32_t KVH, int32_t G, float scale, int32_t ns,
                                                                 T* __restrict__ out, const float* __restrict__ ws)
{
    constexpr int E = D / 64;
    const int lane = threadIdx.x & 63, R = n_q * G;
    const int row = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * 4 + (threadIdx.x >> 6)));
    if (row >= R * KVH) return;
    const int kvh = row / R, r = row - kvh * R, s = r / G;
    const int64_t rows = (int64_t)KVH * R;
    const float2* wml = reinterpret_cast<const float2*>(ws + rows * ns * D);
    float M = -1e30f, den = 0.0f;
    float num[E] = {};
    for (int z = 0; z < ns; z++) M = fmaxf(M, wml[z * rows + row].x);
#pragma unroll 4
    for (int z = 0; z < ns; z++) {
        const float2 ml = wml[z * rows + row];
        const float* o = ws + (z * rows + row) * D + lane * E;
        const float f = __builtin_amdgcn_exp2f(ml.x - M);
#pragma unroll
        for (int e = 0; e < E; e++) num[e] += f * o[e];
        den += f * ml.y;
    }
    const int64_t off = ((int64_t)s * G * KVH + (int64_t)kvh * G + (r - s * G)) * D;
    f4 y = f4{};
#pragma unroll
    for (int e = 0; e < E; e++) y[e] = num[e] / den;
    if (__any(attn_redo(y, den, M))) {  // not with finite inputs
        attn_row_general<T, D>(q + off, k + (int64_t)kvh * D, v + (int64_t)kvh * D, (int64_t)KVH * D, len0 + s, scale,
                               M, den, out + off, lane);
        return;
    }
#pragma unroll
    for (int e = 0; e < E; e++) out[off + lane * E + e] = (T)y[e];
}

// The tile kernels' calls: head_dim 64 or 128, 16-byte aligned q, K and V and
// 16-byte (fp16: 8-byte) aligned out (their loads and stores), byte offsets
// within one kv head's K and V rows and row numbers in 31 bits, and a positive
// scale (they take the maximum before scaling).
// fp32 calls over fewer than 128 positions keep k_attention while its blocks,
// one per head and query, fit the chip at once: a single stage here costs more
// (graph replay: 38 queries, 12 heads of 128, 7.2 us against 13.6; 15, 24 of 64, 4.9
// against 8.2; 7 queries after 360 positions, 14 of 64, 15.3 against 13.3).  So do
// those a little past the first stage with fewer blocks (32 queries after 100, 14 of
// 64, 8.8 against 10.6, 12 of 128, 13.7 against 14.7; 8 after 150 / 250, 14 of 64, 8.7 / 12.4
// against 10.7 / 13.4; 24 after 150 / 250, 32 heads, 11.6 / 17.1 against 10.8 / 13.7; 64 after
// 150 / 200, 12 of 128, 22.6 / 28.9 against 26.8 / 31.7, 48 after 300 34.7 against 36.5), and
// fp16 calls of a few queries over up to 40 positions at head_dim 128 (8 after 20, 12
// heads, 6.3 against 7.4; 24 after 20 7.2 against 7.2).
bool attention_prefill_ok(const void* out, const void* q, const void* k, const void* v, int64_t n_q, int64_t len0,
                          int64_t H, int64_t KVH, int64_t D, float scale, int dtype)
{
    const int64_t es = dtype == VVH_F16 ? 2 : 4;
    const int64_t span = len0 + n_q - 1, rows = n_q * H;
    if (dtype == VVH_F32 && ((span < 128 && rows <= 2048) || (span <= 152 && rows <= 512) ||
                             (D == 64 && span <= 270 && rows <= 256) ||
                             (D == 128 && span <= 270 && rows > 512 && rows <= 800)))
        return false;
    if (dtype == VVH_F16 && D == 128 && span <= 40 && rows <= 256) return false;
    return (D == 64 || D == 128) && scale > 0.0f && scale < INFINITY &&
           ((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k) | reinterpret_cast<uintptr_t>(v)) & 15) == 0 &&
           (reinterpret_cast<uintptr_t>(out) & (uintptr_t)(4 * es - 1)) == 0 && n_q * (H / KVH) <= (1 << 30) &&
           (len0 + n_q) * KVH * D * es < ((int64_t)1 << 31);
}

// Rows per block (32: 4 waves, one 32-key group each; 64: 8 waves) and blocks
// sharing a row block's keys, the least of a model of the call fitted to forced
// choices (graph replay): a stage of 128 keys costs a block about 1.4 us at
// head_dim 128 and 1.1 at 64 with either shape, and the call's time follows its
// longest block or, with more blocks than fit the chip at once (one per CU at
// head_dim 128, two at 64), their sum; a split call adds the merge's launch and
// its partials, written and read at about 1.5 TB/s.  Measured, 32 rows / 64 rows, splits in brackets:
// 512 queries, 14 heads on 2 of 64: 7.7 / 9.2 us (2: 12.1 / 12.1); 2048, 12 on 2
// of 128: 51.4 / 33.7; 500 after 3500 positions, same heads: 46.5 / 46.7 (2:
// 53.1 / 33.8, 4: - / 40.1); 7 after 4000: 45.6 / 44.7 (8: 15.2 / 15.1); 256 from
// the start: 9.0 / 10.7; 1500, 32 on 4 of 64: 31.3 / 28.1.
AttnPrefillPlan attention_prefill_plan(int64_t n_q, int64_t len0, int64_t H, int64_t KVH, int64_t D, int dtype,
                                       int64_t cus)
{
    const bool f32 = dtype == VVH_F32;
    const int64_t R = n_q * (H / KVH), slots = D == 64 && !f32 ? 2 * cus : cus;
    const int64_t keys = f32 ? 8192 / D : 128;  // per stage
    const int64_t longest = (len0 + n_q - 1 + keys - 1) / keys;
    const double mean = (double)(len0 + n_q / 2 + keys - 1) / (double)keys;
    const double stage_us = f32 ? (D == 64 ? 2.0 : 3.9) : (D == 64 ? 1.1 : 1.42);
    AttnPrefillPlan best{};
    double best_t = INFINITY;
    for (const int64_t rows : {32, 64}) {
        if (f32 && rows != (D == 64 ? 32 : 64)) continue;  // 4 waves: 4 key groups, or 2 of each
        const int64_t blocks = (R + rows - 1) / rows * KVH;
        const int64_t smax = std::max<int64_t>(1, std::min<int64_t>({longest, slots / blocks, 32}));
        for (int64_t sp = 1; sp <= smax; sp++) {
            const double st = std::max((double)((longest + sp - 1) / sp), (double)blocks * mean / (double)slots);
            double t = (rows == 32 ? 2.0 : 3.0) + stage_us * st;
            if (sp > 1) t += 5.0 + 0.1 * (double)sp + (double)(sp * n_q * H * (D + 2) * 8) / 1.5e6;
            if (t < best_t) {
                best_t = t;
                best = AttnPrefillPlan{rows, blocks, sp};
            }
        }
    }
    return best;
}

// Whether a call that would split its keys and has no workspace for the partials
// gives each row block all its keys, or takes k_attention.  fp32 tiles of few rows
// over short spans lose (graph replay, us, k_attention / unsplit: 8 queries after 400
// positions, 12 heads of 128, 29.3 / 40.9, after 1500 98.8 / 121.6, after 2500 335 / 197, 8 on
// 8 of 128 163 / 191; 100 queries 62.5 / 46.7, after 100 25.0 / 27.5; 8, 14 of 64, after 250
// 12.4 / 13.6, after 400 16.7 / 16.8); fp16 tiles do not (4 after 1000, 12 of 128, 60.4 / 14.7).
bool attention_prefill_unsplit_pays(int64_t n_q, int64_t len0, int64_t H, int64_t KVH, int64_t D, int dtype)
{
    if (dtype != VVH_F32) return true;
    const int64_t span = len0 + n_q - 1, blocks = n_q * H;
    if (D == 64) return blocks > 512 || span > 300;
    return blocks > 512 ? blocks > 1300 || span > 200 : span > (H == KVH ? 3000 : 2048);
}

int64_t attention_prefill_ws_floats(const AttnPrefillPlan& p, int64_t n_q, int64_t H, int64_t D)
{
    return p.splits > 1 ? p.splits * n_q * H * (D + 2) : 0;
}

int launch_attention_prefill(const AttnPrefillPlan& p, void* out, const void* q, const void* k, const void* v,
                             int64_t n_q, int64_t len0, int64_t H, int64_t KVH, int64_t D, float scale, int dtype,
                             float* ws, void* stream)
{
    const double sd = (double)scale * 1.4426950408889634;
    const float sl = (float)sd;
    const dim3 grid((unsigned)p.blocks, (unsigned)p.splits), mgrid((unsigned)((n_q * H + 3) / 4));
    const int32_t nq = (int32_t)n_q, l0 = (int32_t)len0, kvh = (int32_t)KVH, g = (int32_t)(H / KVH);
    hipStream_t s = static_cast<hipStream_t>(stream);
    auto merge = [&]<typename T>(auto kern, T* o) {
        if (p.splits > 1)
            hipLaunchKernelGGL(kern, mgrid, dim3(256), 0, s, (const T*)q, (const T*)k, (const T*)v, nq, l0, kvh, g, scale,
                               (int32_t)p.splits, o, ws);
    };
    if (dtype == VVH_F32) {
        auto go = [&](auto kern) {
            hipLaunchKernelGGL(kern, grid, dim3(256), 0, s, (const float*)q, (const float*)k, (const float*)v, nq, l0, kvh,
                               g, scale, sl, (float)(sd - (double)sl), (float*)out, ws);
        };
        D == 64 ? go(k_attention_prefill_f32<64, 1, 4>) : go(k_attention_prefill_f32<128, 2, 2>);
        D == 64 ? merge(k_attention_prefill_merge<float, 64>, (float*)out)
                : merge(k_attention_prefill_merge<float, 128>, (float*)out);
        return (int)hipGetLastError();
    }
    auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, grid, dim3(unsigned(8 * p.rows)), 0, s, (const f16*)q, (const f16*)k, (const f16*)v, nq,
                           l0, kvh, g, scale, sl, (f16*)out, ws);
    };
    if (D == 64) p.rows == 32 ? go(k_attention_prefill<64, 1>) : go(k_attention_prefill<64, 2>);
    else p.rows == 32 ? go(k_attention_prefill<128, 1>) : go(k_attention_prefill<128, 2>);
    D == 64 ? merge(k_attention_prefill_merge<f16, 64>, (f16*)out) : merge(k_attention_prefill_merge<f16, 128>, (f16*)out);
    return (int)hipGetLastError();
}

}  // namespace vvh
