// Device code for the quantized engine's projections on either side of the
// attention block (gfx950, wave64): W8A8 matrix-vector products with one
// float scale per group of gs consecutive values of a row, as
// QuantizedTransformer::quantize (QuantizedTransformer.cpp:338-357) and
// ::matmul (:359-652) compute them.
//   - q8_gemv_kernel<..., kQ8InRms, false>: xb = rmsnorm(x),
//     quantized per group, then q, k, v = the stacked int8 Wq/Wk/Wv . xb
//     (QuantizedTransformer.cpp:664-678);
//   - q8_gemv_kernel<..., kQ8InF32, true>: the attention output
//     quantized per group, then x += Wo . that (the wo matmul and the residual
//     after the attention block).
//
// One workgroup per CU where the rows allow it: the fp32 input vector (and the
// rms weight) is read, normalised and quantized once per workgroup and shared
// through LDS, so that the int8 weights, which are a quarter of the fp32 bytes
// per row, are not outweighed by every workgroup re-reading 16-32 KiB of
// activations from L2.  A wave takes whole rows (or halves of them at n =
// 8192): each load instruction reads 1 KiB of one row contiguously, and every
// width that is a multiple of 1024 uses every lane.
//
// Arithmetic, matched to the reference bit for bit:
//   - group scale sx = max|v| * (1/127) (the reference's release build folds
//     its division by 127 into this product), id = 1/sx rounded to nearest
//     (0 for an all-zero group), q = round-half-away(v * id);
//   - the int8 dot product of a group is exact in int32 (v_dot4_i32_i8), and
//     a row's groups are accumulated in order with one fused multiply-add
//     each: val = fma((float)idot_g, ws_g * sx_g, val).  The group products
//     are formed in parallel and the ordered chain runs in one lane per row.
// The rmsnorm in front of the q/k/v product computes 1/sqrt(mean(x^2) +
// 1e-5) exactly rounded, where the reference uses a hardware reciprocal
// square-root estimate plus one Newton step; the two differ in the last bit
// or two, which can move a quantized value by one step.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "decode_attention.hpp"  // raw buffer access helpers
#include "gemv.hpp"

namespace leap {

struct Q8Args {
    const float *x;      // [n] input: the residual stream (with rmsnorm) or the attention output
    const float *rms_w;  // [n] rms_att weight of the layer (rmsnorm variant only)
    const int8_t *w;     // [rows][n] int8 weights (Wq, Wk, Wv stacked, or Wo)
    const float *ws;     // [rows][n / gs] group scales
    float *out0;         // rows [0, n0): q, or the residual stream x (x[r] += val)
    float *out1;         // rows [n0, n0 + n1): k
    float *out2;         // rows [n0 + n1, rows): v
    int rows, n0, n1;
    int8_t *xq_out;      // [n] the quantized input as every workgroup computed it (written by workgroup 0)
    float *xs_out;       // [n / gs] its group scales
};

// What the kernel's input vector is.
constexpr int kQ8InRms = 0;   // fp32 residual stream: rmsnorm with rms_w, then quantize
constexpr int kQ8InF32 = 1;   // fp32 vector (the attention output): quantize

// Butterfly over aligned groups of L lanes (L a power of two <= 16) with the
// DPP patterns of wave_sum; every lane of a group ends with the group's
// result.  Integer sums are exact in any order; max is order-free.
template <int L>
__device__ __forceinline__ int group_sum_i32(int v)
{
    if constexpr (L >= 2) v += __builtin_amdgcn_mov_dpp(v, 0xB1, 0xF, 0xF, true);   // quad_perm [1,0,3,2]
    if constexpr (L >= 4) v += __builtin_amdgcn_mov_dpp(v, 0x4E, 0xF, 0xF, true);   // quad_perm [2,3,0,1]
    if constexpr (L >= 8) v += __builtin_amdgcn_mov_dpp(v, 0x141, 0xF, 0xF, true);  // row_half_mirror
    if constexpr (L >= 16) v += __builtin_amdgcn_mov_dpp(v, 0x140, 0xF, 0xF, true); // row_mirror
    return v;
}

template <int CTRL>
__device__ __forceinline__ float dpp_f(float x)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), CTRL, 0xF, 0xF, true));
}

template <int L>
__device__ __forceinline__ float group_max(float v)
{
    if constexpr (L >= 2) v = fmaxf(v, dpp_f<0xB1>(v));
    if constexpr (L >= 4) v = fmaxf(v, dpp_f<0x4E>(v));
    if constexpr (L >= 8) v = fmaxf(v, dpp_f<0x141>(v));
    if constexpr (L >= 16) v = fmaxf(v, dpp_f<0x140>(v));
    return v;
}

// Group maximum over aligned groups of W lanes (W a power of two <= 64).
template <int W>
__device__ __forceinline__ float group_max_w(float v)
{
    if constexpr (W <= 16) {
        return group_max<W>(v);
    } else {
        v = group_max<16>(v);
        v = fmaxf(v, __shfl_xor(v, 16));
        if constexpr (W >= 64) v = fmaxf(v, __shfl_xor(v, 32));
        return v;
    }
}

// A workgroup of NWV waves owns rows [row0, row0 + per_wg), per_wg <= J * NWV /
// WPR: teams of WPR waves, team t taking rows row0 + t + j * NWV / WPR, j < J.
// Wave p of a team holds the row's 1 KiB pieces [p * NL / WPR, (p + 1) * NL /
// WPR) of n = NL * 1024 values, 16 a lane, so a group of gs values is L = gs/16
// adjacent lanes.  The host picks (J, NWV, WPR) from the rows per CU
// (pick_q8), so that each CU has the same number of rows and the waves of a
// workgroup nearly so; rows past the workgroup's read zeros (an offset past
// the descriptor's range) and write slots that nobody reads.
//
// Bounded by the CU's intake: its rows, plus 16-32 KiB of input ahead of
// them, then the serial tail (dot products, one barrier, the ordered chain of
// n / gs fused multiply-adds).  Before, teams of four waves took a row and
// every launch ran 1024 threads; widths that are not 256 times a power of two
// idled 64-96 of a team's 256 threads, and the rows per team came in steps
// that left 1.2-1.5 rounds of workgroups at Llama-2's widths.  us per launch,
// back to back over 1 GiB of weights, before -> now: Llama-3-8B q/k/v (6144 x
// 4096) 7.29 -> 6.33, wo 5.44 -> 5.05 (of the sub-block's 21.2 the bare streams
// of its three grids take 16.2); Llama-2-13B q/k/v (15360 x 5120) 24.4 -> 16.2,
// wo 9.3 -> 6.8; Llama-2-7B q/k/v (12288 x 4096) 14.3 -> 10.7; Llama-3-70B
// q/k/v (10240 x 8192) 18.8 -> 17.2, wo 14.2 -> 14.1; TinyLlama q/k/v (2560 x
// 2048) 4.14 -> 2.95, wo 3.47 -> 2.96; Llama-3.2-3B q/k/v (5120 x 3072) 5.51 ->
// 5.11, wo 4.40 -> 3.88.
//
// Issue order: the input first, then the rows' scales and the weight rows
// (96 KiB a workgroup for Wq/Wk/Wv at Llama-3-8B), all before anything waits.
// J is a compile-time count so that every load is unconditional: load waits
// count outstanding loads in issue order, and with a runtime row count the
// wait for the input had to assume the longest queue, which made the
// normalisation wait for every weight row (0.8 us at Llama-3-8B).  The input
// work runs while the weights stream.
//
// Arguments: the input and weight pointers and the row counts come first as
// scalars, which the dispatch preloads into scalar registers (the library is
// built with -mllvm -amdgpu-kernarg-preload-count=14), so that the first
// loads do not wait for a load of the arguments; the rest of Q8Args (the
// outputs) is read after the weight rows are issued (late_args).
constexpr unsigned kQ8ArgsOffset = 4 * sizeof(void *) + 8;  // Q8Args after the preloaded x, rms_w, w, ws, rows, per_wg
static_assert(alignof(Q8Args) == 8, "argument layout");
#define LEAP_Q8_PRELOAD_PARAMS                                                                                  \
    const float *pre_x, const float *pre_rms_w, const int8_t *pre_w, const float *pre_ws, int pre_rows, int pre_per_wg

// Float4 pairs (8 registers each) of the ordered chain that are read ahead, of
// n4: all of them while they fit beside the rest, else the most that divide n4.
// More than these spill: with 16 waves (128 registers) Llama-3-70B q/k/v 17.2
// -> 20.6 us; at group size 32 with 8 waves (256) or 12 (168) all 32 or 24 took
// 20-116 bytes of scratch (sub-block of 3072 with 24 KV heads 17.1 us, now 16.5;
// of Llama-3-8B 17.6 either way).
__host__ __device__ constexpr int q8_chain_unroll(int n4, int waves)
{
    const int most = waves >= 16 ? 8 : waves >= 12 ? 20 : 24;
    int u = n4 < most ? n4 : most;
    while (n4 % u) u--;
    return u;
}

// What a kernel instance of (NL, L, J, NWV, WPR) is made of.
template <int NL, int L, int J, int NWV, int WPR>
struct Q8Shape {
    static constexpr int n = NL * 1024;
    static constexpr int NG = NL * 64 / L;       // groups per row
    static constexpr int THREADS = NWV * 64;
    static constexpr int TEAMS = NWV / WPR;
    static constexpr int SLOTS = TEAMS * J;      // rows per workgroup at most
    static constexpr int NLW = NL / WPR;         // loads per wave and row
    static constexpr int NGW = NLW * 64 / L;     // a wave's groups of a row
    static constexpr int SK = (NGW + 63) / 64;   // scale loads per wave and row
    static constexpr int IV = (n / 4 + THREADS - 1) / THREADS;  // input float4s per thread
    static_assert(NWV % WPR == 0 && NL % WPR == 0 && NG % 4 == 0 && L <= 16, "wave layout");
};

// Issue the loads of this wave's scales and weight rows.
template <class S, int J, int WPR>
__device__ __forceinline__ void q8_issue_rows(const int8_t *w, const float *ws, int rows, int row0, int row_end, int wave,
                                              int lane, float (&sc)[J][S::SK], u32x4 (&wv)[J][S::NLW])
{
    const int team = wave / WPR, piece = wave % WPR;
    const uint32_t w_bytes = (uint32_t)rows * (uint32_t)S::n, s_bytes = (uint32_t)rows * (S::NG * 4u);
    const __amdgpu_buffer_rsrc_t w_rsrc = make_rsrc(w, w_bytes);
    const __amdgpu_buffer_rsrc_t s_rsrc = make_rsrc(ws, s_bytes);
#pragma unroll
    for (int j = 0; j < J; j++) {
        const int r = row0 + team + j * S::TEAMS;
#pragma unroll
        for (int k = 0; k < S::SK; k++) {
            const int g = lane + 64 * k;  // of the wave's groups
            const bool in = r < row_end && g < S::NGW;
            const uint32_t off = (uint32_t)r * (S::NG * 4u) + 4u * (uint32_t)(piece * S::NGW + g);
            sc[j][k] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(s_rsrc, (int)(in ? off : s_bytes), 0, kNt));
        }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < J; j++) {
        const int r = row0 + team + j * S::TEAMS;
        const uint32_t off = r < row_end ? (uint32_t)r * (uint32_t)S::n : w_bytes;
#pragma unroll
        for (int c = 0; c < S::NLW; c++)
            wv[j][c] = __builtin_amdgcn_raw_buffer_load_b128(
                w_rsrc, (int)(off + 16u * (uint32_t)lane + 1024u * (uint32_t)(piece * S::NLW + c)), 0, kNt);
    }
    __builtin_amdgcn_sched_barrier(0);
}

template <int NL, int L, int J, int NWV, int WPR, int kIn, bool kResid>
__global__ __launch_bounds__(NWV * 64) void q8_gemv_kernel(LEAP_Q8_PRELOAD_PARAMS, Q8Args args)
{
    using S = Q8Shape<NL, L, J, NWV, WPR>;
    constexpr int n = S::n, NG = S::NG, IV = S::IV, THREADS = S::THREADS;
    constexpr int W = 4 * L;  // threads per group in the quantize step
    __shared__ __align__(16) int8_t lds_xq[n];
    __shared__ float lds_xs[NG];
    // (float)idot and ws * sx of (row slot, group), [slot][group] with the
    // rows padded so that the chain lanes' 128-bit reads spread over the banks
    constexpr int NGP = NG + 4;
    __shared__ __align__(16) float lds_f[S::SLOTS * NGP];
    __shared__ __align__(16) float lds_c[S::SLOTS * NGP];
    __shared__ float ss_part[NWV];
    static_assert(2 * S::SLOTS * NGP * 4 + n + NG * 4 + NWV * 4 <= 64 * 1024, "LDS budget");
    const int tid = threadIdx.x, lane = tid % 64;
    const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
    const int row0 = blockIdx.x * pre_per_wg;
    const int row_end = min(row0 + pre_per_wg, pre_rows);

    // 1. the input (and rms weights): float4s tid, tid + THREADS, ... (past n,
    // zeros); then the rows
    const __amdgpu_buffer_rsrc_t x_rsrc = make_rsrc(pre_x, n * 4u);
    const __amdgpu_buffer_rsrc_t g_rsrc = make_rsrc(pre_rms_w, n * 4u);
    float4 v[IV], gw[IV];
#pragma unroll
    for (int i = 0; i < IV; i++) v[i] = buf_load4(x_rsrc, 16u * (uint32_t)(tid + i * THREADS));
    if constexpr (kIn == kQ8InRms) {
#pragma unroll
        for (int i = 0; i < IV; i++) gw[i] = buf_load4(g_rsrc, 16u * (uint32_t)(tid + i * THREADS));
    }
    __builtin_amdgcn_sched_barrier(0);
    float sc[J][S::SK];
    u32x4 wv[J][S::NLW];
    q8_issue_rows<S, J, WPR>(pre_w, pre_ws, pre_rows, row0, row_end, wave, lane, sc, wv);

    // 2. the input normalised (if asked) and quantized into LDS: group max
    // over W lanes, scale, round half away from zero
    if constexpr (kIn == kQ8InRms) {
        float ss = 0.f;
#pragma unroll
        for (int i = 0; i < IV; i++) ss += dot4f(v[i], v[i]);
        ss = wave_sum(ss);
        if (lane == 0) ss_part[wave] = ss;
        __syncthreads();
        ss = 0.f;
#pragma unroll
        for (int w = 0; w < NWV; w++) ss += ss_part[w];
        const float scale = 1.0f / sqrtf(ss / (float)n + 1e-5f);
#pragma unroll
        for (int i = 0; i < IV; i++)
            v[i] = make_float4(gw[i].x * (scale * v[i].x), gw[i].y * (scale * v[i].y), gw[i].z * (scale * v[i].z),
                               gw[i].w * (scale * v[i].w));
    }
#pragma unroll
    for (int i = 0; i < IV; i++) {
        float m = fmaxf(fmaxf(fabsf(v[i].x), fabsf(v[i].y)), fmaxf(fabsf(v[i].z), fabsf(v[i].w)));
        m = group_max_w<W>(fmaxf(m, 0.f));  // (a group of NaNs: 0)
        const float sx = m * (1.0f / 127.0f);
        const float id = sx != 0.0f ? __frcp_rn(sx) : 0.0f;
        auto q8 = [&](float t) { return (int)(int8_t)(int)roundf(t * id) & 0xFF; };
        const int at = tid + i * THREADS;
        if (n / 4 % THREADS == 0 || at < n / 4) {
            reinterpret_cast<int *>(lds_xq)[at] = q8(v[i].x) | (q8(v[i].y) << 8) | (q8(v[i].z) << 16) | (q8(v[i].w) << 24);
            if (at % W == 0) lds_xs[at / W] = sx;
        }
    }
    __syncthreads();
    // The outputs, from here on: the barriers above wait for every scalar
    // load in flight, and these are needed only at the end.
    const Q8Args a = late_args(args, kQ8ArgsOffset);
    if (blockIdx.x == 0 && a.xq_out) {  // the quantized input, for stage checks
        for (int i = tid; i < n / 4; i += THREADS)
            reinterpret_cast<int *>(a.xq_out)[i] = reinterpret_cast<const int *>(lds_xq)[i];
        for (int i = tid; i < NG; i += THREADS) a.xs_out[i] = lds_xs[i];
    }

    // 3. exact group dot products, one (float, scale product) pair per group
    const int team = wave / WPR, piece = wave % WPR;
#pragma unroll
    for (int k = 0; k < S::SK; k++) {
        const int g = lane + 64 * k;
        if (g < S::NGW) {
            const float xs = lds_xs[piece * S::NGW + g];
#pragma unroll
            for (int j = 0; j < J; j++) lds_c[(team + j * S::TEAMS) * NGP + piece * S::NGW + g] = sc[j][k] * xs;
        }
    }
#pragma unroll
    for (int c = 0; c < S::NLW; c++) {
        const int at = piece * S::NLW + c;
        const u32x4 xq = *reinterpret_cast<const u32x4 *>(lds_xq + 1024 * at + 16 * lane);
#pragma unroll
        for (int j = 0; j < J; j++) {
            int d = __builtin_amdgcn_sdot4((int)xq.x, (int)wv[j][c].x, 0, false);
            d = __builtin_amdgcn_sdot4((int)xq.y, (int)wv[j][c].y, d, false);
            d = __builtin_amdgcn_sdot4((int)xq.z, (int)wv[j][c].z, d, false);
            d = __builtin_amdgcn_sdot4((int)xq.w, (int)wv[j][c].w, d, false);
            d = group_sum_i32<L>(d);
            if (lane % L == 0) lds_f[(team + j * S::TEAMS) * NGP + at * (64 / L) + lane / L] = (float)d;
        }
    }
    __syncthreads();

    // 4. the ordered accumulation, one lane per row
    if (tid < row_end - row0) {
        float val = 0.f;
        const float4 *f4 = reinterpret_cast<const float4 *>(lds_f + tid * NGP);
        const float4 *c4 = reinterpret_cast<const float4 *>(lds_c + tid * NGP);
        // every LDS read ahead of the chain (0.05-0.3 us per launch against 4
        // groups ahead) as far as the registers of a wave hold them
        constexpr int kChainUnroll = q8_chain_unroll(NG / 4, NWV);
#pragma unroll kChainUnroll
        for (int j = 0; j < NG / 4; j++) {
            const float4 f = f4[j], c = c4[j];
            val = __builtin_fmaf(f.x, c.x, val);
            val = __builtin_fmaf(f.y, c.y, val);
            val = __builtin_fmaf(f.z, c.z, val);
            val = __builtin_fmaf(f.w, c.w, val);
        }
        const int r = row0 + tid;
        if constexpr (kResid) {
            a.out0[r] += val;
        } else {
            if (r < a.n0)
                a.out0[r] = val;
            else if (r < a.n0 + a.n1)
                a.out1[r - a.n0] = val;
            else
                a.out2[r - a.n0 - a.n1] = val;
        }
    }
}

// The int8 weights alone (measurement only): the grid, block size, scale
// loads and row loads of q8_gemv_kernel<NL, L, J, NWV, WPR, ...> over w
// [rows][n] and its scales ws [rows][n / gs], summed and kept only behind a
// test that real data never meets.  The launch plus the bare weight stream of
// one int8 projection.
template <int NL, int L, int J, int NWV, int WPR>
__global__ __launch_bounds__(NWV * 64) void q8_floor_kernel(LEAP_Q8_PRELOAD_PARAMS, Q8Args a)
{
    using S = Q8Shape<NL, L, J, NWV, WPR>;
    (void)pre_x;
    (void)pre_rms_w;
    const int tid = threadIdx.x;
    const int row0 = blockIdx.x * pre_per_wg;
    float sc[J][S::SK];
    u32x4 wv[J][S::NLW];
    q8_issue_rows<S, J, WPR>(pre_w, pre_ws, pre_rows, row0, min(row0 + pre_per_wg, pre_rows),
                             __builtin_amdgcn_readfirstlane(tid / 64), tid % 64, sc, wv);
    unsigned acc = 0;
    float s = 0.f;
#pragma unroll
    for (int j = 0; j < J; j++) {
#pragma unroll
        for (int c = 0; c < S::NLW; c++) acc ^= (wv[j][c].x ^ wv[j][c].y) ^ (wv[j][c].z ^ wv[j][c].w);
#pragma unroll
        for (int k = 0; k < S::SK; k++) s += sc[j][k];
    }
    if (acc == 0x7EADBEEFu && __builtin_bit_cast(unsigned, s) == 0x7FC0DEADu) a.out0[tid] = s;
}

}  // namespace leap
