// Dense projections on gfx950: the attention's qkv and o projections in their default form, int8 weights with a
// per-row scale (replaces quantize_rows_i8_k, gemv_i8 and gemm_i8_k / gemm(), kernels.cuh:98-156,250-337), and the
// reference's other matrix forms, int4 / int6 with a scale per 64 inputs and fp16 (quantize_rows_q4_k / _q6_k,
// gemv_q4_k / gemv_q6_k / gemv_f16_k, gemm_wmma_k, gemm_i8_k<true>: kernels.cuh:68-93,225-337,486-590).
//
//   quantize_rows_kernel   fp16 [O][I] -> int8 [O][I] + scale absmax/127 per row (bit-exact: IEEE divide, rint).
//   gemv1_kernel<NT, R>    y[t][o] = s[o] * sum_i q[o][i] x[t][i] for NT <= 8 rows of x, fp32 sums. HBM-bound on the
//                          weights, which are read once for all NT rows. A wavefront takes R weight rows over 1/KS of
//                          I, a lane 16 weights of each (32 where I is 16384), sums them in order and over
//                          the wavefront, and the KS parts of a row are added in LDS. KS and the sum order depend on
//                          O and I only, so any row of a multi-row call is bit-identical to the same row alone.
//   gemv_kernel<NT>        The same for longer parts, which a lane walks in steps.
//   gemm_tile_kernel       S > 8 rows (prefill): Y = X . W^T * s on v_mfma_f32_16x16x32_f16. Weights are widened to
//                          fp16 exactly (integers), activations rounded to fp16 as the reference does
//                          (kernels.cuh:306-307), fp32 accumulation, the row scale applied last. One workgroup per
//                          tile, 16 x 16 to 288 x 256 outputs, chosen so that the call's tiles fill the chip.
//   quantize_gs64_kernel   fp16 rows -> int4 / int6 codes + a scale per 64-input group (bit-exact).
//   gemv_mat_kernel        the GEMV of the int4 / int6 / fp16 forms: a lane per 16-weight unit of R rows, each unit
//                          summed in order and scaled, wavefront and part sums as gemv_kernel.
//   gemv_mat_x_kernel      the same without a loop where a part of a row is one load a lane, with the input rows in LDS.
//   gemm_tile_kernel<form> the same GEMM for every form: the staging widens int4 / int6 weights times their group
//                          scale to fp16 (or copies fp16 weights) where int8 is widened exactly.
#include <algorithm>
#include <cstdlib>
#include "common.hpp"

namespace moex {

namespace {

// sum over the wavefront, every lane receives it: the 32- and 16-lane swaps (v_permlane32/16_swap), then DPP within each
// 16-lane row (rotate by 8 and 4, then the quad swaps). All VALU: the ds_bpermute round trips of __shfl_xor were most
// of a GEMV's time after its loads had landed (o_proj, 2 rows: 9.0 -> 6.2 us without them)
template <int CTRL> __device__ __forceinline__ float dpp_f(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, false));
}
__device__ __forceinline__ float wave_sum(float v) {
    const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    const auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(b[0]) + __uint_as_float(b[1]);
    v += dpp_f<0x128>(v);  // row_ror:8
    v += dpp_f<0x124>(v);  // row_ror:4
    v += dpp_f<0x4e>(v);   // quad_perm [2, 3, 0, 1]
    return v + dpp_f<0xb1>(v);  // quad_perm [1, 0, 3, 2]
}
// N values summed over the wavefront together: the 32- and 16-lane swaps each fold two values into one register (a pair
// of values costs one swap and one add instead of two of each), then DPP within the 16-lane rows. On return v[k] holds,
// in all lanes of row q = lane / 16, the sum of value wave_sums_index(k, q). The tree over the lanes is the same for
// every N and value (lanes 32 apart, 16, 8, 4, 2, 1).
template <int N> __device__ __forceinline__ void wave_sums(float (&v)[N]) {
    constexpr int H = (N + 1) / 2, Q = (H + 1) / 2;
#pragma unroll
    for (int k = 0; k < H; k++) {
        const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[k]), __float_as_uint(k + H < N ? v[k + H] : v[k]),
                                                        false, false);
        v[k] = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    }
#pragma unroll
    for (int k = 0; k < Q; k++) {
        const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v[k]), __float_as_uint(k + Q < H ? v[k + Q] : v[k]),
                                                        false, false);
        v[k] = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    }
#pragma unroll
    for (int k = 0; k < Q; k++) {
        v[k] += dpp_f<0x128>(v[k]);
        v[k] += dpp_f<0x124>(v[k]);
        v[k] += dpp_f<0x4e>(v[k]);
        v[k] += dpp_f<0xb1>(v[k]);
    }
}
// the value whose sum v[k] holds in row q, or N if none (its lanes hold a copy of another)
template <int N> __device__ __forceinline__ int wave_sums_index(int k, int q) {
    constexpr int H = (N + 1) / 2, Q = (H + 1) / 2;
    const int h = k + ((q & 1) ? Q : 0);
    if ((q & 1) && h >= H) return N;
    const int i = h + ((q & 2) ? H : 0);
    return i < N ? i : N;
}

__global__ void __launch_bounds__(256) quantize_rows_kernel(const uint16_t* __restrict__ W, int8_t* __restrict__ q,
                                                            float* __restrict__ s, int I) {
    __shared__ float red[4];
    const size_t row = blockIdx.x;
    const _Float16* wr = reinterpret_cast<const _Float16*>(W) + row * I;
    float m = 0.f;
    for (int i = threadIdx.x; i < I; i += 256) m = fmaxf(m, fabsf((float)wr[i]));
#pragma unroll
    for (int o = 32; o; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    const float sc = m > 0.f ? m / 127.f : 1.f;
    for (int i = threadIdx.x; i < I; i += 256) q[row * I + i] = (int8_t)(int)__builtin_rintf((float)wr[i] / sc);
    if (threadIdx.x == 0) s[row] = sc;
}

// A transfer of 16 bytes a lane from base + off (uniform base, 32-bit byte offset) to lds + 16 * lane, in inline asm: the
// compiler cannot tell which LDS bytes it writes and would make the next LDS read wait for every load in flight. The
// kernels wait for their own transfers.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void dma16x(const void* base, uint32_t off, const unsigned char* lds) {
    const uint32_t m = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)lds);
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(m)
                 : "memory", "m0");
}
#pragma clang diagnostic pop
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
constexpr int GV_R = 8;       // weight rows of a row group
// 16-byte chunks per lane and row loaded before any is used: 16 KB per wavefront in flight, 8 KB from NT = 5 on
// (registers)
template <int NT> constexpr int gv_u() { return NT <= 4 ? 2 : 1; }
constexpr int GV_WAVES = 8;   // wavefronts per workgroup

// A grid of nb workgroups; in round j, wavefront wv of workgroup b takes row group b + nb * (wv / KS + j * 8 / KS)
// over the KS-th part wv % KS of I, and the KS partial sums of a group are added in LDS in part order. KS (1, 2, 4
// or 8) depends on O and I only, so the sum order of a row never depends on NT.
template <int NT>
__global__ void __launch_bounds__(64 * GV_WAVES) gemv_kernel(const int8_t* __restrict__ q, const float* __restrict__ s,
                                                             const float* __restrict__ x, float* __restrict__ y, int I,
                                                             int O, int KS) {
    constexpr int GV_U = gv_u<NT>();
    extern __shared__ __align__(16) float xs[];  // [NT][I], then the partial sums [GV_WAVES][NT][GV_R]
    float* red = xs + NT * I;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, nb = gridDim.x;
    const int ngroups = (O + GV_R - 1) / GV_R, gpr = GV_WAVES / KS;  // groups per workgroup and round
    const int rounds = (ngroups + nb * gpr - 1) / (nb * gpr);
    const int part = wv % KS, slice = I / 16 / KS, cb = part * slice, ce = cb + slice;  // 16-byte chunks of a row
    u32x4 w[GV_U][GV_R];
#define GV_LOAD(g_, c0_)                                                                                         \
    do {                                                                                                         \
        _Pragma("unroll") for (int u = 0; u < GV_U; u++)                                                         \
        _Pragma("unroll") for (int r = 0; r < GV_R; r++) {                                                       \
            const u32x4* row_ = reinterpret_cast<const u32x4*>(q + (size_t)min((g_) * GV_R + r, O - 1) * I);     \
            const int c_ = (c0_) + 64 * u + lane;                                                                \
            w[u][r] = c_ < ce ? __builtin_nontemporal_load(row_ + c_) : u32x4{0u, 0u, 0u, 0u};                  \
        }                                                                                                        \
    } while (0)
    for (int e = tid; e < NT * I / 4; e += 64 * GV_WAVES)
        reinterpret_cast<float4*>(xs)[e] = reinterpret_cast<const float4*>(x)[e];
    __syncthreads();
    for (int j = 0; j < rounds; j++) {
        const int g = blockIdx.x + nb * (wv / KS + j * gpr);
        if (g < ngroups) {
            float acc[NT][GV_R];
#pragma unroll
            for (int t = 0; t < NT; t++)
#pragma unroll
                for (int r = 0; r < GV_R; r++) acc[t][r] = 0.f;
            for (int c0 = cb; c0 < ce; c0 += 64 * GV_U) {
                GV_LOAD(g, c0);
#pragma unroll
                for (int u = 0; u < GV_U; u++) {
                    const int c = c0 + 64 * u + lane;
                    if (c >= ce) continue;  // only when a part is shorter than 64 chunks (I % 1024 != 0)
#pragma unroll
                    for (int t = 0; t < NT; t++) {
#pragma unroll
                        for (int d = 0; d < 4; d++) {
                            const float4 xv = reinterpret_cast<const float4*>(xs + t * I)[4 * c + d];
#pragma unroll
                            for (int r = 0; r < GV_R; r++) {
                                const uint32_t wd = w[u][r][d];
                                acc[t][r] += (float)(int8_t)(wd) * xv.x;
                                acc[t][r] += (float)(int8_t)(wd >> 8) * xv.y;
                                acc[t][r] += (float)(int8_t)(wd >> 16) * xv.z;
                                acc[t][r] += (float)(int8_t)(wd >> 24) * xv.w;
                            }
                        }
                    }
                }
            }
#pragma unroll
            for (int t = 0; t < NT; t++)
#pragma unroll
                for (int r = 0; r < GV_R; r++) {
                    const float v = wave_sum(acc[t][r]);
                    if (lane == 0) red[(wv * NT + t) * GV_R + r] = v;
                }
        }
        __syncthreads();
        if (g < ngroups && part == 0 && lane < NT * GV_R) {
            const int t = lane / GV_R, r = lane % GV_R, o = g * GV_R + r;
            float v = red[(wv * NT + t) * GV_R + r];
            for (int p = 1; p < KS; p++) v += red[((wv + p) * NT + t) * GV_R + r];
            if (o < O) y[(size_t)t * O + o] = v * s[o];
        }
        __syncthreads();  // the partial sums are read before the next round writes them
    }
#undef GV_LOAD
}

// The same product when a part of a row is at most 64 U chunks, U loads a lane (U = 1: I up to 8192, the attention's qkv and
// o shapes among them; U = 2: 16384, where at most two input rows come at once): a wavefront takes R rows, sends all
// of its loads before any product and needs no loop. Same sum order as gemv_kernel.
// It is bound by the weight stream and the launch for few input rows, by the FMAs (and the widening, once per group of
// 4 input rows) for many. One or two input rows are read by each lane straight from L2; more are copied into LDS once
// per workgroup by DMA (float4 e of the rows in slot e ^ (e / 8) % 4: the lanes of a read, 64 bytes apart, then hit
// different banks), as eight wavefronts each reading 4 or 8 rows from L2 took longer than the weights, and their
// values left no registers for the weights in flight. The wait for the transfers counts on the R weight loads being
// issued after them: q is no __restrict__ pointer, since loads through a noalias, read-only kernel argument count as
// loads of constant memory, which the compiler may move across the transfers' asm statements. Graph-replayed over rotating weights, us, before -> now (before:
// every input row from L2, 8 rows a wavefront, qkv's rows not split, six cross-lane steps per sum):
//   input rows          1           2           3            4            6            8
//   qkv  9216 x 2048    7.0 -> 5.2  8.7 -> 6.0  12.3 -> 6.6  21.0 -> 7.7  16.3 -> 9.2  20.9 -> 10.6
//   o    2048 x 4096    4.2 -> 3.9  4.8 -> 4.9  5.4 -> 4.8   6.2 -> 5.1   7.7 -> 6.1   9.3 -> 6.7
template <int NT, int R, int U>
__global__ void __launch_bounds__(64 * GV_WAVES, 2) gemv1_kernel(const int8_t* q, const float* __restrict__ s,
                                                                 const float* __restrict__ x, float* __restrict__ y,
                                                                 int I, int O, int KS) {
    constexpr bool XL = NT > 2;
    extern __shared__ __align__(16) float xs[];  // XL: the input rows [NT][I]; then the partial sums [GV_WAVES][NT * R]
    float* red = xs + (XL ? NT * I : 0);
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int gpw = GV_WAVES / KS, part = wv % KS, slice = I / 16 / KS, cb = part * slice;
    const int g = blockIdx.x * gpw + wv / KS;
    static_assert(U == 1 || !XL, "two loads a lane: input rows from L2");
    int c[U];
#pragma unroll
    for (int u = 0; u < U; u++) c[u] = min(cb + 64 * u + lane, I / 16 - 1);
    constexpr int TB = NT < 4 ? NT : 4;
    float4 xv[U][TB][4];
    if constexpr (XL) {
        if ((reinterpret_cast<uintptr_t>(x) & 15) == 0) {
            const int n = NT * I / 256;  // 1 KB transfers
            for (int i = wv; i < n; i += GV_WAVES) {
                const uint32_t e = 64 * i + lane;
                dma16x(x, 16 * (e ^ ((e >> 3) & 3)), reinterpret_cast<const unsigned char*>(xs) + 1024 * i);
            }
        } else {
            // rows off a 16-byte boundary: the same slots by loads and LDS writes (8 rows: qkv 10.8 us against 10.6 with
            // transfers, o 6.9 against 6.7; gemv_kernel, which ran them before, 26.2 and 14.2)
#pragma unroll 4
            for (uint32_t e = tid; e < (uint32_t)NT * I / 4; e += 64 * GV_WAVES) {
                const float* p = x + 4 * (e ^ ((e >> 3) & 3));
                reinterpret_cast<float4*>(xs)[e] = make_float4(p[0], p[1], p[2], p[3]);
            }
        }
    } else {
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int t = 0; t < NT; t++)
#pragma unroll
                for (int d = 0; d < 4; d++) xv[u][t][d] = reinterpret_cast<const float4*>(x + (size_t)t * I)[4 * c[u] + d];
    }
    u32x4 w[U][R];
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
        for (int r = 0; r < R; r++)  // rows past the last repeat it
            w[u][r] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(q + (size_t)min(g * R + r, O - 1) * I) + c[u]);
    // XL: this wavefront's transfers have landed when only its R weight loads are in flight
    if constexpr (XL) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(R) : "memory");
    float acc[NT * R];
#pragma unroll
    for (int t0 = 0; t0 < NT; t0 += TB) {  // input rows in groups whose values fit the registers
        if constexpr (XL) {
#pragma unroll
            for (int t = t0; t < NT && t < t0 + TB; t++)
#pragma unroll
                for (int d = 0; d < 4; d++) {
                    const uint32_t e = t * (I / 4) + 4 * c[0] + d;
                    xv[0][t - t0][d] = reinterpret_cast<const float4*>(xs)[e ^ ((e >> 3) & 3)];
                }
        }
#pragma unroll
        for (int r = 0; r < R; r++) {
            float a[TB];
#pragma unroll
            for (int u = 0; u < U; u++) {
#pragma unroll
                for (int t = 0; t < TB; t++) a[t] = u ? acc[(t0 + t) * R + r] : 0.f;
#pragma unroll
                for (int d = 0; d < 4; d++) {
                    const uint32_t wd = w[u][r][d];
                    const float w0 = (float)(int8_t)wd, w1 = (float)(int8_t)(wd >> 8), w2 = (float)(int8_t)(wd >> 16),
                                w3 = (float)(int8_t)(wd >> 24);
#pragma unroll
                    for (int t = 0; t < TB && t0 + t < NT; t++) {
                        a[t] = fmaf(w0, xv[u][t][d].x, a[t]);
                        a[t] = fmaf(w1, xv[u][t][d].y, a[t]);
                        a[t] = fmaf(w2, xv[u][t][d].z, a[t]);
                        a[t] = fmaf(w3, xv[u][t][d].w, a[t]);
                    }
                }
#pragma unroll
                for (int t = 0; t < TB && t0 + t < NT; t++) {
                    float& s_ = acc[(t0 + t) * R + r];
                    s_ = 64 * u + lane < slice ? a[t] : u ? s_ : 0.f;  // lanes past the part add nothing
                }
            }
        }
        if constexpr (NT > TB) asm volatile("" ::: "memory");  // the next group's values are read after these are used
    }
    wave_sums(acc);
#pragma unroll
    for (int k = 0; k < ((NT * R + 1) / 2 + 1) / 2; k++) {
        const int i = wave_sums_index<NT * R>(k, lane >> 4);
        if ((lane & 15) == 0 && i < NT * R) red[wv * NT * R + i] = acc[k];
    }
    __syncthreads();
    const int rows = gpw * R;  // of this workgroup
    for (int e = tid; e < NT * rows; e += 64 * GV_WAVES) {
        const int t = e / rows, rr = e % rows, gl = rr / R, r = rr % R, o = (blockIdx.x * gpw + gl) * R + r;
        if (o >= O) continue;
        float v = red[gl * KS * NT * R + t * R + r];
        for (int p = 1; p < KS; p++) v += red[(gl * KS + p) * NT * R + t * R + r];
        y[(size_t)t * O + o] = v * s[o];
    }
}

// ---- prefill GEMM ----
// The weight forms of a dense matrix (struct Mat, kernels.cuh:186-196): int8 with a row scale, int4 and int6 with a
// scale per 64 inputs (gs64), fp16.
enum { MF_I8 = 0, MF_Q4 = 1, MF_Q6 = 2, MF_F16 = 3 };

// A product rounded to fp32 before anything else rounds it: without the barrier the compiler may fuse a multiply
// with its fp16 conversion (v_fma_mix*), one rounding instead of the reference's two.
__device__ __forceinline__ float r32(float x) {
    asm volatile("" : "+v"(x));
    return x;
}
// 16 weights of one row at k .. k + 15 (k % 16 == 0) -> 8 dwords of fp16 pairs, as the reference's GEMMs widen them:
// int8 exactly (row scale applied after the sums); int4 / int6 times the group scale in fp32, then rounded to fp16
// (kernels.cuh:276-279, 313-317: __float2half / __floats2half2_rn of (float)v * s); fp16 as stored.
struct WStage {
    uint4 a;      // int8: 16 codes; int4 / int6: .x, .y the 16 low nibbles; fp16: halves 0-7
    uint4 b;      // fp16: halves 8-15
    uint32_t h;   // int6: the 16 high 2-bit fields
    float sc;     // int4 / int6: the group scale
};
// loaded from element offset off (row * I + k) past a uniform element base, the tile's first row and K step
template <int FMT, class off_t>
__device__ __forceinline__ void wstage_load_at(WStage& w, const void* W, const uint8_t* Wh, const float* s, size_t base,
                                               off_t off) {
    if constexpr (FMT == MF_I8) {
        w.a = *reinterpret_cast<const uint4*>(reinterpret_cast<const int8_t*>(W) + base + off);
    } else if constexpr (FMT == MF_F16) {
        const uint4* p = reinterpret_cast<const uint4*>(reinterpret_cast<const uint8_t*>(W) + 2 * base + (size_t)(2 * off));
        w.a = p[0];
        w.b = p[1];
    } else {
        const uint2 lo = *reinterpret_cast<const uint2*>(reinterpret_cast<const uint8_t*>(W) + base / 2 + off / 2);
        w.a = make_uint4(lo.x, lo.y, 0u, 0u);
        if constexpr (FMT == MF_Q6) w.h = *reinterpret_cast<const uint32_t*>(Wh + base / 4 + off / 4);
        w.sc = *reinterpret_cast<const float*>(reinterpret_cast<const uint8_t*>(s + base / 64) + off / 64 * 4);
    }
}
// a use of everything that wstage_load_at has loaded
template <int FMT>
__device__ __forceinline__ void wstage_use(const WStage& w) {
    if constexpr (FMT == MF_I8) asm volatile("" ::"v"(w.a.x), "v"(w.a.y), "v"(w.a.z), "v"(w.a.w));
    else if constexpr (FMT == MF_F16)
        asm volatile("" ::"v"(w.a.x), "v"(w.a.y), "v"(w.a.z), "v"(w.a.w), "v"(w.b.x), "v"(w.b.y), "v"(w.b.z), "v"(w.b.w));
    else asm volatile("" ::"v"(w.a.x), "v"(w.a.y), "v"(w.sc));
    if constexpr (FMT == MF_Q6) asm volatile("" ::"v"(w.h));
}
template <int FMT>
__device__ __forceinline__ void wstage_widen(const WStage& w, bool ok, uint32_t (&h)[8]) {
    if constexpr (FMT == MF_I8) {
        i8x4_to_h4(ok ? w.a.x : 0u, h[0], h[1]);
        i8x4_to_h4(ok ? w.a.y : 0u, h[2], h[3]);
        i8x4_to_h4(ok ? w.a.z : 0u, h[4], h[5]);
        i8x4_to_h4(ok ? w.a.w : 0u, h[6], h[7]);
    } else if constexpr (FMT == MF_F16) {
        h[0] = ok ? w.a.x : 0u; h[1] = ok ? w.a.y : 0u; h[2] = ok ? w.a.z : 0u; h[3] = ok ? w.a.w : 0u;
        h[4] = ok ? w.b.x : 0u; h[5] = ok ? w.b.y : 0u; h[6] = ok ? w.b.z : 0u; h[7] = ok ? w.b.w : 0u;
    } else {
        float v[16];
#pragma unroll
        for (int e = 0; e < 16; e++) {
            const uint32_t dw = e < 8 ? w.a.x : w.a.y;
            int q;
            if constexpr (FMT == MF_Q4) q = (int)__builtin_amdgcn_sbfe(dw, 4 * (e & 7), 4);  // two's complement nibble
            else q = (int)(((dw >> (4 * (e & 7))) & 15u) | (((w.h >> (2 * e)) & 3u) << 4)) - 32;  // 6-bit code, offset 32
            v[e] = r32((float)q * w.sc);
        }
#pragma unroll
        for (int i = 0; i < 8; i++) h[i] = ok ? h22u(half2_t{(_Float16)v[2 * i], (_Float16)v[2 * i + 1]}) : 0u;
    }
}

// gemm_tile_kernel: Y = X . W^T (* s) on v_mfma_f32_16x16x32_f16, one workgroup of 8 wavefronts per tile of BM weight
// rows x BN tokens. Wavefronts form a GM x GN x KW grid: each computes 16 WM x 16 WN outputs over the KW-th part of
// every K step of 32 KW BKU inputs; the KW partial sums of an output are added through LDS at the end, in part order.
// Weights go through registers, PD steps ahead, and are widened on their way into LDS (two buffers); activations the
// same way from fp32, or (XH) rounded to fp16 once before the kernel and moved into LDS by DMA.
//
// What bounds it. The large tiles: LDS traffic (a 144 x 64 wavefront tile reads 13 KB per 36 MFMAs of 16 cycles, ~90 B
// a cycle of the CU's 128, besides the staging's writes) beside the MFMAs, and the clock under MFMA load. 288 x 256
// outputs are what 256 VGPRs and 160 KB of LDS hold, and at 2048 tokens the qkv matrix is 256 such tiles, one a CU.
// The small tiles: the latency of a K step's loads; a tile that one CU runs alone has all of its K parts inside one
// workgroup, so no partial sum goes through memory and no second launch adds them.
// Measured (graph-replayed calls over 300 MB of rotating weights, us; before: 128 x 128 tiles on 4 wavefronts or 4 + 4
// split roles, an fp16 rounding launch for every call, K split over workgroups with a reduction launch), int8:
//   tokens              9          64         300        512        1024       2048
//   qkv  9216 x 2048    21.1->10.4 33.0->16.1 47.9->31.7 50.8->39.2 74.0->58.7 140->90.6 (853 TFLOPS)
//   o    2048 x 4096    17.9->10.1 25.0->11.9 34.6->23.3 38.9->25.6 53.4->36.1 79.5->53.8 (639 TFLOPS)
// int4 at 300 tokens: qkv 45.4 -> 32.2, o 31.9 -> 23.5; fp16 at 2048: 137 -> 85.8, 81.8 -> 58.9.
template <int WM_, int WN_, int GM_, int GN_, int KW_, int BKU_, int PD_, bool XH_ = false, int WPE_ = 2>
struct GemmTile {
    static constexpr int WM = WM_, WN = WN_, GM = GM_, GN = GN_, KW = KW_, BKU = BKU_, PD = PD_;
    static constexpr bool XH = XH_;
    static constexpr int WPE = WPE_;  // wavefronts per SIMD the registers allow
    using off_t = std::conditional_t<(16 * WM * GM * 16 * WN * GN > 256), uint32_t, size_t>;  // offsets inside a tile
    static constexpr int BM = 16 * WM * GM, BN = 16 * WN * GN, BK = 32 * KW * BKU, LD = BK + 8, XLD = XH ? BK : LD;
    static constexpr int STAGE = BM * LD + BN * XLD;                   // halves of a K step's operands
    static constexpr int RED = KW > 1 ? KW * BN * (BM + 4) * 4 : 0;    // bytes of the partial sums
    static constexpr int LDS = 2 * STAGE * 2 > RED ? 2 * STAGE * 2 : RED;
    static constexpr int NW = (BM * (BK / 16) + 511) / 512;            // 16-weight units a thread stages
    static constexpr int NX = XH ? 1 : (BN * (BK / 4) + 511) / 512;    // 4-activation units a thread stages
    static constexpr int ND = BN * BK * 2 / 8192;                      // 1 KB transfers a wavefront issues (XH)
    static_assert(GM * GN * KW == 8 && LDS <= 160 * 1024, "tile");
    static_assert(!XH || BK <= 512, "a transfer holds whole rows of a K step");
};
template <int N> __device__ __forceinline__ void gemm_vm_wait() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }
// The XH wait counts on a K step's weight loads being issued between its transfers and the wait: W, Wh and s are no
// __restrict__ pointers there (see gemv1_kernel), and every load has a use, the last ones after the loop. The other tiles
// wait for nothing by count and leave the order to the compiler.
// Four outputs (row scales) of a lane from p on, n of them inside the row: 16-byte accesses at any 4-byte alignment, which the
// hardware takes as they are. With 4-byte stores wherever O or Y was not a multiple of 16 bytes, a line was written in four
// passes, and four scale loads a lane cost an int8 tile with a short K as much as its outputs (us, 4-byte accesses -> so:
// 11925 x 320, 1625 tokens int8 59.0 -> 42.7, fp16 65.2 -> 40.0; 11971 x 1088, 389 tokens fp16 37.9 -> 29.9; 6722 x 128, 1005
// tokens int8 26.1 -> 16.5). inside (uniform): the whole tile is.
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
__device__ __forceinline__ f32x4u load4(const float* p, int n, bool inside) {
    if (inside || n >= 4) return *reinterpret_cast<const f32x4u*>(p);
    f32x4u v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int e = 0; e < 3; e++)
        if (e < n) v[e] = p[e];
    return v;
}
__device__ __forceinline__ void store4(float* p, float4_t v, int n, bool inside) {
    if (inside) {
        *reinterpret_cast<f32x4u*>(p) = v;
    } else {
        asm volatile("");  // keeps the two stores apart: merged, the branch is taken lane by lane, 1 to 2 % of a small call
        if (n >= 4) {
            *reinterpret_cast<f32x4u*>(p) = v;
        } else {
#pragma unroll
            for (int e = 0; e < 3; e++)
                if (e < n) p[e] = v[e];
        }
    }
}
template <class C, class T>
using weight_ptr = std::conditional_t<C::XH, const T*, const T* __restrict__>;
// SPLIT: workgroup (x, y) takes spp K steps of tile x from spp y on and writes their sums, without the row scales, to the
// y-th [S][O] of Y. An instance of its own, as the parts' bounds would cost every call 0.2 to 0.4 us.
template <int FMT, class C, bool SPLIT>
__global__ void __launch_bounds__(512, C::WPE) gemm_tile_kernel(weight_ptr<C, void> W, weight_ptr<C, uint8_t> Wh,
                                                           weight_ptr<C, float> s, const void* __restrict__ Xv,
                                                           float* __restrict__ Y, int S, int I, int O, int spp) {
    extern __shared__ __align__(16) _Float16 gl[];
    const int tid = threadIdx.x, lane = tid & 63, m16 = lane & 15, g = lane >> 4;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nO = (O + C::BM - 1) / C::BM, nt = gridDim.x;
    // XCD-aware order (block b runs on XCD b % 8): each XCD takes a run of tiles, weight tiles fastest, so that a token
    // tile's activations are read into as few L2s as possible
    const int q8 = nt >> 3, r8 = nt & 7, xc = blockIdx.x & 7, xi = blockIdx.x >> 3;
    const int tile = (xc < r8 ? xc * (q8 + 1) : r8 * (q8 + 1) + (xc - r8) * q8) + xi;
    const int o0 = (tile % nO) * C::BM, s0 = (tile / nO) * C::BN;
    // the whole K steps [kb, kb + nk); a ragged one follows the last
    const int kb = SPLIT ? spp * (int)blockIdx.y : 0, nk = SPLIT ? min(spp, I / C::BK - kb) : I / C::BK;
    WStage wst[C::PD][C::NW];
    float4 xst[C::PD][C::NX];
    constexpr int WU = C::BK / 16, XU = C::BK / 4;  // units of a row
    // XH: transfer d of wavefront wv covers rows of the tile in 1 KB runs; lane l moves 16-byte piece sl of a row into
    // slot l % PC (piece = slot ^ row % 8), so that the 16 rows of an operand read hit different banks
    constexpr int PC = C::BK / 8, RPI = 64 / PC;
    uint32_t xd[C::XH ? C::ND : 1];
    if constexpr (C::XH) {
#pragma unroll
        for (int d = 0; d < C::ND; d++) {
            const int r = (wv * C::ND + d) * RPI + lane / PC, sl = lane % PC;
            xd[d] = ((uint32_t)min(r, S - 1 - s0) * I + 8 * (sl ^ (r & 7))) * 2;
        }
    }
    auto dma = [&](int kt, int buf) {
        if constexpr (C::XH) {
            const _Float16* base = reinterpret_cast<const _Float16*>(Xv) + (size_t)s0 * I + (kb + kt) * C::BK;
            const unsigned char* dst = reinterpret_cast<const unsigned char*>(gl + buf * C::STAGE + C::BM * C::LD);
#pragma unroll
            for (int d = 0; d < C::ND; d++) dma16x(base, xd[d], dst + (wv * C::ND + d) * 1024);
        }
    };
    // a thread's units: offsets from the tile's first row (rows past the matrix repeat the last one: their outputs are
    // not stored), the K step added to the uniform bases
    typename C::off_t wro[C::NW], xro[C::NX];
#pragma unroll
    for (int u = 0; u < C::NW; u++) {
        const int e = tid + 512 * u;
        wro[u] = (typename C::off_t)min(e / WU, O - 1 - o0) * I + 16 * (e % WU);
    }
#pragma unroll
    for (int u = 0; u < C::NX; u++) {
        const int e = tid + 512 * u;
        xro[u] = ((typename C::off_t)min(e / XU, S - 1 - s0) * I + 4 * (e % XU)) * 4;
    }
    auto load = [&](WStage(&w)[C::NW], float4(&x)[C::NX], int kt, auto rag) {
        constexpr bool RAG = decltype(rag)::value;
        const size_t wbase = (size_t)o0 * I + (size_t)(kb + kt) * C::BK;
        const char* xb = reinterpret_cast<const char*>(Xv) + ((size_t)s0 * I + (size_t)(kb + kt) * C::BK) * 4;
#pragma unroll
        for (int u = 0; u < C::NW; u++) {
            typename C::off_t off = wro[u];  // RAG: inputs past the row's end are read inside it, zeroed when stored
            if (RAG) off -= max(0, (kb + kt) * C::BK + 16 * ((tid + 512 * u) % WU) - (I - 16));
            wstage_load_at<FMT>(w[u], W, Wh, s, wbase, off);
        }
        if constexpr (C::XH) return;
#pragma unroll
        for (int u = 0; u < C::NX; u++) {
            if ((C::BN * XU) % 512 != 0 && tid + 512 * u >= C::BN * XU) break;
            typename C::off_t off = xro[u];
            if (RAG) off -= 4 * max(0, (kb + kt) * C::BK + 4 * ((tid + 512 * u) % XU) - (I - 4));
            x[u] = *reinterpret_cast<const float4*>(xb + off);
        }
    };
    auto store = [&](const WStage(&w)[C::NW], const float4(&x)[C::NX], int kt, auto rag) {
        constexpr bool RAG = decltype(rag)::value;
        _Float16* b = gl + (kt & 1) * C::STAGE;
#pragma unroll
        for (int u = 0; u < C::NW; u++) {
            const int e = tid + 512 * u, r = e / WU, k = 16 * (e % WU);
            if ((C::BM * WU) % 512 != 0 && e >= C::BM * WU) break;
            uint32_t h[8];
            wstage_widen<FMT>(w[u], !RAG || (kb + kt) * C::BK + k < I, h);
            uint4* d = reinterpret_cast<uint4*>(b + r * C::LD + k);
            d[0] = make_uint4(h[0], h[1], h[2], h[3]);
            d[1] = make_uint4(h[4], h[5], h[6], h[7]);
        }
        if constexpr (C::XH) return;
        b += C::BM * C::LD;
#pragma unroll
        for (int u = 0; u < C::NX; u++) {
            const int e = tid + 512 * u, r = e / XU, k = 4 * (e % XU);
            if ((C::BN * XU) % 512 != 0 && e >= C::BN * XU) break;
            const bool ok = !RAG || (kb + kt) * C::BK + k < I;
            const float4 v = x[u];
            *reinterpret_cast<uint2*>(b + r * C::LD + k) =
                make_uint2(ok ? h22u(half2_t{(_Float16)v.x, (_Float16)v.y}) : 0u, ok ? h22u(half2_t{(_Float16)v.z, (_Float16)v.w}) : 0u);
        }
    };
    const int kg = wv / (C::GM * C::GN), wg = wv % (C::GM * C::GN), wr = (wg / C::GN) * 16 * C::WM, wt = (wg % C::GN) * 16 * C::WN;
    float4_t acc[C::WM][C::WN];
#pragma unroll
    for (int i = 0; i < C::WM; i++)
#pragma unroll
        for (int j = 0; j < C::WN; j++) acc[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};
    auto bar = [] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
    const _Float16* ws0 = gl + (wr + m16) * C::LD + kg * 32 * C::BKU + 8 * g;
    const _Float16* xs0 = gl + C::BM * C::LD + (wt + m16) * C::XLD + (C::XH ? 0 : kg * 32 * C::BKU + 8 * g);
    int xu[C::BKU];  // halves from xs0 to the operand of sub-step u
#pragma unroll
    for (int u = 0; u < C::BKU; u++) xu[u] = C::XH ? 8 * ((4 * (kg * C::BKU + u) + g) ^ (m16 & 7)) : 32 * u;
    auto compute = [&](int kt) {
        const _Float16* wb = ws0 + (kt & 1) * C::STAGE;
        const _Float16* xb = xs0 + (kt & 1) * C::STAGE;
#pragma unroll
        for (int u = 0; u < C::BKU; u++) {
            half8_t b[C::WN];
#pragma unroll
            for (int j = 0; j < C::WN; j++) b[j] = *reinterpret_cast<const half8_t*>(xb + 16 * j * C::XLD + xu[u]);
#pragma unroll
            for (int i = 0; i < C::WM; i++) {
                const half8_t a = *reinterpret_cast<const half8_t*>(wb + 16 * i * C::LD + 32 * u);
#pragma unroll
                for (int j = 0; j < C::WN; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b[j], acc[i][j], 0, 0, 0);
            }
        }
    };
    constexpr int LPU = FMT == MF_I8 ? 1 : FMT == MF_Q6 ? 3 : 2;  // loads of a weight unit
    constexpr std::false_type whole{};
    if (nk > 0) {
        dma(0, 0);
#pragma unroll
        for (int p = 0; p < C::PD; p++) load(wst[p], xst[p], min(p, nk - 1), whole);
        store(wst[0], xst[0], 0, whole);
        load(wst[0], xst[0], min(C::PD, nk - 1), whole);
        if constexpr (C::XH) gemm_vm_wait<C::NW * LPU>();
        bar();
    }
    // Step kt: its operands are in buffer kt % 2; the next step's weights and activations, loaded PD steps ago, are
    // widened into the other buffer and the registers refilled. The two wavefronts of a SIMD stage at opposite ends
    // of the step, so that one's MFMAs run beside the other's loads and LDS writes. No condition inside: past the
    // last step the last one is loaded and stored again, into a buffer that nobody reads.
    auto steps = [&](auto first) {
        for (int k0 = 0; k0 < nk; k0 += C::PD) {
#pragma unroll
            for (int p = 0; p < C::PD; p++) {
                const int kt = k0 + p;
                if (C::PD > 1 && kt >= nk) break;
                WStage(&w)[C::NW] = wst[(p + 1) % C::PD];
                float4(&x)[C::NX] = xst[(p + 1) % C::PD];
                if constexpr (decltype(first)::value) {
                    store(w, x, kt + 1, whole);
                    dma(min(kt + 1, nk - 1), (kt + 1) & 1);
                    load(w, x, min(kt + 1 + C::PD, nk - 1), whole);
                    compute(kt);
                } else {
                    dma(min(kt + 1, nk - 1), (kt + 1) & 1);
                    compute(kt);
                    store(w, x, kt + 1, whole);
                    load(w, x, min(kt + 1 + C::PD, nk - 1), whole);
                }
                if constexpr (C::XH) gemm_vm_wait<C::NW * LPU>();  // the step's transfers; the weight loads after them fly on
                bar();
            }
        }
    };
    if (wv < 4) steps(std::true_type{});
    else steps(std::false_type{});
    if constexpr (C::XH) {
#pragma unroll
        for (int p = 0; p < C::PD; p++)
#pragma unroll
            for (int u = 0; u < C::NW; u++) wstage_use<FMT>(wst[p][u]);
    } else {
        if ((!SPLIT || nk < spp) && (kb + nk) * C::BK < I) {  // the ragged last step: inputs past I are zero in both operands
            load(wst[0], xst[0], nk, std::true_type{});
            store(wst[0], xst[0], nk, std::true_type{});
            bar();
            compute(nk);
            bar();
        }
    }
    if (SPLIT) Y += (size_t)blockIdx.y * S * O;
    const bool inside = o0 + C::BM <= O;  // uniform
    // acc[i][j] element e: weight row wr + 16 i + 4 g + e, token wt + 16 j + m16
    if constexpr (C::KW == 1) {
#pragma unroll
        for (int i = 0; i < C::WM; i++) {
            const int o = o0 + wr + 16 * i + 4 * g;
            if (o >= O) continue;
            f32x4u sc = {1.f, 1.f, 1.f, 1.f};
            if constexpr (FMT == MF_I8 && !SPLIT) sc = load4(s + o, O - o, inside);
#pragma unroll
            for (int j = 0; j < C::WN; j++) {
                const int t = s0 + wt + 16 * j + m16;
                if (t >= S) continue;
                store4(Y + (size_t)t * O + o, acc[i][j] * sc, O - o, inside);
            }
        }
    } else {
        float* red = reinterpret_cast<float*>(gl);  // [part][token][row], rows padded by 4
        constexpr int RL = C::BM + 4;
#pragma unroll
        for (int i = 0; i < C::WM; i++)
#pragma unroll
            for (int j = 0; j < C::WN; j++) {
                const float4_t v = acc[i][j];
                *reinterpret_cast<float4*>(red + ((size_t)kg * C::BN + wt + 16 * j + m16) * RL + wr + 16 * i + 4 * g) =
                    make_float4(v[0], v[1], v[2], v[3]);
            }
        bar();
        for (int e = tid; e < C::BN * (C::BM / 4); e += 512) {
            const int tl = e / (C::BM / 4), rl = 4 * (e % (C::BM / 4)), t = s0 + tl, o = o0 + rl;
            if (t >= S || o >= O) continue;
            float4 a = *reinterpret_cast<const float4*>(red + (size_t)tl * RL + rl);
#pragma unroll
            for (int p = 1; p < C::KW; p++) {
                const float4 b = *reinterpret_cast<const float4*>(red + ((size_t)p * C::BN + tl) * RL + rl);
                a.x += b.x; a.y += b.y; a.z += b.z; a.w += b.w;
            }
            f32x4u v = {a.x, a.y, a.z, a.w};
            if constexpr (FMT == MF_I8 && !SPLIT) v *= load4(s + o, O - o, inside);
            store4(Y + (size_t)t * O + o, v, O - o, inside);
        }
    }
}
// The parts of a K split summed in part order (deterministic), times the row scale (int8; s = nullptr: none)
__global__ void __launch_bounds__(256) gemm_reduce_kernel(const float* __restrict__ part, const float* __restrict__ s,
                                                          float* __restrict__ Y, size_t n, int O, int nks) {
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
        float a = part[i];
        for (int k = 1; k < nks; k++) a += part[k * n + i];
        Y[i] = s ? a * s[i % O] : a;
    }
}
// Activations rounded to fp16 once (round to nearest even, as kernels.cuh:306-307 rounds them inside gemm_i8_k): the
// GEMM tiles re-read them once per weight tile, so fp16 halves that traffic and takes the rounding off the staging.
__global__ void __launch_bounds__(256) round_f16_kernel(const float4* __restrict__ X, uint2* __restrict__ Xh, size_t n4) {
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n4; i += (size_t)gridDim.x * 256) {
        const float4 v = X[i];
        Xh[i] = make_uint2(h22u(half2_t{(_Float16)v.x, (_Float16)v.y}), h22u(half2_t{(_Float16)v.z, (_Float16)v.w}));
    }
}

template <int NT, int R, int U>
bool launch_gemv1_r(const int8_t* q, const float* s, const float* x, float* y, int I, int O, int ks, hipStream_t st) {
    const size_t lds = (NT > 2 ? (size_t)NT * I * 4 : 0) + (size_t)GV_WAVES * NT * R * 4;
    if (lds > 160 * 1024) return false;
    static bool once = [] {
        MOEX_CK(hipFuncSetAttribute(reinterpret_cast<const void*>(gemv1_kernel<NT, R, U>),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
        return true;
    }();
    (void)once;
    const int gpw = GV_WAVES / ks, wgs = ((O + R - 1) / R + gpw - 1) / gpw;
    hipLaunchKernelGGL((gemv1_kernel<NT, R, U>), dim3(wgs), dim3(64 * GV_WAVES), lds, st, q, s, x, y, I, O, ks);
    MOEX_LAUNCHED();
    return true;
}
template <int NT, int U>
bool launch_gemv1(const int8_t* q, const float* s, const float* x, float* y, int I, int O, int ks, int cus,
                  hipStream_t st) {
    // the rows per wavefront with the cheapest rounds over the chip: R rows and a fixed part of about two rows' time each.
    // Of 2, 3, 4, 6, 9 and 12 it was the fastest or within 12 % of it for 1 to 8 input rows on qkv (9) and o_proj (4).
    // Two loads a lane (16384 inputs) leave registers for 8 and pay for one round only, where the looped kernel has too few
    // workgroups (us, looped -> so, 1 / 2 input rows: 512 x 16384 7.7 / 11.5 -> 5.1 / 5.7, 2048 x 16384 13.3 / 17.1 -> 9.5 /
    // 10.9)
    int best = 0;
    long cost = 0;
    for (int R : {2, 3, 4, 6, U > 1 ? 8 : 9, 12}) {
        if (U > 1 && R > 8) break;
        const long gpw = GV_WAVES / ks, wgs = ((O + R - 1) / R + gpw - 1) / gpw, e = (wgs + cus - 1) / cus * (R + 2);
        if (!best || e < cost) {
            best = R;
            cost = e;
        }
    }
    if constexpr (U == 1) {
        switch (best) {
            case 6: return launch_gemv1_r<NT, 6, U>(q, s, x, y, I, O, ks, st);
            case 9: return launch_gemv1_r<NT, 9, U>(q, s, x, y, I, O, ks, st);
            case 12: return launch_gemv1_r<NT, 12, U>(q, s, x, y, I, O, ks, st);
        }
    }
    if constexpr (U == 2) {
        if (best == 6) return launch_gemv1_r<NT, 6, U>(q, s, x, y, I, O, ks, st);
        if (best == 8) return launch_gemv1_r<NT, 8, U>(q, s, x, y, I, O, ks, st);
    }
    switch (best) {
        case 2: return launch_gemv1_r<NT, 2, U>(q, s, x, y, I, O, ks, st);
        case 3: return launch_gemv1_r<NT, 3, U>(q, s, x, y, I, O, ks, st);
        default: return launch_gemv1_r<NT, 4, U>(q, s, x, y, I, O, ks, st);
    }
}

template <int NT>
void launch_gemv_t(const int8_t* q, const float* s, const float* x, float* y, int I, int O, hipStream_t st) {
    static bool once = [] {
        MOEX_CK(hipFuncSetAttribute(reinterpret_cast<const void*>(gemv_kernel<NT>),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
        return true;
    }();
    (void)once;
    const int groups = (O + GV_R - 1) / GV_R;
    // split each row over up to 8 wavefronts until 8 wavefronts per CU have 8 rows each, and where I allows it until a part
    // is one load a lane (I % 512 == 0, so the parts are equal). With longer parts left to the looped kernel, us, then -> now,
    // 1 / 2 / 4 / 8 input rows: 9216 x 1536 7.0 / 8.7 / 12.3 / 19.1 -> 4.7 / 5.5 / 7.1 / 10.0; 16384 x 2048 9.3 / 11.8 / 17.8 /
    // 27.5 -> 7.7 / 9.0 / 10.9 / 19.3; 12288 x 4096 13.8 / 18.4 / 28.3 / 44.1 -> 10.3 / 12.8 / 14.1 / 25.5
    int ks = 1;
    while (ks < GV_WAVES && ((groups * ks < 2048 && (I / 16) % (128 * ks) == 0) || (I <= 8192 && I / 16 / ks > 64))) ks *= 2;
    static const int cus = [] {
        int dev = 0, v = 0;
        if (hipGetDevice(&dev) == hipSuccess &&
            hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && v > 0)
            return v;
        return 256;
    }();
    if (I / 16 / ks <= 64 && launch_gemv1<NT, 1>(q, s, x, y, I, O, ks, cus, st)) return;
    // longer parts: two chunks a lane where one round of workgroups holds the matrix, else the looped kernel, with 4
    // wavefronts per CU (8: 4476 x 12288, 2 rows, 24.7 us, 4: 20.7)
    const bool two = I / 16 / ks <= 128 && (O + 7) / 8 <= cus * (GV_WAVES / ks);
    if constexpr (NT <= 2) {
        if (two && launch_gemv1<NT, 2>(q, s, x, y, I, O, ks, cus, st)) return;
    }
    if (I / 16 / ks > 64 && !two) {
        ks = 1;
        while (ks < GV_WAVES && groups * ks < 1024 && (I / 16) % (128 * ks) == 0) ks *= 2;
    }
    const int nb = std::min(cus, groups * ks);
    const size_t lds = (size_t)NT * I * 4 + GV_WAVES * NT * GV_R * 4;
    hipLaunchKernelGGL(gemv_kernel<NT>, dim3(nb), dim3(64 * GV_WAVES), lds, st, q, s, x, y, I, O, ks);
    MOEX_LAUNCHED();
}

// ---- int4 / int6 gs64 quantizers (quantize_rows_q4_k, quantize_rows_q6_k: kernels.cuh:552-590) ----
// A workgroup per row; each wavefront takes 64-weight groups g = w, w + 4, .., a lane per weight. Scale = group absmax
// / 7 (int4) or / 31 (int6), 1 for an all-zero group; codes round-half-even(w / scale) clamped to [-8, 7] /
// [-32, 31] (int6 stored + 32). Packing: weight i's nibble at bits 4 (i % 2) of byte i / 2 of the row's low plane
// (low nibble first); int6 adds its high 2 bits at bits 2 (i % 4) of byte i / 4 of the high plane. The lanes OR their
// fields together across 8 (nibbles) or 16 (2-bit fields) lanes and one lane writes the dword.
template <bool SIX>
__global__ void __launch_bounds__(256) quantize_gs64_kernel(const uint16_t* __restrict__ W, uint8_t* __restrict__ q,
                                                            uint8_t* __restrict__ qh, float* __restrict__ s, int I) {
    const size_t row = blockIdx.x;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, G = I / 64;
    const _Float16* wr = reinterpret_cast<const _Float16*>(W) + row * I;
    for (int g = wv; g < G; g += 4) {
        const float w = (float)wr[g * 64 + lane];
        float m = fabsf(w);
#pragma unroll
        for (int o = 32; o; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
        const float sc = m > 0.f ? m / (SIX ? 31.f : 7.f) : 1.f;
        uint32_t lo, hi = 0;
        if (SIX) {
            const uint32_t u = (uint32_t)((int)fminf(31.f, fmaxf(-32.f, __builtin_rintf(w / sc))) + 32);
            lo = (u & 15u) << (4 * (lane & 7));
            hi = (u >> 4) << (2 * (lane & 15));
        } else {
            const int v = max(-8, min(7, (int)__builtin_rintf(w / sc)));
            lo = ((uint32_t)v & 15u) << (4 * (lane & 7));
        }
#pragma unroll
        for (int o = 1; o < 8; o <<= 1) lo |= __shfl_xor(lo, o);
        if ((lane & 7) == 0) reinterpret_cast<uint32_t*>(q + row * (I / 2) + g * 32)[lane >> 3] = lo;
        if (SIX) {
#pragma unroll
            for (int o = 1; o < 16; o <<= 1) hi |= __shfl_xor(hi, o);
            if ((lane & 15) == 0) reinterpret_cast<uint32_t*>(qh + row * (I / 4) + g * 16)[lane >> 4] = hi;
        }
        if (lane == 0) s[row * G + g] = sc;
    }
}

// ---- GEMV of the int4 / int6 / fp16 forms (gemv_q4_k, gemv_q6_k, gemv_f16_k: kernels.cuh:68-93,486-550) ----
// y[t][o] = sum over the row's 16-weight units c of (sum_k w[o][16c + k] x[t][16c + k]) * scale[o][c / 4] (fp16: no
// scale), fp32 sums. Layout as gemv_kernel: a wavefront takes R rows over the KS-th part of the row's units, a lane
// per unit (8 B of int4, 8 + 4 B of int6, 32 B of fp16 a row), reads its 16 inputs per row of x from L2, sums the
// unit in k order, and the KS parts of a row are added in LDS in part order. KS and R depend on O, I and the form
// only, so every row of a multi-row call is bit-identical to the same row alone.
template <int FMT>
struct MatUnit {
    uint4 a[FMT == MF_F16 ? 2 : 1];  // int4 / int6: .x, .y the 16 low nibbles; fp16: 16 halves
    uint32_t h;                      // int6: the 16 high 2-bit fields
    float sc;
};
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
template <int FMT>
__device__ __forceinline__ void mat_unit_load(MatUnit<FMT>& u, const uint8_t* W, const uint8_t* Wh, const float* s,
                                              size_t row, int I, int c) {
    if constexpr (FMT == MF_F16) {
        const u32x4* p = reinterpret_cast<const u32x4*>(W + (row * I + 16 * (size_t)c) * 2);
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const u32x4 v = __builtin_nontemporal_load(p + i);
            u.a[i] = make_uint4(v[0], v[1], v[2], v[3]);
        }
    } else {
        const u32x2 v = __builtin_nontemporal_load(reinterpret_cast<const u32x2*>(W + row * (I / 2)) + c);
        u.a[0] = make_uint4(v[0], v[1], 0u, 0u);
        if constexpr (FMT == MF_Q6) u.h = __builtin_nontemporal_load(reinterpret_cast<const uint32_t*>(Wh + row * (I / 4)) + c);
        u.sc = s[row * (I / 64) + c / 4];
    }
}
// weight k of the unit, without its scale (k a constant after unrolling)
template <int FMT> __device__ __forceinline__ float mat_unit_weight(const MatUnit<FMT>& u, int k) {
    if constexpr (FMT == MF_F16) {
        const uint4& q = u.a[k / 8];
        const uint32_t d2 = ((k / 2) & 3) == 0 ? q.x : ((k / 2) & 3) == 1 ? q.y : ((k / 2) & 3) == 2 ? q.z : q.w;
        return (float)u2h2(d2)[k & 1];
    } else {
        const uint32_t dw = k < 8 ? u.a[0].x : u.a[0].y;
        if constexpr (FMT == MF_Q4) {
            return (float)(int)__builtin_amdgcn_sbfe(dw, 4 * (k & 7), 4);  // the signed nibble (the builtin returns it as unsigned)
        } else {
            const uint32_t hb = (u.h >> (2 * k)) & 3u;
            return (float)((int)(((dw >> (4 * (k & 7))) & 15u) | (hb << 4)) - 32);
        }
    }
}
template <int FMT>
__device__ __forceinline__ float mat_unit_dot(const MatUnit<FMT>& u, const float4 (&x)[4]) {
    float d = 0.f;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const float xv[4] = {x[j].x, x[j].y, x[j].z, x[j].w};
#pragma unroll
        for (int n = 0; n < 4; n++) d = fmaf(mat_unit_weight<FMT>(u, 4 * j + n), xv[n], d);
    }
    return FMT == MF_F16 ? d : d * u.sc;
}
constexpr int GM_WAVES = 8;
// (wavefronts a SIMD: 5 int6 rows in 4 took 130 registers left alone, 2 too many for 4 of them: 9814 x 1536 19.6 -> 16.2 us)
template <int FMT, int NT, int R>
__global__ void __launch_bounds__(64 * GM_WAVES, NT == 5 ? 4 : 2) gemv_mat_kernel(const uint8_t* __restrict__ W,
                                                                 const uint8_t* __restrict__ Wh,
                                                                 const float* __restrict__ s,
                                                                 const float* __restrict__ x, float* __restrict__ y,
                                                                 int I, int O, int KS) {
    __shared__ float red[GM_WAVES][NT][R];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, nb = gridDim.x;
    const int U = I / 16, ngroups = (O + R - 1) / R, gpr = GM_WAVES / KS;
    const int rounds = (ngroups + nb * gpr - 1) / (nb * gpr);
    const int part = wv % KS, slice = U / KS, cb = part * slice, ce = cb + slice;
    for (int j = 0; j < rounds; j++) {
        const int g = blockIdx.x + nb * (wv / KS + j * gpr);
        if (g < ngroups) {
            float acc[NT * R];
#pragma unroll
            for (int i = 0; i < NT * R; i++) acc[i] = 0.f;
            for (int c = cb + lane; c < ce; c += 64) {
                MatUnit<FMT> u[R];
#pragma unroll
                for (int r = 0; r < R; r++) mat_unit_load<FMT>(u[r], W, Wh, s, (size_t)min(g * R + r, O - 1), I, c);
#pragma unroll
                for (int t = 0; t < NT; t++) {
                    float4 xv[4];
                    const float4* xp = reinterpret_cast<const float4*>(x + (size_t)t * I + 16 * (size_t)c);
#pragma unroll
                    for (int i = 0; i < 4; i++) xv[i] = xp[i];
#pragma unroll
                    for (int r = 0; r < R; r++) acc[t * R + r] += mat_unit_dot<FMT>(u[r], xv);
                }
            }
            wave_sums(acc);
#pragma unroll
            for (int k = 0; k < ((NT * R + 1) / 2 + 1) / 2; k++) {
                const int i = wave_sums_index<NT * R>(k, lane >> 4);
                if ((lane & 15) == 0 && i < NT * R) red[wv][i / R][i % R] = acc[k];
            }
        }
        __syncthreads();
        if (g < ngroups && part == 0 && lane < NT * R) {
            const int t = lane / R, r = lane % R, o = g * R + r;
            float v = red[wv][t][r];
            for (int p = 1; p < KS; p++) v += red[wv + p][t][r];
            if (o < O) y[(size_t)t * O + o] = v;
        }
        __syncthreads();  // the partial sums are read before the next round writes them
    }
}

// The same product when a part of a row is at most 64 units (one load step a lane) and the input rows fit LDS: one row
// group a wavefront and no loop, so a workgroup's loads all go out at once and R follows from whole rounds of the chip.
// The input rows go into LDS once per workgroup by DMA, in gemv1_kernel's layout, instead of being read from L2 by every
// wavefront (8 rows of inputs are ten times the bytes of 4 int6 weight rows), and a unit is widened once per group of
// input rows. One int4 / int6 row's inputs are read straight from L2 (int4 qkv 5.0 against 5.3 us); beside the wider fp16
// weights LDS is better for one row too (8.8 against 10.1). Same sum order as gemv_mat_kernel, so a row's bits are those
// of its own call. Bound by the weight stream and the launch for one or two rows, by the widening and the FMAs for more.
// Graph-replayed over rotating weights, us, before -> now (before: gemv_mat_kernel; int4 and fp16 row by row):
//   input rows               1           2            3           4           6            8
//   int6 qkv 9216 x 2048     7.1 -> 6.1  9.4 -> 8.1   11.1 -> 7.5 13.1 -> 9.1 23.7 -> 10.5 27.6 -> 11.8
//   int6 o   2048 x 4096     4.7 -> 4.6  5.4 -> 5.0   7.0 -> 5.3  7.9 -> 5.7  11.1 -> 6.4  12.4 -> 7.1
//   int4 qkv, o              6.0 -> 5.0, 4.0 -> 3.8   12.1 -> 6.3, 7.7 -> 4.2
//   fp16 qkv, o              10.5 -> 8.8, 6.6 -> 5.5  21.0 -> 9.3, 12.9 -> 6.1
template <int FMT, int NT> constexpr bool mat_xl = NT > 1 || FMT == MF_F16;  // input rows through LDS
template <int FMT, int NT, int R>
__global__ void __launch_bounds__(64 * GM_WAVES, 2) gemv_mat_x_kernel(const uint8_t* __restrict__ W,
                                                                      const uint8_t* __restrict__ Wh,
                                                                      const float* __restrict__ s,
                                                                      const float* __restrict__ x, float* __restrict__ y,
                                                                      int I, int O, int KS) {
    constexpr bool XL = mat_xl<FMT, NT>;
    extern __shared__ __align__(16) float xs[];  // XL: the input rows [NT][I]; then the partial sums [GM_WAVES][NT * R]
    float* red = xs + (XL ? NT * I : 0);
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int gpw = GM_WAVES / KS, part = wv % KS, slice = I / 16 / KS;
    const int g = blockIdx.x * gpw + wv / KS;
    const bool on = lane < slice;
    const int c = min(part * slice + lane, I / 16 - 1);
    constexpr int TB = NT <= 4 ? NT : (NT + 1) / 2;  // input rows whose values fit the registers
    float4 xv[TB][4];
    if constexpr (XL) {
        const int n = NT * I / 256;  // 1 KB transfers
        for (int i = wv; i < n; i += GM_WAVES) {
            const uint32_t e = 64 * i + lane;
            dma16x(x, 16 * (e ^ ((e >> 3) & 3)), reinterpret_cast<const unsigned char*>(xs) + 1024 * i);
        }
    } else {
#pragma unroll
        for (int d = 0; d < 4; d++) xv[0][d] = reinterpret_cast<const float4*>(x)[4 * c + d];
    }
    MatUnit<FMT> u[R];
#pragma unroll
    for (int r = 0; r < R; r++) mat_unit_load<FMT>(u[r], W, Wh, s, (size_t)min(g * R + r, O - 1), I, c);
    if constexpr (XL) asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");  // the products need both anyway
    float acc[NT * R];
#pragma unroll
    for (int t0 = 0; t0 < NT; t0 += TB) {
        if constexpr (XL) {
#pragma unroll
            for (int t = t0; t < NT && t < t0 + TB; t++)
#pragma unroll
                for (int d = 0; d < 4; d++) {
                    const uint32_t e = t * (I / 4) + 4 * c + d;
                    xv[t - t0][d] = reinterpret_cast<const float4*>(xs)[e ^ ((e >> 3) & 3)];
                }
        }
#pragma unroll
        for (int r = 0; r < R; r++) {
            float a[TB];
#pragma unroll
            for (int t = 0; t < TB; t++) a[t] = 0.f;
#pragma unroll
            for (int d = 0; d < 4; d++) {
                float w[4];
#pragma unroll
                for (int i = 0; i < 4; i++) w[i] = mat_unit_weight<FMT>(u[r], 4 * d + i);
#pragma unroll
                for (int t = 0; t < TB && t0 + t < NT; t++) {
                    a[t] = fmaf(w[0], xv[t][d].x, a[t]);
                    a[t] = fmaf(w[1], xv[t][d].y, a[t]);
                    a[t] = fmaf(w[2], xv[t][d].z, a[t]);
                    a[t] = fmaf(w[3], xv[t][d].w, a[t]);
                }
            }
#pragma unroll
            for (int t = 0; t < TB && t0 + t < NT; t++)
                acc[(t0 + t) * R + r] = on ? 0.f + (FMT == MF_F16 ? a[t] : a[t] * u[r].sc) : 0.f;  // no -0
        }
        if constexpr (NT > TB) asm volatile("" ::: "memory");  // the next group's values are read after these are used
    }
    wave_sums(acc);
#pragma unroll
    for (int k = 0; k < ((NT * R + 1) / 2 + 1) / 2; k++) {
        const int i = wave_sums_index<NT * R>(k, lane >> 4);
        if ((lane & 15) == 0 && i < NT * R) red[wv * NT * R + i] = acc[k];
    }
    __syncthreads();
    const int rows = gpw * R;  // of this workgroup
    for (int e = tid; e < NT * rows; e += 64 * GM_WAVES) {
        const int t = e / rows, rr = e % rows, gl = rr / R, r = rr % R, o = (blockIdx.x * gpw + gl) * R + r;
        if (o >= O) continue;
        float v = red[gl * KS * NT * R + t * R + r];
        for (int p = 1; p < KS; p++) v += red[(gl * KS + p) * NT * R + t * R + r];
        y[(size_t)t * O + o] = v;
    }
}

int dense_cus() {
    static const int cus = [] {
        int dev = 0, v = 0;
        if (hipGetDevice(&dev) == hipSuccess &&
            hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && v > 0)
            return v;
        return 256;
    }();
    return cus;
}

template <int FMT, int NT, int R>
void launch_gemv_mat_x(const uint8_t* W, const uint8_t* Wh, const float* s, const float* x, float* y, int I, int O, int ks,
                       size_t lds, hipStream_t st) {
    static bool once = [] {
        MOEX_CK(hipFuncSetAttribute(reinterpret_cast<const void*>(gemv_mat_x_kernel<FMT, NT, R>),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
        return true;
    }();
    (void)once;
    const int gpw = GM_WAVES / ks, wgs = ((O + R - 1) / R + gpw - 1) / gpw;
    hipLaunchKernelGGL((gemv_mat_x_kernel<FMT, NT, R>), dim3(wgs), dim3(64 * GM_WAVES), lds, st, W, Wh, s, x, y, I, O, ks);
    MOEX_LAUNCHED();
}

template <int FMT, int NT>
void launch_gemv_mat_t(const uint8_t* W, const uint8_t* Wh, const float* s, const float* x, float* y, int I, int O,
                       hipStream_t st) {
    // parts of at least 64 units (one load step a lane wherever I allows: a second, dependent step cost the qkv
    // shape 8.4 -> 6.4 us for int4); rows per wavefront: 4, fewer while the grid would leave CUs without a
    // workgroup; up to two workgroups per CU at once before the kernel loops over further rounds
    const int U = I / 16, cus = dense_cus();
    int ks = 1;
    while (ks < GM_WAVES && U % (2 * ks) == 0 && U / (2 * ks) >= 64) ks *= 2;
    const int gpr = GM_WAVES / ks;
    {
        // the rows per wavefront with the cheapest rounds over the chip, as launch_gemv1: of 2, 3, 4 and 6 the fastest or
        // within 6 % of it for 1 to 8 input rows on qkv (3) and o_proj (4). The transfers are of 16 bytes a lane and 1 KB
        // each: input rows of another alignment or length take the kernel below
        constexpr bool XL = mat_xl<FMT, NT>;
        const size_t lds = (XL ? (size_t)NT * I * 4 : 0) + (size_t)GM_WAVES * NT * 4 * 6;
        // (one fp16 row of a matrix that leaves half the chip idle gains nothing from LDS either, and pays for the
        // copy: 579 x 2048 3.75 us, 3.50 without)
        const bool few = FMT == MF_F16 && NT == 1 && 2 * (((O + 1) / 2 + gpr - 1) / gpr) <= cus;
        if (U / ks <= 64 && lds <= 160 * 1024 && !few &&
            (!XL || (I % 256 == 0 && (reinterpret_cast<uintptr_t>(x) & 15) == 0))) {
            int best = 0;
            long cost = 0;
            for (int R : {2, 3, 4, 6}) {
                const long wgs = ((O + R - 1) / R + gpr - 1) / gpr, e = (wgs + cus - 1) / cus * (R + 2);
                if (!best || e < cost) {
                    best = R;
                    cost = e;
                }
            }
            switch (best) {
                case 2: launch_gemv_mat_x<FMT, NT, 2>(W, Wh, s, x, y, I, O, ks, lds, st); break;
                case 3: launch_gemv_mat_x<FMT, NT, 3>(W, Wh, s, x, y, I, O, ks, lds, st); break;
                case 4: launch_gemv_mat_x<FMT, NT, 4>(W, Wh, s, x, y, I, O, ks, lds, st); break;
                default: launch_gemv_mat_x<FMT, NT, 6>(W, Wh, s, x, y, I, O, ks, lds, st); break;
            }
            return;
        }
    }
    int R = 4;
    while (R > 1 && ((O + R - 1) / R + gpr - 1) / gpr < cus) R /= 2;
    const int nb = std::min(2 * cus, ((O + R - 1) / R + gpr - 1) / gpr);
    if (R == 4)
        hipLaunchKernelGGL((gemv_mat_kernel<FMT, NT, 4>), dim3(nb), dim3(64 * GM_WAVES), 0, st, W, Wh, s, x, y, I, O, ks);
    else if (R == 2)
        hipLaunchKernelGGL((gemv_mat_kernel<FMT, NT, 2>), dim3(nb), dim3(64 * GM_WAVES), 0, st, W, Wh, s, x, y, I, O, ks);
    else
        hipLaunchKernelGGL((gemv_mat_kernel<FMT, NT, 1>), dim3(nb), dim3(64 * GM_WAVES), 0, st, W, Wh, s, x, y, I, O, ks);
    MOEX_LAUNCHED();
}

// ---- the GEMM's choice of tile ----
// A call runs ceil(tiles / CUs) rounds of one tile per CU (the smallest tiles share a CU, at the same cost), and us0 +
// us1 * I / 1024 is a tile's time, fitted to every tile at 9 to 2048 tokens on the qkv and o_proj shapes, int8 and int4
// (int6 is within 35 %, tile against tile closer; fp16 weights cost the fp32-reading tiles 15 % more than the XH ones:
// o_proj at 1300 tokens 58 us with 128 x 128 against 48 with 128 x 128 XH, int8 49 against 54). The XH tiles' rounding
// launch costs 8 us + 1 us per million activations, so they pay where a call runs several rounds or the tile is large
// (o_proj at 3000 tokens, int8: 95 -> 80). The tile with the smallest
// estimate runs: at 12 token counts from 12 to 900 on both shapes and forms it was the fastest or within 5 %, and 3 % off the
// fastest in the mean over 100 other matrices of 64 to 2048 inputs, which us0 of 128 x 128 XH, 32 x 32 and 32 x 16 was set by. The 48
// token tiles fill the chip where those of 32 and 64 leave a part of it or a round short (int8 / int4, us, with the best
// of the others against them): qkv at 40 tokens 13.0 / 14.4 -> 12.3 / 12.2, at 100 20.2 / 20.8 -> 17.3 / 20.3; o_proj
// at 300 21.9 / 25.2 -> 21.3 / 21.2, at 600 33.7 / 37.0 -> 26.8 / 33.9. 112 x 128 was never the best by more than 1 %.
// 128 x 96 runs where it fills the chip in one round only (`one`): o_proj of 1025 to 1536 tokens, which 128 x 128 tiles leave
// half idle (int8 / fp16, us, with the best of the others against it: 1100 tokens 53 / 49 -> 44 / 45, 1500 49 / 50 ->
// 46 / 47; 9216 x 3072, 288 tokens, 44 / 41 -> 35 / 37); over several rounds 128 x 128 was up to 15 % faster.
struct GemmCost { int BM, BN; bool xh; int BK; float us0, us1; bool split, one; };
using GemmA = GemmTile<9, 4, 2, 4, 1, 2, 1, true>;  // 288 x 256
using GemmB = GemmTile<9, 2, 1, 8, 1, 2, 1, true>;  // 144 x 256
using GemmC = GemmTile<9, 2, 1, 4, 2, 1, 2>;        // 144 x 128
using GemmD = GemmTile<4, 2, 2, 4, 1, 2, 3>;        // 128 x 128
using GemmE = GemmTile<4, 2, 2, 4, 1, 2, 2, true>;  // 128 x 128
using GemmF = GemmTile<4, 2, 2, 2, 2, 1, 3>;        // 128 x 64
using GemmG = GemmTile<4, 2, 1, 2, 4, 1, 2>;        // 64 x 64
using GemmH = GemmTile<4, 2, 1, 1, 8, 1, 2>;        // 64 x 32
using GemmI = GemmTile<2, 2, 1, 1, 8, 1, 1, false, 4>;       // 32 x 32
using GemmJ = GemmTile<2, 1, 1, 1, 8, 1, 2, false, 4>;       // 32 x 16
using GemmK = GemmTile<1, 1, 1, 1, 8, 1, 2, false, 4>;       // 16 x 16
using GemmL = GemmTile<4, 3, 2, 1, 4, 1, 2>;        // 128 x 48
using GemmM = GemmTile<2, 3, 2, 1, 4, 1, 2>;        // 64 x 48
using GemmN = GemmTile<4, 3, 2, 2, 2, 2, 2, true>;  // 128 x 96
// the tiles that are built with a K split too
template <class C>
constexpr bool gemm_splits = std::is_same_v<C, GemmE> || std::is_same_v<C, GemmF> || std::is_same_v<C, GemmH> ||
                             std::is_same_v<C, GemmI> || std::is_same_v<C, GemmK> || std::is_same_v<C, GemmG>;
template <class C> constexpr GemmCost gemm_cost(float us0, float us1, bool one = false) {
    return {C::BM, C::BN, C::XH, C::BK, us0, us1, gemm_splits<C>, one};
}
constexpr GemmCost GEMM_COST[] = {
    gemm_cost<GemmA>(10.f, 33.f),   gemm_cost<GemmB>(8.f, 20.7f),   gemm_cost<GemmC>(6.f, 16.6f), gemm_cost<GemmD>(6.6f, 11.f),
    gemm_cost<GemmE>(3.f, 8.8f),    gemm_cost<GemmF>(5.6f, 7.37f),  gemm_cost<GemmG>(3.6f, 4.87f), gemm_cost<GemmH>(4.4f, 2.71f),
    gemm_cost<GemmI>(1.1f, 2.42f),  gemm_cost<GemmJ>(.7f, 1.94f),   gemm_cost<GemmK>(1.f, 1.44f), gemm_cost<GemmL>(6.f, 5.61f),
    gemm_cost<GemmM>(2.f, 4.02f),   gemm_cost<GemmN>(7.f, 7.2f, true)};

// nks parts of K (at most: no empty one is left) where the tile has a split instance
template <int FMT, class C, bool SPLIT>
int launch_gemm_s(const void* W, const uint8_t* Wh, const float* s, const void* X, float* Y, int S, int I, int O, int nks,
                  hipStream_t st) {
    static bool once = [] {
        MOEX_CK(hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_tile_kernel<FMT, C, SPLIT>),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
        return true;
    }();
    (void)once;
    const int tiles = ((O + C::BM - 1) / C::BM) * ((S + C::BN - 1) / C::BN);
    const int ns = (I + C::BK - 1) / C::BK, spp = (ns + nks - 1) / nks, parts = (ns + spp - 1) / spp;
    hipLaunchKernelGGL((gemm_tile_kernel<FMT, C, SPLIT>), dim3(tiles, parts), dim3(512), C::LDS, st, W, Wh, s, X, Y, S, I, O,
                       spp);
    MOEX_LAUNCHED();
    return parts;
}
template <int FMT, class C>
void launch_gemm_t(const void* W, const uint8_t* Wh, const float* s, const void* X, float* Y, int S, int I, int O,
                   hipStream_t st, int& nks) {
    if constexpr (gemm_splits<C>) {
        if (nks > 1) {
            nks = launch_gemm_s<FMT, C, true>(W, Wh, s, X, Y, S, I, O, nks, st);
            return;
        }
    }
    launch_gemm_s<FMT, C, false>(W, Wh, s, X, Y, S, I, O, 1, st);
}

// A long K and few tiles: K of more than 4096 inputs (so not the attention's shapes) is split over nks workgroups a tile, parts
// of 2048 inputs at least, where the shorter tiles save more than the second launch (4 us) and the parts' traffic cost, and 5 %. us, whole K in one
// workgroup -> split, int8 / fp16: 64 x 40448, 9 tokens 57 / 54 -> 13 / 12; 128 x 16384, 100 tokens 24 / 24 -> 12 / 12;
// 2048 x 16384, 300 tokens 68 / 80 -> 47 / 62, 1100 tokens 179 / 194 -> 121 / 126; 1024 x 8192, 17 tokens 14 / 14 -> 11 / 11.
// With parts of 4096 at least, 4936 x 10240 with 100 tokens took 51 / 54 (40 / 44 so), 64 x 6144 with 11 11 / 11 (7 / 8), 1920 x 10240
// with 300 48 / 54 (37 / 41).
struct GemmPick { int tile, nks; };
GemmPick gemm_pick(int S, int I, int O, bool xh, bool split, bool f16) {
    const int cus = dense_cus();
    GemmPick best = {-1, 1};
    float us = 0.f;
    for (int c = 0; c < (int)(sizeof(GEMM_COST) / sizeof(GEMM_COST[0])); c++) {
        const GemmCost& t = GEMM_COST[c];
        if (t.xh && (!xh || I % t.BK != 0)) continue;  // whole K steps only
        // a tile's offsets stay within 32 bits (the smallest tile's are 64-bit)
        if (t.BM * t.BN > 256 && (size_t)std::max(t.BM, t.BN) * I * 4 >= (size_t)1 << 32) continue;
        const size_t tiles = (size_t)((O + t.BM - 1) / t.BM) * ((S + t.BN - 1) / t.BN);
        if (t.one && tiles > (size_t)cus) continue;
        for (int nks = 1; nks == 1 || (split && t.split && I > 4096 && nks <= I / 2048 && tiles * nks <= (size_t)2 * cus); nks++) {
            float e = (float)((tiles * nks + cus - 1) / cus) * (t.us0 + t.us1 * (float)I * (1.f / 1024.f) / (float)nks) *
                          (f16 && !t.xh ? 1.15f : 1.f) + (t.xh ? 8.f + 1e-6f * (float)S * (float)I : 0.f);
            if (nks > 1) e = 1.05f * e + 4.f + 2e-6f * (float)nks * (float)S * (float)O;
            if (best.tile < 0 || e < us) {
                best = {c, nks};
                us = e;
            }
        }
    }
    return best;
}

template <int FMT>
void launch_gemm(const void* W, const uint8_t* Wh, const float* s, const float* X, float* Y, int S, int I, int O,
                 hipStream_t st) {
    // quiet: while a workspace cannot be had (a capture before an eager call of this size, or no memory) the best tile that
    // needs none runs: one that rounds the activations itself, over the whole of K
    const size_t n4 = (size_t)S * I / 4;
    uint2* Xh = nullptr;
    float* part = nullptr;
    GemmPick p;
    for (bool xh = true, split = true;;) {
        p = gemm_pick(S, I, O, xh, split, FMT == MF_F16);
        if (p.nks > 1 && !(part = reinterpret_cast<float*>(stream_workspace((size_t)p.nks * S * O * 4, st, 3, true)))) split = false;
        else if (GEMM_COST[p.tile].xh && !(Xh = reinterpret_cast<uint2*>(stream_workspace(n4 * 8, st, 2, true)))) xh = false;
        else break;
    }
    const void* Xg = X;
    if (GEMM_COST[p.tile].xh) {
        hipLaunchKernelGGL(round_f16_kernel, dim3((unsigned)std::min<size_t>((n4 + 255) / 256, 4096)), dim3(256), 0, st,
                           reinterpret_cast<const float4*>(X), Xh, n4);
        MOEX_LAUNCHED();
        Xg = Xh;
    }
    float* const out = Y;
    if (p.nks > 1) Y = part;
    switch (p.tile) {
        case 0: launch_gemm_t<FMT, GemmA>(W, Wh, s, Xg, Y, S, I, O, st, p.nks); break;
        case 1: launch_gemm_t<FMT, GemmB>(W, Wh, s, Xg, Y, S, I, O, st, p.nks); break;
        case 2: launch_gemm_t<FMT, GemmC>(W, Wh, s, Xg, Y, S, I, O, st, p.nks); break;
        case 3: launch_gemm_t<FMT, GemmD>(W, Wh, s, Xg, Y, S, I, O, st, p.nks); break;
        case 4: launch_gemm_t<FMT, GemmE>(W, Wh, s, Xg, Y, S, I, O, st, p.nks); break;
        case 5: launch_gemm_t<FMT, GemmF>(W, Wh, s, Xg, Y, S, I, O, st, p.nks); break;
        case 6: launch_gemm_t<FMT, GemmG>(W, Wh, s, Xg, Y, S, I, O, st, p.nks); break;
        case 7: launch_gemm_t<FMT, GemmH>(W, Wh, s, Xg, Y, S, I, O, st, p.nks); break;
        case 8: launch_gemm_t<FMT, GemmI>(W, Wh, s, Xg, Y, S, I, O, st, p.nks); break;
        case 9: launch_gemm_t<FMT, GemmJ>(W, Wh, s, Xg, Y, S, I, O, st, p.nks); break;
        case 10: launch_gemm_t<FMT, GemmK>(W, Wh, s, Xg, Y, S, I, O, st, p.nks); break;
        case 11: launch_gemm_t<FMT, GemmL>(W, Wh, s, Xg, Y, S, I, O, st, p.nks); break;
        case 12: launch_gemm_t<FMT, GemmM>(W, Wh, s, Xg, Y, S, I, O, st, p.nks); break;
        default: launch_gemm_t<FMT, GemmN>(W, Wh, s, Xg, Y, S, I, O, st, p.nks); break;
    }
    if (p.nks > 1) {
        const size_t n = (size_t)S * O;
        hipLaunchKernelGGL(gemm_reduce_kernel, dim3((unsigned)std::min<size_t>((n + 255) / 256, 2048)), dim3(256), 0, st, part,
                           FMT == MF_I8 ? s : nullptr, out, n, O, p.nks);
        MOEX_LAUNCHED();
    }
}

}  // namespace

void launch_quantize_rows_i8(const uint16_t* W, int8_t* q, float* s, int O, int I, hipStream_t st) {
    hipLaunchKernelGGL(quantize_rows_kernel, dim3(O), dim3(256), 0, st, W, q, s, I);
    MOEX_LAUNCHED();
}

void launch_gemv_i8(const int8_t* q, const float* s, const float* x, float* y, int NT, int I, int O, hipStream_t st) {
    switch (NT) {
        case 1: launch_gemv_t<1>(q, s, x, y, I, O, st); break;
        case 2: launch_gemv_t<2>(q, s, x, y, I, O, st); break;
        case 3: launch_gemv_t<3>(q, s, x, y, I, O, st); break;
        case 4: launch_gemv_t<4>(q, s, x, y, I, O, st); break;
        case 5: launch_gemv_t<5>(q, s, x, y, I, O, st); break;
        case 6: launch_gemv_t<6>(q, s, x, y, I, O, st); break;
        case 7: launch_gemv_t<7>(q, s, x, y, I, O, st); break;
        default: launch_gemv_t<8>(q, s, x, y, I, O, st); break;
    }
}

void launch_quantize_rows_gs64(const uint16_t* W, uint8_t* q, uint8_t* qh, float* s, int O, int I, bool six,
                               hipStream_t st) {
    if (six) hipLaunchKernelGGL(quantize_gs64_kernel<true>, dim3(O), dim3(256), 0, st, W, q, qh, s, I);
    else hipLaunchKernelGGL(quantize_gs64_kernel<false>, dim3(O), dim3(256), 0, st, W, q, qh, s, I);
    MOEX_LAUNCHED();
}

void launch_gemv_mat(const moex_mat& m, const float* x, float* y, int NT, int I, int O, hipStream_t st) {
    if (m.q4) {
        if (NT == 2) launch_gemv_mat_t<MF_Q4, 2>(m.q4, nullptr, m.s, x, y, I, O, st);  // the rows' own bits, one pass
        else launch_gemv_mat_t<MF_Q4, 1>(m.q4, nullptr, m.s, x, y, I, O, st);
    } else if (m.q6) {
        switch (NT) {
            case 1: launch_gemv_mat_t<MF_Q6, 1>(m.q6, m.q6h, m.s, x, y, I, O, st); break;
            case 2: launch_gemv_mat_t<MF_Q6, 2>(m.q6, m.q6h, m.s, x, y, I, O, st); break;
            case 3: launch_gemv_mat_t<MF_Q6, 3>(m.q6, m.q6h, m.s, x, y, I, O, st); break;
            case 4: launch_gemv_mat_t<MF_Q6, 4>(m.q6, m.q6h, m.s, x, y, I, O, st); break;
            case 5: launch_gemv_mat_t<MF_Q6, 5>(m.q6, m.q6h, m.s, x, y, I, O, st); break;
            case 6: launch_gemv_mat_t<MF_Q6, 6>(m.q6, m.q6h, m.s, x, y, I, O, st); break;
            case 7: launch_gemv_mat_t<MF_Q6, 7>(m.q6, m.q6h, m.s, x, y, I, O, st); break;
            default: launch_gemv_mat_t<MF_Q6, 8>(m.q6, m.q6h, m.s, x, y, I, O, st); break;
        }
    } else {
        const uint8_t* W = reinterpret_cast<const uint8_t*>(m.f16);
        if (NT == 2) launch_gemv_mat_t<MF_F16, 2>(W, nullptr, nullptr, x, y, I, O, st);
        else launch_gemv_mat_t<MF_F16, 1>(W, nullptr, nullptr, x, y, I, O, st);
    }
}

void launch_gemm_i8(const int8_t* q, const float* s, const float* X, float* Y, int S, int I, int O, hipStream_t st) {
    launch_gemm<MF_I8>(q, nullptr, s, X, Y, S, I, O, st);
}

void launch_gemm_mat(const moex_mat& m, const float* X, float* Y, int S, int I, int O, hipStream_t st) {
    if (m.q4) launch_gemm<MF_Q4>(m.q4, nullptr, m.s, X, Y, S, I, O, st);
    else if (m.q6) launch_gemm<MF_Q6>(m.q6, m.q6h, m.s, X, Y, S, I, O, st);
    else launch_gemm<MF_F16>(m.f16, nullptr, nullptr, X, Y, S, I, O, st);
}

}  // namespace moex
