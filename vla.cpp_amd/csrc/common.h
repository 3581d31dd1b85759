// Shared device helpers for the gfx950 kernels: bf16 bit conversions, vector
// types, wavefront (64-lane) reductions and the MFMA fragment typedefs.
#pragma once
#include "vla_kernels.h"

#include <hip/hip_runtime.h>
#include <stdint.h>

#define VLA_WAVE 64

#if defined(__HIP_DEVICE_COMPILE__) && !defined(__gfx950__)
#error "these kernels are written for gfx950 (MI355X) only"
#endif

namespace vk {

// Overrides of the by-shape kernel selection, for tests and tuning.  Read from the
// environment once (vla_kernels_init, or the first launch that asks) and again only by
// vla_kernels_reload_env: no launch path calls getenv.
struct Tuning {
    int attn_dl = -1;           // VLA_ATTN_DL: 0 pins the register-staged LDS kernel for 64- and 128-wide bf16 heads
    int attn_slices = 0;        // VLA_ATTN_SLICES: 1 | 2 key slices per row tile in the direct-to-LDS kernel
    int attn_split = -1;        // VLA_ATTN_SPLIT: key slices across workgroups (<= 0 pins one)
    bool attn_split_set = false;
    bool attn_part_f32 = false;  // VLA_ATTN_PART_F32: the tiled kernel, with fp32 partials where fp16 would be used
    bool attn_no_arrive = false; // VLA_ATTN_NO_ARRIVE: no in-launch merge by the last slice to arrive
    bool attn_no_direct = false; // VLA_ATTN_NO_DIRECT: never the register-direct kernel
    bool attn_no_stream = false; // VLA_ATTN_NO_STREAM: never the streaming (LDS-ring) form of the register-direct kernel
    int gemm_rows_max = 512;     // VLA_GEMM_ROWS_MAX: projections of at most this many rows may take the narrow-tile kernels, 0 = never
    int gemm_rows_plan = 0;      // VLA_GEMM_ROWS_PLAN: 1..4 pins those kernels' rows x columns per workgroup (16x16, 32x16, 64x16, 64x32; fp32: 1 and 3), 0 = by shape
    bool attn_no_small = false;  // VLA_ATTN_NO_SMALL: fp32 launches with few row tiles do not split their keys beyond the usual rule
    int attn_rows = -1;          // VLA_ATTN_ROWS: 0 never, 1 always (as far as they serve the shape) the kernels of a wavefront per key block for 48- and 64-wide heads and per 64-key unit for 256-wide bf16 ones; unset = by shape
    int attn_direct_rows = 32;   // VLA_ATTN_DIRECT_ROWS: row limit of the register-direct kernel
    int gemm_tile = -1;          // VLA_GEMM_TILE: 0..5, wide tiles 16..21, plain products also 22..24
    int gemm_panel = 0;          // VLA_GEMM_PANEL: N tiles per panel of an XCD's walk over its tiles; 0 = by size
    int gemm_dl = -1;            // VLA_GEMM_DL: 0 pins the register-staged GEMM
    int gemm_stages = 0;         // VLA_GEMM_STAGES: ring depth of the direct-to-LDS GEMM
    int ternary_tile = 0;        // VLA_TERNARY_TILE: 64 | 128 | 256 (32x32x32 kernels) | 16 (128 x 256) | 17 (128 x 128) | 18 (64 x 128) | 19 (64 x 64) | 20 (64 x 256) | 21 (32 x 64) (16x16x64 kernels)
};
const Tuning& tuning();

// Scratch memory the library owns on behalf of entry points whose signature has no
// workspace argument: one block per (purpose, device, stream), grown on demand and never
// freed before the process ends, so a captured graph that holds an older block keeps
// pointing at live memory and calls on different streams never share a block.  New blocks
// are zero-filled.  Allocates (never under stream capture: run a shape once before
// capturing it).  Returns nullptr when the allocation fails.
enum { SCRATCH_ATTN = 0, SCRATCH_ROWSUM = 1 };
void* stream_scratch(int purpose, hipStream_t stream, size_t bytes);

typedef uint16_t bf16_t;  // raw bf16 bits

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef int i32x4_t __attribute__((ext_vector_type(4)));
typedef int i32x16_t __attribute__((ext_vector_type(16)));
typedef uint16_t u16x4_t __attribute__((ext_vector_type(4)));
typedef uint16_t u16x8_t __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

// bf16 <-> f32, round to nearest even, NaN quieted: the hardware converter (v_cvt_pk_bf16_f32),
// one instruction where the integer formulation takes seven.
__device__ __forceinline__ float bf2f(bf16_t h) { return __uint_as_float(((uint32_t)h) << 16); }
__device__ __forceinline__ bf16_t f2bf(float f) { return __builtin_bit_cast(bf16_t, (__bf16)f); }
// Two floats -> packed bf16 pair with the hardware converter (v_cvt_pk_bf16_f32,
// round to nearest even).
typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pack_bf2(float lo, float hi) {
    const f32x2_t v = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));
}

// Element traits: storage type <-> float.
template <typename T> struct Elem;
template <> struct Elem<float> {
    static constexpr int kVec = 4;  // elements per 16-byte vector
    __device__ static __forceinline__ float load(const float* p) { return *p; }
    __device__ static __forceinline__ void store(float* p, float v) { *p = v; }
    __device__ static __forceinline__ float round(float v) { return v; }  // the value a store and a load would give back
};
template <> struct Elem<bf16_t> {
    static constexpr int kVec = 8;
    __device__ static __forceinline__ float load(const bf16_t* p) { return bf2f(*p); }
    __device__ static __forceinline__ void store(bf16_t* p, float v) { *p = f2bf(v); }
    __device__ static __forceinline__ float round(float v) { return bf2f(f2bf(v)); }
};

// 64-lane wavefront reductions; every lane ends with the result.  No trip through LDS (a
// ds_bpermute butterfly costs six dependent LDS round trips, which is most of the time of a
// kernel that is one wavefront's chain of dependent steps): inside a row of 16 lanes the
// partners come from DPP operands (neighbour, neighbour pair, the mirrored half, the
// mirrored row), the four rows are combined by gfx950's row swaps (v_permlane16_swap of a
// register with itself leaves rows (0, 0, 2, 2) in one copy and (1, 1, 3, 3) in the other;
// v_permlane32_swap does the same for the halves).  Both partners of a step form the same
// sum of the same two values, so every lane ends with the same bits.
template <int CTRL>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, false);
}
constexpr int DPP_XOR1 = 0xB1, DPP_XOR2 = 0x4E, DPP_HALF_MIRROR = 0x141, DPP_ROW_MIRROR = 0x140;
template <typename Op>
__device__ __forceinline__ uint32_t wave_combine_u32(uint32_t v, Op op) {
    v = op(v, dpp_u32<DPP_XOR1>(v));
    v = op(v, dpp_u32<DPP_XOR2>(v));
    v = op(v, dpp_u32<DPP_HALF_MIRROR>(v));
    v = op(v, dpp_u32<DPP_ROW_MIRROR>(v));
    u32x2_t r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    v = op(r[0], r[1]);
    r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    return op(r[0], r[1]);
}
__device__ __forceinline__ float wave_max(float v) {
    return __uint_as_float(wave_combine_u32(__float_as_uint(v), [](uint32_t a, uint32_t b) {
        return __float_as_uint(fmaxf(__uint_as_float(a), __uint_as_float(b)));
    }));
}
__device__ __forceinline__ float wave_sum(float v) {
    return __uint_as_float(wave_combine_u32(__float_as_uint(v), [](uint32_t a, uint32_t b) {
        return __float_as_uint(__uint_as_float(a) + __uint_as_float(b));
    }));
}
__device__ __forceinline__ int wave_sum_i(int v) {
    return (int)wave_combine_u32((uint32_t)v, [](uint32_t a, uint32_t b) { return a + b; });
}

// A value combined over the two halves of the wavefront (lanes r and r + 32): one row swap
// instead of a trip through LDS.
__device__ __forceinline__ float halves_max(float x) {
    const u32x2_t r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float halves_sum(float x) {
    const u32x2_t r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// A value combined over the four 16-lane rows of the wavefront (lanes c, c + 16, c + 32, c + 48)
// with gfx950's row swaps instead of two trips through LDS: after v_permlane16_swap of a register
// with itself one copy holds rows (0, 0, 2, 2) and the other rows (1, 1, 3, 3); v_permlane32_swap does
// the same for the two halves.
__device__ __forceinline__ float rows_max(float x) {
    u32x2_t r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
    r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float rows_sum(float x) {
    u32x2_t r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Block reductions through LDS for blocks of up to 16 wavefronts.  `red` holds
// at least 16 floats.  All threads of the block must call.
__device__ __forceinline__ float block_max(float v, float* red) {
    v = wave_max(v);
    const int w = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[w] = v;
    __syncthreads();
    float r = red[0];
    for (int i = 1; i < nw; ++i) r = fmaxf(r, red[i]);
    return r;
}
__device__ __forceinline__ float block_sum(float v, float* red) {
    v = wave_sum(v);
    const int w = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[w] = v;
    __syncthreads();
    float r = 0.f;
    for (int i = 0; i < nw; ++i) r += red[i];
    return r;
}

// One bf16 row through RMSNorm and the per-row int8 quantisation of the BitNet activations,
// by one wavefront (bitvla_rmsnorm_bf16 then act_quant, src/kernels/bitnet_kernels.h:49-54,
// without the round trip): lane L holds the 16-byte vectors L, L + 64, ... of the row, NV of
// them.  y = x * rsqrt(mean(x^2) + eps) * w is rounded to bf16 as it would be stored; the
// scale is 127 / max(amax, 1e-5); q = clamp(round-half-even(y * scale)).  The int8 row goes
// to qrow (global or LDS, 8 bytes per vector); scale and the sum of the row's int8 values
// are returned in every lane.  K % 8 == 0 and K <= 512 NV.
// GLU: the row is formed on the fly from a fused projection, x[k] = bf16(relu(gate[k])^2 * up[k])
// with gate = xr and up = xr + K (gate_up_fused_sqrelu_mul_bf16, src/kernels/bitvla/bitvla_lm_cuda.cu:525-548).
// WAVES > 1: the row is shared by the WAVES wavefronts of a workgroup (`lane` = the thread's
// index in it, vectors lane, lane + 64 WAVES, ...; `red` = 16 floats of LDS for the three
// reductions; every thread of the workgroup calls).  The squares are then added in another
// order than by one wavefront, so the two forms agree to rounding, not bit for bit.
// (Loads, weights and rounding under a branch per vector and word: a launch of the decode projections, 2560-wide rows, 0.65 us longer.)
// Two loads per vector and no other branch than the stores': addresses past the row are clamped and the values replaced by zeros
// (which change neither sums nor maxima), a missing or unaligned weight is read or made up once, in front of the arithmetic.
template <int NV, bool GLU = false, int WAVES = 1>
__device__ __forceinline__ void rms_act_quant_row(const bf16_t* __restrict__ xr, const bf16_t* __restrict__ w, int K,
                                                  float eps, int lane, int8_t* qrow, float& scale_out, int& sum_out,
                                                  float* red = nullptr) {
    constexpr int LS = 64 * WAVES;  // vectors per pass over the row
    const int nvec = K / 8;
    // Every value kept between the passes is a bf16 (the input, then the rounded normalised
    // row), so the row stays packed: 4 registers per 16-byte vector.
    u32x4_t xp[NV], up[GLU ? NV : 1];
    u32x4_t wv[NV];  // the weight's vectors, requested with the row's so that one round trip covers both
    auto lo = [](uint32_t u) { return __uint_as_float(u << 16); };
    auto hi = [](uint32_t u) { return __uint_as_float(u & 0xffff0000u); };
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const long k0 = (long)min(lane + LS * i, nvec - 1) * 8;
        xp[i] = *reinterpret_cast<const u32x4_t*>(xr + k0);
        if (GLU) up[i] = *reinterpret_cast<const u32x4_t*>(xr + K + k0);
    }
    if (w && !((uintptr_t)w & 15)) {  // uniform
#pragma unroll
        for (int i = 0; i < NV; ++i) wv[i] = *reinterpret_cast<const u32x4_t*>(w + (long)min(lane + LS * i, nvec - 1) * 8);
    } else {
#pragma unroll
        for (int i = 0; i < NV; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const bf16_t* we = w ? w + (long)min(lane + LS * i, nvec - 1) * 8 + 2 * e : nullptr;
                wv[i][e] = we ? (uint32_t)we[0] | ((uint32_t)we[1] << 16) : 0x3f803f80u;  // none: ones
            }
    }
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const bool in = lane + LS * i < nvec;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (GLU) {
                float g0 = lo(xp[i][e]), g1 = hi(xp[i][e]);
                if (g0 < 0.f) g0 = 0.f;
                if (g1 < 0.f) g1 = 0.f;
                xp[i][e] = pack_bf2(g0 * g0 * lo(up[i][e]), g1 * g1 * hi(up[i][e]));
            }
            xp[i][e] = in ? xp[i][e] : 0u;
            const float a = lo(xp[i][e]), b = hi(xp[i][e]);
            ss += a * a;
            ss += b * b;
        }
    }
    const float inv = 1.0f / sqrtf((WAVES > 1 ? block_sum(ss, red) : wave_sum(ss)) / (float)K + eps);
    // the packed words are opaque from here on, or the compiler keeps the first pass's unpacked
    // floats alive across the reduction (8 registers per vector instead of 4)
#pragma unroll
    for (int i = 0; i < NV; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) asm volatile("" : "+v"(xp[i][e]));
    float amax = 0.f;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const bool in = lane + LS * i < nvec;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float o0 = lo(xp[i][e]) * inv * lo(wv[i][e]), o1 = hi(xp[i][e]) * inv * hi(wv[i][e]);
            const uint32_t pr = in ? pack_bf2(o0, o1) : 0u;  // the activation as the bf16 it would be stored as (0 x inv may be NaN past the row)
            xp[i][e] = pr;
            amax = fmaxf(amax, fmaxf(fabsf(lo(pr)), fabsf(hi(pr))));
        }
    }
    amax = WAVES > 1 ? block_max(amax, red) : wave_max(amax);
    if (amax < 1e-5f) amax = 1e-5f;
    const float scale = 127.0f / amax;
#pragma unroll
    for (int i = 0; i < NV; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) asm volatile("" : "+v"(xp[i][e]));
    int sum = 0;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        // Clamped, then rounded to the nearest even integer by adding 1.5 x 2^23, whose ulp is 1: the low byte of the sum's bits is
        // the integer's (rounding first gives the same, the bounds being integers; NaN becomes -128 as before).
        uint32_t t[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const uint32_t u = xp[i][e >> 1];
            const float qf = fminf(fmaxf(((e & 1) ? hi(u) : lo(u)) * scale, -128.0f), 127.0f);
            t[e] = __float_as_uint(qf + 12582912.0f);
        }
        uint32_t pk[2];
#pragma unroll
        for (int h = 0; h < 2; ++h)  // bytes 0 of four words
            pk[h] = __builtin_amdgcn_perm(t[4 * h + 1], t[4 * h], 0x0c0c0400u) | (__builtin_amdgcn_perm(t[4 * h + 3], t[4 * h + 2], 0x0c0c0400u) << 16);
        sum = __builtin_amdgcn_sdot4((int)pk[0], 0x01010101, sum, false);  // + the four signed bytes
        sum = __builtin_amdgcn_sdot4((int)pk[1], 0x01010101, sum, false);
        if (lane + LS * i < nvec) *reinterpret_cast<u32x2_t*>(qrow + (long)(lane + LS * i) * 8) = u32x2_t{pk[0], pk[1]};
    }
    scale_out = scale;
    sum = wave_sum_i(sum);
    if (WAVES > 1) {  // exact in any order
        int* redi = reinterpret_cast<int*>(red);
        __syncthreads();
        if ((lane & 63) == 0) redi[lane >> 6] = sum;
        __syncthreads();
        sum = 0;
        for (int i = 0; i < WAVES; ++i) sum += redi[i];
    }
    sum_out = sum;
}

// ggml_silu / ggml_gelu (tanh form) / ggml_relu, fp32 (src/layers/ffn.h:24-40, src/modules/action_expert.cpp:41-59).
__device__ __forceinline__ float apply_act(float x, int act) {
    if (act == VLA_ACT_SILU) return x / (1.0f + __expf(-x));
    if (act == VLA_ACT_GELU) return 0.5f * x * (1.0f + tanhf(0.79788456080286535588f * x * (1.0f + 0.044715f * x * x)));
    if (act == VLA_ACT_RELU) return x > 0.f ? x : 0.f;
    return x;
}

// x / (1 + e) in seven instructions, correctly rounded: the hardware reciprocal (1 ulp), the quotient, and one step on its exact
// remainder.  On 2^24 values from -87 to 30 and over all exponents the bits of the division (which is some 15 instructions), but for
// |x| < 2^-124, where it is the nearest denormal or the one beside it.  A quarter of both sides, so that the reciprocal is a
// normal number up to e = 2^128; v_div_fixup puts right what infinities make of the remainder.
__device__ __forceinline__ float div_1p(float x, float e) {
    const float d = fmaf(e, 0.25f, 0.25f), n = 0.25f * x, r = __builtin_amdgcn_rcpf(d), q = n * r;
    return __builtin_amdgcn_div_fixupf(fmaf(fmaf(-d, q, n), r, q), d, n);
}
// The same for values that are rounded to bf16 next, N at a time.  The exact division and tanhf above are some 25 and 45
// instructions per value, and a 128 x 128 tile has 64 per thread: 12 of the 65 us that 1323 x 6144 x 1536 with GELU took on such
// tiles (on the wide tiles now 30.9 us, 28.3 without an activation).  Here 9 and 11: GELU's tanh form is written as the sigmoid
// it is, 0.5 x (1 + tanh u) = x / (1 + exp(-2 u)).  SiLU has the bits of the exact form.  GELU against float64, 4 M values of N(0, 1):
// 4.2e-8 of the norm (tanhf 3.8e-8; N(0, 0.3^2) 4.0e-8, tanhf 4.2e-8), largest error 1.6e-6 of the value (tanhf 0.35, where 1 + tanh u
// cancels); rounded to bf16 both are 1.665157630e-3 of the norm, and 29 values are not the nearest (tanhf 111).
// The multiply-add is spelled out: every kernel gives the same bits.
template <int N>
__device__ __forceinline__ void apply_act_bf16(float (&v)[N], int act) {
    if (act == VLA_ACT_SILU) {
#pragma unroll
        for (int e = 0; e < N; ++e) v[e] = div_1p(v[e], __builtin_amdgcn_exp2f(v[e] * -1.44269504088896341f));
    } else if (act == VLA_ACT_GELU) {
        constexpr float k1 = -2.0f * 0.79788456080286535588f * 1.44269504088896341f, k3 = k1 * 0.044715f;
#pragma unroll
        for (int e = 0; e < N; ++e) v[e] = div_1p(v[e], __builtin_amdgcn_exp2f(v[e] * fmaf(k3, v[e] * v[e], k1)));
    } else if (act == VLA_ACT_RELU) {
#pragma unroll
        for (int e = 0; e < N; ++e) v[e] = v[e] > 0.f ? v[e] : 0.f;
    }
}

// s_waitcnt on the vector-memory counter alone (vmcnt[3:0] in bits 3:0, vmcnt[5:4] in bits
// 15:14; the export and LDS/scalar counter fields at their maxima, i.e. not waited on).
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
    static_assert(N >= 0 && N <= 63, "vmcnt is a 6-bit counter");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}
// Division by a launch-wide constant without the divider sequence (some thirty dependent instructions per quotient, in
// front of a kernel's first load): the host forms 2^32 / d + 1 once, the quotient of any x < 2^16 is then the high half
// of one multiplication (exact while d < 2^16).  mg == 0 keeps the plain division (d or the dividends out of range).
struct DivC {
    unsigned d, mg;
};
inline DivC make_divc(long d, long max_x) {
    DivC c;
    c.d = (unsigned)d;
    c.mg = (d > 1 && d < 65536 && max_x < 65536) ? (unsigned)((1ull << 32) / (unsigned long long)d) + 1u : 0u;
    return c;
}
__device__ __forceinline__ unsigned div_c(unsigned x, DivC c) { return c.mg ? __umulhi(x, c.mg) : (c.d == 1 ? x : x / c.d); }

// One 16-byte load per lane from global memory straight into LDS, no register in between:
// lane i's bytes land at lds_base + 16 i (lds_base wavefront-uniform, held in M0); the
// per-lane global address is free.  Completion is tracked by vmcnt like any vector load.
// Issued from inline assembly so that the wait counts stay under this file's control.
// The ISA asks for one wait state between a scalar write of M0 and the LDS load that reads it; the compiler puts none inside
// an asm statement, hence the s_nop in each of these.
__device__ __forceinline__ void load_to_lds16(const void* gptr, uint32_t lds_base) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds_base), "v"(gptr) : "memory");
}
// One 16-byte load per lane from uniform base + 32-bit lane offset straight into LDS (see load_to_lds16).
__device__ __forceinline__ void load_to_lds16_at(const void* base, uint32_t off, uint32_t lds_base) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_base), "v"(off), "s"(base) : "memory");
}
// The same to lds_base + plus (a constant): no scalar register per destination.
__device__ __forceinline__ void load_to_lds16_plus(const void* base, uint32_t off, uint32_t lds_base, int plus) {
    asm volatile("s_add_u32 m0, %0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_base), "v"(off), "s"(base), "i"(plus) : "memory", "scc");
}
// The same if c (uniform), without a branch that the compiler sees.
__device__ __forceinline__ void load_to_lds16_plus_if(bool c, const void* base, uint32_t off, uint32_t lds_base, int plus) {
    asm volatile("s_cmp_eq_u32 %4, 0\n\ts_cbranch_scc1 skip%=\n\ts_add_u32 m0, %0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\nskip%=:" ::"s"(lds_base), "v"(off), "s"(base), "i"(plus), "s"(__builtin_amdgcn_readfirstlane(c ? 1 : 0)) : "memory", "scc");
}

}  // namespace vk
