// What the projection kernels share: the argument block, the workgroup -> tile walk, the mapping of
// 64-column tiles to rows of W, and the epilogues' arithmetic.
#pragma once

#include "common.h"
#include "tile_rules.h"
#include "vla_kernels.h"

namespace vk {

constexpr int BN = 64;                     // epilogue sub-tile; column-tile unit of the N mapping
constexpr int C_STRIDE = BN + 4;           // floats

enum { EPI_PLAIN = 0, EPI_QKV = 1, EPI_TERNARY = 2, EPI_GLU = 3 };
enum { NORM_NONE = 0, NORM_RMS = 1, NORM_LAYER = 2, NORM_LAYER_PRE = 3 };  // row statistics taken inside gemm_dl_kernel (PRE: LayerNorm from sums handed over by the producing launch)
constexpr int STAT_MAX_TILES = 24;  // 64-column tiles of a row whose sums a consumer adds up (four threads per row, six pairs each)

struct GemmArgs {
    // Field order: what the single-token decode projections read (a chain of short launches, each waiting for its
    // arguments' cache lines before anything else) sits in the first two 64-byte lines of the block, the rotation
    // tables in the third; the tiled kernels' walk constants and epilogue extras follow.
    const void* A;
    const void* W;
    const float* bias;
    int M, N, K, n_tiles;
    // TERNARY (part): weight scales; row statistics of A taken inside the launch (see norm_eps below)
    int ws_num;
    // Row statistics of A taken inside the GEMM (direct-to-LDS kernel, kNorm): RMS when
    // colsum is null, else LayerNorm with colsum[n] = sum_k W[n][k] (fp32 [N])
    float norm_eps;
    const float* ws;
    const void* norm_w;  // ternary GEMV with the RMSNorm and quantisation of its rows inside: A is bf16, this the norm weight
    // PLAIN, GLU
    const void* residual;
    void* Y;
    int out_bf16;
    int act;  // VLA_ACT_*: PLAIN applies it after the bias, GLU to the gate
    // QKV
    void* q_out;
    void* k_cache;
    void* vt_cache;
    int t_max, tok_offset, Hkv, D;
    const float* cos_t;
    const float* sin_t;
    int S, Hq, nk, nv;
    int xm, xn;
    int pn;  // N tiles per panel of an XCD's walk (see xcd_tile)
    const float* col_gate;  // PLAIN: fp32 [N] factor on the projection before the residual is added, or null
    // TERNARY
    int32_t* acc_out;
    const float* s;
    const int32_t* rowsum;
    const float* colsum;
    // Row statistics handed from the launch that writes a row to the launch that normalises it: a PLAIN
    // launch with bf16 output leaves (sum of squares, sum) of the 64 values it wrote per (row, 64-column
    // tile) in stats_out [M][N / 64][2]; a QKV launch with the LayerNorm inside adds up the n_stat pairs
    // of a row from stats_in instead of summing the row from its operand tiles.
    float* stats_out;
    const float* stats_in;
    int n_stat;
    // The tile walk's constants (see xcd_tile), formed once on the host (xcd_split) so that a workgroup finds its tile
    // with a few multiplications: every division by a run-time value costs a wavefront some thirty dependent scalar
    // instructions in front of its first load.  cn, cm: tiles per XCD column / row; per_panel = pn cm; full = cn / pn
    // whole panels; w_last = cn - full pn; mg_*: 2^32 / d + 1 for d = cn, per_panel, pn, w_last (x / d = mulhi(x, mg)
    // for x < 2^16); xn_shift = log2 xn.
    int cn, cm, per_panel, full, w_last, xn_shift;
    unsigned mg_cn, mg_pp, mg_pn, mg_wl;
    DivC div_s;  // QKV, wide tiles: rows per observation
};

// Workgroup -> tile.  Workgroup i runs on XCD i % 8; the XCDs form an xm x xn grid over the
// tile grid and XCD (xr, xc) owns the tiles (m, n) with m % xm == xr, n % xn == xc.  Its
// workgroups walk them panel by panel: pn of its N tiles at a time, every M tile of the XCD
// against that panel before the next panel starts, so that the panel's rows of W stay in the
// XCD's L2 while the rows of A stream past them once per panel.  (With all of W in one
// panel and W larger than the L2, W would stream again for every few M tiles instead.)
__device__ __forceinline__ unsigned div_magic(unsigned x, unsigned d, unsigned mg) { return d == 1 ? x : __umulhi(x, mg); }
__device__ __forceinline__ bool xcd_tile(const GemmArgs& a, int n_wg_tiles, int m_wg_tiles, int& mtw, int& ntw) {
    const unsigned xcd = blockIdx.x & 7, local = blockIdx.x >> 3;  // local < 2^16 (checked where the grid is sized)
    unsigned ml, nl;
    if (a.pn >= a.cn) {
        ml = div_magic(local, a.cn, a.mg_cn);
        nl = local - ml * a.cn;
    } else {
        unsigned p = div_magic(local, a.per_panel, a.mg_pp), rem = local - p * a.per_panel, w = a.pn, mg = a.mg_pn;
        if (p >= (unsigned)a.full) {  // the last, narrower panel
            p = a.full;
            rem = local - a.full * a.per_panel;
            w = a.w_last;
            mg = a.mg_wl;
        }
        ml = div_magic(rem, w, mg);
        nl = p * a.pn + rem - ml * w;
    }
    ntw = (int)(nl * a.xn + (xcd & (a.xn - 1)));
    mtw = (int)(ml * a.xm + (xcd >> a.xn_shift));
    return ntw < n_wg_tiles && mtw < m_wg_tiles;
}

// W-row bases of the two 32-column halves of output tile `nt`.
struct TileCols {
    int base0, base1;  // rows of W feeding tile columns [0,32) and [32,64)
    int seg;           // 0 Q, 1 K, 2 V (QKV mode)
    int col0, col1;    // segment-local column of tile column 0 and of tile column 32
    bool rope;
};

template <int kEpi>
__device__ __forceinline__ TileCols tile_cols(const GemmArgs& a, int nt) {
    TileCols t;
    if (kEpi == EPI_GLU) {  // W = [gate rows; up rows]: the tile pairs 32 gate columns with their up columns
        t.base0 = nt * 32;
        t.base1 = a.N / 2 + nt * 32;
        t.seg = 0;
        t.col0 = t.base0;
        t.col1 = t.base1;
        t.rope = false;
        return t;
    }
    if (kEpi != EPI_QKV) {
        t.base0 = nt * BN;
        t.base1 = t.base0 + 32;
        t.seg = 0;
        t.col0 = t.base0;
        t.col1 = t.base1;
        t.rope = false;
        return t;
    }
    const int tq = a.Hq * a.D / BN, tk = a.nk * a.D / BN;
    int lt = nt, seg_base = 0;
    t.seg = 0;
    if (nt >= tq + tk) {
        t.seg = 2;
        lt = nt - tq - tk;
        seg_base = (a.Hq + a.nk) * a.D;
    } else if (nt >= tq) {
        t.seg = 1;
        lt = nt - tq;
        seg_base = a.Hq * a.D;
    }
    t.rope = (a.cos_t != nullptr) && t.seg != 2;
    if (t.rope) {
        const int tph = a.D / BN;  // tiles per head
        const int head = lt / tph, chunk = lt % tph;
        t.col0 = head * a.D + chunk * 32;
        t.col1 = t.col0 + a.D / 2;
    } else {
        t.col0 = lt * BN;
        t.col1 = t.col0 + 32;
    }
    t.base0 = seg_base + t.col0;
    t.base1 = seg_base + t.col1;
    return t;
}

// Rows of W of a narrow tile's 16 columns: 8 + 8 (see gemm_narrow_kernel).
struct RowCols {
    int base_lo, base_hi;  // rows of W of tile columns [0, 8) and [8, 16)
    int seg;               // 0 Q, 1 K, 2 V (QKV mode)
    int col_lo, col_hi;    // segment-local column of tile column 0 and of tile column 8
    bool rope;
};
template <int kEpi>
__device__ __forceinline__ RowCols row_cols(const GemmArgs& a, int t) {
    RowCols rc;
    rc.seg = 0;
    rc.rope = false;
    if (kEpi == EPI_GLU) {
        rc.base_lo = rc.col_lo = t * 8;
        rc.base_hi = rc.col_hi = a.N / 2 + t * 8;
        return rc;
    }
    if (kEpi != EPI_QKV) {
        rc.base_lo = rc.col_lo = t * 16;
        rc.base_hi = rc.col_hi = t * 16 + 8;
        return rc;
    }
    const int tq = a.Hq * a.D / 16, tk = a.nk * a.D / 16;
    int lt = t, seg_base = 0;
    if (t >= tq + tk) {
        rc.seg = 2;
        lt = t - tq - tk;
        seg_base = (a.Hq + a.nk) * a.D;
    } else if (t >= tq) {
        rc.seg = 1;
        lt = t - tq;
        seg_base = a.Hq * a.D;
    }
    rc.rope = (a.cos_t != nullptr) && rc.seg != 2;
    if (rc.rope) {
        const int tph = a.D / 16;  // tiles per head
        const int head = lt / tph, chunk = lt % tph;
        rc.col_lo = head * a.D + chunk * 8;
        rc.col_hi = rc.col_lo + a.D / 2;
    } else {
        rc.col_lo = lt * 16;
        rc.col_hi = rc.col_lo + 8;
    }
    rc.base_lo = seg_base + rc.col_lo;
    rc.base_hi = seg_base + rc.col_hi;
    return rc;
}

// The last min(nkt, LEFT) tiles of the ring: with LEFT tiles in flight, the oldest has landed
// when at most (LEFT - 1) NLOAD loads are still due.
template <int LEFT, int NLOAD, typename Body>
__device__ __forceinline__ void narrow_tail(int nkt, Body body) {
    if (LEFT <= nkt) {  // uniform
        wait_vmcnt<(LEFT - 1) * NLOAD>();
        body(LEFT == 1);
    }
    if constexpr (LEFT > 1) narrow_tail<LEFT - 1, NLOAD>(nkt, body);
}

// acc + lo^2 + hi^2 of the two bf16 values packed in u (taken by value: a bit_cast applied
// directly to a vector element expression reads element 0).
__device__ __forceinline__ float add_squares_bf16x2(uint32_t u, float acc) {
    const bf16x2_t v = __builtin_bit_cast(bf16x2_t, u);
    return __builtin_amdgcn_fdot2_f32_bf16(v, v, acc, false);
}
// acc + lo + hi
__device__ __forceinline__ float add_pair_bf16x2(uint32_t u, float acc) {
    const bf16x2_t v = __builtin_bit_cast(bf16x2_t, u);
    const bf16x2_t ones = __builtin_bit_cast(bf16x2_t, 0x3f803f80u);
    return __builtin_amdgcn_fdot2_f32_bf16(v, ones, acc, false);
}

// Epilogue arithmetic that several kernels share to the bit: the fused multiply-adds are spelled
// out, so that no kernel contracts the other product of a sum.
__device__ __forceinline__ void rotate_pair(float& x0, float& x1, float c, float s) {  // NeoX rotation of (x0, x1)
    const float a = x0, b = x1;
    x0 = fmaf(a, c, -(b * s));
    x1 = fmaf(b, c, a * s);
}
// rstd acc - (mean rstd) colsum: the projection of the centred and scaled row
__device__ __forceinline__ float center_scale(float acc, float rstd, float mean_rstd, float colsum) { return fmaf(acc, rstd, -(mean_rstd * colsum)); }

// The activation of a projection's outputs; fp32 outputs keep the exact forms.
template <int N>
__device__ __forceinline__ void epilogue_act(float (&v)[N], int act, int out_bf16) {
    if (out_bf16) {
        apply_act_bf16(v, act);
    } else {
#pragma unroll
        for (int e = 0; e < N; ++e) v[e] = apply_act(v[e], act);
    }
}

__device__ const float kNoBiasRegs[16] = {};
// Epilogue of 16 values of one row of a 64-column sub-tile: columns jg .. jg + 7 (lo) and 32 + jg .. 32 + jg + 7 (hi), the
// row's norm already applied.  The four threads of a row are neighbouring lanes in launches that leave row sums.
// BIAS_REGS: the bias of the 16 columns was fetched by the caller.
template <typename T, int kEpi, bool BIAS_REGS = false>
__device__ __forceinline__ void epilogue_16(const GemmArgs& a, int m, int nt, const TileCols& tc, int jg, float (&lo)[8], float (&hi)[8],
                                            bool have_res, u32x4_t res_lo, u32x4_t res_hi, const float (&bias_regs)[16]) {
    if (kEpi == EPI_GLU) {
        // lo = gate columns nt*32 + jg .. +7, hi = the up columns of the same outputs
        const int I = a.N / 2, n0 = nt * 32 + jg;  // I is a multiple of 32: the 8 outputs are inside the row
        float (&v)[8] = lo;
        if (a.bias) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                lo[e] += BIAS_REGS ? bias_regs[e] : a.bias[n0 + e];
                hi[e] += BIAS_REGS ? bias_regs[8 + e] : a.bias[I + n0 + e];
            }
        }
        epilogue_act(v, a.act, a.out_bf16);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] *= hi[e];
        const long o = (long)m * I + n0;
        if (a.out_bf16) {
            const u32x4_t pk = {pack_bf2(v[0], v[1]), pack_bf2(v[2], v[3]), pack_bf2(v[4], v[5]), pack_bf2(v[6], v[7])};
            *reinterpret_cast<u32x4_t*>((bf16_t*)a.Y + o) = pk;
        } else {
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const f32x4_t pk = {v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]};
                *reinterpret_cast<f32x4_t*>((float*)a.Y + o + 4 * q) = pk;
            }
        }
        return;
    }

    if (kEpi == EPI_PLAIN) {
        float st1 = 0.f, st2 = 0.f;  // sum and sum of squares of the 16 values this thread writes (as written: rounded to bf16)
#pragma unroll
        for (int hlf = 0; hlf < 2; ++hlf) {
            const int n0 = nt * BN + hlf * 32 + jg;
            if (n0 >= a.N) continue;
            float (&v)[8] = hlf ? hi : lo;
            const long o = (long)m * a.N + n0;
            const bool full = (n0 + 8 <= a.N) && (a.N % 8 == 0);
            // per-column operands: indices clamped into the row instead of a branch per element
            // (columns past N are never stored), so the eight loads are in flight together
            if (a.bias) {
                // BIAS_REGS: this thread's 2 x 8 values, fetched by the caller ahead of the epilogue
                float bv[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) bv[e] = BIAS_REGS ? bias_regs[hlf * 8 + e] : a.bias[min(n0 + e, a.N - 1)];
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] += bv[e];
            }
            if (a.act != VLA_ACT_NONE) epilogue_act(v, a.act, a.out_bf16);
            if (a.col_gate) {
                float gv[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) gv[e] = a.col_gate[min(n0 + e, a.N - 1)];
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] *= gv[e];
            }
            if (full && a.out_bf16) {  // 8 consecutive bf16 = one 16-byte access each way
                if (a.residual) {
                    // res_lo / res_hi: this thread's two residual vectors when fetched before the k loop
                    u32x4_t rr = hlf ? res_hi : res_lo;
                    if (!have_res) rr = *reinterpret_cast<const u32x4_t*>((const bf16_t*)a.residual + o);
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        v[2 * e] += __uint_as_float(rr[e] << 16);
                        v[2 * e + 1] += __uint_as_float(rr[e] & 0xffff0000u);
                    }
                }
                const u32x4_t pk = {pack_bf2(v[0], v[1]), pack_bf2(v[2], v[3]), pack_bf2(v[4], v[5]), pack_bf2(v[6], v[7])};
                *reinterpret_cast<u32x4_t*>((bf16_t*)a.Y + o) = pk;
                if (a.stats_out) {  // two bf16 values per instruction, exact products, fp32 sums
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        st1 = add_pair_bf16x2(pk[e], st1);
                        st2 = add_squares_bf16x2(pk[e], st2);
                    }
                }
            } else if (full) {
                if (a.residual) {
#pragma unroll
                    for (int q = 0; q < 2; ++q) {
                        const f32x4_t rr = *reinterpret_cast<const f32x4_t*>((const float*)a.residual + o + 4 * q);
#pragma unroll
                        for (int e = 0; e < 4; ++e) v[4 * q + e] += rr[e];
                    }
                }
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    const f32x4_t pk = {v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]};
                    *reinterpret_cast<f32x4_t*>((float*)a.Y + o + 4 * q) = pk;
                }
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    if (n0 + e >= a.N) continue;
                    float x = v[e];
                    if (a.out_bf16) {
                        if (a.residual) x += bf2f(((const bf16_t*)a.residual)[o + e]);
                        ((bf16_t*)a.Y)[o + e] = f2bf(x);
                    } else {
                        if (a.residual) x += ((const float*)a.residual)[o + e];
                        ((float*)a.Y)[o + e] = x;
                    }
                }
            }
        }
        if (a.stats_out) {
            // the four threads of a row are neighbouring lanes: the row's 64 values of this tile
            st1 += __uint_as_float(dpp_u32<DPP_XOR1>(__float_as_uint(st1)));
            st2 += __uint_as_float(dpp_u32<DPP_XOR1>(__float_as_uint(st2)));
            st1 += __uint_as_float(dpp_u32<DPP_XOR2>(__float_as_uint(st1)));
            st2 += __uint_as_float(dpp_u32<DPP_XOR2>(__float_as_uint(st2)));
            if (jg == 0) *reinterpret_cast<f32x2_t*>(a.stats_out + ((long)m * (a.N / BN) + nt) * 2) = f32x2_t{st2, st1};
        }
        return;
    }

    // QKV: bias, rotation, scatter.
    const int b = m / a.S, s = m % a.S;
    if (a.bias) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            lo[e] += BIAS_REGS ? bias_regs[e] : a.bias[tc.base0 + jg + e];
            hi[e] += BIAS_REGS ? bias_regs[8 + e] : a.bias[tc.base1 + jg + e];
        }
    }
    if (tc.rope) {
        const int half = a.D >> 1;
        const int p0 = (tc.col0 % a.D) + jg;  // pair index inside the head
        const float* cr = a.cos_t + (long)s * half + p0;
        const float* sr = a.sin_t + (long)s * half + p0;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float c = cr[e], sn = sr[e];
            rotate_pair(lo[e], hi[e], c, sn);
        }
    }
    const bool is_bf16 = (sizeof(T) == 2);
#pragma unroll
    for (int hlf = 0; hlf < 2; ++hlf) {
        const float* v = hlf ? hi : lo;
        const int col = (hlf ? tc.col1 : tc.col0) + jg;  // segment-local, 8 consecutive columns
        if (tc.seg == 0) {
            const long o = (long)m * (a.Hq * a.D) + col;
            if (is_bf16) {
                u32x4_t pk = {pack_bf2(v[0], v[1]), pack_bf2(v[2], v[3]), pack_bf2(v[4], v[5]), pack_bf2(v[6], v[7])};
                *reinterpret_cast<u32x4_t*>((bf16_t*)a.q_out + o) = pk;
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) ((float*)a.q_out)[o + e] = v[e];
            }
        } else if (tc.seg == 1) {
            const int head = col / a.D, d0 = col % a.D;
            const long o = (((long)b * a.Hkv + head) * a.t_max + a.tok_offset + s) * a.D + d0;
            if (is_bf16) {
                u32x4_t pk = {pack_bf2(v[0], v[1]), pack_bf2(v[2], v[3]), pack_bf2(v[4], v[5]), pack_bf2(v[6], v[7])};
                *reinterpret_cast<u32x4_t*>((bf16_t*)a.k_cache + o) = pk;
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) ((float*)a.k_cache)[o + e] = v[e];
            }
        } else {
            const int head = col / a.D, d0 = col % a.D;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const long o = (((long)b * a.Hkv + head) * a.D + d0 + e) * a.t_max + a.tok_offset + s;
                if (is_bf16) ((bf16_t*)a.vt_cache)[o] = f2bf(v[e]);
                else ((float*)a.vt_cache)[o] = v[e];
            }
        }
    }
}

// Epilogue of one 64x64 sub-tile held in the LDS C tile: thread t owns row t/4 and
// columns jg..jg+7 and 32+jg..32+jg+7 of the sub-tile.
template <typename T, int kEpi, bool BIAS_REGS = false>
__device__ __forceinline__ void epilogue_64x64(const GemmArgs& a, const uint32_t* C, int m0, int nt, const TileCols& tc,
                                               int tid, bool have_res = false, u32x4_t res_lo = u32x4_t{0u, 0u, 0u, 0u},
                                               u32x4_t res_hi = u32x4_t{0u, 0u, 0u, 0u}, int norm_mode = 0,
                                               const float* row_stat = nullptr, int stat_stride = 0,
                                               const float (&bias_regs)[16] = kNoBiasRegs) {
    const int erow = tid >> 2, jg = (tid & 3) * 8;
    const int m = m0 + erow;
    if (m >= a.M) return;
    const uint32_t* crow = C + erow * C_STRIDE;

    if (kEpi == EPI_TERNARY) {
        const int rs2 = 2 * a.rowsum[m];
        const float sm = a.s ? a.s[m] : 1.f;
        const int group = a.N / a.ws_num;
#pragma unroll
        for (int hlf = 0; hlf < 2; ++hlf)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int n = nt * BN + hlf * 32 + jg + e;
                if (n >= a.N) continue;
                const int v = (int)crow[hlf * 32 + jg + e] - rs2;
                if (a.acc_out) a.acc_out[(long)m * a.N + n] = v;
                if (a.Y) {
                    bf16_t o = f2bf((float)v / sm * a.ws[n / group]);
                    if (a.residual) o = f2bf(bf2f(o) + bf2f(((const bf16_t*)a.residual)[(long)m * a.N + n]));
                    ((bf16_t*)a.Y)[(long)m * a.N + n] = o;
                }
            }
        return;
    }

    float lo[8], hi[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        lo[e] = __uint_as_float(crow[jg + e]);
        hi[e] = __uint_as_float(crow[32 + jg + e]);
    }
    if (norm_mode) {
        // row_stat: per row of the sub-tile (sum of squares, sum) of the A row, as two partial
        // pairs stat_stride floats apart (one from each of the two wavefronts sharing the row)
        const float inv_k = 1.0f / (float)a.K;
        const float sq = row_stat[2 * erow] + row_stat[stat_stride + 2 * erow];
        if (norm_mode == NORM_LAYER && kEpi == EPI_QKV) {
            // sum_k (x - mean) rstd W[n][k] = rstd acc - (mean rstd) colsum[n]
            const float mean = (row_stat[2 * erow + 1] + row_stat[stat_stride + 2 * erow + 1]) * inv_k;
            const float f = rsqrtf(fmaxf(sq * inv_k - mean * mean, 0.f) + a.norm_eps);
            const float ms = mean * f;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                lo[e] = center_scale(lo[e], f, ms, a.colsum[tc.base0 + jg + e]);
                hi[e] = center_scale(hi[e], f, ms, a.colsum[tc.base1 + jg + e]);
            }
        } else {
            const float f = rsqrtf(sq * inv_k + a.norm_eps);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                lo[e] *= f;
                hi[e] *= f;
            }
        }
    }
    epilogue_16<T, kEpi, BIAS_REGS>(a, m, nt, tc, jg, lo, hi, have_res, res_lo, res_hi, bias_regs);
}

// The walk constants of xcd_tile for the XCD grid and panel width already in a; returns the grid size.
inline unsigned xcd_walk(GemmArgs& a, int m_wg, int n_wg) {
    auto magic = [](int d) { return d > 1 ? (unsigned)((1ull << 32) / (unsigned)d) + 1u : 0u; };
    a.cn = (n_wg + a.xn - 1) / a.xn;
    a.cm = (m_wg + a.xm - 1) / a.xm;
    a.per_panel = a.pn * a.cm;
    a.full = a.cn / a.pn;
    a.w_last = a.cn - a.full * a.pn;
    a.xn_shift = a.xn == 1 ? 0 : a.xn == 2 ? 1 : a.xn == 4 ? 2 : 3;
    a.mg_cn = magic(a.cn);
    a.mg_pp = magic(a.per_panel);
    a.mg_pn = magic(a.pn);
    a.mg_wl = magic(a.w_last);
    const long wgs = (long)a.cm * a.cn;
    if (wgs >= 65536) return 0;  // the tile walk's divisions are exact below 2^16 workgroups per XCD
    return (unsigned)(wgs * 8);
}

// The same with the XCD grid by shape (xcd_grid in tile_rules.h).
inline unsigned xcd_split(GemmArgs& a, int m_wg, int n_wg, double w_bytes_per_elem, int tile_cols, double a_bytes_per_elem) {
    const vla_rules::XcdGrid g = vla_rules::xcd_grid(a.M, a.N, a.K, m_wg, n_wg, w_bytes_per_elem, tile_cols, a_bytes_per_elem, tuning().gemm_panel);
    a.xm = g.xm;
    a.xn = g.xn;
    a.pn = g.pn;
    return xcd_walk(a, m_wg, n_wg);
}

}  // namespace vk
