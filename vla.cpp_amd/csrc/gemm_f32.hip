// fp32 projections of few rows: narrow tiles, 16x16x4 MFMA, K shared out over wavefronts and accumulators.
#include "gemm_f32.h"
#include "tile_rules.h"

namespace {

using namespace vk;

// The fp32 counterpart of the bf16 narrow-tile kernel: a workgroup owns 16 RB rows and 16 columns (8 + 8, see row_cols),
// both operands go straight into an LDS ring (rows of KB bytes, 16-byte pieces XOR-swizzled by the row, which keeps the
// fragment reads free of bank conflicts), NS - 1 stages in flight, one barrier per stage.
// v_mfma_f32_16x16x4_f32 multiplies full fp32 at twice the rate of plain FMAs, but one block over all of K is K / 4
// products of 32 clocks in a row: with one row block the four wavefronts share K (16-k groups in turn).  A wavefront
// keeps 16 accumulators in turn, which also shortens the sums: K / 64 values of k follow one another (K / 256 MFMA products of four) before
// the partial sums are added in pairs, as in an FMA kernel with a value of k per lane, whose error against float64 it has (50 x
// 720 x 960: 9.9e-8 of the norm; tiled kernel 5.6e-7).  Half as many accumulators cost 1.2e-7 and gained 0.2 us.  With four row blocks a
// wavefront has all of K to itself, K / 16 values: 1.5e-7 for K = 1024 (tiled kernel 8e-7).  Adding its accumulators up every 128 k would make
// that 0.95e-7, but the additions are not hidden behind the products: 51 x 2560 x 1024 9.0 -> 10.4 us, where 16 x 16 tiles take 9.1.
// NORM: the rows' RMSNorm inside.  The operand is x w (the weight, resident in LDS, is applied to the fragments), the sum of
// squares is taken from the fragments, and row c of the result is scaled by 1 / sqrt(mean + eps).
// A lane (c, q) reads 16 bytes, k = 4 q .. 4 q + 3 of a 16-k group, of row c; product t of the group takes element t of both
// operands (k = t, 4 + t, 8 + t, 12 + t).  W is the left operand, so that a lane ends with columns 4 q .. 4 q + 3 of row c.
// What bounds it: start and first loads (3 us), then per 256 k and wavefront 512 clocks of products beside 32 KiB of fill.
// Against an FMA kernel of 8 columns per workgroup (us): 50 x 720 x 960 10.8 -> 4.9, 50 x 1600 x 720 12.4 -> 6.1, 50 x 720 x 2048 13.1 -> 6.5,
// 51 x 2560 x 1024 QKV 18.0 -> 10.3; against the tiled kernel: 50 x 4096 x 720 gated 19.8 -> 9.3, 241 x 640 x 960 22.5 -> 10.5, 100 x 720 x 2048
// 43.5 -> 10.3.
template <int kEpi, int RB, int KB, int NS, bool VEC, bool NORM>
__global__ void __launch_bounds__(256) gemm_narrow_f32_kernel(GemmArgs a) {
    constexpr int BK = KB / 4, STAGE = (RB + 1) * 16 * KB, LPS = KB / 256, NLOAD = (RB + 1) * LPS;  // LPS: loads per thread and slab of 16 rows
    constexpr int KS = 4 / RB;        // wavefronts sharing a row block's K
    constexpr int NG = KB / 64 / KS;  // 16-k groups of a stage per wavefront
    constexpr int NACC = 16;
    static_assert((RB == 1 || RB == 4) && NG % 4 == 0, "one row block per workgroup or per wavefront; every accumulator has its turn in a stage");
    constexpr int IN_FLIGHT = (NS - 2) * NLOAD;
    static_assert(IN_FLIGHT <= 63 && NS * STAGE <= 160 * 1024, "ring depth");
    // NORM: the norm's weight and, after the walk, the wavefronts' partial sums of squares
    constexpr int NORM_BYTES = NORM ? F32_NORM_MAX_K * 4 : 0;
    __shared__ __attribute__((aligned(1024))) unsigned char lds[NS * STAGE + NORM_BYTES];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 15, q = lane >> 4;
    const int n_t16 = (a.N + 15) / 16;
    // the row groups of a column tile sit eight workgroups apart, on one XCD: the second one finds the weight rows in the L2
    const int n_rg = (a.M + RB * 16 - 1) / (RB * 16);
    const int rg = ((int)blockIdx.x >> 3) % n_rg, t16 = (((int)blockIdx.x >> 3) / n_rg) * 8 + ((int)blockIdx.x & 7);
    if (t16 >= n_t16) return;
    const int m0 = rg * RB * 16;
    const RowCols rc = row_cols<kEpi>(a, t16);

    // Loader: load j of a slab fills its rows (16 / LPS) j .. + 16 / LPS - 1, KB bytes each, 1 KiB per wavefront.  Rows past M
    // or N and pieces past K are read from valid addresses; their products are dropped or zeroed.
    const int lrow = wave * (1024 / KB) + lane / (KB / 16), pos = lane % (KB / 16);
    const float* src[NLOAD];
    int koff[LPS];
#pragma unroll
    for (int j = 0; j < LPS; ++j) {
        const int row = j * (16 / LPS) + lrow;
        koff[j] = (pos ^ row) * 4;
#pragma unroll
        for (int i = 0; i < RB; ++i) src[i * LPS + j] = (const float*)a.A + (long)min(m0 + i * 16 + row, a.M - 1) * a.K;
        src[RB * LPS + j] = (const float*)a.W + (long)min(row < 8 ? rc.base_lo + row : rc.base_hi + row - 8, a.N - 1) * a.K;
    }
    const uint32_t lds0 = (uint32_t)(uintptr_t)lds + wave * 1024;  // low 32 bits of a shared-aperture address = LDS offset
    const int nkt = (a.K + BK - 1) / BK;
    auto issue = [&](int kt, int stage) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < LPS; ++j) {
            const long k = min(kt * BK + koff[j], a.K - 4);
#pragma unroll
            for (int i = 0; i <= RB; ++i) load_to_lds16(src[i * LPS + j] + k, lds0 + stage * STAGE + (i * LPS + j) * 4096);
        }
    };
    if (NORM) {  // older than every operand load, so that the first stage's wait covers it
        for (int k = wave * 256; k < a.K; k += 1024)  // uniform
            load_to_lds16((const float*)a.norm_w + min(k + lane * 4, a.K - 4), (uint32_t)(uintptr_t)lds + NS * STAGE + k * 4);
    }
#pragma unroll
    for (int t = 0; t < NS - 1; ++t)
        if (t < nkt) issue(t, t);  // uniform

    const int rb = wave % RB, ks = wave / RB;
    f32x4_t acc[NACC];
#pragma unroll
    for (int j = 0; j < NACC; ++j) acc[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    f32x4_t ssq = {0.f, 0.f, 0.f, 0.f};  // squares of this lane's pieces of its row
    const int fx0 = (rb * 16 + c) * KB, fw0 = (RB * 16 + c) * KB;
    auto multiply = [&](int stage, int kt, int k_left) __attribute__((always_inline)) {  // k_left: k of this tile inside K (the last tile), or BK
        const unsigned char* base = lds + stage * STAGE;
        f32x4_t fx[NG], fw[NG];
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            const int off = ((4 * (g * KS + ks) + q) ^ c) * 16;
            fx[g] = *reinterpret_cast<const f32x4_t*>(base + fx0 + off);
            fw[g] = *reinterpret_cast<const f32x4_t*>(base + fw0 + off);
        }
        f32x4_t nw[NORM ? NG : 1];
        if (NORM) {  // past K: some weight, beside an operand that is zeroed
#pragma unroll
            for (int g = 0; g < NG; ++g) nw[g] = *reinterpret_cast<const f32x4_t*>(lds + NS * STAGE + min(kt * BK + (g * KS + ks) * 16 + 4 * q, F32_NORM_MAX_K - 4) * 4);
        }
        if (k_left < BK) {  // K is a multiple of 4: a piece is inside or outside as a whole
            const f32x4_t z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int g = 0; g < NG; ++g)
                if ((g * KS + ks) * 16 + 4 * q >= k_left) fx[g] = fw[g] = z;
        }
        __builtin_amdgcn_sched_barrier(0);  // all reads requested before the first product
        if (NORM) {
#pragma unroll
            for (int g = 0; g < NG; ++g) {
#pragma unroll
                for (int e = 0; e < 4; ++e) ssq[e] = fmaf(fx[g][e], fx[g][e], ssq[e]);
                fx[g] *= nw[g];
            }
        }
#pragma unroll
        for (int g = 0; g < NG; ++g)
#pragma unroll
            for (int t = 0; t < 4; ++t)
                acc[(g * 4 + t) % NACC] = __builtin_amdgcn_mfma_f32_16x16x4f32(fw[g][t], fx[g][t], acc[(g * 4 + t) % NACC], 0, 0, 0);
    };
    int cs = 0, ls = NS - 1, kt = 0;
    for (; kt + NS - 1 < nkt; ++kt) {
        wait_vmcnt<IN_FLIGHT>();
        __syncthreads();  // this stage has landed for every wavefront; stage ls has been read by everyone
        issue(kt + NS - 1, ls);
        multiply(cs, kt, BK);
        cs = (cs + 1 == NS) ? 0 : cs + 1;
        ls = (ls + 1 == NS) ? 0 : ls + 1;
    }
    narrow_tail<NS - 1, NLOAD>(nkt, [&](bool last) __attribute__((always_inline)) {
        __syncthreads();
        multiply(cs, kt, last ? a.K - (nkt - 1) * BK : BK);
        ++kt;
        cs = (cs + 1 == NS) ? 0 : cs + 1;
    });
#pragma unroll
    for (int w = NACC / 2; w >= 1; w /= 2)
#pragma unroll
        for (int j = 0; j < w; ++j) acc[j] += acc[j + w];
    f32x4_t sum = acc[0];
    float sq = NORM ? rows_sum((ssq[0] + ssq[1]) + (ssq[2] + ssq[3])) : 0.f;  // of row c, over this wavefront's share of K
    if (KS > 1) {
        __syncthreads();  // the ring has been read by everyone
        f32x4_t* part = reinterpret_cast<f32x4_t*>(lds);  // [ks][rb][lane]
        float* part_sq = reinterpret_cast<float*>(lds + KS * RB * 1024);  // [ks][rb][c]
        if (ks > 0) {
            part[(ks * RB + rb) * 64 + lane] = sum;
            if (NORM && q == 0) part_sq[(ks * RB + rb) * 16 + c] = sq;
        }
        __syncthreads();
        if (ks > 0) return;
        sum = (sum + part[(RB + rb) * 64 + lane]) + (part[(2 * RB + rb) * 64 + lane] + part[(3 * RB + rb) * 64 + lane]);
        if (NORM) sq = (sq + part_sq[(RB + rb) * 16 + c]) + (part_sq[(2 * RB + rb) * 16 + c] + part_sq[(3 * RB + rb) * 16 + c]);
    }
    if (NORM) {
        const float rstd = 1.0f / sqrtf(sq / (float)a.K + a.norm_eps);
        sum *= f32x4_t{rstd, rstd, rstd, rstd};
    }

    const int m = m0 + rb * 16 + c;
    const bool live = m < a.M;
    const int n0 = q < 2 ? rc.base_lo + 4 * q : rc.base_hi + 4 * q - 8;  // W row (= bias index) of v[0]
    float v[4] = {sum[0], sum[1], sum[2], sum[3]};
    if (a.bias) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] += a.bias[min(n0 + e, a.N - 1)];
    }
    if (kEpi == EPI_PLAIN) {
        if (a.act != VLA_ACT_NONE) {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = apply_act(v[e], a.act);
        }
        if (a.col_gate) {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] *= a.col_gate[min(n0 + e, a.N - 1)];
        }
        if (!live) return;
        const long o = (long)m * a.N + n0;
        if (VEC && !a.out_bf16) {  // N % 4 == 0: 4 consecutive columns are inside the row or outside as a whole
            if (n0 >= a.N) return;
            f32x4_t y = {v[0], v[1], v[2], v[3]};
            if (a.residual) y += *reinterpret_cast<const f32x4_t*>((const float*)a.residual + o);
            *reinterpret_cast<f32x4_t*>((float*)a.Y + o) = y;
            return;
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (n0 + e >= a.N) continue;
            if (a.out_bf16) ((bf16_t*)a.Y)[o + e] = f2bf(a.residual ? v[e] + bf2f(((const bf16_t*)a.residual)[o + e]) : v[e]);
            else ((float*)a.Y)[o + e] = a.residual ? v[e] + ((const float*)a.residual)[o + e] : v[e];
        }
        return;
    }
    float other[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) other[e] = __shfl_xor(v[e], 32, 64);
    if (kEpi == EPI_GLU) {  // I is a multiple of 32: no column of a tile lies past the row
        if (q >= 2 || !live) return;
        const long o = (long)m * (a.N / 2) + n0;
        f32x4_t y;
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] = apply_act(v[e], a.act) * other[e];
        if (VEC && !a.out_bf16) {
            *reinterpret_cast<f32x4_t*>((float*)a.Y + o) = y;
            return;
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (a.out_bf16) ((bf16_t*)a.Y)[o + e] = f2bf(y[e]);
            else ((float*)a.Y)[o + e] = y[e];
        }
        return;
    }
    // QKV: rotation, scatter
    const int b = min(m, a.M - 1) / a.S, s = min(m, a.M - 1) % a.S;
    if (rc.rope) {
        const long ri = (long)s * (a.D >> 1) + (rc.col_lo % a.D) + (q & 1) * 4;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float lo = q < 2 ? v[e] : other[e], hi = q < 2 ? other[e] : v[e];
            rotate_pair(lo, hi, a.cos_t[ri + e], a.sin_t[ri + e]);
            v[e] = q < 2 ? lo : hi;
        }
    }
    if (!live) return;
    const int col = q < 2 ? rc.col_lo + 4 * q : rc.col_hi + 4 * q - 8;  // segment-local, 4 consecutive columns of one head
    const int head = col / a.D, d = col % a.D;
    if (rc.seg == 2) {
        float* vt = (float*)a.vt_cache + (((long)b * a.Hkv + head) * a.D + d) * (long)a.t_max + a.tok_offset + s;
#pragma unroll
        for (int e = 0; e < 4; ++e) vt[(long)e * a.t_max] = v[e];
        return;
    }
    float* dst = rc.seg == 0 ? (float*)a.q_out + (long)m * (a.Hq * a.D) + col
                             : (float*)a.k_cache + (((long)b * a.Hkv + head) * a.t_max + a.tok_offset + s) * a.D + d;
    if (VEC) {
        *reinterpret_cast<f32x4_t*>(dst) = f32x4_t{v[0], v[1], v[2], v[3]};
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) dst[e] = v[e];
    }
}

template <int kEpi, bool VEC, bool NORM>
void launch_plan(const GemmArgs& a, int plan, hipStream_t st) {
    const unsigned grid = (unsigned)vla_rules::narrow_grid(a.M, a.N, plan);
    // Three stages (96 KiB: all of K = 720 requested at once) while every workgroup has a CU of its own, else two (64 KiB), so
    // that two share a CU: 50 x 720 x 960 (180 workgroups) 4.9 us and 5.2, 50 x 1600 x 720 (400) 7.4 us and 6.1.
    if (plan) gemm_narrow_f32_kernel<kEpi, 4, 512, 3, VEC, NORM><<<grid, 256, 0, st>>>(a);
    else if (grid <= 256) gemm_narrow_f32_kernel<kEpi, 1, 1024, 3, VEC, NORM><<<grid, 256, 0, st>>>(a);
    else gemm_narrow_f32_kernel<kEpi, 1, 1024, 2, VEC, NORM><<<grid, 256, 0, st>>>(a);
}

}  // namespace

namespace vk {

template <int kEpi>
void launch_narrow_f32(const GemmArgs& a, int plan, hipStream_t st) {
    // four columns at a time where they are inside a row as a whole and aligned, else one by one
    const uintptr_t io = kEpi == EPI_QKV ? (uintptr_t)a.q_out | (uintptr_t)a.k_cache : (uintptr_t)a.Y | (uintptr_t)a.residual;
    const bool vec = (kEpi != EPI_PLAIN || a.N % 4 == 0) && io % 16 == 0;
    if constexpr (kEpi != EPI_PLAIN) {
        if (a.norm_eps >= 0.f) {
            if (vec) launch_plan<kEpi, true, true>(a, plan, st);
            else launch_plan<kEpi, false, true>(a, plan, st);
            return;
        }
    }
    if (vec) launch_plan<kEpi, true, false>(a, plan, st);
    else launch_plan<kEpi, false, false>(a, plan, st);
}
template void launch_narrow_f32<EPI_PLAIN>(const GemmArgs&, int, hipStream_t);
template void launch_narrow_f32<EPI_QKV>(const GemmArgs&, int, hipStream_t);
template void launch_narrow_f32<EPI_GLU>(const GemmArgs&, int, hipStream_t);

}  // namespace vk
