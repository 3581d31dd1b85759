// bf16 projections of many rows: large tiles, 16x16x32 MFMA, both operands through an LDS ring.
#include "gemm_wide.h"

namespace {

using namespace vk;

// wait until at most `tiles` tiles of NL loads are due (uniform run-time count, at most MAX)
template <int NL, int MAX>
__device__ __forceinline__ void wait_tiles(int tiles) {
    if constexpr (MAX <= 0) {
        wait_vmcnt<0>();
    } else {
        if (tiles >= MAX) wait_vmcnt<MAX * NL>();
        else wait_tiles<NL, MAX - 1>(tiles);
    }
}

// NV (4 or 8) consecutive columns from n0 on of row m, plain epilogue: bias (fetched by the caller), activation, gate, residual (have_res: the
// first NV / 2 words of res), store.
template <int NV>
__device__ __forceinline__ void plain_cols(const GemmArgs& a, int m, int n0, float (&v)[NV], const float (&bias)[NV], bool have_res, u32x4_t res) {
    if (n0 >= a.N) return;
    const long o = (long)m * a.N + n0;
    if (a.bias) {
#pragma unroll
        for (int e = 0; e < NV; ++e) v[e] += bias[e];
    }
    if (a.act != VLA_ACT_NONE) epilogue_act(v, a.act, a.out_bf16);
    if (a.col_gate) {
#pragma unroll
        for (int e = 0; e < NV; ++e) v[e] *= a.col_gate[min(n0 + e, a.N - 1)];
    }
    if (a.N % 8 == 0 && a.out_bf16) {
        if (a.residual) {
            if (!have_res) {
                const bf16_t* r = (const bf16_t*)a.residual + o;
                if constexpr (NV == 8) {
                    res = *reinterpret_cast<const u32x4_t*>(r);
                } else {
                    const u32x2_t h = *reinterpret_cast<const u32x2_t*>(r);
                    res[0] = h[0];
                    res[1] = h[1];
                }
            }
#pragma unroll
            for (int e = 0; e < NV / 2; ++e) {
                v[2 * e] += __uint_as_float(res[e] << 16);
                v[2 * e + 1] += __uint_as_float(res[e] & 0xffff0000u);
            }
        }
        bf16_t* y = (bf16_t*)a.Y + o;
        if constexpr (NV == 8) *reinterpret_cast<u32x4_t*>(y) = u32x4_t{pack_bf2(v[0], v[1]), pack_bf2(v[2], v[3]), pack_bf2(v[4], v[5]), pack_bf2(v[6], v[7])};
        else *reinterpret_cast<u32x2_t*>(y) = u32x2_t{pack_bf2(v[0], v[1]), pack_bf2(v[2], v[3])};
    } else if (a.N % 8 == 0) {
#pragma unroll
        for (int h = 0; h < NV / 4; ++h) {
            f32x4_t x = {v[4 * h], v[4 * h + 1], v[4 * h + 2], v[4 * h + 3]};
            if (a.residual) x += *reinterpret_cast<const f32x4_t*>((const float*)a.residual + o + 4 * h);
            *reinterpret_cast<f32x4_t*>((float*)a.Y + o + 4 * h) = x;
        }
    } else {
#pragma unroll
        for (int e = 0; e < NV; ++e) {
            if (n0 + e >= a.N) continue;
            if (a.out_bf16) {
                const float r = a.residual ? bf2f(((const bf16_t*)a.residual)[o + e]) : 0.f;
                ((bf16_t*)a.Y)[o + e] = f2bf(a.residual ? v[e] + r : v[e]);
            } else {
                const float r = a.residual ? ((const float*)a.residual)[o + e] : 0.f;
                ((float*)a.Y)[o + e] = a.residual ? v[e] + r : v[e];
            }
        }
    }
}

// The epilogue of a wavefront of RM x RN blocks, RN < 4: rows m + 16 i, columns n0 + 8 q .. + 7 and, RN = 3, n0 + 32 + 4 q .. + 3.  Bias and a bf16
// residual (which may be the output buffer: a lane stores no other lane's elements) are requested ahead of the first store.
template <int RM, int RN>
__device__ __forceinline__ void plain_rows(const GemmArgs& a, const f32x4_t (&acc)[RM][RN], int m, int n0, int q) {
    const int n8 = n0 + 8 * q, n4 = n0 + 32 + 4 * q;
    float b8[8] = {}, b4[4] = {};
    if (a.bias) {
#pragma unroll
        for (int e = 0; e < 8; ++e) b8[e] = a.bias[min(n8 + e, a.N - 1)];
        if (RN == 3) {
#pragma unroll
            for (int e = 0; e < 4; ++e) b4[e] = a.bias[min(n4 + e, a.N - 1)];
        }
    }
    const bool have_res = a.residual != nullptr && a.out_bf16 && a.N % 8 == 0;
    u32x4_t res[RM] = {};
    u32x2_t res4[RM] = {};
    if (have_res) {
#pragma unroll
        for (int i = 0; i < RM; ++i) {
            const bf16_t* r = (const bf16_t*)a.residual + (long)min(m + 16 * i, a.M - 1) * a.N;
            res[i] = *reinterpret_cast<const u32x4_t*>(r + min(n8, a.N - 8));
            if (RN == 3) res4[i] = *reinterpret_cast<const u32x2_t*>(r + min(n4, a.N - 4));
        }
    }
#pragma unroll
    for (int i = 0; i < RM; ++i) {
        if (m + 16 * i >= a.M) continue;
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = acc[i][e >> 2][e & 3];
        plain_cols(a, m + 16 * i, n8, v, b8, have_res, res[i]);
        if constexpr (RN == 3) {
            float u[4] = {acc[i][2][0], acc[i][2][1], acc[i][2][2], acc[i][2][3]};
            plain_cols(a, m + 16 * i, n4, u, b4, have_res, u32x4_t{res4[i][0], res4[i][1], 0u, 0u});
        }
    }
}

// Workgroup tile (16 RM WM) x (16 RN WN); wavefront (wm, wn) of WM x WN owns RM x RN blocks (RN = 4 if not said otherwise) of 16 x 16 over all of K:
// v_mfma_f32_16x16x32_bf16, ascending k, whose sums have the bits of the 32x32x16 kernels.  W is the left operand, so
// that a lane (c, q) = (lane % 16, lane / 16) ends with four columns of row c per block; the loader places the rows of W
// so that a wavefront's four blocks are columns 8 q .. 8 q + 7 of both 32-column halves of a 64-column sub-tile (the
// epilogue's layout; rotation and gate partners are in the same lane): no trip through LDS at the end.
//
// What bounds it: three rates of similar size.  A 64-k step of a 192 x 192 tile is 1152 clocks of MFMA on every SIMD, 168
// KiB of fragment reads (an LDS that gives eight or more wavefronts about 215 bytes per clock) and 48 KiB from the L2 (50
// bytes per clock and CU when they hit, half of that when the weights come from memory).  Hence
//  - wavefront tiles of RM x 4 blocks (reads per product 1 / 4 + 1 / RM);
//  - operands straight into LDS, 128-byte rows, pieces XOR-swizzled by (row >> 1) & 7 (free of bank conflicts);
//  - fragments of the next 32 k are read between the products of these 32 k: the products of a phase never wait for
//    reads, and because a step's last fragments are in registers before its barrier, that barrier both publishes tile
//    kt + 1 and frees the stage of tile kt, whose refill with tile kt + NS starts right behind it: NS stages keep NS - 1
//    to NS tiles of requests in flight, at one barrier per 64 k.
// The phase behind the barrier runs at raised wave priority: of a SIMD's wavefronts the one that is through the barrier
// issues its products first instead of alternating, and the others' reads fall behind them (4096 x 4096 x 4096 113 -> 100 us
// as a kernel without epilogue variants).
// Against the direct-to-LDS kernel (128 x 128 tiles of four wavefronts, 32x32x16; us, weights not in the caches): 1323 x 6144 x 1536
// 46.3 -> 28.3 (0.88 PFLOP/s; loads alone 22 to 26, MFMA and LDS alone 23), 816 x 8192 x 1024 gated 21.4 -> 19.6, 1323 x 4608 x 1536 with the
// LayerNorm inside 34.8 -> 30.5, 13824 x 3072 x 2048 186 -> 144, 4096 x 4096 x 4096 147 -> 102 (1.35 PFLOP/s).
//
// RN = 2, 3 (plain epilogue): 32- and 48-column wavefronts of tiles that cover a narrow product in one round.  Such a launch is bound by what its
// CUs draw from the L2s (12 to 14 TB/s in all when the weights come from memory, 21 to 25 when every line hits, loads alone; requesting the
// lines ahead of the ring changes nothing), so that of the tiles that fit a round the one with the fewest operand rows per output is the
// fastest: 1323 x 1536 x 6144 264 tiles of 128 x 64 55.2 us, 176 of 128 x 96 42.6; 1323 x 1536 x 1536 15.1 -> 12.9 (96 x 96, two a CU); 1600 x 720 x 2048
// 13.8 -> 12.0 (96 x 64, two a CU).
template <int kEpi, int kNorm, int RM, int RN, int WM, int WN, int NS>
__global__ void __launch_bounds__(64 * WM * WN) gemm_wide_kernel(GemmArgs a) {
    constexpr int CW = 16 * RN, BM = 16 * RM * WM, BW = CW * WN, NW = WM * WN, KB = 128, BK = 64;
    constexpr int STAGE = (BM + BW) * KB, VA = BM / 8 / NW, VW = BW / 8 / NW, NL = VA + VW;
    constexpr int SB = (RM + WN - 1) / WN;  // row blocks whose norm a wavefront sums up
    static_assert(BM % (8 * NW) == 0 && BW % (8 * NW) == 0, "a load instruction of a wavefront fills eight rows of one operand");
    static_assert(RN == 4 || (RN >= 2 && RN < 4 && kEpi == EPI_PLAIN && kNorm == NORM_NONE), "narrower wavefront tiles know the plain epilogue only");
    static_assert(NS >= 2 && NS * STAGE <= 160 * 1024, "ring exceeds the LDS");
    static_assert((NS - 1) * NL <= 63, "ring depth exceeds the vector-memory counter");
    __shared__ __attribute__((aligned(1024))) unsigned char lds[NS * STAGE];

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WN, wn = wave % WN, c = lane & 15, q = lane >> 4;
    const int n_wg_tiles = RN == 4 ? (a.n_tiles + WN - 1) / WN : (a.N + BW - 1) / BW, m_wg_tiles = (a.M + BM - 1) / BM;
    int mtw, ntw;
    if (!xcd_tile(a, n_wg_tiles, m_wg_tiles, mtw, ntw)) return;
    const int m0 = mtw * BM;

    // Loader: load l of this wavefront fills the eight LDS rows of slab l NW + wave (A: l < VA, else W); a lane fetches
    // piece (lane % 8) ^ swz of row lane / 8.  Rows past M or N are read from the last valid one and their products
    // dropped.  Addresses: a uniform base per load, advanced by the k tile, and a 32-bit lane offset.
    const int lrow = lane >> 3, swz = ((wave & 1) * 4 + (lrow >> 1)) & 7;  // (row >> 1) & 7; NW is even
    const int koff = ((lane & 7) ^ swz) * 16;
    const unsigned char* base[NL];
    uint32_t off[NL];
#pragma unroll
    for (int l = 0; l < NL; ++l) {
        if (l < VA) {
            base[l] = (const unsigned char*)a.A + (long)m0 * a.K * 2;
            off[l] = (uint32_t)(min((l * NW + wave) * 8 + lrow, a.M - 1 - m0) * a.K * 2 + koff);
        } else if constexpr (RN < 4) {
            // a wavefront's blocks 0 and 1 are its columns 8 q .. 8 q + 7, block 2 is 32 + 4 q .. 32 + 4 q + 3
            const int s = ((l - VA) * NW + wave) * 8 + lrow, j = (s % CW) >> 4, cc = s & 15, b = ntw * BW;
            const int col = s / CW * CW + (j == 2 ? 32 + cc : 8 * (cc >> 2) + 4 * j + (cc & 3));
            base[l] = (const unsigned char*)a.W + (long)b * a.K * 2;
            off[l] = (uint32_t)(min(col, a.N - 1 - b) * a.K * 2 + koff);
        } else {
            const int slab = (l - VA) * NW + wave, s = (slab & 7) * 8 + lrow, cc = s & 15;
            const TileCols t = tile_cols<kEpi>(a, ntw * WN + (slab >> 3));
            const int b = min((slab & 4) ? t.base1 : t.base0, a.N - 1);
            base[l] = (const unsigned char*)a.W + (long)b * a.K * 2;
            off[l] = (uint32_t)(min(8 * (cc >> 2) + 4 * ((s >> 4) & 1) + (cc & 3), a.N - 1 - b) * a.K * 2 + koff);
        }
    }
    const int nkt = (a.K + BK - 1) / BK, k_left = a.K - (nkt - 1) * BK;
    // the last tile's pieces past K are read from the row's last valid piece (and their fragments zeroed)
    const uint32_t last_adj = (uint32_t)(min(koff, (k_left - 8) * 2) - koff);
    const uint32_t lds0 = (uint32_t)(uintptr_t)lds + wave * 1024;  // low 32 bits of a shared-aperture address = LDS offset
    auto issue = [&](int l, int kt, int st, uint32_t adj) __attribute__((always_inline)) {
        load_to_lds16_at(base[l] + (long)kt * KB, off[l] + adj, lds0 + st * STAGE + l * (NW * 1024));
    };
#pragma unroll
    for (int t = 0; t < NS; ++t)
        if (t < nkt) {  // uniform
            const uint32_t adj = t == nkt - 1 ? last_adj : 0u;
#pragma unroll
            for (int l = 0; l < NL; ++l) issue(l, t, t, adj);
        }

    f32x4_t acc[RM][RN];
#pragma unroll
    for (int i = 0; i < RM; ++i)
#pragma unroll
        for (int j = 0; j < RN; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    // Row sums for the norm, in the other kernels' order (a lane sums its piece of every 32 k, one accumulator per word);
    // the WN wavefronts that read the same rows take every WN-th row block each.
    float ssq[SB][4] = {}, ssum[SB][4] = {};

    const int fa = (wm * RM * 16 + c) * KB, fw = (BM + wn * CW + c) * KB, fsw = (c >> 1) & 7;
    typedef u32x4_t FragA[RM];
    typedef u32x4_t FragW[RN];
    FragA a0, a1;
    FragW w0, w1;
    // RM groups of four products on (xa, xw); between the groups the reads of the next fragments (ya, yw: chunk ch of
    // stage sr; the ones needed first are read first) and, LOAD, the requests of tile kl into stage sl.
    auto phase = [&](FragA& xa, FragW& xw, FragA& ya, FragW& yw, int sr, int ch, bool read, auto do_load, int kl, int sl, uint32_t adj) __attribute__((always_inline)) {
        constexpr bool LOAD = decltype(do_load)::value;
        const unsigned char* b = lds + sr * STAGE + (((4 * ch + q) ^ fsw) * 16);
#pragma unroll
        for (int i = 0; i < RM; ++i) {
            if (read) {  // uniform
#pragma unroll
                for (int r = i * (RM + RN) / RM; r < (i + 1) * (RM + RN) / RM; ++r) {
                    if (r < RN) yw[r] = *reinterpret_cast<const u32x4_t*>(b + fw + r * 16 * KB);
                    else ya[r - RN] = *reinterpret_cast<const u32x4_t*>(b + fa + (r - RN) * 16 * KB);
                }
            }
            if (LOAD) {
#pragma unroll
                for (int l = i * NL / RM; l < (i + 1) * NL / RM; ++l) issue(l, kl, sl, adj);
            }
#pragma unroll
            for (int j = 0; j < RN; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, xw[j]), __builtin_bit_cast(bf16x8_t, xa[i]), acc[i][j], 0, 0, 0);
            if (kNorm) {
                if (i % WN == wn) {  // uniform
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        ssq[i / WN][e] = add_squares_bf16x2(xa[i][e], ssq[i / WN][e]);
                        if (kNorm == NORM_LAYER) ssum[i / WN][e] = add_pair_bf16x2(xa[i][e], ssum[i / WN][e]);
                    }
                }
            }
            __builtin_amdgcn_sched_barrier(0);  // keeps the reads and loads where they were placed
        }
    };
    auto mask = [&](FragA& xa, FragW& xw, int ch) __attribute__((always_inline)) {  // last tile: a piece is inside K or outside as a whole
        if (ch * 32 + 8 * q >= k_left) {
            const u32x4_t z = {0u, 0u, 0u, 0u};
#pragma unroll
            for (int i = 0; i < RM; ++i) xa[i] = z;
#pragma unroll
            for (int j = 0; j < RN; ++j) xw[j] = z;
        }
    };
    auto meet = [&]() __attribute__((always_inline)) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // this wavefront's fragments of the stage are in registers
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };

    wait_tiles<NL, NS - 1>(nkt - 1);
    meet();
    {
        const unsigned char* b = lds + ((q ^ fsw) * 16);
#pragma unroll
        for (int j = 0; j < RN; ++j) w0[j] = *reinterpret_cast<const u32x4_t*>(b + fw + j * 16 * KB);
#pragma unroll
        for (int i = 0; i < RM; ++i) a0[i] = *reinterpret_cast<const u32x4_t*>(b + fa + i * 16 * KB);
    }
    int st = 0, kt = 0;
    for (; kt + NS < nkt; ++kt) {
        const int sn = (st + 1 == NS) ? 0 : st + 1;
        phase(a0, w0, a1, w1, st, 1, true, std::false_type{}, 0, 0, 0u);
        wait_vmcnt<(NS - 2) * NL>();  // tile kt + 1 has landed (this wavefront's part of it)
        meet();
        __builtin_amdgcn_s_setprio(1);
        phase(a1, w1, a0, w0, sn, 0, true, std::true_type{}, kt + NS, st, kt + NS == nkt - 1 ? last_adj : 0u);
        __builtin_amdgcn_s_setprio(0);
        st = sn;
    }
    // the last NS tiles: nothing left to request (a ring that kept re-fetching past the end would add NS tiles of traffic)
    for (; kt < nkt; ++kt) {
        const int sn = (st + 1 == NS) ? 0 : st + 1;
        const bool last = kt == nkt - 1;
        if (last && k_left < BK) mask(a0, w0, 0);
        phase(a0, w0, a1, w1, st, 1, true, std::false_type{}, 0, 0, 0u);
        if (!last) {
            wait_tiles<NL, NS - 2>(nkt - 2 - kt);
            meet();
        } else if (k_left < BK) {
            mask(a1, w1, 1);
        }
        phase(a1, w1, a0, w0, sn, 0, !last, std::false_type{}, 0, 0, 0u);
        st = sn;
    }

    if constexpr (RN < 4) {
        plain_rows<RM, RN>(a, acc, m0 + wm * RM * 16 + c, ntw * BW + wn * CW, q);
        return;
    } else {
    // Epilogue: this lane's rows m0 + 16 (wm RM + i) + c, columns 8 q .. + 7 of both halves of sub-tile nt.
    const int nt = ntw * WN + wn, jg = q * 8;
    float* row_f = reinterpret_cast<float*>(lds);  // (rstd, mean rstd) of the tile's rows
    if (kNorm) {
        meet();  // every wavefront is through with the ring
        const float inv_k = 1.0f / (float)a.K;
#pragma unroll
        for (int i = 0; i < RM; ++i) {
            if (i % WN != wn) continue;  // uniform
            const float sq = rows_sum((ssq[i / WN][0] + ssq[i / WN][1]) + (ssq[i / WN][2] + ssq[i / WN][3]));
            f32x2_t f = {0.f, 0.f};
            if (kNorm == NORM_LAYER) {
                const float mean = rows_sum((ssum[i / WN][0] + ssum[i / WN][1]) + (ssum[i / WN][2] + ssum[i / WN][3])) * inv_k;
                f[0] = rsqrtf(fmaxf(sq * inv_k - mean * mean, 0.f) + a.norm_eps);
                f[1] = mean * f[0];
            } else {
                f[0] = rsqrtf(sq * inv_k + a.norm_eps);
            }
            if (q == 0) *reinterpret_cast<f32x2_t*>(row_f + ((wm * RM + i) * 16 + c) * 2) = f;
        }
        meet();
    }
    if (nt >= a.n_tiles) return;
    const TileCols tc = tile_cols<kEpi>(a, nt);
    float bias[16] = {}, cs[16] = {};
    if (a.bias) {
#pragma unroll
        for (int e = 0; e < 16; ++e) bias[e] = a.bias[min((e < 8 ? tc.base0 : tc.base1) + jg + (e & 7), a.N - 1)];
    }
    if (kNorm == NORM_LAYER) {
#pragma unroll
        for (int e = 0; e < 16; ++e) cs[e] = a.colsum[(e < 8 ? tc.base0 : tc.base1) + jg + (e & 7)];
    }
    // A bf16 residual of up to four of the lane's rows is requested before the first of them is stored (it may be the output
    // buffer: a lane stores no other lane's elements).  All eight of the 256 x 256 tile at once are 64 registers beside 128
    // accumulators and spilled.
    constexpr int RG = RM < 4 ? RM : 4;
    const bool have_res = kEpi == EPI_PLAIN && a.residual != nullptr && a.out_bf16 && a.N % 8 == 0;
    u32x4_t res[RG][2] = {};
    // QKV: what belongs to the lane's columns is formed once for all of its rows.  dst[h]: element (b = 0, s = 0) of half h's
    // first column; rows are s_stride apart within an observation, observations b_stride.
    bf16_t* dst[2] = {nullptr, nullptr};
    long s_stride = 0, b_stride = 0;
    int p0 = 0;
    if (kEpi == EPI_QKV) {
        if (tc.rope) p0 = tc.col0 % a.D + jg;  // pair index inside the head
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int col = (h ? tc.col1 : tc.col0) + jg, head = col / a.D, d = col - head * a.D;  // segment-local, 8 columns of one head
            if (tc.seg == 0) dst[h] = (bf16_t*)a.q_out + col;
            else if (tc.seg == 1) dst[h] = (bf16_t*)a.k_cache + ((long)head * a.t_max + a.tok_offset) * a.D + d;
            else dst[h] = (bf16_t*)a.vt_cache + ((long)head * a.D + d) * a.t_max + a.tok_offset;
        }
        s_stride = tc.seg == 0 ? a.Hq * a.D : tc.seg == 1 ? a.D : 1;
        b_stride = tc.seg == 0 ? (long)a.S * a.Hq * a.D : (long)a.Hkv * a.D * a.t_max;
    }
#pragma unroll
    for (int i = 0; i < RM; ++i) {
        if (have_res && i % RG == 0) {
#pragma unroll
            for (int j = 0; j < RG; ++j)
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int m = min(m0 + (wm * RM + i + j) * 16 + c, a.M - 1), n = min(nt * 64 + h * 32 + jg, a.N - 8);
                    res[j][h] = *reinterpret_cast<const u32x4_t*>((const bf16_t*)a.residual + (long)m * a.N + n);
                }
        }
        const int mr = (wm * RM + i) * 16 + c;
        float lo[8], hi[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            lo[e] = acc[i][e >> 2][e & 3];
            hi[e] = acc[i][2 + (e >> 2)][e & 3];
        }
        if (kNorm) {
#pragma clang fp contract(off)  // the other kernels round the scaled value before a bias is added
            const f32x2_t f = *reinterpret_cast<const f32x2_t*>(row_f + mr * 2);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                lo[e] = kNorm == NORM_LAYER ? center_scale(lo[e], f[0], f[1], cs[e]) : lo[e] * f[0];
                hi[e] = kNorm == NORM_LAYER ? center_scale(hi[e], f[0], f[1], cs[8 + e]) : hi[e] * f[0];
            }
        }
        if (m0 + mr >= a.M) continue;
        if (kEpi != EPI_QKV) {
            epilogue_16<bf16_t, kEpi, true>(a, m0 + mr, nt, tc, jg, lo, hi, have_res, res[i % RG][0], res[i % RG][1], bias);
            continue;
        }
        const int b = (int)div_c((unsigned)(m0 + mr), a.div_s), s = m0 + mr - b * a.S;
        if (a.bias) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                lo[e] += bias[e];
                hi[e] += bias[8 + e];
            }
        }
        if (tc.rope) {
            const float* cr = a.cos_t + (long)s * (a.D >> 1) + p0;
            const float* sr = a.sin_t + (long)s * (a.D >> 1) + p0;
#pragma unroll
            for (int e = 0; e < 8; ++e) rotate_pair(lo[e], hi[e], cr[e], sr[e]);
        }
        const long o = b * b_stride + s * s_stride;
        const u32x4_t pk[2] = {{pack_bf2(lo[0], lo[1]), pack_bf2(lo[2], lo[3]), pack_bf2(lo[4], lo[5]), pack_bf2(lo[6], lo[7])},
                               {pack_bf2(hi[0], hi[1]), pack_bf2(hi[2], hi[3]), pack_bf2(hi[4], hi[5]), pack_bf2(hi[6], hi[7])}};
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            if (tc.seg != 2) {  // uniform
                *reinterpret_cast<u32x4_t*>(dst[h] + o) = pk[h];
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) dst[h][o + (long)e * a.t_max] = (bf16_t)(pk[h][e >> 1] >> (16 * (e & 1)));
            }
        }
    }
    }
}

template <int kEpi, int RM, int WM, int WN, int NS, int RN = 4>
bool launch_tile(GemmArgs a, hipStream_t st) {
    const unsigned grid = xcd_split(a, (a.M + 16 * RM * WM - 1) / (16 * RM * WM), RN == 4 ? (a.n_tiles + WN - 1) / WN : (a.N + 16 * RN * WN - 1) / (16 * RN * WN), 2.0, 16 * RN * WN, 2.0);
    if (!grid) return false;  // more workgroups than the tile walk can count
    constexpr int T = 64 * WM * WN;
    if (kEpi == EPI_QKV) a.div_s = make_divc(a.S, a.M);
    if constexpr (kEpi == EPI_QKV) {
        if (a.norm_eps >= 0.f && a.colsum) {
            gemm_wide_kernel<kEpi, NORM_LAYER, RM, RN, WM, WN, NS><<<grid, T, 0, st>>>(a);
            return true;
        }
    }
    if constexpr (kEpi == EPI_QKV || kEpi == EPI_GLU) {
        if (a.norm_eps >= 0.f) {
            gemm_wide_kernel<kEpi, NORM_RMS, RM, RN, WM, WN, NS><<<grid, T, 0, st>>>(a);
            return true;
        }
    }
    gemm_wide_kernel<kEpi, NORM_NONE, RM, RN, WM, WN, NS><<<grid, T, 0, st>>>(a);
    return true;
}

}  // namespace

namespace vk {

template <int kEpi>
bool launch_wide(const GemmArgs& a, int tile, hipStream_t st) {
    if constexpr (kEpi == EPI_PLAIN) {
        switch (tile) {
            case vla_rules::PLAIN_96X96_PAIRS: return launch_tile<kEpi, 3, 2, 2, 3, 3>(a, st);
            case vla_rules::PLAIN_128X96: return launch_tile<kEpi, 4, 2, 2, 5, 3>(a, st);
            case vla_rules::PLAIN_96X64_PAIRS: return launch_tile<kEpi, 3, 2, 2, 4, 2>(a, st);
            default: break;
        }
    }
    switch (tile) {
        case vla_rules::WIDE_256X256: return launch_tile<kEpi, 8, 2, 4, 2>(a, st);
        case vla_rules::WIDE_192X192: return launch_tile<kEpi, 3, 4, 3, 3>(a, st);
        case vla_rules::WIDE_256X128: return launch_tile<kEpi, 4, 4, 2, 3>(a, st);
        case vla_rules::WIDE_192X128: return launch_tile<kEpi, 3, 4, 2, 3>(a, st);
        case vla_rules::WIDE_128X128: return launch_tile<kEpi, 2, 4, 2, 4>(a, st);
        default: return launch_tile<kEpi, 2, 4, 2, 2>(a, st);
    }
}
template bool launch_wide<EPI_PLAIN>(const GemmArgs&, int, hipStream_t);
template bool launch_wide<EPI_QKV>(const GemmArgs&, int, hipStream_t);
template bool launch_wide<EPI_GLU>(const GemmArgs&, int, hipStream_t);

}  // namespace vk
