// MFMA projections for the attention path on gfx950.
//
// One 64x64 output tile per 256-thread workgroup (four 64-lane wavefronts, each
// a 32x32 MFMA accumulator), A and W tiles staged through padded LDS rows of
// 128 bytes, the next tile's global loads in flight while the current one is
// multiplied.  Three instantiations share the loop:
//
//   bf16 : v_mfma_f32_32x32x16_bf16                       (configs 1-3)
//   fp32 : v_mfma_f32_32x32x2_f32, full fp32 products     (config 0, 1e-5 bar)
//   int8 : v_mfma_i32_32x32x32_i8 against 2-bit ternary weights decoded while
//          they are staged (BitVLA, exact int32 accumulators)
//
// and three epilogues, all run from an LDS copy of the accumulator tile:
//
//   PLAIN   y = x.W^T + bias + residual        (ggml_mul_mat + add; Wo)
//   QKV     bias, NeoX RoPE on the Q and K columns, Q to a token-major buffer,
//           K / V straight into the resident cache at token tok_offset + s
//   TERNARY acc - 2*rowsum (code offset), optional raw int32 dump, bf16 out =
//           float(acc) / s[m] * ws[group]
//
// MFMA operand layout used throughout (64 lanes, g = lane / 32, r = lane % 32):
// a lane supplies 16 bytes of row r of its operand at k offset
// chunk*kChunk + g*(kChunk/2); the 32x32 result holds, in element 4j+i of lane
// (g, r), C[8j + 4g + i][r].

#include <stdlib.h>
#include <string.h>
#include <type_traits>

#include "common.h"
#include "gemm_common.h"
#include "fused_f32.h"
#include "gemm_f32.h"
#include "gemm_wide.h"
#include "tile_rules.h"
#include "vla_kernels.h"

namespace {

using namespace vk;

template <typename T> struct Traits;
template <> struct Traits<bf16_t> {
    typedef f32x16_t Acc;
    static constexpr int kElemBytes = 2;
    static constexpr int kChunkBytes = 32;  // bytes of k per MFMA group per row
    __device__ static __forceinline__ void mma(Acc& acc, const u32x4_t& a, const u32x4_t& b) {
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b),
                                                      acc, 0, 0, 0);
    }
};
template <> struct Traits<float> {
    typedef f32x16_t Acc;
    static constexpr int kElemBytes = 4;
    static constexpr int kChunkBytes = 32;
    __device__ static __forceinline__ void mma(Acc& acc, const u32x4_t& a, const u32x4_t& b) {
        const f32x4_t fa = __builtin_bit_cast(f32x4_t, a), fb = __builtin_bit_cast(f32x4_t, b);
#pragma unroll
        for (int t = 0; t < 4; ++t) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[t], fb[t], acc, 0, 0, 0);
    }
};
template <> struct Traits<int8_t> {
    typedef i32x16_t Acc;
    static constexpr int kElemBytes = 1;
    static constexpr int kChunkBytes = 32;
    __device__ static __forceinline__ void mma(Acc& acc, const u32x4_t& a, const u32x4_t& b) {
        acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(__builtin_bit_cast(i32x4_t, a), __builtin_bit_cast(i32x4_t, b), acc,
                                                   0, 0, 0);
    }
};

// Packed ternary weights are stored "MFMA-fragment-major": for each block of 32 output
// columns and each group of 32 k, 64 consecutive words [g][r] hold the 16 codes
// k = 32*kk + 16*g .. +15 of column 32*nb + r -- exactly what lane (g, r) of a wavefront
// feeds to v_mfma_i32_32x32x32_i8, so a fragment is one coalesced 256-byte load.
__host__ __device__ __forceinline__ long tern_word_index(long n, int w, int K) {
    return (((n >> 5) * (K / 32) + (w >> 1)) * 2 + (w & 1)) * 32 + (n & 31);
}

// Accumulator element -> raw 32-bit LDS cell (by value: a bit_cast applied
// directly to a vector element expression reads element 0).
__device__ __forceinline__ uint32_t acc_bits(float v) { return __float_as_uint(v); }
__device__ __forceinline__ uint32_t acc_bits(int v) { return (uint32_t)v; }

// Workgroup tile (64*TM) x (64*TN), 2 x 2 wavefronts; wavefront (wm, wn) owns the 32x32
// MFMA blocks in block rows wm + 2i (i < TM) and block columns wn + 2j (j < TN), so every
// 64x64 sub-tile is made of one block from each wavefront.  KB = bytes of K per staged row.
template <typename T, int kEpi, int TM, int TN, int KB, int DEPTH>
__global__ void __launch_bounds__(256) gemm_kernel(GemmArgs a) {
    typedef Traits<T> TR;
    constexpr int EB = TR::kElemBytes;
    constexpr int BK = KB / EB;        // k elements per tile
    constexpr int EPV = 16 / EB;       // elements per 16-byte vector
    constexpr int STRIDE = KB + 16;    // padded LDS row
    constexpr int ROWS_A = 64 * TM, ROWS_W = 64 * TN;
    constexpr int VPR = KB / 16;       // 16-byte vectors per staged row
    constexpr int VA = ROWS_A * VPR / 256, VW = ROWS_W * VPR / 256;  // vectors per thread
    static_assert(kEpi != EPI_TERNARY || (TM == 1 && TN == 1 && KB == 128), "ternary staging assumes 64x64x128 tiles");

    // two operand buffers: tile kt is multiplied out of buffer kt & 1 while tile kt + 1 is
    // being stored into the other one, so a k-tile costs one barrier
    constexpr int BUF = (ROWS_A + ROWS_W) * STRIDE;
    __shared__ __attribute__((aligned(16))) unsigned char lds[2 * BUF];
    static_assert(sizeof(float) * 64 * C_STRIDE <= sizeof(lds), "C sub-tile must fit in the operand buffers");

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int g = lane >> 5, r = lane & 31;
    // Linear workgroup id -> (M tile, N tile).  id % 8 is the XCD a workgroup is dispatched
    // to; the 8 XCDs form an xm x xn grid and XCD (i, j) owns the M tiles = i (mod xm) and
    // the N tiles = j (mod xn), so each L2 fetches 1/xm of A and 1/xn of W instead of the
    // whole of either (the host picks the split that minimises the total).
    const int n_wg_tiles = (a.n_tiles + TN - 1) / TN, m_wg_tiles = (a.M + ROWS_A - 1) / ROWS_A;
    int mtw, ntw;
    if (!xcd_tile(a, n_wg_tiles, m_wg_tiles, mtw, ntw)) return;
    const int m0 = mtw * ROWS_A;
    TileCols tc[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) tc[j] = tile_cols<kEpi>(a, ntw * TN + j);

    typename TR::Acc acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0;

    const int nkt = (a.K + BK - 1) / BK;

    // Operand staging: global -> registers -> LDS, with DEPTH k-tiles of loads in flight
    // (a ring of register stages with compile-time indices).  The loads are unconditional:
    // rows past M or N and k past K are redirected to valid addresses (their products land
    // in outputs that are dropped, or are zeroed when the one partial k-tile is stored), and
    // the ring keeps re-reading the last tile once the real ones are exhausted, so the loop
    // body has no load under a branch and the wait counts stay exact.
    const unsigned char* ap[VA];
    int a_koff[VA];
#pragma unroll
    for (int v = 0; v < VA; ++v) {
        const int idx = tid + v * 256;
        const int m = min(m0 + idx / VPR, a.M - 1);
        a_koff[v] = (idx % VPR) * EPV;
        ap[v] = (const unsigned char*)a.A + (long)m * a.K * EB;
    }
    const unsigned char* wp[VW];
    if (kEpi != EPI_TERNARY) {
#pragma unroll
        for (int v = 0; v < VW; ++v) {
            const int idx = tid + v * 256;
            constexpr int RPV = 256 / VPR;                     // rows covered by one vector index step
            const int sub = (v * RPV) / 64, wr = (idx / VPR) & 63;  // sub is compile-time per unrolled v
            int n = (wr < 32) ? tc[sub].base0 + wr : tc[sub].base1 + wr - 32;
            n = min(max(n, 0), a.N - 1);
            wp[v] = (const unsigned char*)a.W + (long)n * a.K * EB;
        }
    } else {
        // 64 rows x 128 k of 2-bit codes = 64 x 8 words; two words per thread: the two
        // 16-k halves (g = 0, 1) of 32-k group q of the tile.
        const int n = min(ntw * BN + (tid >> 2), a.N - 1);
        wp[0] = (const unsigned char*)((const uint32_t*)a.W + tern_word_index(n, (tid & 3) * 2, a.K));
    }
    u32x4_t ra[DEPTH][VA], rw[DEPTH][VW];
    // Load vector i of tile kt into ring stage st; i runs over the VA vectors of A and then
    // the VW vectors of W (the ternary staging has a single W entry of two words).
    constexpr int NLOAD = VA + ((kEpi != EPI_TERNARY) ? VW : 1);
    auto load_vec = [&](int st, int kt, int i) __attribute__((always_inline)) {
        const int k0 = kt * BK;
        if (i < VA) {
            const int k = min(k0 + a_koff[i], a.K - EPV);
            ra[st][i] = *reinterpret_cast<const u32x4_t*>(ap[i] + (long)k * EB);
        } else if (kEpi != EPI_TERNARY) {
            const int v = i - VA;
            const int k = min(k0 + a_koff[v % VA], a.K - EPV);  // same column pattern as A (VPR | 256)
            rw[st][v] = *reinterpret_cast<const u32x4_t*>(wp[v] + (long)k * EB);
        } else {
            const uint32_t* w = (const uint32_t*)wp[0] + (long)(k0 / 32) * 64;
            rw[st][0][0] = w[0];
            rw[st][0][1] = w[32];
        }
    };
    auto load_tile = [&](int st, int kt) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NLOAD; ++i) load_vec(st, kt, i);
    };
    auto mask_partial = [&](int st, int kt) __attribute__((always_inline)) {  // zero what lies past K
#pragma unroll
        for (int v = 0; v < VA; ++v)
            if (kt * BK + a_koff[v] >= a.K) {
                const u32x4_t z = {0u, 0u, 0u, 0u};
                ra[st][v] = z;
            }
        if (kEpi != EPI_TERNARY) {
#pragma unroll
            for (int v = 0; v < VW; ++v)
                if (kt * BK + a_koff[v % VA] >= a.K) {
                    const u32x4_t z = {0u, 0u, 0u, 0u};
                    rw[st][v] = z;
                }
        }
    };
    auto store_tile = [&](int st, int buf) __attribute__((always_inline)) {
        unsigned char* ldsA = lds + buf * BUF;
        unsigned char* ldsW = ldsA + ROWS_A * STRIDE;
#pragma unroll
        for (int v = 0; v < VA; ++v) {
            const int idx = tid + v * 256;
            *reinterpret_cast<u32x4_t*>(ldsA + (idx / VPR) * STRIDE + (idx % VPR) * 16) = ra[st][v];
        }
        if (kEpi != EPI_TERNARY) {
#pragma unroll
            for (int v = 0; v < VW; ++v) {
                const int idx = tid + v * 256;
                *reinterpret_cast<u32x4_t*>(ldsW + (idx / VPR) * STRIDE + (idx % VPR) * 16) = rw[st][v];
            }
        } else {
            // Decode 2 words -> 32 codes (unsigned 0..3; the -2 offset is folded
            // into the epilogue as -2*rowsum).  Word layout: value b+4j sits at
            // bits 8b+2j, so (w >> 2j) & 0x03030303 is values 4j..4j+3.
            const int row = tid >> 2, q = tid & 3;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const uint32_t w = rw[st][0][h];
                u32x4_t d;
                d[0] = w & 0x03030303u;
                d[1] = (w >> 2) & 0x03030303u;
                d[2] = (w >> 4) & 0x03030303u;
                d[3] = (w >> 6) & 0x03030303u;
                *reinterpret_cast<u32x4_t*>(ldsW + row * STRIDE + q * 32 + h * 16) = d;
            }
        }
    };
    // Multiplies the tile in LDS buffer buf.  With LOAD set, the loads of tile kt_load into
    // ring stage st_load are issued a few per k-chunk between the MFMA groups instead of in
    // one burst: a burst keeps every wavefront of the workgroup waiting at the texture
    // unit's queue before any of them starts on the LDS reads, so load issue and multiply
    // would run one after the other instead of side by side.
    auto multiply = [&](int buf, auto do_load, int st_load, int kt_load) __attribute__((always_inline)) {
        constexpr bool LOAD = decltype(do_load)::value;
        constexpr int NCH = KB / TR::kChunkBytes;
        const unsigned char* ldsA = lds + buf * BUF;
        const unsigned char* ldsW = ldsA + ROWS_A * STRIDE;
        // operand fragments are read one k-chunk ahead of the MFMAs that use them, so the
        // LDS latency of chunk ch + 1 passes under the MFMAs of chunk ch
        u32x4_t fa[2][TM], fw[2][TN];
        auto read_frags = [&](int slot, int ch) __attribute__((always_inline)) {
            const int off = ch * TR::kChunkBytes + g * 16;
#pragma unroll
            for (int i = 0; i < TM; ++i) fa[slot][i] = *reinterpret_cast<const u32x4_t*>(ldsA + ((wm + 2 * i) * 32 + r) * STRIDE + off);
#pragma unroll
            for (int j = 0; j < TN; ++j) fw[slot][j] = *reinterpret_cast<const u32x4_t*>(ldsW + ((wn + 2 * j) * 32 + r) * STRIDE + off);
        };
        read_frags(0, 0);
#pragma unroll
        for (int ch = 0; ch < NCH; ++ch) {
            if (ch + 1 < NCH) read_frags((ch + 1) & 1, ch + 1);
            if (LOAD) {
#pragma unroll
                for (int i = ch * NLOAD / NCH; i < (ch + 1) * NLOAD / NCH; ++i) load_vec(st_load, kt_load, i);
            }
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) TR::mma(acc[i][j], fa[ch & 1][i], fw[ch & 1][j]);
            __builtin_amdgcn_sched_barrier(0);  // keeps the reads and loads where they were placed
        }
    };

    // Stage st of the ring holds tile kt with kt % DEPTH == st.  Main loop: whole groups
    // of DEPTH full tiles, no branch around a load.  The remaining tiles (fewer than DEPTH
    // full ones and at most one partial) are already in flight when the main loop ends
    // and are drained without further loads.  The LDS store of tile kt + 1 follows the
    // multiply of tile kt in program order, so it runs under the MFMAs still in flight.
#pragma unroll
    for (int st = 0; st < DEPTH; ++st) load_tile(st, min(st, nkt - 1));
    if (BK > a.K) mask_partial(0, 0);
    store_tile(0, 0);
    __syncthreads();
    const int n_main = (a.K / BK) / DEPTH;
    for (int gi = 0; gi < n_main; ++gi) {
#pragma unroll
        for (int st = 0; st < DEPTH; ++st) {
            const int kt = gi * DEPTH + st;
            // stage st held tile kt, already in LDS: refill it with tile kt + DEPTH
            multiply(kt & 1, std::true_type{}, st, min(kt + DEPTH, nkt - 1));
            if ((kt + 2) * BK > a.K) mask_partial((st + 1) % DEPTH, kt + 1);  // uniform; only the last tile can be partial
            store_tile((st + 1) % DEPTH, (kt + 1) & 1);  // past the last tile: a repeat of it, never read
            __syncthreads();
        }
    }
#pragma unroll
    for (int st = 0; st < DEPTH; ++st) {
        const int kt = n_main * DEPTH + st;
        if (kt < nkt) {  // uniform
            multiply(kt & 1, std::false_type{}, 0, 0);
            if (kt + 1 < nkt) {
                if ((kt + 2) * BK > a.K) mask_partial((st + 1) % DEPTH, kt + 1);
                store_tile((st + 1) % DEPTH, (kt + 1) & 1);
            }
            __syncthreads();
        }
    }

    // Epilogue, one 64x64 sub-tile at a time through an LDS copy of the accumulators.
    uint32_t* C = reinterpret_cast<uint32_t*>(lds);
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            if (i + j > 0) __syncthreads();
#pragma unroll
            for (int jj = 0; jj < 4; ++jj)
#pragma unroll
                for (int ii = 0; ii < 4; ++ii)
                    C[(wm * 32 + 8 * jj + 4 * g + ii) * C_STRIDE + wn * 32 + r] = acc_bits(acc[i][j][4 * jj + ii]);
            __syncthreads();
            const int nt_sub = ntw * TN + j;
            if (nt_sub < a.n_tiles) epilogue_64x64<T, kEpi>(a, C, m0 + i * 64, nt_sub, tc[j], tid);
        }
}

// ---- bf16 GEMM with operand tiles loaded straight into LDS --------------------------
// Same tiling, wavefront layout, XCD mapping and epilogues as gemm_kernel, for bf16
// operands with K a multiple of 16.  A stage of the LDS ring holds one k-tile of A and W
// rows, KB bytes per row and no padding: a load instruction of a wavefront fills 1 KiB of
// consecutive LDS (1024 / KB rows).  Bank conflicts of the fragment reads are avoided by a
// swizzle instead of padding: the 16-byte piece c of row `row` is kept at piece position
// c ^ swz(row), swz = (row >> 1) & 7 for 128-byte rows and row & 15 for 256-byte rows (16
// consecutive fragment rows then cover all 64 banks exactly once); the loading lane picks
// the global piece that belongs in its LDS slot.  NS - 1 tiles of loads are in flight; a
// k-tile costs one barrier, and no wavefront spends issue slots on LDS stores.
template <int kEpi, int TM, int TN, int KB, int NS, int kNorm>
__global__ void __launch_bounds__(256) gemm_dl_kernel(GemmArgs a) {
    typedef bf16_t T;
    typedef Traits<bf16_t> TR;
    constexpr int EB = 2, BK = KB / EB, EPV = 8;
    constexpr int ROWS_A = 64 * TM, ROWS_W = 64 * TN;
    constexpr int VPR = KB / 16;        // 16-byte pieces per row
    constexpr int RPS = 256 / VPR;      // rows filled by one load per thread of the workgroup
    constexpr int VA = ROWS_A / RPS, VW = ROWS_W / RPS, NLOAD = VA + VW;
    constexpr int NCH = KB / 32;        // 16-k MFMA chunks per tile
    constexpr int STAGE = (ROWS_A + ROWS_W) * KB;
    constexpr int C_BYTES = 4 * 64 * C_STRIDE;
    constexpr int EPI_BYTES = 2 * C_BYTES + ROWS_A * 16;  // two C sub-tiles, then two (sum of squares, sum) pairs per tile row (kNorm)
    constexpr int LDS_BYTES = NS * STAGE > EPI_BYTES ? NS * STAGE : EPI_BYTES;
    constexpr int IN_FLIGHT = (NS - 2) * NLOAD;  // loads younger than the tile about to be multiplied
    static_assert(KB == 128 || KB == 256, "swizzle is defined for 128- and 256-byte rows");
    static_assert(NS >= 2 && IN_FLIGHT <= 63, "ring depth exceeds the vector-memory counter");
    __shared__ __attribute__((aligned(1024))) unsigned char lds[LDS_BYTES];

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    const int g = lane >> 5, r = lane & 31;
    const int n_wg_tiles = (a.n_tiles + TN - 1) / TN, m_wg_tiles = (a.M + ROWS_A - 1) / ROWS_A;
    int mtw, ntw;
    if (!xcd_tile(a, n_wg_tiles, m_wg_tiles, mtw, ntw)) return;
    const int m0 = mtw * ROWS_A;
    TileCols tc[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) tc[j] = tile_cols<kEpi>(a, ntw * TN + j);

    typename TR::Acc acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0;

    const int nkt = (a.K + BK - 1) / BK, nkt_full = a.K / BK;
    // kNorm: the GEMM multiplies raw rows of A and scales row m of the result by
    // rsqrt(mean_k A[m][k]^2 + eps); the squares are summed from the same LDS fragments
    // the MFMAs read (lane (g, r) sees 8 of every 16 k of its rows; the two halves meet
    // after the loop), two bf16 products per instruction.  NORM_LAYER also sums the values:
    // row m of the result becomes rstd (acc - mean colsum[n]), the projection of the
    // centred and scaled row.  The two wavefronts that read the same A rows (wn = 0, 1)
    // take alternate k-chunks, and each of a fragment's four words has its own
    // accumulator, so a chunk adds one dependent operation per accumulator.
    float ssq[TM][4], ssum[TM][4];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) ssq[i][e] = ssum[i][e] = 0.f;

    // A bf16 residual is fetched now, ahead of every operand load, instead of in the
    // epilogue where nothing is left to hide its latency (the epilogue thread layout:
    // row tid / 4, columns 8 (tid % 4) .. +7 of each 32-column half of a 64x64 sub-tile).
    u32x4_t res_pf[TM][TN][2] = {};
    const bool pf = kEpi == EPI_PLAIN && a.residual != nullptr && a.out_bf16 && a.N % 8 == 0;
    if (pf) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int hlf = 0; hlf < 2; ++hlf) {
                    const int m = min(m0 + i * 64 + (tid >> 2), a.M - 1);
                    const int n0 = min((ntw * TN + j) * BN + hlf * 32 + (tid & 3) * 8, a.N - 8);
                    res_pf[i][j][hlf] = *reinterpret_cast<const u32x4_t*>((const bf16_t*)a.residual + (long)m * a.N + n0);
                }
    }

    // NORM_LAYER_PRE: the row sums handed over by the producing launch, six (sum of squares, sum) pairs per thread
    // and tile row (the four threads of a row take the tiles t % 4), requested ahead of the operand loads as well.
    f32x2_t st_pf[TM][STAT_MAX_TILES / 4] = {};
    if (kNorm == NORM_LAYER_PRE) {
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            const float* sp = a.stats_in + (long)min(m0 + i * 64 + (tid >> 2), a.M - 1) * a.n_stat * 2;
#pragma unroll
            for (int t = 0; t < STAT_MAX_TILES / 4; ++t) st_pf[i][t] = *reinterpret_cast<const f32x2_t*>(sp + min((tid & 3) + 4 * t, a.n_stat - 1) * 2);
        }
    }

    // Loader side.  Thread tid fills LDS slot tid of each 256-slot slab; slab v of A holds
    // rows v*RPS .. v*RPS+RPS-1.  The slot is piece position tid % VPR of row tid / VPR, so
    // the lane fetches the logical piece (tid % VPR) ^ swz(row); swz only involves the low
    // row bits, which do not depend on the slab.  Rows past M or N and k past K are
    // redirected to valid addresses: their products land in outputs that are dropped, and
    // k-chunks past K are never multiplied.
    const int lrow = tid / VPR;
    const int lsw = (KB == 128) ? ((lrow >> 1) & 7) : (lrow & 15);
    const int koff = ((tid % VPR) ^ lsw) * EPV;
    const unsigned char* ap[VA];
#pragma unroll
    for (int v = 0; v < VA; ++v) ap[v] = (const unsigned char*)a.A + (long)min(m0 + v * RPS + lrow, a.M - 1) * a.K * EB;
    const unsigned char* wp[VW];
#pragma unroll
    for (int v = 0; v < VW; ++v) {
        const int sub = (v * RPS) / 64, wr = (v * RPS + lrow) & 63;  // sub is compile-time per unrolled v
        int n = (wr < 32) ? tc[sub].base0 + wr : tc[sub].base1 + wr - 32;
        n = min(max(n, 0), a.N - 1);
        wp[v] = (const unsigned char*)a.W + (long)n * a.K * EB;
    }
    const uint32_t lds0 = (uint32_t)(uintptr_t)lds + wave * 1024;  // low 32 bits of a shared-aperture address = LDS offset
    auto issue = [&](int i, int kt, int stage) __attribute__((always_inline)) {
        const long kb = (long)min(kt * BK + koff, a.K - EPV) * EB;
        if (i < VA) load_to_lds16(ap[i] + kb, lds0 + stage * STAGE + i * 4096);
        else load_to_lds16(wp[i - VA] + kb, lds0 + stage * STAGE + ROWS_A * KB + (i - VA) * 4096);
    };

    // Consumer side.  Fragment row r of any 32-row block has swz = (r >> 1) & 7 (or r & 15);
    // the lane wants logical piece 2 ch + g, i.e. position (2 ch) ^ (g ^ swz).
    const int fsw = (KB == 128) ? ((r >> 1) & 7) : (r & 15);
    const int xo = (g ^ fsw) * 16;
    const int fragA = (wm * 32 + r) * KB, fragW = ROWS_A * KB + (wn * 32 + r) * KB;
    auto multiply = [&](int stage, auto do_load, int st_load, int kt_load, int n_chunks) __attribute__((always_inline)) {
        constexpr bool LOAD = decltype(do_load)::value;
        // fragments are read PF k-chunks ahead of the MFMAs that use them: one chunk of MFMAs
        // is shorter than the LDS latency, so a single chunk of lookahead leaves every chunk
        // waiting on its reads
        constexpr int PF = NCH >= 4 ? 2 : 1, SLOTS = PF + 1;
        const unsigned char* base = lds + stage * STAGE;
        u32x4_t fa[SLOTS][TM], fw[SLOTS][TN];
        auto read_frags = [&](int slot, int ch) __attribute__((always_inline)) {
            const int off = (ch * 32) ^ xo;
#pragma unroll
            for (int i = 0; i < TM; ++i) fa[slot][i] = *reinterpret_cast<const u32x4_t*>(base + fragA + i * 64 * KB + off);
#pragma unroll
            for (int j = 0; j < TN; ++j) fw[slot][j] = *reinterpret_cast<const u32x4_t*>(base + fragW + j * 64 * KB + off);
        };
#pragma unroll
        for (int ch = 0; ch < PF; ++ch) read_frags(ch % SLOTS, ch);
#pragma unroll
        for (int ch = 0; ch < NCH; ++ch) {
            if (ch + PF < NCH) read_frags((ch + PF) % SLOTS, ch + PF);
            if (LOAD) {
#pragma unroll
                for (int i = ch * NLOAD / NCH; i < (ch + 1) * NLOAD / NCH; ++i) issue(i, kt_load, st_load);
            }
            if (LOAD || ch < n_chunks) {  // uniform; only the partial last tile has fewer chunks
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j) TR::mma(acc[i][j], fa[ch % SLOTS][i], fw[ch % SLOTS][j]);
                if ((kNorm == NORM_RMS || kNorm == NORM_LAYER) && (ch & 1) == wn) {
#pragma unroll
                    for (int i = 0; i < TM; ++i)
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            ssq[i][e] = add_squares_bf16x2(fa[ch % SLOTS][i][e], ssq[i][e]);
                            if (kNorm == NORM_LAYER) ssum[i][e] = add_pair_bf16x2(fa[ch % SLOTS][i][e], ssum[i][e]);
                        }
                }
            }
            __builtin_amdgcn_sched_barrier(0);  // keeps the reads and loads where they were placed
        }
    };

    // Stage kt % NS holds tile kt.  Before tile kt is multiplied every wavefront waits for
    // its own loads of that tile (the IN_FLIGHT younger ones may still be pending) and all
    // meet at the barrier, which also tells that stage (kt - 1) % NS has been read by
    // everyone: the loads of tile kt + NS - 1 go there.  Past the last tile the ring keeps
    // re-fetching it into free stages, so the counts stay the same to the end.
#pragma unroll
    for (int t = 0; t < NS - 1; ++t)
#pragma unroll
        for (int i = 0; i < NLOAD; ++i) issue(i, min(t, nkt - 1), t);
    int cs = 0, ls = NS - 1;
    for (int kt = 0; kt < nkt_full; ++kt) {
        wait_vmcnt<IN_FLIGHT>();
        __syncthreads();
        multiply(cs, std::true_type{}, ls, min(kt + NS - 1, nkt - 1), NCH);
        cs = (cs + 1 == NS) ? 0 : cs + 1;
        ls = (ls + 1 == NS) ? 0 : ls + 1;
    }
    if (nkt > nkt_full) {
        wait_vmcnt<IN_FLIGHT>();
        __syncthreads();
        multiply(cs, std::false_type{}, 0, 0, (a.K - nkt_full * BK) / 16);
    }
    // The bias columns of every sub-tile's epilogue (thread layout as for the residual) are
    // requested here, while the ring's last loads drain, and not behind each sub-tile's barrier.
    float bias_pf[TN][16] = {};
    if (kEpi == EPI_PLAIN && a.bias != nullptr) {
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e)
                bias_pf[j][e] = a.bias[min((ntw * TN + j) * BN + (e >> 3) * 32 + (tid & 3) * 8 + (e & 7), a.N - 1)];
    }
    wait_vmcnt<0>();  // the re-fetches must have landed before the ring is reused for C
    __syncthreads();

    // The accumulators leave through LDS one 64x64 sub-tile at a time (the epilogue wants whole
    // rows of a sub-tile per thread: rotation partners, 16-byte stores).  Two staging buffers in
    // turn: sub-tile n + 1 is written between the same pair of barriers in which sub-tile n is
    // read, so a sub-tile costs one barrier, and its LDS writes overlap the previous epilogue's
    // memory traffic.
    uint32_t* Cb[2] = {reinterpret_cast<uint32_t*>(lds), reinterpret_cast<uint32_t*>(lds + C_BYTES)};
    float* row_stat = reinterpret_cast<float*>(lds + 2 * C_BYTES);  // [wn][ROWS_A][2]
    if (kNorm == NORM_LAYER_PRE) {
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            float q = 0.f, u = 0.f;
#pragma unroll
            for (int t = 0; t < STAT_MAX_TILES / 4; ++t) {
                const bool on = (tid & 3) + 4 * t < a.n_stat;  // the clamped repeats of the last tile do not count
                q += on ? st_pf[i][t][0] : 0.f;
                u += on ? st_pf[i][t][1] : 0.f;
            }
            q += __uint_as_float(dpp_u32<DPP_XOR1>(__float_as_uint(q)));
            u += __uint_as_float(dpp_u32<DPP_XOR1>(__float_as_uint(u)));
            q += __uint_as_float(dpp_u32<DPP_XOR2>(__float_as_uint(q)));
            u += __uint_as_float(dpp_u32<DPP_XOR2>(__float_as_uint(u)));
            if ((tid & 3) == 0) {  // the epilogue adds two partial pairs per row: the totals and zeros
                float* dst = row_stat + (i * 64 + (tid >> 2)) * 2;
                dst[0] = q;
                dst[1] = u;
                dst[ROWS_A * 2] = 0.f;
                dst[ROWS_A * 2 + 1] = 0.f;
            }
        }
    } else if (kNorm) {
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            float q = (ssq[i][0] + ssq[i][1]) + (ssq[i][2] + ssq[i][3]);
            float u = (ssum[i][0] + ssum[i][1]) + (ssum[i][2] + ssum[i][3]);
            q += __shfl_xor(q, 32, 64);
            u += __shfl_xor(u, 32, 64);
            if (g == 0) {
                float* dst = row_stat + (wn * ROWS_A + (wm + 2 * i) * 32 + r) * 2;
                dst[0] = q;
                dst[1] = u;
            }
        }
    }
    constexpr int NSUB = TM * TN;
    auto stage_c = [&](int n) __attribute__((always_inline)) {
        const int i = n / TN, j = n % TN;
        uint32_t* C = Cb[n & 1];
#pragma unroll
        for (int jj = 0; jj < 4; ++jj)
#pragma unroll
            for (int ii = 0; ii < 4; ++ii)
                C[(wm * 32 + 8 * jj + 4 * g + ii) * C_STRIDE + wn * 32 + r] = acc_bits(acc[i][j][4 * jj + ii]);
    };
    stage_c(0);
#pragma unroll
    for (int n = 0; n < NSUB; ++n) {
        const int i = n / TN, j = n % TN;
        __syncthreads();  // sub-tile n is staged, and the buffer of sub-tile n - 1 has been read by everyone
        if (n + 1 < NSUB) stage_c(n + 1);
        const int nt_sub = ntw * TN + j;
        if (nt_sub < a.n_tiles)
            epilogue_64x64<T, kEpi, kEpi == EPI_PLAIN>(a, Cb[n & 1], m0 + i * 64, nt_sub, tc[j], tid, pf, res_pf[i][j][0],
                                                       res_pf[i][j][1], kNorm == NORM_LAYER_PRE ? NORM_LAYER : kNorm, row_stat + i * 128, ROWS_A * 2, bias_pf[j]);
    }
}

// ---- Few rows of a bf16 projection: narrow tiles over the whole chip ----
// The suffix rows of one or a few observations through a projection.  The weights are read once and from
// memory (a step touches every layer's weights once, more than the caches hold), and what a
// CU gets out of memory is bounded by its own requests in flight and by its path to the L2
// (about 55 bytes per clock), not by the chip: the tiled kernels' 64-column tiles put such a
// launch on N / 64 CUs, a tenth of the chip.  Here a workgroup owns 16 RB rows and 16 NB
// columns, so that a CU moves 32 K (RB + NB) bytes; RB and NB are chosen per shape for the
// fewest bytes per CU (narrow_plan in tile_rules.h).  As in gemm_dl_kernel the operands go straight into an
// LDS ring (128 k per stage, 256-byte rows, pieces XOR-swizzled by the row, NS - 1 stages in
// flight, one barrier per stage): a load instruction covers whole cache lines of four rows.
// Fetching MFMA fragments from memory instead -- 16 rows x 16 bytes per quarter of a wavefront
// -- is limited to about 16 bytes per clock and CU by the address unit, whatever is in flight.
// A wavefront owns whole 16 x 16 blocks over all of K (v_mfma_f32_16x16x32_bf16, ascending k,
// whose sums have the bits of the tiled kernels' 32x32x16: a row's result does not depend on
// the batch it is in); W is the left operand, so that lane (c, q) = (lane % 16, lane / 16) ends
// with columns 4 q .. 4 q + 3 of row c and the epilogue needs no LDS.  The 16 columns are 8 + 8:
// for rotated segments the columns d .. d + 7 of a head and their partners d + D / 2, for gated
// projections 8 gate columns and their up columns (the partner is lane ^ 32), else 16
// consecutive columns.
// Against the tiled kernel (us, weights not in the caches): 16 rows x 1536 x 1536 7.9 -> 4.2, 50 x 720 x 2048
// 9.3 -> 4.7, 50 x 4096 x 720 gated 7.0 -> 4.9, 50 x 1536 x 6144 28.4 -> 11.3.  At 2 to 5 TB/s out of the L2s such a
// launch is mostly its fixed cost: start, first loads, epilogue.
// RB: 16-row blocks, NB: 16-column tiles per workgroup; VEC: outputs and residual four columns at a time, else one by one
template <int kEpi, int kNorm, int RB, int NB, int NS, bool VEC = true>
__global__ void __launch_bounds__(256) gemm_narrow_kernel(GemmArgs a) {
    constexpr int KB = 256, BK = 128, STAGE = (RB + NB) * 16 * KB, NLOAD = RB + NB;
    constexpr int IN_FLIGHT = (NS - 2) * NLOAD;
    static_assert(NB == 1 || RB == 4, "a wavefront per row block; fewer than four repeat each other's products");
    static_assert(IN_FLIGHT <= 63, "ring depth exceeds the vector-memory counter");
    __shared__ __attribute__((aligned(1024))) unsigned char lds[NS * STAGE];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 15, q = lane >> 4;
    const int n_t16 = (a.N + 15) / 16;
    // Workgroup -> (row group, columns).  The row groups of a column group sit eight apart, on
    // one XCD: the second one finds the weight rows in the L2.
    const int n_rg = (a.M + RB * 16 - 1) / (RB * 16);
    const int rg = ((int)blockIdx.x >> 3) % n_rg, tg = (((int)blockIdx.x >> 3) / n_rg) * 8 + ((int)blockIdx.x & 7);
    if (tg * NB >= n_t16) return;
    const int m0 = rg * RB * 16;
    RowCols rc[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) rc[nb] = row_cols<kEpi>(a, min(tg * NB + nb, n_t16 - 1));

    // Loader: thread tid fills slot tid of each 4 KiB slab (16 rows of 256 bytes): position
    // tid % 16 of row tid / 16, which holds logical piece (tid % 16) ^ row.  Rows past M or N and
    // pieces past K are read from valid addresses; their products are dropped or zeroed.
    const int lrow = tid >> 4, koff = ((tid & 15) ^ lrow) * 8;
    const unsigned char* src[NLOAD];
#pragma unroll
    for (int i = 0; i < RB; ++i) src[i] = (const unsigned char*)a.A + (long)min(m0 + i * 16 + lrow, a.M - 1) * a.K * 2;
#pragma unroll
    for (int i = 0; i < NB; ++i)
        src[RB + i] = (const unsigned char*)a.W + (long)min(lrow < 8 ? rc[i].base_lo + lrow : rc[i].base_hi + lrow - 8, a.N - 1) * a.K * 2;
    const uint32_t lds0 = (uint32_t)(uintptr_t)lds + wave * 1024;  // low 32 bits of a shared-aperture address = LDS offset
    const int nkt = (a.K + BK - 1) / BK;
    auto issue = [&](int kt, int stage) __attribute__((always_inline)) {
        const long kb = (long)min(kt * BK + koff, a.K - 8) * 2;
#pragma unroll
        for (int i = 0; i < NLOAD; ++i) load_to_lds16(src[i] + kb, lds0 + stage * STAGE + i * 4096);
    };
#pragma unroll
    for (int t = 0; t < NS - 1; ++t)
        if (t < nkt) issue(t, t);  // uniform

    // wavefront -> row block; each multiplies it with all NB column tiles
    const bool active = wave < RB;
    const int rb = wave % RB;
    f32x4_t acc[NB];
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    // Row sums for the norm, in the tiled kernels' order: lane (c, q) sums its piece of every 32
    // k with one accumulator per word; the pairs q, q ^ 1 are those kernels' two lane halves, the
    // pairs q, q ^ 2 their two wavefronts.
    float ssq[4] = {0.f, 0.f, 0.f, 0.f}, ssum[4] = {0.f, 0.f, 0.f, 0.f};
    const int fx0 = (rb * 16 + c) * KB, fw0 = (RB * 16 + c) * KB;
    auto multiply = [&](int stage, int k_left) __attribute__((always_inline)) {  // k_left: k of this tile inside K (the partial last tile), or BK
        const unsigned char* base = lds + stage * STAGE;
        u32x4_t fx[4], fw[4][NB];
#pragma unroll
        for (int ch = 0; ch < 4; ++ch) {
            const int off = ((4 * ch + q) ^ c) * 16;
            fx[ch] = *reinterpret_cast<const u32x4_t*>(base + fx0 + off);
#pragma unroll
            for (int j = 0; j < NB; ++j) fw[ch][j] = *reinterpret_cast<const u32x4_t*>(base + fw0 + j * 16 * KB + off);
        }
        if (k_left < BK) {  // K is a multiple of 8: a piece is inside or outside as a whole
            const u32x4_t z = {0u, 0u, 0u, 0u};
#pragma unroll
            for (int ch = 0; ch < 4; ++ch)
                if (ch * 32 + 8 * q >= k_left) {
                    fx[ch] = z;
#pragma unroll
                    for (int j = 0; j < NB; ++j) fw[ch][j] = z;
                }
        }
        __builtin_amdgcn_sched_barrier(0);  // all reads requested before the first product: left alone they are spread for fewer registers
#pragma unroll
        for (int ch = 0; ch < 4; ++ch) {
#pragma unroll
            for (int j = 0; j < NB; ++j)
                acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, fw[ch][j]), __builtin_bit_cast(bf16x8_t, fx[ch]),
                                                                 acc[j], 0, 0, 0);
            if (kNorm) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    ssq[e] = add_squares_bf16x2(fx[ch][e], ssq[e]);
                    if (kNorm == NORM_LAYER) ssum[e] = add_pair_bf16x2(fx[ch][e], ssum[e]);
                }
            }
        }
    };
    // A wavefront without a block of its own multiplies along with another's (no branch in the
    // loop) and drops the result.  The last NS - 1 tiles are multiplied without further loads:
    // a ring that kept re-fetching past the end would double the traffic of a short K.
    int cs = 0, ls = NS - 1, kt = 0;
    for (; kt + NS - 1 < nkt; ++kt) {
        wait_vmcnt<IN_FLIGHT>();
        __syncthreads();  // this stage has landed for every wavefront; stage ls has been read by everyone
        issue(kt + NS - 1, ls);
        multiply(cs, BK);
        cs = (cs + 1 == NS) ? 0 : cs + 1;
        ls = (ls + 1 == NS) ? 0 : ls + 1;
    }
    narrow_tail<NS - 1, NLOAD>(nkt, [&](bool last) __attribute__((always_inline)) {
        __syncthreads();
        multiply(cs, last ? a.K - (nkt - 1) * BK : BK);
        cs = (cs + 1 == NS) ? 0 : cs + 1;
    });
    if (!active) return;

    float f = 1.f, ms = 0.f;
    if (kNorm) {
        const float inv_k = 1.0f / (float)a.K;
        const float sq = rows_sum((ssq[0] + ssq[1]) + (ssq[2] + ssq[3]));
        if (kNorm == NORM_LAYER) {
            // sum_k (x - mean) rstd W[n][k] = rstd acc - (mean rstd) colsum[n]
            const float mean = rows_sum((ssum[0] + ssum[1]) + (ssum[2] + ssum[3])) * inv_k;
            f = rsqrtf(fmaxf(sq * inv_k - mean * mean, 0.f) + a.norm_eps);
            ms = mean * f;
        } else {
            f = rsqrtf(sq * inv_k + a.norm_eps);
        }
    }
    const int m = m0 + rb * 16 + c;
#pragma unroll
    for (int j = 0; j < NB; ++j) {
        const RowCols& t = rc[j];
        const bool live = m < a.M && tg * NB + j < n_t16;
        const int n0 = q < 2 ? t.base_lo + 4 * q : t.base_hi + 4 * q - 8;  // W row (= bias, column-sum index) of v[0]
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = acc[j][e];
        if (kNorm == NORM_LAYER) {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = center_scale(v[e], f, ms, a.colsum[min(n0 + e, a.N - 1)]);
        } else if (kNorm) {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] *= f;
        }
        if (a.bias) {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] += a.bias[min(n0 + e, a.N - 1)];
        }
        if (kEpi == EPI_PLAIN) {
            if (a.act != VLA_ACT_NONE) epilogue_act(v, a.act, a.out_bf16);
            if (a.col_gate) {
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] *= a.col_gate[min(n0 + e, a.N - 1)];
            }
            if (!live) continue;
            const long o = (long)m * a.N + n0;
            if (VEC && a.N % 4 == 0) {  // 4 consecutive columns are inside the row or outside as a whole
                if (n0 >= a.N) continue;
                if (a.out_bf16) {
                    if (a.residual) {
                        const u32x2_t rr = *reinterpret_cast<const u32x2_t*>((const bf16_t*)a.residual + o);
#pragma unroll
                        for (int e = 0; e < 2; ++e) {
                            v[2 * e] += __uint_as_float(rr[e] << 16);
                            v[2 * e + 1] += __uint_as_float(rr[e] & 0xffff0000u);
                        }
                    }
                    *reinterpret_cast<u32x2_t*>((bf16_t*)a.Y + o) = u32x2_t{pack_bf2(v[0], v[1]), pack_bf2(v[2], v[3])};
                } else {
                    if (a.residual) {
                        const f32x4_t rr = *reinterpret_cast<const f32x4_t*>((const float*)a.residual + o);
#pragma unroll
                        for (int e = 0; e < 4; ++e) v[e] += rr[e];
                    }
                    *reinterpret_cast<f32x4_t*>((float*)a.Y + o) = f32x4_t{v[0], v[1], v[2], v[3]};
                }
                continue;
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
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
            continue;
        }
        float other[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) other[e] = __shfl_xor(v[e], 32, 64);
        if (kEpi == EPI_GLU) {  // I is a multiple of 32: no column of a tile lies past the row
            if (q >= 2 || !live) continue;
            float y[4] = {v[0], v[1], v[2], v[3]};
            epilogue_act(y, a.act, a.out_bf16);
#pragma unroll
            for (int e = 0; e < 4; ++e) y[e] *= other[e];
            const long o = (long)m * (a.N / 2) + n0;
            if (!VEC) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    if (a.out_bf16) ((bf16_t*)a.Y)[o + e] = f2bf(y[e]);
                    else ((float*)a.Y)[o + e] = y[e];
                }
            } else if (a.out_bf16) {
                *reinterpret_cast<u32x2_t*>((bf16_t*)a.Y + o) = u32x2_t{pack_bf2(y[0], y[1]), pack_bf2(y[2], y[3])};
            } else {
                *reinterpret_cast<f32x4_t*>((float*)a.Y + o) = f32x4_t{y[0], y[1], y[2], y[3]};
            }
            continue;
        }
        // QKV: rotation, scatter
        const int b = min(m, a.M - 1) / a.S, s = min(m, a.M - 1) % a.S;
        if (t.rope) {
            const long ri = (long)s * (a.D >> 1) + (t.col_lo % a.D) + (q & 1) * 4;
            const f32x4_t cr = *reinterpret_cast<const f32x4_t*>(a.cos_t + ri), sr = *reinterpret_cast<const f32x4_t*>(a.sin_t + ri);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float lo = q < 2 ? v[e] : other[e], hi = q < 2 ? other[e] : v[e];
                rotate_pair(lo, hi, cr[e], sr[e]);
                v[e] = q < 2 ? lo : hi;
            }
        }
        if (!live) continue;
        const int col = q < 2 ? t.col_lo + 4 * q : t.col_hi + 4 * q - 8;  // segment-local, 4 consecutive columns of one head
        const u32x2_t pk = {pack_bf2(v[0], v[1]), pack_bf2(v[2], v[3])};
        auto store = [&](bf16_t* dst) __attribute__((always_inline)) {
            if (VEC) {
                *reinterpret_cast<u32x2_t*>(dst) = pk;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) dst[e] = (bf16_t)(pk[e >> 1] >> (16 * (e & 1)));
            }
        };
        if (t.seg == 0) {
            store((bf16_t*)a.q_out + (long)m * (a.Hq * a.D) + col);
        } else {
            const int head = col / a.D, d = col % a.D;
            if (t.seg == 1) {
                store((bf16_t*)a.k_cache + (((long)b * a.Hkv + head) * a.t_max + a.tok_offset + s) * a.D + d);
            } else {
                bf16_t* vt = (bf16_t*)a.vt_cache + (((long)b * a.Hkv + head) * a.D + d) * (long)a.t_max + a.tok_offset + s;
#pragma unroll
                for (int e = 0; e < 4; ++e) vt[(long)e * a.t_max] = (bf16_t)(pk[e >> 1] >> (16 * (e & 1)));
            }
        }
    }
}

// Large-M ternary GEMM (BitVLA prefill: M = batch x prefix tokens).  Workgroup tile
// (64*WM) x 256 with WM x 2 wavefronts, each owning 64 x 128 = 2 x 4 MFMA blocks (128
// accumulator registers), so one 16-byte A fragment feeds four MFMAs and one weight
// fragment two.  int8 activations go global -> registers -> double-buffered LDS (one
// barrier per 128-k tile).  The 2-bit weights never touch LDS: the fragment-major layout
// makes each (32 columns x 32 k) fragment one coalesced 256-byte load per wavefront; a
// word is expanded to bytes with shift/mask right before use and its register is
// refilled at once with the word of the next k-tile, a full tile of MFMAs ahead of need.
template <int WM>
__global__ void __launch_bounds__(WM * 128, 2) ternary_gemm_big_kernel(GemmArgs a) {
    constexpr int NT = WM * 128, ROWS = WM * 64, STRIDE = 144, VA = ROWS * 8 / NT;
    constexpr int T_STRIDE = 272;  // bf16 transpose staging: 128 columns + 16 bytes of padding
    __shared__ __attribute__((aligned(16))) unsigned char lds[2][ROWS * STRIDE];
    static_assert(sizeof(lds) >= (size_t)(WM * 2) * 32 * T_STRIDE, "epilogue staging must fit in the A buffers");

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int g = lane >> 5, r = lane & 31;
    // id % 8 (the XCD) = M tile % 8: workgroups sharing an L2 share their activation rows,
    // the larger operand, and stream the whole (4x smaller) packed weight matrix.
    const int m_tiles = (a.M + ROWS - 1) / ROWS, mt_pad = (m_tiles + 7) & ~7;
    const int mt = blockIdx.x % mt_pad;
    if (mt >= m_tiles) return;
    const int m0 = mt * ROWS, n0 = (blockIdx.x / mt_pad) * 256 + wn * 128;

    const int kgroups = a.K / 32, nblocks = (a.N + 31) / 32;
    const uint32_t* wp[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        int nb = n0 / 32 + j;
        nb = nb < nblocks ? nb : nblocks - 1;  // columns past N: any valid block, result dropped
        wp[j] = (const uint32_t*)a.W + (long)nb * kgroups * 64 + lane;
    }
    const unsigned char* ap[VA];
#pragma unroll
    for (int v = 0; v < VA; ++v) {
        const int idx = tid + v * NT;
        const int m = min(m0 + idx / 8, a.M - 1);  // rows past M: a valid row, result dropped
        ap[v] = (const unsigned char*)a.A + (long)m * a.K + (idx % 8) * 16;
    }

    i32x16_t acc[2][4];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0;

    u32x4_t ra[VA];
    uint32_t bw[4][4];  // [k group of the tile][column block]
    const int nkt = a.K / 128;

#pragma unroll
    for (int ch = 0; ch < 4; ++ch)
#pragma unroll
        for (int j = 0; j < 4; ++j) bw[ch][j] = wp[j][ch * 64];
#pragma unroll
    for (int v = 0; v < VA; ++v) ra[v] = *reinterpret_cast<const u32x4_t*>(ap[v]);
#pragma unroll
    for (int v = 0; v < VA; ++v) {
        const int idx = tid + v * NT;
        *reinterpret_cast<u32x4_t*>(&lds[0][(idx / 8) * STRIDE + (idx % 8) * 16]) = ra[v];
    }
    __syncthreads();

    for (int kt = 0; kt < nkt; ++kt) {
        const unsigned char* cur = lds[kt & 1];
        const int kn = kt + 1 < nkt ? kt + 1 : kt;  // the last tile re-reads itself; copy unused
#pragma unroll
        for (int v = 0; v < VA; ++v) ra[v] = *reinterpret_cast<const u32x4_t*>(ap[v] + (long)kn * 128);
        u32x4_t fa[2][2];
#pragma unroll
        for (int i = 0; i < 2; ++i)
            fa[0][i] = *reinterpret_cast<const u32x4_t*>(cur + (wm * 64 + i * 32 + r) * STRIDE + g * 16);
#pragma unroll
        for (int ch = 0; ch < 4; ++ch) {
            u32x4_t fw[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t w = bw[ch][j];
                fw[j][0] = w & 0x03030303u;
                fw[j][1] = (w >> 2) & 0x03030303u;
                fw[j][2] = (w >> 4) & 0x03030303u;
                fw[j][3] = (w >> 6) & 0x03030303u;
                bw[ch][j] = wp[j][(kn * 4 + ch) * 64];
            }
            if (ch < 3) {
#pragma unroll
                for (int i = 0; i < 2; ++i)
                    fa[(ch + 1) & 1][i] =
                        *reinterpret_cast<const u32x4_t*>(cur + (wm * 64 + i * 32 + r) * STRIDE + (ch + 1) * 32 + g * 16);
            }
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) Traits<int8_t>::mma(acc[i][j], fa[ch & 1][i], fw[j]);
        }
        unsigned char* nxt = lds[(kt + 1) & 1];
#pragma unroll
        for (int v = 0; v < VA; ++v) {
            const int idx = tid + v * NT;
            *reinterpret_cast<u32x4_t*>(nxt + (idx / 8) * STRIDE + (idx % 8) * 16) = ra[v];
        }
        __syncthreads();
    }

    // Accumulator element 4jj+ii of block (i, j) is row 8jj + 4g + ii, column r.
    if (a.acc_out) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int m = m0 + wm * 64 + i * 32 + 8 * (e >> 2) + 4 * g + (e & 3);
                if (m >= a.M) continue;
                const int rs2 = 2 * a.rowsum[m];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int n = n0 + j * 32 + r;
                    if (n < a.N) a.acc_out[(long)m * a.N + n] = acc[i][j][e] - rs2;
                }
            }
    }
    if (!a.Y) return;

    // bf16 output: out = float(acc - 2*rowsum) / s[m] * ws[group], staged per wavefront as
    // 32 rows x 128 columns in LDS and written with 16-byte stores (16 lanes per row).
    const int group = a.N / a.ws_num;
    float wsc[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int n = n0 + j * 32 + r;
        wsc[j] = n < a.N ? a.ws[n / group] : 0.f;
    }
    // The division is the correctly rounded IEEE quotient.  When every scale of the
    // wavefront's 64 rows is far from the exponent limits it is computed as the refinement
    // sequence of the full-range expansion without its operand scaling (identical bits):
    // y ~ 1/s by one Newton step on v_rcp_f32, then q0 = a*y, two residual corrections.
    // Lane l holds the activation scale and the row sum of the wavefront's row l: one coalesced
    // load each.  The loops below pick a row's pair out of these with v_readlane (the row of an
    // accumulator element is a compile-time constant apart from the lane's half g) instead of
    // fetching it from memory where it is needed, which cost a round trip per pair of rows.
    const int lane_row = min(m0 + wm * 64 + lane, a.M - 1);
    const float s_lane = a.s[lane_row];
    const int rs_lane = a.rowsum[lane_row];
    const float sabs = fabsf(s_lane);
    const bool fast = __builtin_amdgcn_ballot_w64(sabs > 0x1p-60f && sabs < 0x1p60f) == ~0ull;
    unsigned char* tp = &lds[0][0] + wave * (32 * T_STRIDE);
    const bool vec_ok = (a.N % 8) == 0;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        // the residual vectors of this half of the rows, requested ahead of the staging arithmetic
        u32x4_t res_v[8] = {};
        const bool res_vec = a.residual != nullptr && vec_ok;
        if (res_vec) {
#pragma unroll
            for (int p = 0; p < 8; ++p) {
                const int m = min(m0 + wm * 64 + i * 32 + p * 4 + (lane >> 4), a.M - 1), n = min(n0 + (lane & 15) * 8, a.N - 8);
                res_v[p] = *reinterpret_cast<const u32x4_t*>((const bf16_t*)a.residual + (long)m * a.N + n);
            }
        }
        if (fast) {
#pragma unroll
            for (int jj = 0; jj < 4; ++jj)
#pragma unroll
                for (int ip = 0; ip < 4; ip += 2) {
                    const int row = 8 * jj + 4 * g + ip;
                    float sm[2], y[2];
                    int rs2[2];
#pragma unroll
                    for (int t = 0; t < 2; ++t) {
                        // row of the wavefront's tile: i * 32 + 8 jj + 4 g + ip + t (rows past M repeat row M - 1, as lane_row does)
                        const int r0 = i * 32 + 8 * jj + ip + t;
                        const int rs_g0 = __builtin_amdgcn_readlane(rs_lane, r0), rs_g1 = __builtin_amdgcn_readlane(rs_lane, r0 + 4);
                        const int sb_g0 = __builtin_amdgcn_readlane(__float_as_int(s_lane), r0);
                        const int sb_g1 = __builtin_amdgcn_readlane(__float_as_int(s_lane), r0 + 4);
                        rs2[t] = 2 * (g ? rs_g1 : rs_g0);
                        sm[t] = __int_as_float(g ? sb_g1 : sb_g0);
                        const float y0 = __builtin_amdgcn_rcpf(sm[t]);
                        y[t] = __builtin_fmaf(__builtin_fmaf(-sm[t], y0, 1.0f), y0, y0);
                    }
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        float o[2];
#pragma unroll
                        for (int t = 0; t < 2; ++t) {
                            const float av = (float)(acc[i][j][4 * jj + ip + t] - rs2[t]);
                            const float q0 = av * y[t];
                            const float q1 = __builtin_fmaf(__builtin_fmaf(-sm[t], q0, av), y[t], q0);
                            o[t] = __builtin_fmaf(__builtin_fmaf(-sm[t], q1, av), y[t], q1) * wsc[j];
                        }
                        const uint32_t pk = pack_bf2(o[0], o[1]);
                        *reinterpret_cast<bf16_t*>(tp + row * T_STRIDE + (j * 32 + r) * 2) = (bf16_t)(pk & 0xffff);
                        *reinterpret_cast<bf16_t*>(tp + (row + 1) * T_STRIDE + (j * 32 + r) * 2) = (bf16_t)(pk >> 16);
                    }
                }
        } else {
#pragma unroll 1
            for (int e = 0; e < 16; ++e) {
                const int row = 8 * (e >> 2) + 4 * g + (e & 3);
                const int mm = min(m0 + wm * 64 + i * 32 + row, a.M - 1);
                const int rs2 = 2 * a.rowsum[mm];
                const float sm = a.s[mm];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    int v = 0;
#pragma unroll
                    for (int e2 = 0; e2 < 16; ++e2) v = (e2 == e) ? acc[i][j][e2] : v;
                    *reinterpret_cast<bf16_t*>(tp + row * T_STRIDE + (j * 32 + r) * 2) =
                        f2bf((float)(v - rs2) / sm * wsc[j]);
                }
            }
        }
#pragma unroll
        for (int p = 0; p < 8; ++p) {
            const int row = p * 4 + (lane >> 4), c16 = lane & 15;
            const u32x4_t v = *reinterpret_cast<const u32x4_t*>(tp + row * T_STRIDE + c16 * 16);
            const int m = m0 + wm * 64 + i * 32 + row, n = n0 + c16 * 8;
            if (m >= a.M) continue;
            bf16_t* dst = (bf16_t*)a.Y + (long)m * a.N + n;
            const bf16_t* res = a.residual ? (const bf16_t*)a.residual + (long)m * a.N + n : nullptr;
            if (vec_ok && n + 8 <= a.N) {
                u32x4_t o = v;
                if (res) {  // out = bf16(out + residual), both already bf16
                    const u32x4_t rr = res_v[p];
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        o[e] = pack_bf2(__uint_as_float(v[e] << 16) + __uint_as_float(rr[e] << 16),
                                        __uint_as_float(v[e] & 0xffff0000u) + __uint_as_float(rr[e] & 0xffff0000u));
                }
                *reinterpret_cast<u32x4_t*>(dst) = o;
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    if (n + e < a.N) {
                        const bf16_t o = (bf16_t)(v[e >> 1] >> (16 * (e & 1)));
                        dst[e] = res ? f2bf(bf2f(o) + bf2f(res[e])) : o;
                    }
            }
        }
    }
}

// ---- Large-M ternary GEMM on v_mfma_i32_16x16x64_i8 (BitVLA prefill) ------------------
// The 16x16x64 form moves a quarter of the accumulator registers per multiply-add that the
// 32x32x32 form does, and on this part that is what the matrix pipe's clock follows: the
// same product streams about a fifth faster.  Everything around the MFMAs is built so that
// nothing the compiler schedules can sit between a load and its first use:
//
//  - int8 activation tiles (128 rows x 128 k) go from global memory straight into a
//    three-stage LDS ring (global_load_lds_dwordx4, rows unpadded, 16-byte pieces
//    XOR-swizzled by (row >> 1) & 7 so that a fragment read touches every bank once);
//  - a wavefront's packed weight words (one dword = 16 codes of one column) go from the
//    fragment-major layout into registers with inline-assembly loads, refilled in place
//    right after they are expanded, a full k-tile ahead of their next use;
//  - both kinds are counted by hand: every pass issues the same loads in the same order,
//    so "the words of this chunk have landed" is always s_waitcnt vmcnt(NB / 2 + 4), and the
//    activation tile of a pass is older than that.  One barrier per k-tile.
//
// The product is formed as D = W . A^T: a lane ends up with four consecutive output
// columns of one row, so the row's scale and row sum are per-lane constants (no lane
// exchange), the accumulators start at -2 * rowsum (the code offset), and the bf16 results
// go to the LDS staging area as 16-byte pieces (a 16-lane group takes the even columns of
// a 32-column block in one MFMA and the odd ones in the next, so that its two weight words
// are one 8-byte load and its eight outputs per row are consecutive).
//
// Registers written by the inline-assembly loads are "in flight" until the matching wait.
// Each of them is an in/out operand of that wait, which keeps the compiler from reading it
// early and from giving the register to anything else in between.  The kernel must not
// spill (a spilled in-flight register is stored before its data arrives and its register
// reused while the load is still due): vla_cpp_amd/build.py checks the scratch size.
template <int IMM>
__device__ __forceinline__ void tern_wload_i(u32x2_t& dst, uint32_t voff, const void* sbase) {
    asm volatile("global_load_dwordx2 %0, %1, %2 offset:%3" : "+v"(dst) : "v"(voff), "s"(sbase), "n"(IMM) : "memory");
}
__device__ __forceinline__ void tern_aload_lds(uint32_t voff, const void* sbase, uint32_t lds_base) {
    load_to_lds16_at(sbase, voff, lds_base);
}
__device__ __forceinline__ void tern_gload(uint32_t& dst, const void* p) {
    asm volatile("global_load_dword %0, %1, off" : "=v"(dst) : "v"(p) : "memory");
}
template <int CNT>
__device__ __forceinline__ void tern_wait_words(u32x2_t (&w)[4]) {
    asm volatile("s_waitcnt vmcnt(%4)" : "+v"(w[0]), "+v"(w[1]), "+v"(w[2]), "+v"(w[3]) : "n"(CNT));
}

// 2 x 2 wavefronts, each 64 rows x 128 columns (4 x 8 blocks of 16 x 16); workgroup tile 128 x 256.
__global__ void __launch_bounds__(256, 2) ternary_gemm_x16_kernel(GemmArgs a) {
    constexpr int NB = 8, MB = 4, NS = 3, ROWS = 128, CW = 16 * NB, COLS = 2 * CW, STAGE = ROWS * 128;
    constexpr int CNT = NB / 2 + 4;    // loads younger than a chunk's words when they are waited for
    constexpr int T_STRIDE = 272;      // staging row: 128 bf16 + 16 bytes
    __shared__ __attribute__((aligned(1024))) unsigned char lds[NS * STAGE];
    static_assert(NS * STAGE >= 4 * 16 * T_STRIDE, "epilogue staging must fit in the ring");

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    const int q = lane >> 4, c = lane & 15;
    int mt, nt;
    if (!xcd_tile(a, (a.N + COLS - 1) / COLS, (a.M + ROWS - 1) / ROWS, mt, nt)) return;
    const int m0 = mt * ROWS, n0 = nt * COLS + wn * CW;

    // Row constants of the lane's four output rows m = m0 + 64 wm + 16 mb + c: requested
    // before everything else, valid after the first wait of the ring.
    uint32_t rs_raw[MB], sc_raw[MB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
        const int m = min(m0 + wm * 64 + mb * 16 + c, a.M - 1);
        tern_gload(rs_raw[mb], a.rowsum + m);
        tern_gload(sc_raw[mb], a.s ? a.s + m : (const float*)(a.rowsum + m));
    }
    // The 16 lanes c of a k quarter q take the columns 2 c (block 2 p) and 2 c + 1 (block 2 p + 1) of the 32-column
    // block n0 / 32 + p: the two words sit side by side in the fragment-major layout (k group 2 chunk + q / 2, half
    // q % 2), one 8-byte load.  Byte offsets; both operands fit 32 bits (checked by the launcher).
    const int kgroups = a.K / 32, nblocks = (a.N + 31) / 32;
    uint32_t woff[NB / 2];
#pragma unroll
    for (int p = 0; p < NB / 2; ++p) {
        const int nb32 = min(n0 / 32 + p, nblocks - 1);  // columns past N: any valid block, result dropped
        woff[p] = ((uint32_t)nb32 * (uint32_t)kgroups * 64u + (uint32_t)((q >> 1) * 64 + (q & 1) * 32 + 2 * c)) * 4u;
    }
    // Activation loader: wavefront w fills the 1 KiB slabs 4 w + v of a stage (8 rows each);
    // the lane's slot is piece position lane % 8 of row lane / 8 and holds logical piece (lane % 8) ^ ((row >> 1) & 7).
    uint32_t aoff[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const int row = (wave * 4 + v) * 8 + (lane >> 3);
        const int piece = (lane & 7) ^ ((row >> 1) & 7);
        aoff[v] = (uint32_t)min(m0 + row, a.M - 1) * (uint32_t)a.K + (uint32_t)(piece * 16);  // rows past M: a valid row, result dropped
    }
    const uint32_t lds0 = (uint32_t)(uintptr_t)lds + wave * 4096;  // low 32 bits of a shared-aperture address = LDS offset

    u32x2_t bw[2][NB / 2] = {};  // [chunk][32-column block]: the words of blocks 2 p and 2 p + 1
    const int nkt = a.K / 128;
    const unsigned char* Ab = (const unsigned char*)a.A;
    const unsigned char* Wb = (const unsigned char*)a.W;
#define TERN_WLOAD(ch, base) \
    _Pragma("unroll") for (int p = 0; p < NB / 2; ++p) tern_wload_i<(ch) * 512>(bw[ch][p], woff[p], base);
#define TERN_ALOAD(ch, abase, lbase)                                   \
    tern_aload_lds(aoff[(ch) * 2], abase, (lbase) + ((ch) * 2) * 1024); \
    tern_aload_lds(aoff[(ch) * 2 + 1], abase, (lbase) + ((ch) * 2 + 1) * 1024);

    // Prologue = the issue order of two passes before the first: activation tile 0, then
    // (words of tile 0, activation tile 1) chunk by chunk.  Past the last tile the ring
    // keeps re-fetching it, so the counts stay the same to the end.
#pragma unroll
    for (int v = 0; v < 4; ++v) tern_aload_lds(aoff[v], Ab, lds0 + v * 1024);
    {
        const unsigned char* a1 = Ab + (long)min(1, nkt - 1) * 128;
        TERN_WLOAD(0, Wb) TERN_ALOAD(0, a1, lds0 + STAGE)
        TERN_WLOAD(1, Wb) TERN_ALOAD(1, a1, lds0 + STAGE)
    }
    // Fragment reads: row 64 wm + 16 mb + c, logical piece 4 ch + q at position (4 ch + q) ^ ((c >> 1) & 7).
    const int fsw = (c >> 1) & 7;
    const int fragA = (wm * 64 + c) * 128;

    // Words of (tile 0, chunk 0) have landed, and with them everything older: activation tile 0 and the row constants.
    tern_wait_words<CNT>(bw[0]);
    asm volatile("" : "+v"(rs_raw[0]), "+v"(rs_raw[1]), "+v"(rs_raw[2]), "+v"(rs_raw[3]), "+v"(sc_raw[0]), "+v"(sc_raw[1]), "+v"(sc_raw[2]), "+v"(sc_raw[3]));
    i32x4_t acc[NB][MB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
        const int init = -2 * (int)rs_raw[mb];  // 2-bit codes are t + 2: sum_k q (t + 2) - 2 rowsum
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) acc[nb][mb] = i32x4_t{init, init, init, init};
    }
    int cs = 0, ls = 2;
    for (int kt = 0; kt < nkt; ++kt) {
        const unsigned char* cur = lds + cs * STAGE;
        const unsigned char* wn_base = Wb + (long)min(kt + 1, nkt - 1) * 1024;
        const unsigned char* an_base = Ab + (long)min(kt + 2, nkt - 1) * 128;
        const uint32_t lds_ld = lds0 + ls * STAGE;
        u32x4_t fa[2][MB];
        __syncthreads();  // every wavefront's loads of this tile have landed; stage ls has been read by everyone
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
            fa[0][mb] = *reinterpret_cast<const u32x4_t*>(cur + fragA + mb * 16 * 128 + ((q ^ fsw) * 16));
#pragma unroll
        for (int ch = 0; ch < 2; ++ch) {
            if (ch > 0) tern_wait_words<CNT>(bw[ch]);
            u32x4_t fw[NB];
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) {
                const uint32_t w = bw[ch][nb >> 1][nb & 1];
                fw[nb][0] = w & 0x03030303u;
                fw[nb][1] = (w >> 2) & 0x03030303u;
                fw[nb][2] = (w >> 4) & 0x03030303u;
                fw[nb][3] = (w >> 6) & 0x03030303u;
            }
            // refill the words just expanded with the next k-tile's, then two activation slabs of the tile after that
            if (ch == 0) { TERN_WLOAD(0, wn_base) TERN_ALOAD(0, an_base, lds_ld) }
            if (ch == 1) { TERN_WLOAD(1, wn_base) TERN_ALOAD(1, an_base, lds_ld) }
            if (ch == 0) {
#pragma unroll
                for (int mb = 0; mb < MB; ++mb)
                    fa[1][mb] = *reinterpret_cast<const u32x4_t*>(cur + fragA + mb * 16 * 128 + (((4 + q) ^ fsw) * 16));
            }
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                for (int mb = 0; mb < MB; ++mb)
                    acc[nb][mb] = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(i32x4_t, fw[nb]),
                                                                        __builtin_bit_cast(i32x4_t, fa[ch][mb]), acc[nb][mb], 0, 0, 0);
        }
        tern_wait_words<CNT>(bw[0]);  // the next tile's first chunk (and, older than it, the next activation tile)
        cs = (cs + 1 == NS) ? 0 : cs + 1;
        ls = (ls + 1 == NS) ? 0 : ls + 1;
    }
#undef TERN_WLOAD
#undef TERN_ALOAD
    // the ring's trailing loads (repeats of the last tile) still target the word registers and the LDS stages
    asm volatile("s_waitcnt vmcnt(0)"
                 : "+v"(bw[0][0]), "+v"(bw[0][1]), "+v"(bw[0][2]), "+v"(bw[0][3]), "+v"(bw[1][0]), "+v"(bw[1][1]), "+v"(bw[1][2]), "+v"(bw[1][3]));
    __syncthreads();

    // acc[nb][mb][i]: column n = n0 + 32 (nb / 2) + 2 (4 q + i) + nb % 2, row m = m0 + 64 wm + 16 mb + c
    if (a.acc_out) {
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
            const int m = m0 + wm * 64 + mb * 16 + c;
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int n = n0 + (nb >> 1) * 32 + 2 * (4 * q + i) + (nb & 1);
                    if (m < a.M && n < a.N) a.acc_out[(long)m * a.N + n] = acc[nb][mb][i];
                }
        }
    }
    if (!a.Y) return;

    // bf16 output: out = float(acc) / s[m] * ws[group], staged per wavefront as 16 rows x 128
    // columns and written with 16-byte stores (16 lanes per row), the residual added on the way.
    // The quotient is the correctly rounded one.  For a positive scale away from the exponent
    // limits it is computed with the scale's exponent taken out: y ~ 1 / mantissa by one Newton
    // step on v_rcp_f32, q0 = a y, one residual correction; for |a| < 2^20 that sequence gives
    // the IEEE quotient for every mantissa (checked exhaustively on the device), and the power
    // of two goes back in exactly.  Larger accumulators take a second correction (the compiler's
    // own sequence without its operand scaling); other scales take the division operator.
    const int group = a.N / a.ws_num;
    float wsc[NB / 2];  // one weight scale per 32-column block (the launcher checks that a scale group is a multiple of 32 columns)
    bool ok = true;
#pragma unroll
    for (int p = 0; p < NB / 2; ++p) {
        wsc[p] = a.ws[min(n0 + p * 32, a.N - 1) / group];
        const float wa = fabsf(wsc[p]);
        ok = ok && (wa == 0.f || (wa > 0x1p-60f && wa < 0x1p60f));  // 2^-e ws below is then exact
    }
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
        const float sm = __uint_as_float(sc_raw[mb]);
        ok = ok && sm > 0x1p-60f && sm < 0x1p60f;
    }
    const bool fast = __builtin_amdgcn_ballot_w64(ok) == ~0ull;
    const bool one_step = a.K < 8192;  // |acc| <= 128 K < 2^20
    unsigned char* tp = &lds[0] + wave * (16 * T_STRIDE);
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
        u32x4_t res_v[4] = {};
        if (a.residual) {  // this row block's residual vectors, requested ahead of the staging arithmetic
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                const int m = min(m0 + wm * 64 + mb * 16 + p * 4 + (lane >> 4), a.M - 1), n = min(n0 + (lane & 15) * 8, a.N - 8);
                res_v[p] = *reinterpret_cast<const u32x4_t*>((const bf16_t*)a.residual + (long)m * a.N + n);
            }
        }
        const float sm = __uint_as_float(sc_raw[mb]);
        if (fast) {
            const uint32_t sb = sc_raw[mb];
            const float mant = __uint_as_float((sb & 0x007fffffu) | 0x3f800000u);      // in [1, 2)
            const float pw = __uint_as_float(0x7f000000u - (sb & 0x7f800000u));         // 2^-(exponent of sm), exact
            const float y0 = __builtin_amdgcn_rcpf(mant);
            const float y = __builtin_fmaf(__builtin_fmaf(-mant, y0, 1.0f), y0, y0);
#pragma unroll
            for (int p = 0; p < NB / 2; ++p) {
                const float pws = pw * wsc[p];  // exact: (q 2^-e) ws and q (2^-e ws) round the same product once
                u32x4_t o;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    float r2[2];
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const float av = (float)acc[2 * p + h][mb][i];
                        const float q0 = av * y;
                        float q1 = __builtin_fmaf(__builtin_fmaf(-mant, q0, av), y, q0);
                        if (!one_step) q1 = __builtin_fmaf(__builtin_fmaf(-mant, q1, av), y, q1);
                        r2[h] = q1 * pws;
                    }
                    o[i] = pack_bf2(r2[0], r2[1]);
                }
                *reinterpret_cast<u32x4_t*>(tp + c * T_STRIDE + (p * 32 + 8 * q) * 2) = o;
            }
        } else {
#pragma unroll
            for (int p = 0; p < NB / 2; ++p) {
                u32x4_t o;
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    o[i] = pack_bf2((float)acc[2 * p][mb][i] / sm * wsc[p], (float)acc[2 * p + 1][mb][i] / sm * wsc[p]);
                *reinterpret_cast<u32x4_t*>(tp + c * T_STRIDE + (p * 32 + 8 * q) * 2) = o;
            }
        }
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            const int row = p * 4 + (lane >> 4), c16 = lane & 15;
            u32x4_t v = *reinterpret_cast<const u32x4_t*>(tp + row * T_STRIDE + c16 * 16);
            const int m = m0 + wm * 64 + mb * 16 + row, n = n0 + c16 * 8;
            if (m >= a.M || n + 8 > a.N) continue;
            if (a.residual) {  // out = bf16(out + residual), both already bf16
                const u32x4_t rr = res_v[p];
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    v[e] = pack_bf2(__uint_as_float(v[e] << 16) + __uint_as_float(rr[e] << 16),
                                    __uint_as_float(v[e] & 0xffff0000u) + __uint_as_float(rr[e] & 0xffff0000u));
            }
            // streaming store: the 2 M N bytes leave the L2 as they are produced instead of waiting, dirty, for the
            // write-back at the end of the kernel (each XCD's L2 would hold its whole share until then)
            __builtin_nontemporal_store(v, reinterpret_cast<u32x4_t*>((bf16_t*)a.Y + (long)m * a.N + n));
        }
    }
}

// ---- Ternary GEMM, both operands through an LDS ring ----------------------------------
// 2 x 2 wavefronts, each 16 MB rows x 16 NB columns of 16 x 16 x 64 products (transposed, D = W .
// A^T, as above): workgroup tile 32 MB x 32 NB.  A stage of the ring holds 128 k of the activation
// rows (pieces XOR-swizzled by (row >> 1) & 7) and the packed words of the same 128 k, 1 KiB per
// 32-column block, copied as they lie in the fragment-major layout; a lane's two words of a block
// are one 8-byte read.  NS - 1 stages are in flight, one barrier per stage.  For a few hundred rows
// (one observation's prefix) the 128 x 256 tiles above leave most of the chip idle -- 40 of 256
// CUs at 512 x 2560 -- and a wavefront alone on its SIMD waits for every load it makes.  Bound by
// the L2 -> CU fill (about 10 TB/s over the chip) below 128 x 128.  512 rows, M x N x K: 512 x 3840 x
// 2560 19.0 -> 9.9 us, 512 x 2560 x 2560 20.5 -> 9.6, 512 x 13824 x 2560 34.2 -> 21.9, 512 x 2560 x
// 6912 33.8 -> 17.1 (64 x 64 tiles with the words staged through registers before).
template <int MB, int NB, int NS>
__global__ void __launch_bounds__(256) ternary_gemm_ring_kernel(GemmArgs a) {
    constexpr int ROWS = 32 * MB, CW = 16 * NB, COLS = 2 * CW, ABYTES = ROWS * 128, STAGE = ABYTES + NB * 1024;
    constexpr int WL = NB >= 4 ? NB / 4 : 1, NLOAD = MB + WL;  // load instructions per wavefront and stage: activations, words
    constexpr int T_STRIDE = 2 * CW + 16;                      // epilogue staging row: CW bf16 + 16 bytes
    constexpr int LPR = CW / 8, RPP = 64 / LPR, PASSES = 16 / RPP;  // 16-byte pieces of a staging row, rows per store pass, passes
    static_assert((NS - 2) * NLOAD <= 63, "ring depth exceeds the vector-memory counter");
    static_assert(NS * STAGE >= 4 * 16 * T_STRIDE, "epilogue staging must fit in the ring");
    __shared__ __attribute__((aligned(1024))) unsigned char lds[NS * STAGE];

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    const int q = lane >> 4, c = lane & 15;
    int mt, nt;
    if (!xcd_tile(a, (a.N + COLS - 1) / COLS, (a.M + ROWS - 1) / ROWS, mt, nt)) return;
    const int m0 = mt * ROWS, n0 = nt * COLS + wn * CW;

    // Loader: wavefront w fills the activation slabs MB w + v (8 rows, 1 KiB each) and the word
    // slabs WL w + v (one 32-column block each; with two blocks the wavefronts 2 and 3 repeat them).
    const int kgroups = a.K / 32, nblocks = (a.N + 31) / 32, nkt = a.K / 128;
    const unsigned char* src[NLOAD];
#pragma unroll
    for (int v = 0; v < MB; ++v) {
        const int row = (wave * MB + v) * 8 + (lane >> 3), piece = (lane & 7) ^ ((row >> 1) & 7);
        src[v] = (const unsigned char*)a.A + (long)min(m0 + row, a.M - 1) * a.K + piece * 16;  // rows past M: a valid row, result dropped
    }
#pragma unroll
    for (int v = 0; v < WL; ++v)  // columns past N: any valid block, result dropped
        src[MB + v] = (const unsigned char*)a.W + (long)min(nt * NB + (wave * WL + v) % NB, nblocks - 1) * kgroups * 256 + lane * 16;
    const uint32_t lds0 = (uint32_t)(uintptr_t)lds;  // low 32 bits of a shared-aperture address = LDS offset
    auto issue = [&](int kt, int stage) __attribute__((always_inline)) {
#pragma unroll
        for (int v = 0; v < MB; ++v) load_to_lds16(src[v] + (long)kt * 128, lds0 + stage * STAGE + (wave * MB + v) * 1024);
#pragma unroll
        for (int v = 0; v < WL; ++v) load_to_lds16(src[MB + v] + (long)kt * 1024, lds0 + stage * STAGE + ABYTES + ((wave * WL + v) % NB) * 1024);
    };
#pragma unroll
    for (int t = 0; t < NS - 1; ++t)
        if (t < nkt) issue(t, t);  // uniform

    i32x4_t acc[NB][MB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) acc[nb][mb] = i32x4_t{0, 0, 0, 0};
    // Fragment reads: row 16 MB wm + 16 mb + c, logical piece 4 ch + q at position (4 ch + q) ^ ((c >> 1) & 7); words
    // (k group 2 ch + q / 2, half q % 2, columns 2 c and 2 c + 1) of block wn NB / 2 + p.
    const int fsw = (c >> 1) & 7;
    const int fragA = (wm * MB * 16 + c) * 128, fragW = ABYTES + wn * (NB / 2) * 1024 + ((q >> 1) * 64 + (q & 1) * 32 + 2 * c) * 4;
    auto multiply = [&](int stage) __attribute__((always_inline)) {
        const unsigned char* cur = lds + stage * STAGE;
        u32x4_t fa[2][MB];
        u32x2_t w[2][NB / 2];
#pragma unroll
        for (int ch = 0; ch < 2; ++ch) {
#pragma unroll
            for (int p = 0; p < NB / 2; ++p) w[ch][p] = *reinterpret_cast<const u32x2_t*>(cur + fragW + p * 1024 + ch * 512);
#pragma unroll
            for (int mb = 0; mb < MB; ++mb)
                fa[ch][mb] = *reinterpret_cast<const u32x4_t*>(cur + fragA + mb * 16 * 128 + (((4 * ch + q) ^ fsw) * 16));
        }
        __builtin_amdgcn_sched_barrier(0);  // all reads requested before the first product
#pragma unroll
        for (int ch = 0; ch < 2; ++ch)
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) {
                const uint32_t x = w[ch][nb >> 1][nb & 1];
                const u32x4_t fw = {x & 0x03030303u, (x >> 2) & 0x03030303u, (x >> 4) & 0x03030303u, (x >> 6) & 0x03030303u};
#pragma unroll
                for (int mb = 0; mb < MB; ++mb)
                    acc[nb][mb] = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(i32x4_t, fw), __builtin_bit_cast(i32x4_t, fa[ch][mb]),
                                                                        acc[nb][mb], 0, 0, 0);
            }
    };
    int cs = 0, ls = NS - 1, kt = 0;
    for (; kt + NS - 1 < nkt; ++kt) {
        wait_vmcnt<(NS - 2) * NLOAD>();
        __syncthreads();  // this stage has landed for every wavefront; stage ls has been read by everyone
        issue(kt + NS - 1, ls);
        multiply(cs);
        cs = (cs + 1 == NS) ? 0 : cs + 1;
        ls = (ls + 1 == NS) ? 0 : ls + 1;
    }
    // the row constants of the epilogue (rows m0 + 16 MB wm + 16 mb + c), under the last tiles
    int rs_row[MB];
    float sc_row[MB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
        const int m = min(m0 + (wm * MB + mb) * 16 + c, a.M - 1);
        rs_row[mb] = a.rowsum[m];
        sc_row[mb] = a.s ? a.s[m] : 1.f;
    }
    narrow_tail<NS - 1, NLOAD>(nkt, [&](bool) __attribute__((always_inline)) {
        __syncthreads();
        multiply(cs);
        cs = (cs + 1 == NS) ? 0 : cs + 1;
    });
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)  // 2-bit codes are t + 2: sum_k q (t + 2) - 2 rowsum
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[nb][mb][i] -= 2 * rs_row[mb];
    __syncthreads();  // the ring becomes the epilogue's staging area

    // acc[nb][mb][i]: column n = n0 + 32 (nb / 2) + 2 (4 q + i) + nb % 2, row m = m0 + 16 MB wm + 16 mb + c
    if (a.acc_out) {
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
            const int m = m0 + (wm * MB + mb) * 16 + c;
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int n = n0 + (nb >> 1) * 32 + 2 * (4 * q + i) + (nb & 1);
                    if (m < a.M && n < a.N) a.acc_out[(long)m * a.N + n] = acc[nb][mb][i];
                }
        }
    }
    if (!a.Y) return;

    // bf16 output: out = float(acc) / s[m] * ws[group], staged per wavefront as 16 rows x CW
    // columns and written with 16-byte stores (LPR lanes per row), the residual added on the way.
    // The quotient is the correctly rounded one.  For a positive scale away from the exponent
    // limits it is computed with the scale's exponent taken out: y ~ 1 / mantissa by one Newton
    // step on v_rcp_f32, q0 = a y, one residual correction; for |a| < 2^20 that sequence gives
    // the IEEE quotient for every mantissa (checked exhaustively on the device), and the power
    // of two goes back in exactly.  Larger accumulators take a second correction (the compiler's
    // own sequence without its operand scaling); other scales take the division operator.
    const int group = a.N / a.ws_num;
    float wsc[NB / 2];  // one weight scale per 32-column block (the launcher checks that a scale group is a multiple of 32 columns)
    bool ok = true;
#pragma unroll
    for (int p = 0; p < NB / 2; ++p) {
        wsc[p] = a.ws[min(n0 + p * 32, a.N - 1) / group];
        const float wa = fabsf(wsc[p]);
        ok = ok && (wa == 0.f || (wa > 0x1p-60f && wa < 0x1p60f));  // 2^-e ws below is then exact
    }
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
        const float sm = sc_row[mb];
        ok = ok && sm > 0x1p-60f && sm < 0x1p60f;
    }
    const bool fast = __builtin_amdgcn_ballot_w64(ok) == ~0ull;
    const bool one_step = a.K < 8192;  // |acc| <= 128 K < 2^20
    unsigned char* tp = &lds[0] + wave * (16 * T_STRIDE);
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
        u32x4_t res_v[PASSES] = {};
        if (a.residual) {  // this row block's residual vectors, requested ahead of the staging arithmetic
#pragma unroll
            for (int p = 0; p < PASSES; ++p) {
                const int m = min(m0 + (wm * MB + mb) * 16 + p * RPP + lane / LPR, a.M - 1), n = min(n0 + (lane % LPR) * 8, a.N - 8);
                res_v[p] = *reinterpret_cast<const u32x4_t*>((const bf16_t*)a.residual + (long)m * a.N + n);
            }
        }
        const float sm = sc_row[mb];
        if (fast) {
            const uint32_t sb = __float_as_uint(sc_row[mb]);
            const float mant = __uint_as_float((sb & 0x007fffffu) | 0x3f800000u);      // in [1, 2)
            const float pw = __uint_as_float(0x7f000000u - (sb & 0x7f800000u));         // 2^-(exponent of sm), exact
            const float y0 = __builtin_amdgcn_rcpf(mant);
            const float y = __builtin_fmaf(__builtin_fmaf(-mant, y0, 1.0f), y0, y0);
#pragma unroll
            for (int p = 0; p < NB / 2; ++p) {
                const float pws = pw * wsc[p];  // exact: (q 2^-e) ws and q (2^-e ws) round the same product once
                u32x4_t o;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    float r2[2];
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const float av = (float)acc[2 * p + h][mb][i];
                        const float q0 = av * y;
                        float q1 = __builtin_fmaf(__builtin_fmaf(-mant, q0, av), y, q0);
                        if (!one_step) q1 = __builtin_fmaf(__builtin_fmaf(-mant, q1, av), y, q1);
                        r2[h] = q1 * pws;
                    }
                    o[i] = pack_bf2(r2[0], r2[1]);
                }
                *reinterpret_cast<u32x4_t*>(tp + c * T_STRIDE + (p * 32 + 8 * q) * 2) = o;
            }
        } else {
#pragma unroll
            for (int p = 0; p < NB / 2; ++p) {
                u32x4_t o;
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    o[i] = pack_bf2((float)acc[2 * p][mb][i] / sm * wsc[p], (float)acc[2 * p + 1][mb][i] / sm * wsc[p]);
                *reinterpret_cast<u32x4_t*>(tp + c * T_STRIDE + (p * 32 + 8 * q) * 2) = o;
            }
        }
#pragma unroll
        for (int p = 0; p < PASSES; ++p) {
            const int row = p * RPP + lane / LPR, c16 = lane % LPR;
            u32x4_t v = *reinterpret_cast<const u32x4_t*>(tp + row * T_STRIDE + c16 * 16);
            const int m = m0 + (wm * MB + mb) * 16 + row, n = n0 + c16 * 8;
            if (m >= a.M || n + 8 > a.N) continue;
            if (a.residual) {  // out = bf16(out + residual), both already bf16
                const u32x4_t rr = res_v[p];
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    v[e] = pack_bf2(__uint_as_float(v[e] << 16) + __uint_as_float(rr[e] << 16),
                                    __uint_as_float(v[e] & 0xffff0000u) + __uint_as_float(rr[e] & 0xffff0000u));
            }
            // streaming store: the 2 M N bytes leave the L2 as they are produced instead of waiting, dirty, for the
            // write-back at the end of the kernel (each XCD's L2 would hold its whole share until then)
            __builtin_nontemporal_store(v, reinterpret_cast<u32x4_t*>((bf16_t*)a.Y + (long)m * a.N + n));
        }
    }
}

// Ternary GEMV for a handful of rows (single-token decode, M <= 32).  A workgroup owns 32
// output columns; its 8 wavefronts each take one eighth of K and multiply it with
// v_mfma_i32_32x32x32_i8 as C[n][m] = sum_k W[n][k] * A[m][k] (weight fragment as the A
// operand: one coalesced 256-byte load per 32 k; activation rows as the B operand, lanes
// past M feed zeros).  Every load of a wavefront's slice is issued before the first is
// used; the eight partial 32 x 32 int32 tiles are summed through LDS (exact) and the
// epilogue of the tiled kernels follows, with an optional bf16 residual add.
constexpr int GEMV_WAVES = 8;
template <int MAXG>  // k groups of 32 per wavefront held in registers: K <= 256 * MAXG
__global__ void __launch_bounds__(GEMV_WAVES * 64) ternary_gemv_kernel(GemmArgs a) {
    __shared__ int part[GEMV_WAVES][32][33];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int g = lane >> 5, r = lane & 31;
    const int nb = blockIdx.x;                       // 32-column block
    const int kgroups = a.K / 32;
    const int per_wave = (kgroups + GEMV_WAVES - 1) / GEMV_WAVES;
    const int kg0 = wave * per_wave, kg1 = min(kgroups, kg0 + per_wave);
    const uint32_t* wp = (const uint32_t*)a.W + (long)nb * kgroups * 64 + lane;
    const bool row_ok = r < a.M;
    const unsigned char* ap = (const unsigned char*)a.A + (long)(row_ok ? r : 0) * a.K + g * 16;

    uint32_t wv[MAXG];
    u32x4_t av[MAXG];
#pragma unroll
    for (int i = 0; i < MAXG; ++i) {
        const int kg = min(kg0 + i, kgroups - 1);    // past the slice: a valid group, not multiplied
        wv[i] = wp[(long)kg * 64];
        av[i] = *reinterpret_cast<const u32x4_t*>(ap + kg * 32);
    }
    i32x16_t acc;
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[e] = 0;
#pragma unroll
    for (int i = 0; i < MAXG; ++i) {
        if (kg0 + i < kg1) {                         // uniform
            const uint32_t w = wv[i];
            const u32x4_t fw = {w & 0x03030303u, (w >> 2) & 0x03030303u, (w >> 4) & 0x03030303u, (w >> 6) & 0x03030303u};
            const u32x4_t z = {0u, 0u, 0u, 0u};
            Traits<int8_t>::mma(acc, fw, row_ok ? av[i] : z);
        }
    }
    // element 4j+i of lane (g, r) is C[n = 8j + 4g + i][m = r]
#pragma unroll
    for (int e = 0; e < 16; ++e) part[wave][8 * (e >> 2) + 4 * g + (e & 3)][r] = acc[e];
    __syncthreads();
    // thread -> (m, n): 512 threads cover 16 rows x 32 columns per pass, n fastest
    const int group = a.N / a.ws_num;
    for (int m = tid >> 5; m < a.M; m += GEMV_WAVES * 2) {
        const int nl = tid & 31, n = nb * 32 + nl;
        if (n >= a.N) continue;
        int v = 0;
#pragma unroll
        for (int w = 0; w < GEMV_WAVES; ++w) v += part[w][nl][m];
        v -= 2 * a.rowsum[m];
        if (a.acc_out) a.acc_out[(long)m * a.N + n] = v;
        if (a.Y) {
            bf16_t o = f2bf((float)v / (a.s ? a.s[m] : 1.f) * a.ws[n / group]);
            if (a.residual) o = f2bf(bf2f(o) + bf2f(((const bf16_t*)a.residual)[(long)m * a.N + n]));
            ((bf16_t*)a.Y)[(long)m * a.N + n] = o;
        }
    }
}

// The same GEMV with the producer of its activations inside: A holds the bf16 rows before
// RMSNorm, and wavefront w of every workgroup normalises and quantises row w (the code of
// the stand-alone kernel, so the bits are the same) into LDS while the weight loads are in
// flight.  Saves the separate norm + quantise launch in front of each decode projection
// (bitvla.cpp's attn_norm -> QKV and sub_norm -> O pairs).  M <= GEMV_WAVES, K <= 512 NV.
//
// ROPE: the fused Q | K | V projection of one appended token per batch row, with the split,
// the NeoX rotation and the cache append of qkv_split_rope_append_kernel in the epilogue.  The
// weight rows are in "paired" order (vla_ternary_pair_rope_rows_host): inside the Q and K
// columns every 32-row block holds 16 rotation pairs, d in lanes 0-15 and d + D/2 in lanes
// 16-31, so a pair meets through one shuffle.  The projection is rounded to bf16 before the
// rotation, as the stand-alone chain stores it.
//
// GLU: A is a fused [gate | up] projection of 2 K columns and the rows are relu(gate)^2 * up
// (the FFN's sub-norm -> down projection step, bitvla_lm_cuda.cu:505-517).
constexpr int GEMV_FUSED_MAX_K = 7168;
template <int MAXG, int NV, bool ROPE, bool GLU = false>
__global__ void __launch_bounds__(GEMV_WAVES * 64) ternary_gemv_norm_kernel(GemmArgs a) {
    // int8 rows (stride K + 32 bytes: eight rows' 16-byte fragments fall on distinct banks),
    // later the partial accumulator tiles
    constexpr int KMAX = NV * 512 < GEMV_FUSED_MAX_K ? NV * 512 : GEMV_FUSED_MAX_K;
    constexpr int kPartBytes = GEMV_WAVES * 32 * 33 * 4, kRowBytes = GEMV_WAVES * (KMAX + 32);
    __shared__ __align__(16) unsigned char smem[kPartBytes > kRowBytes ? kPartBytes : kRowBytes];
    __shared__ float s_sh[GEMV_WAVES];
    __shared__ int rs_sh[GEMV_WAVES];
    int (*part)[32][33] = reinterpret_cast<int (*)[32][33]>(smem);
    // Every kernel argument the launch will need, fetched in one batch at its start: left to the compiler the ones of
    // the epilogue are requested where they are first used, a second wait for the scalar cache in the middle of a
    // launch that is one chain of dependent steps.
    asm volatile("" ::"s"(a.A), "s"(a.W), "s"(a.norm_w), "s"(a.ws), "s"(a.q_out), "s"(a.k_cache), "s"(a.vt_cache), "s"(a.cos_t),
                 "s"(a.sin_t), "s"(a.residual), "s"(a.Y), "s"(a.t_max), "s"(a.tok_offset), "s"(a.Hkv), "s"(a.D), "s"(a.K), "s"(a.N),
                 "s"(a.M));
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int g = lane >> 5, r = lane & 31;
    const int nb = blockIdx.x;
    const int kgroups = a.K / 32;
    const int per_wave = (kgroups + GEMV_WAVES - 1) / GEMV_WAVES;
    const int kg0 = wave * per_wave, kg1 = min(kgroups, kg0 + per_wave);
    const uint32_t* wp = (const uint32_t*)a.W + (long)nb * kgroups * 64 + lane;
    const int stride = a.K + 32;

    uint32_t wv[MAXG];
#pragma unroll
    for (int i = 0; i < MAXG; ++i) wv[i] = wp[(long)min(kg0 + i, kgroups - 1) * 64];
    // What the epilogue reads from memory is fetched now, behind the weight loads, instead of
    // after the last barrier where nothing is left to hide a round trip to memory.  Epilogue
    // thread -> (row em = tid / 32, column en): M <= GEMV_WAVES, so one pass covers every row.
    const int group = a.N / a.ws_num;
    const int em = tid >> 5, enl = tid & 31, en = nb * 32 + enl;
    // (no branch around any of these loads: addresses are clamped into the arrays instead, and
    // a value that is not needed is dropped -- a load under a branch is waited for at the join,
    // together with every load issued before it)
    const bool e_ok = em < a.M && en < a.N;
    const int ec = min(en, a.N - 1), emc = min(em, a.M - 1);
    const float ws_pf = a.ws[ec / group];
    bf16_t res_pf = 0;
    float cos_pf = 0.f, sin_pf = 0.f;
    if constexpr (ROPE) {
        const int pi = 16 * ((ec % a.D) >> 5) + (enl & 15);  // < D / 2 for every column
        cos_pf = a.cos_t[pi];
        sin_pf = a.sin_t[pi];
    } else {
        // without a residual: the first element of the activations, dropped in the epilogue
        const bf16_t* rp = a.residual ? (const bf16_t*)a.residual + (long)emc * a.N + ec : (const bf16_t*)a.A;
        res_pf = *rp;
    }
    if (wave < a.M) {  // uniform per wavefront
        float scale;
        int sum;
        rms_act_quant_row<NV, GLU>((const bf16_t*)a.A + (long)wave * a.K * (GLU ? 2 : 1), (const bf16_t*)a.norm_w, a.K,
                                   a.norm_eps, lane, (int8_t*)smem + wave * stride, scale, sum);
        if (lane == 0) {
            s_sh[wave] = scale;
            rs_sh[wave] = sum;
        }
    }
    __syncthreads();
    const bool row_ok = r < a.M;
    const unsigned char* ap = smem + (row_ok ? r : 0) * stride + g * 16;
    u32x4_t av[MAXG];
#pragma unroll
    for (int i = 0; i < MAXG; ++i) av[i] = *reinterpret_cast<const u32x4_t*>(ap + min(kg0 + i, kgroups - 1) * 32);
    __syncthreads();  // the rows are in registers: the partial tiles may overwrite them
    i32x16_t acc;
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[e] = 0;
#pragma unroll
    for (int i = 0; i < MAXG; ++i) {
        if (kg0 + i < kg1) {
            const uint32_t w = wv[i];
            const u32x4_t fw = {w & 0x03030303u, (w >> 2) & 0x03030303u, (w >> 4) & 0x03030303u, (w >> 6) & 0x03030303u};
            const u32x4_t z = {0u, 0u, 0u, 0u};
            Traits<int8_t>::mma(acc, fw, row_ok ? av[i] : z);
        }
    }
#pragma unroll
    for (int e = 0; e < 16; ++e) part[wave][8 * (e >> 2) + 4 * g + (e & 3)][r] = acc[e];
    __syncthreads();
    if (e_ok) {
        const int m = em, nl = enl, n = en;
        int v = 0;
#pragma unroll
        for (int w = 0; w < GEMV_WAVES; ++w) v += part[w][nl][m];
        v -= 2 * rs_sh[m];
        bf16_t o = f2bf((float)v / s_sh[m] * ws_pf);
        if constexpr (ROPE) {  // N is a multiple of 32 here: no lane of a half-wavefront is missing
            const float own = bf2f(o);
            const float other = __shfl_xor(own, 16, 64);
            const int hh = n / a.D, r = n % a.D, half = a.D >> 1;
            if (hh < a.Hq + a.Hkv) {
                const bool lower = nl < 16;
                const int pi = 16 * (r >> 5) + (nl & 15);
                const float c = cos_pf, sn = sin_pf;
                const float x0 = lower ? own : other, x1 = lower ? other : own;
                const float lo = x0 * c - x1 * sn, hi = x1 * c + x0 * sn;
                const int d = lower ? pi : pi + half;
                const bf16_t rot = f2bf(lower ? lo : hi);
                if (hh < a.Hq) ((bf16_t*)a.q_out)[((long)m * a.Hq + hh) * a.D + d] = rot;
                else ((bf16_t*)a.k_cache)[(((long)m * a.Hkv + (hh - a.Hq)) * a.t_max + a.tok_offset) * a.D + d] = rot;
            } else {
                ((bf16_t*)a.vt_cache)[(((long)m * a.Hkv + (hh - a.Hq - a.Hkv)) * a.D + r) * (long)a.t_max + a.tok_offset] = o;
            }
        } else {
            if (a.residual) o = f2bf(bf2f(o) + bf2f(res_pf));
            ((bf16_t*)a.Y)[(long)m * a.N + n] = o;
        }
    }
}

template <typename T, int kEpi, int TM, int TN, int KB, int DEPTH>
void launch_cfg(GemmArgs a, hipStream_t st) {
    const unsigned grid = xcd_split(a, (a.M + 64 * TM - 1) / (64 * TM), (a.n_tiles + TN - 1) / TN, kEpi == EPI_TERNARY ? 0.25 : sizeof(T), 64 * TN,
                                    kEpi == EPI_TERNARY ? 1.0 : sizeof(T));
    gemm_kernel<T, kEpi, TM, TN, KB, DEPTH><<<grid, 256, 0, st>>>(a);
}

template <int kEpi, int TM, int TN, int KB, int NS>
void launch_dl(GemmArgs a, hipStream_t st) {
    const unsigned grid = xcd_split(a, (a.M + 64 * TM - 1) / (64 * TM), (a.n_tiles + TN - 1) / TN, 2.0, 64 * TN, 2.0);
    if constexpr (kEpi == EPI_QKV) {
        if (a.norm_eps >= 0.f && a.colsum) {
            if (a.stats_in) gemm_dl_kernel<kEpi, TM, TN, KB, NS, NORM_LAYER_PRE><<<grid, 256, 0, st>>>(a);
            else gemm_dl_kernel<kEpi, TM, TN, KB, NS, NORM_LAYER><<<grid, 256, 0, st>>>(a);
            return;
        }
    }
    if constexpr (kEpi == EPI_QKV || kEpi == EPI_GLU) {
        if (a.norm_eps >= 0.f) {
            gemm_dl_kernel<kEpi, TM, TN, KB, NS, NORM_RMS><<<grid, 256, 0, st>>>(a);
            return;
        }
    }
    gemm_dl_kernel<kEpi, TM, TN, KB, NS, NORM_NONE><<<grid, 256, 0, st>>>(a);
}

// rows x columns per workgroup, or -1 for the tiled kernel
int narrow_plan(const GemmArgs& a, bool qkv) {
    const int force = tuning().gemm_rows_plan;
    return force > 0 && force <= 4 ? force - 1 : vla_rules::narrow_plan(a.M, a.N, a.K, qkv);
}

template <int kEpi, int kNorm>
void launch_narrow(const GemmArgs& a, int p, hipStream_t st) {
    // Outputs or a residual that four columns at a time would not hit aligned: a form of its own (a branch in the others'
    // epilogues costs 0.05 us of a launch of 5).  The caller checks the operands and the rotation tables.
    const uintptr_t io = kEpi == EPI_QKV ? (uintptr_t)a.q_out | (uintptr_t)a.k_cache : (uintptr_t)a.Y | (uintptr_t)a.residual;
    if ((kEpi != EPI_PLAIN || a.N % 4 == 0) && (io & (kEpi == EPI_QKV || a.out_bf16 ? 7 : 15))) {  // other N go one by one anyway
        gemm_narrow_kernel<kEpi, kNorm, 1, 1, 6, false><<<(unsigned)vla_rules::narrow_grid(a.M, a.N, 0), 256, 0, st>>>(a);
        return;
    }
    const unsigned grid = (unsigned)vla_rules::narrow_grid(a.M, a.N, p);
    // Ring depths: more stages only delay the first one, fewer leave a CU short of requests; with
    // more workgroups than CUs two of them share a CU's LDS and its requests.
    switch (p) {
        case 0: gemm_narrow_kernel<kEpi, kNorm, 1, 1, 6><<<grid, 256, 0, st>>>(a); break;
        case 1:
            if (vla_rules::narrow_wgs(a.M, a.N, 1) > 256) gemm_narrow_kernel<kEpi, kNorm, 2, 1, 4><<<grid, 256, 0, st>>>(a);
            else gemm_narrow_kernel<kEpi, kNorm, 2, 1, 6><<<grid, 256, 0, st>>>(a);
            break;
        case 2: gemm_narrow_kernel<kEpi, kNorm, 4, 1, 4><<<grid, 256, 0, st>>>(a); break;
        default: gemm_narrow_kernel<kEpi, kNorm, 4, 2, 4><<<grid, 256, 0, st>>>(a); break;
    }
}

// false, launching nothing: more workgroups than the tile walk can count (millions of rows)
template <int MB, int NB, int NS>
bool launch_ring(GemmArgs a, hipStream_t st) {
    const unsigned grid = xcd_split(a, (a.M + 32 * MB - 1) / (32 * MB), (a.N + 32 * NB - 1) / (32 * NB), 0.25, 32 * NB, 1.0);
    if (grid) ternary_gemm_ring_kernel<MB, NB, NS><<<grid, 256, 0, st>>>(a);
    return grid != 0;
}
bool launch_x16(GemmArgs a, hipStream_t st) {
    const int m_wg = (a.M + 127) / 128, n_wg = (a.N + 255) / 256;
    unsigned grid;
    if (m_wg % 8 == 0) {
        // whole M tiles per XCD: workgroups sharing an L2 share their activation rows, the larger
        // operand, and stream the (4x smaller) packed weights tile column by tile column
        a.xm = 8;
        a.xn = a.pn = 1;
        grid = xcd_walk(a, m_wg, n_wg);
    } else {
        grid = xcd_split(a, m_wg, n_wg, 0.25, 256, 1.0);
    }
    if (grid) ternary_gemm_x16_kernel<<<grid, 256, 0, st>>>(a);
    return grid != 0;
}

template <typename T, int kEpi>
int launch(GemmArgs a, int n_tiles, vla_stream_t stream) {
    if (a.M == 0 || n_tiles == 0) return VLA_K_OK;
    a.n_tiles = n_tiles;
    hipStream_t st = (hipStream_t)stream;
    if constexpr (std::is_same<T, float>::value) {
        // a few fp32 rows: narrow tiles (VLA_GEMM_TILE pins the tiled kernel instead)
        bool rows_ok = a.M <= tuning().gemm_rows_max && (a.norm_eps < 0.f || (a.norm_w && a.K <= F32_NORM_MAX_K && (uintptr_t)a.norm_w % 16 == 0)) && tuning().gemm_tile < 0 && ((uintptr_t)a.A | (uintptr_t)a.W) % 16 == 0;
        const int force = tuning().gemm_rows_plan;
        const int plan = !rows_ok ? -1 : force == 1 || force == 3 ? force - 1 : vla_rules::narrow_plan_f32(a.M, a.N, kEpi == EPI_GLU);
        if (plan >= 0) {
            launch_narrow_f32<kEpi>(a, plan, st);
            return hipGetLastError() == hipSuccess ? VLA_K_OK : VLA_K_ERR_LAUNCH;
        }
    }
    if constexpr (std::is_same<T, bf16_t>::value && kEpi != EPI_TERNARY) {
        // few bf16 rows (the suffix of one or a few observations through a projection): narrow tiles over the whole chip
        bool rows_ok = a.M <= tuning().gemm_rows_max && a.K % 8 == 0 && a.K >= 64 && tuning().gemm_tile < 0 && tuning().gemm_dl != 0 &&
                       (uintptr_t)a.A % 16 == 0 && (uintptr_t)a.W % 16 == 0 && !(a.colsum && a.norm_eps < 0.f) && !a.stats_out && !a.stats_in;
        if (kEpi == EPI_QKV)  // 8 + 8 columns of one head, rotation tables read 16 bytes at a time
            rows_ok = rows_ok && a.D % 16 == 0 && a.N % 16 == 0 && (((uintptr_t)a.cos_t | (uintptr_t)a.sin_t) & 15) == 0;
        if (kEpi == EPI_PLAIN) rows_ok = rows_ok && a.norm_eps < 0.f;
        if (a.norm_eps >= 0.f) rows_ok = rows_ok && a.K % 16 == 0;  // what the tiled kernel takes with a norm inside, at every number of rows
        const int plan = rows_ok ? narrow_plan(a, kEpi == EPI_QKV) : -1;
        if (plan >= 0) {
            if (a.norm_eps < 0.f) launch_narrow<kEpi, NORM_NONE>(a, plan, st);
            else if constexpr (kEpi == EPI_QKV) {
                if (a.colsum) launch_narrow<kEpi, NORM_LAYER>(a, plan, st);
                else launch_narrow<kEpi, NORM_RMS>(a, plan, st);
            } else if constexpr (kEpi == EPI_GLU) {
                launch_narrow<kEpi, NORM_RMS>(a, plan, st);
            }
            return hipGetLastError() == hipSuccess ? VLA_K_OK : VLA_K_ERR_LAUNCH;
        }
    }
    if constexpr (kEpi != EPI_TERNARY) {
        // VLA_GEMM_TILE = 0..5 pins the tile configuration and VLA_GEMM_STAGES the ring depth
        // of the direct-to-LDS kernel, 16..24 a tile of the wide-tile kernel (tests and tuning; 22..24 plain products only, 16 in their place elsewhere); unset = by shape.
        int cfg = tuning().gemm_tile;
        const bool pinned = cfg >= 0;
        const int pinned_wide = cfg >= 16 && cfg < 16 + vla_rules::PLAIN_TILES ? (kEpi == EPI_PLAIN || cfg < 16 + vla_rules::WIDE_TILES ? cfg - 16 : 0) : -1;
        const long m128 = (a.M + 127) / 128, m64 = (a.M + 63) / 64;
        const long wgs0 = m128 * ((n_tiles + 1) / 2), wgs2 = m128 * n_tiles, wgs4 = m64 * n_tiles;
        if (!pinned) cfg = sizeof(T) == 4 ? vla_rules::f32_tile(a.M, n_tiles) : vla_rules::dl_tile(a.M, n_tiles);
        // bf16 operands with 16-byte aligned rows and K a multiple of the MFMA depth take the
        // direct-to-LDS kernel (VLA_GEMM_DL=0 pins the register-staged one).  Its ring depth
        // trades loads in flight against LDS per workgroup: a workgroup is short-lived, so
        // what matters first is that the whole grid is resident at once (160 KiB of LDS per
        // CU, 256 CUs), and only then how far ahead each workgroup fetches.
        bool dl = false;
        if constexpr (std::is_same<T, bf16_t>::value) {
            dl = tuning().gemm_dl != 0 && a.K % 16 == 0 && ((uintptr_t)a.A % 16 == 0) && ((uintptr_t)a.W % 16 == 0);
        }
        if (a.norm_eps >= 0.f && !(dl && (kEpi == EPI_QKV || kEpi == EPI_GLU))) return VLA_K_ERR_SHAPE;  // only that kernel takes the row statistics
        if (a.colsum && kEpi != EPI_QKV) return VLA_K_ERR_SHAPE;
        if constexpr (std::is_same<T, bf16_t>::value) {
            // The wide tiles where they are predicted faster (32-bit lane offsets inside a tile; row sums handed from launch
            // to launch stay with the kernel below).
            if (dl && a.K <= (1 << 20) && !a.stats_in && !a.stats_out) {
                const int wide = pinned ? pinned_wide : kEpi == EPI_PLAIN ? vla_rules::plain_tile(a.M, a.N, a.K) : vla_rules::wide_tile(a.M, a.N, a.K, kEpi != EPI_QKV ? 0 : a.colsum ? 2 : 1);
                if (wide >= 0 && launch_wide<kEpi>(a, wide, st)) return hipGetLastError() == hipSuccess ? VLA_K_OK : VLA_K_ERR_LAUNCH;
            }
        }
        if (dl) {
            int ns = tuning().gemm_stages;
            const long wgs = cfg == 0 ? wgs0 : (cfg == 2 || cfg == 3 ? wgs2 : wgs4);
            switch (cfg) {
                case 5:  // 40 KiB per stage, one workgroup per CU
                    launch_dl<kEpi, 2, 3, 128, 3>(a, st);
                    break;
                case 0:  // 32 KiB per stage
                    if (ns == 0) ns = wgs <= 256 ? 3 : 2;
                    if (ns <= 2) launch_dl<kEpi, 2, 2, 128, 2>(a, st);
                    else launch_dl<kEpi, 2, 2, 128, 3>(a, st);
                    break;
                case 1:  // 32 KiB per stage
                    if (ns == 0) ns = 4;
                    if (ns <= 3) launch_dl<kEpi, 1, 1, 256, 3>(a, st);
                    else launch_dl<kEpi, 1, 1, 256, 4>(a, st);
                    break;
                case 2:  // 24 KiB per stage
                    if (ns == 0) ns = wgs <= 256 ? 4 : (wgs <= 512 ? 3 : 2);
                    if (ns <= 2) launch_dl<kEpi, 2, 1, 128, 2>(a, st);
                    else if (ns == 3) launch_dl<kEpi, 2, 1, 128, 3>(a, st);
                    else launch_dl<kEpi, 2, 1, 128, 4>(a, st);
                    break;
                case 3:  // 24 KiB per stage
                    if (ns == 0) ns = wgs <= 256 ? 4 : 3;
                    if (ns <= 3) launch_dl<kEpi, 1, 2, 128, 3>(a, st);
                    else launch_dl<kEpi, 1, 2, 128, 4>(a, st);
                    break;
                default:  // 16 KiB per stage
                    if (ns == 0) ns = wgs <= 512 ? 4 : 3;
                    if (ns <= 3) launch_dl<kEpi, 1, 1, 128, 3>(a, st);
                    else launch_dl<kEpi, 1, 1, 128, 4>(a, st);
                    break;
            }
            return hipGetLastError() == hipSuccess ? VLA_K_OK : VLA_K_ERR_LAUNCH;
        }
        switch (cfg) {
            case 0: launch_cfg<T, kEpi, 2, 2, 128, 3>(a, st); break;
            case 1: launch_cfg<T, kEpi, 1, 1, 256, 4>(a, st); break;
            case 2: launch_cfg<T, kEpi, 2, 1, 128, 4>(a, st); break;
            case 3: launch_cfg<T, kEpi, 1, 2, 128, 4>(a, st); break;
            case 5: launch_cfg<T, kEpi, 2, 2, 128, 3>(a, st); break;  // the register-staged kernel has no 192-column tile
            default: launch_cfg<T, kEpi, 1, 1, 128, 6>(a, st); break;
        }
    } else {
        // VLA_TERNARY_TILE = 64 | 128 | 256 pins a tile of the 32x32x32 kernels, 16..21 one of the 16x16x64 kernels (tests and tuning); unset = by shape.
        const int force = tuning().ternary_tile;
        const int n256 = (a.N + 255) / 256;
        const long wg128 = (long)((a.M + 127) / 128) * n256;
        const int gemv_groups = (a.K / 32 + GEMV_WAVES - 1) / GEMV_WAVES;  // k groups per wavefront
        // The 16x16x64 kernel addresses both operands with 32-bit byte offsets, writes 8-column vectors and keeps one
        // weight scale per 32-column block; anything else stays with the 32x32x32 kernels.
        const int ws_group = a.N / (a.ws_num > 0 ? a.ws_num : 1);
        const bool x16_ok = a.N % 8 == 0 && (a.Y == nullptr || ws_group % 32 == 0) && (long)a.M * a.K < (1l << 32) &&
                            (long)((a.N + 31) / 32) * a.K * 8 < (1l << 32) && ((uintptr_t)a.A % 16 == 0) && a.K % 16 == 0;
        // The LDS-ring tiles copy the weights and write the rows in 16-byte pieces; unaligned buffers stay with the other
        // kernels, 128 x 256 tiles from half the chip on and the 64 x 64 ones, whose weight and row accesses are 4 bytes
        // and less, below.
        const bool ring_ok = (((uintptr_t)a.W | (uintptr_t)a.Y | (uintptr_t)a.residual) & 15) == 0;
        const bool x16_asked = force == 0 || (force >= 16 && force < 64);
        bool done = false;
        if (force == 0 && a.M <= 32 && gemv_groups <= 28) {
            const unsigned grid = (unsigned)((a.N + 31) / 32);
            if (gemv_groups <= 10) ternary_gemv_kernel<10><<<grid, GEMV_WAVES * 64, 0, st>>>(a);
            else ternary_gemv_kernel<28><<<grid, GEMV_WAVES * 64, 0, st>>>(a);
            done = true;
        } else if (x16_ok && x16_asked && (ring_ok || force == 16 || wg128 >= 128)) {
            // the 16x16x64 kernels
            switch (!ring_ok ? 16 : force ? force : vla_rules::ternary_tile(a.M, a.N, a.K)) {
                case 17: done = launch_ring<4, 4, 4>(a, st); break;
                case 18: done = launch_ring<2, 4, 5>(a, st); break;
                case 19: done = launch_ring<2, 2, 6>(a, st); break;
                case 20: done = launch_ring<2, 8, 4>(a, st); break;
                case 21: done = launch_ring<1, 2, 8>(a, st); break;
                default: done = launch_x16(a, st); break;  // 128 x 256 tiles, two workgroups per CU
            }
        }
        // What those do not take: the 32x32x32 kernels, with 128 x 256 tiles where they fill half the chip (two
        // workgroups per CU, measured faster than one of 256 x 256: fewer wavefronts per barrier).
        if (done) {
        } else if (force == 256) {
            const unsigned grid = (unsigned)(((((a.M + 255) / 256) + 7) & ~7) * n256);
            ternary_gemm_big_kernel<4><<<grid, 512, 0, st>>>(a);
        } else if (force == 128 || (x16_asked && wg128 >= 128)) {
            const unsigned grid = (unsigned)(((((a.M + 127) / 128) + 7) & ~7) * n256);
            ternary_gemm_big_kernel<2><<<grid, 256, 0, st>>>(a);
        } else {
            launch_cfg<T, EPI_TERNARY, 1, 1, 128, 4>(a, st);
        }
    }
    return hipGetLastError() == hipSuccess ? VLA_K_OK : VLA_K_ERR_LAUNCH;
}

// Row sums for the exact-signature BitVLA entry points.
__global__ void rowsum_i8_kernel(const int8_t* __restrict__ A, int32_t* __restrict__ rowsum, int K) {
    const int8_t* r = A + (long)blockIdx.x * K;
    int s = 0;
    for (int k = threadIdx.x; k < K; k += 64) s += r[k];
    s = wave_sum_i(s);
    if (threadIdx.x == 0) rowsum[blockIdx.x] = s;
}

template <bool ROPE, bool GLU = false>
int launch_gemv_norm(const GemmArgs& a, vla_stream_t stream) {
    const unsigned grid = (unsigned)((a.N + 31) / 32);
    const int groups = (a.K / 32 + GEMV_WAVES - 1) / GEMV_WAVES, nvec = a.K / 8;
    hipStream_t st = (hipStream_t)stream;
#define VLA_GEMV_NORM(G, NV) ternary_gemv_norm_kernel<G, NV, ROPE, GLU><<<grid, GEMV_WAVES * 64, 0, st>>>(a)
    if (groups <= 10) {
        if (nvec <= 128) VLA_GEMV_NORM(10, 2);
        else if (nvec <= 256) VLA_GEMV_NORM(10, 4);
        else VLA_GEMV_NORM(10, 5);  // up to 2560 wide, the model's rows: three vectors of eight would be padding
    } else if (groups <= 16) {
        VLA_GEMV_NORM(16, 8);
    } else {
        if constexpr (ROPE) return VLA_K_ERR_SHAPE;  // the QKV projection's K is the model width, never that long
        else VLA_GEMV_NORM(28, 16);
    }
#undef VLA_GEMV_NORM
    return hipGetLastError() == hipSuccess ? VLA_K_OK : VLA_K_ERR_LAUNCH;
}

}  // namespace

extern "C" {

int vla_linear(const void* x, const void* W, const float* bias, const void* residual, void* y, int dtype,
               int out_dtype, int M, int N, int K, vla_stream_t stream) {
    if (!x || !W || !y || M < 0 || N <= 0 || K <= 0) return VLA_K_ERR_ARG;
    if (out_dtype != VLA_DT_F32 && out_dtype != VLA_DT_BF16) return VLA_K_ERR_ARG;
    GemmArgs a = {};
    a.norm_eps = -1.f;
    a.A = x; a.W = W; a.bias = bias; a.M = M; a.N = N; a.K = K;
    a.residual = residual; a.Y = y; a.out_bf16 = (out_dtype == VLA_DT_BF16);
    const int nt = (N + BN - 1) / BN;
    if (dtype == VLA_DT_BF16) {
        if (K % 8) return VLA_K_ERR_SHAPE;
        return launch<bf16_t, EPI_PLAIN>(a, nt, stream);
    }
    if (dtype == VLA_DT_F32) {
        if (K % 4) return VLA_K_ERR_SHAPE;
        return launch<float, EPI_PLAIN>(a, nt, stream);
    }
    return VLA_K_ERR_ARG;
}

static int qkv_rope_impl(const void* x, const void* W, const float* bias, int dtype, int M, int K, int S, int n_q_heads,
                         int n_kv_heads, int has_k, int has_v, int head_dim, const float* cos_tab, const float* sin_tab,
                         void* q_out, void* k_cache, void* vt_cache, int t_max, int tok_offset, float rms_eps,
                         vla_stream_t stream, const float* colsum = nullptr, const float* stats_in = nullptr, int n_stat = 0,
                         const float* norm_w = nullptr) {
    if (!x || !W || M < 0 || K <= 0 || S <= 0 || n_q_heads < 0 || n_kv_heads < 0 || head_dim <= 0) return VLA_K_ERR_ARG;
    const int nk = has_k ? n_kv_heads : 0, nv = has_v ? n_kv_heads : 0;
    if (n_q_heads > 0 && !q_out) return VLA_K_ERR_ARG;
    if ((nk > 0 && !k_cache) || (nv > 0 && !vt_cache)) return VLA_K_ERR_ARG;
    if ((cos_tab == nullptr) != (sin_tab == nullptr)) return VLA_K_ERR_ARG;
    if (M % S) return VLA_K_ERR_SHAPE;
    if (nk + nv > 0 && (tok_offset < 0 || tok_offset + S > t_max)) return VLA_K_ERR_SHAPE;
    const int D = head_dim;
    // every segment is a whole number of 64-column tiles, 8-column groups stay inside a head
    if ((n_q_heads * D) % BN || (nk * D) % BN || (nv * D) % BN || D % 8) return VLA_K_ERR_SHAPE;
    if (cos_tab && D % BN) return VLA_K_ERR_SHAPE;  // rotation pairs both halves of a head inside one tile
    GemmArgs a = {};
    a.norm_eps = rms_eps;
    a.colsum = colsum;
    a.stats_in = stats_in;
    a.n_stat = n_stat;
    a.norm_w = norm_w;
    a.A = x; a.W = W; a.bias = bias; a.M = M; a.K = K;
    a.N = (n_q_heads + nk + nv) * D;
    a.S = S; a.Hq = n_q_heads; a.nk = nk; a.nv = nv; a.D = D; a.Hkv = n_kv_heads;
    a.cos_t = cos_tab; a.sin_t = sin_tab; a.q_out = q_out; a.k_cache = k_cache; a.vt_cache = vt_cache;
    a.t_max = t_max; a.tok_offset = tok_offset;
    const int nt = a.N / BN;
    if (dtype == VLA_DT_BF16) {
        if (K % 8) return VLA_K_ERR_SHAPE;
        return launch<bf16_t, EPI_QKV>(a, nt, stream);
    }
    if (dtype == VLA_DT_F32) {
        if (K % 4) return VLA_K_ERR_SHAPE;
        return launch<float, EPI_QKV>(a, nt, stream);
    }
    return VLA_K_ERR_ARG;
}

int vla_attn_qkv_rope(const void* x, const void* W, const float* bias, int dtype, int M, int K, int S, int n_q_heads,
                      int n_kv_heads, int has_k, int has_v, int head_dim, const float* cos_tab, const float* sin_tab,
                      void* q_out, void* k_cache, void* vt_cache, int t_max, int tok_offset, vla_stream_t stream) {
    return qkv_rope_impl(x, W, bias, dtype, M, K, S, n_q_heads, n_kv_heads, has_k, has_v, head_dim, cos_tab, sin_tab, q_out,
                         k_cache, vt_cache, t_max, tok_offset, -1.f, stream);
}

int vla_linear_act(const void* x, const void* W, const float* bias, const void* residual, void* y, int dtype,
                   int out_dtype, int M, int N, int K, int act, vla_stream_t stream) {
    if (!x || !W || !y || M < 0 || N <= 0 || K <= 0) return VLA_K_ERR_ARG;
    if (out_dtype != VLA_DT_F32 && out_dtype != VLA_DT_BF16) return VLA_K_ERR_ARG;
    if (act < VLA_ACT_NONE || act > VLA_ACT_RELU) return VLA_K_ERR_ARG;
    GemmArgs a = {};
    a.norm_eps = -1.f;
    a.A = x; a.W = W; a.bias = bias; a.M = M; a.N = N; a.K = K;
    a.residual = residual; a.Y = y; a.out_bf16 = (out_dtype == VLA_DT_BF16); a.act = act;
    const int nt = (N + BN - 1) / BN;
    if (dtype == VLA_DT_BF16) {
        if (K % 8) return VLA_K_ERR_SHAPE;
        return launch<bf16_t, EPI_PLAIN>(a, nt, stream);
    }
    if (dtype == VLA_DT_F32) {
        if (K % 4) return VLA_K_ERR_SHAPE;
        return launch<float, EPI_PLAIN>(a, nt, stream);
    }
    return VLA_K_ERR_ARG;
}

int vla_linear_gated(const void* x, const void* W, const float* bias, const float* col_gate, const void* residual, void* y,
                     int dtype, int out_dtype, int M, int N, int K, vla_stream_t stream) {
    if (!x || !W || !y || !col_gate || M < 0 || N <= 0 || K <= 0) return VLA_K_ERR_ARG;
    if (out_dtype != VLA_DT_F32 && out_dtype != VLA_DT_BF16) return VLA_K_ERR_ARG;
    GemmArgs a = {};
    a.norm_eps = -1.f;
    a.A = x; a.W = W; a.bias = bias; a.M = M; a.N = N; a.K = K;
    a.residual = residual; a.Y = y; a.out_bf16 = (out_dtype == VLA_DT_BF16); a.col_gate = col_gate;
    const int nt = (N + BN - 1) / BN;
    if (dtype == VLA_DT_BF16) {
        if (K % 8) return VLA_K_ERR_SHAPE;
        return launch<bf16_t, EPI_PLAIN>(a, nt, stream);
    }
    if (dtype == VLA_DT_F32) {
        if (K % 4) return VLA_K_ERR_SHAPE;
        return launch<float, EPI_PLAIN>(a, nt, stream);
    }
    return VLA_K_ERR_ARG;
}

int vla_glu_linear(const void* x, const void* W_gate_up, const float* bias, void* y, int dtype, int out_dtype, int M, int I,
                   int K, int act, float rms_eps, vla_stream_t stream) {
    if (!x || !W_gate_up || !y || M < 0 || I <= 0 || K <= 0) return VLA_K_ERR_ARG;
    if (out_dtype != VLA_DT_F32 && out_dtype != VLA_DT_BF16) return VLA_K_ERR_ARG;
    if (act < VLA_ACT_NONE || act > VLA_ACT_RELU) return VLA_K_ERR_ARG;
    if (I % 32) return VLA_K_ERR_SHAPE;  // a tile pairs 32 gate columns with their 32 up columns
    GemmArgs a = {};
    a.norm_eps = rms_eps >= 0.f ? rms_eps : -1.f;
    a.A = x; a.W = W_gate_up; a.bias = bias; a.M = M; a.N = 2 * I; a.K = K;
    a.Y = y; a.out_bf16 = (out_dtype == VLA_DT_BF16); a.act = act;
    const int nt = I / 32;
    if (dtype == VLA_DT_BF16) {
        if (K % 8) return VLA_K_ERR_SHAPE;
        return launch<bf16_t, EPI_GLU>(a, nt, stream);
    }
    if (dtype == VLA_DT_F32) {
        if (K % 4) return VLA_K_ERR_SHAPE;
        return launch<float, EPI_GLU>(a, nt, stream);
    }
    return VLA_K_ERR_ARG;
}

int vla_rmsnorm_attn_qkv_rope(const void* x, const void* W_folded, const float* bias, int dtype, int M, int K, int S,
                              int n_q_heads, int n_kv_heads, int has_k, int has_v, int head_dim, const float* cos_tab,
                              const float* sin_tab, void* q_out, void* k_cache, void* vt_cache, int t_max, int tok_offset,
                              float rms_eps, vla_stream_t stream) {
    if (rms_eps < 0.f) return VLA_K_ERR_ARG;
    if (dtype != VLA_DT_BF16) return VLA_K_ERR_SHAPE;
    return qkv_rope_impl(x, W_folded, bias, dtype, M, K, S, n_q_heads, n_kv_heads, has_k, has_v, head_dim, cos_tab, sin_tab,
                         q_out, k_cache, vt_cache, t_max, tok_offset, rms_eps, stream);
}

int vla_layernorm_attn_qkv_rope(const void* x, const void* W_folded, const float* colsum, const float* bias, int dtype, int M,
                                int K, int S, int n_q_heads, int n_kv_heads, int has_k, int has_v, int head_dim,
                                const float* cos_tab, const float* sin_tab, void* q_out, void* k_cache, void* vt_cache,
                                int t_max, int tok_offset, float ln_eps, vla_stream_t stream) {
    if (ln_eps < 0.f || !colsum) return VLA_K_ERR_ARG;
    if (dtype != VLA_DT_BF16) return VLA_K_ERR_SHAPE;
    return qkv_rope_impl(x, W_folded, bias, dtype, M, K, S, n_q_heads, n_kv_heads, has_k, has_v, head_dim, cos_tab, sin_tab,
                         q_out, k_cache, vt_cache, t_max, tok_offset, ln_eps, stream, colsum);
}

int vla_layernorm_attn_qkv_rope_stats(const void* x, const void* W_folded, const float* colsum, const float* bias,
                                      const float* row_stats, int n_stat_tiles, int dtype, int M, int K, int S, int n_q_heads,
                                      int n_kv_heads, int has_k, int has_v, int head_dim, const float* cos_tab,
                                      const float* sin_tab, void* q_out, void* k_cache, void* vt_cache, int t_max,
                                      int tok_offset, float ln_eps, vla_stream_t stream) {
    if (ln_eps < 0.f || !colsum || !row_stats) return VLA_K_ERR_ARG;
    if (dtype != VLA_DT_BF16 || n_stat_tiles < 1 || n_stat_tiles > STAT_MAX_TILES || K != n_stat_tiles * BN) return VLA_K_ERR_SHAPE;
    return qkv_rope_impl(x, W_folded, bias, dtype, M, K, S, n_q_heads, n_kv_heads, has_k, has_v, head_dim, cos_tab, sin_tab,
                         q_out, k_cache, vt_cache, t_max, tok_offset, ln_eps, stream, colsum, row_stats, n_stat_tiles);
}

int vla_linear_row_stats(const void* x, const void* W, const float* bias, const void* residual, void* y, float* row_stats,
                         int dtype, int M, int N, int K, vla_stream_t stream) {
    if (!x || !W || !y || !row_stats || M < 0 || N <= 0 || K <= 0) return VLA_K_ERR_ARG;
    if (dtype != VLA_DT_BF16 || N % BN || K % 8) return VLA_K_ERR_SHAPE;
    GemmArgs a = {};
    a.norm_eps = -1.f;
    a.A = x; a.W = W; a.bias = bias; a.M = M; a.N = N; a.K = K;
    a.residual = residual; a.Y = y; a.out_bf16 = 1;
    a.stats_out = row_stats;
    return launch<bf16_t, EPI_PLAIN>(a, N / BN, stream);
}

int vla_fold_norm_weight_host(const void* W, const void* g, int dtype, int N, int K, void* W_out) {
    if (!W || !g || !W_out || N <= 0 || K <= 0) return VLA_K_ERR_ARG;
    if (dtype == VLA_DT_F32) {
        for (long n = 0; n < N; ++n)
            for (int k = 0; k < K; ++k) ((float*)W_out)[n * K + k] = ((const float*)W)[n * K + k] * ((const float*)g)[k];
        return VLA_K_OK;
    }
    if (dtype == VLA_DT_BF16) {
        const uint16_t* w = (const uint16_t*)W;
        const uint16_t* gg = (const uint16_t*)g;
        for (long n = 0; n < N; ++n)
            for (int k = 0; k < K; ++k) {
                uint32_t wb = (uint32_t)w[n * K + k] << 16, gb = (uint32_t)gg[k] << 16;
                float wf, gf;
                memcpy(&wf, &wb, 4);
                memcpy(&gf, &gb, 4);
                const float p = wf * gf;
                uint32_t pb;
                memcpy(&pb, &p, 4);
                if ((pb & 0x7fffffffu) > 0x7f800000u) pb |= 0x00400000u;                // NaN stays NaN
                else pb += 0x7fffu + ((pb >> 16) & 1u);                                  // round to nearest even
                ((uint16_t*)W_out)[n * K + k] = (uint16_t)(pb >> 16);
            }
        return VLA_K_OK;
    }
    return VLA_K_ERR_ARG;
}

int vla_fold_adaln_weight_host(const void* W, const float* bias, const float* scale, const float* shift, int N, int K,
                               void* W_out, float* colsum_out, float* bias_out) {
    if (!W || !scale || !shift || !W_out || !colsum_out || !bias_out || N <= 0 || K <= 0) return VLA_K_ERR_ARG;
    const uint16_t* w = (const uint16_t*)W;
    for (long n = 0; n < N; ++n) {
        double cs = 0.0, bs = bias ? (double)bias[n] : 0.0;
        for (int k = 0; k < K; ++k) {
            const uint32_t wb = (uint32_t)w[n * K + k] << 16;
            float wf;
            memcpy(&wf, &wb, 4);
            bs += (double)wf * (double)shift[k];
            const float p = wf * (1.0f + scale[k]);
            uint32_t pb;
            memcpy(&pb, &p, 4);
            if ((pb & 0x7fffffffu) > 0x7f800000u) pb |= 0x00400000u;  // NaN stays NaN
            else pb += 0x7fffu + ((pb >> 16) & 1u);                    // round to nearest even
            pb &= 0xffff0000u;
            ((uint16_t*)W_out)[n * K + k] = (uint16_t)(pb >> 16);
            float rf;
            memcpy(&rf, &pb, 4);
            cs += (double)rf;
        }
        colsum_out[n] = (float)cs;
        bias_out[n] = (float)bs;
    }
    return VLA_K_OK;
}

int vla_ternary_gemm(const int8_t* A, const uint32_t* W_packed, uint16_t* out, int32_t* acc_out, const float* s,
                     const int32_t* rowsum, const float* ws, int ws_num, int M, int N, int K, vla_stream_t stream) {
    if (!A || !W_packed || !rowsum || (!out && !acc_out) || M < 0 || N <= 0 || K <= 0) return VLA_K_ERR_ARG;
    if (out && (!s || !ws || ws_num <= 0)) return VLA_K_ERR_ARG;
    if (K % 128 || (out && N % ws_num)) return VLA_K_ERR_SHAPE;
    GemmArgs a = {};
    a.norm_eps = -1.f;
    a.A = A; a.W = W_packed; a.M = M; a.N = N; a.K = K;
    a.Y = out; a.acc_out = acc_out; a.s = s; a.rowsum = rowsum; a.ws = ws; a.ws_num = ws_num > 0 ? ws_num : 1;
    return launch<int8_t, EPI_TERNARY>(a, (N + BN - 1) / BN, stream);
}

int vla_ternary_gemm_add(const int8_t* A, const uint32_t* W_packed, uint16_t* out, const uint16_t* residual, const float* s,
                         const int32_t* rowsum, const float* ws, int ws_num, int M, int N, int K, vla_stream_t stream) {
    if (!A || !W_packed || !rowsum || !out || !s || !ws || ws_num <= 0 || M < 0 || N <= 0 || K <= 0) return VLA_K_ERR_ARG;
    if (K % 128 || N % ws_num) return VLA_K_ERR_SHAPE;
    GemmArgs a = {};
    a.norm_eps = -1.f;
    a.A = A; a.W = W_packed; a.M = M; a.N = N; a.K = K;
    a.Y = out; a.residual = residual; a.s = s; a.rowsum = rowsum; a.ws = ws; a.ws_num = ws_num;
    return launch<int8_t, EPI_TERNARY>(a, (N + BN - 1) / BN, stream);
}

int vla_rmsnorm_ternary_gemv(const uint16_t* x, const uint16_t* norm_w, float eps, const uint32_t* W_packed, uint16_t* out,
                             const uint16_t* residual, const float* ws, int ws_num, int M, int N, int K,
                             vla_stream_t stream) {
    if (!x || !W_packed || !out || !ws || ws_num <= 0 || M < 0 || N <= 0 || K <= 0) return VLA_K_ERR_ARG;
    if (M > GEMV_WAVES || K > GEMV_FUSED_MAX_K || K % 128 || N % ws_num || (((uintptr_t)x) & 15)) return VLA_K_ERR_SHAPE;
    if (M == 0) return VLA_K_OK;
    GemmArgs a = {};
    a.A = x; a.norm_w = norm_w; a.norm_eps = eps; a.W = W_packed; a.M = M; a.N = N; a.K = K;
    a.Y = out; a.residual = residual; a.ws = ws; a.ws_num = ws_num;
    return launch_gemv_norm<false>(a, stream);
}

int vla_sqrelu_rmsnorm_ternary_gemv(const uint16_t* gate_up, const uint16_t* norm_w, float eps, const uint32_t* W_packed,
                                    uint16_t* out, const uint16_t* residual, const float* ws, int ws_num, int M, int N, int K,
                                    vla_stream_t stream) {
    if (!gate_up || !W_packed || !out || !ws || ws_num <= 0 || M < 0 || N <= 0 || K <= 0) return VLA_K_ERR_ARG;
    if (M > GEMV_WAVES || K > GEMV_FUSED_MAX_K || K % 128 || N % ws_num || (((uintptr_t)gate_up) & 15)) return VLA_K_ERR_SHAPE;
    if (M == 0) return VLA_K_OK;
    GemmArgs a = {};
    a.A = gate_up; a.norm_w = norm_w; a.norm_eps = eps; a.W = W_packed; a.M = M; a.N = N; a.K = K;
    a.Y = out; a.residual = residual; a.ws = ws; a.ws_num = ws_num;
    return launch_gemv_norm<false, true>(a, stream);
}

int vla_rmsnorm_ternary_gemv_rope_append(const uint16_t* x, const uint16_t* norm_w, float eps, const uint32_t* W_paired,
                                         const float* ws, int ws_num, const float* cos_row, const float* sin_row,
                                         uint16_t* q_out, uint16_t* k_cache, uint16_t* vt_cache, int batch, int n_q_heads,
                                         int n_kv_heads, int head_dim, int K, int t_max, int tok_offset,
                                         vla_stream_t stream) {
    if (!x || !W_paired || !ws || !cos_row || !sin_row || !q_out || !k_cache || !vt_cache || ws_num <= 0 || batch < 0 ||
        n_q_heads <= 0 || n_kv_heads <= 0 || head_dim <= 0 || K <= 0)
        return VLA_K_ERR_ARG;
    const int N = (n_q_heads + 2 * n_kv_heads) * head_dim;
    if (batch > GEMV_WAVES || K > 4096 || K % 128 || head_dim % 32 || N % ws_num || (N / ws_num) % head_dim ||
        tok_offset < 0 || tok_offset >= t_max || (((uintptr_t)x) & 15))
        return VLA_K_ERR_SHAPE;
    if (batch == 0) return VLA_K_OK;
    GemmArgs a = {};
    a.A = x; a.norm_w = norm_w; a.norm_eps = eps; a.W = W_paired; a.M = batch; a.N = N; a.K = K;
    a.ws = ws; a.ws_num = ws_num; a.cos_t = cos_row; a.sin_t = sin_row;
    a.q_out = q_out; a.k_cache = k_cache; a.vt_cache = vt_cache;
    a.Hq = n_q_heads; a.Hkv = n_kv_heads; a.D = head_dim; a.t_max = t_max; a.tok_offset = tok_offset; a.S = 1;
    return launch_gemv_norm<true>(a, stream);
}

int vla_ternary_pair_rope_rows_host(const uint32_t* packed, int n_q_heads, int n_kv_heads, int head_dim, int K,
                                    uint32_t* paired) {
    if (!packed || !paired || packed == paired || n_q_heads <= 0 || n_kv_heads <= 0 || head_dim <= 0 || K <= 0)
        return VLA_K_ERR_ARG;
    if (head_dim % 32 || K % 32) return VLA_K_ERR_SHAPE;
    const int half = head_dim / 2, kw = K / 16;
    const long rope_rows = (long)(n_q_heads + n_kv_heads) * head_dim, N = rope_rows + (long)n_kv_heads * head_dim;
    for (long n = 0; n < N; ++n) {
        long src = n;
        if (n < rope_rows) {
            const int r = (int)(n % head_dim), nl = r % 32;
            src = n - r + (nl < 16 ? 16 * (r / 32) + nl : half + 16 * (r / 32) + (nl - 16));
        }
        for (int w = 0; w < kw; ++w) paired[tern_word_index(n, w, K)] = packed[tern_word_index(src, w, K)];
    }
    return VLA_K_OK;
}

static int bitvla_ws_num(int N, int K) {  // the reference's per-shape table, bitnet_kernels.cu:31-116
    if (N == 3840 && K == 2560) return 3;
    if (N == 13824 && K == 2560) return 2;
    if (N == 4800 && K == 3200) return 6;
    if (N == 20480 && K == 3200) return 2;
    return 1;
}

int bitlinear_int8xint2_m(int8_t* A, int8_t* B, uint16_t* out, float* s, float* ws, int M, int N, int K,
                          vla_stream_t stream) {
    if (!A || !B || !out || !s || !ws || M < 0) return VLA_K_ERR_ARG;
    if (M == 0) return VLA_K_OK;
    // the reference's signature carries no row sums: they go into a block the library keeps
    // for this stream (calls on one stream are ordered, other streams have their own block)
    int32_t* rowsum = (int32_t*)stream_scratch(SCRATCH_ROWSUM, (hipStream_t)stream, (size_t)M * sizeof(int32_t));
    if (!rowsum) return VLA_K_ERR_LAUNCH;
    rowsum_i8_kernel<<<M, 64, 0, (hipStream_t)stream>>>(A, rowsum, K);
    return vla_ternary_gemm(A, (const uint32_t*)B, out, nullptr, s, rowsum, ws, bitvla_ws_num(N, K), M, N, K, stream);
}

int bitlinear_int8xint2(int8_t* A, int8_t* B, uint16_t* out, float* s, float* ws, int M, int N, int K,
                        vla_stream_t stream) {
    return bitlinear_int8xint2_m(A, B, out, s, ws, M, N, K, stream);
}

int vla_ternary_quant_host(const float* W, int64_t n, int8_t* ternary, float* absmean) {
    if (!W || !ternary || !absmean || n < 0) return VLA_K_ERR_ARG;
    double sum = 0.0;
    for (int64_t i = 0; i < n; ++i) sum += fabs((double)W[i]);
    float mean = n > 0 ? (float)(sum / (double)n) : 0.0f;
    if (mean < 1e-5f) mean = 1e-5f;
    *absmean = mean;
    const float inv = 1.0f / mean;
    for (int64_t i = 0; i < n; ++i) {
        float q = nearbyintf(W[i] * inv);
        q = q > 1.0f ? 1.0f : (q < -1.0f ? -1.0f : q);
        ternary[i] = (int8_t)q;
    }
    return VLA_K_OK;
}

long vla_ternary_packed_words(int N, int K) { return (long)((N + 31) / 32 * 32) * (K / 16); }

static void tern_fill_pad_rows(int N, int K, uint32_t* packed) {
    for (long n = N; n < (N + 31) / 32 * 32; ++n)
        for (int w = 0; w < K / 16; ++w) packed[tern_word_index(n, w, K)] = 0xAAAAAAAAu;  // code 2 = weight 0
}

int vla_ternary_pack_host(const int8_t* ternary, int N, int K, uint32_t* packed) {
    if (!ternary || !packed || N <= 0 || K <= 0) return VLA_K_ERR_ARG;
    if (K % 32) return VLA_K_ERR_SHAPE;
    const int kw = K / 16;
    for (long n = 0; n < N; ++n)
        for (int w = 0; w < kw; ++w) {
            uint32_t word = 0;
            for (int v = 0; v < 16; ++v) {
                const int t = ternary[n * K + w * 16 + v];
                if (t < -2 || t > 1) return VLA_K_ERR_ARG;
                word |= (uint32_t)((t + 2) & 3) << (8 * (v & 3) + 2 * (v >> 2));
            }
            packed[tern_word_index(n, w, K)] = word;
        }
    tern_fill_pad_rows(N, K, packed);
    return VLA_K_OK;
}

// A ladder slot is the same 16-value word; only the word order differs
// (src/models/bitvla.cpp:453-483): inside each 16-row block the words run
// (k_0: 128 k) (major_k: 32 k) (y_half: 8 rows) (sub_k: 16 k) (row in half).
int vla_ternary_repack_ladder_host(const uint8_t* ladder, int N, int K, uint32_t* packed) {
    if (!ladder || !packed || N <= 0 || K <= 0) return VLA_K_ERR_ARG;
    if (N % 16 || K % 128) return VLA_K_ERR_SHAPE;
    const uint32_t* src = (const uint32_t*)ladder;
    const int kw = K / 16;
    for (long n = 0; n < N; ++n)
        for (int w = 0; w < kw; ++w) {
            const long n_block = n / 16;
            const int y = (int)(n % 16), y_half = y / 8, y_in_h = y % 8;
            const int k_0 = w / 8, tx = w % 8, major_k = tx / 2, sub_k = tx % 2;
            const long slot = n_block * K + (long)k_0 * 128 + major_k * 32 + y_half * 16 + sub_k * 8 + y_in_h;
            packed[tern_word_index(n, w, K)] = src[slot];
        }
    tern_fill_pad_rows(N, K, packed);
    return VLA_K_OK;
}

}  // extern "C"

namespace vk {

int f32_rmsnorm_attn_qkv_rope(const float* x, const float* norm_w, float eps, const float* W, const float* bias, int M, int K, int S,
                              int n_q_heads, int n_kv_heads, int has_k, int has_v, int head_dim, const float* cos_tab,
                              const float* sin_tab, void* q_out, void* k_cache, void* vt_cache, int t_max, int tok_offset,
                              vla_stream_t stream) {
    if (!norm_w || eps < 0.f) return VLA_K_ERR_ARG;
    return qkv_rope_impl(x, W, bias, VLA_DT_F32, M, K, S, n_q_heads, n_kv_heads, has_k, has_v, head_dim, cos_tab, sin_tab, q_out, k_cache,
                         vt_cache, t_max, tok_offset, eps, stream, nullptr, nullptr, 0, norm_w);
}

int f32_rmsnorm_glu_linear(const float* x, const float* norm_w, float eps, const float* W_gate_up, void* y, int M, int I, int K, int act,
                           vla_stream_t stream) {
    if (!x || !norm_w || !W_gate_up || !y || eps < 0.f || M < 0 || I <= 0 || K <= 0) return VLA_K_ERR_ARG;
    if (I % 32 || K % 4) return VLA_K_ERR_SHAPE;
    GemmArgs a = {};
    a.norm_eps = eps;
    a.norm_w = norm_w;
    a.A = x; a.W = W_gate_up; a.M = M; a.N = 2 * I; a.K = K;
    a.Y = y; a.act = act;
    return launch<float, EPI_GLU>(a, I / 32, stream);
}

}  // namespace vk
