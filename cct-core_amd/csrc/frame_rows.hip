// Frame block-reduce modes on the BF16 / FP16 matrix cores, walking down the rows:
//
//   out[b*Mout + m](y, x) = sum_{r < R} sum_{t < F*F} A[m][r][t] * X_{b*N + r}(y - h + ti, x - h + tj)
//
// (the contraction of igemm_f32.hip; ConvolveHyperKernel.scala:153-167, 327-332,
// borders 235-317), for operands of T terms:
//
//   BF16, FP16    T = 1: operands rounded once, one product.
//   split-BF16    T = 2: x = x0 + x1, the products x0 w0 + x0 w1 + x1 w0.
//   FP32          T = 3: x = x0 + x1 + x2 with x0 = bf16(x), x1 = bf16(x - x0),
//     x2 = x - x0 - x1.  Round to nearest leaves remainders of 16 and 8 bits, so the
//     terms hold all 24 bits of x.  Of the nine products of two operands the six
//     with term indexes summing to at most 2 are computed, each exact on the
//     MFMA with FP32 accumulation; the other three come to 2^-24 of the product
//     at most.  So a sum of one product may be off by two half-ulps where an FP32 multiply
//     is off by one (1.82 measured; 3.8% of such products are not correctly rounded),
//     while in longer sums fewer roundings halve the error (9x9 below); the
//     implicit-GEMM hint keeps to FP32 products.  Six BF16 MFMAs do the work of one
//     FP32 MFMA in 6/16 of its cycles.
//
// gfx950 mapping: v_mfma_f32_32x32x16, A = filters (32 output planes x 16 input
// planes at one tap), B = pixels (16 planes x 32 pixels of a row).  A block of
// four waves owns 4*RW x 32 pixels and 32 output planes; a wave owns RW rows.
// Input planes are staged 16 at a time, split, 8 planes (16 bytes) of a pixel to
// an LDS slot; with 16-byte loads of 4 columns where rows are 16-byte aligned
// (BF16, 24 -> 24 planes and the like: 1.02-1.07x the 4-byte loads at up to two
// rows a wave, 0.95x at four, which keeps the 4-byte ones).  For tap column j a
// wave holds the F tap rows of its filters in
// registers and walks down the tile: the pixels of tile row y, read from LDS once
// per tap column, meet tap row i for every output row y - i the wave owns.  So an
// LDS read of a pixel fragment feeds up to F tap rows and a filter fragment RW
// rows: FP32 9x9, RW = 8: 48 16-byte reads of pixels and 27 filter fragments for 432
// MFMAs of 32 cycles a tap column.
// Filter fragments come straight from the packed bank in L2 (1 KiB contiguous
// each) and pass through a ring of registers: each is loaded into the registers of
// the fragment it replaces right after that one's last use, a tap column ahead.
//
// A lane's accumulators hold one pixel of 16 output planes, so a store
// instruction writes whole 32-pixel rows of two planes at any alignment.
//
// Measured against the kernels it replaced (us a call): FP32 9x9, 32 -> 32 planes,
// 8 images 256x256: 730 -> 327; split-BF16 3x3, 64 -> 64 planes, 32 images 128x128:
// 170 -> 122; FP32 2x up-sampled 7x7, 32 -> 32 planes, 8 images 256x256: 485 -> 257 (126 of
// matrix cores at their peak, 55 of output stores); BF16 and FP16 3x3 to 9x9 over 1350
// random calls (3 to 64 planes, 24 to 256 a side): 1.5x.  What bounds it: the matrix cores
// in FP32 (busy 75% of the cycles at 9x9, 69% at 7x7, 62% up-sampled, at the clock that
// the power limit leaves: 327 us are 64% of the nominal rate); for one term the
// latency of staging and of the filter stream (35% busy at 7x7, 49% at 9x9).
#include <algorithm>
#include <type_traits>

#include "epi.h"
#include "lp.h"
#include "stage.h"

namespace cogconv {

typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int FR_RC = 16;  // planes of a staged chunk (one MFMA k slice)
// Whether every 32-pixel run of an output tile is a whole 128-byte line.
__host__ __device__ __forceinline__ bool stream_rows(int OW, const float* out) {
    return (OW & 31) == 0 && (reinterpret_cast<uintptr_t>(out) & 127) == 0;
}

// How taps meet the staged samples.
//   FR_UNIT  unit steps: output row r sees tap row i at staged row r + i.
//   FR_UP0 / FR_UP1  input up-sampled by 2, filter halo h even / odd: output row
//     2r + p sees the tap rows i = h + p (mod 2), at stored row
//     r + ceil((i - h) / 2); staged row 0 is stored row r0 - floor(h / 2); the
//     same for columns.  Wave s of a pair (s = 0, 1) sums the even tap rows of
//     the tap columns j = s (mod 2), then the odd ones of the others: two of the
//     four output phases of its rows, (F*F + 1) / 2 taps for s = 0 and one less
//     for s = 1, half a tap column held at a time.
//   FR_DOWN  every second output.
template <int F, int RW, int S, int T>
struct FrameRows {
    static constexpr bool UP = S == FR_UP0 || S == FR_UP1;
    static constexpr int P = S == FR_UP1;                       // parity of h
    static constexpr int STEP = S == FR_DOWN ? 2 : 1;
    static constexpr int NP = UP ? 2 : 1;                       // phases of a dimension
    static constexpr int off(int i) { return UP ? (i + 1 - P) / 2 : i; }
    static constexpr int taps(int set) { return UP ? (F - set + 1) / 2 : F; }  // even / odd tap rows
    static constexpr int TH = 4 * RW / NP;                      // output rows (of a phase) of a block
    static constexpr int TR = STEP * (TH - 1) + off(F - 1) + 1; // staged rows
    static constexpr int TC = STEP * 31 + off(F - 1) + 1;       // staged columns
    static constexpr int HC = (TC + 1) / 2;                     // FR_DOWN: even columns first, then odd ones
    static constexpr int NPIX = TR * TC;
    // Aligned groups of 4 columns over a tile: it starts up to S4 columns into one
    // (at -h mod 4, for h = 0, (F - 1) / 2 and F - 1).
    static constexpr int S4 = F == 3 ? 3 : (F == 9 ? 0 : 2);
    static constexpr int NG = (TC + S4 + 3) / 4;
    static constexpr int LDS = 2 * T * NPIX * 16 + 16;          // and the tile's extreme magnitudes
};

template <int PREC>
__device__ __forceinline__ floatx16 fr_mfma(typename LpType<PREC>::V a, typename LpType<PREC>::V b, floatx16 c) {
    if constexpr (PREC == COGCONV_FP16)
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// Packed bank: [32-plane output block][16-plane chunk][tap column j][tap row i][term][lane][8], where lane l
// holds output plane l % 32 and input planes 8 (l / 32) .. + 7 (zeros past the planes), taps flipped for the
// convolution orientation.  After it, for the FP32 plans, one uint2 a [block][chunk][j][i]: the fragment's largest
// magnitude (bits), and whether it holds operands under LP_SMALL.
template <int PREC, int T>
__global__ void k_pack_rows(Geom g, PlaneMap m, int Mout, int chunks, long total, const float* __restrict__ Wt,
                            typename LpType<PREC>::T* __restrict__ Wp) {
    typedef typename LpType<PREC>::T E;
    typedef typename LpType<PREC>::V V;
    const int F = g.FH, taps = F * F;
    const bool bpf = m.mode == COGCONV_BACK_PROJECT_FRAME_BLOCK_REDUCE_SUM;
    const int L = m.T / m.N;
    uint2* range = reinterpret_cast<uint2*>(Wp + total * T * 8);
    for (long idx = blockIdx.x * (long)blockDim.x + threadIdx.x; idx < total; idx += (long)gridDim.x * blockDim.x) {
        const int lane = (int)(idx & 63);
        long rest = idx >> 6;
        const int i = (int)(rest % F);
        rest /= F;
        const int j = (int)(rest % F);
        rest /= F;
        const int ch = (int)(rest % chunks);
        const int mm = (int)(rest / chunks) * 32 + (lane & 31);
        const int t = g.flip ? taps - 1 - (i * F + j) : i * F + j;
        V v[T];
        unsigned most = 0u, least = ~0u;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const int r = ch * FR_RC + 8 * (lane >> 5) + e;
            float w = 0.f;
            if (r < m.R && mm < Mout) w = Wt[(size_t)(bpf ? r * L + mm : mm * m.N + r) * taps + t];
            most = max(most, magnitude(w));
            least = min(least, magnitude(w) - 1u);
            E q[T];
            split_terms<T>(w, q);
#pragma unroll
            for (int k = 0; k < T; k++) v[k][e] = q[k];
        }
#pragma unroll
        for (int k = 0; k < T; k++) *reinterpret_cast<V*>(Wp + (((idx >> 6) * T + k) * 64 + lane) * 8) = v[k];
        if (T == 3) {  // `total` is whole waves
            most = wave_max(most);
            const bool small = any_small(least);
            if (lane == 0) range[idx >> 6] = make_uint2(most, small);
        }
    }
}

// VEC: 16-byte staging loads.  STORES: 0 picks the stores' cache policy at run time;
// at four rows a wave, where the two forms side by side spill, 1 is the cached
// and 2 the streamed one.
// INLINE: the workgroup packs its filters itself, chunk by chunk, into LDS: no
// packed bank, one launch.
template <int F, int RW, int MW, int OCC, int S, int PREC, bool VEC, int STORES, bool INLINE>
__global__ __launch_bounds__(256 * MW, OCC) void k_frame_rows(Geom g, PlaneMap m, IgemmCfg c, const float* __restrict__ X,
                                                         const float* __restrict__ Wt,
                                                         const typename LpType<PREC>::T* __restrict__ Wp,
                                                         float* __restrict__ O,
                                                         const cogconv_image_io* __restrict__ tab, Epi e) {
    constexpr int T = lp_terms(PREC);
    typedef FrameRows<F, RW, S, T> Z;
    typedef typename LpType<PREC>::T E;
    typedef typename LpType<PREC>::V V;
    constexpr int TC = Z::TC, NPIX = Z::NPIX, NP = Z::NP, NA = NP * RW, NT = Z::taps(0);
    constexpr bool EXACT = T == 3;  // FP32 results
    static_assert(!EXACT || (!INLINE && MW == 1), "the redo's bounds are those of one packed output block");
    extern __shared__ __attribute__((aligned(16))) unsigned char fr_smem[];
    unsigned* sRange = reinterpret_cast<unsigned*>(fr_smem + 2 * T * NPIX * 16);

    // Output-plane blocks of one tile are adjacent block indices (same XCD).
    int bid = xcd_swizzle(blockIdx.x, gridDim.x);
    const int mGroups = (c.mTiles + MW - 1) / MW;
    const int mg = bid % mGroups * MW;
    bid /= mGroups;
    const int tc = bid % c.tilesC;
    bid /= c.tilesC;
    const int tr = bid % c.tilesR;
    const int b = bid / c.tilesR;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6) & 3;
    // A wave's output block; one past the last works on the last and stores nothing.
    const int mOwn = mg + (MW > 1 ? __builtin_amdgcn_readfirstlane(tid >> 8) : 0), mt = min(mOwn, c.mTiles - 1);
    const int half = lane >> 5, l32 = lane & 31;
    const int pair = wave & 1;  // FR_UP
    const int row0 = (Z::UP ? wave >> 1 : wave) * RW;
    const int Mout = c.Mout, m0 = mt * 32;
    constexpr int NTH = 256 * MW;
    const int HW = g.H * g.W, OHW = g.OH * g.OW;
    const float* Xb = tab ? tab[b].in0 : X + (size_t)b * m.N * HW;
    float* Ob = tab ? tab[b].out : O + (size_t)b * Mout * OHW;
    const __amdgpu_buffer_rsrc_t xr = buffer_rsrc(Xb, (uint32_t)m.N * HW * 4u);  // the plan bounds this by 2^31

    // Staging units of this thread, numbers tid, tid + 256 MW, ...: a pixel (all 16
    // planes of a chunk), or (VEC) 8 planes of an aligned group of 4 columns, which
    // a row of W % 4 == 0 columns holds or leaves out as a whole.  Byte offsets
    // within a plane with the border applied, or out of range (reads 0).
    constexpr int NS = VEC ? (2 * Z::NG * Z::TR + NTH - 1) / NTH : (NPIX + NTH - 1) / NTH;
    // The next chunk's loads run under this one's MFMAs where registers allow.
    constexpr bool AHEAD = NS <= (VEC ? 1 : S == FR_DOWN ? 3 : 2) && !(MW == 2 && RW == 4 && T == 1);
    const int y0 = tr * Z::TH * Z::STEP - (Z::UP ? g.hR >> 1 : g.hR);
    const int x0 = tc * 32 * Z::STEP - (Z::UP ? g.hC >> 1 : g.hC);
    int pOff[NS];
    int pix[VEC ? NS : 1];          // VEC: 4 * (half * T * NPIX + pixel of the group's first column) + clamp
#pragma unroll
    for (int k = 0; k < NS; k++) {
        const int u = tid + NTH * k;
        int ty, x;
        bool live;
        if constexpr (VEC) {
            const int h = u / (Z::NG * Z::TR), q = u - h * (Z::NG * Z::TR);
            ty = q / Z::NG;
            x = (x0 & ~3) + 4 * (q - ty * Z::NG);
            live = h < 2;
            const int side = g.border == COGCONV_BORDER_CLAMP ? (x < 0 ? 1 : (x >= g.W ? 2 : 0)) : 0;
            pix[k] = 4 * (h * T * NPIX + ty * TC + x - x0) + side;
            // The clamped column is in the first or the last group.
            if (side) x = side == 1 ? 0 : g.W - 4;
        } else {
            ty = u / TC;
            const int slot = u - ty * TC;
            x = x0 + (S == FR_DOWN ? (slot < Z::HC ? 2 * slot : 2 * (slot - Z::HC) + 1) : slot);
            live = u < NPIX;
        }
        int y = y0 + ty;
        const int xo = stage_col_offset(g, x);
        bool in = (unsigned)y < (unsigned)g.H;
        if (g.border == COGCONV_BORDER_CYCLIC) {
            y %= g.H;
            y += y < 0 ? g.H : 0;
            in = true;
        } else {
            in = in || g.border == COGCONV_BORDER_CLAMP;
            y = min(max(y, 0), g.H - 1);
        }
        pOff[k] = in && xo >= 0 && live ? 4 * y * g.W + xo : STAGE_OOB;
    }

    // EXACT: the five products with a low term sum apart from the leading one: in
    // one accumulator each would round at the running sum's magnitude, six
    // roundings a slice (9x9, 32 planes: relative error 7.9e-7, 3.0e-7 apart, and
    // 6.4e-7 for the FP32 MFMA kernel, which rounds every 4 planes).
    // Accumulator set * RW + r: row r of the wave (FR_UP: even, odd tap rows).
    floatx16 acc[NA], low[EXACT ? NA : 1];
#pragma unroll
    for (int r = 0; r < NA; r++)
#pragma unroll
        for (int v = 0; v < 16; v++) {
            acc[r][v] = 0.f;
            if (EXACT) low[EXACT ? r : 0][v] = 0.f;
        }

    // The block's filter stream: per (chunk, tap column) F * T fragments of 1 KiB.
    const int chunks = c.RC / FR_RC;
    constexpr int FRAG = 1024, COLB = F * T * FRAG;
    const __amdgpu_buffer_rsrc_t wr = buffer_rsrc(reinterpret_cast<const char*>(Wp) + (size_t)mt * chunks * F * COLB,
                                                  (uint32_t)(chunks * F * COLB));
    // FR_UP: the wave's k-th tap column of a chunk, even tap rows for k < kOdd.
    const int kOdd = (F - pair + 1) / 2;
    auto tap_column = [&](int k) __attribute__((always_inline)) {
        return !Z::UP ? k : (k < kOdd ? pair + 2 * k : 1 - pair + 2 * (k - kOdd));
    };
    // Byte offset of the fragments after column k of chunk ch (past the end: reads 0).
    auto next_column = [&](int ch, int k) __attribute__((always_inline)) {
        ch += k + 1 == F;
        k = k + 1 == F ? 0 : k + 1;
        return lane * 16 + (ch * F + tap_column(k)) * COLB + (Z::UP && k >= kOdd ? T * FRAG : 0);
    };
    // Filters held: a tap column, loaded one ahead, or all F of a chunk (DEEP, where
    // they fit registers), loaded a chunk ahead.
    constexpr bool DEEP = S == FR_UNIT && F == 3 && T == 1 && MW * RW < 8 && !INLINE;
    V a[DEEP ? F : 1][NT][T];
    unsigned char* sFilt = fr_smem + Z::LDS;  // INLINE: the chunk's fragments, in the bank's order
    auto fragment = [&](int at, int i, int t) __attribute__((always_inline)) {
        return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b128(wr, at, (NP * i * T + t) * FRAG, 0));
    };
    if (!INLINE)
#pragma unroll
    for (int k = 0; k < (DEEP ? F : 1); k++)
#pragma unroll
        for (int i = 0; i < NT; i++)
#pragma unroll
            for (int t = 0; t < T; t++) a[k][i][t] = fragment(DEEP ? lane * 16 + k * COLB : next_column(-1, F - 1), i, t);
    // EXACT: whether the bank (smallW) and the tile (sRange[0]) hold operands under LP_SMALL.
    const uint2* range = reinterpret_cast<const uint2*>(Wp + (size_t)c.mTiles * chunks * F * F * T * 512) +
                         (size_t)mt * chunks * F * F;
    bool smallW = false;
    if (EXACT) {
        for (int i = lane; i < chunks * F * F; i += 64) smallW |= range[i].y != 0;
        if (tid < 2) sRange[tid] = 0u;
        __syncthreads();  // before the first chunk's stores
    }

    const int rdBase = ((half * T) * NPIX + row0 * Z::STEP * TC + l32) * 16;
    // The wave's k-th tap column of chunk ch, tap rows of set SET.
    auto column = [&](int ch, int k, auto SET) __attribute__((always_inline)) {
        constexpr int N = Z::taps(SET);
        const int j = tap_column(k), next = DEEP ? lane * 16 + ((ch + 1) * F + k) * COLB : next_column(ch, k);
        const int d = DEEP ? k : 0;
        const int off = S == FR_DOWN ? (j & 1) * Z::HC + (j >> 1) : Z::off(j);
        const unsigned char* bp = fr_smem + rdBase + (Z::off(SET) * TC + off) * 16;
        if (INLINE)
#pragma unroll
            for (int i = 0; i < N; i++)
#pragma unroll
                for (int t = 0; t < T; t++)
                    a[0][i][t] = *reinterpret_cast<const V*>(sFilt + ((k * F + i) * T + t) * FRAG + lane * 16);
#pragma unroll
        for (int y = 0; y < Z::STEP * (RW - 1) + N; y++) {
            V bv[T];
#pragma unroll
            for (int t = 0; t < T; t++) bv[t] = *reinterpret_cast<const V*>(bp + (t * NPIX + y * TC) * 16);
            // Products in order of the pixel term, so the first MFMAs wait for one read only.
#pragma unroll
            for (int tb = 0; tb < T; tb++)
#pragma unroll
                for (int ta = 0; ta + tb < T; ta++)
#pragma unroll
                    for (int i = 0; i < N; i++) {
                        const int r = y - i;
                        if (r < 0 || r % Z::STEP || r / Z::STEP >= RW) continue;
                        const int at = SET * RW + r / Z::STEP;
                        if (!EXACT || ta + tb == 0) acc[at] = fr_mfma<PREC>(a[d][i][ta], bv[tb], acc[at]);
                        else low[EXACT ? at : 0] = fr_mfma<PREC>(a[d][i][ta], bv[tb], low[EXACT ? at : 0]);
                    }
            // A tap row that has met its last row gives its registers to the next tap column's.
            if (!INLINE && y >= Z::STEP * (RW - 1)) {
                const int i = y - Z::STEP * (RW - 1);
#pragma unroll
                for (int t = 0; t < T; t++) a[d][i][t] = fragment(next, i, t);
            }
        }
        // The odd tap rows are one fewer: the last register set is only needed by
        // the even ones of the next chunk.
        if (N < NT)
#pragma unroll
            for (int t = 0; t < T; t++) a[0][NT - 1][t] = fragment(k + 1 == F ? next : STAGE_OOB, NT - 1, t);
    };
    // A chunk is staged in batches of loads: every plane of the thread's units (one
    // memory round trip) where they are loaded ahead, otherwise (VEC) a unit at a
    // time, or a half of the planes of at most 8 pixels.
    constexpr int NB = AHEAD ? NS : VEC ? 1 : NS <= 8 ? NS : 4, HB = !VEC && NS <= (S == FR_DOWN ? 3 : 2) ? 2 : 1;
    float v[NB][VEC ? 1 : 8 * HB];
    floatx4 v4[NB][VEC ? 8 : 1];
    auto load = [&](int ch, int h0, int k0) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < NB; k++) {
            if (k0 + k >= NS) continue;
            if constexpr (VEC) {
                const int r8 = ch * FR_RC + 8 * (tid + NTH * (k0 + k) >= Z::NG * Z::TR);
#pragma unroll
                for (int q = 0; q < 8; q++) {
                    // The plane is per lane (the two halves meet in a wave): plane, then a scalar one.
                    const int at = r8 + q < m.R ? pOff[k0 + k] + 4 * (r8 - ch * FR_RC) * HW : STAGE_OOB;
                    v4[k][q] = __builtin_bit_cast(
                        floatx4, __builtin_amdgcn_raw_buffer_load_b128(xr, pOff[k0 + k] < 0 ? STAGE_OOB : at,
                                                                       4 * (ch * FR_RC + q) * HW, 0));
                }
            } else {
#pragma unroll
                for (int q = 0; q < 8 * HB; q++) {
                    const int r = ch * FR_RC + 8 * h0 + q;
                    v[k][q] = buffer_load_f32(xr, r < m.R ? pOff[k0 + k] : STAGE_OOB, 4 * r * HW);
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);  // keep every load ahead of the first store
    };
    unsigned most = 0u;
    auto store = [&](int h0, int k0) __attribute__((always_inline)) {
        unsigned least = ~0u;
        // One slot: 8 planes of a pixel, every term.
        auto slot = [&](const float (&x)[8], int at) __attribute__((always_inline)) {
            V s[T];
#pragma unroll
            for (int q = 0; q < 8; q++) {
                if (EXACT) {
                    most = max(most, magnitude(x[q]));
                    least = min(least, magnitude(x[q]) - 1u);
                }
                E t3[T];
                split_terms<T>(x[q], t3);
#pragma unroll
                for (int t = 0; t < T; t++) s[t][q] = t3[t];
            }
#pragma unroll
            for (int t = 0; t < T; t++) *reinterpret_cast<V*>(fr_smem + (at + t * NPIX) * 16) = s[t];
        };
#pragma unroll
        for (int k = 0; k < NB; k++) {
            const int u = tid + NTH * (k0 + k);
            if (k0 + k >= NS) continue;
            if constexpr (VEC) {
                if (u >= 2 * Z::NG * Z::TR) continue;
                const int h = u >= Z::NG * Z::TR, q = u - h * (Z::NG * Z::TR);
                const int tx = (x0 & ~3) - x0 + 4 * (q % Z::NG), side = pix[k0 + k] & 3;
#pragma unroll
                for (int c4 = 0; c4 < 4; c4++) {
                    if (tx + c4 < 0 || tx + c4 >= TC) continue;
                    float x[8];
#pragma unroll
                    for (int p = 0; p < 8; p++) {
                        const floatx4 w = v4[k][p];
                        x[p] = w[c4];
                        x[p] = side == 1 ? w[0] : x[p];
                        x[p] = side == 2 ? w[3] : x[p];
                    }
                    slot(x, (pix[k0 + k] >> 2) + c4);
                }
            } else {
                if (u >= NPIX) continue;
#pragma unroll
                for (int h = 0; h < HB; h++) {
                    float x[8];
#pragma unroll
                    for (int p = 0; p < 8; p++) x[p] = v[k][8 * h + p];
                    slot(x, (h0 + h) * T * NPIX + u);
                }
            }
        }
        if (EXACT && any_small(least) && lane == 0) sRange[0] = 1u;
    };
    // INLINE: unit u of a chunk is 8 planes of one output and tap, tap fastest (the
    // order of the filters in memory); FB units of a thread at a time.
    constexpr int FN = F * F * 64, FU = (FN + NTH - 1) / NTH, FB = FU <= 3 ? FU : 4;
    float fv[INLINE ? FB : 1][8];
    const bool bpf = m.mode == COGCONV_BACK_PROJECT_FRAME_BLOCK_REDUCE_SUM;
    const int planeW = (bpf ? m.T / m.N : 1) * F * F * 4;  // bytes between an output's planes
    const __amdgpu_buffer_rsrc_t fr = buffer_rsrc(Wt, (uint32_t)m.T * F * F * 4u);
    auto load_filters = [&](int ch, int k0) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < FB; k++) {
            const int u = tid + NTH * (k0 + k);
            const int t = u % (F * F), mm = u / (F * F) & 31, h = u / (F * F) >> 5;
            const bool live = k0 + k < FU && u < FN && m0 + mm < Mout;
            const int at = ((bpf ? m0 + mm : (m0 + mm) * m.N) * F * F + t) * 4 + 8 * h * planeW;
#pragma unroll
            for (int q = 0; q < 8; q++)
                fv[INLINE ? k : 0][q] = buffer_load_f32(fr, live && ch * FR_RC + 8 * h + q < m.R ? at : STAGE_OOB,
                                                        (ch * FR_RC + q) * planeW);
        }
    };
    auto store_filters = [&](int k0) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < FB; k++) {
            const int u = tid + NTH * (k0 + k);
            if (k0 + k >= FU || u >= FN) continue;
            const int t = u % (F * F), pos = g.flip ? F * F - 1 - t : t;  // tap row pos / F, column pos % F
            V s[T];
#pragma unroll
            for (int q = 0; q < 8; q++) {
                const float w = fv[INLINE ? k : 0][q];
                E t3[T];
                split_terms<T>(w, t3);
#pragma unroll
                for (int e = 0; e < T; e++) s[e][q] = t3[e];
            }
#pragma unroll
            for (int e = 0; e < T; e++)
                *reinterpret_cast<V*>(sFilt + ((pos % F * F + pos / F) * T + e) * FRAG + u / (F * F) * 16) = s[e];
        }
    };
    if (AHEAD) load(0, 0, 0);
    if (INLINE && FB == FU) load_filters(0, 0);
    for (int ch = 0; ch < chunks; ch++) {
        if (ch) __syncthreads();
        if (AHEAD) {
            store(0, 0);
        } else {
#pragma unroll
            for (int h = 0; h < 2; h += VEC ? 2 : HB)
#pragma unroll
                for (int k0 = 0; k0 < NS; k0 += NB) {
                    load(ch, h, k0);
                    store(h, k0);
                }
        }
        if (INLINE) {
            if (FB == FU) {
                store_filters(0);
            } else {
#pragma unroll 1
                for (int k0 = 0; k0 < FU; k0 += FB) {
                    load_filters(ch, k0);
                    store_filters(k0);
                }
            }
        }
        __syncthreads();
        if (AHEAD && ch + 1 < chunks) load(ch + 1, 0, 0);
        if (INLINE && FB == FU && ch + 1 < chunks) load_filters(ch + 1, 0);
        constexpr int UNROLL = DEEP || (INLINE && F == 3) ? F : 1;
#pragma unroll UNROLL
        for (int k = 0; k < (Z::UP ? kOdd : F); k++) column(ch, k, std::integral_constant<int, 0>());
        if constexpr (Z::UP)
#pragma unroll 1
            for (int k = kOdd; k < F; k++) column(ch, k, std::integral_constant<int, 1>());
    }

    // Lane (half, l32), register v of an accumulator: output plane m0 + 8 (v / 4) + 4 half + v % 4, pixel l32
    // of the row.
    const int orow0 = tr * Z::TH + row0, ocol0 = tc * 32 + l32;
    auto out_row = [&](int q) __attribute__((always_inline)) { return NP * (orow0 + q % RW) + (Z::UP ? q / RW ^ Z::P : 0); };
    auto out_col = [&](int q) __attribute__((always_inline)) {
        return NP * ocol0 + (Z::UP ? q / RW ^ pair ^ Z::P : 0);
    };
    // Two kinds of outputs are computed again below, by FP32 MFMAs:
    // non-finite ones (an infinite or NaN operand, or one that rounds to infinity,
    // reaches them as inf * 0 or inf - inf of its terms), and those so small that
    // products or terms under BF16's and FP32's normal range may matter to
    // them: each of the n products of a pair of operands loses at most 2^-123,
    // and where the tile (the bank) holds operands under LP_SMALL, whose
    // last term may be lost, 2^-125 of the bank's (the tile's) largest.  Operands
    // under 2^-134 lose every term, so where the tile or the bank holds small ones
    // a sum of exactly 0 is such an output too (elsewhere it is a sum of zeros).
    float tiny = 0x1p-100f * (float)(chunks * FR_RC * F * F);
    bool zeros = false;
    if (EXACT) {
        constexpr unsigned FINITE = 0x7f7fffffu;
        float bound = 1.f;
        smallW = __any(smallW);  // the same in every wave
        zeros = sRange[0] != 0 || smallW;
        if (sRange[0]) {
            unsigned wMost = 0u;
            for (int i = lane; i < chunks * F * F; i += 64) wMost = max(wMost, range[i].x);
            bound += __uint_as_float(min(wave_max(wMost), FINITE));
        }
        if (smallW) {
            most = wave_max(most);
            if (lane == 0) atomicMax(&sRange[1], most);
            __syncthreads();
            bound += __uint_as_float(min(sRange[1], FINITE));
        }
        tiny *= bound;
    }
    if constexpr (EXACT) {
        float z = 0.f;
        unsigned least = ~0u;  // the smallest magnitude but 0, as 2 bits - 1
#pragma unroll
        for (int r = 0; r < NA; r++)
#pragma unroll
            for (int v = 0; v < 16; v++) {
                acc[r][v] += low[r][v];
                z = fmaf(acc[r][v], 0.f, z);
                least = min(least, (__float_as_uint(acc[r][v]) << 1) - 1u);
            }
        bool redo = z != z;
        if (zeros || least < (__float_as_uint(tiny) << 1) - 1u) {
#pragma unroll
            for (int r = 0; r < NA; r++)
#pragma unroll
                for (int v = 0; v < 16; v++) redo |= fabsf(acc[r][v]) < tiny && (acc[r][v] != 0.f || zeros);
        }
        if (__builtin_expect(__any(redo), 0)) {  // wave-uniform
            // The wave's outputs once more, v_mfma_f32_32x32x2 on operands as they are in
            // memory, two planes a tap (taps off the field multiply 0, as everywhere else;
            // no inserted zero of an up-sampled field multiplies).  A field masked with
            // infinities brings every wave here.  Bound by the scattered filter loads (64 lines
            // of L1 each, for NA rows): one 128x128 image, 32 -> 32 planes, 9x9, a tenth of the
            // samples NaN, 144 us (5.7 ms with a lane summing each of its outputs by itself; 49
            // us without NaNs).
#pragma unroll
            for (int r = 0; r < NA; r++)
#pragma unroll
                for (int v = 0; v < 16; v++) low[r][v] = 0.f;
            const int mm = m0 + l32;
            const int aOff = mm < Mout ? (bpf ? mm : mm * m.N) * F * F * 4 + half * planeW : STAGE_OOB;
            int co[F];  // byte offset of tap column j's sample in a row, of the lane's plane
#pragma unroll
            for (int j = 0; j < F; j++) {
                const int x = Z::UP ? (2 * ocol0 + ((g.hC + j) & 1) - g.hC + j) >> 1 : Z::STEP * ocol0 - g.hC + j;
                co[j] = stage_col_offset(g, x) + half * HW * 4;
            }
#pragma unroll 1
            for (int r0 = 0; r0 < m.R; r0 += 2) {
                const bool live = r0 + half < m.R;
#pragma unroll 1
                for (int i = 0; i < F; i++) {
                    float w[F], a[F];
                    const int row = (g.flip ? F - 1 - i : i) * F * 4;
                    buffer_load_row<F>(fr, live ? aOff : STAGE_OOB, r0 * planeW + row, w);
#pragma unroll
                    for (int j = 0; j < F; j++) a[j] = g.flip ? w[F - 1 - j] : w[j];
#pragma unroll
                    for (int q = 0; q < NA; q++) {
                        int y = Z::STEP * out_row(q) - g.hR + i;
                        if (Z::UP && (y & 1)) continue;
                        y = Z::UP ? y >> 1 : y;
                        bool in = (unsigned)y < (unsigned)g.H;
                        if (g.border == COGCONV_BORDER_CYCLIC) {
                            y %= g.H;
                            y += y < 0 ? g.H : 0;
                            in = true;
                        } else {
                            in = in || g.border == COGCONV_BORDER_CLAMP;
                            y = min(max(y, 0), g.H - 1);
                        }
                        float x[F];
#pragma unroll
                        for (int j = 0; j < F; j++)
                            x[j] = buffer_load_f32(xr, in && live ? co[j] + 4 * y * g.W : STAGE_OOB, 4 * r0 * HW);
#pragma unroll
                        for (int j = 0; j < F; j++) {
                            // The tap columns of the accumulator's column phase (out_col).
                            if (Z::UP && ((g.hC + j) & 1) != ((q / RW ^ pair ^ Z::P) & 1)) continue;
                            low[q] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[j], x[j], low[q], 0, 0, 0);
                        }
                    }
                }
            }
            asm volatile("" : "+v"(tiny));  // (compared anew: the masks of the first comparison would spill)
#pragma unroll
            for (int r = 0; r < NA; r++)
#pragma unroll
                for (int v = 0; v < 16; v++) {
                    const float a = acc[r][v];
                    if (!(fabsf(a) < __builtin_inff()) || (fabsf(a) < tiny && (a != 0.f || zeros))) acc[r][v] = low[r][v];
                }
        }
    }
    if (e.n) {
        // Eight planes of a row at a time in a runtime loop (16 spill registers at
        // three waves a SIMD).
#pragma unroll 1
        for (int t = 0; t < 2 * NA; t++) {
            float v[8];
            int pl[8], pt[8];
            const int mo0 = 16 * (t & 1) + 4 * half;  // plane of v[k]: mo0 + 8 (k / 4) + k % 4
            const int prow = min(out_row(t >> 1), g.OH - 1), pc = min(out_col(t >> 1), g.OW - 1);
#pragma unroll
            for (int q = 0; q < 2 * NA; q++) {
                if (q != t) continue;  // wave-uniform: the accumulators keep compile-time indexes
#pragma unroll
                for (int k = 0; k < 8; k++) v[k] = acc[q >> 1][8 * (q & 1) + k];
            }
#pragma unroll
            for (int k = 0; k < 8; k++) {
                pl[k] = b * Mout + min(m0 + mo0 + 8 * (k >> 2) + (k & 3), Mout - 1);
                pt[k] = prow * g.OW + pc;
            }
            epi_eval_n<8>(e, v, pl, pt);
#pragma unroll
            for (int q = 0; q < 2 * NA; q++) {
                if (q != t) continue;
#pragma unroll
                for (int k = 0; k < 8; k++) acc[q >> 1][8 * (q & 1) + k] = v[k];
            }
        }
    }
    const __amdgpu_buffer_rsrc_t orr = buffer_rsrc(Ob + (size_t)m0 * OHW, (uint32_t)min(32, Mout - m0) * OHW * 4u);
    // Streamed (non-temporal) where a row of 32 pixels is a whole 128-byte line, so
    // that the output does not push the input out of L2; through the caches where
    // lines are shared by two tiles, or by the two waves of an up-sampled pair.
    // (BF16 3x3, 64 -> 64 planes, 32 images: 128x128 100 us streamed, 102 cached, and with
    // 32 input planes 46 and 75; 136x136 135 and 122.)
    auto put = [&](auto POLICY) __attribute__((always_inline)) {
#pragma unroll
        for (int v = 0; v < 16; v++) {
            const int mo = 8 * (v >> 2) + (v & 3);
            const bool ok = m0 + mo + 4 * half < Mout && mOwn == mt;
#pragma unroll
            for (int q = 0; q < NA; q++) {
                const int orow = out_row(q), ocol = out_col(q);
                const int vo = ok && orow < g.OH && ocol < g.OW ? (4 * half * OHW + orow * g.OW + ocol) * 4 : STAGE_OOB;
                const float sum = acc[q][v];
                __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, sum), orr, vo, mo * OHW * 4, POLICY);
            }
        }
    };
    if constexpr (STORES || Z::UP)
        put(std::integral_constant<int, STORES == 2 ? LOAD_NT : 0>());
    else if (stream_rows(g.OW, Ob))
        put(std::integral_constant<int, LOAD_NT>());
    else
        put(std::integral_constant<int, 0>());
}

// The configurations built: (filter, rows a wave, output blocks a workgroup, waves a SIMD, sampling, precision).
#define FR_LP(X, P)                                                                                                \
    X(3, 1, 1, 4, FR_UNIT, P) X(3, 2, 1, 4, FR_UNIT, P) X(3, 4, 1, 3, FR_UNIT, P) X(3, 2, 2, 4, FR_UNIT, P)        \
    X(3, 4, 2, 4, FR_UNIT, P) X(5, 1, 1, 4, FR_UNIT, P) X(5, 2, 1, 4, FR_UNIT, P) X(5, 4, 1, 3, FR_UNIT, P)        \
    X(7, 1, 1, 4, FR_UNIT, P) X(7, 2, 1, 3, FR_UNIT, P) X(7, 4, 1, 3, FR_UNIT, P) X(9, 1, 1, 4, FR_UNIT, P)        \
    X(9, 2, 1, 3, FR_UNIT, P) X(9, 4, 1, 3, FR_UNIT, P)
#define FR_SPLIT(X, F, P) X(F, 1, 1, 3, FR_UNIT, P) X(F, 2, 1, 3, FR_UNIT, P) X(F, 4, 1, 2, FR_UNIT, P)
#define FR_UNIT32(X, P)                                                                                            \
    X(3, 1, 1, 3, FR_UNIT, P) X(3, 2, 1, 3, FR_UNIT, P) X(5, 1, 1, 3, FR_UNIT, P) X(5, 2, 1, 2, FR_UNIT, P)        \
    X(7, 1, 1, 2, FR_UNIT, P) X(7, 2, 1, 2, FR_UNIT, P) X(9, 1, 1, 2, FR_UNIT, P) X(9, 2, 1, 2, FR_UNIT, P)        \
    X(9, 8, 1, 1, FR_UNIT, P)
#define FR_UP2(X, F, S, P) X(F, 1, 1, F < 9 ? 3 : 2, S, P) X(F, 2, 1, 2, S, P)
#define FR_UP(X, P)                                                                                                \
    FR_UP2(X, 3, FR_UP0, P) FR_UP2(X, 3, FR_UP1, P) FR_UP2(X, 5, FR_UP0, P) FR_UP2(X, 7, FR_UP0, P)                \
    FR_UP2(X, 7, FR_UP1, P) FR_UP2(X, 9, FR_UP0, P)
#define FR_DOWN2(X, P)                                                                                             \
    X(3, 1, 1, 2, FR_DOWN, P) X(5, 1, 1, 2, FR_DOWN, P) X(7, 1, 1, 2, FR_DOWN, P) X(9, 1, 1, 2, FR_DOWN, P)
#define FR_CASES(X)                                                                                                \
    FR_UNIT32(X, COGCONV_FP32) FR_UP(X, COGCONV_FP32) FR_DOWN2(X, COGCONV_FP32) FR_LP(X, COGCONV_BF16)             \
    FR_LP(X, COGCONV_FP16) FR_SPLIT(X, 3, COGCONV_SPLIT_BF16) FR_SPLIT(X, 5, COGCONV_SPLIT_BF16)

// Where 16-byte staging loads pay (at four rows a wave their registers cost a block a CU).
static constexpr bool fr_vec(int RW, int S, int prec) { return S == FR_UNIT && prec != COGCONV_FP32 && RW <= 2; }

// Where a workgroup may pack its own filters.  3x3: 1.20x the packed form's time on
// 158 small and middle calls (BF16, FP16, split-BF16; 4 images 75x96, 7 -> 8 planes:
// 7.3 -> 4.8 us), 5x5 BF16 / FP16 1.07x where it wins.  Not built: 7x7 (0.64x: 49
// scattered taps a workgroup and chunk), 5x5 split-BF16 (1.02x where it wins), FP32
// (1.03x).
static constexpr bool fr_inline(int F, int RW, int MW, int S, int prec) {
    return S == FR_UNIT && MW == 1 && prec != COGCONV_FP32 &&
           (F == 3 ? RW <= 2 : F == 5 && RW == 1 && prec != COGCONV_SPLIT_BF16);
}
bool frame_rows_inline(int F, int RW, int MW, int S, int prec) { return fr_inline(F, RW, MW, S, prec); }

static constexpr int fr_stores(int RW, bool stream) { return RW < 4 || RW == 8 ? 0 : 1 + stream; }

static constexpr int fr_key(int F, int RW, int MW, int S, int prec) { return (((prec * 4 + S) * 16 + F) * 16 + RW) * 2 + MW - 1; }

size_t frame_rows_lds_bytes(int F, int RW, int MW, int S, int prec) {
    switch (fr_key(F, RW, MW, S, prec)) {
#define FR_LDS(F, RW, MW, OCC, S, PREC) \
    case fr_key(F, RW, MW, S, PREC): return FrameRows<F, RW, S, lp_terms(PREC)>::LDS;
        FR_CASES(FR_LDS)
#undef FR_LDS
    default: return 0;
    }
}

size_t frame_rows_workspace_bytes(const IgemmCfg& c, int F, int prec) {
    return (size_t)c.mTiles * (c.RC / FR_RC) * F * F * (lp_terms(prec) * 1024 + sizeof(uint2));
}

hipError_t launch_frame_rows(int prec, const Geom& g, const PlaneMap& m, const IgemmCfg& c, const float* x,
                             const float* w, float* out, void* ws, hipStream_t s, int stage, const Epi& ep,
                             const cogconv_image_io* tab, bool x16) {
    const long blocks = (long)c.tilesC * c.tilesR * ((c.mTiles + c.splits - 1) / c.splits) * m.B;
    if (blocks <= 0 || blocks > 0x7fffffffL) return hipErrorInvalidConfiguration;
    if (prec == COGCONV_FP32 && stage != LP_PACK_AND_RUN) return hipErrorInvalidValue;  // the redo reads w itself
    const bool own = c.ring && stage == LP_PACK_AND_RUN;
    if (stage != LP_RUN_ONLY && !own) {
        const long total = (long)c.mTiles * (c.RC / FR_RC) * g.FH * g.FW * 64;
        const dim3 grid((unsigned)std::min((total + 255) / 256, 4096L)), block(256);
        switch (prec) {
#define FR_PACK(PREC)                                                                                              \
    case PREC:                                                                                                     \
        hipLaunchKernelGGL((k_pack_rows<PREC, lp_terms(PREC)>), grid, block, 0, s, g, m, c.Mout, c.RC / FR_RC, total, w, \
                           static_cast<LpType<PREC>::T*>(ws));                                                     \
        break;
            FR_PACK(COGCONV_FP32)
            FR_PACK(COGCONV_BF16)
            FR_PACK(COGCONV_FP16)
            FR_PACK(COGCONV_SPLIT_BF16)
#undef FR_PACK
        default: return hipErrorInvalidValue;
        }
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess || stage == LP_PACK_ONLY) return e;
    }
    const dim3 grid((unsigned)blocks), block(256 * c.splits);
    const bool vec = c.vec4 && (tab ? x16 : (reinterpret_cast<uintptr_t>(x) & 15) == 0);
    const size_t lds = c.lds_bytes + (own ? (size_t)g.FH * g.FW * lp_terms(prec) * 1024 : 0);
    const bool stream = !tab && stream_rows(g.OW, out);
    switch (fr_key(g.FH, c.MB, c.splits, c.variant, prec)) {
#define FR_FORM(F, RW, MW, OCC, S, PREC, VEC, STREAM, OWN) \
    k_frame_rows<F, RW, MW, OCC, S, PREC, VEC, fr_stores(RW, STREAM), OWN && fr_inline(F, RW, MW, S, PREC)>
#define FR_LAUNCH(F, RW, MW, OCC, S, PREC)                                                                         \
    case fr_key(F, RW, MW, S, PREC):                                                                               \
        hipLaunchKernelGGL((own ? (vec ? FR_FORM(F, RW, MW, OCC, S, PREC, fr_vec(RW, S, PREC), false, true)        \
                                       : FR_FORM(F, RW, MW, OCC, S, PREC, false, false, true))                     \
                            : vec    ? FR_FORM(F, RW, MW, OCC, S, PREC, fr_vec(RW, S, PREC), false, false)         \
                            : stream ? FR_FORM(F, RW, MW, OCC, S, PREC, false, true, false)                        \
                                     : FR_FORM(F, RW, MW, OCC, S, PREC, false, false, false)),                     \
                           grid, block, lds, s, g, m, c, x, w, static_cast<const LpType<PREC>::T*>(ws),    \
                           out, tab, ep);                                                                          \
        break;
        FR_CASES(FR_LAUNCH)
#undef FR_LAUNCH
#undef FR_FORM
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace cogconv
