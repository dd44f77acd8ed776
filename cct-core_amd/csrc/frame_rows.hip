// FP32 frame block-reduce modes on the BF16 matrix cores, every FP32 operand
// split exactly into three BF16 terms:
//
//   out[b*Mout + m](y, x) = sum_{r < R} sum_{t < F*F} A[m][r][t] * X_{b*N + r}(y - h + ti, x - h + tj)
//
// (the contraction of igemm_f32.hip; ConvolveHyperKernel.scala:153-167, 327-332,
// borders 235-317).  x = x0 + x1 + x2 with x0 = bf16(x), x1 = bf16(x - x0),
// x2 = x - x0 - x1: round to nearest leaves remainders of 16 and 8 bits, so the
// three terms hold all 24 bits of x.  Of the nine products of two split operands
// the six with term indexes summing to at most 2 are computed, each exact on the
// MFMA with FP32 accumulation; the other three are below 2^-25 of the product,
// under the rounding of one FP32 multiply.  Six BF16 MFMAs do the work of one
// FP32 MFMA in 6/16 of its cycles.
//
// gfx950 mapping: v_mfma_f32_32x32x16_bf16, A = filters (32 output planes x 16
// input planes at one tap), B = pixels (16 planes x 32 pixels of a row).  A block
// of four waves owns 4*RW x 32 pixels and 32 output planes; a wave owns RW rows.
// Input planes are staged 16 at a time, split, 8 planes (16 bytes) of a pixel to
// an LDS slot.  For tap column j a wave holds the F tap rows of its filters in
// registers and walks down the tile: the pixels of tile row y, read from LDS once
// per tap column, meet tap row i for every output row y - i the wave owns.  So an
// LDS read of a pixel fragment feeds up to F tap rows and a filter fragment RW
// rows: RW = 4, 9x9: 63 16-byte reads for 216 MFMAs of 32 cycles a tap column.
// Filter fragments come straight from the packed bank in L2 (1 KiB contiguous
// each), loaded into the registers of the fragment they replace right after its
// last use, a tap column ahead.
//
// A lane's accumulators hold one pixel of 16 output planes, so a store
// instruction writes whole 32-pixel rows of two planes at any alignment.
#include <algorithm>

#include "epi.h"
#include "lp.h"
#include "stage.h"

namespace cogconv {

typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int FR_RC = 16;  // planes of a staged chunk (one MFMA k slice)
// Outputs below this are computed again in plain FP32: operands near its square
// root or above keep every term a normal BF16 number.
constexpr float FR_TINY = 0x1p-100f;

// Splits w into T terms of type V's element: term t rounds what the earlier ones left.
template <int T>
__device__ __forceinline__ void split_terms(float x, __bf16 (&t)[T]) {
#pragma unroll
    for (int k = 0; k < T; k++) {
        t[k] = (__bf16)x;
        if (k + 1 < T) x -= (float)t[k];
    }
}

// Packed bank: [32-plane output block][16-plane chunk][tap column j][tap row i][term][lane][8], where lane l
// holds output plane l % 32 and input planes 8 (l / 32) .. + 7 (zeros past the planes), taps flipped for the
// convolution orientation.
template <int T>
__global__ void k_pack_rows(Geom g, PlaneMap m, int Mout, int chunks, long total, const float* __restrict__ Wt,
                            __bf16* __restrict__ Wp) {
    const int F = g.FH, taps = F * F;
    const bool bpf = m.mode == COGCONV_BACK_PROJECT_FRAME_BLOCK_REDUCE_SUM;
    const int L = m.T / m.N;
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
        bf16x8 v[T];
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const int r = ch * FR_RC + 8 * (lane >> 5) + e;
            float w = 0.f;
            if (r < m.R && mm < Mout) w = Wt[(size_t)(bpf ? r * L + mm : mm * m.N + r) * taps + t];
            __bf16 q[T];
            split_terms<T>(w, q);
#pragma unroll
            for (int k = 0; k < T; k++) v[k][e] = q[k];
        }
#pragma unroll
        for (int k = 0; k < T; k++)
            *reinterpret_cast<bf16x8*>(Wp + (((idx >> 6) * T + k) * 64 + lane) * 8) = v[k];
    }
}

// One output element by plain FP32 multiply-adds, four planes a tap as in the FP32
// MFMA kernel (taps off the field multiply 0, as everywhere else).
__device__ __forceinline__ float frame_point(const Geom& g, const PlaneMap& m, const float* Xb, const float* Wt, int mm,
                                          int orow, int ocol) {
    const bool bpf = m.mode == COGCONV_BACK_PROJECT_FRAME_BLOCK_REDUCE_SUM;
    const int L = m.T / m.N, taps = g.FH * g.FW;
    float s = 0.f;
    for (int r0 = 0; r0 < m.R; r0 += 4)
        for (int i = 0; i < g.FH; i++)
            for (int j = 0; j < g.FW; j++) {
                int y = orow - g.hR + i, c = ocol - g.hC + j;
                bool in = (unsigned)y < (unsigned)g.H && (unsigned)c < (unsigned)g.W;
                if (g.border == COGCONV_BORDER_CYCLIC) {
                    y %= g.H;
                    y += y < 0 ? g.H : 0;
                    c %= g.W;
                    c += c < 0 ? g.W : 0;
                    in = true;
                } else if (g.border == COGCONV_BORDER_CLAMP) {
                    y = min(max(y, 0), g.H - 1);
                    c = min(max(c, 0), g.W - 1);
                    in = true;
                }
                const int t = g.flip ? taps - 1 - (i * g.FW + j) : i * g.FW + j;
                for (int r = r0; r < min(r0 + 4, m.R); r++)
                    s = fmaf(Wt[(size_t)(bpf ? r * L + mm : mm * m.N + r) * taps + t],
                             in ? Xb[((size_t)r * g.H + y) * g.W + c] : 0.f, s);
            }
    return s;
}

template <int F, int RW>
struct FrameRows {
    static constexpr int T = 3;
    static constexpr int TH = 4 * RW;               // output rows of a block
    static constexpr int TR = TH + F - 1;           // staged rows
    static constexpr int TC = 31 + F;               // staged columns
    static constexpr int NPIX = TR * TC;
    static constexpr int LDS = 2 * T * NPIX * 16;
};

template <int F, int RW, int OCC>
__global__ __launch_bounds__(256, OCC) void k_frame_rows(Geom g, PlaneMap m, IgemmCfg c, const float* __restrict__ X,
                                                         const float* __restrict__ Wt, const __bf16* __restrict__ Wp,
                                                         float* __restrict__ O,
                                                         const cogconv_image_io* __restrict__ tab, Epi e) {
    typedef FrameRows<F, RW> S;
    constexpr int T = S::T, TC = S::TC, NPIX = S::NPIX;
    extern __shared__ __attribute__((aligned(16))) unsigned char fr_smem[];

    // Output-plane blocks of one tile are adjacent block indices (same XCD).
    int bid = xcd_swizzle(blockIdx.x, gridDim.x);
    const int mt = bid % c.mTiles;
    bid /= c.mTiles;
    const int tc = bid % c.tilesC;
    bid /= c.tilesC;
    const int tr = bid % c.tilesR;
    const int b = bid / c.tilesR;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int half = lane >> 5, l32 = lane & 31;
    const int Mout = c.Mout, m0 = mt * 32;
    const int HW = g.H * g.W, OHW = g.OH * g.OW;
    const float* Xb = tab ? tab[b].in0 : X + (size_t)b * m.N * HW;
    float* Ob = tab ? tab[b].out : O + (size_t)b * Mout * OHW;
    const __amdgpu_buffer_rsrc_t xr = buffer_rsrc(Xb, (uint32_t)m.N * HW * 4u);  // the plan bounds this by 2^31

    // Staged pixels of this thread: tid, tid + 256, ...; byte offsets within a
    // plane with the border applied, or out of range (reads 0).
    constexpr int NS = (NPIX + 255) / 256;
    int pOff[NS];
#pragma unroll
    for (int k = 0; k < NS; k++) {
        const int p = tid + 256 * k;
        const int ty = p / TC, tx = p - ty * TC;
        int y = tr * S::TH - g.hR + ty;
        const int xo = stage_col_offset(g, tc * 32 - g.hC + tx);
        bool in = (unsigned)y < (unsigned)g.H;
        if (g.border == COGCONV_BORDER_CYCLIC) {
            y %= g.H;
            y += y < 0 ? g.H : 0;
            in = true;
        } else {
            in = in || g.border == COGCONV_BORDER_CLAMP;
            y = min(max(y, 0), g.H - 1);
        }
        pOff[k] = in && xo >= 0 && p < NPIX ? 4 * y * g.W + xo : STAGE_OOB;
    }

    // The five products with a low term sum apart from the leading one: in one
    // accumulator each would round at the running sum's magnitude, six roundings
    // a slice (9x9, 32 planes: relative error 7.9e-7, 3.0e-7 apart, and
    // 6.4e-7 for the FP32 MFMA kernel, which rounds every 4 planes).
    floatx16 acc[RW], low[RW];
#pragma unroll
    for (int r = 0; r < RW; r++)
#pragma unroll
        for (int v = 0; v < 16; v++) acc[r][v] = low[r][v] = 0.f;

    // The block's filter stream: per (chunk, tap column) F * T fragments of 1 KiB.
    const int chunks = c.RC / FR_RC;
    constexpr int FRAG = 1024, COLB = F * T * FRAG;
    const __amdgpu_buffer_rsrc_t wr = buffer_rsrc(reinterpret_cast<const char*>(Wp) + (size_t)mt * chunks * F * COLB,
                                                  (uint32_t)(chunks * F * COLB));
    int wOff = lane * 16;  // of the tap column whose fragments are loaded next (past the end: reads 0)
    bf16x8 a[F][T];
#pragma unroll
    for (int i = 0; i < F; i++)
#pragma unroll
        for (int t = 0; t < T; t++)
            a[i][t] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(wr, wOff, (i * T + t) * FRAG, 0));
    wOff += COLB;

    const int rdBase = ((half * T) * NPIX + wave * RW * TC + l32) * 16;
    for (int ch = 0; ch < chunks; ch++) {
        if (ch) __syncthreads();
#pragma unroll
        for (int h = 0; h < 2; h++) {
            // Batches of at most 8 pixels (64 loads in flight a thread).
            constexpr int NB = NS <= 8 ? NS : 4;
#pragma unroll
            for (int k0 = 0; k0 < NS; k0 += NB) {
                float v[NB][8];
#pragma unroll
                for (int k = 0; k < NB; k++) {
                    if (k0 + k >= NS) continue;
#pragma unroll
                    for (int q = 0; q < 8; q++) {
                        const int r = ch * FR_RC + 8 * h + q;
                        v[k][q] = buffer_load_f32(xr, r < m.R ? pOff[k0 + k] : STAGE_OOB, 4 * r * HW);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);  // keep every load ahead of the first store
#pragma unroll
                for (int k = 0; k < NB; k++) {
                    const int p = tid + 256 * (k0 + k);
                    if (k0 + k >= NS || p >= NPIX) continue;
                    bf16x8 s[T];
#pragma unroll
                    for (int q = 0; q < 8; q++) {
                        __bf16 t3[T];
                        split_terms<T>(v[k][q], t3);
#pragma unroll
                        for (int t = 0; t < T; t++) s[t][q] = t3[t];
                    }
#pragma unroll
                    for (int t = 0; t < T; t++)
                        *reinterpret_cast<bf16x8*>(fr_smem + ((h * T + t) * NPIX + p) * 16) = s[t];
                }
            }
        }
        __syncthreads();
#pragma unroll 1
        for (int j = 0; j < F; j++) {
            const unsigned char* bp = fr_smem + rdBase + j * 16;
#pragma unroll
            for (int y = 0; y < RW + F - 1; y++) {
                bf16x8 bv[T];
#pragma unroll
                for (int t = 0; t < T; t++) bv[t] = *reinterpret_cast<const bf16x8*>(bp + (t * NPIX + y * TC) * 16);
                // Products in order of the pixel term, so the first MFMAs wait for one read only.
#pragma unroll
                for (int tb = 0; tb < T; tb++)
#pragma unroll
                    for (int ta = 0; ta + tb < T; ta++)
#pragma unroll
                        for (int i = 0; i < F; i++) {
                            const int r = y - i;
                            if (r < 0 || r >= RW) continue;
                            if (ta + tb == 0)
                                acc[r] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i][0], bv[0], acc[r], 0, 0, 0);
                            else
                                low[r] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i][ta], bv[tb], low[r], 0, 0, 0);
                        }
                // Tap row y - (RW - 1) has met its last row: its registers take the next tap column's.
                if (y >= RW - 1) {
                    const int i = y - (RW - 1);
#pragma unroll
                    for (int t = 0; t < T; t++)
                        a[i][t] = __builtin_bit_cast(
                            bf16x8, __builtin_amdgcn_raw_buffer_load_b128(wr, wOff, (i * T + t) * FRAG, 0));
                }
            }
            wOff += COLB;
        }
    }

    // Lane (half, l32), register v of acc[r]: output plane m0 + 8 (v / 4) + 4 half + v % 4, pixel l32 of the
    // wave's row r.
    const int orow0 = tr * S::TH + wave * RW, ocol = tc * 32 + l32;
    // Two kinds of outputs are computed again below, by plain FP32 multiply-adds:
    // non-finite ones (an infinite or NaN operand, or one that rounds to infinity,
    // reaches them as inf * 0 or inf - inf of its terms), and those below
    // FR_TINY, where the low terms of operands run out of BF16's exponents.
    float z = 0.f;
    bool redo = false;
#pragma unroll
    for (int r = 0; r < RW; r++)
#pragma unroll
        for (int v = 0; v < 16; v++) {
            acc[r][v] += low[r][v];
            z = fmaf(acc[r][v], 0.f, z);
            redo |= fabsf(acc[r][v]) < FR_TINY && acc[r][v] != 0.f;
        }
    const int pc = min(ocol, g.OW - 1);
    if (e.n || __any(redo || z != z)) {  // wave-uniform
        // Eight planes of a row at a time in a runtime loop (16 spill registers at
        // three waves a SIMD).
#pragma unroll 1
        for (int t = 0; t < 2 * RW; t++) {
            float v[8];
            int pl[8], pt[8];
            const int r = t >> 1, mo0 = 16 * (t & 1) + 4 * half;  // plane of v[k]: mo0 + 8 (k / 4) + k % 4
            const int prow = min(orow0 + r, g.OH - 1);
#pragma unroll
            for (int q = 0; q < 2 * RW; q++) {
                if (q != t) continue;  // wave-uniform: the accumulators keep compile-time indexes
#pragma unroll
                for (int k = 0; k < 8; k++) v[k] = acc[q >> 1][8 * (q & 1) + k];
            }
            unsigned again = 0;
#pragma unroll
            for (int k = 0; k < 8; k++) {
                const int mm = m0 + mo0 + 8 * (k >> 2) + (k & 3);
                const float a = fabsf(v[k]);
                if (mm < Mout && (!(a < __builtin_inff()) || (a < FR_TINY && v[k] != 0.f))) again |= 1u << k;
                pl[k] = b * Mout + min(mm, Mout - 1);
                pt[k] = prow * g.OW + pc;
            }
            if (orow0 + r >= g.OH || ocol >= g.OW) again = 0;
            while (again) {
                const int k = __builtin_ctz(again);
                again &= again - 1;
                const float s = frame_point(g, m, Xb, Wt, m0 + mo0 + 8 * (k >> 2) + (k & 3), prow, pc);
#pragma unroll
                for (int q = 0; q < 8; q++) v[q] = q == k ? s : v[q];
            }
            if (e.n) epi_eval_n<8>(e, v, pl, pt);
#pragma unroll
            for (int q = 0; q < 2 * RW; q++) {
                if (q != t) continue;
#pragma unroll
                for (int k = 0; k < 8; k++) acc[q >> 1][8 * (q & 1) + k] = v[k];
            }
        }
    }
    const __amdgpu_buffer_rsrc_t orr = buffer_rsrc(Ob + (size_t)m0 * OHW, (uint32_t)min(32, Mout - m0) * OHW * 4u);
#pragma unroll
    for (int v = 0; v < 16; v++) {
        const int mo = 8 * (v >> 2) + (v & 3);
        const bool ok = m0 + mo + 4 * half < Mout && ocol < g.OW;
#pragma unroll
        for (int r = 0; r < RW; r++) {
            const int vo = ok && orow0 + r < g.OH ? (4 * half * OHW + (orow0 + r) * g.OW + ocol) * 4 : STAGE_OOB;
            const float sum = acc[r][v];
            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, sum), orr, vo, mo * OHW * 4, LOAD_NT);
        }
    }
}

bool frame_rows_supported(int F) { return F == 3 || F == 5 || F == 7 || F == 9; }

size_t frame_rows_lds_bytes(int F, int RW) {
    switch (F * 10 + RW) {
    case 31: return FrameRows<3, 1>::LDS;
    case 51: return FrameRows<5, 1>::LDS;
    case 71: return FrameRows<7, 1>::LDS;
    case 91: return FrameRows<9, 1>::LDS;
    case 32: return FrameRows<3, 2>::LDS;
    case 52: return FrameRows<5, 2>::LDS;
    case 72: return FrameRows<7, 2>::LDS;
    case 92: return FrameRows<9, 2>::LDS;
    case 98: return FrameRows<9, 8>::LDS;
    default: return 0;
    }
}

size_t frame_rows_workspace_bytes(const IgemmCfg& c, int F) {
    return (size_t)c.mTiles * (c.RC / FR_RC) * F * F * 3 * 1024;
}

hipError_t launch_frame_rows(const Geom& g, const PlaneMap& m, const IgemmCfg& c, const float* x, const float* w,
                             float* out, void* ws, hipStream_t s, const Epi& ep, const cogconv_image_io* tab) {
    const long blocks = (long)c.tilesC * c.tilesR * c.mTiles * m.B;
    if (blocks <= 0 || blocks > 0x7fffffffL) return hipErrorInvalidConfiguration;
    __bf16* wp = static_cast<__bf16*>(ws);
    const long total = (long)c.mTiles * (c.RC / FR_RC) * g.FH * g.FW * 64;
    hipLaunchKernelGGL((k_pack_rows<3>), dim3((unsigned)std::min((total + 255) / 256, 4096L)), dim3(256), 0, s, g, m,
                       c.Mout, c.RC / FR_RC, total, w, wp);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const dim3 grid((unsigned)blocks), block(256);
#define FR_CASE(F, RW, OCC)                                                                                         \
    case F * 10 + RW:                                                                                               \
        hipLaunchKernelGGL((k_frame_rows<F, RW, OCC>), grid, block, c.lds_bytes, s, g, m, c, x, w, wp, out, tab, ep); \
        break;
    switch (g.FH * 10 + c.MB) {
        FR_CASE(3, 1, 3)
        FR_CASE(5, 1, 3)
        FR_CASE(7, 1, 2)
        FR_CASE(9, 1, 2)
        FR_CASE(3, 2, 3)
        FR_CASE(5, 2, 2)
        FR_CASE(7, 2, 2)
        FR_CASE(9, 2, 2)
        FR_CASE(9, 8, 1)
    default: return hipErrorInvalidValue;
    }
#undef FR_CASE
    return hipGetLastError();
}

}  // namespace cogconv
