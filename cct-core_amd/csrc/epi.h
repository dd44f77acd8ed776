// Elementwise epilogue applied to every output element at its store: the
// device side of cogconv_plan_set_epilogue (see Epi in internal.h).
//
// The ops run in order on the value in registers, each as one IEEE float
// operation (or one call of the device math library for exp / log / sqrt /
// tanh), with contraction off, so that a fused store gives bit for bit what
// the same ops give when they run as their own pass over the stored output
// (k_elementwise).
#pragma once

#include "internal.h"

namespace cogconv {

__device__ __forceinline__ float epi_operand(const Epi& e, int slot, int plane, int point) {
    const size_t at = (size_t)(e.srcPlanes[slot] == 1 ? 0 : plane) * e.srcPoints[slot] +
                      (e.srcPoints[slot] == 1 ? 0 : point);
    return e.src[slot][at];
}

__device__ __forceinline__ float epi_eval(const Epi& e, float v, int plane, int point) {
#pragma clang fp contract(off)
    for (int i = 0; i < e.n; i++) {
        const int op = e.op[i];
        float a = e.val[i];
        if (op >= COGCONV_EPI_ADD_FIELD) a = epi_operand(e, e.slot[i], plane, point);
        switch (op) {
        case COGCONV_EPI_ADD_CONST:
        case COGCONV_EPI_ADD_FIELD: v = v + a; break;
        case COGCONV_EPI_SUB_CONST:
        case COGCONV_EPI_SUB_FIELD: v = v - a; break;
        case COGCONV_EPI_RSUB_CONST:
        case COGCONV_EPI_RSUB_FIELD: v = a - v; break;
        case COGCONV_EPI_MUL_CONST:
        case COGCONV_EPI_MUL_FIELD: v = v * a; break;
        case COGCONV_EPI_DIV_CONST:
        case COGCONV_EPI_DIV_FIELD: v = v / a; break;
        case COGCONV_EPI_RDIV_CONST:
        case COGCONV_EPI_RDIV_FIELD: v = a / v; break;
        case COGCONV_EPI_MAX_CONST:
        case COGCONV_EPI_MAX_FIELD: v = fmaxf(v, a); break;
        case COGCONV_EPI_MIN_CONST:
        case COGCONV_EPI_MIN_FIELD: v = fminf(v, a); break;
        case COGCONV_EPI_NEG: v = -v; break;
        case COGCONV_EPI_ABS: v = fabsf(v); break;
        case COGCONV_EPI_SQ: v = v * v; break;
        case COGCONV_EPI_SQRT: v = sqrtf(v); break;
        case COGCONV_EPI_EXP: v = expf(v); break;
        case COGCONV_EPI_LOG: v = logf(v); break;
        case COGCONV_EPI_TANH: v = tanhf(v); break;
        case COGCONV_EPI_SIGNUM: v = v > 0.f ? 1.f : (v < 0.f ? -1.f : 0.f); break;
        default: break;
        }
    }
    return v;
}

// Four adjacent output elements (16-byte aligned) as one store: non-temporal
// (streamed to memory, no cache line kept) when no epilogue reads them back.
__device__ __forceinline__ void store_out4(float* p, float a, float b, float c, float d, const Epi& e) {
    typedef float f4 __attribute__((ext_vector_type(4)));
    const f4 v = {a, b, c, d};
    if (e.n == 0)
        __builtin_nontemporal_store(v, reinterpret_cast<f4*>(p));
    else
        *reinterpret_cast<f4*>(p) = v;
}

// The value stored for output element (plane, point): v itself without an epilogue.
__device__ __forceinline__ float epi(const Epi& e, float v, int plane, int point) {
    return e.n == 0 ? v : epi_eval(e, v, plane, point);
}

// The epilogue over N output elements of a thread, op by op: the descriptor's
// fields (scalar loads of a runtime op index) are fetched once per op instead of
// once per op and element, and the N operand loads of a field op are in flight
// together.  Element by element these dependent loads were most of a small
// launch: bias and rectifier on 16 images 64x64x16 -> 32 planes, 3x3, took
// 22.7 us, and 13.8 us this way (12.4 us without an epilogue).  Every (plane, point)
// must be a valid output element, also where the caller does not store the result.
template <int N>
__device__ __forceinline__ void epi_eval_n(const Epi& e, float (&v)[N], const int (&plane)[N], const int (&point)[N]) {
#pragma clang fp contract(off)
    for (int i = 0; i < e.n; i++) {
        const int op = e.op[i];
        float a[N];
        if (op >= COGCONV_EPI_ADD_FIELD) {
            const int slot = e.slot[i];
            const float* src = e.src[slot];
            const size_t points = (size_t)e.srcPoints[slot];
            const bool perPlane = e.srcPlanes[slot] != 1, perPoint = e.srcPoints[slot] != 1;
#pragma unroll
            for (int k = 0; k < N; k++) a[k] = src[(perPlane ? plane[k] : 0) * points + (perPoint ? point[k] : 0)];
        } else {
            const float c = e.val[i];
#pragma unroll
            for (int k = 0; k < N; k++) a[k] = c;
        }
#define COGCONV_EPI_EACH(expr)        \
    {                                 \
        _Pragma("unroll")             \
        for (int k = 0; k < N; k++) { \
            const float x = v[k];     \
            const float y = a[k];     \
            (void)y;                  \
            v[k] = (expr);            \
        }                             \
        break;                        \
    }
        switch (op) {
        case COGCONV_EPI_ADD_CONST:
        case COGCONV_EPI_ADD_FIELD: COGCONV_EPI_EACH(x + y)
        case COGCONV_EPI_SUB_CONST:
        case COGCONV_EPI_SUB_FIELD: COGCONV_EPI_EACH(x - y)
        case COGCONV_EPI_RSUB_CONST:
        case COGCONV_EPI_RSUB_FIELD: COGCONV_EPI_EACH(y - x)
        case COGCONV_EPI_MUL_CONST:
        case COGCONV_EPI_MUL_FIELD: COGCONV_EPI_EACH(x * y)
        case COGCONV_EPI_DIV_CONST:
        case COGCONV_EPI_DIV_FIELD: COGCONV_EPI_EACH(x / y)
        case COGCONV_EPI_RDIV_CONST:
        case COGCONV_EPI_RDIV_FIELD: COGCONV_EPI_EACH(y / x)
        case COGCONV_EPI_MAX_CONST:
        case COGCONV_EPI_MAX_FIELD: COGCONV_EPI_EACH(fmaxf(x, y))
        case COGCONV_EPI_MIN_CONST:
        case COGCONV_EPI_MIN_FIELD: COGCONV_EPI_EACH(fminf(x, y))
        case COGCONV_EPI_NEG: COGCONV_EPI_EACH(-x)
        case COGCONV_EPI_ABS: COGCONV_EPI_EACH(fabsf(x))
        case COGCONV_EPI_SQ: COGCONV_EPI_EACH(x * x)
        case COGCONV_EPI_SQRT: COGCONV_EPI_EACH(sqrtf(x))
        case COGCONV_EPI_EXP: COGCONV_EPI_EACH(expf(x))
        case COGCONV_EPI_LOG: COGCONV_EPI_EACH(logf(x))
        case COGCONV_EPI_TANH: COGCONV_EPI_EACH(tanhf(x))
        case COGCONV_EPI_SIGNUM: COGCONV_EPI_EACH(x > 0.f ? 1.f : (x < 0.f ? -1.f : 0.f))
        default: break;
        }
#undef COGCONV_EPI_EACH
    }
}

// Re-applies the epilogue to the N adjacent elements from p, of which this
// thread has just stored the first `n` (kernels whose accumulator arrays must
// stay in registers store them plainly first).  A thread reads its own earlier
// stores in program order, so no fence is needed.
template <int N>
__device__ __forceinline__ void epi_rewrite(const Epi& e, float* p, int n, int plane, int point) {
    float v[N];
    int pl[N], pt[N];
#pragma unroll
    for (int k = 0; k < N; k++) {
        const int q = min(k, n - 1);
        v[k] = p[q];
        pl[k] = plane;
        pt[k] = point + q;
    }
    epi_eval_n<N>(e, v, pl, pt);
#pragma unroll
    for (int k = 0; k < N; k++)
        if (k < n) p[k] = v[k];
}

}  // namespace cogconv
