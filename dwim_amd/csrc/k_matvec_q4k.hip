// Q4_K products of a batch of n tokens, routed by size (dwim gpu/cpu.rs:110-149
// is the product, gpu/mod.rs:259 the add, gpu/mod.rs:274-285 the SwiGLU): up to
// four tokens go to the int8 matrix-core matrix-vector kernels
// (k_mv_q4k_mfma.hip, k_mv_q4k_stream.hip), up to 64 to the kernels of the other
// formats (k_rows_few.hip, k_gemm_rows.hip), larger batches to the f16
// matrix-core GEMM of 128-token tiles (k_gemm_q4k.hip).
// Measured on MI355X, us: a 17408×5120 SwiGLU pair at 5 tokens 55 (two runs of
// the few-token kernel 63), at 16 50 (the 128-token tiles 99), at 32 62 (102), at
// 64 84 (114), at 128 172 (131); x += W·h 5120×17408 at 5 33 (49), 16 35 (102), 64
// 81 (106); 1024×1024 at 16 8.4 (28).
#include "runtime.h"

// rmsnorm(x)·norm in `to` or the device's work scratch; x itself without a norm
static const float *normalized(dwim_dev *dev, const float *x, const float *norm, float eps, size_t n, size_t cols,
                               float *to) {
    if (!norm) return x;
    float *xn = to ? to : dev_work(dev, n * cols);
    return xn && launch_rmsnorm(dev->stream, xn, x, norm, n, cols, eps) == hipSuccess ? xn : nullptr;
}

// Q4_K products may be in place.  The kernel of 5 to 64 tokens reads x while
// other workgroups write results; the int8 kernels and the GEMM read it in a
// launch of its own first, so products in place go to those (runs of four
// tokens below kGemmInPlace, whose rows are read before they are written).
constexpr size_t kGemmInPlace = 16;
static bool by_rows(size_t n, const float *out, const float *x) { return n >= kRowsQ4kTokens && n < kGemmTokens && out != x; }
static bool by_gemm(size_t n, const float *out, const float *x) { return n >= (out == x ? kGemmInPlace : kGemmTokens); }

hipError_t launch_matvec_q4k(dwim_dev *dev, const dwim_weight *w, float *out, const float *x, size_t n, int add) {
    if (by_rows(n, out, x)) return launch_rows(dev, w, nullptr, out, x, n, add);
    if (by_gemm(n, out, x)) return launch_gemm_q4k(dev, w, out, x, n, add);
    return launch_mv_q4k_mfma_tokens(dev, &w, &out, &add, 1, 0, x, n, nullptr, 0.0f, nullptr);
}

hipError_t launch_matvec_q4k_multi(dwim_dev *dev, const dwim_weight *const *ws, float *const *outs, int count,
                                   const float *x, size_t n, const float *norm, float eps, float *xn_out) {
    if (count < 1 || count > 4) return hipErrorInvalidValue;
    for (int j = 0; j < count; j++)
        if (ws[j]->cols != ws[0]->cols || ws[j]->fmt != DWIM_Q4_K) return hipErrorInvalidValue;
    if (n < kRowsQ4kTokens) return launch_mv_q4k_mfma_tokens(dev, ws, outs, nullptr, count, 0, x, n, norm, eps, xn_out);
    if (n < kGemmTokens) {
        const float *xn = normalized(dev, x, norm, eps, n, ws[0]->cols, xn_out);
        if (!xn) return hipErrorOutOfMemory;
        bool split = false;  // the activations' parts, shared by the matrices
        for (int j = 0; j < count; j++) {
            const hipError_t e = launch_rows(dev, ws[j], nullptr, outs[j], xn, n, 0, &split);
            if (e != hipSuccess) return e;
        }
        return hipSuccess;
    }
    {
        hipError_t e = norm ? gemm_prepare_rms(dev, x, norm, eps, n, ws[0]->cols, xn_out)
                            : gemm_prepare(dev, x, n, ws[0]->cols);
        for (int j = 0; j < count && e == hipSuccess; j++) e = gemm_run(dev, ws[j], outs[j], n, kGemmStore);
        return e;
    }
}

hipError_t launch_swiglu_q4k(dwim_dev *dev, const dwim_weight *gate, const dwim_weight *up, float *out, const float *x,
                             size_t n, const float *norm, float eps) {
    if (gate->rows != up->rows || gate->cols != up->cols) return hipErrorInvalidValue;
    if (by_rows(n, out, x)) {
        const float *xn = normalized(dev, x, norm, eps, n, gate->cols, nullptr);
        return xn ? launch_rows(dev, gate, up, out, xn, n, 0) : hipErrorOutOfMemory;
    }
    if (!by_gemm(n, out, x)) {
        const dwim_weight *ws[2] = {gate, up};
        float *outs[2] = {out, nullptr};
        return launch_mv_q4k_mfma_tokens(dev, ws, outs, nullptr, 2, 1, x, n, norm, eps, nullptr);
    }
    {
        // x normalized, split once; gate·x into out, then out = silu(out)·(up·x)
        const size_t cols = gate->cols;
        hipError_t e = norm ? gemm_prepare_rms(dev, x, norm, eps, n, cols, nullptr) : gemm_prepare(dev, x, n, cols);
        if (e == hipSuccess) e = gemm_run(dev, gate, out, n, kGemmStore);
        if (e == hipSuccess) e = gemm_run(dev, up, out, n, kGemmSiluGate);
        return e;
    }
}

hipError_t launch_ffn_q4k(dwim_dev *dev, const dwim_weight *gate, const dwim_weight *up, const dwim_weight *down,
                          float *x, size_t n, const float *norm, float eps, float *g, float *u) {
    if (n < kGemmTokens || gate->fmt != DWIM_Q4_K || down->fmt != DWIM_Q4_K || down->cols != gate->rows)
        return hipErrorInvalidValue;
    hipError_t e = gemm_prepare_rms(dev, x, norm, eps, n, gate->cols, nullptr);
    if (e == hipSuccess) e = gemm_run_swiglu_pair(dev, gate, up, g, u, n);
    if (e == hipSuccess) e = gemm_run(dev, down, x, n, kGemmAdd);
    return e;
}
