// Matrix products by format and batch size: out[t][r] (+)= w[r] · x[t] (dwim
// gpu/cpu.rs:110-149, Device::matmul), and the kernel for a
// few tokens through bf16 matrices of few rows (DeltaNet's gate projection) on
// the vector ALUs.
#include "device_util.h"
#include "quant_math.h"
#include "runtime.h"

#include <algorithm>

// A few tokens (a verify batch) through a bf16 matrix of few rows: a block of
// 256 threads per row and run of up to 4 tokens, thread i summing columns
// 8i.. in steps of 2048 for each token (16-byte weight loads, read once for
// the run), then the block's sums meet per token.  Enough blocks to spread the
// rows' bytes over the chip: 96 × 5120 is 96 blocks of 40 KB.
constexpr int kRowTok = 4, kSkRows = 96;

__global__ void __launch_bounds__(256) k_rows_bf16(const uint16_t *__restrict__ w, const float *__restrict__ x,
                                                   float *__restrict__ out, size_t rows, size_t cols, size_t n,
                                                   int add) {
    __shared__ float part[kRowTok][4];
    const size_t row = blockIdx.x, t0 = (size_t)blockIdx.y * kRowTok;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int nt = (int)(n - t0 < (size_t)kRowTok ? n - t0 : (size_t)kRowTok);
    float acc[kRowTok] = {0.0f, 0.0f, 0.0f, 0.0f};
    const uint16_t *wr = w + row * cols;
    for (size_t c = 8 * (size_t)tid; c < cols; c += 8 * 256) {
        const uint4 q = *(const uint4 *)(wr + c);
        const uint32_t v[4] = {q.x, q.y, q.z, q.w};
        float wf[8];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            wf[2 * i] = dq::bf16_to_f32((uint16_t)(v[i] & 0xffffu));
            wf[2 * i + 1] = dq::bf16_to_f32((uint16_t)(v[i] >> 16));
        }
#pragma unroll
        for (int t = 0; t < kRowTok; t++) {
            if (t >= nt) break;
            const float4 a = *(const float4 *)(x + (t0 + t) * cols + c), b = *(const float4 *)(x + (t0 + t) * cols + c + 4);
            acc[t] += ((wf[0] * a.x + wf[1] * a.y) + (wf[2] * a.z + wf[3] * a.w)) +
                      ((wf[4] * b.x + wf[5] * b.y) + (wf[6] * b.z + wf[7] * b.w));
        }
    }
#pragma unroll
    for (int t = 0; t < kRowTok; t++) {
        const float v = group_sum<64>(acc[t]);
        if (lane == 0) part[t][wave] = v;
    }
    __syncthreads();
    if (tid < nt) {
        const float v = (part[tid][0] + part[tid][1]) + (part[tid][2] + part[tid][3]);
        float *o = out + (t0 + tid) * rows + row;
        *o = add ? *o + v : v;
    }
}

// The most tokens that go through the kernel that converts the activations
// itself (k_rows_few.hip); more go through the GEMM (k_gemm_rows.hip), whose
// split of the activations and sum of the parts are launches of their own.
// Measured on MI355X (us, few | GEMM): a 17408×5120 Q4_0 pair at 16 tokens 43 |
// 44, at 32 66 | 48; Q8_0 at 16 53 | 53, at 32 79 | 57; Q6_K at 16 56 | 72, at 32 93
// | 76; bf16 at 32 113 | 121, at 64 254 | 139; a 2304×3072 Q8_0 pair at 32 17.5 | 17.8,
// at 64 32 | 24; 5120×17408 Q4_0 at 16 32 | 47, at 32 44 | 48, at 64 75 | 68; Q6_K,
// whose GEMM scales every 16 columns, at 64 93 | 116; 1024×1024 Q4_0 at 64 12 | 15.
static size_t few_tokens(const dwim_weight *w, bool pair) {
    const bool small = w->rows * w->cols <= (size_t)8 << 20;
    if (!pair && (small || w->fmt == DWIM_Q6_K)) return 64;
    return small || w->fmt == DWIM_BF16 || w->cols >= 2 * w->rows ? 32 : 16;
}

hipError_t launch_rows(dwim_dev *dev, const dwim_weight *w, const dwim_weight *up, float *out, const float *x, size_t n,
                       int add, bool *split) {
    if (n > few_tokens(w, up)) {
        const hipError_t e = launch_gemm_rows(dev, w, up, out, x, n, add, split && *split);
        if (e == hipSuccess && split) *split = true;
        if (e != hipErrorNotSupported) return e;
    }
    // (also a batch whose GEMM cannot have its scratch: the weights read again
    // for every run of tokens)
    const size_t most = std::min((size_t)(up ? 32 : 64), std::max((size_t)1, ((size_t)1 << 32) / w->cols));
    for (size_t t = 0; t < n; t += most) {
        const size_t m = std::min(most, n - t);
        const hipError_t e = launch_rows_few(dev, w, up, out + t * w->rows, x + t * w->cols, m, add);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

void rows_scratch(const dwim_dev *dev, int fmt, size_t rows, size_t cols, size_t most, bool pair, size_t *split,
                  size_t *parts) {
    dwim_weight w{};
    w.fmt = fmt;
    w.rows = rows;
    w.cols = cols;
    for (size_t n = 1; n <= most; n++) {
        if (n > few_tokens(&w, pair)) gemm_rows_scratch(dev, fmt, rows, cols, n, pair, split, parts);
        else *parts = std::max(*parts, rows_few_scratch(dev, fmt, rows, cols, n, pair));
    }
}

hipError_t launch_matvec(dwim_dev *dev, const dwim_weight *wt, float *out, const float *x, size_t n, int add) {
    hipStream_t s = dev->stream;
    switch (wt->fmt) {
    case DWIM_Q4_K: return launch_matvec_q4k(dev, wt, out, x, n, add);
    case DWIM_Q6_K:
        if (n == 1 && !add && wt->cols <= 10240) {  // (a workgroup's 8 waves take 5 blocks each)
            // one token (the output head): the int8 matrix cores over x's planes
            hipError_t e = launch_planes(dev, x, wt->cols, nullptr, 0.0f, nullptr, 0);
            return e != hipSuccess ? e : launch_mv_q6k_mfma(dev, wt, out, 0);
        }
        // a few tokens (a verify batch): the weights read once a run of four
        if (n > 1 && n < 16 && !add && wt->cols % 256 == 0 && wt->cols <= 10240)
            return launch_mv_q6k_tokens(dev, wt, out, x, n);
        return launch_rows(dev, wt, nullptr, out, x, n, add);
    case DWIM_BF16:
        // (1 MB of weights at 96 × 5120, read again from the L2 for every four tokens)
        if (n <= 256 && wt->rows <= kSkRows) {
            k_rows_bf16<<<dim3((unsigned)wt->rows, (unsigned)((n + kRowTok - 1) / kRowTok)), 256, 0, s>>>(
                (const uint16_t *)wt->q, x, out, wt->rows, wt->cols, n, add);
            return hipGetLastError();
        }
        [[fallthrough]];
    default: return launch_rows(dev, wt, nullptr, out, x, n, add);
    }
}

hipError_t launch_swiglu(dwim_dev *dev, const dwim_weight *gate, const dwim_weight *up, float *out, float *scratch,
                         const float *x, size_t n) {
    if (gate->fmt == DWIM_Q4_K && up->fmt == DWIM_Q4_K && gate->cols <= 16 * 5 * 256 / 2)
        return launch_swiglu_q4k(dev, gate, up, out, x, n, nullptr, 0.0f);
    if (gate->fmt == up->fmt && gate->fmt != DWIM_Q4_K) return launch_rows(dev, gate, up, out, x, n, 0);
    hipError_t e = launch_matvec(dev, gate, out, x, n, 0);
    if (e == hipSuccess) e = launch_matvec(dev, up, scratch, x, n, 0);
    if (e == hipSuccess) e = launch_silu_mul(dev->stream, out, scratch, n * gate->rows);
    return e;
}
