// Matrix products by format and batch size: out[t][r] (+)= w[r] · x[t] (dwim
// gpu/cpu.rs:110-149, Device::matmul), and the kernels for a few tokens through
// bf16 matrices on the vector ALUs: of few rows (DeltaNet's gate projection),
// and of any.
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

// Up to four tokens through a bf16 matrix: a group of LPR lanes takes R rows (of
// each matrix of a SwiGLU pair) and walks their columns 8 at a time, every
// activation loaded serving its R rows, every weight its T tokens; the lanes' sums
// meet by lane swaps.  No LDS, no barrier and a wave for every few rows: the
// weights' way from memory bounds it.  The matrix cores' kernel holds 16 rows a wave and a
// workgroup for every 16 or 32 rows, too few in flight for weights of two bytes.
// Measured on MI355X, us, k_rows_few | here, weights from HBM: 5120×5120 1 token
// 16.8 | 10.4 (5.0 TB/s), 2 18.9 | 11.7, 3 23.2 | 14.9, 4 23.3 | 18.7; 5120×17408
// 45.8 | 31.3, 53 | 35, 70 | 51, 70 | 61; 17408×5120 42.6 | 33.4, 45 | 40, 54 | 49, 54 |
// 53; 1000×4096 9.9 | 6.2; 1024×1024 (in the cache) 3.7 | 3.4, 2 4.4 | 3.5; pairs
// 17408×5120 70 | 61, 75 | 66, 83 | 70, 5120×17408 84 | 64, 91 | 73.  At 5
// tokens, read twice here, 1000×4096 would be 8.5 | 9.1, larger ones slower than there.
constexpr int kVecThreads = 256;

template <int R, int T, int LPR, bool PAIR>
__global__ void __launch_bounds__(kVecThreads) k_vec_bf16(const uint16_t *__restrict__ w, const uint16_t *__restrict__ up,
                                                          const float *__restrict__ x, float *out, size_t rows,
                                                          size_t cols, int add) {
    constexpr int M = PAIR ? 2 : 1;
    const size_t row0 = ((size_t)blockIdx.x * kVecThreads + threadIdx.x) / LPR * R;
    const int sl = threadIdx.x & (LPR - 1);
    if (row0 >= rows) return;  // (whole groups: lane swaps stay within one)
    const size_t chunks = cols / 8;
    float acc[M][R][T];
#pragma unroll
    for (int m = 0; m < M; m++)
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
            for (int t = 0; t < T; t++) acc[m][r][t] = 0.0f;
    for (size_t c = sl; c < chunks; c += LPR) {
        // (every load of the step before its sums: left to itself the compiler
        // waits for each before it issues the next)
        uint4 q[M][R];
        float4 xv[T][2];
#pragma unroll
        for (int m = 0; m < M; m++)
#pragma unroll
            for (int r = 0; r < R; r++) {  // (rows past the last: the last, not written)
                const size_t row = row0 + r < rows ? row0 + r : rows - 1;
                q[m][r] = ((const uint4 *)(m ? up : w))[row * chunks + c];
            }
#pragma unroll
        for (int t = 0; t < T; t++)
#pragma unroll
            for (int i = 0; i < 2; i++) xv[t][i] = ((const float4 *)(x + t * cols))[2 * c + i];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int m = 0; m < M; m++)
#pragma unroll
            for (int r = 0; r < R; r++)
#pragma unroll
                for (int t = 0; t < T; t++) {
                    const uint4 v = q[m][r];
                    const float4 a = xv[t][0], b = xv[t][1];
                    auto lo = [](uint32_t u) { return __uint_as_float(u << 16); };
                    auto hi = [](uint32_t u) { return __uint_as_float(u & 0xffff0000u); };
                    float sum = fmaf(hi(v.x), a.y, lo(v.x) * a.x);  // (by itself: see k_rows_few.hip)
                    sum = fmaf(hi(v.y), a.w, fmaf(lo(v.y), a.z, sum));
                    sum = fmaf(hi(v.z), b.y, fmaf(lo(v.z), b.x, sum));
                    acc[m][r][t] += fmaf(hi(v.w), b.w, fmaf(lo(v.w), b.z, sum));
                }
    }
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int t = 0; t < T; t++) {
            const float v = group_sum<LPR>(acc[0][r][t]), u = PAIR ? group_sum<LPR>(acc[M - 1][r][t]) : 0.0f;
            if (sl == 0 && row0 + r < rows) {
                float *o = out + t * rows + row0 + r;
                *o = PAIR ? v * sigmoidf_(v) * u : add ? *o + v : v;
            }
        }
}

template <int R, int T, bool PAIR>
static hipError_t vec_bf16(hipStream_t s, const dwim_weight *w, const dwim_weight *up, float *out, const float *x, int add) {
    // lanes a group: all 64, whose loads are whole lines, unless a fifth of their
    // steps would be past the row's end
    const size_t chunks = w->cols / 8;
    int lpr = 64;
    for (int l = 32; l >= 4; l >>= 1)
        if ((chunks + l - 1) / l * l * 5 < (chunks + lpr - 1) / lpr * lpr * 4) lpr = l;
    const unsigned blocks = (unsigned)(((w->rows + R - 1) / R * lpr + kVecThreads - 1) / kVecThreads);
    const uint16_t *q = (const uint16_t *)w->q, *u = up ? (const uint16_t *)up->q : nullptr;
    switch (lpr) {
    case 64: k_vec_bf16<R, T, 64, PAIR><<<blocks, kVecThreads, 0, s>>>(q, u, x, out, w->rows, w->cols, add); break;
    case 32: k_vec_bf16<R, T, 32, PAIR><<<blocks, kVecThreads, 0, s>>>(q, u, x, out, w->rows, w->cols, add); break;
    case 16: k_vec_bf16<R, T, 16, PAIR><<<blocks, kVecThreads, 0, s>>>(q, u, x, out, w->rows, w->cols, add); break;
    case 8: k_vec_bf16<R, T, 8, PAIR><<<blocks, kVecThreads, 0, s>>>(q, u, x, out, w->rows, w->cols, add); break;
    default: k_vec_bf16<R, T, 4, PAIR><<<blocks, kVecThreads, 0, s>>>(q, u, x, out, w->rows, w->cols, add); break;
    }
    return hipGetLastError();
}

// Tokens that go there.
constexpr size_t kVecTokens = 4;

// Rows a group: where rows are many, more of them share the activations (17408
// rows, one token: 1 row a group 36, 4 33; at 5120 rows 4 took 11.8 for 10.4)
template <int T>
static hipError_t vec_bf16_tokens(hipStream_t s, const dwim_weight *w, const dwim_weight *up, float *out, const float *x,
                                  int add) {
    constexpr int kFew = T == 1 ? 1 : 2, kMany = T == 1 ? 4 : 2;
    const bool many = w->rows >= 16384;
    if (up) return many ? vec_bf16<2, T, true>(s, w, up, out, x, 0) : vec_bf16<1, T, true>(s, w, up, out, x, 0);
    return many ? vec_bf16<kMany, T, false>(s, w, up, out, x, add) : vec_bf16<kFew, T, false>(s, w, up, out, x, add);
}

static hipError_t launch_vec_bf16(hipStream_t s, const dwim_weight *w, const dwim_weight *up, float *out, const float *x,
                                  size_t n, int add) {
    switch (n) {
    case 1: return vec_bf16_tokens<1>(s, w, up, out, x, add);
    case 2: return vec_bf16_tokens<2>(s, w, up, out, x, add);
    case 3: return vec_bf16_tokens<3>(s, w, up, out, x, add);
    default: return vec_bf16_tokens<4>(s, w, up, out, x, add);
    }
}

// Up to four tokens through a small Q4_0 or Q8_0 matrix: a workgroup takes RR rows
// of a tile of 16 (layout.h: chunk m of a row lies 256 bytes after chunk m - 1), a wave
// U × 64 / RR chunks of each at a time, lane (g, c) row c's chunks g, g + 64 / RR, ..;
// the sums meet by lane swaps and once in LDS.  Without the conversion of the activations
// into LDS that k_rows_few starts with, which is most of its time here, and with
// RR = 4 four times its workgroups.
constexpr unsigned vec_loads(int fmt, int rr) { return rr == 16 && fmt == DWIM_Q4_0 ? 1 : 2; }  // U: 8 waves at 1024 columns

template <int FMT, int T, int RR>
__global__ void __launch_bounds__(1024) k_vec_tiles(const uint4 *__restrict__ q, const uint16_t *__restrict__ s,
                                                    const float *__restrict__ x, float *out, unsigned rows, unsigned cols,
                                                    int add) {
    constexpr unsigned G = 64 / RR, U = vec_loads(FMT, RR), kWeights = FMT == DWIM_Q4_0 ? 32 : 16, kPer = 128 / kWeights;
    __shared__ float red[16][T][RR];
    const unsigned lane = threadIdx.x & 63, g = lane / RR, c = lane % RR, wave = threadIdx.x >> 6, KW = blockDim.x >> 6;
    const unsigned units = (cols + 127) / 128, chunks = cols / kWeights;
    const unsigned row0 = blockIdx.x * RR, in_tile = row0 % 16 + c;
    const size_t base = (size_t)(row0 / 16) * units;
    float acc[T];
#pragma unroll
    for (int t = 0; t < T; t++) acc[t] = 0.0f;
    for (unsigned m0 = wave * U * G; m0 < chunks; m0 += KW * U * G) {
        uint4 w[U];
        uint16_t d[U];
#pragma unroll
        for (unsigned i = 0; i < U; i++) {  // (past the row's chunks the last one's, unused)
            const unsigned m = min(m0 + i * G + g, chunks - 1), b = m * kWeights / 32;
            w[i] = q[(base * kPer + m) * 16 + in_tile];
            d[i] = s[((base + b / 4) * 16 + in_tile) * 4 + b % 4];
        }
#pragma unroll
        for (unsigned i = 0; i < U; i++) {
            const unsigned m = m0 + i * G + g;
            if (m >= chunks) continue;
            const uint32_t v[4] = {w[i].x, w[i].y, w[i].z, w[i].w};
            const float scale = dq::from_f16(d[i]);
#pragma unroll
            for (int t = 0; t < T; t++) {
                const float4 *xt = (const float4 *)(x + (size_t)t * cols + m * kWeights);
                float sum = 0.0f;
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const float4 a = xt[k];
                    if constexpr (FMT == DWIM_Q4_0) {
                        const float4 e = xt[4 + k];
                        auto lo = [&](int j) { return (float)((int)(v[k] >> (8 * j) & 15u) - 8); };
                        auto hi = [&](int j) { return (float)((int)(v[k] >> (8 * j + 4) & 15u) - 8); };
                        sum = fmaf(lo(3), a.w, fmaf(lo(2), a.z, fmaf(lo(1), a.y, fmaf(lo(0), a.x, sum))));
                        sum = fmaf(hi(3), e.w, fmaf(hi(2), e.z, fmaf(hi(1), e.y, fmaf(hi(0), e.x, sum))));
                    } else {
                        auto b = [&](int j) { return (float)(int8_t)(v[k] >> (8 * j)); };
                        sum = fmaf(b(3), a.w, fmaf(b(2), a.z, fmaf(b(1), a.y, fmaf(b(0), a.x, sum))));
                    }
                }
                acc[t] = fmaf(scale, sum, acc[t]);
            }
        }
    }
#pragma unroll
    for (int t = 0; t < T; t++) {
        float v = acc[t], a, b;
        if (RR == 4) {  // (rotations of 16 lanes by 4 and 8)
            v += xlane::mov<0x124>(v);
            v += xlane::mov<0x128>(v);
        }
        xlane::swap16(v, a, b);
        xlane::swap32(a + b, a, b);
        if (g == 0) red[wave][t][c] = a + b;
    }
    __syncthreads();
    const unsigned t = threadIdx.x / RR, row = row0 + threadIdx.x % RR;
    if (t >= T || row >= rows) return;
    float v = 0.0f;
    for (unsigned k = 0; k < KW; k++) v += red[k][t][threadIdx.x % RR];
    float *o = out + (size_t)t * rows + row;
    *o = add ? *o + v : v;
}

// What goes there: two to four tokens over rows of few units (RR = 16), one to four
// over few long rows (RR = 4), whose tiles are too few for k_rows_few.  Measured on MI355X, us, k_rows_few | here, Q8_0: 1024×1024 2
// tokens 4.8 | 3.5, 4 5.0 | 3.9; 4096×1024 4 5.5 | 4.0; 8192×1024 2 5.6 | 4.4, 4 5.5 |
// 6.1; 100000×1024 2 (from HBM) 40.3 | 39.3, Q4_0 41.5 | 35.0; 2048×2048 2 5.3 | 4.3, 4
// 5.5 | 6.1; 8192×2048 2 (from HBM) 8.0 | 8.7; 1000×4096 2 6.3 | 6.5; one token 96×5120 5.2 |
// 3.3, 1024×5120 5.3 | 3.0 (from HBM 5.5 | 4.8; 4 tokens 10.2 | 6.4), 1024×17408 12.7 | 8.6,
// 1024×2048 3.4 | 3.2, 2048×5120 from HBM 5.9 | 6.4 (a line is read by two workgroups).
static int vec_tiles(const dwim_weight *w, size_t n) {
    if ((w->fmt != DWIM_Q4_0 && w->fmt != DWIM_Q8_0) || n > 4 || w->rows >= (1u << 31) || w->cols >= (1u << 31)) return 0;
    if (w->rows <= 1024 && w->cols > 2048) return 4;
    if (n == 1) return 0;
    return (w->cols <= 1024 ? n == 2 || w->rows * n <= 16384 : w->cols <= 2048 && n == 2 && w->rows <= 2048) ? 16 : 0;
}

template <int FMT>
static hipError_t launch_vec_tiles(hipStream_t s, const dwim_weight *w, float *out, const float *x, size_t n, int add,
                                   int rr) {
    // (the waves' steps as even as may be, at most 16 waves)
    const size_t step = (size_t)64 / rr * vec_loads(FMT, rr) * (FMT == DWIM_Q4_0 ? 32 : 16);
    const unsigned steps = (unsigned)((w->cols + step - 1) / step), each = (steps + 15) / 16, kw = (steps + each - 1) / each;
    const unsigned blocks = (unsigned)((w->rows + rr - 1) / rr), threads = 64 * kw;
    const unsigned rows = (unsigned)w->rows, cols = (unsigned)w->cols;
    const uint4 *q = (const uint4 *)w->q;
    const uint16_t *sc = (const uint16_t *)w->s;
    switch (n) {
    case 1: k_vec_tiles<FMT, 1, 4><<<blocks, threads, 0, s>>>(q, sc, x, out, rows, cols, add); break;
    case 2:
        if (rr == 4) k_vec_tiles<FMT, 2, 4><<<blocks, threads, 0, s>>>(q, sc, x, out, rows, cols, add);
        else k_vec_tiles<FMT, 2, 16><<<blocks, threads, 0, s>>>(q, sc, x, out, rows, cols, add);
        break;
    case 3:
        if (rr == 4) k_vec_tiles<FMT, 3, 4><<<blocks, threads, 0, s>>>(q, sc, x, out, rows, cols, add);
        else k_vec_tiles<FMT, 3, 16><<<blocks, threads, 0, s>>>(q, sc, x, out, rows, cols, add);
        break;
    default:
        if (rr == 4) k_vec_tiles<FMT, 4, 4><<<blocks, threads, 0, s>>>(q, sc, x, out, rows, cols, add);
        else k_vec_tiles<FMT, 4, 16><<<blocks, threads, 0, s>>>(q, sc, x, out, rows, cols, add);
        break;
    }
    return hipGetLastError();
}

// The most tokens that go through the kernel that converts the activations
// itself (k_rows_few.hip); more go through the GEMM (k_gemm_rows.hip), whose
// split of the activations and sum of the parts are launches of their own.
// Measured on MI355X (us, few | GEMM): a 17408×5120 Q4_0 pair at 16 tokens 43 |
// 44, at 32 66 | 48; Q8_0 at 16 53 | 53, at 32 79 | 57; Q6_K at 16 56 | 72, at 32 93
// | 76; bf16 at 32 113 | 121, at 64 254 | 139; a 2304×3072 Q8_0 pair at 32 17.5 | 17.8,
// at 64 32 | 24; 5120×17408 Q4_0 at 16 32 | 47, at 32 44 | 48, at 64 75 | 68; Q6_K,
// whose GEMM scales every 16 columns, at 64 92 | 117, 5120×5120 35 | 45, but with rows
// for whole rounds of tiles 17408×5120 86 | 59, 20000×2048 44 | 39, 100000×1024 117 | 60;
// bf16 at 32 5120×5120 31 | 34, 17408×5120 70 | 62; 1024×1024 Q4_0 at 64 12 | 15.
static size_t few_tokens(const dwim_weight *w, bool pair) {
    const bool small = w->rows * w->cols <= (size_t)8 << 20;
    const bool many = w->rows > 8192;
    if (!pair && (small || w->fmt == DWIM_Q6_K)) return !small && many ? 32 : 64;
    if (!pair && many && w->fmt == DWIM_BF16) return 16;
    return small || w->fmt == DWIM_BF16 || w->cols >= 2 * w->rows ? 32 : 16;
}

hipError_t launch_rows(dwim_dev *dev, const dwim_weight *w, const dwim_weight *up, float *out, const float *x, size_t n,
                       int add, bool *split) {
    if (up && (up->fmt != w->fmt || up->rows != w->rows || up->cols != w->cols)) return hipErrorInvalidValue;
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
        float *const o = out + t * w->rows;
        const float *const xt = x + t * w->cols;
        if (const int rr = up ? 0 : vec_tiles(w, m)) {
            const hipError_t e = w->fmt == DWIM_Q4_0 ? launch_vec_tiles<DWIM_Q4_0>(dev->stream, w, o, xt, m, add, rr)
                                                     : launch_vec_tiles<DWIM_Q8_0>(dev->stream, w, o, xt, m, add, rr);
            if (e != hipSuccess) return e;
            continue;
        }
        const hipError_t e = w->fmt == DWIM_BF16 && m <= kVecTokens ? launch_vec_bf16(dev->stream, w, up, o, xt, m, add)
                                                                     : launch_rows_few(dev, w, up, o, xt, m, add);
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
