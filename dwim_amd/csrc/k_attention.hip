// Causal grouped-query attention over the key/value caches (dwim
// gpu/cpu.rs:202-236), split over chunks of 64 positions so that a single
// decode token still spreads its cache reads over the whole GPU.  A cache is
// the reference's Q8 (int8 with an f16 scale per block of 32) or f16 (each
// kernel a template on the format, F16; an f16 key or value is read as is).
//
// Pass 1, one block per (chunk, key/value head, token; or group of up to 4
// tokens of a small batch, such as a speculative verify step): the G query
// heads sharing the key/value head score the chunk's positions (a Q8 block of
// 32 per lane, its f16 scale applied to the block's sum, the 8 lanes of a
// position summed by shuffles), take the chunk's softmax numerator and weight
// the chunk's values, for each of the block's tokens in turn over the keys
// and values read once.  Every cache load of the block is issued before any
// arithmetic.  It writes, per token and query head, the chunk's max, sum of
// exponentials and weighted values.  Pass 2, one block per (query head,
// token), merges the chunks.  Each cache byte is read once per token (once
// per 4 tokens of a small batch).
//
// A batch of 16 tokens or more (head_dim 256) runs flash attention on the
// f16 matrix cores over a copy of the cache expanded to f16 hi + lo parts in
// the layout the kernel holds in LDS (k_kv_expand, k_attn_flash below), but for
// short ones (short_batch_tokens), which take the decode pass of k_attn_mfma.
#include "device_util.h"
#include "planes.h"
#include "quant_math.h"
#include "runtime.h"

namespace {

constexpr int kMaxG = 8;
constexpr int kMaxD = 256;
constexpr int kPos = 64;        // positions a partial block scores
constexpr int kPThreads = 512;  // 8 lanes a position
constexpr int kQPer = kMaxG * kMaxD / kPThreads;
constexpr int kTok = 4;         // tokens a block of a several-token batch

typedef _Float16 ahalf8 __attribute__((ext_vector_type(8)));
typedef float afloat4 __attribute__((ext_vector_type(4)));

constexpr int kFD = 256, kFQ = 128, kFThreads = 256;
constexpr size_t kMPerCU = 2;  // blocks of k_attn_mfma resident at once on a CU (its launch bounds)
constexpr size_t kFlashItems = 2;  // blocks a CU when a batch's positions are split


struct Shape {
    size_t n, pos, n_heads, head_dim, n_kv_heads, ch, chunks;
};

// partials: [token][head][chunk][head_dim + 2]  (o[...], max, sum)
//
// One pass over the chunk's kPos positions, every load issued up front.
// Scores: 8 lanes per position, lane b takes Q8 block b (32 elements) of the
// head for all G query heads.  Values: wave w takes elements 32w..32w+31 (one
// Q8 block: one scale per position), lane l elements 32w + 4(l % 8)..+3 of
// positions l/8 + 8i; the 8 position groups meet by shuffles.
DEV float half_of(uint32_t word, int hi) {
    return (float)__builtin_bit_cast(_Float16, (uint16_t)(hi ? word >> 16 : word & 0xffffu));
}
DEV uint32_t word_of(const uint4 &v, int i) { return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w; }

template <int G, bool F16, int T>
__global__ void __launch_bounds__(kPThreads) k_attn_partial(float *__restrict__ partials, const float *__restrict__ q,
                                                            const int8_t *__restrict__ kq,
                                                            const uint16_t *__restrict__ ks,
                                                            const int8_t *__restrict__ vq,
                                                            const uint16_t *__restrict__ vs, Shape sh) {
    // queries, each Q8 block of 32 padded to 36 floats: the 8 lanes of a
    // position, reading blocks 0..7 at once, then hit 8 different banks
    __shared__ float q_s[T * G * kMaxD / 32 * 36];
    __shared__ float p_s[T * G * kPos];
    __shared__ float stat_s[T * G * 2];
    const size_t chunk = blockIdx.x, kvh = blockIdx.y, t0 = blockIdx.z * (size_t)T;
    const int nt = (int)min((size_t)T, sh.n - t0);  // the block's tokens: t0 .. t0 + nt - 1
    const int D = (int)sh.head_dim;
    const size_t kv_dim = sh.n_kv_heads * sh.head_dim;
    const size_t p0 = chunk * kPos;
    const size_t head0 = kvh * G;
    const size_t part_stride = sh.chunks * (size_t)(D + 2);  // next head
    // token t0 + tt attends up to its own position: cnt_of(tt) of the
    // chunk's positions (0 past its last)
    auto cnt_of = [&](int tt) -> int {
        const size_t len = sh.pos + t0 + tt + 1;
        return p0 >= len ? 0 : (int)min((size_t)kPos, len - p0);
    };
    auto part_of = [&](int tt) -> float * {
        return partials + (((t0 + tt) * sh.n_heads + head0) * sh.chunks + chunk) * (size_t)(D + 2);
    };
    const int cnt = cnt_of(nt - 1);  // the last token's: the most
    if (cnt == 0) {
        // a chunk past every token's last position: empty
        if (threadIdx.x < (unsigned)(nt * G)) {
            float *part = part_of((int)threadIdx.x / G) + (threadIdx.x % G) * part_stride;
            part[D] = -INFINITY;
            part[D + 1] = 0.0f;
        }
        return;
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    // the queries first: in-order completion then lets the scores wait for
    // the queries and keys alone, and the values arrive meanwhile
    float qr[T][kQPer];
#pragma unroll
    for (int tt = 0; tt < T; tt++)
#pragma unroll
        for (int k = 0; k < kQPer; k++) {
            const size_t i = threadIdx.x + k * kPThreads;
            qr[tt][k] = tt < nt && i < (size_t)(G * D) ? q[((t0 + tt) * sh.n_heads + head0) * D + i] : 0.0f;
        }
    // key and value loads, unconditional (positions past the chunk's end read
    // its last position, masked later) and unconverted, so that every load is
    // in flight before the first wait
    const int kp = threadIdx.x >> 3, b = threadIdx.x & 7, nblk = D / 32;
    const bool klive = kp < cnt && b < nblk;
    uint4 kr[F16 ? 4 : 2];
    uint16_t kbits = 0;
    {
        const size_t off = (p0 + min(kp, cnt - 1)) * kv_dim + kvh * D + 32 * min(b, nblk - 1);
        if constexpr (F16) {
            const uint4 *src = (const uint4 *)((const uint16_t *)kq + off);
#pragma unroll
            for (int i = 0; i < 4; i++) kr[i] = src[i];
        } else {
            kr[0] = ((const uint4 *)(kq + off))[0];
            kr[1] = ((const uint4 *)(kq + off))[1];
            kbits = ks[off / 32];
        }
    }
    // values: wave w < nblk takes block w of the head (4 values a lane)
    const bool vlive = wave < nblk;
    uint32_t vw[kPos / 8][F16 ? 2 : 1];
    uint16_t vbits[kPos / 8];
#pragma unroll
    for (int i = 0; i < kPos / 8; i++) {
        const int vp = min((lane >> 3) + 8 * i, cnt - 1);
        const size_t off = (p0 + vp) * kv_dim + kvh * D + 32 * min(wave, nblk - 1) + 4 * (lane & 7);
        if constexpr (F16) {
            const uint2 x = *(const uint2 *)((const uint16_t *)vq + off);
            vw[i][0] = x.x;
            vw[i][F16 ? 1 : 0] = x.y;
            vbits[i] = 0;
        } else {
            vw[i][0] = *(const uint32_t *)(vq + off);
            vbits[i] = vs[off / 32];
        }
    }
    // (the query loads were issued first, so this waits for them alone)
#pragma unroll
    for (int tt = 0; tt < T; tt++)
        for (int k = 0; k < kQPer; k++) {
            const unsigned i = threadIdx.x + k * kPThreads;
            if (i < (unsigned)(G * D)) q_s[(tt * G * nblk + i / 32) * 36 + i % 32] = qr[tt][k];
        }
    __syncthreads();

    const float scale = 1.0f / sqrtf((float)D);
    {
        const float ksc = F16 ? 1.0f : dq::from_f16(kbits);
        float kv[32];
#pragma unroll
        for (int i = 0; i < 32; i++) {
            if constexpr (F16) {
                kv[i] = half_of(word_of(kr[i / 8], (i % 8) / 2), i % 2);
            } else {
                const uint32_t w = word_of(kr[i / 16], (i % 16) / 4);
                kv[i] = (float)(int8_t)((w >> (8 * (i & 3))) & 0xff);
            }
        }
        // every token's G heads against the keys read once
#pragma unroll
        for (int r = 0; r < T * G; r++) {
            if (T > 1 && r >= nt * G) continue;  // (uniform)
            float sc = 0.0f;
            if (klive) {
                const float *qg = q_s + (r * nblk + b) * 36;
#pragma unroll
                for (int i = 0; i < 32; i++) sc += qg[i] * kv[i];
            }
            sc = group_sum<8>(sc * ksc);
            if (b == 0 && kp < cnt) p_s[r * kPos + kp] = scale * sc;
        }
    }
    __syncthreads();
    // softmax numerators: wave w takes rows (token, head) w, w + 8, ..., a
    // lane per position
    for (int r = wave; r < nt * G; r += kPThreads / 64) {
        const int c = cnt_of(r / G);
        const float sc = lane < c ? p_s[r * kPos + lane] : -INFINITY;
        const float m = group_max<64>(sc);
        const float e = lane < c ? expf(sc - m) : 0.0f;
        const float l = group_sum<64>(e);
        if (lane < cnt) p_s[r * kPos + lane] = e;  // (0 past the token's last position)
        if (lane == 0) {
            stat_s[2 * r] = c ? m : -INFINITY;
            stat_s[2 * r + 1] = l;
        }
    }
    __syncthreads();
    if (vlive) {
        float vv[kPos / 8][4];
#pragma unroll
        for (int i = 0; i < kPos / 8; i++) {
            if constexpr (F16) {
                vv[i][0] = half_of(vw[i][0], 0);
                vv[i][1] = half_of(vw[i][0], 1);
                vv[i][2] = half_of(vw[i][F16 ? 1 : 0], 0);
                vv[i][3] = half_of(vw[i][F16 ? 1 : 0], 1);
            } else {
                const uint32_t w = vw[i][0];
                const float vsc = dq::from_f16(vbits[i]);
                vv[i][0] = (float)(int8_t)(w & 0xff) * vsc;
                vv[i][1] = (float)(int8_t)((w >> 8) & 0xff) * vsc;
                vv[i][2] = (float)(int8_t)((w >> 16) & 0xff) * vsc;
                vv[i][3] = (float)(int8_t)(w >> 24) * vsc;
            }
        }
        for (int tt = 0; tt < nt; tt++) {
            float acc[G][4];
#pragma unroll
            for (int g = 0; g < G; g++)
#pragma unroll
                for (int e = 0; e < 4; e++) acc[g][e] = 0.0f;
#pragma unroll
            for (int i = 0; i < kPos / 8; i++) {
                const int vp = (lane >> 3) + 8 * i;
#pragma unroll
                for (int g = 0; g < G; g++) {
                    const float pr = vp < cnt ? p_s[(tt * G + g) * kPos + vp] : 0.0f;
                    acc[g][0] += pr * vv[i][0];
                    acc[g][1] += pr * vv[i][1];
                    acc[g][2] += pr * vv[i][2];
                    acc[g][3] += pr * vv[i][3];
                }
            }
            // the 8 position groups (lanes 8 apart) meet: lanes l, l ^ 8 by a
            // row rotation, l ^ 16 and l ^ 32 by permlane swaps
#pragma unroll
            for (int g = 0; g < G; g++)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    float v = acc[g][e];
                    v += xlane::mov<0x128>(v);
                    float x, y;
                    xlane::swap16(v, x, y);
                    v = x + y;
                    xlane::swap32(v, x, y);
                    acc[g][e] = x + y;
                }
            // position group pg stores head pg's four values (a partial row
            // is (D + 2) floats: 8-byte alignment only)
            const int pg = lane >> 3;
            float o[4] = {acc[0][0], acc[0][1], acc[0][2], acc[0][3]};
#pragma unroll
            for (int g = 1; g < G; g++)
#pragma unroll
                for (int e = 0; e < 4; e++) o[e] = pg == g ? acc[g][e] : o[e];
            if (pg < G) {
                float2 *dst = (float2 *)(part_of(tt) + pg * part_stride + 32 * wave + 4 * (lane & 7));
                dst[0] = make_float2(o[0], o[1]);
                dst[1] = make_float2(o[2], o[3]);
            }
        }
    }
    if (threadIdx.x < (unsigned)(nt * G)) {
        float *part = part_of((int)threadIdx.x / G) + (threadIdx.x % G) * part_stride;
        part[D] = stat_s[2 * threadIdx.x];
        part[D + 1] = stat_s[2 * threadIdx.x + 1];
    }
}

// ---------------------------------------------------------------- decode, matrix cores
//
// The same partial rows for head_dim 256 with the scores and the weighted
// values on the f16 matrix cores (v_mfma_f32_16x16x32_f16).  A block of 4
// waves takes a run of sh.ch positions (64 a step) of one key/value head and
// its query rows, a row a (token, head) pair: the G heads of one token, or
// of up to kTok tokens of a small batch, in RT tiles of 16 rows.  (The queries
// are staged times qscale, a power of two.)
//   * Scores, wave w the step's positions 16w..16w+15: for each Q8 block of
//     32 dimensions, the queries' f16 hi and lo parts (staged in LDS once) as
//     A against the keys as B, exact in f16 (int8, or the f16 cache as is),
//     then times the block's per-position scale, in f32.
//   * Softmax over the step, a running max and sum per row (flash style).
//   * Values, wave w the dimensions 64w..64w+63: the probabilities times the
//     values' per-position scale of the dimension's Q8 block, split into f16
//     hi and lo parts, as A against the values as B (transposed into LDS,
//     8 positions of one dimension a lane).
// Every product is exact up to the hi/lo split (2^-22 relative) and summed
// in f32.  WIDE (batches, over Q8 caches): the values' scales of a step and Q8 block are
// taken times a power of two that brings the largest to [2^14, 2^15), so that
// no probability times a scale is small in f16 (small ones cost 6e-6 of the
// result; k_attn_flash 4e-7), and a step's products are summed by themselves.
constexpr int kMStep = 64;       // positions a step
constexpr int kMThreads = 256;
constexpr int kQStride = 256 + 8;  // halfs a staged query row (bank spread)
constexpr int kPStride = kMStep + 4;
constexpr int kVRow = kFD + 16;           // Q8: bytes of a value row as the cache holds it (bank spread)
constexpr int kVRow16 = 2 * kFD + 32;     // f16: bytes of such a row

// Eight int8 values (two little-endian words) as f16, exactly: each byte
// biased to u = b + 128 and placed under the f16 exponent of 1024
// (0x64uu = 1024 + u), then 1152 subtracted, two values a packed op.
DEV ahalf8 i8x8_to_f16(uint32_t w0, uint32_t w1) {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    const h2 bias = h2{(_Float16)1152.0f, (_Float16)1152.0f};
    const uint32_t x0 = w0 ^ 0x80808080u, x1 = w1 ^ 0x80808080u;
    const h2 a = __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, x0, 0x04010400u)) - bias;
    const h2 b = __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, x0, 0x04030402u)) - bias;
    const h2 c = __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, x1, 0x04010400u)) - bias;
    const h2 d = __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, x1, 0x04030402u)) - bias;
    return ahalf8{a[0], a[1], b[0], b[1], c[0], c[1], d[0], d[1]};
}

// LDS of k_attn_mfma: queries hi and lo, probabilities, value scales, the
// rows' max / sum / rescale, the transposed values
constexpr size_t mfma_lds(int rt, bool f16) {
    return (size_t)16 * rt * kQStride * 2 * 2 + (size_t)16 * rt * kPStride * 4 + (size_t)(kFD / 32) * kMStep * 4 +
           (size_t)16 * rt * 3 * 4 + (size_t)kMStep * (f16 ? kVRow16 : kVRow);
}

template <int RT, bool F16, bool WIDE>
__global__ void __launch_bounds__(kMThreads, 2) k_attn_mfma(float *__restrict__ partials, const float *__restrict__ q,
                                                         const int8_t *__restrict__ kq,
                                                         const uint16_t *__restrict__ ks,
                                                         const int8_t *__restrict__ vq,
                                                         const uint16_t *__restrict__ vs, Shape sh, int G, int T,
                                                         float qscale) {
    constexpr int NR = 16 * RT;  // rows, padded
    constexpr int D = kFD;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds_raw[];
    __shared__ float unscale[WIDE ? 8 : 1];  // of a step's scales, by Q8 block
    _Float16 *q_hi = (_Float16 *)lds_raw, *q_lo = q_hi + NR * kQStride;
    float *p_s = (float *)(q_lo + NR * kQStride);
    float(*vsc_s)[kMStep] = (float(*)[kMStep])(p_s + NR * kPStride);
    float *m_s = (float *)(vsc_s + D / 32), *l_s = m_s + NR, *a_s = l_s + NR;
    uint8_t *vt_raw = (uint8_t *)(a_s + NR);
    const size_t chunk = blockIdx.x, kvh = blockIdx.y, t0 = blockIdx.z * (size_t)T;
    const int nt = (int)min((size_t)T, sh.n - t0), R = nt * G;
    const size_t kv_dim = sh.n_kv_heads * D, head0 = kvh * G;
    const size_t c0 = chunk * sh.ch;
    const size_t len_last = sh.pos + t0 + nt;  // positions the group's last token sees
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r16 = lane & 15, kq4 = lane >> 4;
    auto part_of = [&](int r) -> float * {
        return partials + (((t0 + r / G) * sh.n_heads + head0 + r % G) * sh.chunks + chunk) * (size_t)(D + 2);
    };
    if (c0 >= len_last) {
        if (threadIdx.x < (unsigned)R) {
            float *part = part_of((int)threadIdx.x);
            part[D] = -INFINITY;
            part[D + 1] = 0.0f;
        }
        return;
    }
    // the queries, hi and lo parts (rows past R zero)
    for (int r = wave; r < NR; r += kMThreads / 64) {
        float4 x = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (r < R) x = *(const float4 *)(q + ((t0 + r / G) * sh.n_heads + head0 + r % G) * D + 4 * lane);
        const float xs[4] = {x.x * qscale, x.y * qscale, x.z * qscale, x.w * qscale};
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const _Float16 h = (_Float16)xs[e];
            q_hi[r * kQStride + 4 * lane + e] = h;
            q_lo[r * kQStride + 4 * lane + e] = (_Float16)(xs[e] - (float)h);
        }
    }
    if (threadIdx.x < (unsigned)NR) {
        m_s[threadIdx.x] = -INFINITY;
        l_s[threadIdx.x] = 0.0f;
    }
    afloat4 o[RT][4];
#pragma unroll
    for (int rt = 0; rt < RT; rt++)
#pragma unroll
        for (int j = 0; j < 4; j++) o[rt][j] = afloat4{0.0f, 0.0f, 0.0f, 0.0f};
    const float scale = 0.0625f / qscale;  // 1 / sqrt(256), powers of two
    const int steps = (int)(sh.ch / kMStep);
    // ---- loads: this wave's keys (position 16w + r16, 8 dimensions of each
    // Q8 block) and their scales; a 4-dimension x 16-position patch of the
    // values and (wave 0) the value scales.  A step's loads are issued while
    // the previous step computes: the values' once they are in LDS, the
    // keys' once the scores are taken.
    // the value patch: Q8, dimensions 16·(t % 16).. of positions 4·(t / 16)..;
    // f16, dimensions 8·(t % 32).. of positions 8·(t / 32)..
    constexpr int VP = F16 ? 8 : 4;                                   // positions a thread
    const int vd = F16 ? 8 * (threadIdx.x & 31) : 16 * (threadIdx.x & 15);
    const int vp0 = F16 ? 8 * (threadIdx.x >> 5) : 4 * (threadIdx.x >> 4);
    uint4 kf[F16 ? 8 : 4];  // Q8: two blocks a uint4
    uint4 kscale = make_uint4(0, 0, 0, 0);
    uint4 vw[VP];
    uint4 vscale = make_uint4(0, 0, 0, 0);
    auto load_keys = [&](size_t ps, int cnt) __attribute__((always_inline)) {
        const size_t kpos = ps + min(16 * wave + r16, cnt - 1);
        const size_t kbase = kpos * kv_dim + kvh * D + 8 * kq4;
        if constexpr (F16) {
#pragma unroll
            for (int b = 0; b < 8; b++) kf[b] = *(const uint4 *)((const uint16_t *)kq + kbase + 32 * b);
        } else {
#pragma unroll
            for (int b = 0; b < 8; b += 2) {
                const uint2 x = *(const uint2 *)(kq + kbase + 32 * b), y = *(const uint2 *)(kq + kbase + 32 * (b + 1));
                kf[b / 2] = make_uint4(x.x, x.y, y.x, y.y);
            }
            kscale = *(const uint4 *)(ks + kpos * (kv_dim / 32) + kvh * 8);
        }
    };
    auto load_values = [&](size_t ps, int cnt) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < VP; j++) {
            const size_t off = (ps + min(vp0 + j, cnt - 1)) * kv_dim + kvh * D + vd;
            vw[j] = F16 ? *(const uint4 *)((const uint16_t *)vq + off) : *(const uint4 *)(vq + off);
        }
        if (!F16 && threadIdx.x < kMStep)
            vscale = *(const uint4 *)(vs + (ps + min((int)threadIdx.x, cnt - 1)) * (kv_dim / 32) + kvh * 8);
    };
    auto count = [&](size_t ps) { return (int)min((size_t)kMStep, len_last - ps); };
    load_keys(c0, count(c0));
    load_values(c0, count(c0));
    for (int s = 0; s < steps; s++) {
        const size_t ps = c0 + (size_t)s * kMStep;
        if (ps >= len_last) break;
        const size_t pn = ps + kMStep;  // the next step
        const bool next = s + 1 < steps && pn < len_last;
        __syncthreads();  // (the previous step is done with vt, p_s and vsc_s; the queries are staged)
        // ---- the values, in LDS as the cache holds them (read transposed below)
        if constexpr (F16) {
            typedef unsigned u4n __attribute__((ext_vector_type(4)));
#pragma unroll
            for (int j = 0; j < VP; j++)
                *(u4n *)(vt_raw + (vp0 + j) * kVRow16 + 2 * vd) = u4n{vw[j].x, vw[j].y, vw[j].z, vw[j].w};
        } else {
            // Q8: the rows as the cache holds them (read transposed below)
            // (as a native vector: a uint4 struct copy would keep vw in memory)
            typedef unsigned u4n __attribute__((ext_vector_type(4)));
#pragma unroll
            for (int j = 0; j < VP; j++)
                *(u4n *)(vt_raw + (vp0 + j) * kVRow + vd) = u4n{vw[j].x, vw[j].y, vw[j].z, vw[j].w};
            if (threadIdx.x < kMStep) {
                const uint32_t w4[4] = {vscale.x, vscale.y, vscale.z, vscale.w};
#pragma unroll
                for (int b = 0; b < 8; b++) {
                    const float d = dq::from_f16((uint16_t)(w4[b / 2] >> (16 * (b % 2))));
                    float up = 1.0f;
                    if constexpr (WIDE) {  // (wave 0)
                        const float top = group_max<64>(fabsf(d));
                        const int sh2 = top > 0.0f ? 141 - (int)(__float_as_uint(top) >> 23) : 0;
                        up = __uint_as_float((unsigned)(sh2 + 127) << 23);
                        if (lane == 0) unscale[b] = __uint_as_float((unsigned)(127 - sh2) << 23);
                    }
                    vsc_s[b][threadIdx.x] = d * up;
                }
            }
        }
        if (next) load_values(pn, count(pn));
        // ---- scores: rows 4·kq4 + e of each tile, position 16w + r16
        {
            afloat4 sc[RT];
#pragma unroll
            for (int rt = 0; rt < RT; rt++) sc[rt] = afloat4{0.0f, 0.0f, 0.0f, 0.0f};
            const uint32_t ksw[4] = {kscale.x, kscale.y, kscale.z, kscale.w};
#pragma unroll
            for (int b = 0; b < 8; b++) {
                ahalf8 kb;
                if constexpr (F16) {
                    kb = __builtin_bit_cast(ahalf8, kf[b]);
                } else {
                    const uint4 &x = kf[b / 2];
                    kb = (b % 2) ? i8x8_to_f16(x.z, x.w) : i8x8_to_f16(x.x, x.y);
                }
                const float kscl = F16 ? 1.0f : dq::from_f16((uint16_t)(ksw[b / 2] >> (16 * (b % 2))));
#pragma unroll
                for (int rt = 0; rt < RT; rt++) {
                    const int qo = (rt * 16 + r16) * kQStride + 32 * b + 8 * kq4;
                    const ahalf8 ah = *(const ahalf8 *)(q_hi + qo), al = *(const ahalf8 *)(q_lo + qo);
                    afloat4 c = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah, kb, afloat4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
                    c = __builtin_amdgcn_mfma_f32_16x16x32_f16(al, kb, c, 0, 0, 0);
#pragma unroll
                    for (int e = 0; e < 4; e++) sc[rt][e] += c[e] * kscl;
                }
                // (a block at a time: the scheduler would otherwise hoist every
                // block's query reads, and their registers cost a block a CU)
                __builtin_amdgcn_sched_barrier(0);
            }
            const int p = 16 * wave + r16;
#pragma unroll
            for (int rt = 0; rt < RT; rt++)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const int r = rt * 16 + 4 * kq4 + e;
                    // row r's token sees positions up to sh.pos + t0 + r / G
                    const bool live = r < R && ps + p <= sh.pos + t0 + r / G;
                    p_s[r * kPStride + p] = live ? sc[rt][e] * scale : -INFINITY;
                }
        }
        if (next) load_keys(pn, count(pn));
        __syncthreads();
        // ---- softmax numerators with a running max and sum: wave w takes
        // rows w, w + 4, ..., a lane per position (the padding rows past R
        // are never written out, and their products stay in their own rows)
        for (int r = wave; r < R; r += kMThreads / 64) {
            const float x = p_s[r * kPStride + lane];
            const float mo = m_s[r];
            const float mn = fmaxf(mo, group_max<64>(x));
            const float e = mn == -INFINITY ? 0.0f : expf(x - mn);
            const float l = group_sum<64>(e);
            p_s[r * kPStride + lane] = e;
            if (lane == 0) {
                const float a = mn == -INFINITY ? 1.0f : expf(mo - mn);
                a_s[r] = a;
                m_s[r] = mn;
                l_s[r] = l_s[r] * a + l;
            }
        }
        __syncthreads();
        // ---- values: dimensions 64w + 16j + r16 (j < 4: Q8 blocks 2w, 2w + 1)
#pragma unroll
        for (int rt = 0; rt < RT; rt++) {
            float a[4];
#pragma unroll
            for (int e = 0; e < 4; e++) a[e] = a_s[rt * 16 + 4 * kq4 + e];
#pragma unroll
            for (int j = 0; j < 4; j++)
#pragma unroll
                for (int e = 0; e < 4; e++) o[rt][j][e] *= a[e];
        }
        afloat4 part[WIDE ? RT : 1][WIDE ? 4 : 1];  // this step's
        if constexpr (WIDE)
#pragma unroll
            for (int rt = 0; rt < RT; rt++)
#pragma unroll
                for (int j = 0; j < 4; j++) part[rt][j] = afloat4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int k2 = 0; k2 < 2; k2++) {
            const int pp = 32 * k2 + 8 * kq4;  // this lane's 8 positions
            ahalf8 vb[4];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                if constexpr (F16) {
                    // ds_read_b64_tr_b16, twice (positions pp.., pp + 4..):
                    // lane 16g + m + 4b names the row of position b at
                    // dimensions d0 + 4m..+3; lane 16g + 4m + i receives
                    // element i of its m's 4 rows, i.e. dimension d0 + r16
                    const int tb = (lane & 15) >> 2, tm = lane & 3;
                    typedef short v4s_ __attribute__((ext_vector_type(4)));
                    const uint8_t *row = vt_raw + 2 * (64 * wave + 16 * j + 4 * tm);
                    const v4s_ x0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                        (__attribute__((address_space(3))) v4s_ *)(row + (pp + tb) * kVRow16));
                    const v4s_ x1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                        (__attribute__((address_space(3))) v4s_ *)(row + (pp + 4 + tb) * kVRow16));
                    // (whole words: assembled element by element, the
                    // compiler took x0[2..3] for copies of x0[0..1])
                    typedef unsigned u2n_ __attribute__((ext_vector_type(2)));
                    typedef unsigned u4n_ __attribute__((ext_vector_type(4)));
                    const u2n_ a0 = __builtin_bit_cast(u2n_, x0), a1 = __builtin_bit_cast(u2n_, x1);
                    vb[j] = __builtin_bit_cast(ahalf8, u4n_{a0.x, a0.y, a1.x, a1.y});
                } else {
                    // ds_read_b64_tr_b8: lane 16g + 2b + h names the row of
                    // position pp_g + b at dimensions d0 + 8h..+7; lane 16g +
                    // 8h + i receives byte i of the 8 rows of its h, i.e.
                    // dimension d0 + r16 of positions pp_g..pp_g + 7
                    const int tb = (lane & 15) >> 1, th = lane & 1;
                    typedef int v2i_ __attribute__((ext_vector_type(2)));
                    const v2i_ x = __builtin_amdgcn_ds_read_tr8_b64_v2i32(
                        (__attribute__((address_space(3))) v2i_ *)(vt_raw + (pp + tb) * kVRow + 64 * wave + 16 * j +
                                                                     8 * th));
                    vb[j] = i8x8_to_f16((uint32_t)x[0], (uint32_t)x[1]);
                }
            }
#pragma unroll
            for (int rt = 0; rt < RT; rt++) {
                const float4 pa = *(const float4 *)(p_s + (rt * 16 + r16) * kPStride + pp);
                const float4 pb = *(const float4 *)(p_s + (rt * 16 + r16) * kPStride + pp + 4);
                const float pr[8] = {pa.x, pa.y, pa.z, pa.w, pb.x, pb.y, pb.z, pb.w};
#pragma unroll
                for (int h = 0; h < 2; h++) {  // Q8 block 2w + h: tiles j = 2h, 2h + 1
                    ahalf8 ph, pl;
#pragma unroll
                    for (int i = 0; i < 8; i++) {
                        float x = F16 ? pr[i] : pr[i] * vsc_s[2 * wave + h][pp + i];
                        // (one product: left to itself the compiler rounds hi from
                        // it, and lo from the exact product less another hi, which
                        // differ now and then: 5e-6 of the results, and 1% of the
                        // time of a token at 32k positions)
                        if (WIDE) asm volatile("" : "+v"(x));
                        const _Float16 hh = (_Float16)x;
                        ph[i] = hh;
                        pl[i] = (_Float16)(x - (float)hh);
                    }
#pragma unroll
                    for (int jj = 0; jj < 2; jj++) {
                        const int j = 2 * h + jj;
                        afloat4 &to = WIDE ? part[WIDE ? rt : 0][WIDE ? j : 0] : o[rt][j];
                        to = __builtin_amdgcn_mfma_f32_16x16x32_f16(ph, vb[j], to, 0, 0, 0);
                        to = __builtin_amdgcn_mfma_f32_16x16x32_f16(pl, vb[j], to, 0, 0, 0);
                    }
                }
            }
        }
        if constexpr (WIDE)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const float down = unscale[2 * wave + j / 2];
#pragma unroll
                for (int rt = 0; rt < RT; rt++)
#pragma unroll
                    for (int e = 0; e < 4; e++) o[rt][j][e] = fmaf(part[rt][j][e], down, o[rt][j][e]);
            }
    }
    // ---- the partial rows: row 4·kq4 + e of tile rt, dimension 64w + 16j + r16
#pragma unroll
    for (int rt = 0; rt < RT; rt++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int r = rt * 16 + 4 * kq4 + e;
            if (r >= R) continue;
            float *part = part_of(r);
#pragma unroll
            for (int j = 0; j < 4; j++) part[64 * wave + 16 * j + r16] = o[rt][j][e];
        }
    if (threadIdx.x < (unsigned)R) {
        float *part = part_of((int)threadIdx.x);
        part[D] = m_s[threadIdx.x];
        part[D + 1] = l_s[threadIdx.x];
    }
}

// out[t][h] = Σ_c e^(m_c − M) o_c / Σ_c e^(m_c − M) l_c, times sigmoid(gate)
// when a gate is given (gpu/cpu.rs:244-248); with one token, its planes too.
// A head's elements split over DS = head_dim / 64 blocks (blockIdx.x = head ·
// DS + slice; one block for a head_dim not a multiple of 64) of 16 threads a
// chunk row, four elements a thread, and 16 groups of them (more for a
// smaller row): group cg takes every 16th chunk, all its loads issued at
// once (up to kU chunks, so that a 4k context needs one round trip), merging
// them as it goes (the batch's max first, then one rescale); the groups meet
// in LDS.
constexpr int kCThreads = 256;
constexpr int kU = 8;

DEV int combine_slices(int D) { return D % 64 == 0 ? D / 64 : 1; }

__global__ void __launch_bounds__(kCThreads) k_attn_combine(float *__restrict__ out, const float *__restrict__ partials,
                                                            Shape sh, const float *__restrict__ gate,
                                                            planes::View pv) {
    __shared__ float gm[kCThreads / 8], gl[kCThreads / 8];  // (head_dim >= 32: 8 threads a row at least)
    __shared__ float4 part_s[kCThreads];
    const int D = (int)sh.head_dim, DS = combine_slices(D), TPR = D / (4 * DS);
    const size_t h = blockIdx.x / DS, t = blockIdx.y;
    const int slice = (int)(blockIdx.x % DS);
    const int dg = (int)threadIdx.x % TPR, cg = (int)threadIdx.x / TPR, CG = kCThreads / TPR;
    const int e0 = slice * (D / DS) + 4 * dg;  // the thread's first element
    const size_t stride = (size_t)(D + 2);
    const float *part = partials + (t * sh.n_heads + h) * sh.chunks * stride;
    float M = -INFINITY, L = 0.0f;
    float4 acc = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    // (threads past the last whole group take no chunks)
    for (size_t c0 = cg; cg < CG && c0 < sh.chunks; c0 += (size_t)kU * CG) {
        float m[kU], l[kU];
        float2 oa[kU], ob[kU];
#pragma unroll
        for (int u = 0; u < kU; u++) {
            const size_t c = c0 + (size_t)u * CG;
            const size_t cc = c < sh.chunks ? c : c0;  // past the end: a chunk already counted, dropped below
            const float *row = part + cc * stride;
            m[u] = c < sh.chunks ? row[D] : -INFINITY;
            l[u] = row[D + 1];
            oa[u] = *(const float2 *)(row + e0);  // (D + 2)·4 bytes apart: 8-byte aligned only
            ob[u] = *(const float2 *)(row + e0 + 2);
        }
        float Mb = M;
#pragma unroll
        for (int u = 0; u < kU; u++) Mb = fmaxf(Mb, m[u]);
        if (Mb == -INFINITY) continue;  // nothing yet
        const float ra = expf(M - Mb);  // (M = −∞: 0)
        L *= ra;
        acc.x *= ra;
        acc.y *= ra;
        acc.z *= ra;
        acc.w *= ra;
#pragma unroll
        for (int u = 0; u < kU; u++) {
            // an empty chunk, or none: no term (its row holds only m and l)
            const bool live = m[u] != -INFINITY;
            const float rb = expf(m[u] - Mb);
            if (!live) oa[u] = ob[u] = make_float2(0.0f, 0.0f);
            L += live ? l[u] * rb : 0.0f;
            acc.x += oa[u].x * rb;
            acc.y += oa[u].y * rb;
            acc.z += ob[u].x * rb;
            acc.w += ob[u].y * rb;
        }
        M = Mb;
    }
    // the groups meet: every thread of a group holds the same M and L
    if (dg == 0) {
        gm[cg] = M;
        gl[cg] = L;
    }
    part_s[threadIdx.x] = acc;
    __syncthreads();
    if (cg != 0) return;
    float Mt = -INFINITY;
    for (int k = 0; k < CG; k++) Mt = fmaxf(Mt, gm[k]);
    float Lt = 0.0f;
    float4 sum = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    for (int k = 0; k < CG; k++) {
        if (gm[k] == -INFINITY) continue;
        const float r = expf(gm[k] - Mt);
        const float4 o = part_s[k * TPR + dg];
        Lt += gl[k] * r;
        sum.x += o.x * r;
        sum.y += o.y * r;
        sum.z += o.z * r;
        sum.w += o.w * r;
    }
    const size_t i = (t * sh.n_heads + h) * D + e0;
    float4 o = make_float4(sum.x / Lt, sum.y / Lt, sum.z / Lt, sum.w / Lt);
    if (gate) {
        const float4 gv = *(const float4 *)(gate + i);
        o.x *= sigmoidf_(gv.x);
        o.y *= sigmoidf_(gv.y);
        o.z *= sigmoidf_(gv.z);
        o.w *= sigmoidf_(gv.w);
    }
    *(float4 *)(out + i) = o;
    if (pv.q) {
        // token t's planes in the t-th area from pv's (a group of 16 is 4 lanes)
        const planes::View pt = t ? planes::view(pv.q + t * planes::kAreaBytes, pv.cols) : pv;
        planes::write4x4(pt, (h * D + e0) / 4, o);
    }
}

// ---------------------------------------------------------------- prefill


DEV ahalf8 hi8(const float *v) {
    ahalf8 h;
#pragma unroll
    for (int i = 0; i < 8; i++) h[i] = (_Float16)v[i];
    return h;
}
DEV ahalf8 lo8(const float *v, const ahalf8 &h) {
    ahalf8 l;
#pragma unroll
    for (int i = 0; i < 8; i++) l[i] = (_Float16)(v[i] - (float)h[i]);
    return l;
}

// ---------------------------------------------------------------- prefill, expanded cache
//
// The batch path in two launches.  k_kv_expand writes, per key/value head
// and step of 32 positions, 64 KB exactly as k_attn_flash holds a step in
// LDS, so that the attention kernel copies each step straight from global
// memory into LDS (global_load_lds, no registers, no conversion): the A
// operands of v_mfma_f32_32x32x16_f16, 1 KB each, lane l's 16 bytes at 16·l
// (r = l % 32, half = l / 32), the f16 hi parts and then the lo parts of
//   * keys, [16 dimensions 16·ks..]: position r, dimensions 16·ks + 8·half..;
//   * values, [16 positions 16·kp..][32 dimensions 32·dt..]: dimension 32·dt
//     + r, positions 16·kp + 4·half.. and 16·kp + 8 + 4·half.. (four and
//     four: the positions whose scores a lane of that half holds, so that the
//     probabilities are the other operand as they are).
// A Q8 value k8·s (an int8 times an f16 scale, 19 significant bits) is hi +
// lo exactly; an f16 cache's value is its hi part, and its lo parts, all
// zero, are neither written nor read.  Positions past the last are zeros.
constexpr unsigned kXStep = 32;                  // positions a step
constexpr size_t kXStepBytes = 65536;            // a step of one key/value head
constexpr int kXThreads = 256;

template <bool F16>
__global__ void __launch_bounds__(kXThreads) k_kv_expand(uint4 *__restrict__ xs, const int8_t *__restrict__ kq,
                                                          const uint16_t *__restrict__ ks,
                                                          const int8_t *__restrict__ vq,
                                                          const uint16_t *__restrict__ vs, unsigned len,
                                                          unsigned steps, unsigned kv_heads) {
    __shared__ float vt[kXStep][kFD + 1];
    const unsigned s = blockIdx.x, kvh = blockIdx.y, t = threadIdx.x;
    const unsigned r = t >> 3, c8 = t & 7;  // position r of the step, 32 dimensions 32·c8..
    const unsigned p = s * kXStep + r;
    const bool live = p < len;
    const size_t off = (size_t)(live ? p : 0) * kv_heads * kFD + (size_t)kvh * kFD + 32 * c8;
    uint4 *step = xs + ((size_t)kvh * steps + s) * (kXStepBytes / 16);
    float kv[32], vv[32];
    if constexpr (F16) {
        const uint4 *k16 = (const uint4 *)((const uint16_t *)kq + off), *v16 = (const uint4 *)((const uint16_t *)vq + off);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint4 a = k16[i], b = v16[i];
            const uint32_t aw[4] = {a.x, a.y, a.z, a.w}, bw[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
            for (int e = 0; e < 8; e++) {
                kv[8 * i + e] = half_of(aw[e / 2], e % 2);
                vv[8 * i + e] = half_of(bw[e / 2], e % 2);
            }
        }
    } else {
        const float ksc = dq::from_f16(ks[off / 32]), vsc = dq::from_f16(vs[off / 32]);
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const uint4 a = ((const uint4 *)(kq + off))[i], b = ((const uint4 *)(vq + off))[i];
            const uint32_t aw[4] = {a.x, a.y, a.z, a.w}, bw[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
            for (int e = 0; e < 16; e++) {
                kv[16 * i + e] = (float)(int8_t)((aw[e / 4] >> (8 * (e % 4))) & 0xffu) * ksc;
                vv[16 * i + e] = (float)(int8_t)((bw[e / 4] >> (8 * (e % 4))) & 0xffu) * vsc;
            }
        }
    }
#pragma unroll
    for (int i = 0; i < 32; i++) {
        kv[i] = live ? kv[i] : 0.0f;
        vt[r][32 * c8 + i] = live ? vv[i] : 0.0f;
    }
    // keys: 8-dimension groups 4·c8 + j of position r
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const ahalf8 h = hi8(kv + 8 * j);
        const unsigned c = 4 * c8 + j, at = (c >> 1) * 64 + (c & 1) * 32 + r;
        step[at] = __builtin_bit_cast(uint4, h);
        if (!F16) step[1024 + at] = __builtin_bit_cast(uint4, lo8(kv + 8 * j, h));
    }
    __syncthreads();
    // values: thread t takes dimension t, positions by 8 of an operand's lane
    uint4 *vdst = step + 2048;
    const unsigned d = t;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const unsigned kp = j >> 1, half = j & 1;
        float x[8];
#pragma unroll
        for (int i = 0; i < 8; i++) x[i] = vt[16 * kp + 8 * (i >> 2) + 4 * half + (i & 3)][d];
        const ahalf8 h = hi8(x);
        const unsigned at = (kp * 8 + (d >> 5)) * 64 + half * 32 + (d & 31);
        vdst[at] = __builtin_bit_cast(uint4, h);
        if (!F16) vdst[1024 + at] = __builtin_bit_cast(uint4, lo8(x, h));
    }
}

// Causal GQA for a batch of tokens over the expanded cache, on the f16
// matrix cores.  A row is a (token, query head) pair of one key/value head,
// token after token; a block of 4 waves takes 128 rows and a run of steps of
// 32 positions, a wave 32 rows with one SIMD to itself.  The scores are taken
// transposed, Sᵀ = K·Qᵀ, so that a lane holds 16 scores of one row: the
// softmax needs one exchange with the other half wave, its running max, sum
// and rescale are one value a lane, and the probabilities are the B operand of
// Oᵀ = Vᵀ·Pᵀ where they are.  Scores take three products (k hi·q hi, k hi·q lo,
// k lo·q hi; the queries times 1/16 = 1/sqrt(256), exact), values too (V hi·P
// hi, V lo·P hi, V hi·P lo).  Per step one barrier: every wave waits for its
// own copies (issued a step earlier), the barrier makes them visible and frees
// what the step before read; then the scores of step s + 1 are taken on the
// matrix cores while the softmax of step s runs beside them.
//
// What bounds it: 96 MFMAs a wave and step, 3072 cycles (1.3 us), which the
// softmax and the step's copies run beside where the order of the instructions
// lets them; LDS reads are 2048 cycles of a CU's.  1000 tokens of 24 / 4 heads
// at position 3001 (q8) took 428 us with a wave to 16 rows (the same LDS reads
// for half the products, and every wave's softmax at once after each barrier)
// and take 324; 256 tokens at 8192, 881 and 231 (both with the expansion).
// Copies all issued at a step's start, scores and softmax one after the other:
// 30 us more.  Rescaling O with every new max took 200 us more.
constexpr int kFlashLds = 2 * (int)kXStepBytes;

struct FlashArgs {
    float *out, *partials;  // partials: where parts > 1, [token][head][part][head_dim + 2]
    const float *q, *gate;
    const uint8_t *xs;  // the expanded cache, [kv head][step][64 KB]
    unsigned n, pos, heads, kv_heads, steps, tiles, parts;
};

typedef float afloat16 __attribute__((ext_vector_type(16)));

DEV afloat16 mfma32(const ahalf8 &a, const ahalf8 &b, const afloat16 &c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

// grid: kv_heads × tiles × parts (a key/value head's blocks on the same XCDs
// where the heads divide 8; the longest tiles first)
template <bool F16>
__global__ void __launch_bounds__(kFThreads, 1) k_attn_flash(const FlashArgs a) {
    extern __shared__ uint4 smem[];  // keys of two steps, values of two steps: 2048 × 16 bytes each
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r32 = lane & 31,
              half = lane >> 5;
    const unsigned G = a.heads / a.kv_heads, kvh = blockIdx.x % a.kv_heads, item = blockIdx.x / a.kv_heads;
    const unsigned tile = a.tiles - 1 - item / a.parts, part = item % a.parts;
    const unsigned row0 = tile * kFQ + 32 * w, row = row0 + r32;
    const bool live = row < a.n * G;
    const unsigned t = min(row / G, a.n - 1), head = kvh * G + row % G;
    const unsigned first = min(row0 / G, a.n - 1);                // the wave's first token
    const unsigned last = min((tile * kFQ + kFQ - 1) / G, a.n - 1);  // the block's last
    const unsigned all = (a.pos + last + kXStep) / kXStep, per = (all + a.parts - 1) / a.parts;
    const unsigned s0 = part * per, s1 = min(all, s0 + per);
    float *prow = a.partials + (((size_t)t * a.heads + head) * a.parts + part) * (kFD + 2);
    if (s0 >= s1) {  // (only where parts > 1)
        if (live && half == 0) {
            prow[kFD] = -INFINITY;
            prow[kFD + 1] = 0.0f;
        }
        return;
    }
    constexpr int kCopies = F16 ? 4 : 8;  // 1 KB pieces a wave copies of a step's keys, and of its values
    const uint8_t *src = a.xs + (size_t)kvh * a.steps * kXStepBytes + 1024 * kCopies * w + 16 * lane;
    // piece k of step s's keys or values
    auto copy = [&](unsigned s, int values, int k) __attribute__((always_inline)) {
        lds_copy16(src + (size_t)min(s, s1 - 1) * kXStepBytes + 32768 * values + 1024 * k,
                   (uint8_t *)smem + 65536 * values + 32768 * (s & 1) + 1024 * (kCopies * w + k));
    };
    ahalf8 qh[16], ql[16];
    {
        const float *qr = a.q + ((size_t)t * a.heads + head) * kFD + 8 * half;
        float4 qx[32];
#pragma unroll
        for (int g = 0; g < 32; g++) qx[g] = *(const float4 *)(qr + 8 * (g & ~1) + 4 * (g & 1));
        // the first step's keys and values, the second's keys
#pragma unroll
        for (int k = 0; k < kCopies; k++) {
            copy(s0, 0, k);
            copy(s0, 1, k);
        }
        if (s0 + 1 < s1) {
#pragma unroll
            for (int k = 0; k < kCopies; k++) copy(s0 + 1, 0, k);
        }
#pragma unroll
        for (int g = 0; g < 16; g++) {
            const float4 x0 = qx[2 * g], x1 = qx[2 * g + 1];
            float v[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
#pragma unroll
            for (int i = 0; i < 8; i++) v[i] *= 0.0625f;
            qh[g] = hi8(v);
            ql[g] = lo8(v, qh[g]);
        }
    }
    float m = -INFINITY, l = 0.0f;
    afloat16 o[8], zero;
#pragma unroll
    for (int i = 0; i < 16; i++) zero[i] = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; i++) o[i] = zero;
    // scores of step s: lane (half, r): positions 8·(i / 4) + 4·half + i % 4 of
    // row r; `beside(g)` after the g'th group of products, in that order (one
    // wave a SIMD: what the matrix cores run beside is what comes after them;
    // the operands are read four groups ahead)
    auto scores = [&](unsigned s, auto beside) __attribute__((always_inline)) {
        const uint4 *K = smem + (s & 1) * 2048 + lane;
        afloat16 c0 = zero, c1 = zero;
        ahalf8 kh[4], kl[4];
        auto read = [&](int g) __attribute__((always_inline)) {
            kh[g & 3] = __builtin_bit_cast(ahalf8, K[64 * g]);
            if (!F16) kl[g & 3] = __builtin_bit_cast(ahalf8, K[1024 + 64 * g]);
        };
#pragma unroll
        for (int g = 0; g < 4; g++) read(g);
#pragma unroll
        for (int g = 0; g < 16; g++) {
            c1 = mfma32(kh[g & 3], ql[g], c1);
            c0 = mfma32(kh[g & 3], qh[g], c0);
            if (!F16) c1 = mfma32(kl[g & 3], qh[g], c1);
            if (g + 4 < 16) read(g + 4);
            beside(g);
            __builtin_amdgcn_sched_barrier(0);
        }
        return c0 + c1;
    };
    __builtin_amdgcn_s_waitcnt(0x0f70);
    __syncthreads();
    afloat16 x = scores(s0, [](int) {});
    for (unsigned s = s0; s < s1; s++) {
        __builtin_amdgcn_s_waitcnt(0x0f70);  // this wave's copies of the keys of s + 1, the values of s
        __syncthreads();
        const unsigned p0 = s * kXStep;
        if (p0 + kXStep - 1 > a.pos + first) {
#pragma unroll
            for (int i = 0; i < 16; i++)
                if (p0 + 8 * (i / 4) + 4 * half + i % 4 > a.pos + t) x[i] = -INFINITY;
        }
        float mx = x[0];
#pragma unroll
        for (int i = 1; i < 16; i++) mx = fmaxf(mx, x[i]);
        float lo, hi;
        xlane::swap32(mx, lo, hi);
        // the reference the probabilities are taken from follows the max at a
        // distance of up to 8 (e^8 is well inside f16): rescaling O is rare then
        const float top = fmaxf(lo, hi), mn = top > m + 8.0f ? top : m;
        // ---- the next step's scores (past the last: of the copies of its own
        // keys, unused) and copies, beside this step's probabilities
        float p[16], sum = 0.0f;
        ahalf8 ph[2], pl[2];
        const afloat16 next = scores(s + 1, [&](int g) __attribute__((always_inline)) {
            if (g < kCopies) {
                copy(s + 2, 0, g);
                copy(s + 1, 1, g);
            }
            p[g] = x[g] == -INFINITY ? 0.0f : expf(x[g] - mn);
            sum += p[g];
            const _Float16 h = (_Float16)p[g];
            ph[g / 8][g % 8] = h;
            pl[g / 8][g % 8] = (_Float16)(p[g] - (float)h);
        });
        xlane::swap32(sum, lo, hi);
        sum = lo + hi;
        // (rows whose reference stays rescale by 1)
        if (__any(mn != m)) {
            const float alpha = mn == -INFINITY ? 1.0f : expf(m - mn);
            m = mn;
            l *= alpha;
            // (O is zero before the first step; in the accumulation registers, so
            // that it stays there: a block of asm waits itself for the matrix
            // cores' results and for its own)
            if (s > s0) {
                asm volatile("s_nop 15\n\ts_nop 15");
#pragma unroll
                for (int i = 0; i < 8; i++)
#pragma unroll
                    for (int j = 0; j < 16; j++) {
                        float e = o[i][j], tmp;
                        asm volatile("v_accvgpr_read_b32 %1, %0\n\ts_nop 1\n\tv_mul_f32 %1, %1, %2\n\ts_nop 1\n\tv_accvgpr_write_b32 %0, %1"
                                     : "+a"(e), "=&v"(tmp)
                                     : "v"(alpha));
                        o[i][j] = e;
                    }
                asm volatile("s_nop 15");
            }
        }
        l += sum;
        // ---- Oᵀ += Vᵀ·Pᵀ, 32 dimensions a tile
        const uint4 *V = smem + 4096 + (s & 1) * 2048 + lane;
        ahalf8 vh[2][2], vl[2][2];
        auto read = [&](int u) __attribute__((always_inline)) {
#pragma unroll
            for (int e = 0; e < 2; e++) {
                vh[u & 1][e] = __builtin_bit_cast(ahalf8, V[(2 * u + e) * 64]);
                if (!F16) vl[u & 1][e] = __builtin_bit_cast(ahalf8, V[1024 + (2 * u + e) * 64]);
            }
        };
        read(0);
#pragma unroll
        for (int u = 0; u < 8; u++) {  // two tiles of 32 dimensions
            const int kp = u / 4, d = u % 4 * 2;
            if (u < 7) read(u + 1);
#pragma unroll
            for (int e = 0; e < 2; e++) o[d + e] = mfma32(vh[u & 1][e], pl[kp], o[d + e]);
#pragma unroll
            for (int e = 0; e < 2; e++) o[d + e] = mfma32(vh[u & 1][e], ph[kp], o[d + e]);
            if (!F16) {
#pragma unroll
                for (int e = 0; e < 2; e++) o[d + e] = mfma32(vl[u & 1][e], ph[kp], o[d + e]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        x = next;
    }
    __builtin_amdgcn_s_waitcnt(0x0f70);  // (no copy outlives its block)
    if (!live) return;
    // ---- lane (half, r): dimensions 32·d + 8·j + 4·half.. of row r
    if (a.parts > 1) {
#pragma unroll
        for (int d = 0; d < 8; d++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                float2 *dst = (float2 *)(prow + 32 * d + 8 * j + 4 * half);  // (8-byte alignment only)
                dst[0] = make_float2(o[d][4 * j], o[d][4 * j + 1]);
                dst[1] = make_float2(o[d][4 * j + 2], o[d][4 * j + 3]);
            }
        if (half == 0) {
            prow[kFD] = m;
            prow[kFD + 1] = l;
        }
        return;
    }
    const float inv = 1.0f / l;
    const size_t at = ((size_t)t * a.heads + head) * kFD + 4 * half;
#pragma unroll
    for (int d = 0; d < 8; d++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const size_t idx = at + 32 * d + 8 * j;
            float4 r = make_float4(o[d][4 * j] * inv, o[d][4 * j + 1] * inv, o[d][4 * j + 2] * inv, o[d][4 * j + 3] * inv);
            if (a.gate) {
                const float4 g = *(const float4 *)(a.gate + idx);
                r.x *= sigmoidf_(g.x);
                r.y *= sigmoidf_(g.y);
                r.z *= sigmoidf_(g.z);
                r.w *= sigmoidf_(g.w);
            }
            *(float4 *)(a.out + idx) = r;
        }
}

// Where a batch's (key/value head, 128 rows) tiles leave CUs idle, their
// positions are split over blocks and the parts merged by k_attn_combine.  In
// microseconds: a block costs 2.4 a step and five steps' worth besides, the
// merge its launch, a row's blocks and the partial results, written and read.
// Whole / so split, 24 / 4 heads: 16 tokens at position 65000 6600 / 263 us (a
// whole block of the kernel before), 100 at 8000 (f16) 841 / 104; 512 at 512 in
// two parts 141, whole 98.  At most kFlashItems blocks a CU bound the scratch.
unsigned flash_parts(const dwim_dev *dev, size_t n, size_t pos, size_t n_heads, size_t n_kv_heads, size_t room) {
    const size_t rows = n * n_heads, tiles = (n * (n_heads / n_kv_heads) + kFQ - 1) / kFQ * n_kv_heads;
    const size_t steps = (pos + n + kXStep - 1) / kXStep, cus = (size_t)dev->cus;
    size_t best = 1;
    double least = 0.0;
    for (size_t p = 1; p <= steps && (p == 1 || (p * tiles <= kFlashItems * cus && p * rows * (kFD + 2) <= room)); p++) {
        const double rounds = (double)((p * tiles + cus - 1) / cus);
        const double cost = 2.4 * rounds * (double)((steps + p - 1) / p + 5) +
                            (p > 1 ? 4.0 + (3e-3 + 6e-4 * (double)p) * (double)rows : 0.0);
        if (p == 1 || cost < least) {
            least = cost;
            best = p;
        }
    }
    return (unsigned)best;
}

// Tokens a block where a batch of few rows over few positions goes to the
// decode pass (k_attn_mfma), 0 where not: as long as that pass's blocks are all resident at
// once.  There is no cache to expand then, and none of what a block of
// k_attn_flash does once (its queries, a prologue of two steps, the scores of
// the step past the last), most of its time when the steps are few.  Measured on
// MI355X (us, flash | so), 24 / 4 heads, q8: 16 tokens at position 0 16.4 | 13.6, at
// 100 23 | 14, at 1000 35 | 22.5; 32 at 0 17.6 | 16.7, at 200 32 | 19.  The pass takes
// 0.2 us more a token (its merge): 64 at 0 20 | 24, hence the limit of rows.
constexpr size_t kShortRows = 768;
size_t short_batch_tokens(const dwim_dev *dev, size_t n, size_t pos, size_t n_heads, size_t n_kv_heads) {
    const size_t G = n_heads / n_kv_heads, slots = kMPerCU * (size_t)dev->cus;
    const size_t base = (pos + n + kMStep - 1) / kMStep * n_kv_heads;
    if (n * n_heads > kShortRows) return 0;
    // (one tile of 16 rows a block, else two: 16 tokens of 24 / 4 heads 12 | 16 us)
    for (size_t T : {std::min((size_t)kTok, 16 / G), (size_t)kTok})
        if (base * ((n + T - 1) / T) <= slots) return T;
    return 0;
}
}  // namespace

// The partial results of a batch's positions split over blocks, for any
// batch of 16 tokens or more.
size_t attention_flash_floats(const dwim_dev *dev) {
    return kFlashItems * (size_t)dev->cus * kFQ * (kFD + 2);
}

// The decode path's partial results: [token][head][chunk][head_dim + 2] floats.
size_t attention_partials_floats(size_t n, size_t pos, size_t n_heads, size_t head_dim) {
    const size_t chunks = (pos + n + kPos - 1) / kPos;
    return n * n_heads * chunks * (head_dim + 2);
}

// Grows the device's partials buffer to `floats` (a model reserves its
// largest once, when it is built, so that no forward pass allocates).
hipError_t attention_reserve(dwim_dev *dev, size_t floats) {
    return dev_grow(dev, (void **)&dev->partials, &dev->partials_cap, floats, sizeof(float));
}

namespace {

// one token over at most this many positions: the one-chunk VALU pass, a
// single round of blocks (4k positions: 14.1 against 14.2 us with the merge;
// 32k: 47.8 against 31.2)
constexpr size_t kValuLen = 6144;

template <int RT, bool F16, bool WIDE>
hipError_t mfma_pass(dwim_dev *dev, dim3 grid, float *partials, const float *q, const dwim_cache *k,
                     const dwim_cache *v, const Shape &sh, int G, int T, float qscale) {
    constexpr size_t lds = mfma_lds(RT, F16);
    // once a process (thread-safe: a function-local static)
    static const hipError_t raised =
        hipFuncSetAttribute((const void *)k_attn_mfma<RT, F16, WIDE>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (raised != hipSuccess) return raised;
    k_attn_mfma<RT, F16, WIDE><<<grid, kMThreads, lds, dev->stream>>>(partials, q, k->q, k->s, v->q, v->s, sh, G, T, qscale);
    return hipGetLastError();
}

template <bool F16>
hipError_t flash_pass(dwim_dev *dev, const FlashArgs &fa) {
    // once a process (thread-safe: a function-local static)
    static const hipError_t raised =
        hipFuncSetAttribute((const void *)k_attn_flash<F16>, hipFuncAttributeMaxDynamicSharedMemorySize, kFlashLds);
    if (raised != hipSuccess) return raised;
    k_attn_flash<F16><<<fa.tiles * fa.parts * fa.kv_heads, kFThreads, kFlashLds, dev->stream>>>(fa);
    return hipGetLastError();
}

// Both entry points' launches: the batch path on the matrix cores (its
// positions split where `room` floats of `partials` allow), or the chunked
// decode path with its partial results in `partials` (at least
// attention_partials_floats).
hipError_t attention_run(dwim_dev *dev, float *partials, float *out, const float *q, const dwim_cache *k,
                         const dwim_cache *v, size_t n, size_t pos, size_t n_heads, size_t head_dim,
                         size_t n_kv_heads, const float *gate, planes::View pv, uint8_t *kvx, size_t room) {
    const size_t few = n >= 16 && !pv.q && head_dim == (size_t)kFD ? short_batch_tokens(dev, n, pos, n_heads, n_kv_heads) : 0;
    const bool fits = partials && n * n_heads * ((pos + n + kMStep - 1) / kMStep) * (kFD + 2) <= room;
    if (n >= 16 && !pv.q && head_dim == (size_t)kFD && n_heads % n_kv_heads == 0 && !(few && fits)) {
        // a batch of tokens over the expanded cache (kvx: attention_kvx_bytes)
        const size_t len = pos + n, steps = (len + kXStep - 1) / kXStep;
        dim3 gx((unsigned)steps, (unsigned)n_kv_heads);
        if (k->f16)
            k_kv_expand<true><<<gx, kXThreads, 0, dev->stream>>>((uint4 *)kvx, k->q, k->s, v->q, v->s, (unsigned)len,
                                                               (unsigned)steps, (unsigned)n_kv_heads);
        else
            k_kv_expand<false><<<gx, kXThreads, 0, dev->stream>>>((uint4 *)kvx, k->q, k->s, v->q, v->s, (unsigned)len,
                                                                (unsigned)steps, (unsigned)n_kv_heads);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        const size_t rows = n * (n_heads / n_kv_heads);
        const unsigned tiles = (unsigned)((rows + kFQ - 1) / kFQ);
        const unsigned parts = flash_parts(dev, n, pos, n_heads, n_kv_heads, partials ? room : 0);
        FlashArgs fa{out, partials, q, gate, kvx, (unsigned)n, (unsigned)pos, (unsigned)n_heads, (unsigned)n_kv_heads,
                     (unsigned)steps, tiles, parts};
        e = k->f16 ? flash_pass<true>(dev, fa) : flash_pass<false>(dev, fa);
        if (e != hipSuccess || parts == 1) return e;
        dim3 g2((unsigned)n_heads * (unsigned)(head_dim / 64), (unsigned)n);
        k_attn_combine<<<g2, kCThreads, 0, dev->stream>>>(out, partials, Shape{n, pos, n_heads, head_dim, n_kv_heads, 0, parts},
                                                          gate, pv);
        return hipGetLastError();
    }
    const size_t len = pos + n;
    if (head_dim == (size_t)kFD && (n > 1 || len > kValuLen)) {
        // the matrix-core pass: a run of 64-position steps a block, as few as
        // keep every block resident at once (two a CU): a second round of a
        // few blocks costs a whole block's time (32k + 1 positions: 412 blocks
        // of 5 steps, not 516 of 4; in the model 43.3 against 47.5 us a
        // 4-token pass, 9.4 against 10.9 us its merge)
        const int G = (int)(n_heads / n_kv_heads), T = few ? (int)few : n > 1 ? kTok : 1;
        const float qscale = few ? 0.0625f : 1.0f;  // (a batch's queries have the range k_attn_flash gives them)
        const size_t groups = (n + T - 1) / T, base = (len + kMStep - 1) / kMStep * n_kv_heads * groups;
        const size_t slots = kMPerCU * (size_t)dev->cus;
        const size_t ch = kMStep * std::max<size_t>(1, (base + slots - 1) / slots), chunks = (len + ch - 1) / ch;
        Shape sh{n, pos, n_heads, head_dim, n_kv_heads, ch, chunks};
        dim3 g1((unsigned)chunks, (unsigned)n_kv_heads, (unsigned)groups);
        auto pass = T * G <= 16 ? (k->f16 ? mfma_pass<1, true, false> : few ? mfma_pass<1, false, true> : mfma_pass<1, false, false>)
                                : (k->f16 ? mfma_pass<2, true, false> : few ? mfma_pass<2, false, true> : mfma_pass<2, false, false>);
        hipError_t e = pass(dev, g1, partials, q, k, v, sh, G, T, qscale);
        if (e != hipSuccess) return e;
        dim3 g2((unsigned)n_heads * (unsigned)(head_dim / 64), (unsigned)n);
        k_attn_combine<<<g2, kCThreads, 0, dev->stream>>>(out, partials, sh, gate, pv);
        return hipGetLastError();
    }
    const size_t ch = kPos, chunks = (len + ch - 1) / ch;
    Shape sh{n, pos, n_heads, head_dim, n_kv_heads, ch, chunks};
    // one token a block, or a few tokens' queries against the chunk read once
    const bool grouped = n > 1;
    dim3 g1((unsigned)chunks, (unsigned)n_kv_heads, (unsigned)(grouped ? (n + kTok - 1) / kTok : n));
    switch (n_heads / n_kv_heads) {
#define DWIM_PARTIAL_T(G, T)                                                                                    \
    if (k->f16) k_attn_partial<G, true, T><<<g1, kPThreads, 0, dev->stream>>>(partials, q, k->q, k->s, v->q, v->s, sh); \
    else k_attn_partial<G, false, T><<<g1, kPThreads, 0, dev->stream>>>(partials, q, k->q, k->s, v->q, v->s, sh);
#define DWIM_PARTIAL(G)                                                                                        \
    case G:                                                                                                    \
        if (grouped) {                                                                                         \
            DWIM_PARTIAL_T(G, kTok)                                                                            \
        } else {                                                                                               \
            DWIM_PARTIAL_T(G, 1)                                                                               \
        }                                                                                                      \
        break;
        DWIM_PARTIAL(1) DWIM_PARTIAL(2) DWIM_PARTIAL(3) DWIM_PARTIAL(4) DWIM_PARTIAL(5) DWIM_PARTIAL(6)
        DWIM_PARTIAL(7) DWIM_PARTIAL(8)
#undef DWIM_PARTIAL
#undef DWIM_PARTIAL_T
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const unsigned ds = head_dim % 64 == 0 ? (unsigned)(head_dim / 64) : 1u;
    dim3 g2((unsigned)n_heads * ds, (unsigned)n);
    k_attn_combine<<<g2, kCThreads, 0, dev->stream>>>(out, partials, sh, gate, pv);
    return hipGetLastError();
}

bool attention_shape_ok(size_t n_heads, size_t head_dim, size_t n_kv_heads) {
    return !(head_dim % 32 || head_dim > kMaxD || n_kv_heads == 0 || n_heads % n_kv_heads ||
             n_heads / n_kv_heads > kMaxG);
}

}  // namespace

hipError_t launch_attention(dwim_dev *dev, float *out, const float *q, const dwim_cache *k, const dwim_cache *v,
                            size_t n, size_t pos, size_t n_heads, size_t head_dim, size_t n_kv_heads) {
    return launch_attention_gated(dev, out, q, k, v, n, pos, n_heads, head_dim, n_kv_heads, nullptr, -1);
}

hipError_t launch_attention_gated(dwim_dev *dev, float *out, const float *q, const dwim_cache *k,
                                  const dwim_cache *v, size_t n, size_t pos, size_t n_heads, size_t head_dim,
                                  size_t n_kv_heads, const float *gate, int area) {
    if (!attention_shape_ok(n_heads, head_dim, n_kv_heads)) return hipErrorInvalidValue;
    planes::View pv{};
    if (area >= 0) {
        // one token's planes, or 2..4 tokens' in a set of batch areas
        const bool areas_ok = n == 1 || (n <= 4 && (area == kBatchArea || area == kBatchArea2));
        if (!areas_ok || head_dim % 32 || n_heads * head_dim > planes::kMaxCols || (n_heads * head_dim) % 256)
            return hipErrorInvalidValue;
        pv = planes_area(dev, area, n_heads * head_dim);
        dev->prepared = 0;
    }
    const bool batch = n >= 16 && area < 0 && head_dim == (size_t)kFD;
    if (!batch) {
        hipError_t e = attention_reserve(dev, attention_partials_floats(n, pos, n_heads, head_dim));
        if (e != hipSuccess) return e;
        return attention_run(dev, dev->partials, out, q, k, v, n, pos, n_heads, head_dim, n_kv_heads, gate, pv,
                             nullptr, dev->partials_cap);
    }
    hipError_t e = attention_kvx_reserve(dev, attention_kvx_bytes(pos + n, n_kv_heads));
    if (e != hipSuccess) return e;
    // (without it, in a capture: what there is)
    (void)dev_grow_unless_capturing(dev, (void **)&dev->partials, &dev->partials_cap, attention_flash_floats(dev),
                                    sizeof(float));
    return attention_run(dev, dev->partials, out, q, k, v, n, pos, n_heads, head_dim, n_kv_heads, gate, pv,
                         (uint8_t *)dev->kvx, dev->partials_cap);
}

// The expanded cache of a batch over `len` positions (head_dim 256).
size_t attention_kvx_bytes(size_t len, size_t n_kv_heads) {
    return (len + kXStep - 1) / kXStep * kXStepBytes * n_kv_heads;
}

hipError_t attention_kvx_reserve(dwim_dev *dev, size_t bytes) {
    return dev_grow(dev, &dev->kvx, &dev->kvx_cap, bytes, 1);
}

// ---------------------------------------------------------------- without allocating
//
// dwim_attention_noalloc keeps the decode path's partial results in this
// file-scope array instead of the device's grown buffer.  Every GPU holds its
// own copy of it (64 MiB) until the process ends; its address on a device is
// taken once, when the device is opened (attention_scratch_init), and used
// wherever host code needs the array.  Calls on one GPU share it, so calls
// that overlap on one device race.  Nothing in it needs to start at zero:
// each chunk's partial row is written before the combine reads it.
namespace {
constexpr size_t kScratchFloats = (size_t)16 << 20;
__device__ __align__(256) float scratch[kScratchFloats];
}  // namespace

hipError_t attention_scratch_init(dwim_dev *dev) {
    void *ptr = nullptr;
    hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    dev->attn_scratch = (float *)ptr;
    return hipSuccess;
}

extern "C" int dwim_attention_noalloc(dwim_dev *dev, dwim_buf *out, const dwim_buf *q, const dwim_cache *k_cache,
                                      const dwim_cache *v_cache, size_t pos, size_t n_heads, size_t head_dim,
                                      size_t n_kv_heads) {
    DWIM_CHECK(head_dim % 32 == 0 && head_dim <= 256 && head_dim > 0,
               "attention: heads are whole blocks of 32, at most 256");
    DWIM_CHECK(n_kv_heads > 0 && n_heads % n_kv_heads == 0 && n_heads / n_kv_heads <= 8,
               "attention: at most 8 query heads to a key/value head");
    const size_t width = n_heads * head_dim;
    DWIM_CHECK(q->len % width == 0 && out->len == q->len, "attention: q and out are whole tokens");
    const size_t n = q->len / width, kv_dim = n_kv_heads * head_dim;
    DWIM_CHECK((pos + n) * kv_dim <= k_cache->len && (pos + n) * kv_dim <= v_cache->len,
               "attention: the caches do not hold the tokens' positions");
    DWIM_CHECK(k_cache->f16 == v_cache->f16, "attention: the key and value caches are of different formats");
    DWIM_CHECK(dev->attn_scratch != nullptr, "attention_noalloc: the device's scratch array has no address");
    if (n == 0) return 0;
    const bool batch = n >= 16 && head_dim == (size_t)kFD;
    // the decode path's partial results, or a batch's expanded cache
    const size_t need = batch ? attention_kvx_bytes(pos + n, n_kv_heads)
                              : attention_partials_floats(n, pos, n_heads, head_dim) * sizeof(float);
    DWIM_CHECK(need <= kScratchFloats * sizeof(float),
               "attention_noalloc: " + std::to_string(n) + " tokens at position " + std::to_string(pos) + " need " +
                   std::to_string(need) + " bytes of " + (batch ? "expanded cache" : "partial results") +
                   ", more than the " + std::to_string(kScratchFloats * 4) + " bytes of its scratch array");
    // (a batch's partial results in what its expanded cache leaves)
    const size_t held = batch ? need / sizeof(float) : 0;
    DWIM_HIP(attention_run(dev, dev->attn_scratch + held, out->data, q->data, k_cache, v_cache, n, pos, n_heads,
                           head_dim, n_kv_heads, nullptr, planes::View{}, (uint8_t *)dev->attn_scratch,
                           kScratchFloats - held));
    return 0;
}
