// The gated delta rule of linear attention, token after token
// (dwim gpu/cpu.rs:298-363).  For value head h (key head h / (n_v/n_k)) and
// each token: g = exp(a·softplus(alpha + dt_bias)), beta = sigmoid(beta_logit);
// S *= g; kv = Sᵀk; S += k ⊗ (v − kv)·beta; o = Sᵀq / sqrt(d); with the state
// S stored s[key][value].
//
// Every value column j of S evolves on its own: kv[j], the update of column j
// and o[j] read only column j.  So a block owns 16 columns of one head (grid
// = 8 × n_v_heads) and keeps its 128×16 slice of the fp32 state in registers
// across all the batch's tokens: thread (column c, part p) holds keys
// 8p..8p+7 of column c, and the 16 parts of a column are 16 adjacent lanes
// whose partial sums meet by DPP moves.  The token loop is a chain of
// dependent steps, so it is kept short and free of global loads: the inputs
// of a run of 64 tokens (keys, queries, the block's values, the gates g and
// beta) are staged in LDS at once, the next run's loaded into registers while
// this run's tokens are computed, and each sum runs in two accumulators.  The
// slice is read from HBM once and written once per call, through LDS so that
// both are coalesced.
#include "device_util.h"
#include "planes.h"
#include "runtime.h"

#include <algorithm>

typedef float v4f __attribute__((ext_vector_type(4)));

namespace {

constexpr int kD = 128;      // head_dim (the reference asserts 128, gpu/cuda/mod.rs:1437)
constexpr int kCols = 16;    // value columns per block
constexpr int kParts = 16;   // key parts per column
constexpr int kKeys = kD / kParts;
constexpr int kThreads = kCols * kParts;
constexpr int kRun = 64;  // tokens whose inputs a block stages in LDS at once

// sum over 16 aligned adjacent lanes, every lane getting it: quad xor 1 and
// 2, then the half-row mirror (lane i and 7 − i) and the row mirror (i and
// 15 − i)
DEV float sum16(float v) {
    v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xb1, 0xf, 0xf, false));
    v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x4e, 0xf, 0xf, false));
    v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x141, 0xf, 0xf, false));
    v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x140, 0xf, 0xf, false));
    return v;
}

__global__ void __launch_bounds__(kThreads) k_delta_net(float *__restrict__ out, const float *__restrict__ q,
                                                        const float *__restrict__ k, const float *__restrict__ v,
                                                        const float *__restrict__ gates,
                                                        const float *__restrict__ decay, float *state,
                                                        const float *state_in, size_t n, int n_k_heads, int n_v_heads,
                                                        Rms rms) {
    // a run's keys and queries [token][key] (also the state slice's staging
    // at the start and the end), values [token][column] and gates
    __shared__ v4f kq[2][kRun][kD / 4];
    __shared__ float vs[kRun][kCols];
    __shared__ float2 gb[kRun];  // per token: g, beta
    __shared__ float red[kThreads / 64];
    float(*tile)[kCols + 1] = (float(*)[kCols + 1]) & kq[0][0][0];  // [kD][kCols + 1]
    // the gates' RMS scale, when the gate projection took x·w unscaled
    float gs = 1.0f;
    if (rms.ss) {
        float t = 0.0f;
        for (unsigned g = threadIdx.x; g < rms.groups; g += kThreads) t += rms.ss[g];
        t = block_sum<kThreads>(t, red);
        gs = 1.0f / sqrtf(t / rms.cols + rms.eps);
    }
    const int h = blockIdx.y, c0 = blockIdx.x * kCols;
    const int kh = h / (n_v_heads / n_k_heads);
    const int c = threadIdx.x / kParts, p = threadIdx.x % kParts;
    float *S = state + (size_t)h * kD * kD;
    const float *Sin = state_in + (size_t)h * kD * kD;

    // state slice in (from state_in, out to state): rows of 16 columns, coalesced
    for (int e = threadIdx.x; e < kD * kCols; e += kThreads) tile[e / kCols][e % kCols] = Sin[(e / kCols) * kD + c0 + e % kCols];
    __syncthreads();
    float s[kKeys];
#pragma unroll
    for (int i = 0; i < kKeys; i++) s[i] = tile[p * kKeys + i][c];

    const float scale = 1.0f / sqrtf((float)kD);
    const float a = decay[h], dt = decay[n_v_heads + h];
    // a run's inputs, loaded into registers while the run before it is
    // computed: thread i takes float4s i, i + 256, ... of the run's keys and
    // queries ([2][kRun][32] float4s), and value (token i / 16, column i % 16)
    // for i < kRun·16 (four a thread), and the gate logits of token i < kRun
    constexpr int kKQ = 2 * kRun * kD / 4 / kThreads, kV = kRun * kCols / kThreads;
    v4f rkq[kKQ];  // (vector types: an array of float4 structs stays in private memory)
    float rv[kV], ra = 0.0f, rb = 0.0f;
    auto fetch = [&](size_t r0) {
        const size_t rn = n - r0 < (size_t)kRun ? n - r0 : (size_t)kRun;
#pragma unroll
        for (int u = 0; u < kKQ; u++) {
            const int f = threadIdx.x + kThreads * u, which = f / (kRun * kD / 4), tok = (f / (kD / 4)) % kRun;
            const size_t t = r0 + ((size_t)tok < rn ? tok : 0);
            rkq[u] = ((const v4f *)((which ? q : k) + (t * n_k_heads + kh) * kD))[f % (kD / 4)];
        }
#pragma unroll
        for (int u = 0; u < kV; u++) {
            const int f = threadIdx.x + kThreads * u, tok = f / kCols;
            const size_t t = r0 + ((size_t)tok < rn ? tok : 0);
            rv[u] = v[(t * n_v_heads + h) * kD + c0 + f % kCols];
        }
        if (threadIdx.x < kRun) {
            const size_t t = r0 + (threadIdx.x < rn ? threadIdx.x : 0);
            ra = gates[t * 2 * n_v_heads + h];
            rb = gates[t * 2 * n_v_heads + n_v_heads + h];
        }
    };
    if (n > 0) fetch(0);
    for (size_t r0 = 0; r0 < n; r0 += kRun) {
        const size_t rn = n - r0 < (size_t)kRun ? n - r0 : (size_t)kRun;
        __syncthreads();  // the run before has been read
#pragma unroll
        for (int u = 0; u < kKQ; u++) {
            const int f = threadIdx.x + kThreads * u;
            (&kq[0][0][0])[f] = rkq[u];
        }
#pragma unroll
        for (int u = 0; u < kV; u++) (&vs[0][0])[threadIdx.x + kThreads * u] = rv[u];
        // g = exp(a·softplus(alpha + dt_bias)), beta = sigmoid(beta_logit)
        if (threadIdx.x < kRun) gb[threadIdx.x] = make_float2(expf(a * softplusf_(gs * ra + dt)), sigmoidf_(gs * rb));
        __syncthreads();
        if (r0 + kRun < n) fetch(r0 + kRun);
        for (size_t tt = 0; tt < rn; tt++) {
            const size_t t = r0 + tt;
            float kk[kKeys], qq[kKeys];
#pragma unroll
            for (int i = 0; i < kKeys / 4; i++) {
                const v4f k4 = kq[0][tt][p * (kKeys / 4) + i], q4 = kq[1][tt][p * (kKeys / 4) + i];
                kk[4 * i] = k4.x; kk[4 * i + 1] = k4.y; kk[4 * i + 2] = k4.z; kk[4 * i + 3] = k4.w;
                qq[4 * i] = q4.x; qq[4 * i + 1] = q4.y; qq[4 * i + 2] = q4.z; qq[4 * i + 3] = q4.w;
            }
            const float2 g2 = gb[tt];
            const float g = g2.x, beta = g2.y;
            float kv0 = 0.0f, kv1 = 0.0f;
#pragma unroll
            for (int i = 0; i < kKeys; i += 2) {
                s[i] *= g;
                s[i + 1] *= g;
                kv0 += s[i] * kk[i];
                kv1 += s[i + 1] * kk[i + 1];
            }
            const float kv = sum16(kv0 + kv1);
            const float ub = (vs[tt][c] - kv) * beta;
            float o0 = 0.0f, o1 = 0.0f;
#pragma unroll
            for (int i = 0; i < kKeys; i += 2) {
                s[i] += kk[i] * ub;
                s[i + 1] += kk[i + 1] * ub;
                o0 += s[i] * qq[i];
                o1 += s[i + 1] * qq[i + 1];
            }
            const float o = sum16(o0 + o1) * scale;
            if (p == 0) out[(t * n_v_heads + h) * kD + c0 + c] = o;
        }
    }

    // state slice out, through LDS
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kKeys; i++) tile[p * kKeys + i][c] = s[i];
    __syncthreads();
    for (int e = threadIdx.x; e < kD * kCols; e += kThreads) S[(e / kCols) * kD + c0 + e % kCols] = tile[e / kCols][e % kCols];
}


// ---- A small batch's whole mixer step --------------------------------------
//
// For batches of up to kSmallT tokens (speculative-decoding verify batches,
// the rewind's re-run, small prompt pieces): the conv of 4 taps + SiLU over
// the batch with its carried state (gpu/cpu.rs:250-296), the l2 norms of q
// and k (:157-166 without weights) and the delta rule (:298-363), in one
// launch of k_delta_net's blocks (16 value columns of one head a block, the
// state slice in registers).  Each block makes its key head's q and k itself
// (a channel a thread, the window sliding in registers, each token's norm a
// block sum) and its own 16 value channels, straight into the LDS the token
// loop reads; the conv state carried to the next batch is written by the key
// head's first block (q and k channels) and by each block (its value
// channels).  The same arithmetic as the three calls it replaces.
constexpr int kSmallT = 16;

__global__ void __launch_bounds__(kThreads) k_gdn_tokens(float *__restrict__ out, const float *__restrict__ qkv,
                                                         const float *__restrict__ conv_state,
                                                         float *__restrict__ conv_state_out,
                                                         const float *__restrict__ conv_w,
                                                         const float *__restrict__ gates,
                                                         const float *__restrict__ decay, float *state,
                                                         const float *state_in, int n, int n_k_heads, int n_v_heads,
                                                         float eps, GdnSteps steps, GdnGate gg) {
    __shared__ float kqs[2][kSmallT][kD];          // normalized k, q of each token
    __shared__ float tile[kD][kCols + 1];          // the state slice's staging
    __shared__ float vs[kSmallT][kCols];
    __shared__ float2 gb[kSmallT];
    __shared__ float red[kSmallT][kThreads / 64];
    __shared__ float o_s[4][kCols];  // (with gg.planes: the first 4 tokens' o)
    const int h = blockIdx.y, c0 = blockIdx.x * kCols, tid = threadIdx.x;
    const int ratio = n_v_heads / n_k_heads, kh = h / ratio;
    const int c = tid / kParts, p = tid % kParts;
    const size_t ch = (size_t)(2 * n_k_heads + n_v_heads) * kD;
    float *S = state + (size_t)h * kD * kD;
    const float *Sin = state_in + (size_t)h * kD * kD;

    // ---- loads: the state slice, this thread's q or k channel over the
    // batch (with its window and weights), the block's value channels, the
    // gate logits
    // (every load of the block issues before any is waited for: the slice
    // into registers here, into LDS once the others are issued)
    constexpr int kTileLoads = kD * kCols / kThreads;
    float tl[kTileLoads];
#pragma unroll
    for (int u = 0; u < kTileLoads; u++) {
        const int e = tid + u * kThreads;
        tl[u] = Sin[(e / kCols) * kD + c0 + e % kCols];
    }
    const size_t qk = tid < kD ? (size_t)kh * kD + tid : (size_t)(n_k_heads + kh) * kD + (tid - kD);
    float win[kSmallT + 3];
#pragma unroll
    for (int j = 0; j < 3; j++) win[j] = conv_state[(size_t)j * ch + qk];
#pragma unroll
    for (int t = 0; t < kSmallT; t++) win[3 + t] = t < n ? qkv[(size_t)t * ch + qk] : 0.0f;
    const float4 w = ((const float4 *)conv_w)[qk];
    const size_t vc = (size_t)(2 * n_k_heads + h) * kD + c0 + (tid % kCols);
    const bool vlane = tid < kCols;
    const float a = decay[h], dt = decay[n_v_heads + h];
    // the value lanes' channels (loaded by all of wave 0, so that the loads
    // issue here, unconditionally within the wave) and the gate logits
    float vw[kSmallT + 3];
    float4 vwt = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (tid < 64) {
#pragma unroll
        for (int j = 0; j < 3; j++) vw[j] = conv_state[(size_t)j * ch + vc];
#pragma unroll
        for (int t = 0; t < kSmallT; t++) vw[3 + t] = t < n ? qkv[(size_t)t * ch + vc] : 0.0f;
        vwt = ((const float4 *)conv_w)[vc];
    }
    // (with gg.planes: wave 0, lane 16t + c, takes token t's column c at the end)
    float zv = 0.0f, nwv = 0.0f;
    if (gg.planes && tid < 64 && (tid >> 4) < n) {
        zv = gg.z[(size_t)(tid >> 4) * n_v_heads * kD + (size_t)h * kD + c0 + (tid & 15)];
        nwv = gg.norm_w[c0 + (tid & 15)];
    }
    float g_alpha = 0.0f, g_beta = 0.0f;
    if (tid < n) {
        g_alpha = gates[(size_t)tid * 2 * n_v_heads + h];
        g_beta = gates[(size_t)tid * 2 * n_v_heads + n_v_heads + h];
    }

    // ---- q and k: conv + SiLU, each token's sum of squares a block sum
    // over its half (q: waves 0-1, k: waves 2-3)
    float y[kSmallT];
#pragma unroll
    for (int t = 0; t < kSmallT; t++) {
        y[t] = 0.0f;
        if (t < n) {  // (uniform: the batch's tokens only)
            float acc = 0.0f;
            acc += w.x * win[t];
            acc += w.y * win[t + 1];
            acc += w.z * win[t + 2];
            acc += w.w * win[t + 3];
            y[t] = acc * sigmoidf_(acc);
            const float sq = group_sum<64>(y[t] * y[t]);
            if ((tid & 63) == 0) red[t][tid >> 6] = sq;
        }
    }
    // the last three inputs carry over: after the batch, window entries
    // n..n+2 (the state's rows when the batch is shorter); with steps, also
    // after each earlier token t, entries t+1..t+3 (the conv state of t + 1
    // kept).  Stored from the window's registers, every index a constant (a
    // branch per batch size), so that no store waits for a load of its own.
    // (a macro rather than a lambda over the array, which would put the
    // window in scratch memory)
#define DWIM_GDN_CARRY(WV, IDX)                                                                   \
    {                                                                                            \
        float c0 = 0.0f, c1 = 0.0f, c2 = 0.0f;                                                   \
        _Pragma("unroll") for (int m = 1; m <= kSmallT; m++) if (m == n) {                       \
            c0 = WV[m];                                                                          \
            c1 = WV[m + 1];                                                                      \
            c2 = WV[m + 2];                                                                      \
        }                                                                                        \
        conv_state_out[(IDX)] = c0;                                                              \
        conv_state_out[ch + (IDX)] = c1;                                                         \
        conv_state_out[2 * ch + (IDX)] = c2;                                                     \
        _Pragma("unroll") for (int t = 0; t < kMaxSteps && t + 1 < kSmallT; t++) {               \
            if (t + 1 < n && steps.conv[t]) {                                                    \
                steps.conv[t][(IDX)] = WV[t + 1];                                                \
                steps.conv[t][ch + (IDX)] = WV[t + 2];                                           \
                steps.conv[t][2 * ch + (IDX)] = WV[t + 3];                                       \
            }                                                                                    \
        }                                                                                        \
    }
    if (blockIdx.x == 0 && h % ratio == 0) DWIM_GDN_CARRY(win, qk)
    if (vlane) {
#pragma unroll
        for (int t = 0; t < kSmallT; t++) {
            if (t < n) {
                float acc = 0.0f;
                acc += vwt.x * vw[t];
                acc += vwt.y * vw[t + 1];
                acc += vwt.z * vw[t + 2];
                acc += vwt.w * vw[t + 3];
                vs[t][tid] = acc * sigmoidf_(acc);
            }
        }
        DWIM_GDN_CARRY(vw, vc)
    }
    // g = exp(a·softplus(alpha + dt_bias)), beta = sigmoid(beta_logit)
    if (tid < n) gb[tid] = make_float2(expf(a * softplusf_(g_alpha + dt)), sigmoidf_(g_beta));
#pragma unroll
    for (int u = 0; u < kTileLoads; u++) {
        const int e = tid + u * kThreads;
        tile[e / kCols][e % kCols] = tl[u];
    }
    __syncthreads();
    {
        const int half = tid >> 7;  // 0: q, 1: k
#pragma unroll
        for (int t = 0; t < kSmallT; t++) {
            if (t < n) {
                const float ss = red[t][2 * half] + red[t][2 * half + 1];
                kqs[half ? 0 : 1][t][tid & (kD - 1)] = y[t] * (1.0f / sqrtf(ss + eps));
            }
        }
    }
    float s[kKeys];
#pragma unroll
    for (int i = 0; i < kKeys; i++) s[i] = tile[p * kKeys + i][c];
    __syncthreads();

    // ---- the token loop (k_delta_net's)
    const float scale = 1.0f / sqrtf((float)kD);
    for (int t = 0; t < n; t++) {
        float kk[kKeys], qq[kKeys];
#pragma unroll
        for (int i = 0; i < kKeys; i++) {
            kk[i] = kqs[0][t][p * kKeys + i];
            qq[i] = kqs[1][t][p * kKeys + i];
        }
        const float2 g2 = gb[t];
        const float g = g2.x, beta = g2.y;
        float kv0 = 0.0f, kv1 = 0.0f;
#pragma unroll
        for (int i = 0; i < kKeys; i += 2) {
            s[i] *= g;
            s[i + 1] *= g;
            kv0 += s[i] * kk[i];
            kv1 += s[i + 1] * kk[i + 1];
        }
        const float kv = sum16(kv0 + kv1);
        const float ub = (vs[t][c] - kv) * beta;
        float o0 = 0.0f, o1 = 0.0f;
#pragma unroll
        for (int i = 0; i < kKeys; i += 2) {
            s[i] += kk[i] * ub;
            s[i + 1] += kk[i + 1] * ub;
            o0 += s[i] * qq[i];
            o1 += s[i + 1] * qq[i + 1];
        }
        const float o = sum16(o0 + o1) * scale;
        if (p == 0 && out) out[((size_t)t * n_v_heads + h) * kD + c0 + c] = o;
        if (p == 0 && gg.planes && t < 4) o_s[t][c] = o;
        if (t + 1 < n && t < kMaxSteps && steps.state[t]) {
            // the state after token t, for a rewind that keeps t + 1 tokens
            // (through LDS, a row's 16 columns in one run, as at the end)
            float *St = steps.state[t] + (size_t)h * kD * kD;
            __syncthreads();  // (the previous step's copy is done with the tile)
#pragma unroll
            for (int i = 0; i < kKeys; i++) tile[p * kKeys + i][c] = s[i];
            __syncthreads();
            for (int e = tid; e < kD * kCols; e += kThreads) St[(e / kCols) * kD + c0 + e % kCols] = tile[e / kCols][e % kCols];
        }
    }

    // ---- the state slice out, through LDS
    __syncthreads();  // (a step's copy may still read the tile; o_s is written)
    if (gg.planes && tid < 64 && (tid >> 4) < n) {
        // token t's gated output of the block's 16 columns as one planes group
        // (whole groups of 16 lanes), unnormalized, and their Σo²
        const int t = tid >> 4, cc = tid & 15;
        const float ov = o_s[t][cc];
        const float ss = group_sum<16>(ov * ov);
        if (cc == 0) gg.head_ss[((size_t)t * n_v_heads + h) * (kD / kCols) + blockIdx.x] = ss;
        const float r = zv * sigmoidf_(zv) * (ov * nwv);
        planes::write16(planes::view(gg.planes + (size_t)t * planes::kAreaBytes, (size_t)n_v_heads * kD),
                        (size_t)h * kD + c0 + cc, r);
    }
#pragma unroll
    for (int i = 0; i < kKeys; i++) tile[p * kKeys + i][c] = s[i];
    __syncthreads();
    for (int e = tid; e < kD * kCols; e += kThreads) S[(e / kCols) * kD + c0 + e % kCols] = tile[e / kCols][e % kCols];
}
#undef DWIM_GDN_CARRY

// ---- The chunked form, for batches of at least kC tokens -------------------
//
// Over a chunk of kC tokens with log decays lg_t and cumulative sums L_t (from
// the chunk's start, so γ_t = exp(L_t) ≤ 1), the token loop above unrolls to
// (the WY form of the delta rule):
//   U = X·(V − diag(γ)·K·S) = Ũ − W·S   (kC × 128, per value column),
//       X = (I + A)⁻¹·diag(β),   A_ti = β_t·exp(L_t − L_i)·k_t·k_i (i < t),
//       Ũ = X·V,   W = X·diag(γ)·K
//   O = (diag(γ)·Q·S + M·U) / sqrt(d),  M_ti = exp(L_t − L_i)·q_t·k_i (i ≤ t)
//   S ← γ_C·S + Kᵀ·diag(exp(L_C − L_t))·U
// where S is the state at the chunk's start.  Padding tokens past the batch
// have lg = 0, β = 0 and zero k, q, v, and change nothing.  Two kernels:
// k_dn_prep builds Ũ, W, M and the decays of every (value head, chunk) in
// parallel (K·Kᵀ, Q·Kᵀ and X's products on the fp32 matrix cores; X by forward
// substitution, a column a lane), and k_dn_chunks walks the chunks of a head in
// order with 16 of the state's value columns in registers, every product on
// the fp32 matrix cores (v_mfma_f32_16x16x4_f32).  The algebra is exact; the
// keys are unit vectors (the conv's l2 norm), so A's entries are at most 1 in
// size and the substitution is well conditioned.
//
// What bounds the second is the chain from chunk to chunk: two products a
// chunk that need all of the one before (W·S over every key, Kᵀ·U over every
// token), 32 MFMAs a wave each, and an exchange through LDS after either; with
// the two products of O that is 110 MFMAs a wave, 3.0 us where a CU holds two
// blocks.  At 1023 tokens of 16/48 heads it measured 5.0 us a chunk (80 us).
// With X alone prepared (U = X·(V − γ·K·S), K·S and Q·S summed over the waves'
// keys through LDS) there were three exchanges and 8.2 us a chunk (132 us);
// with two exchanges, but row-major matrices and loads behind branches (waits
// for all of them at once), 7.6.  k_dn_prep is bound by its chain of phases
// (load, K·Kᵀ, the substitution's 64 steps, X's products): 40 us there with a
// block a value head, three a CU; with a block a key head, so one a CU, 44
// for X and M alone and 100 with W and Ũ.
constexpr int kC = 64;
constexpr int kLdA = kC + 4, kLdK = kD + 4;  // LDS rows of A (or X) and K: 16-byte aligned, columns in distinct banks

// What the first kernel leaves for the second, but for the decays in
// "fragments": the 16×16 tile (i, j) of a matrix of J tiles a row is 64 × 16
// bytes at (i·J + j)·256 floats, lane (kq, r)'s four values together, so that a
// wave's load or store of a fragment is 1 KB in one piece.
struct Chunks {
    float *W;    // [n_v][chunks]: −W, tiles of (tokens, keys): token r, keys 4kq..
    float *U;    // [n_v][chunks]: Ũ, tiles of (tokens, values): tokens 4kq.., value r
    float *M;    // [n_v][chunks]: tiles of (tokens t, tokens i): t = r, i = 4kq..
    float *dec;  // [n_v][chunks][2][kC]: γ_t = exp(L_t), then exp(L_C − L_t)
    float *KT;   // [n_k][chunks]: tiles of (keys, tokens): key r, tokens 4kq..
    float *Q;    // [n_k][chunks]: tiles of (tokens, keys): token r, keys 4kq..
};
constexpr size_t kRunTokens = 4096;  // tokens a pair of launches: 320 MB of the matrices at 16/48 heads
constexpr size_t kWide = (size_t)kC * kD, kSquare = (size_t)kC * kC;  // floats of a chunk's matrices

__host__ Chunks chunks_of(float *work, size_t nch, size_t n_k, size_t n_v) {
    Chunks c;
    c.W = work;
    c.U = c.W + n_v * nch * kWide;
    c.M = c.U + n_v * nch * kWide;
    c.dec = c.M + n_v * nch * kSquare;
    c.KT = c.dec + n_v * nch * 2 * kC;
    c.Q = c.KT + n_k * nch * kWide;
    return c;
}

DEV v4f mfma4(float a, float b, v4f c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// grid (chunks, value heads), 256 threads.
__global__ void __launch_bounds__(256, 3) k_dn_prep(const float *__restrict__ q, const float *__restrict__ k,
                                                 const float *__restrict__ v, const float *__restrict__ gates,
                                                 const float *__restrict__ decay, const Chunks out, size_t n, int n_k,
                                                 int n_v) {
    __shared__ double Ls[kC];        // cumulative log decays
    __shared__ float bs[kC], gs[kC];  // β, γ
    __shared__ __attribute__((aligned(16))) float A[kC][kLdA];  // Aᵀ, then X
    __shared__ __attribute__((aligned(16))) float Ks[kC][kLdK];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, r = lane & 15, kq = lane >> 4;
    const size_t ch = blockIdx.x, nch = gridDim.x, t0 = ch * kC;
    const int h = blockIdx.y, ratio = n_v / n_k, kh = h / ratio;
    const size_t stride = (size_t)n_k * kD, vstride = (size_t)n_v * kD, at = (size_t)h * nch + ch;
    v4f kl[8];  // K's rows 8i + threadIdx.x / 32
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const size_t t = t0 + 8 * i + threadIdx.x / 32;
        kl[i] = *(const v4f *)(k + (t < n ? t : 0) * stride + kh * kD + threadIdx.x % 32 * 4);
    }
    // the decays: g_t = exp(lg_t), lg_t = a·softplus(alpha + dt_bias), beta_t =
    // sigmoid(beta logit); L_t = Σ lg up to t, in double: differences of sums
    // of up to 64 terms are taken below
    if (w == 0) {
        const size_t t = t0 + lane;
        float lg = 0.0f, beta = 0.0f;
        if (t < n) {
            lg = decay[h] * softplusf_(gates[t * 2 * n_v + h] + decay[n_v + h]);
            beta = sigmoidf_(gates[t * 2 * n_v + n_v + h]);
        }
        double L = lg;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const double u = __shfl_up(L, o, 64);
            if (lane >= o) L += u;
        }
        const double LC = __shfl(L, 63, 64);
        const float gamma = expf((float)L);
        out.dec[at * 2 * kC + lane] = gamma;
        out.dec[at * 2 * kC + kC + lane] = expf((float)(LC - L));
        Ls[lane] = L;
        bs[lane] = beta;
        gs[lane] = gamma;
    }
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const int t = 8 * i + threadIdx.x / 32;
        *(v4f *)&Ks[t][threadIdx.x % 32 * 4] = t0 + t < n ? kl[i] : v4f{0.0f, 0.0f, 0.0f, 0.0f};
    }
    __syncthreads();
    // Aᵀ (A_ti at row i, column t): the ten tiles on and above the diagonal;
    // lane (kq, r) feeds A[r][kq] and B[kq][r] with keys 4kq + j of each 16.
    // L falls with t, so each decay here and below is exp of a value ≤ 0
    for (int job = w; job < 10; job += 4) {
        int ti = job, tj = 0;
        while (ti > tj) ti -= ++tj;
        v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int m = 0; m < 8; m++) {
            const v4f a = *(const v4f *)&Ks[16 * ti + r][16 * m + 4 * kq];
            const v4f b = *(const v4f *)&Ks[16 * tj + r][16 * m + 4 * kq];
            acc = mfma4(a.x, b.x, acc);
            acc = mfma4(a.y, b.y, acc);
            acc = mfma4(a.z, b.z, acc);
            acc = mfma4(a.w, b.w, acc);
        }
        const int t = 16 * tj + r;
        const double L = Ls[t];
        const float beta = bs[t];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int i = 16 * ti + 4 * kq + j;
            const float e = expf((float)(t > i ? L - Ls[i] : 0.0));
            A[i][t] = t > i ? beta * e * acc[j] : 0.0f;
        }
    }
    __syncthreads();
    // one wave solves for X, the others prepare the rest meanwhile (which one
    // goes by the block, so that a CU's solvers are on different SIMDs)
    const int solver = (int)((ch + h) & 3);
    if (w == solver) {
        // (I + A)·X = diag(β), right-looking: once row i of X is known, its
        // terms join every later row's sum; lane j holds column j
        float acc[kC];
#pragma unroll
        for (int t = 0; t < kC; t++) acc[t] = 0.0f;
#pragma unroll
        for (int i = 0; i < kC; i++) {
            const float xi = (i == lane ? bs[i] : 0.0f) - acc[i];
#pragma unroll
            for (int t = (i + 4) & ~3; t < kC; t += 4) {
                const v4f a = *(const v4f *)&A[i][t];
                acc[t] += a.x * xi;
                acc[t + 1] += a.y * xi;
                acc[t + 2] += a.z * xi;
                acc[t + 3] += a.w * xi;
            }
#pragma unroll
            for (int t = i + 1; t < ((i + 4) & ~3); t++) acc[t] += A[i][t] * xi;
            acc[i] = xi;
            // the sums are brought up to date row by row (left to itself the
            // compiler defers them and keeps all of A in registers)
#pragma unroll
            for (int t = i + 1; t < kC; t++) asm volatile("" : "+v"(acc[t]));
        }
#pragma unroll
        for (int i = 0; i < kC; i++) A[i][lane] = acc[i];
    } else {
        const int part = (w - solver - 1) & 3;  // 0..2
        // M_ti = exp(L_t − L_i)·q_t·k_i for i ≤ t, taken as K·Qᵀ (rows i,
        // columns t); the tiles of i past t's are never read
        for (int job = part; job < 10; job += 3) {
            int ti = job, tt = 0;
            while (ti > tt) ti -= ++tt;
            const size_t tq = t0 + 16 * tt + r;
            const float *pq = q + (tq < n ? tq : 0) * stride + kh * kD + 4 * kq;
            v4f y[8];
#pragma unroll
            for (int m = 0; m < 8; m++) y[m] = *(const v4f *)(pq + 16 * m);
            v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
            const bool keep = ti == 0 && h % ratio == 0;  // Q's fragments, once a key head
#pragma unroll
            for (int m = 0; m < 8; m++) {
                const v4f a = *(const v4f *)&Ks[16 * ti + r][16 * m + 4 * kq];
                const v4f b = tq < n ? y[m] : v4f{0.0f, 0.0f, 0.0f, 0.0f};
                if (keep) *(v4f *)(out.Q + ((size_t)kh * nch + ch) * kWide + ((tt * 8 + m) * 64 + lane) * 4) = b;
                acc = mfma4(a.x, b.x, acc);
                acc = mfma4(a.y, b.y, acc);
                acc = mfma4(a.z, b.z, acc);
                acc = mfma4(a.w, b.w, acc);
            }
            const int t = 16 * tt + r;
            const double L = Ls[t];
            v4f mv;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int i = 16 * ti + 4 * kq + j;
                const float e = expf((float)(t >= i ? L - Ls[i] : 0.0));
                mv[j] = t >= i ? e * acc[j] : 0.0f;
            }
            *(v4f *)(out.M + at * kSquare + ((tt * 4 + ti) * 64 + lane) * 4) = mv;
        }
        // Kᵀ's fragments
        if (h % ratio == 0)
            for (int job = part; job < 32; job += 3) {
                const int kt = job / 4, ut = job % 4;
                v4f x;
#pragma unroll
                for (int j = 0; j < 4; j++) x[j] = Ks[16 * ut + 4 * kq + j][16 * kt + r];
                *(v4f *)(out.KT + ((size_t)kh * nch + ch) * kWide + (job * 64 + lane) * 4) = x;
            }
    }
    // −W = −X·diag(γ)·K and Ũ = X·V, 16 columns of either at a time: wave w's are
    // 16w.. and 64 + 16w..; a lane's 16 values of their 64 rows (V's loaded
    // ahead), X (lower triangular) from LDS.  W's fragments hold a token a
    // lane, Ũ's a value: W is taken transposed.
    float b[2][4][4];
#pragma unroll
    for (int g = 0; g < 2; g++)
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const size_t t = t0 + 16 * (i / 4) + 4 * kq + i % 4;
            b[g][i / 4][i % 4] = v[(t < n ? t : 0) * vstride + h * kD + 64 * g + 16 * w + r];
        }
    __syncthreads();
#pragma unroll
    for (int job = 0; job < 4; job++) {
        const int g = job & 1, m = 4 * g + w;
        const bool values = job >= 2;
        v4f acc[4][2];  // (two chains: half the roundings of one)
#pragma unroll
        for (int ti = 0; ti < 4; ti++) acc[ti][0] = acc[ti][1] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int ui = 0; ui < 4; ui++) {
            v4f x;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int i = 16 * ui + 4 * kq + j;
                x[j] = values ? (t0 + i < n ? b[g][ui][j] : 0.0f) : -gs[i] * Ks[i][16 * m + r];
            }
#pragma unroll
            for (int ti = ui; ti < 4; ti++) {
                const v4f a = *(const v4f *)&A[16 * ti + r][16 * ui + 4 * kq];
#pragma unroll
                for (int j = 0; j < 4; j++)
                    acc[ti][j & 1] = values ? mfma4(a[j], x[j], acc[ti][j & 1]) : mfma4(x[j], a[j], acc[ti][j & 1]);
            }
        }
        float *o = (values ? out.U : out.W) + at * kWide + lane * 4;
#pragma unroll
        for (int ti = 0; ti < 4; ti++) *(v4f *)(o + (ti * 8 + m) * 256) = acc[ti][0] + acc[ti][1];
    }
}

// grid: 8 column blocks × n_v heads (all the blocks of a key head on one XCD
// when n_k is a multiple of 8), 256 threads.  Wave w owns keys 32w..32w+31 of
// the block's 16 columns of the state (two 16×16 accumulator tiles) and the
// chunk's tokens 16w..16w+15; the state and U go through LDS as the MFMA's
// accumulators hold them (lane (kq, r): rows 4kq.. of column r, 16 bytes), which
// is also how its B operand takes them.
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) k_dn_chunks(
    float *__restrict__ out, const Chunks in, float *__restrict__ state, size_t n, int n_k, int n_v) {
    __shared__ v4f Ss[8][4][16], Us[4][4][16], Ud[4][4][16];  // [16 rows][kq][column]
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, r = lane & 15, kq = lane >> 4;
    const int ratio = n_v / n_k;
    const unsigned b = blockIdx.x;
    int h, cb;
    if (n_k % 8 == 0) {
        const unsigned idx = b / 8, per = (unsigned)(ratio * 8);
        const int kh = (int)(b % 8) * (n_k / 8) + (int)(idx / per);
        h = kh * ratio + (int)((idx % per) / 8);
        cb = (int)(idx % 8);
    } else {
        h = (int)(b / 8);
        cb = (int)(b % 8);
    }
    const int kh = h / ratio, c0 = cb * kCols;
    const size_t vstride = (size_t)n_v * kD;
    float *S = state + (size_t)h * kD * kD;
    v4f s[2];
#pragma unroll
    for (int kt = 0; kt < 2; kt++)
#pragma unroll
        for (int i = 0; i < 4; i++) s[kt][i] = S[(32 * w + 16 * kt + 4 * kq + i) * kD + c0 + r];
    const size_t nch = (n + kC - 1) / kC;
    const float scale = 1.0f / sqrtf((float)kD);
    // every global load is issued a chunk ahead, right after the last use of
    // what it replaces (past the last chunk the last one's again, so that no
    // branch comes between a load and its wait): W, Q and M of tokens 16w..,
    // Kᵀ of the wave's keys
    const float *Wp = in.W + (size_t)h * nch * kWide + (w * 8 * 64 + lane) * 4;
    const float *Up = in.U + (size_t)h * nch * kWide + ((w * 8 + cb) * 64 + lane) * 4;
    const float *Qp = in.Q + (size_t)kh * nch * kWide + (w * 8 * 64 + lane) * 4;
    const float *Kp = in.KT + (size_t)kh * nch * kWide + (w * 8 * 64 + lane) * 4;
    const float *Mp = in.M + (size_t)h * nch * kSquare + (w * 4 * 64 + lane) * 4;
    const float *Dp = in.dec + (size_t)h * nch * 2 * kC;
    v4f wf[8], qf[8], mf[4], kf[2][4], uf, gg, ee, gn, en;
    float gC, gCn;
    auto fetch_w = [&](size_t ch) {
#pragma unroll
        for (int m = 0; m < 8; m++) wf[m] = *(const v4f *)(Wp + ch * kWide + m * 256);
        uf = *(const v4f *)(Up + ch * kWide);
    };
    auto fetch_q = [&](size_t ch) {
#pragma unroll
        for (int m = 0; m < 8; m++) qf[m] = *(const v4f *)(Qp + ch * kWide + m * 256);
    };
    auto fetch_k = [&](size_t ch) {
#pragma unroll
        for (int kt = 0; kt < 2; kt++)
#pragma unroll
            for (int t = 0; t < 4; t++) kf[kt][t] = *(const v4f *)(Kp + ch * kWide + (kt * 4 + t) * 256);
    };
    auto fetch_m = [&](size_t ch) {  // (tiles past the diagonal: the diagonal's again, unused)
#pragma unroll
        for (int t = 0; t < 4; t++) mf[t] = *(const v4f *)(Mp + ch * kSquare + (t < w ? t : w) * 256);
    };
    auto fetch_decay = [&](size_t ch) {
        const float *d = Dp + ch * 2 * kC;
        gn = *(const v4f *)(d + 16 * w + 4 * kq);
        en = *(const v4f *)(d + kC + 16 * w + 4 * kq);
        gCn = d[kC - 1];
    };
    fetch_decay(0);
    fetch_w(0);
    fetch_q(0);
    fetch_k(0);
    fetch_m(0);
#pragma unroll
    for (int kt = 0; kt < 2; kt++) Ss[2 * w + kt][kq][r] = s[kt];
    __syncthreads();
    auto chunk = [&](size_t ch, bool whole) {
        const size_t next = ch + 1 < nch ? ch + 1 : ch;
        gg = gn;
        ee = en;
        gC = gCn;
        fetch_decay(next);
        v4f sf[8];
#pragma unroll
        for (int m = 0; m < 8; m++) sf[m] = Ss[m][kq][r];
        // U = Ũ − W·S of this wave's tokens (four chains; Ũ, like S and O's first
        // term below, joins at the end: a chain rounds at its own size)
        v4f u[4];
#pragma unroll
        for (int j = 0; j < 4; j++) u[j] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int m = 0; m < 8; m++) {
            u[0] = mfma4(wf[m].x, sf[m].x, u[0]);
            u[1] = mfma4(wf[m].y, sf[m].y, u[1]);
            u[2] = mfma4(wf[m].z, sf[m].z, u[2]);
            u[3] = mfma4(wf[m].w, sf[m].w, u[3]);
        }
        const v4f ut = uf + ((u[0] + u[1]) + (u[2] + u[3]));
        Us[w][kq][r] = ut;
        Ud[w][kq][r] = v4f{ut[0] * ee[0], ut[1] * ee[1], ut[2] * ee[2], ut[3] * ee[3]};
        fetch_w(next);
        // O starts as γ·Q·S
        v4f o[2] = {v4f{0.0f, 0.0f, 0.0f, 0.0f}, v4f{0.0f, 0.0f, 0.0f, 0.0f}};
#pragma unroll
        for (int m = 0; m < 8; m++) {
            o[0] = mfma4(qf[m].x, sf[m].x, o[0]);
            o[1] = mfma4(qf[m].y, sf[m].y, o[1]);
            o[0] = mfma4(qf[m].z, sf[m].z, o[0]);
            o[1] = mfma4(qf[m].w, sf[m].w, o[1]);
        }
        v4f ot = o[0] + o[1];
#pragma unroll
        for (int i = 0; i < 4; i++) ot[i] *= gg[i];
        fetch_q(next);
        __syncthreads();
        // S = γ_C·S + Kᵀ·diag(exp(L_C − L_t))·U of this wave's keys
        v4f d[2][2];
#pragma unroll
        for (int kt = 0; kt < 2; kt++) d[kt][0] = d[kt][1] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const v4f x = Ud[t][kq][r];
#pragma unroll
            for (int kt = 0; kt < 2; kt++) {
                d[kt][0] = mfma4(kf[kt][t].x, x.x, d[kt][0]);
                d[kt][1] = mfma4(kf[kt][t].y, x.y, d[kt][1]);
                d[kt][0] = mfma4(kf[kt][t].z, x.z, d[kt][0]);
                d[kt][1] = mfma4(kf[kt][t].w, x.w, d[kt][1]);
            }
        }
#pragma unroll
        for (int kt = 0; kt < 2; kt++) {
            s[kt] = s[kt] * gC + (d[kt][0] + d[kt][1]);
            Ss[2 * w + kt][kq][r] = s[kt];
        }
        fetch_k(next);
        // O += M·U, M lower triangular
        o[0] = o[1] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int t = 0; t < 4; t++) {
            if (t > w) break;
            const v4f x = Us[t][kq][r];
            o[0] = mfma4(mf[t].x, x.x, o[0]);
            o[1] = mfma4(mf[t].y, x.y, o[1]);
            o[0] = mfma4(mf[t].z, x.z, o[0]);
            o[1] = mfma4(mf[t].w, x.w, o[1]);
        }
        ot += o[0] + o[1];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const size_t t = ch * kC + 16 * w + 4 * kq + i;
            if (whole || t < n) out[t * vstride + h * kD + c0 + r] = ot[i] * scale;
        }
        fetch_m(next);
        __syncthreads();
    };
    const size_t whole = n / kC;
    for (size_t ch = 0; ch < whole; ch++) chunk(ch, true);
    if (whole < nch) chunk(whole, false);
#pragma unroll
    for (int kt = 0; kt < 2; kt++)
#pragma unroll
        for (int i = 0; i < 4; i++) S[(32 * w + 16 * kt + 4 * kq + i) * kD + c0 + r] = s[kt][i];
}

}  // namespace

// The chunked form's per-chunk matrices (W, Ũ, M, the decays and Kᵀ) for n tokens.
size_t delta_net_work_floats(size_t n, size_t n_k_heads, size_t n_v_heads) {
    if (n < (size_t)kC) return 0;
    const size_t nch = (std::min(n, kRunTokens) + kC - 1) / kC;
    return nch * (n_v_heads * (2 * kWide + kSquare + 2 * kC) + n_k_heads * 2 * kWide);
}

hipError_t delta_net_reserve(dwim_dev *dev, size_t n, size_t n_k_heads, size_t n_v_heads) {
    return dev_grow(dev, (void **)&dev->dn_work, &dev->dn_work_cap, delta_net_work_floats(n, n_k_heads, n_v_heads),
                    sizeof(float));
}

hipError_t launch_gdn_tokens(dwim_dev *dev, float *out, const float *qkv, const float *conv_state,
                             float *conv_state_out, const float *conv_w, const float *gates, const float *decay,
                             float *state, const float *state_in, size_t n, size_t n_k_heads, size_t n_v_heads,
                             size_t head_dim, float eps, const GdnSteps *steps, const GdnGate *gate) {
    if (head_dim != kD || n < 1 || n > (size_t)kSmallT || n_k_heads == 0 || n_v_heads % n_k_heads)
        return hipErrorInvalidValue;
    if (gate && (n > 4 || !gate->z || !gate->norm_w || !gate->planes || !gate->head_ss ||
                 n_v_heads * kD > planes::kMaxCols || (n_v_heads * kD) % 256))
        return hipErrorInvalidValue;
    dim3 grid(kD / kCols, (unsigned)n_v_heads);
    k_gdn_tokens<<<grid, kThreads, 0, dev->stream>>>(out, qkv, conv_state, conv_state_out, conv_w, gates, decay, state,
                                                     state_in ? state_in : state, (int)n, (int)n_k_heads,
                                                     (int)n_v_heads, eps, steps ? *steps : GdnSteps{},
                                                     gate ? *gate : GdnGate{});
    return hipGetLastError();
}

hipError_t launch_delta_net(dwim_dev *dev, float *out, const float *q, const float *k, const float *v,
                            const float *gates, const float *decay, float *state, size_t n, size_t n_k_heads,
                            size_t n_v_heads, size_t head_dim, const Rms *rms, bool unit_keys, const float *state_in) {
    if (head_dim != (size_t)kD || n_k_heads == 0 || n_v_heads % n_k_heads) return hipErrorInvalidValue;
    if (unit_keys && n >= (size_t)kC && !(rms && rms->ss)) {
        if (state_in && state_in != state) return hipErrorInvalidValue;  // (the token loop reads one state, writes another)
        hipError_t e = delta_net_reserve(dev, n, n_k_heads, n_v_heads);
        if (e != hipSuccess) return e;
        const int nk = (int)n_k_heads, nv = (int)n_v_heads;
        for (size_t t = 0; t < n; t += kRunTokens) {
            const size_t m = std::min(kRunTokens, n - t), nch = (m + kC - 1) / kC, kt = t * n_k_heads * kD, vt = t * n_v_heads * kD;
            const Chunks c = chunks_of(dev->dn_work, nch, n_k_heads, n_v_heads);
            k_dn_prep<<<dim3((unsigned)nch, (unsigned)n_v_heads), 256, 0, dev->stream>>>(
                q + kt, k + kt, v + vt, gates + t * 2 * n_v_heads, decay, c, m, nk, nv);
            k_dn_chunks<<<(unsigned)(8 * n_v_heads), 256, 0, dev->stream>>>(out + vt, c, state, m, nk, nv);
        }
        return hipGetLastError();
    }
    dim3 grid(kD / kCols, (unsigned)n_v_heads);
    k_delta_net<<<grid, kThreads, 0, dev->stream>>>(out, q, k, v, gates, decay, state, state_in ? state_in : state, n,
                                                    (int)n_k_heads,
                                                    (int)n_v_heads, rms ? *rms : Rms{});
    return hipGetLastError();
}
