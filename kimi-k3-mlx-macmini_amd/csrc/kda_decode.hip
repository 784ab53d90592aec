// Kimi Delta Attention recurrent step for one token: the state update and read-out of
// every value head, in place on the fp32 state.
//
// Reference: KDAAttention._recurrent (air_llm/models/kimi_k3/attention_kda.py:65-90), the
// upstream naive_recurrent_kda (k3ref/_vendor/kda_naive.py:46-60):
//   S = S * exp(g)[:, None];  S = S + (beta k) (x) (v - k . S);  o = (scale q) . S
// with S [K, V] per value head, g the per-key-channel log decay.
//
// The state is the whole cost: 96 heads x 128 x 128 fp32 = 6 MiB read and written per
// token.  A block owns 32 value columns of one head, so every column's reduction over the
// 128 key channels stays inside the block and the state is read and written exactly once:
// thread t holds rows r, r + 32, r + 64, r + 96 (r = t / 8) of columns 4 (t % 8) .. +3, so
// eight lanes read one 128-byte row segment.  The two reductions over the key channels
// (k . S' for the delta, q . S'' for the read-out) run as xor shuffles inside a wave, then
// across the four waves through LDS in a fixed order.
#include "dense_rows.h"

namespace k3 {
namespace {

constexpr int kKdaK = 128;   // key channels (state rows) per head
constexpr int kKdaVS = 32;   // value columns per block

struct KdaArgs {
    const void *q, *k;        // [T, HQ, K]
    const void *v;            // [T, HV, V]
    const void *g;            // [T, HV, K] log decay
    const void *beta;         // [T, HV]
    int in_bf16;              // q, k, v, g, beta: bf16 (1) or fp32 (0)
    float *S;                 // [HV, K, V] fp32, updated in place
    void *out;                // [T, HV, V]
    int out_bf16;
    int vec;                  // q, k, g are 16-byte aligned and out holds aligned pairs (many tokens)
    int HV, G, V, T;          // G = HV / HQ value heads per q/k head
    float scale;
};

__device__ __forceinline__ float ldx(const void *p, int64_t i, int bf) {
    return bf ? bf16_to_f32(static_cast<const uint16_t *>(p)[i]) : static_cast<const float *>(p)[i];
}

// sum over the 8 lanes of a wave that share lane % 8 (the wave's 8 row groups)
__device__ __forceinline__ float sum_row_groups(float x) {
    x += __shfl_xor(x, 8);
    x += __shfl_xor(x, 16);
    x += __shfl_xor(x, 32);
    return x;
}

// The update of one block's 32 columns of head h's state, given this thread's four rows'
// key values kk, scaled query values qq and decay factors dk, its four columns' values vv
// and the head's beta.  x holds the thread's state values (loaded by the caller, stored by
// the caller once its tokens are done).
// Returns the read-out of column t (valid in threads t < 32).
__device__ __forceinline__ float kda_apply(float4 (&x)[4], const float (&kk)[4],
                                           const float (&qq)[4], const float (&dk)[4], const float (&vv)[4], float b,
                                           float (*red)[4][kKdaVS]) {
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6, cg = t & 7;
    // decay, then k . S' over the 128 channels
#pragma unroll
    for (int j = 0; j < 4; ++j) x[j].x *= dk[j], x[j].y *= dk[j], x[j].z *= dk[j], x[j].w *= dk[j];
    float p[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        p[0] = fmaf(kk[j], x[j].x, p[0]);
        p[1] = fmaf(kk[j], x[j].y, p[1]);
        p[2] = fmaf(kk[j], x[j].z, p[2]);
        p[3] = fmaf(kk[j], x[j].w, p[3]);
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) p[c] = sum_row_groups(p[c]);
    if (lane < 8) {
#pragma unroll
        for (int c = 0; c < 4; ++c) red[0][wave][4 * lane + c] = p[c];
    }
    __syncthreads();
    float d[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const int i = 4 * cg + c;
        d[c] = vv[c] - (((red[0][0][i] + red[0][1][i]) + red[0][2][i]) + red[0][3][i]);
    }
    // the delta update, written back; then q . S''
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const float bk = b * kk[j];
        x[j].x = fmaf(bk, d[0], x[j].x);
        x[j].y = fmaf(bk, d[1], x[j].y);
        x[j].z = fmaf(bk, d[2], x[j].z);
        x[j].w = fmaf(bk, d[3], x[j].w);
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) p[c] = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        p[0] = fmaf(qq[j], x[j].x, p[0]);
        p[1] = fmaf(qq[j], x[j].y, p[1]);
        p[2] = fmaf(qq[j], x[j].z, p[2]);
        p[3] = fmaf(qq[j], x[j].w, p[3]);
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) p[c] = sum_row_groups(p[c]);
    if (lane < 8) {
#pragma unroll
        for (int c = 0; c < 4; ++c) red[1][wave][4 * lane + c] = p[c];
    }
    __syncthreads();
    return t < kKdaVS ? ((red[1][0][t] + red[1][1][t]) + red[1][2][t]) + red[1][3][t] : 0.f;
}

__device__ __forceinline__ void kda_store_state(const float4 (&x)[4], float *const (&Sp)[4]) {
#pragma unroll
    for (int j = 0; j < 4; ++j) *reinterpret_cast<float4 *>(Sp[j]) = x[j];
}

// the four state rows t/8 + 32j of columns c0 .. c0+3 of head h
__device__ __forceinline__ void kda_load_state(float *S, int h, int V, int c0, float4 (&x)[4], float *(&Sp)[4]) {
    const int r = threadIdx.x >> 3;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        Sp[j] = S + (static_cast<int64_t>(h) * kKdaK + r + 32 * j) * V + c0;
        x[j] = *reinterpret_cast<const float4 *>(Sp[j]);
    }
}

// One token.
__global__ __launch_bounds__(256) void kda_decode_kernel(KdaArgs a) {
    __shared__ float red[2][4][kKdaVS];
    const int nvb = a.V / kKdaVS;
    const int h = blockIdx.x / nvb, vb = blockIdx.x % nvb;
    const int hq = h / a.G;
    const int t = threadIdx.x, cg = t & 7, r = t >> 3;
    const int c0 = vb * kKdaVS + 4 * cg;
    const int bf = a.in_bf16;
    float *Sp[4];
    float4 x[4];
    kda_load_state(a.S, h, a.V, c0, x, Sp);
    float kk[4], qq[4], dk[4], vv[4];
    const int64_t qo = static_cast<int64_t>(hq) * kKdaK, go = static_cast<int64_t>(h) * kKdaK;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        kk[j] = ldx(a.k, qo + r + 32 * j, bf);
        qq[j] = ldx(a.q, qo + r + 32 * j, bf) * a.scale;
        dk[j] = expf(ldx(a.g, go + r + 32 * j, bf));
    }
    const int64_t vo = static_cast<int64_t>(h) * a.V + c0;
#pragma unroll
    for (int c = 0; c < 4; ++c) vv[c] = ldx(a.v, vo + c, bf);
    const float o = kda_apply(x, kk, qq, dk, vv, ldx(a.beta, h, bf), red);
    if (t < kKdaVS) {
        const int64_t oi = static_cast<int64_t>(h) * a.V + vb * kKdaVS + t;
        if (a.out_bf16)
            static_cast<uint16_t *>(a.out)[oi] = f32_to_bf16(o);
        else
            static_cast<float *>(a.out)[oi] = o;
    }
    kda_store_state(x, Sp);
}

// Many tokens, in order.  The tokens are a serial chain, so what bounds the launch is the
// length of one token's step; the state stays in registers throughout.  A wave owns 8 value
// columns: lane (rg, cp) holds rows 4 rg .. + 3 and 64 + 4 rg .. + 3 of columns 2 cp, 2 cp + 1,
// so a column's reduction over the 128 key channels is 8 terms in a lane and four DPP steps
// inside a 16-lane row, with no LDS round trip and no barrier.  Both reductions run on the
// decayed state at once, since
//   q . (S' + (beta k) (x) d) = q . S' + (q . k) (beta d),  d = v - k . S'
// and q . k needs no state.  The inputs of 16 tokens at a time (scaled q, k, exp(g), v, beta,
// q . k) are staged in LDS, double buffered, one barrier per 16 tokens, and each token's are
// read one token ahead.
// 256 tokens, 96 heads of 128 x 128: 470 us with two barriers and two LDS reductions per
// token, 110 us now (0.43 us per token: about 100 VALU operations of the two waves a SIMD
// holds; 384 blocks leave half the CUs one wave per SIMD).  A branch per token around the
// output's store: 131 us.
constexpr int kKdaChunk = 16;

__device__ __forceinline__ float row16_sum(float v) {  // sum over the 16 lanes of a DPP row, in all of them
    v += dpp_or_zero<0xb1>(v);
    v += dpp_or_zero<0x4e>(v);
    v += dpp_or_zero<0x141>(v);
    v += dpp_or_zero<0x140>(v);
    return v;
}

// four of them side by side, so no step waits for the one before it
__device__ __forceinline__ void row16_sum4(float &a, float &b, float &c, float &d) {
    a += dpp_or_zero<0xb1>(a), b += dpp_or_zero<0xb1>(b), c += dpp_or_zero<0xb1>(c), d += dpp_or_zero<0xb1>(d);
    a += dpp_or_zero<0x4e>(a), b += dpp_or_zero<0x4e>(b), c += dpp_or_zero<0x4e>(c), d += dpp_or_zero<0x4e>(d);
    a += dpp_or_zero<0x141>(a), b += dpp_or_zero<0x141>(b), c += dpp_or_zero<0x141>(c), d += dpp_or_zero<0x141>(d);
    a += dpp_or_zero<0x140>(a), b += dpp_or_zero<0x140>(b), c += dpp_or_zero<0x140>(c), d += dpp_or_zero<0x140>(d);
}

__global__ __launch_bounds__(256) void kda_sequence_kernel(KdaArgs a) {
    __shared__ float4 in[2][kKdaChunk][3][kKdaK / 4];  // k, q, decay
    __shared__ float2 vs[2][kKdaChunk][kKdaVS / 2];
    __shared__ float2 bq[2][kKdaChunk];                // beta, q . k
    const int nvb = a.V / kKdaVS;
    const int h = blockIdx.x / nvb, vb = blockIdx.x % nvb;
    const int hq = h / a.G, HQ = a.HV / a.G;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, rg = lane & 15, cp = lane >> 4;
    const int col = vb * kKdaVS + wave * 8 + 2 * cp;
    const int bf = a.in_bf16;
    float S[8][2];
    float *Sp = a.S + (static_cast<int64_t>(h) * kKdaK + 4 * rg) * a.V + col;
#pragma unroll
    for (int r = 0; r < 8; ++r) {
        const float2 v = *reinterpret_cast<const float2 *>(Sp + static_cast<int64_t>((r >> 2) * 64 + (r & 3)) * a.V);
        S[r][0] = v.x, S[r][1] = v.y;
    }
    // staging: thread (token tid / 16, channels 8 (tid % 16) .. + 7)
    const int st = tid >> 4, sp = tid & 15;
    float k8[8], q8[8], g8[8], v2[2], sb;
    auto load8 = [&](const void *p, int64_t i, float (&o)[8]) {
        if (!a.vec) {
#pragma unroll
            for (int x = 0; x < 8; ++x) o[x] = ldx(p, i + x, bf);
        } else if (bf) {
            const uint4 u = *reinterpret_cast<const uint4 *>(static_cast<const uint16_t *>(p) + i);
            const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
            for (int x = 0; x < 4; ++x) o[2 * x] = __uint_as_float(w[x] << 16), o[2 * x + 1] = __uint_as_float(w[x] & 0xffff0000u);
        } else {
            const float4 *f = reinterpret_cast<const float4 *>(static_cast<const float *>(p) + i);
            const float4 x = f[0], y = f[1];
            o[0] = x.x, o[1] = x.y, o[2] = x.z, o[3] = x.w, o[4] = y.x, o[5] = y.y, o[6] = y.z, o[7] = y.w;
        }
    };
    auto load = [&](int i0) {
        const int64_t i = min(i0 + st, a.T - 1);  // past the end: the last token, not used
        load8(a.k, (i * HQ + hq) * kKdaK + 8 * sp, k8);
        load8(a.q, (i * HQ + hq) * kKdaK + 8 * sp, q8);
        load8(a.g, (i * a.HV + h) * kKdaK + 8 * sp, g8);
        const int64_t vo = (i * a.HV + h) * a.V + vb * kKdaVS + 2 * sp;
        v2[0] = ldx(a.v, vo, bf), v2[1] = ldx(a.v, vo + 1, bf);
        sb = ldx(a.beta, i * a.HV + h, bf);
    };
    auto store = [&](int buf) {
        float dot = 0.f;
#pragma unroll
        for (int x = 0; x < 8; ++x) {
            q8[x] *= a.scale;
            dot = fmaf(q8[x], k8[x], dot);
            g8[x] = expf(g8[x]);
        }
        dot = row16_sum(dot);
#pragma unroll
        for (int x = 0; x < 2; ++x) {
            in[buf][st][0][2 * sp + x] = make_float4(k8[4 * x], k8[4 * x + 1], k8[4 * x + 2], k8[4 * x + 3]);
            in[buf][st][1][2 * sp + x] = make_float4(q8[4 * x], q8[4 * x + 1], q8[4 * x + 2], q8[4 * x + 3]);
            in[buf][st][2][2 * sp + x] = make_float4(g8[4 * x], g8[4 * x + 1], g8[4 * x + 2], g8[4 * x + 3]);
        }
        vs[buf][st][sp] = make_float2(v2[0], v2[1]);
        if (sp == 0) bq[buf][st] = make_float2(sb, dot);
    };
    struct Token {
        float4 k[2], q[2], d[2];
        float2 v, bq;
    };
    auto read = [&](int buf, int i, Token &t) {
#pragma unroll
        for (int x = 0; x < 2; ++x) t.k[x] = in[buf][i][0][rg + 16 * x], t.q[x] = in[buf][i][1][rg + 16 * x], t.d[x] = in[buf][i][2][rg + 16 * x];
        t.v = vs[buf][i][wave * 4 + cp];
        t.bq = bq[buf][i];
    };
    load(0);
    store(0);
    __syncthreads();
    for (int i0 = 0, buf = 0; i0 < a.T; i0 += kKdaChunk, buf ^= 1) {
        const int n = min(kKdaChunk, a.T - i0);
        const bool more = i0 + kKdaChunk < a.T;
        if (more) load(i0 + kKdaChunk);
        // one token: the state's step; lane rg == i of each row keeps the read-out
        float y[2] = {0.f, 0.f};
        auto token = [&](const Token &t, int i) {
            const float kk[8] = {t.k[0].x, t.k[0].y, t.k[0].z, t.k[0].w, t.k[1].x, t.k[1].y, t.k[1].z, t.k[1].w};
            const float qq[8] = {t.q[0].x, t.q[0].y, t.q[0].z, t.q[0].w, t.q[1].x, t.q[1].y, t.q[1].z, t.q[1].w};
            const float dd[8] = {t.d[0].x, t.d[0].y, t.d[0].z, t.d[0].w, t.d[1].x, t.d[1].y, t.d[1].z, t.d[1].w};
            float p[2] = {0.f, 0.f}, o[2] = {0.f, 0.f};
#pragma unroll
            for (int r = 0; r < 8; ++r)
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    S[r][c] *= dd[r];
                    p[c] = fmaf(kk[r], S[r][c], p[c]);
                    o[c] = fmaf(qq[r], S[r][c], o[c]);
                }
            row16_sum4(p[0], p[1], o[0], o[1]);
            const float d[2] = {t.bq.x * (t.v.x - p[0]), t.bq.x * (t.v.y - p[1])};
#pragma unroll
            for (int r = 0; r < 8; ++r)
#pragma unroll
                for (int c = 0; c < 2; ++c) S[r][c] = fmaf(kk[r], d[c], S[r][c]);
#pragma unroll
            for (int c = 0; c < 2; ++c) y[c] = rg == i ? fmaf(t.bq.y, d[c], o[c]) : y[c];
        };
        Token t0, t1;
        read(buf, 0, t0);
        for (int i = 0; i < n; i += 2) {
            read(buf, min(i + 1, n - 1), t1);
            token(t0, i);
            if (i + 1 >= n) break;
            read(buf, min(i + 2, n - 1), t0);
            token(t1, i + 1);
        }
        if (rg < n) {
            const int64_t oi = (static_cast<int64_t>(i0 + rg) * a.HV + h) * a.V + col;
            if (!a.vec) {
                for (int c = 0; c < 2; ++c) {
                    if (a.out_bf16)
                        static_cast<uint16_t *>(a.out)[oi + c] = f32_to_bf16(y[c]);
                    else
                        static_cast<float *>(a.out)[oi + c] = y[c];
                }
            } else if (a.out_bf16) {
                *reinterpret_cast<uint32_t *>(static_cast<uint16_t *>(a.out) + oi) =
                    f32_to_bf16(y[0]) | (static_cast<uint32_t>(f32_to_bf16(y[1])) << 16);
            } else {
                *reinterpret_cast<float2 *>(static_cast<float *>(a.out) + oi) = make_float2(y[0], y[1]);
            }
        }
        if (more) {
            store(buf ^ 1);
            __syncthreads();
        }
    }
#pragma unroll
    for (int r = 0; r < 8; ++r)
        *reinterpret_cast<float2 *>(Sp + static_cast<int64_t>((r >> 2) * 64 + (r & 3)) * a.V) = make_float2(S[r][0], S[r][1]);
}

// ------------------------------------------------------------------ around the recurrence, many tokens
// The recurrence's inputs of B sequences of T tokens from the projections (token-major rows
// b * T + t): short convolutions with SiLU, L2 norms of q and k, decay gate, beta, as
// kda_step_kernel builds them for one token.  A block takes one head and eight tokens.
// Outputs are time-major, [T, B, H, 128] and [T, B, H].
struct KdaPrepArgs {
    const float *raw[3];                     // q, k, v projections [B * T, P]
    const float *fb, *b_raw;                 // [B * T, P], [B * T, H]
    const float *conv[3];                    // [P, kc]
    const float *win[3];                     // [B, kc - 1, P], or null (zeros)
    float *win_out[3];                       // [B, kc - 1, P]
    const float *A_log, *dt_bias;
    float lower;
    float *q, *k, *v, *g, *beta;
    int B, T, H, kc;
};
constexpr int kPrepTokens = 8;

__global__ __launch_bounds__(128) void kda_prep_kernel(KdaPrepArgs a) {
    __shared__ float part[2][kPrepTokens][2];
    // blocks: head, then eight tokens, then sequence
    const int nt = (a.T + kPrepTokens - 1) / kPrepTokens, tile = blockIdx.x / a.H;
    const int c = threadIdx.x, h = blockIdx.x % a.H, t0 = tile % nt * kPrepTokens, b = tile / nt;
    const int P = a.H * kKdaK, ch = h * kKdaK + c, kc = a.kc, lane = c & 63, wave = c >> 6;
    const int64_t row0 = static_cast<int64_t>(b) * a.T;
    // input i of the padded sequence: the window, then the tokens
    auto xp = [&](int m, int i) -> float {  // (uniform choices; one load, unconditional but for a null window)
        const bool tok = i >= kc - 1;
        if (!tok && !a.win[m]) return 0.f;
        const float *p = tok ? a.raw[m] + (row0 + i - (kc - 1)) * P : a.win[m] + (static_cast<int64_t>(b) * (kc - 1) + i) * P;
        return p[ch];
    };
    float y[3][kPrepTokens];
#pragma unroll
    for (int m = 0; m < 3; ++m) {
        const float *cw = a.conv[m] + static_cast<int64_t>(ch) * kc;
        if (kc == 4) {
            float x[kPrepTokens + 3];
#pragma unroll
            for (int i = 0; i < kPrepTokens + 3; ++i) x[i] = xp(m, min(t0 + i, a.T + 2));
            const float w0 = cw[0], w1 = cw[1], w2 = cw[2], w3 = cw[3];
#pragma unroll
            for (int i = 0; i < kPrepTokens; ++i)
                y[m][i] = fmaf(w3, x[i + 3], fmaf(w2, x[i + 2], fmaf(w1, x[i + 1], w0 * x[i])));
        } else {
#pragma unroll
            for (int i = 0; i < kPrepTokens; ++i) {
                const int t = min(t0 + i, a.T - 1);
                float z = 0.f;
                for (int j = 0; j < kc; ++j) z = fmaf(cw[j], xp(m, t + j), z);
                y[m][i] = z;
            }
        }
#pragma unroll
        for (int i = 0; i < kPrepTokens; ++i) y[m][i] = y[m][i] / (1.0f + expf(-y[m][i]));
        if (t0 == 0)
            for (int j = 0; j < kc - 1; ++j) a.win_out[m][(static_cast<int64_t>(b) * (kc - 1) + j) * P + ch] = xp(m, a.T + j);
    }
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int i = 0; i < kPrepTokens; ++i) {
            const float s = wave_sum_all(y[m][i] * y[m][i]);
            if (lane == 0) part[m][i][wave] = s;
        }
    __syncthreads();
    const float ea = expf(a.A_log[h]), db = a.dt_bias[ch];
#pragma unroll
    for (int i = 0; i < kPrepTokens; ++i) {
        const int t = t0 + i;
        if (t < a.T) {
            const int64_t th = (static_cast<int64_t>(t) * a.B + b) * a.H + h, o = th * kKdaK + c;
            a.q[o] = y[0][i] / sqrtf(part[0][i][0] + part[0][i][1] + 1e-6f);
            a.k[o] = y[1][i] / sqrtf(part[1][i][0] + part[1][i][1] + 1e-6f);
            a.v[o] = y[2][i];
            const float z = ea * (a.fb[(row0 + t) * P + ch] + db);
            a.g[o] = a.lower / (1.0f + expf(-z));
            if (c == 0) a.beta[th] = 1.0f / (1.0f + expf(-a.b_raw[(row0 + t) * a.H + h]));
        }
    }
}

// out [B * T, P] = o * rsqrt(mean(o^2) + eps) * w * sigmoid(og): o time-major [T, B, H, 128], one
// wave per (token, head) (ops.py:36-39).
__global__ __launch_bounds__(256) void kda_gated_norm_kernel(const float *o, const float *og, const float *w, float eps,
                                                             float *out, int B, int T, int H) {
    const int64_t id = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (id >= static_cast<int64_t>(B) * T * H) return;
    const int h = static_cast<int>(id % H);
    const int64_t row = id / H, b = row / T, t = row % T;
    const float2 x = reinterpret_cast<const float2 *>(o + ((t * B + b) * H + h) * kKdaK)[lane];
    const float s = 1.0f / sqrtf(wave_sum_all(x.x * x.x + x.y * x.y) * (1.0f / kKdaK) + eps);
    const float2 g = reinterpret_cast<const float2 *>(og + id * kKdaK)[lane], wn = reinterpret_cast<const float2 *>(w)[lane];
    reinterpret_cast<float2 *>(out + id * kKdaK)[lane] =
        make_float2(x.x * s * wn.x / (1.0f + expf(-g.x)), x.y * s * wn.y / (1.0f + expf(-g.y)));
}

// ------------------------------------------------------------------ whole KDA layer step
// KDAAttention.__call__ for one token (attention_kda.py:94-115): the recurrence block also
// builds its inputs from the projection outputs: the short convolutions with SiLU
// (ops.py:46-60) of q, k (all 128 channels of the head) and v (the block's 32 columns),
// the L2 normalisation of q and k (ops.py:31-33, eps 1e-6), the decay gate
// lower_bound * sigmoid(exp(A_log[h]) * (f_b(f_a x) + dt_bias)) and beta = sigmoid(b x).
// The convolution states are read from conv_in and written to conv_out (distinct buffers),
// so no block reads a state another block rewrites.
struct KdaStepArgs {
    const float *q_raw, *k_raw, *v_raw;     // [P] projections of x
    const float *fb, *b_raw;                 // [P] f_b(f_a x), [H] b x
    const float *q_conv, *k_conv, *v_conv;   // [P, kc]
    const float *conv_in;                    // [3, kc - 1, P] (q, k, v), oldest first
    float *conv_out;                         // [3, kc - 1, P]
    const float *A_log, *dt_bias;            // [>= H], [P]
    float lower, scale;
    float *S;                                // [H, 128, 128] fp32, in place
    const float *og;                         // [P] g_proj x (the output gate logits)
    float *o;                                // [P] fp32: o * sigmoid(og)
    float *hss;                              // [H, 4] sum of o^2 over each block's 32 columns
    int H, kc;
};

__global__ __launch_bounds__(256) void kda_step_kernel(KdaStepArgs a) {
    __shared__ float red[2][4][kKdaVS];
    __shared__ float qs[kKdaK], ks[kKdaK], gs[kKdaK], vsh[kKdaVS], nrm[4];
    constexpr int V = kKdaK, nvb = kKdaK / kKdaVS;
    const int h = blockIdx.x / nvb, vb = blockIdx.x % nvb;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6, cg = t & 7, r = t >> 3;
    const int P = a.H * kKdaK, kc = a.kc;
    const int c0 = vb * kKdaVS + 4 * cg;
    float *Sp[4];
    float4 x[4];
    kda_load_state(a.S, h, V, c0, x, Sp);
    // q (threads 0..127) and k (128..255): convolution, SiLU, then the L2 norm of the head
    {
        const int m = t >> 7, ch = h * kKdaK + (t & 127);
        const float *cw = (m ? a.k_conv : a.q_conv) + static_cast<int64_t>(ch) * kc;
        const float *cin = a.conv_in + static_cast<int64_t>(m) * (kc - 1) * P + ch;
        const float xr = (m ? a.k_raw : a.q_raw)[ch];
        float y = 0.f;
        for (int j = 0; j < kc - 1; ++j) y = fmaf(cw[j], cin[static_cast<int64_t>(j) * P], y);
        y = fmaf(cw[kc - 1], xr, y);
        y = y / (1.0f + expf(-y));
        if (vb == 0) {
            float *cout = a.conv_out + static_cast<int64_t>(m) * (kc - 1) * P + ch;
            for (int j = 0; j < kc - 2; ++j) cout[static_cast<int64_t>(j) * P] = cin[static_cast<int64_t>(j + 1) * P];
            cout[static_cast<int64_t>(kc - 2) * P] = xr;
        }
        const float ss = wave_sum_all(y * y);
        if (lane == 0) nrm[wave] = ss;
        __syncthreads();
        const float n = m ? nrm[2] + nrm[3] : nrm[0] + nrm[1];
        const float yn = y / sqrtf(n + 1e-6f);
        if (m == 0)
            qs[t] = yn * a.scale;
        else
            ks[t - 128] = yn;
    }
    // v for this block's columns (and their convolution states), the decay gate, beta
    if (t < kKdaVS) {
        const int ch = h * kKdaK + vb * kKdaVS + t;
        const float *cw = a.v_conv + static_cast<int64_t>(ch) * kc;
        const float *cin = a.conv_in + static_cast<int64_t>(2) * (kc - 1) * P + ch;
        const float xr = a.v_raw[ch];
        float y = 0.f;
        for (int j = 0; j < kc - 1; ++j) y = fmaf(cw[j], cin[static_cast<int64_t>(j) * P], y);
        y = fmaf(cw[kc - 1], xr, y);
        vsh[t] = y / (1.0f + expf(-y));
        float *cout = a.conv_out + static_cast<int64_t>(2) * (kc - 1) * P + ch;
        for (int j = 0; j < kc - 2; ++j) cout[static_cast<int64_t>(j) * P] = cin[static_cast<int64_t>(j + 1) * P];
        cout[static_cast<int64_t>(kc - 2) * P] = xr;
    }
    if (t >= 128) {
        const int i = t - 128, ch = h * kKdaK + i;
        const float z = expf(a.A_log[h]) * (a.fb[ch] + a.dt_bias[ch]);
        gs[i] = a.lower / (1.0f + expf(-z));
    }
    const float b = 1.0f / (1.0f + expf(-a.b_raw[h]));
    __syncthreads();
    float kk[4], qq[4], dk[4], vv[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        kk[j] = ks[r + 32 * j];
        qq[j] = qs[r + 32 * j];
        dk[j] = expf(gs[r + 32 * j]);
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) vv[c] = vsh[4 * cg + c];
    const float o = kda_apply(x, kk, qq, dk, vv, b, red);
    kda_store_state(x, Sp);
    // the block's share of the head's sum of squares (for the gated RMSNorm), and o gated
    if (t < kKdaVS) {
        float ss = o * o;
        ss += __shfl_xor(ss, 1);
        ss += __shfl_xor(ss, 2);
        ss += __shfl_xor(ss, 4);
        ss += __shfl_xor(ss, 8);
        ss += __shfl_xor(ss, 16);
        if (t == 0) a.hss[h * nvb + vb] = ss;
        const int64_t c = static_cast<int64_t>(h) * V + vb * kKdaVS + t;
        a.o[c] = o / (1.0f + expf(-a.og[c]));
    }
}

}  // namespace
}  // namespace k3

using namespace k3;

static int kda_recurrent_impl(const void *q, const void *k, const void *v, const void *g, const void *beta,
                              int in_dtype, float *state, void *out, int out_dtype, int64_t T, int64_t qk_heads,
                              int64_t v_heads, int64_t key_dim, int64_t value_dim, float scale, void *stream) {
    if (!q || !k || !v || !g || !beta || !state || !out) return set_error(K3_ERR_NULL, "kda recurrence: null pointer");
    if (in_dtype != K3_F32 && in_dtype != K3_BF16)
        return set_error(K3_ERR_DTYPE, "kda recurrence: in_dtype %d", in_dtype);
    if (out_dtype != K3_F32 && out_dtype != K3_BF16)
        return set_error(K3_ERR_DTYPE, "kda recurrence: out_dtype %d", out_dtype);
    if (key_dim != kKdaK)
        return set_error(K3_ERR_SHAPE, "kda recurrence: key_dim=%lld; the kernel takes %d", (long long)key_dim, kKdaK);
    if (value_dim <= 0 || value_dim % kKdaVS || value_dim > 4096)
        return set_error(K3_ERR_SHAPE, "kda recurrence: value_dim=%lld must be a positive multiple of %d, <= 4096",
                         (long long)value_dim, kKdaVS);
    if (qk_heads <= 0 || v_heads <= 0 || v_heads % qk_heads || v_heads > (1 << 20))
        return set_error(K3_ERR_SHAPE, "kda recurrence: v_heads=%lld must be a positive multiple of qk_heads=%lld",
                         (long long)v_heads, (long long)qk_heads);
    if (T <= 0 || T > (1 << 24)) return set_error(K3_ERR_SHAPE, "kda recurrence: T=%lld", (long long)T);
    if (!aligned16(state)) return set_error(K3_ERR_ALIGN, "kda recurrence: the state must be 16-byte aligned");
    KdaArgs a{};
    a.q = q, a.k = k, a.v = v, a.g = g, a.beta = beta;
    a.in_bf16 = in_dtype == K3_BF16;
    a.S = state;
    a.out = out;
    a.out_bf16 = out_dtype == K3_BF16;
    a.HV = static_cast<int>(v_heads);
    a.G = static_cast<int>(v_heads / qk_heads);
    a.V = static_cast<int>(value_dim);
    a.T = static_cast<int>(T);
    a.vec = aligned16(q) && aligned16(k) && aligned16(g) && (reinterpret_cast<uintptr_t>(out) & 7) == 0;
    a.scale = scale;
    const int64_t blocks = v_heads * (value_dim / kKdaVS);
    if (T == 1)
        kda_decode_kernel<<<dim3(static_cast<unsigned>(blocks)), 256, 0, static_cast<hipStream_t>(stream)>>>(a);
    else
        kda_sequence_kernel<<<dim3(static_cast<unsigned>(blocks)), 256, 0, static_cast<hipStream_t>(stream)>>>(a);
    return check_hip(hipGetLastError(), "kda recurrence launch");
}

extern "C" int k3_kda_recurrent_decode(const void *q, const void *k, const void *v, const void *g, const void *beta,
                                       int in_dtype, float *state, void *out, int out_dtype, int64_t qk_heads,
                                       int64_t v_heads, int64_t key_dim, int64_t value_dim, float scale,
                                       void *stream) {
    return kda_recurrent_impl(q, k, v, g, beta, in_dtype, state, out, out_dtype, 1, qk_heads, v_heads, key_dim,
                              value_dim, scale, stream);
}

extern "C" int k3_kda_recurrent(const void *q, const void *k, const void *v, const void *g, const void *beta,
                                int in_dtype, float *state, void *out, int out_dtype, int64_t T, int64_t qk_heads,
                                int64_t v_heads, int64_t key_dim, int64_t value_dim, float scale, void *stream) {
    return kda_recurrent_impl(q, k, v, g, beta, in_dtype, state, out, out_dtype, T, qk_heads, v_heads, key_dim,
                              value_dim, scale, stream);
}

extern "C" int k3_kda_prefill_inputs(const float *q_raw, const float *k_raw, const float *v_raw, const float *fb,
                                     const float *b_raw, const float *q_conv, const float *k_conv, const float *v_conv,
                                     const float *q_win, const float *k_win, const float *v_win, float *q_win_out,
                                     float *k_win_out, float *v_win_out, const float *A_log, const float *dt_bias,
                                     float *q, float *k, float *v, float *g, float *beta, int64_t B, int64_t T,
                                     int64_t heads, int64_t head_dim, int64_t conv_size, float gate_lower_bound,
                                     void *stream) {
    const bool windows = conv_size != 1;    // (one tap keeps no inputs: the windows are empty)
    if (!q_raw || !k_raw || !v_raw || !fb || !b_raw || !q_conv || !k_conv || !v_conv ||
        (windows && (!q_win_out || !k_win_out || !v_win_out)) || !A_log || !dt_bias || !q || !k || !v || !g || !beta || (!q_win != !k_win) || (!q_win != !v_win))
        return set_error(K3_ERR_NULL, "kda prefill inputs: null pointer");
    if (head_dim != kKdaK) return set_error(K3_ERR_SHAPE, "kda prefill inputs: head_dim=%lld; the kernels take %d",
                                            (long long)head_dim, kKdaK);
    if (conv_size < 1 || conv_size > (1 << 16))
        return set_error(K3_ERR_SHAPE, "kda prefill inputs: conv_size=%lld", (long long)conv_size);
    if (B <= 0 || T <= 0 || heads <= 0 || B > (1 << 24) || T > (1 << 24) || heads > (1 << 20) ||
        B * cdiv(T, kPrepTokens) >= (1ll << 25) || B * cdiv(T, kPrepTokens) * heads >= (1ll << 25))
        return set_error(K3_ERR_SHAPE, "kda prefill inputs: B=%lld, T=%lld, heads=%lld", (long long)B, (long long)T,
                         (long long)heads);
    KdaPrepArgs a{};
    a.raw[0] = q_raw, a.raw[1] = k_raw, a.raw[2] = v_raw, a.fb = fb, a.b_raw = b_raw;
    a.conv[0] = q_conv, a.conv[1] = k_conv, a.conv[2] = v_conv;
    a.win[0] = q_win, a.win[1] = k_win, a.win[2] = v_win;
    a.win_out[0] = q_win_out, a.win_out[1] = k_win_out, a.win_out[2] = v_win_out;
    a.A_log = A_log, a.dt_bias = dt_bias, a.lower = gate_lower_bound;
    a.q = q, a.k = k, a.v = v, a.g = g, a.beta = beta;
    a.B = static_cast<int>(B), a.T = static_cast<int>(T), a.H = static_cast<int>(heads), a.kc = static_cast<int>(conv_size);
    kda_prep_kernel<<<dim3(static_cast<unsigned>(heads * cdiv(T, kPrepTokens) * B)), 128, 0, static_cast<hipStream_t>(stream)>>>(a);
    return check_hip(hipGetLastError(), "kda prefill inputs launch");
}

extern "C" int k3_kda_gated_norm(const float *o, const float *gate, const float *w, float eps, float *out, int64_t B,
                                 int64_t T, int64_t heads, int64_t head_dim, void *stream) {
    if (!o || !gate || !w || !out) return set_error(K3_ERR_NULL, "kda gated norm: null pointer");
    if (head_dim != kKdaK) return set_error(K3_ERR_SHAPE, "kda gated norm: head_dim=%lld; the kernel takes %d",
                                            (long long)head_dim, kKdaK);
    if (B <= 0 || T <= 0 || heads <= 0 || B * T * heads >= (1ll << 31))
        return set_error(K3_ERR_SHAPE, "kda gated norm: B=%lld, T=%lld, heads=%lld", (long long)B, (long long)T, (long long)heads);
    if (!aligned16(o) || !aligned16(gate) || !aligned16(w) || !aligned16(out))
        return set_error(K3_ERR_ALIGN, "kda gated norm: 16-byte alignment");
    kda_gated_norm_kernel<<<dim3(static_cast<unsigned>(cdiv(B * T * heads, 4))), 256, 0, static_cast<hipStream_t>(stream)>>>(
        o, gate, w, eps, out, static_cast<int>(B), static_cast<int>(T), static_cast<int>(heads));
    return check_hip(hipGetLastError(), "kda gated norm launch");
}

namespace {
struct KdaStepWs {
    size_t q, k, v, og, fa, b, fb, o, hss, total;
};
KdaStepWs kda_step_ws(int64_t H) {
    const size_t P = static_cast<size_t>(H) * kKdaK;
    KdaStepWs L{};
    size_t off = 0;
    auto take = [&](size_t n) { const size_t at = off; off += (n * 4 + 255) & ~size_t(255); return at; };
    L.q = take(P), L.k = take(P), L.v = take(P), L.og = take(P), L.fa = take(kKdaK), L.b = take(H), L.fb = take(P);
    L.o = take(P);
    L.hss = take(static_cast<size_t>(H) * (kKdaK / kKdaVS));
    L.total = off;
    return L;
}
}  // namespace

extern "C" int64_t k3_kda_step_workspace_size(int64_t heads) { return static_cast<int64_t>(kda_step_ws(heads).total); }

extern "C" int k3_kda_step_decode(const void *x, int x_dtype, const void *q_proj, const void *k_proj,
                                  const void *v_proj, const void *g_proj, const void *o_proj, const void *f_a,
                                  const void *f_b, const void *b_proj, const float *q_conv, const float *k_conv,
                                  const float *v_conv, const float *conv_in, float *conv_out, const float *o_norm,
                                  const float *A_log, const float *dt_bias, float *state, void *out, int out_dtype,
                                  int64_t hidden, int64_t heads, int64_t head_dim, int64_t conv_size,
                                  float gate_lower_bound, float eps, void *workspace, int64_t workspace_bytes,
                                  void *stream) {
    if (!x || !q_proj || !k_proj || !v_proj || !g_proj || !o_proj || !f_a || !f_b || !b_proj || !q_conv || !k_conv ||
        !v_conv || !conv_in || !conv_out || !o_norm || !A_log || !dt_bias || !state || !out || !workspace)
        return set_error(K3_ERR_NULL, "kda step: null pointer");
    if (x_dtype != K3_F32 && x_dtype != K3_BF16) return set_error(K3_ERR_DTYPE, "kda step: x_dtype %d", x_dtype);
    if (out_dtype != K3_F32 && out_dtype != K3_BF16) return set_error(K3_ERR_DTYPE, "kda step: out_dtype %d", out_dtype);
    if (head_dim != kKdaK) return set_error(K3_ERR_SHAPE, "kda step: head_dim=%lld; the kernels take %d",
                                            (long long)head_dim, kKdaK);
    const int64_t P = heads * head_dim;
    if (heads <= 0 || P > kMaxWidth || hidden <= 0 || hidden % 8 || hidden > kMaxWidth)
        return set_error(K3_ERR_SHAPE, "kda step: heads*head_dim and hidden must be <= %d (hidden a multiple of 8)",
                         kMaxWidth);
    if (conv_size < 2 || conv_size > 8) return set_error(K3_ERR_SHAPE, "kda step: conv_size=%lld", (long long)conv_size);
    if (conv_in == conv_out) return set_error(K3_ERR_SHAPE, "kda step: conv_in and conv_out must be distinct buffers");
    if (!aligned16(x) || !aligned16(q_proj) || !aligned16(k_proj) || !aligned16(v_proj) || !aligned16(g_proj) ||
        !aligned16(o_proj) || !aligned16(f_a) || !aligned16(f_b) || !aligned16(b_proj) || !aligned16(o_norm) ||
        !aligned16(state) || !aligned16(workspace))
        return set_error(K3_ERR_ALIGN, "kda step: vectors, weights, state and workspace must be 16-byte aligned");
    if (P * hidden * 2 >= (1ll << 31)) return set_error(K3_ERR_SHAPE, "kda step: a weight matrix exceeds 2 GiB");
    const KdaStepWs L = kda_step_ws(heads);
    if (workspace_bytes < static_cast<int64_t>(L.total))
        return set_error(K3_ERR_WORKSPACE, "kda step: workspace %lld < %zu bytes", (long long)workspace_bytes, L.total);
    char *ws = static_cast<char *>(workspace);
    float *wq = reinterpret_cast<float *>(ws + L.q), *wk = reinterpret_cast<float *>(ws + L.k);
    float *wv = reinterpret_cast<float *>(ws + L.v), *wog = reinterpret_cast<float *>(ws + L.og);
    float *wfa = reinterpret_cast<float *>(ws + L.fa), *wb = reinterpret_cast<float *>(ws + L.b);
    float *wfb = reinterpret_cast<float *>(ws + L.fb), *wo = reinterpret_cast<float *>(ws + L.o);
    float *whss = reinterpret_cast<float *>(ws + L.hss);
    auto st = static_cast<hipStream_t>(stream);
    // K1: rows of q, k, v, g, f_a and b against x
    RowsArgs a1{};
    a1.x = x, a1.x_bf16 = x_dtype == K3_BF16, a1.K = static_cast<int>(hidden);
    const void *w1[6] = {q_proj, k_proj, v_proj, g_proj, f_a, b_proj};
    float *y1[6] = {wq, wk, wv, wog, wfa, wb};
    const int n1[6] = {static_cast<int>(P), static_cast<int>(P), static_cast<int>(P), static_cast<int>(P), kKdaK,
                       static_cast<int>(heads)};
    for (int i = 0; i < 6; ++i) a1.w[i] = static_cast<const uint16_t *>(w1[i]), a1.N[i] = n1[i], a1.y[i] = y1[i];
    int rc = launch_rows<kModeX>(a1, st);
    if (rc) return rc;
    // K2: rows of f_b against f_a x
    RowsArgs a2{};
    a2.o = wfa, a2.K = kKdaK;
    a2.w[0] = static_cast<const uint16_t *>(f_b), a2.N[0] = static_cast<int>(P), a2.y[0] = wfb;
    rc = launch_rows<kModeGate>(a2, st);
    if (rc) return rc;
    // K3: convolutions, norms, gate and the recurrence
    KdaStepArgs k{};
    k.q_raw = wq, k.k_raw = wk, k.v_raw = wv, k.fb = wfb, k.b_raw = wb;
    k.q_conv = q_conv, k.k_conv = k_conv, k.v_conv = v_conv, k.conv_in = conv_in, k.conv_out = conv_out;
    k.A_log = A_log, k.dt_bias = dt_bias, k.lower = gate_lower_bound, k.scale = 1.0f / sqrtf(static_cast<float>(kKdaK));
    k.S = state, k.og = wog, k.o = wo, k.hss = whss, k.H = static_cast<int>(heads), k.kc = static_cast<int>(conv_size);
    kda_step_kernel<<<dim3(static_cast<unsigned>(heads * (kKdaK / kKdaVS))), 256, 0, st>>>(k);
    rc = check_hip(hipGetLastError(), "kda step: recurrence launch");
    if (rc) return rc;
    // K4: rows of o_proj against the gated heads scaled by their RMS norms, in the persistent
    // row form (one block per CU stages the 48 KB vector once): measured faster for this
    // launch, while K1 measured slower in that form
    RowsArgs a4{};
    a4.o = wo, a4.gl = whss, a4.nw = o_norm, a4.eps = eps, a4.K = static_cast<int>(P);
    a4.w[0] = static_cast<const uint16_t *>(o_proj), a4.N[0] = static_cast<int>(hidden);
    a4.out = out, a4.out_bf16 = out_dtype == K3_BF16;
    return launch_rows_loop<kModeHeadNorm>(a4, st);
}
