// MLA attention for many query tokens over the latent cache, in fp32 arithmetic on the bf16
// matrix cores.
//
// Reference: the multi-token branch of MLAAttention.__call__
// (air_llm/models/kimi_k3/attention_mla.py:193-212): scores of every query against every cached
// position, causal mask, softmax, context, per head.  The reference keeps the cache latent
// and works in its 576 columns; for many queries it costs less to expand the cache once per
// head (192 score columns and 128 value columns instead of 576 and 512) and the result is
// the same.
//
// fp32 operands (queries, expanded keys and values, probabilities) enter as three bf16 terms
// whose sum is exact, rounded to nearest (split3_near); of the nine products of two such values the
// six of at least 2^-16 of the largest are taken.  What is left out is at most 2^-23 of the
// product, 0.1 x 2^-24 root mean square over pairs of normal values and of either sign (0.9 x 2^-24
// at most over two million of them), so it stays below fp32's rounding of the product.  Terms cut
// instead of rounded left out 0.7 x 2^-24 on average, up to 2^-21, always with the product's sign.
//
//   expand     k3_dense's KV form: keys and values of all heads, already split (mla_expand_kv)
//   split_rot  fp32 cache only: the rotary rows as three terms
//   attention  block = (head, 128 queries), eight waves of 16 queries; 32 cached tokens per
//              step, staged in LDS double buffered, XOR-swizzled 16-byte chunks.  A wave forms
//              the scores transposed (tokens x queries), so a query's scores, its running
//              maximum and its sums stay in one lane column, and the probabilities leave the
//              softmax in the very order the context product takes them.
// What bounds it: the six-fold products (1.3e11 at 1000 tokens and 64 heads, about 100 us of the
// matrix cores) beside LDS reads of 52 KB per wave and step, with two waves per SIMD to overlap
// a step's scores, softmax and context.  Measured at 1000 tokens, 64 heads: attention 147 us,
// expansion 59 us; the fp32 absorbed form in library products took 1.9 ms with its passes.
#include <algorithm>

#include "k3_common.h"

namespace k3 {
namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kThreads = 512, kBQ = 128, kBT = 32;
constexpr int kNope = 128, kRope = 64, kV = 128, kQ = kNope + kRope;

struct AttnArgs {
    const float *q;          // [T, heads, 192], row pitch ldq
    int64_t ldq;
    const uint16_t *kp, *vt; // expanded keys and values of this launch's heads
    const void *rot;         // bf16 rows [Tk, 64] of pitch ld_rot, or three-term rows [tpad, 3, 64]
    int64_t ld_rot;
    const float *gate;       // [T, heads * 128] logits or null
    float *out;              // [T, heads * 128]
    int64_t ldo;             // pitch of gate and out
    int T, Tk, tpad, heads, nq;
    float c;                 // scale * log2(e)
};

__global__ __launch_bounds__(256) void split_rot_kernel(const float *rot, int64_t ld, uint16_t *out, int Tk, int tpad) {
    const int id = blockIdx.x * 256 + threadIdx.x, t = id >> 6, c = id & 63;
    if (t >= tpad) return;
    uint32_t a, b, d;
    split3_near(t < Tk ? rot[t * ld + c] : 0.f, a, b, d);
    uint16_t *o = out + static_cast<int64_t>(t) * 3 * kRope + c;
    o[0] = static_cast<uint16_t>(a >> 16), o[kRope] = static_cast<uint16_t>(b >> 16), o[2 * kRope] = static_cast<uint16_t>(d >> 16);
}

// 8 fp32 values -> three fragments
template <bool SMALL>
__device__ __forceinline__ void split8(const float (&v)[8], bf16x8 (&f)[3]) {
    uint32_t t[3][8];
#pragma unroll
    for (int i = 0; i < 8; ++i) split3_near<SMALL>(v[i], t[0][i], t[1][i], t[2][i]);
#pragma unroll
    for (int x = 0; x < 3; ++x)
        f[x] = __builtin_bit_cast(bf16x8, make_uint4(hi16x2(t[x][0], t[x][1]), hi16x2(t[x][2], t[x][3]),
                                                     hi16x2(t[x][4], t[x][5]), hi16x2(t[x][6], t[x][7])));
}

__device__ __forceinline__ f32x4 mfma(const bf16x8 &a, const bf16x8 &b, const f32x4 &c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// RT: terms of the rotary rows (bf16 cache 1, fp32 cache 3)
template <int RT>
__global__ __launch_bounds__(kThreads, 2) void attention_kernel(AttnArgs a) {
    constexpr int kK = kBT * kNope * 2, kR = kBT * kRope * 2, kVt = kV * kBT * 2;  // bytes of one term
    constexpr int kOffR = 3 * kK, kOffV = kOffR + RT * kR, kStage = kOffV + 3 * kVt;
    extern __shared__ char lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, q = lane >> 4;
    // The long query tiles first (a tile's work grows with its position); blocks b % 8 run on
    // one XCD, which takes the heads h % 8 == b % 8, so its L2 holds their keys and values.
    const int nb = a.heads * a.nq, li = blockIdx.x >> 3, hx = a.heads >> 3;
    int head, qt;
    if ((a.heads & 7) == 0) {
        head = (blockIdx.x & 7) + 8 * (li % hx), qt = a.nq - 1 - li / hx;
    } else {
        head = blockIdx.x % a.heads, qt = a.nq - 1 - static_cast<int>(blockIdx.x) / a.heads;
    }
    if (static_cast<int>(blockIdx.x) >= nb) return;
    const int past = a.Tk - a.T;                       // query t sees cached positions 0 .. past + t
    const int q0 = qt * kBQ + wave * 16;               // this wave's first query
    const int last = past + min(qt * kBQ + kBQ, a.T) - 1;   // last position any query of the block sees
    const int nsteps = last / kBT + 1;
    const bool active = q0 < a.T;
    const int wlast = past + min(q0 + 16, a.T) - 1;    // .. any query of the wave sees

    // ---- queries: fragments of the transposed product's B operand
    bf16x8 qf[6][3];
    {
        const int t = min(q0 + r16, a.T - 1);
        const float *qr = a.q + t * a.ldq + head * kQ + 8 * q;
#pragma unroll
        for (int ks = 0; ks < 6; ++ks) {
            const float4 x = *reinterpret_cast<const float4 *>(qr + ks * 32), y = *reinterpret_cast<const float4 *>(qr + ks * 32 + 4);
            const float v[8] = {x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w};
            split8<false>(v, qf[ks]);
        }
    }

    // ---- staging of one step: 16 bytes per thread and term of keys and values; rotary rows by
    // the first four waves
    const char *kp = reinterpret_cast<const char *>(a.kp + mla_k_index(head, a.tpad, 0, 0)) + (tid >> 4) * 768 + (tid & 15) * 16;
    const char *vt = reinterpret_cast<const char *>(a.vt + mla_v_index(head, a.tpad, 0, 0, 0)) + tid * 16;
    const int rk = (tid >> 3) & 31, rc = tid & 7;
    u32x4 RK[3], RV[3], RR[RT];
    // (native vectors, straight-line and unconditional, past the last step that step again: as
    // uint4 structs the staged values went through private memory and every step waited for
    // its loads)
    auto load = [&](int step) {
        const int s = min(step, nsteps - 1);
#pragma unroll
        for (int x = 0; x < 3; ++x) {
            RK[x] = *reinterpret_cast<const u32x4 *>(kp + static_cast<int64_t>(s) * (kBT * 768) + x * 256);
            RV[x] = *reinterpret_cast<const u32x4 *>(vt + static_cast<int64_t>(s) * (3 * kVt) + x * kVt);
        }
        const int t = s * kBT + rk;    // rows past the cache (never seen): its last row
        const uint16_t *row = RT == 1 ? static_cast<const uint16_t *>(a.rot) + min(t, a.Tk - 1) * a.ld_rot
                                      : static_cast<const uint16_t *>(a.rot) + static_cast<int64_t>(t) * 3 * kRope;
#pragma unroll
        for (int x = 0; x < RT; ++x) RR[x] = *reinterpret_cast<const u32x4 *>(row + x * kRope + rc * 8);
    };
    auto store = [&](int buf) {
        char *L = lds + buf * kStage;
#pragma unroll
        for (int x = 0; x < 3; ++x) {
            *reinterpret_cast<u32x4 *>(L + x * kK + (tid >> 4) * 256 + (((tid & 15) ^ ((tid >> 4) & 15)) << 4)) = RK[x];
            *reinterpret_cast<u32x4 *>(L + kOffV + x * kVt + (tid >> 2) * 64 + (((tid & 3) ^ ((tid >> 3) & 3)) << 4)) = RV[x];
        }
        if (wave < 4) {
#pragma unroll
            for (int x = 0; x < RT; ++x)
                *reinterpret_cast<u32x4 *>(L + kOffR + x * kR + rk * 128 + ((rc ^ (rk & 7)) << 4)) = RR[x];
        }
    };

    f32x4 o[8];
#pragma unroll
    for (int d = 0; d < 8; ++d) o[d] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, l = 0.f;      // of query r16: maximum of c * score, this lane's part of the sum

    auto step = [&](int s, int buf) {
        const char *L = lds + buf * kStage;
        // scores: two tiles of 16 tokens; the main products and the small ones apart
        f32x4 hi[2], lo[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) hi[h] = lo[h] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < 6; ++ks) {
            constexpr int kTerms[2] = {3, RT};
            bf16x8 kf[2][3];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int row = 16 * h + r16;
#pragma unroll
                for (int x = 0; x < kTerms[ks >= 4]; ++x)
                    kf[h][x] = ks < 4 ? *reinterpret_cast<const bf16x8 *>(L + x * kK + row * 256 + (((4 * ks + q) ^ (row & 15)) << 4))
                                      : *reinterpret_cast<const bf16x8 *>(L + kOffR + x * kR + row * 128 +
                                                                          (((4 * (ks - 4) + q) ^ (row & 7)) << 4));
            }
#pragma unroll
            for (int x = 2; x >= 0; --x)           // terms x (tokens) and y (queries), x + y <= 2
#pragma unroll
                for (int y = 2 - x; y >= 0; --y) {
                    if (x >= kTerms[ks >= 4]) continue;
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        if (x + y)
                            lo[h] = mfma(kf[h][x], qf[ks][y], lo[h]);
                        else
                            hi[h] = mfma(kf[h][0], qf[ks][0], hi[h]);
                    }
                }
        }
        // softmax: lane (r16, q) holds tokens 16 h + 4q + v of query r16
        float p[8];
        const bool edge = s * kBT + kBT - 1 > past + q0;
        const int seen = past + q0 + r16 - s * kBT;    // last visible token of this step
        float mx = m;
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                // (an infinite score stands in hi alone: infinity times a zero or negative term is in lo)
                float z = (__builtin_isinf(hi[h][v]) ? hi[h][v] : hi[h][v] + lo[h][v]) * a.c;
                if (edge && 16 * h + 4 * q + v > seen) z = -INFINITY;
                p[4 * h + v] = z;
            }
#pragma unroll
        for (int i = 0; i < 8; ++i) mx = fmaxf(mx, p[i]);
        mx = fmaxf(mx, __shfl_xor(mx, 16));
        mx = fmaxf(mx, __shfl_xor(mx, 32));
        // (every score so far -infinity: weights of zero, not of -infinity - -infinity)
        const float ref = mx == -INFINITY ? 0.f : mx;
        const float al = __builtin_amdgcn_exp2f(m - ref);
        m = mx;
        l *= al;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            p[i] = __builtin_amdgcn_exp2f(p[i] - ref);
            l += p[i];
        }
#pragma unroll
        for (int d = 0; d < 8; ++d) o[d] *= al;
        bf16x8 pf[3];
        split8<true>(p, pf);
        // context, transposed: rows 16 d + r16 of the values against the probabilities
#pragma unroll
        for (int d = 0; d < 8; d += 2) {
            bf16x8 vf[2][3];
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const int row = 16 * (d + e) + r16;
#pragma unroll
                for (int x = 0; x < 3; ++x)
                    vf[e][x] = *reinterpret_cast<const bf16x8 *>(L + kOffV + x * kVt + row * 64 + ((q ^ ((row >> 1) & 3)) << 4));
            }
#pragma unroll
            for (int x = 2; x >= 0; --x)
#pragma unroll
                for (int y = 2 - x; y >= 0; --y)
#pragma unroll
                    for (int e = 0; e < 2; ++e) o[d + e] = mfma(vf[e][x], pf[y], o[d + e]);
        }
    };

    load(0);
    store(0);
    load(1);
    for (int s = 0;; s += 2) {
        __syncthreads();
        if (active && s * kBT <= wlast) step(s, 0);
        __builtin_amdgcn_sched_barrier(0);
        if (s + 1 >= nsteps) break;
        store(1);
        load(s + 2);
        __syncthreads();
        if (active && (s + 1) * kBT <= wlast) step(s + 1, 1);
        __builtin_amdgcn_sched_barrier(0);
        if (s + 2 >= nsteps) break;
        store(0);
        load(s + 3);
    }
    l += __shfl_xor(l, 16);
    l += __shfl_xor(l, 32);
    const int t = q0 + r16;
    if (t >= a.T) return;
    const float r = 1.0f / l;
    float *out = a.out + t * a.ldo + head * kV + 4 * q;
#pragma unroll
    for (int d = 0; d < 8; ++d) {
        f32x4 v = o[d] * r;
        if (a.gate) {
            const f32x4 g = *reinterpret_cast<const f32x4 *>(a.gate + t * a.ldo + head * kV + 16 * d + 4 * q);
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = v[i] / (1.0f + expf(-g[i]));
        }
        *reinterpret_cast<f32x4 *>(out + 16 * d) = v;
    }
}

// The heads are expanded in groups whose keys and values stay within this many bytes.
constexpr int64_t kGroupBytes = 1ll << 30;

struct Ws {
    int64_t tpad, group, k, v, rot, total;
};
Ws ws_layout(int64_t Tk, int64_t heads) {
    Ws w{};
    w.tpad = cdiv(Tk, kBT) * kBT;
    const int64_t per = w.tpad * 3 * 128 * 2;          // bytes of one head's keys (and of its values)
    w.group = std::max<int64_t>(1, std::min(heads, kGroupBytes / (2 * per)));
    if (w.group >= 8 && w.group < heads) w.group &= ~int64_t(7);
    w.k = 0, w.v = w.group * per, w.rot = 2 * w.group * per;
    w.total = w.rot + w.tpad * 3 * kRope * 2;
    return w;
}

template <int RT>
int launch_attention(const AttnArgs &a, hipStream_t st) {
    constexpr int bytes = 2 * (3 * kBT * kNope * 2 + RT * kBT * kRope * 2 + 3 * kV * kBT * 2);
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void *>(&attention_kernel<RT>),
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    const int rc = check_hip(attr, "mla prefill: LDS size attribute");
    if (rc) return rc;
    attention_kernel<RT><<<dim3(static_cast<unsigned>(a.heads * a.nq)), kThreads, bytes, st>>>(a);
    return check_hip(hipGetLastError(), "mla prefill: attention launch");
}

}  // namespace
}  // namespace k3

using namespace k3;

extern "C" int64_t k3_mla_prefill_workspace_size(int64_t Tk, int64_t heads) {
    return Tk > 0 && heads > 0 ? ws_layout(Tk, heads).total : 0;
}

extern "C" int k3_mla_prefill(const float *q, int64_t ldq, const void *kv_b, const void *lat, int64_t ld_lat,
                              const void *rot, int64_t ld_rot, int cache_dtype, const float *gate, float *out, int64_t T,
                              int64_t Tk, int64_t heads, int64_t kv_lora_rank, int64_t rope_dim, int64_t nope_dim,
                              int64_t v_dim, float scale, void *workspace, int64_t workspace_bytes, void *stream) {
    if (!q || !kv_b || !lat || !rot || !out || !workspace) return set_error(K3_ERR_NULL, "mla prefill: null pointer");
    if (cache_dtype != K3_BF16 && cache_dtype != K3_F32) return set_error(K3_ERR_DTYPE, "mla prefill: cache_dtype %d", cache_dtype);
    if (kv_lora_rank != 512 || rope_dim != kRope || nope_dim != kNope || v_dim != kV)
        return set_error(K3_ERR_SHAPE, "mla prefill: the kernels take kv_lora_rank 512, rope 64, nope 128, v 128");
    const int64_t es = cache_dtype == K3_F32 ? 4 : 2;
    if (T <= 0 || Tk < T || Tk > (1 << 24) || heads <= 0 || heads > 4096 || ldq < heads * kQ || ldq % 4 || ld_lat < 512 ||
        (ld_lat * es) % 16 || ld_rot < kRope || (ld_rot * es) % 16 || ld_lat > (1 << 20))
        return set_error(K3_ERR_SHAPE, "mla prefill: T=%lld, Tk=%lld, heads=%lld or a row pitch", (long long)T, (long long)Tk,
                         (long long)heads);
    if (!aligned16(q) || !aligned16(kv_b) || !aligned16(lat) || !aligned16(rot) || !aligned16(out) || !aligned16(workspace) ||
        (gate && !aligned16(gate)))
        return set_error(K3_ERR_ALIGN, "mla prefill: pointers must be 16-byte aligned");
    const Ws w = ws_layout(Tk, heads);
    if (workspace_bytes < w.total)
        return set_error(K3_ERR_WORKSPACE, "mla prefill: workspace %lld < %lld bytes", (long long)workspace_bytes, (long long)w.total);
    auto st = static_cast<hipStream_t>(stream);
    char *ws = static_cast<char *>(workspace);
    AttnArgs a{};
    a.ldq = ldq, a.ldo = heads * kV;
    a.T = static_cast<int>(T), a.Tk = static_cast<int>(Tk), a.tpad = static_cast<int>(w.tpad);
    a.nq = static_cast<int>(cdiv(T, kBQ));
    a.c = scale * 1.4426950408889634f;
    a.rot = rot, a.ld_rot = ld_rot;
    if (cache_dtype == K3_F32) {
        uint16_t *r3 = reinterpret_cast<uint16_t *>(ws + w.rot);
        split_rot_kernel<<<dim3(static_cast<unsigned>(cdiv(w.tpad * kRope, 256))), 256, 0, st>>>(
            static_cast<const float *>(rot), ld_rot, r3, a.Tk, a.tpad);
        const int rc = check_hip(hipGetLastError(), "mla prefill: rotary split launch");
        if (rc) return rc;
        a.rot = r3;
    }
    uint16_t *kp = reinterpret_cast<uint16_t *>(ws + w.k), *vt = reinterpret_cast<uint16_t *>(ws + w.v);
    for (int64_t h0 = 0; h0 < heads; h0 += w.group) {
        const int64_t n = std::min(w.group, heads - h0);
        int rc = mla_expand_kv(lat, cache_dtype, ld_lat, static_cast<const uint16_t *>(kv_b) + h0 * 256 * 512, Tk, n, kp, vt,
                               w.tpad, st);
        if (rc) return rc;
        a.q = q + h0 * kQ, a.out = out + h0 * kV, a.gate = gate ? gate + h0 * kV : nullptr;
        a.kp = kp, a.vt = vt, a.heads = static_cast<int>(n);
        rc = cache_dtype == K3_F32 ? launch_attention<3>(a, st) : launch_attention<1>(a, st);
        if (rc) return rc;
    }
    return K3_OK;
}
