// Dense projections for many tokens: out[M, N] = a[M, K] w[N, K]^T in fp32, a fp32 or bf16,
// w bf16, several weight matrices against one a in a single launch.
//
// The reference promotes a bf16 weight against an fp32 activation to an fp32 product
// (air_llm/models/kimi_k3/moe.py:67-68, attention_mla.py:168-216, attention_kda.py:94-115).
// Here an fp32 value is the exact sum of three bf16 terms (8 + 8 + 8 significant bits, cut
// off, not rounded, so no term overflows), each term meets the bf16 weight in the bf16
// matrix cores with exact products, and everything accumulates in fp32: the arithmetic of an
// fp32 product with another summation order, at a third of the bf16 rate instead of the
// fp32 matrix rate (a sixteenth).
//
// Block: 256 weight rows x BM tokens, eight waves, K in steps of 64 (one 128-byte line per
// weight row).  Operands load line-contiguous into registers one step ahead; the terms are
// split as they are stored to LDS, once per block, in 16-byte chunks XOR-swizzled by the row.
// Weight rows are the MFMA A operand, so a lane ends with four consecutive outputs of a token.
// BM falls with M (128 / 64 / 32), and K is split over blocks, with the partial sums added
// in order by a second launch, while there are fewer blocks than CUs.
// Measured against three library products of the terms and two adds (fp32 a): 1000 x 7168 x 8192
// 400 -> 314 us (1.12 PFLOP/s executed), 256 x 7168 x 12288 347 -> 141 us, 16 x 7168 x 8192 104 -> 33 us;
// bf16 a, six matrices of 49,376 rows in all at K 7168: 2 tokens 153 -> 120 us (5.9 TB/s), 256 tokens
// 349 -> 217 us.  What bounds it: the matrix cores at the clock they hold under load (46% busy by
// counter, LDS 24%, no bank conflicts), CUs without a tile where the tiles are more than half the
// CUs and no multiple of them (make_plan) and, at few tokens, HBM.
#include <algorithm>
#include <type_traits>

#include "k3_common.h"
#include "moe_common.h"

namespace k3 {
namespace {

constexpr int kBN = 256, kBK = 64, kThreads = 512;
constexpr int kMaxSeg = 8;
constexpr int kTargetBlocks = 256;   // one per CU
constexpr uint32_t kOob = 0xf0000000u;

struct DenseArgs {
    const void *a;           // [M, K], row pitch lda elements
    int64_t lda;
    int M, K;
    int mt, nt, ksplit, ksteps;      // token tiles, weight tiles, K pieces, 64-steps per piece
    int nseg;
    const uint16_t *w[kMaxSeg];      // [N, K] bf16 each
    float *out[kMaxSeg];             // [M, N] fp32 each
    int N[kMaxSeg], t0[kMaxSeg];     // rows and first weight tile of each matrix
    const float *add;                // [M, N] fp32 added to the (single) output, or null
    float *part;                     // [ksplit][M'][nt * 256] when ksplit > 1 (M' = mt * BM)
    uint16_t *kp, *vt;               // MLA keys and values (k3_common.h): bf16 terms
    int tpad;
};

// KV: the expansion of the MLA latent cache into keys and values.  A weight tile is one head's
// kv_b rows, 128 key rows (waves wn == 0) then 128 value rows (wn == 1, WN == 2), and the results
// are stored as three bf16 terms in the order the attention reads them; the value waves swap
// the MFMA operands, so a lane ends with four consecutive tokens of one value column.
template <int TERMS, int WM, int MT, bool KV>
__global__ __launch_bounds__(kThreads, 2) void dense_kernel(DenseArgs a) {
    constexpr int WN = 8 / WM, NT = kBN / WN / 16, BM = WM * MT * 16;
    constexpr int kW = kBN * 128, kA = BM * 128, kStage = kW + TERMS * kA;
    extern __shared__ char lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn = wave % WN, wm = wave / WN;
    const int r16 = lane & 15, q = lane >> 4;

    // Blocks b % 8 run on one XCD; it takes a contiguous eighth of the work list, token tiles
    // fastest, so the tiles that share weight rows share them in its L2.
    const int total = a.mt * a.nt * a.ksplit, per = (total + 7) >> 3;
    const int w = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if ((blockIdx.x >> 3) >= per || w >= total) return;
    const int mtile = w % a.mt, ks = (w / a.mt) % a.ksplit, ntile = w / a.mt / a.ksplit;
    int sg = 0;
    for (int i = 1; i < a.nseg; ++i) sg = ntile >= a.t0[i] ? i : sg;
    const int n0 = (ntile - a.t0[sg]) * kBN, m0 = mtile * BM;
    const int N = a.N[sg];
    const int k0 = ks * a.ksteps * kBK, kend = min(a.K, k0 + a.ksteps * kBK);
    const int NS = (kend - k0 + kBK - 1) / kBK;

    // ---- loads
    const int nrows = min(kBN, N - n0), mrows = min(BM, a.M - m0);
    const auto rw = make_rsrc(a.w[sg] + static_cast<int64_t>(n0) * a.K, static_cast<uint32_t>(nrows) * a.K * 2u);
    constexpr int ES = TERMS == 1 ? 2 : 4;                 // bytes per element of a
    constexpr int RPI = TERMS == 1 ? 8 : 4;                // rows per wave instruction
    constexpr int NA = BM / 8 / RPI > 0 ? BM / 8 / RPI : 1;
    const auto ra = make_rsrc(static_cast<const char *>(a.a) + static_cast<int64_t>(m0) * a.lda * ES,
                              static_cast<uint32_t>((static_cast<int64_t>(mrows - 1) * a.lda + a.K) * ES));
    const int wc = lane & 7, ac = TERMS == 1 ? lane & 7 : lane & 15;  // 16-byte chunk of a row's step
    uint32_t woff[4], aoff[NA];
#pragma unroll
    for (int n = 0; n < 4; ++n) {
        const int row = wave * 32 + 8 * n + (lane >> 3);
        woff[n] = row < nrows ? static_cast<uint32_t>(row) * a.K * 2u + wc * 16u + k0 * 2u : kOob;
    }
    const int arow0 = wave * NA * RPI + (TERMS == 1 ? lane >> 3 : lane >> 4);
#pragma unroll
    for (int n = 0; n < NA; ++n) {
        const int row = arow0 + n * RPI;
        aoff[n] = row < mrows ? static_cast<uint32_t>(row * a.lda * ES) + ac * 16u + k0 * ES : kOob;
    }
    uint4 RW[4], RA[NA];
    uint2 RT[NA][3];                                       // the split terms of RA (fp32 a)
    auto load_w = [&](int S) {
        const bool ok = k0 + S * kBK + wc * 8 < kend;
#pragma unroll
        for (int n = 0; n < 4; ++n) RW[n] = buf_load16(rw, ok ? woff[n] + S * (kBK * 2u) : kOob);
    };
    auto load_a = [&](int S) {
        const bool ok = k0 + S * kBK + ac * (16 / ES) < kend;
#pragma unroll
        for (int n = 0; n < NA; ++n) RA[n] = buf_load16(ra, ok ? aoff[n] + S * (kBK * ES) : kOob);
    };
    auto store_w = [&](int buf) {
#pragma unroll
        for (int n = 0; n < 4; ++n) {
            const int row = wave * 32 + 8 * n + (lane >> 3);
            *reinterpret_cast<uint4 *>(lds + buf * kStage + row * 128 + ((wc ^ (row & 7)) << 4)) = RW[n];
        }
    };
    auto split = [&] {
        if constexpr (TERMS == 3) {
#pragma unroll
            for (int n = 0; n < NA; ++n) {
                const uint32_t v[4] = {RA[n].x, RA[n].y, RA[n].z, RA[n].w};
                uint32_t t[3][4];
#pragma unroll
                for (int i = 0; i < 4; ++i) split3(__uint_as_float(v[i]), t[0][i], t[1][i], t[2][i]);
#pragma unroll
                for (int x = 0; x < 3; ++x) RT[n][x] = make_uint2(hi16x2(t[x][0], t[x][1]), hi16x2(t[x][2], t[x][3]));
            }
        }
    };
    auto store_a = [&](int buf) {
        char *A = lds + buf * kStage + kW;
#pragma unroll
        for (int n = 0; n < NA; ++n) {
            const int row = arow0 + n * RPI;
            if (BM / 8 / RPI > 0 || row < BM) {
                if constexpr (TERMS == 1) {
                    *reinterpret_cast<uint4 *>(A + row * 128 + ((ac ^ (row & 7)) << 4)) = RA[n];
                } else {
                    char *p = A + row * 128 + (((ac >> 1) ^ (row & 7)) << 4) + (ac & 1) * 8;
#pragma unroll
                    for (int x = 0; x < 3; ++x) *reinterpret_cast<uint2 *>(p + x * kA) = RT[n][x];
                }
            }
        }
    };

    f32x4 acc[NT][MT];
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int i = 0; i < MT; ++i) acc[j][i] = f32x4{0.f, 0.f, 0.f, 0.f};
    // Few tokens (BM 32, where registers are free): each step's sum of 64 products goes into a
    // sum of eight steps and that into the total, and the second and third terms have sums of
    // their own, so a long K rounds no more than the one-token row kernels' trees do.
    constexpr bool kFold = WM == 1;
    constexpr int FN = kFold ? NT : 1, FM = kFold ? MT : 1;
    f32x4 tot[FN][FM], mid[FN][FM], lo[FN][FM];
    if constexpr (kFold) {
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int i = 0; i < MT; ++i) tot[j][i] = mid[j][i] = lo[j][i] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    auto fold = [](f32x4 (&from)[NT][MT], f32x4 (&to)[NT][MT]) {
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int i = 0; i < MT; ++i) to[j][i] += from[j][i], from[j][i] = f32x4{0.f, 0.f, 0.f, 0.f};
    };
    bf16x8 wv[NT], av[TERMS][MT];
    auto read = [&](int buf, int kk) {
        const char *W = lds + buf * kStage + (wn * NT * 16 + r16) * 128;
        const char *A = lds + buf * kStage + kW + (wm * MT * 16 + r16) * 128;
        const int c = ((4 * kk + q) ^ (r16 & 7)) << 4;
#pragma unroll
        for (int j = 0; j < NT; ++j) wv[j] = *reinterpret_cast<const bf16x8 *>(W + j * 2048 + c);
#pragma unroll
        for (int t = 0; t < TERMS; ++t)
#pragma unroll
            for (int i = 0; i < MT; ++i) av[t][i] = *reinterpret_cast<const bf16x8 *>(A + t * kA + i * 2048 + c);
    };
    auto multiply = [&](auto swap) {
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int t = TERMS - 1; t >= 0; --t)
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int i = 0; i < MT; ++i) {
                    f32x4 &c = kFold && t ? lo[kFold ? j : 0][kFold ? i : 0] : acc[j][i];
                    c = swap ? __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[t][i], wv[j], c, 0, 0, 0)
                             : __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv[j], av[t][i], c, 0, 0, 0);
                }
        __builtin_amdgcn_s_setprio(0);
    };
    auto phase = [&] {
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
    };
    // Two groups of four waves, one wave of each per SIMD, run half a beat apart: while one
    // multiplies (and splits the fp32 values it loaded), the other reads its next operands
    // from LDS and stores its part of the next step, so the matrix cores do not wait for LDS.
    // A buffer is overwritten at the earliest one barrier after its last read and read at the
    // earliest one barrier after its last store.
    const bool late = wave >= 4;
    load_w(0);
    load_a(0);
    store_w(0);
    split();
    store_a(0);
    load_w(1);
    load_a(1);
    phase();
    if (late) phase();
    auto steps = [&](auto swap) {
        for (int S = 0; S < NS; ++S) {
            const int buf = S & 1;
            read(buf, 0);
            store_w(buf ^ 1);
            load_w(S + 2);
            phase();
            split();
            multiply(swap);
            phase();
            read(buf, 1);
            store_a(buf ^ 1);
            load_a(S + 2);
            phase();
            multiply(swap);
            if constexpr (kFold) {
                fold(acc, mid);
                if ((S & 7) == 7) fold(mid, tot);
            }
            phase();
        }
    };
    if constexpr (KV) {
        if (wn)  // (uniform per wave; both sides meet the same barriers)
            steps(std::true_type{});
        else
            steps(std::false_type{});
    } else {
        steps(std::false_type{});
    }
    if (!late) phase();
    if constexpr (kFold) {
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int i = 0; i < MT; ++i) acc[j][i] = (tot[j][i] + mid[j][i]) + lo[j][i];
    }

    if constexpr (KV) {
        static_assert(WN == 2, "one wave column per half of a head's rows");
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            const int mt0 = m0 + (wm * MT + i) * 16, key = mt0 + (wn ? 4 * q : r16);
            if (key < a.tpad) {
#pragma unroll
                for (int j = 0; j < NT; ++j) {
                    uint32_t t[3][4];
#pragma unroll
                    for (int x = 0; x < 4; ++x) split3_near(acc[j][i][x], t[0][x], t[1][x], t[2][x]);
#pragma unroll
                    for (int x = 0; x < 3; ++x) {
                        uint16_t *dst = wn ? a.vt + mla_v_index(ntile, a.tpad, x, 16 * j + r16, mt0) + q * 8
                                           : a.kp + mla_k_index(ntile, a.tpad, key, x) + 16 * j + 4 * q;
                        *reinterpret_cast<uint2 *>(dst) = make_uint2(hi16x2(t[x][0], t[x][1]), hi16x2(t[x][2], t[x][3]));
                    }
                }
            }
        }
        return;
    }

    // ---- lane: outputs n0 + 16 j + 4q .. + 3 of token r16
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        const int m = m0 + (wm * MT + i) * 16 + r16;
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            const int nl = (wn * NT + j) * 16 + 4 * q, n = n0 + nl;
            f32x4 v = acc[j][i];
            if (a.ksplit > 1) {
                *reinterpret_cast<f32x4 *>(a.part + ((static_cast<int64_t>(ks) * a.mt * BM + m) * a.nt + ntile) * kBN + nl) = v;
            } else if (m < a.M) {
                const int64_t o = static_cast<int64_t>(m) * N + n;
                float *out = a.out[sg] + o;
                if ((N & 3) == 0) {
                    if (n < N) {
                        if (a.add) v += *reinterpret_cast<const f32x4 *>(a.add + o);
                        *reinterpret_cast<f32x4 *>(out) = v;
                    }
                } else {
#pragma unroll
                    for (int x = 0; x < 4; ++x)
                        if (n + x < N) out[x] = v[x] + (a.add ? a.add[o + x] : 0.f);
                }
            }
        }
    }
}

// The K pieces' partial sums, added in order: one thread per four outputs of a token.
__global__ __launch_bounds__(256) void dense_reduce_kernel(DenseArgs a, int mpad) {
    const int cols = a.nt * (kBN / 4);
    const int64_t id = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (id >= static_cast<int64_t>(a.M) * cols) return;
    const int m = static_cast<int>(id / cols), c = static_cast<int>(id % cols), ntile = c / (kBN / 4);
    int sg = 0;
    for (int i = 1; i < a.nseg; ++i) sg = ntile >= a.t0[i] ? i : sg;
    const int N = a.N[sg], n = c * 4 - a.t0[sg] * kBN;
    if (n >= N) return;
    const f32x4 *p = reinterpret_cast<const f32x4 *>(a.part) + static_cast<int64_t>(m) * cols + c;
    f32x4 v = p[0];
    for (int s = 1; s < a.ksplit; ++s) v += p[static_cast<int64_t>(s) * mpad * cols];
    const int64_t o = static_cast<int64_t>(m) * N + n;
#pragma unroll
    for (int x = 0; x < 4; ++x)
        if (n + x < N) a.out[sg][o + x] = v[x] + (a.add ? a.add[o + x] : 0.f);
}

struct Plan {
    int bm, mt, ksplit, ksteps;
};
// BM: the smallest tile that takes M in one, 128 (bf16 a: 256) above.  ksplit: enough blocks
// for every CU, in pieces of at least four steps.  A tile is never shared by two blocks once there
// are more than 128, so 1000 tokens against 8192 + 1536 + 576 rows are 164 blocks (64% of the CUs),
// 700 against 7168 168, 256 against 4 x 12,288 192, 1000 against 12,288 384 in two turns (75%).
Plan make_plan(int64_t M, int64_t K, int nt, bool f32) {
    Plan p{};
    p.bm = M <= 32 ? 32 : (M <= 64 ? 64 : (M <= 128 || f32 ? 128 : 256));
    p.mt = static_cast<int>(cdiv(M, p.bm));
    const int steps = static_cast<int>(cdiv(K, kBK)), tiles = p.mt * nt;
    int s = std::max(1, std::min(kTargetBlocks / tiles, steps / 4));
    p.ksteps = static_cast<int>(cdiv(steps, s));
    p.ksplit = static_cast<int>(cdiv(steps, p.ksteps));
    return p;
}

template <int TERMS, int WM, int MT, bool KV = false>
int launch_dense(const DenseArgs &a, hipStream_t st) {
    constexpr int BM = WM * MT * 16, bytes = 2 * (kBN * 128 + TERMS * BM * 128);
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void *>(&dense_kernel<TERMS, WM, MT, KV>),
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    int rc = check_hip(attr, "dense: LDS size attribute");
    if (rc) return rc;
    const int64_t total = static_cast<int64_t>(a.mt) * a.nt * a.ksplit;
    dense_kernel<TERMS, WM, MT, KV><<<dim3(static_cast<unsigned>(8 * cdiv(total, 8))), kThreads, bytes, st>>>(a);
    rc = check_hip(hipGetLastError(), "dense launch");
    if (rc || a.ksplit == 1) return rc;
    const int64_t threads = static_cast<int64_t>(a.M) * a.nt * (kBN / 4);
    dense_reduce_kernel<<<dim3(static_cast<unsigned>(cdiv(threads, 256))), 256, 0, st>>>(a, a.mt * BM);
    return check_hip(hipGetLastError(), "dense reduction launch");
}

int count_tiles(const int64_t *N, int nseg) {
    int64_t t = 0;
    for (int i = 0; i < nseg; ++i) t += cdiv(N[i], kBN);
    return t < (1 << 20) ? static_cast<int>(t) : -1;
}

// ------------------------------------------------------------------ row-wise kernels
// out = w * x * rsqrt(mean(x^2) + eps), one wave per row (KimiRMSNorm, ops.py:11-14).
__global__ __launch_bounds__(256) void rmsnorm_rows_kernel(const float *x, int64_t ldx, const float *w, float eps,
                                                           float *out, int M, int K) {
    const int m = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (m >= M) return;
    const float *xr = x + m * ldx;
    float ss = 0.f;
    for (int k = lane * 4; k < K; k += 256) {
        const float4 v = *reinterpret_cast<const float4 *>(xr + k);
        ss += v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w;
    }
    const float s = 1.0f / sqrtf(wave_sum_all(ss) / K + eps);
    for (int k = lane * 4; k < K; k += 256) {
        const float4 v = *reinterpret_cast<const float4 *>(xr + k), g = *reinterpret_cast<const float4 *>(w + k);
        *reinterpret_cast<float4 *>(out + static_cast<int64_t>(m) * K + k) =
            make_float4(g.x * (v.x * s), g.y * (v.y * s), g.z * (v.z * s), g.w * (v.w * s));
    }
}

// out = act(g, u), four values per thread
__global__ __launch_bounds__(256) void act_rows_kernel(const float *g, const float *u, float *out, int64_t n4, int kind,
                                                       float beta, float lbeta) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (i >= n4) return;
    const float4 a = reinterpret_cast<const float4 *>(g)[i], b = reinterpret_cast<const float4 *>(u)[i];
    reinterpret_cast<float4 *>(out)[i] = make_float4(act_fn(a.x, b.x, kind, beta, lbeta), act_fn(a.y, b.y, kind, beta, lbeta),
                                                     act_fn(a.z, b.z, kind, beta, lbeta), act_fn(a.w, b.w, kind, beta, lbeta));
}

}  // namespace

int mla_expand_kv(const void *lat, int cache_dtype, int64_t ld_lat, const void *kv_b, int64_t Tk, int64_t heads,
                  uint16_t *kp, uint16_t *vt, int64_t tpad, hipStream_t st) {
    DenseArgs d{};
    d.a = lat, d.lda = ld_lat, d.M = static_cast<int>(Tk), d.K = 512;
    d.w[0] = static_cast<const uint16_t *>(kv_b);
    d.N[0] = static_cast<int>(heads * 256);
    d.nt = static_cast<int>(heads), d.nseg = 1, d.ksplit = 1, d.ksteps = 512 / kBK;
    d.kp = kp, d.vt = vt, d.tpad = static_cast<int>(tpad);
    const bool f32 = cache_dtype == K3_F32;
    d.mt = static_cast<int>(cdiv(Tk, 128));
    return f32 ? launch_dense<3, 4, 2, true>(d, st) : launch_dense<1, 4, 2, true>(d, st);
}

}  // namespace k3

using namespace k3;

extern "C" int64_t k3_dense_workspace_size(int64_t M, int64_t K, const int64_t *N, int64_t n_mats, int a_dtype) {
    if (M <= 0 || K <= 0 || !N || n_mats <= 0 || n_mats > kMaxSeg) return 0;
    const int nt = count_tiles(N, static_cast<int>(n_mats));
    if (nt <= 0) return 0;
    const Plan p = make_plan(M, K, nt, a_dtype == K3_F32);
    return p.ksplit > 1 ? static_cast<int64_t>(p.ksplit) * p.mt * p.bm * nt * kBN * 4 : 0;
}

extern "C" int k3_dense(const void *a, int a_dtype, int64_t lda, const void *const *w, void *const *out,
                        const int64_t *N, int64_t n_mats, const float *add, int64_t M, int64_t K, void *workspace,
                        int64_t workspace_bytes, void *stream) {
    if (!a || !w || !out || !N) return set_error(K3_ERR_NULL, "dense: null pointer");
    if (a_dtype != K3_F32 && a_dtype != K3_BF16) return set_error(K3_ERR_DTYPE, "dense: a_dtype %d", a_dtype);
    if (n_mats <= 0 || n_mats > kMaxSeg) return set_error(K3_ERR_SHAPE, "dense: 1 to %d weight matrices", kMaxSeg);
    if (add && n_mats != 1) return set_error(K3_ERR_SHAPE, "dense: an added matrix takes one weight matrix");
    const int es = a_dtype == K3_F32 ? 4 : 2;
    if (M <= 0 || K <= 0 || K % 8 || K > (1 << 20) || M > (1 << 24) || lda < K || (lda * es) % 16 ||
        lda > (1 << 20))
        return set_error(K3_ERR_SHAPE, "dense: M=%lld, K=%lld (a multiple of 8), lda=%lld", (long long)M, (long long)K,
                         (long long)lda);
    DenseArgs d{};
    for (int i = 0; i < n_mats; ++i) {
        if (!w[i] || !out[i]) return set_error(K3_ERR_NULL, "dense: null pointer");
        if (N[i] <= 0 || N[i] > (1 << 24)) return set_error(K3_ERR_SHAPE, "dense: N=%lld", (long long)N[i]);
        if (!aligned16(w[i]) || !aligned16(out[i])) return set_error(K3_ERR_ALIGN, "dense: weights and outputs must be 16-byte aligned");
        d.w[i] = static_cast<const uint16_t *>(w[i]);
        d.out[i] = static_cast<float *>(out[i]);
        d.N[i] = static_cast<int>(N[i]);
        d.t0[i] = i ? d.t0[i - 1] + static_cast<int>(cdiv(N[i - 1], kBN)) : 0;
    }
    if (!aligned16(a) || (add && !aligned16(add))) return set_error(K3_ERR_ALIGN, "dense: a must be 16-byte aligned");
    d.nt = count_tiles(N, static_cast<int>(n_mats));
    if (d.nt <= 0) return set_error(K3_ERR_SHAPE, "dense: too many weight rows");
    const Plan p = make_plan(M, K, d.nt, a_dtype == K3_F32);
    if (static_cast<int64_t>(p.mt) * d.nt * p.ksplit >= (1ll << 30)) return set_error(K3_ERR_SHAPE, "dense: problem too large");
    const int64_t need = p.ksplit > 1 ? static_cast<int64_t>(p.ksplit) * p.mt * p.bm * d.nt * kBN * 4 : 0;
    if (need && (!workspace || workspace_bytes < need || !aligned16(workspace)))
        return set_error(K3_ERR_WORKSPACE, "dense: workspace %lld < %lld bytes", (long long)workspace_bytes, (long long)need);
    d.a = a, d.lda = lda, d.M = static_cast<int>(M), d.K = static_cast<int>(K);
    d.mt = p.mt, d.ksplit = p.ksplit, d.ksteps = p.ksteps, d.nseg = static_cast<int>(n_mats);
    d.add = add, d.part = static_cast<float *>(workspace);
    auto st = static_cast<hipStream_t>(stream);
    if (a_dtype == K3_F32) {
        if (p.bm == 32) return launch_dense<3, 1, 2>(d, st);
        if (p.bm == 64) return launch_dense<3, 2, 2>(d, st);
        return launch_dense<3, 4, 2>(d, st);
    }
    if (p.bm == 32) return launch_dense<1, 1, 2>(d, st);
    if (p.bm == 64) return launch_dense<1, 2, 2>(d, st);
    if (p.bm == 128) return launch_dense<1, 2, 4>(d, st);
    return launch_dense<1, 4, 4>(d, st);
}

extern "C" int k3_rmsnorm_rows(const float *x, int64_t ldx, const float *w, float eps, float *out, int64_t M, int64_t K,
                               void *stream) {
    if (!x || !w || !out) return set_error(K3_ERR_NULL, "rmsnorm: null pointer");
    if (M <= 0 || K <= 0 || K % 4 || ldx < K || ldx % 4 || M > (1 << 24) || K > (1 << 24))
        return set_error(K3_ERR_SHAPE, "rmsnorm: M=%lld, K=%lld (a multiple of 4)", (long long)M, (long long)K);
    if (!aligned16(x) || !aligned16(w) || !aligned16(out)) return set_error(K3_ERR_ALIGN, "rmsnorm: 16-byte alignment");
    rmsnorm_rows_kernel<<<dim3(static_cast<unsigned>(cdiv(M, 4))), 256, 0, static_cast<hipStream_t>(stream)>>>(
        x, ldx, w, eps, out, static_cast<int>(M), static_cast<int>(K));
    return check_hip(hipGetLastError(), "rmsnorm launch");
}

extern "C" int k3_act_rows(const float *g, const float *u, float *out, int64_t n, int act_kind, float beta,
                           float linear_beta, void *stream) {
    if (!g || !u || !out) return set_error(K3_ERR_NULL, "act: null pointer");
    if (act_kind != K3_ACT_SILU && act_kind != K3_ACT_SITU) return set_error(K3_ERR_SHAPE, "act: act_kind");
    if (n <= 0 || n % 4 || n >= (1ll << 38)) return set_error(K3_ERR_SHAPE, "act: n=%lld must be a multiple of 4", (long long)n);
    if (!aligned16(g) || !aligned16(u) || !aligned16(out)) return set_error(K3_ERR_ALIGN, "act: 16-byte alignment");
    act_rows_kernel<<<dim3(static_cast<unsigned>(cdiv(n / 4, 256))), 256, 0, static_cast<hipStream_t>(stream)>>>(
        g, u, out, n / 4, act_kind, beta, linear_beta);
    return check_hip(hipGetLastError(), "act launch");
}
