// MXFP4 matmul for the tokens gathered for one expert (more than a GEMV's four): y[M, N] =
// x[M, K] w[N, K]^T, w E2M1 with one E8M0 scale per 32, on the bf16 matrix cores.
//
// Reference: the Metal kernel takes M tokens in one call (air_llm/kernels/metal/
// mxfp4_matvec.py:89-95).  The GEMV form runs four tokens per launch and reads the weights once
// per launch: at 37 tokens ten launches.
//
// One 32-element group is one K step of v_mfma_f32_16x16x32_bf16: the codes become bf16
// unscaled (exact), bf16 x is exact and fp32 x enters as three bf16 terms whose sum is exact
// (split3), and each group's sum is scaled once by its power-of-two scale as it is added to
// the fp32 total, as in the GEMV.
//
// Block: R weight rows x 16 TT tokens, eight waves, WR over the rows and 8 / WR over the groups of
// a step (their sums meet in LDS at the end).  Operands load line-contiguous into registers, two
// steps ahead, and go through LDS (x in 16-byte chunks XOR-swizzled by the row).  What bounds a
// small call is latency and the x rows every block reads, so R is 16 while that gives less
// than two blocks per CU, else 64.
// Measured: 37 tokens of a [3072 x 3584] projection 51.6 us (ten GEMV launches) -> 8.9 us.  It is
// bound by its chain of steps (seven of 512 elements: barrier, LDS, products) and the 190 KB of
// x every block reads; one step of 256 elements instead of 512: 11.5 against 11.2 us at 64 token
// slots, 48 slots instead of 64 for 37 tokens: 11.2 -> 9.1 us.
#include <algorithm>

#include "k3_common.h"
#include "mxfp4_gemv.h"

namespace k3 {
namespace {

constexpr int kThreads = 512;
constexpr int kMaxScale = 16 * 1024;   // LDS bytes for a block's scale rows
constexpr uint32_t kOob = 0xf0000000u;

template <int TERMS, int WR, int TT>
struct Shape {
    static constexpr int R = 16 * WR, WK = 8 / WR;
    // elements per step: what two steps of x leave room for in LDS (a step costs a barrier and
    // an LDS round trip whatever its length), and one 16-byte weight load per thread
    static constexpr int KC = WR == 4 ? (TERMS == 1 ? 256 : 128)
                                      : TERMS == 1 ? (TT >= 3 ? 512 : 1024) : (TT >= 3 ? 128 : 512 / TT);
    static constexpr int G = KC / 32, GW = G / WK > 0 ? G / WK : 1;  // groups per step, per wave
    static constexpr int XT = 16 * TT * KC * 2;                  // bytes of one x term
    static constexpr int W = R * KC / 2;
    static constexpr int Stage = TERMS * XT + W;
    static constexpr int Acc = 8 * TT * 1024;                    // the waves' sums
    static constexpr int lds(int scale) { return std::max(2 * Stage, Acc) + scale; }
};

template <int TERMS, int WR, int TT>
__global__ __launch_bounds__(kThreads, 2) void mxfp4_gemm_kernel(GemvArgs a) {
    using Sh = Shape<TERMS, WR, TT>;
    constexpr int KC = Sh::KC, G = Sh::G, GW = Sh::GW, WK = Sh::WK;
    extern __shared__ char lds[];
    char *const sc = lds + (2 * Sh::Stage > Sh::Acc ? 2 * Sh::Stage : Sh::Acc);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wr = wave % WR, wk = wave / WR, r16 = lane & 15, q = lane >> 4;
    const int K = static_cast<int>(a.K), KB = K >> 5, NS = (K + KC - 1) / KC;
    const int64_t n0 = static_cast<int64_t>(blockIdx.x) * Sh::R;
    const int m0 = blockIdx.y * 16 * TT;
    const int nrows = static_cast<int>(a.N - n0 < Sh::R ? a.N - n0 : Sh::R), mrows = min(16 * TT, a.M - m0);

    // ---- loads.  x: KC * element size bytes per row and step, 16-byte chunks
    constexpr int ES = TERMS == 1 ? 2 : 4, XC = KC * ES / 16;        // chunks per x row: 32 to 128
    constexpr int XR = kThreads / XC, NX = 16 * TT / XR;             // rows per pass, passes
    const int xc = tid % XC, xr = tid / XC;
    const auto rx = make_rsrc(static_cast<const char *>(a.x) + static_cast<int64_t>(m0) * a.ldx * ES,
                              static_cast<uint32_t>(static_cast<int64_t>(mrows) * a.ldx * ES));
    constexpr int WC = KC / 32;                                      // 16-byte chunks per weight row: 4 to 32
    const int wc = tid % WC, wrow = tid / WC;                        // rows past R: no load
    const uint32_t row_bytes = static_cast<uint32_t>(K >> 1);
    const auto rw = make_rsrc(static_cast<const char *>(a.packed) + n0 * row_bytes, static_cast<uint32_t>(nrows) * row_bytes);
    uint4 RX[2][NX], RW[2];
    auto load = [&](int s, int set) {
        const bool xok = (s * XC + xc) * (16 / ES) < K, wok = wrow < nrows && s * WC + wc < KB;
#pragma unroll
        for (int n = 0; n < NX; ++n) {
            const int row = xr + n * XR;
            RX[set][n] = buf_load16(rx, xok && row < mrows ? static_cast<uint32_t>(row * a.ldx * ES) + (s * XC + xc) * 16u : kOob);
        }
        RW[set] = buf_load16_nt(rw, wok ? wrow * row_bytes + (s * WC + wc) * 16u : kOob);
    };
    auto store = [&](int set, int buf) {
        char *X = lds + buf * Sh::Stage, *W = X + TERMS * Sh::XT;
#pragma unroll
        for (int n = 0; n < NX; ++n) {
            const int row = xr + n * XR;
            const uint4 v = RX[set][n];
            if constexpr (TERMS == 1) {
                *reinterpret_cast<uint4 *>(X + row * (KC * 2) + ((xc ^ (row & 15)) << 4)) = v;
            } else {
                const uint32_t f[4] = {v.x, v.y, v.z, v.w};
                uint32_t t[3][4];
#pragma unroll
                for (int i = 0; i < 4; ++i) split3(__uint_as_float(f[i]), t[0][i], t[1][i], t[2][i]);
                char *p = X + row * (KC * 2) + (((xc >> 1) ^ (row & 15)) << 4) + (xc & 1) * 8;
#pragma unroll
                for (int x = 0; x < 3; ++x)
                    *reinterpret_cast<uint2 *>(p + x * Sh::XT) = make_uint2(hi16x2(t[x][0], t[x][1]), hi16x2(t[x][2], t[x][3]));
            }
        }
        if (wrow < Sh::R) *reinterpret_cast<uint4 *>(W + wrow * (KC / 2) + ((wc ^ (wrow & (WC - 1))) << 4)) = RW[set];
    };
    load(0, 0);
    load(1, 1);
    // all scales of the block's rows: one contiguous run of bytes, copied as aligned dwords
    const uintptr_t s0 = reinterpret_cast<uintptr_t>(a.scales) + static_cast<uintptr_t>(n0) * KB;
    const int sdelta = static_cast<int>(s0 & 3u), sdw = (nrows * KB + sdelta + 3) >> 2;
    const uint32_t *sp = reinterpret_cast<const uint32_t *>(s0 - sdelta);
    for (int i = tid; i < sdw; i += kThreads) reinterpret_cast<uint32_t *>(sc)[i] = sp[i];
    store(0, 0);
    load(2, 0);

    // two sums per output, alternate groups in each, and the waves' sums added pairwise: as
    // little rounding as the GEMV's lane sums and tree
    f32x4 acc[2][TT];
#pragma unroll
    for (int t = 0; t < TT; ++t) acc[0][t] = acc[1][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int wl = wr * 16 + r16;                                    // this lane's weight row
    auto compute = [&](int s, int buf) {
        const char *X = lds + buf * Sh::Stage, *W = X + TERMS * Sh::XT;
#pragma unroll
        for (int j = 0; j < GW; ++j) {
            const int g = wk * GW + j;                               // group of the step
            if (G < WK && g >= G) break;
            if (s * G + g >= KB) break;
            const uint32_t w = *reinterpret_cast<const uint32_t *>(W + wl * (KC / 2) + ((g ^ (wl & (WC - 1))) << 4) + 4 * q);
            const float scale = e8m0_to_f32(static_cast<uint8_t>(sc[sdelta + min(wl, nrows - 1) * KB + s * G + g]));
            const uint4 wv4 = make_uint4(__builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, 1.0f, 0)),
                                         __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, 1.0f, 1)),
                                         __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, 1.0f, 2)),
                                         __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, 1.0f, 3)));
            const bf16x8 wv = __builtin_bit_cast(bf16x8, wv4);
#pragma unroll
            for (int t = 0; t < TT; ++t) {
                const char *p = X + (16 * t + r16) * (KC * 2) + (((4 * g + q) ^ r16) << 4);
                f32x4 v = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int x = TERMS - 1; x >= 0; --x)
                    v = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<const bf16x8 *>(p + x * Sh::XT), wv, v, 0, 0, 0);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    f32x4 &c = acc[GW == 1 ? buf : j & 1][t];
                    c[i] = fmaf(v[i], scale, c[i]);
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    for (int s = 0;; s += 2) {
        __syncthreads();
        compute(s, 0);
        if (s + 1 >= NS) break;
        store(1, 1);
        load(s + 3, 1);
        __syncthreads();
        compute(s + 1, 1);
        if (s + 2 >= NS) break;
        store(0, 0);
        load(s + 4, 0);
    }

    static_assert(WK == 8 || WK == 2, "the sum below");
    // ---- the waves' sums: wave (wr, wk) leaves [wk][wr][t][lane]
    __syncthreads();
    f32x4 *part = reinterpret_cast<f32x4 *>(lds);
#pragma unroll
    for (int t = 0; t < TT; ++t) part[((wk * WR + wr) * TT + t) * 64 + lane] = acc[0][t] + acc[1][t];
    __syncthreads();
    for (int id = tid; id < WR * TT * 64; id += kThreads) {
        constexpr int kStep = WR * TT * 64;
        f32x4 v = part[id] + part[kStep + id];
        if constexpr (WK == 8)
            v = (v + (part[2 * kStep + id] + part[3 * kStep + id])) +
                ((part[4 * kStep + id] + part[5 * kStep + id]) + (part[6 * kStep + id] + part[7 * kStep + id]));
        const int ln = id & 63, t = (id >> 6) % TT, w = (id >> 6) / TT;
        const int64_t n = n0 + w * 16 + (ln & 15);
        if (n < a.N) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int m = m0 + 16 * t + 4 * (ln >> 4) + i;
                if (m < a.M) {
                    if (a.out_bf16)
                        static_cast<uint16_t *>(a.out)[m * a.ldo + n] = f32_to_bf16(v[i]);
                    else
                        static_cast<float *>(a.out)[m * a.ldo + n] = v[i];
                }
            }
        }
    }
}

template <int TERMS, int WR, int TT>
int launch(const GemvArgs &a, hipStream_t st) {
    using Sh = Shape<TERMS, WR, TT>;
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void *>(&mxfp4_gemm_kernel<TERMS, WR, TT>),
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, Sh::lds(kMaxScale));
    const int rc = check_hip(attr, "mxfp4 matmul: LDS size attribute");
    if (rc) return rc;
    const int scale = static_cast<int>((Sh::R * (a.K / 32) + 7 + 15) & ~15);
    mxfp4_gemm_kernel<TERMS, WR, TT><<<dim3(static_cast<unsigned>(cdiv(a.N, Sh::R)), static_cast<unsigned>(cdiv(a.M, 16 * TT))),
                                       kThreads, Sh::lds(scale), st>>>(a);
    return check_hip(hipGetLastError(), "mxfp4 matmul launch");
}

template <int TERMS, int WR>
int launch_tt(const GemvArgs &a, hipStream_t st) {
    if (a.M <= 16) return launch<TERMS, WR, 1>(a, st);
    if (a.M <= 32) return launch<TERMS, WR, 2>(a, st);
    if (a.M <= 48) return launch<TERMS, WR, 3>(a, st);
    return launch<TERMS, WR, 4>(a, st);
}

}  // namespace

// A few tokens of few weights finish sooner in GEMV launches: the matmul stages whole 16-token
// tiles and walks K in one chain of steps, whatever M and N.  The costs are fits in us of launches
// measured over M 5..37, N 64..8192, K 1024..32,704.
// K below 8192 (GEMV / matmul): fp32 x, K = 7168: 5 tokens of 300 rows 9.0 / 17.5, 8 of 1024 rows
// 13.1 / 17.7, 12 of 1024 rows 19.3 / 17.4, 8 of 2048 rows 23.1 / 17.4; K = 1024: 5 of 300 rows
// 5.3 / 5.0.  bf16 x, K = 7168: 5 tokens of 300 rows 6.9 / 8.1, 8 of 300 rows 8.9 / 8.1.
// From 8192 on a GEMV launch takes four tokens up to the K whose activations a block holds
// (gemv_token_tile: fp32 8192, bf16 16,384), then one.  fp32 x: 8 tokens of 300 rows at K = 8192
// 13.2 / 22, 5 tokens of 1024 rows at 12,288 20.3 / 31.2, of 4096 rows 37.6 / 32.7, 8 tokens of
// 300 rows at 16,384 32.9 / 39.9, 12 tokens 48.6 / 40.0.  bf16 x: 5 tokens of 300 rows at 12,288
// 10.0 / 15.3, 8 tokens 12.7 / 15.3, 12 tokens at 16,384 21.1 / 19.0, 5 of 2048 rows there 17.9 / 19.1.
// Of 1195 measured points with K from 8192 on, every one is within 7% of its shorter form.
static bool gemv_sooner(int64_t M, int64_t N, int64_t K, bool x_bf16) {
    if (M > 20 || K < 2048 || (N > 4096 && (x_bf16 || K >= 8192))) return false;
    const double k = static_cast<double>(K);
    if (K < 8192) {
        const double w = static_cast<double>(N) * k, waves = static_cast<double>(cdiv(N, 16 * 256));
        const double per = x_bf16 ? 0.8e-4 + w / 400e9 : 0.95e-4 + w / 95e9;   // of a GEMV, per token and element
        const double step = (x_bf16 ? k / 1500 : k / 500) * static_cast<double>(cdiv(M, 16));
        return 2.0 * static_cast<double>(cdiv(M, 4)) + static_cast<double>(M) * k * per < (3.2 + step) * waves;
    }
    // (rows of a multiple of 4096 elements meet the same memory channels)
    double matmul = x_bf16 ? (4.4 + 0.7e-3 * k) * (K % 4096 ? 1.0 : 1.18) : 3.2 + k / 455;
    if (M > 16) matmul *= x_bf16 ? 1.4 : 1.7;
    const int rows = static_cast<int>(cdiv(N, 1024));       // a GEMV launch's cost steps with these
    if (gemv_token_tile(K, x_bf16) == 1) {
        const double one = x_bf16 ? 3 + 8.5e-5 * k : 3.45 + 4e-5 * k;
        return static_cast<double>(M) * one * (rows == 1 ? 1.0 : rows == 2 ? 1.45 : 2.0) < matmul;
    }
    double four = x_bf16 ? (K == 8192 ? 4.8 : 5.4 + 9e-5 * k) : 6.5;     // a launch of four tokens, of one
    double one = x_bf16 ? (K == 8192 ? 2.7 : 2.4 + 7.5e-5 * k) : 3.5;
    if (rows > 1) four *= rows > 2 ? 2.4 : x_bf16 && K == 8192 ? 1.33 : 1.8, one *= 1.2;
    const int64_t rest = M % 4;
    const double gemv = static_cast<double>(M / 4) * four + (rest ? one + (four - one) * static_cast<double>(rest - 1) / 3 : 0);
    return gemv < matmul;
}

bool mxfp4_gemm_takes(int64_t M, int64_t N, int64_t K, bool x_bf16) {
    return M > 4 && !gemv_sooner(M, N, K, x_bf16) && M <= 64 * 65535 && N <= (1ll << 26) &&   // (2^32 threads a grid dimension)
           16 * (K / 32) + 32 <= kMaxScale && K * 64 * 4 < (1ll << 31);
}

int mxfp4_gemm_launch(const GemvArgs &a, hipStream_t st) {
    const bool wide = 64 * (a.K / 32) + 32 <= kMaxScale && cdiv(a.N, 16) * cdiv(a.M, 64) >= 2 * 256;
    if (a.x_bf16) return wide ? launch_tt<1, 4>(a, st) : launch_tt<1, 1>(a, st);
    return wide ? launch_tt<3, 4>(a, st) : launch_tt<3, 1>(a, st);
}

}  // namespace k3
