// Grouped routed-expert FFN for many tokens (prefill): every routed (token, slot) pair is
// grouped by expert and each expert runs as a GEMM with M = its token count on the bf16
// matrix cores.  Each expert's MXFP4 weights are read once per 64-token tile; the tiles of an expert
// run side by side on one XCD, so most repeats come from its L2 (2048 tokens over 896 experts, 520
// of them reached, in 845 tiles: 7.0 GB fetched for gate and up, of 6.1 GB of weights).
//
// Reference: LatentMoE.__call__ (air_llm/models/kimi_k3/moe.py:110-132; k3ref
// k3ref/layers.py:241-261): for each distinct routed expert, gather its tokens, run
// expert_forward, scale by the gate weight and add into y.  The reference loops over
// experts on the host; here:
//
//   count    block e counts the pairs routed to expert e                      -> counts[E]
//   plan     one block: exclusive scan of the counts (segment bases) and the list of
//            64-row tiles of every non-empty expert
//   place    block e writes its pairs, in (token, slot) order, into perm[base_e ...]
//   split_x  (fp32 x only) x -> two bf16 terms, hi + lo, about 16 significant bits
//   gateup   block (tile, 128 intermediate indices): gate and up rows against the tile's
//            tokens; act = f(gate, up) in fp32, stored as two bf16 terms (16 bits)
//   down     block (tile, 256 output rows): the same against the two act terms
//            -> fp32 rows per (token, slot) pair
//   combine  y[t] = sum_slot w[t, slot] * y_pair[t, slot], slots in order
//
// Numerics: an E2M1 code times its E8M0 scale is a bf16 value, so the weights enter the
// bf16 MFMA exactly; bf16 x is exact, and fp32 operands keep 16 bits in two terms.  Products
// are exact and accumulate in fp32.  Deterministic: no atomics, fixed summation orders.
#include <algorithm>

#include "k3_common.h"
#include "moe_common.h"

namespace k3 {
namespace {

constexpr int kTM = 64;        // grouped rows (tokens) per tile: four 16-column MFMA tiles

struct GroupArgs {
    const int32_t *idx;    // [P] expert id of pair p = t * k + slot
    int P, E;
    int32_t *counts;       // [E]
    int32_t *base;         // [E]
    int32_t *perm;         // [P]: pairs grouped by expert
    int4 *tiles;           // [max_tiles]: (expert, its first tile, its pairs, its first grouped row)
    int32_t *n_tiles;      // [1]
    int max_tiles;
};

// Stable compaction of the pairs equal to `e`, by one 1024-thread block: wave w scans the
// contiguous range [w * span, (w + 1) * span) of the pairs with ballots, kScanLoads ids per
// lane in flight at once and no barrier inside the scan; the waves' hit counts meet in LDS
// once, and the writing pass places wave w's hits after those of waves 0 .. w - 1, so the
// pairs keep their ascending order.  (One barrier per 256 pairs, one id load per lane at a
// time, ran 28-34 us at 16,384 pairs.)  Returns the block's total.
constexpr int kScanThreads = 1024;
constexpr int kScanWaves = kScanThreads / 64;
constexpr int kScanLoads = 16;  // ids per lane in flight
template <bool WRITE>
__device__ int scan_expert(const GroupArgs &g, int e, int32_t *out) {
    __shared__ int wcnt[kScanWaves];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int span = (g.P + kScanWaves * 64 - 1) / (kScanWaves * 64) * 64;  // a multiple of 64
    const int lo = wave * span, hi = min(g.P, lo + span);
    // one pass over the wave's range; hits(u, mask) for each group of 64 pairs in order
    auto pass = [&](auto &&hits) {
        for (int p0 = lo; p0 < hi; p0 += 64 * kScanLoads) {
            int v[kScanLoads];
#pragma unroll
            for (int u = 0; u < kScanLoads; ++u) {
                const int p = p0 + 64 * u + lane;
                v[u] = p < hi ? g.idx[p] : -1;
            }
#pragma unroll
            for (int u = 0; u < kScanLoads; ++u) hits(p0 + 64 * u + lane, v[u] == e, __ballot(v[u] == e));
        }
    };
    int cnt = 0;
    pass([&](int, bool, uint64_t m) { cnt += __popcll(m); });
    if (lane == 0) wcnt[wave] = cnt;
    __syncthreads();
    int before = 0, total = 0;
#pragma unroll
    for (int w = 0; w < kScanWaves; ++w) {
        before += w < wave ? wcnt[w] : 0;
        total += wcnt[w];
    }
    if (WRITE) {
        pass([&](int p, bool hit, uint64_t m) {
            if (hit) out[before + __popcll(m & ((1ull << lane) - 1ull))] = p;
            before += __popcll(m);
        });
    }
    return total;
}

__global__ __launch_bounds__(kScanThreads) void group_count_kernel(GroupArgs g) {
    const int n = scan_expert<false>(g, blockIdx.x, nullptr);
    if (threadIdx.x == 0) g.counts[blockIdx.x] = n;
}

__global__ __launch_bounds__(kScanThreads) void group_place_kernel(GroupArgs g) {
    scan_expert<true>(g, blockIdx.x, g.perm + g.base[blockIdx.x]);
}

// One block of 1024 threads: segment bases and the tile list (E <= 1024).
__global__ __launch_bounds__(1024) void group_plan_kernel(GroupArgs g) {
    __shared__ int sc[1024], st[1024];
    const int e = threadIdx.x;
    const int c = e < g.E ? g.counts[e] : 0;
    sc[e] = c;
    st[e] = (c + kTM - 1) / kTM;
    __syncthreads();
    for (int off = 1; off < 1024; off <<= 1) {  // inclusive Hillis-Steele scans
        const int a = e >= off ? sc[e - off] : 0, b = e >= off ? st[e - off] : 0;
        __syncthreads();
        sc[e] += a;
        st[e] += b;
        __syncthreads();
    }
    if (e < g.E) {
        g.base[e] = sc[e] - c;
        const int t0 = st[e] - (c + kTM - 1) / kTM;
        for (int j = 0; j * kTM < c; ++j)
            if (t0 + j < g.max_tiles) g.tiles[t0 + j] = make_int4(e, t0, c, sc[e] - c);
    }
    if (e == 1023) *g.n_tiles = min(st[1023], g.max_tiles);
}

// ------------------------------------------------------------------ bf16 terms
// hi + lo of an fp32 value: hi rounded to nearest, lo the rounded remainder (zero where hi
// is not finite, so an infinity stays one).
__device__ __forceinline__ void bf16_split2(float v, uint16_t &hi, uint16_t &lo) {
    hi = f32_to_bf16(v);
    const float h = bf16_to_f32(hi);
    lo = (hi & 0x7f80u) == 0x7f80u ? 0 : f32_to_bf16(v - h);
}

// The activation of moe_common.h's act_fn in straight-line code on the hardware's exp2 and
// reciprocal (each within one unit in the last place).  The exponent's rounding enters the result
// by its size: about 1e-6 relative up to |x| of 20, 4e-6 at 80, against the 2^-17 (7.6e-6) that the
// two-term storage keeps.
__device__ __forceinline__ float fast_sigmoid(float x) {
    return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * x));
}
__device__ __forceinline__ float fast_tanh(float x) {
    const float a = fabsf(x), e = __builtin_amdgcn_exp2f(-2.8853900817779268f * a), s = x * x;
    // below 1/4 the difference 1 - e cancels: the Taylor polynomial, next term 2e-2 x^8
    const float p = x * (1.0f + s * (-0.33333333f + s * (0.13333333f - s * 0.053968254f)));
    return a < 0.25f ? p : copysignf((1.0f - e) * __builtin_amdgcn_rcpf(1.0f + e), x);
}
__device__ __forceinline__ float fast_act(float g, float u, int kind, float beta, float ibeta, float lbeta, float ilbeta) {
    if (kind == K3_ACT_SITU) {
        const float a = beta * fast_tanh(g * ibeta) * fast_sigmoid(g);
        return a * (lbeta > 0.f ? lbeta * fast_tanh(u * ilbeta) : u);
    }
    return g * fast_sigmoid(g) * u;
}

// A two-term row: per 128 elements, 128 hi values then 128 lo values (512 bytes), so one
// staging step of the GEMM reads 512 contiguous bytes per row in either form.
constexpr int kBlk = 128;

struct SplitArgs {
    const float *x;      // [T, H]
    uint16_t *xt;        // [T][Hblk][2][128]
    int T, H, Hblk;
};

__global__ __launch_bounds__(256) void split_x_kernel(SplitArgs a) {
    const int eighths = a.H >> 3;
    const int64_t idx = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (idx >= static_cast<int64_t>(a.T) * eighths) return;
    const int64_t t = idx / eighths;
    const int k = static_cast<int>(idx % eighths) * 8;
    const float4 *src = reinterpret_cast<const float4 *>(a.x + t * a.H + k);
    const float4 f0 = src[0], f1 = src[1];
    const float v[8] = {f0.x, f0.y, f0.z, f0.w, f1.x, f1.y, f1.z, f1.w};
    uint32_t hi[4], lo[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        uint16_t h0, l0, h1, l1;
        bf16_split2(v[2 * i], h0, l0);
        bf16_split2(v[2 * i + 1], h1, l1);
        hi[i] = h0 | (static_cast<uint32_t>(h1) << 16);
        lo[i] = l0 | (static_cast<uint32_t>(l1) << 16);
    }
    uint16_t *dst = a.xt + (t * a.Hblk + (k >> 7)) * (2 * kBlk) + (k & 127);
    *reinterpret_cast<uint4 *>(dst) = make_uint4(hi[0], hi[1], hi[2], hi[3]);
    *reinterpret_cast<uint4 *>(dst + kBlk) = make_uint4(lo[0], lo[1], lo[2], lo[3]);
}

// ------------------------------------------------------------------ grouped GEMMs
struct GemmArgs {
    const void *b;           // B rows: bf16 x [T, K], or two-term rows [., Kblk, 2, 128]
    uint32_t b_bytes;        // size of all B rows (gate/up)
    uint32_t brow;           // bytes per B row
    const uint64_t *table;   // [E][6] expert pointers
    const int32_t *perm, *n_tiles;
    const int4 *tiles;
    uint16_t *act;           // gate/up output: two-term rows [P, Iblk, 2, 128]
    uint32_t act_row;        // bytes per act row
    float *ypair;            // down output [P, N]: row = pair id
    int K, N, NT;            // reduction length, weight rows of one projection, row blocks
    int top_k, act_kind;
    float beta, lbeta;
};

// The GEMM streams weights, so it is bound by HBM as long as the operands reach the matrix
// cores without extra traffic.  What decides that on this chip is the lane order of the
// loads: adjacent lanes on one 128-byte line reach 48 B/clk per CU from L2, while the MFMA
// operand order loaded straight from memory (adjacent lanes on different rows) makes one
// L1 request per lane and stops at 16 B/clk per CU.  So every operand is loaded
// line-contiguous into registers, two steps ahead, and turned into operand order through
// LDS, in 16-byte chunks XOR-swizzled by the row so neither the stores nor the operand
// reads meet bank conflicts:
//   A  256 weight rows x 256 elements (128 bytes a row: one line), double buffered
//   B  64 token rows x 512 bytes (256 elements, or 128 of two terms), double buffered
//   S  256 rows x 32 scale bytes, one load per four steps, double buffered
// 144 KB of LDS, one block of eight waves per CU.  Waves w and w + 4 own the same 64 weight
// rows and split the reduction (their sums meet in LDS at the end), so no wave converts or
// reads what another one does.  Weights become bf16 in registers (4 v_cvt per 8 values of
// a row, reused by the tile's column groups and both terms).
// Measured (2048 tokens, 896 experts top-16, latent 3584 / 3072; the former form fed the scaled
// FP4 x FP8 MFMA in operand order): gate/up 4470 -> 2790 us, down 2366 -> 1970 us; 700 tokens over
// 384 experts: 1850 -> 1340 and 1208 -> 960 us under the profiler.  What bounds it now: a step costs a barrier, the
// LDS round trip and the products in turn, 1.2 us at one column group (its weights take 1.2 us
// of HBM), 1.6 at three, 1.9 at four (matrix cores busy 28% in gate/up, 39% in down).  Measured
// and not kept: the two wave groups half a beat apart (gate/up 3030 -> 3940 us: too little work
// between barriers), sixteen waves of 32 rows (B is read twice as often from LDS: 2720 -> 3800
// us), persistent blocks that read the next tile's record and first lines ahead (3030 -> 3740
// us, static shares), non-temporal weight loads (no change), loads one step further ahead at
// three column groups (no change).
constexpr int kThreads = 512;
constexpr uint32_t kOob = 0xf0000000u;      // past every buffer size the host lets through
constexpr int kABuf = 256 * 128, kBBuf = 64 * 512, kSBuf = 256 * 32;
constexpr int kLdsB = 2 * kABuf, kLdsS = kLdsB + 2 * kBBuf;
constexpr int kLds = kLdsS + 2 * kSBuf;

__device__ __forceinline__ bf16x8 fp4x8_bf16(uint32_t w, float s) {
    const uint4 v = make_uint4(__builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, s, 0)),
                               __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, s, 1)),
                               __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, s, 2)),
                               __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, s, 3)));
    return __builtin_bit_cast(bf16x8, v);
}

// DOWN == false: gate/up + activation; A rows 0..127 of the block are gate rows, 128..255
// the up rows of the same intermediate indices, and wave w % 4 owns 32 of both, so the
// activation of a (token, index) pair meets both products in one lane.
// DOWN == true: 256 rows of W_down, 64 per wave.
// TERMS: bf16 terms of B (bf16 x: 1; fp32 x and act: 2).  NCT: 16-column groups in use.
template <bool DOWN, int TERMS, int NCT>
__device__ __forceinline__ void grouped_tile(const GemmArgs &a, char *lds, int nt, int rows, int pos0,
                                             const uint64_t *ptr) {
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wr = wave & 3, kg = wave >> 2;
    const int r16 = lane & 15, q = lane >> 4;
    const int KB = a.K >> 5;                     // 32-element groups per weight row
    const int NS = (a.K + 255) >> 8;

    // ---- loads: A and S by wave w for block rows 32 w .. + 31, B for token rows 8 w .. + 7
    const int proj = DOWN ? 4 : (wave < 4 ? 0 : 2);
    const uint32_t rowA = static_cast<uint32_t>(a.K >> 1);
    const auto ra = make_rsrc(uniform_ptr(ptr[proj]), static_cast<uint32_t>(a.N) * rowA);
    // scale rows have any alignment: five aligned dwords hold the 16 bytes at any byte offset
    const uintptr_t sbase = reinterpret_cast<uintptr_t>(uniform_ptr(ptr[proj + 1]));
    const uint32_t sdelta = static_cast<uint32_t>(sbase & 3u);
    const auto rs = make_rsrc(reinterpret_cast<const void *>(sbase - sdelta),
                              (static_cast<uint32_t>(a.N * KB) + sdelta + 3u) & ~3u);
    const int grow0 = DOWN ? nt * 256 + wave * 32 : nt * 128 + (wave & 3) * 32;  // weight row of block row 32 w
    const int ac = lane & 7;                     // 16-byte chunk of the 128-byte line
    uint32_t aoff[4];
#pragma unroll
    for (int n = 0; n < 4; ++n) {
        const int row = grow0 + 8 * n + (lane >> 3);
        aoff[n] = row < a.N ? static_cast<uint32_t>(row) * rowA + ac * 16u : kOob;
    }
    const int srow = grow0 + (lane >> 1);
    const uint32_t soff = srow < a.N ? static_cast<uint32_t>(srow * KB) + (lane & 1) * 16u + sdelta : kOob;
    const auto rb = DOWN ? make_rsrc(static_cast<const char *>(a.b) + static_cast<int64_t>(pos0) * a.brow,
                                     static_cast<uint32_t>(rows) * a.brow)
                         : make_rsrc(a.b, a.b_bytes);
    const int bc = lane & 31;                    // 16-byte chunk of the 512 bytes
    const int brow0 = wave * 2 * NCT + (lane >> 5);  // NCT row pairs per wave
    uint32_t boff[NCT];
#pragma unroll
    for (int n = 0; n < NCT; ++n) {
        const int rr = brow0 + 2 * n;
        const int src = DOWN ? rr : a.perm[pos0 + min(rr, rows - 1)] / a.top_k;
        boff[n] = rr < rows ? static_cast<uint32_t>(src) * a.brow + bc * 16u : kOob;
    }
    // register sets: loads run one or two steps ahead of their stores; a step of three or four
    // column groups computes longer than a load takes, and its sums need the registers
    constexpr int D = NCT >= 3 ? 1 : 2;
    uint4 RA[D][4], RB[D][NCT], RS;
    uint32_t RS4;
    auto load_a = [&](int S, int set) {
        const bool ok = S * 8 + ac < KB;
#pragma unroll
        for (int n = 0; n < 4; ++n) RA[set][n] = buf_load16(ra, ok ? aoff[n] + S * 128u : kOob);
    };
    auto load_b = [&](int u, int set) {
        const bool ok = TERMS == 1 ? u * 32 + bc < (a.K >> 3) : u * 16 + (bc & 15) < (a.K >> 3);
#pragma unroll
        for (int n = 0; n < NCT; ++n) RB[set][n] = buf_load16(rb, ok ? boff[n] + u * 512u : kOob);
    };
    auto load_s = [&](int G) {
        const uint32_t off = (soff + G * 32u) & ~3u;
        RS = buf_load16(rs, off);
        RS4 = buf_load4(rs, off + 16u);
    };
    // LDS row of A: 16-byte unit p = 4 kg + q holds what lane (., q) of wave group kg takes in
    // the step, dwords 2kg, 2kg + 1 of groups q and 4 + q.
    // The XOR keys: a 16-byte LDS read runs 16 lanes at a time over all 64 banks, lanes 0-3,
    // 12-15 and 20-27 together (and 4-11, 16-19, 28-31), so the operand rows 0-3, 12-15 of one
    // q meet rows 4-11 of the next q.  akey sends both sets to different units, and
    // neighbouring row pairs' 8-byte stores to different halves; bkey does it for B's rows,
    // whose chunks of neighbouring q are 4 apart.  (3-bit keys of the row: 2-way conflicts,
    // 124 instead of 228 B/clk.)
    auto akey = [](int R) { return ((R & 2) << 1) | (((R >> 2) ^ (R >> 3)) & 1) << 1 | ((R >> 3) & 1); };
    auto bkey = [](int R) { return (((R >> 2) ^ (R >> 3)) & 1) << 3 | ((R >> 3) & 1) << 2 | (R & 3); };
    auto store_a = [&](int set, int buf) {
#pragma unroll
        for (int n = 0; n < 4; ++n) {
            const int R = wave * 32 + 8 * n + (lane >> 3);
            char *row = lds + buf * kABuf + R * 128 + (ac >> 2) * 8;
            *reinterpret_cast<uint2 *>(row + (((ac & 3) ^ akey(R)) << 4)) = make_uint2(RA[set][n].x, RA[set][n].y);
            *reinterpret_cast<uint2 *>(row + (((4 + (ac & 3)) ^ akey(R)) << 4)) = make_uint2(RA[set][n].z, RA[set][n].w);
        }
    };
    auto store_b = [&](int set, int buf) {
#pragma unroll
        for (int n = 0; n < NCT; ++n) {
            const int rr = brow0 + 2 * n;
            *reinterpret_cast<uint4 *>(lds + kLdsB + buf * kBBuf + rr * 512 + ((bc ^ bkey(rr)) << 4)) = RB[set][n];
        }
    };
    // 32 scale bytes per row and four steps, as [q][step][h]: a lane reads its eight in one
    // 8-byte load.  Bytes past the row's end become zero (they meet zero weights, and must
    // not hold another row's infinity).
    auto store_s = [&](int G) {
        const uint32_t sh = soff & 3u;
        uint32_t v[4] = {__builtin_amdgcn_alignbyte(RS.y, RS.x, sh), __builtin_amdgcn_alignbyte(RS.z, RS.y, sh),
                         __builtin_amdgcn_alignbyte(RS.w, RS.z, sh), __builtin_amdgcn_alignbyte(RS4, RS.w, sh)};
        const int left = KB - G * 32 - (lane & 1) * 16;
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            const int n = max(min(left - 4 * d, 4), 0);
            v[d] &= n == 4 ? ~0u : (1u << (8 * n)) - 1u;
        }
        char *row = lds + kLdsS + (G & 1) * kSBuf + (tid >> 1) * 32 + (lane & 1) * 4;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            // bytes i of the step's groups 0-3 and 4-7, for two steps
            const uint32_t lo = __builtin_amdgcn_perm(v[1], v[0], 0x0c0c0400u + 0x0101u * i);
            const uint32_t hi = __builtin_amdgcn_perm(v[3], v[2], 0x0c0c0400u + 0x0101u * i);
            *reinterpret_cast<uint32_t *>(row + i * 8) = lo | (hi << 16);
        }
    };

    f32x4 acc[4][NCT];
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int ct = 0; ct < NCT; ++ct) acc[j][ct] = f32x4{0.f, 0.f, 0.f, 0.f};
    int arow[4];                                 // block row of this lane in each 16-row tile
#pragma unroll
    for (int j = 0; j < 4; ++j)
        arow[j] = (DOWN ? wr * 64 + j * 16 : (j >> 1) * 128 + wr * 32 + (j & 1) * 16) + r16;

    // Lane (r16, q) holds weight row r16's 32-element group 4h + q of the step; MFMA i takes
    // its elements 8i .. 8i + 7 (one dword), against the same elements of the tokens.  Wave
    // group kg takes i = 2kg, 2kg + 1 in both forms, so bf16 x gives the sums that fp32 x
    // with the same values gives.
    uint32_t sw[4][2];                           // this lane's scale bytes of four steps
    auto read_s = [&](int G) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint2 v = *reinterpret_cast<const uint2 *>(lds + kLdsS + (G & 1) * kSBuf + arow[j] * 32 + q * 8);
            sw[j][0] = v.x, sw[j][1] = v.y;
        }
    };
    uint4 wv[4];                                 // this lane's weights of the step: two groups' halves
    auto read_a = [&](int abuf) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
            wv[j] = *reinterpret_cast<const uint4 *>(lds + abuf * kABuf + arow[j] * 128 +
                                                     (((4 * kg + q) ^ akey(arow[j])) << 4));
    };
    auto compute = [&](int P, int h, int bbuf) {
        const char *B = lds + kLdsB + bbuf * kBBuf;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            bf16x8 av[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t w4[4] = {wv[j].x, wv[j].y, wv[j].z, wv[j].w};
                const int byte = (2 * P + h) & 3;
                const uint32_t s4 = sw[j][P >> 1];
                // the conversion takes the scale's exponent bits
                const float sc = __uint_as_float((byte == 3 ? s4 >> 1 : s4 << (23 - 8 * byte)) & 0x7f800000u);
                av[j] = fp4x8_bf16(w4[2 * h + i], sc);
            }
#pragma unroll
            for (int t = 0; t < TERMS; ++t) {
                const int chunk = 16 * (TERMS == 1 ? h : t) + 4 * q + 2 * kg + i;
#pragma unroll
                for (int ct = 0; ct < NCT; ++ct) {
                    const bf16x8 bv = *reinterpret_cast<const bf16x8 *>(B + (ct * 16 + r16) * 512 +
                                                                        ((chunk ^ bkey(r16)) << 4));
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        acc[j][ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[j], bv, acc[j][ct], 0, 0, 0);
                }
            }
        }
    };

    // ---- pipeline: step S computes on buffers S % 2, then stores step S + 1 and issues step
    // S + 1 + D.  (The loads wait in order, so B goes ahead of A: a wait for B leaves the newer
    // A in flight; the fences keep the entry's loads in the loop's order.)
    load_a(0, 0);
    load_s(0);
    load_b(0, 0);
    __builtin_amdgcn_sched_barrier(0);
    if (D == 2) load_b(1, D - 1);
    __builtin_amdgcn_sched_barrier(0);
    if (D == 2) load_a(1, D - 1);
    __builtin_amdgcn_sched_barrier(0);
    store_a(0, 0);
    store_b(0, 0);
    store_s(0);
    __builtin_amdgcn_sched_barrier(0);
    load_b(D, 0);
    __builtin_amdgcn_sched_barrier(0);
    load_a(D, 0);
    __builtin_amdgcn_sched_barrier(0);
    auto step = [&](int S, int P) {
        const int nx = (P + 1) & 1, set = nx & (D - 1);
        __syncthreads();
        if (P == 0) read_s(S >> 2);
        read_a(P & 1);
        if constexpr (TERMS == 1) {
            compute(P, 0, P & 1);
            compute(P, 1, P & 1);
            __builtin_amdgcn_sched_barrier(0);  // the stores wait for loads the sums above cover
            store_b(set, nx);
            load_b(S + 1 + D, set);
        } else {
            compute(P, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            store_b(D - 1, 1);
            load_b(2 * S + 1 + D, D - 1);
            __syncthreads();
            compute(P, 1, 1);
            __builtin_amdgcn_sched_barrier(0);
            store_b(0, 0);
            load_b(2 * S + 2 + D, 0);
        }
        store_a(set, nx);
        if (P == 3) store_s((S >> 2) + 1);
        if (P == 0) load_s((S >> 2) + 1);
        load_a(S + 1 + D, set);
    };
    // (left by break only, so the loop head has one predecessor besides the entry and the
    // compiler's counted waits there stay exact)
    for (int S = 0;; S += 4) {
        step(S, 0);
        if (S + 1 >= NS) break;
        step(S + 1, 1);
        if (S + 2 >= NS) break;
        step(S + 2, 2);
        if (S + 3 >= NS) break;
        step(S + 3, 3);
        if (S + 4 >= NS) break;
    }

    // ---- the two wave groups' sums meet: group kg finishes column groups ct % 2 == kg and
    // hands the others over through LDS
    __syncthreads();
    f32x4 *xch = reinterpret_cast<f32x4 *>(lds);
#pragma unroll
    for (int ct = 0; ct < NCT; ++ct)
        if ((ct & 1) != kg) {
#pragma unroll
            for (int j = 0; j < 4; ++j) xch[((wr * NCT + ct) * 4 + j) * 64 + lane] = acc[j][ct];
        }
    __syncthreads();
    // (C: lane holds weight rows 4q + v of each A tile, column r16 of each column group)
    const float ib = 1.0f / a.beta, il = 1.0f / a.lbeta;
#pragma unroll
    for (int ct = 0; ct < NCT; ++ct) {
        const int rr = ct * 16 + r16;
        if ((ct & 1) == kg && rr < rows) {
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[j][ct] += xch[((wr * NCT + ct) * 4 + j) * 64 + lane];
            if constexpr (DOWN) {
                float *yrow = a.ypair + static_cast<int64_t>(a.perm[pos0 + rr]) * a.N;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int row = nt * 256 + wr * 64 + j * 16 + 4 * q;
                    if (row < a.N) *reinterpret_cast<float4 *>(yrow + row) = __builtin_bit_cast(float4, acc[j][ct]);
                }
            } else if (nt * 128 + wr * 32 < a.N) {
                uint16_t *dst = reinterpret_cast<uint16_t *>(reinterpret_cast<char *>(a.act) +
                                                             static_cast<int64_t>(pos0 + rr) * a.act_row) +
                                nt * (2 * kBlk) + wr * 32 + 4 * q;
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    uint16_t hi[4], lo[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        bf16_split2(fast_act(acc[j][ct][i], acc[j + 2][ct][i], a.act_kind, a.beta, ib, a.lbeta, il), hi[i], lo[i]);
                    *reinterpret_cast<uint2 *>(dst + 16 * j) =
                        make_uint2(hi[0] | (static_cast<uint32_t>(hi[1]) << 16), hi[2] | (static_cast<uint32_t>(hi[3]) << 16));
                    *reinterpret_cast<uint2 *>(dst + kBlk + 16 * j) =
                        make_uint2(lo[0] | (static_cast<uint32_t>(lo[1]) << 16), lo[2] | (static_cast<uint32_t>(lo[3]) << 16));
                }
            }
        }
    }
}

// Block order: the work list is (expert, row block, token tile of the expert), and XCD x
// (blocks b % 8 == x) walks the x-th eighth of it, so the CUs of one XCD read one or two
// experts at a time: neighbouring rows of one weight matrix, the same token rows, and for
// an expert of several tiles the same weight rows, which its L2 then holds.
template <bool DOWN, int TERMS>
__global__ __launch_bounds__(kThreads, 2) void grouped_gemm_kernel(GemmArgs a) {
    extern __shared__ char lds[];
    const int total = *a.n_tiles * a.NT;
    const int per = (total + 7) >> 3, li = blockIdx.x >> 3;
    const int w = (blockIdx.x & 7) * per + li;
    if (li >= per || w >= total) return;
    const int4 rec = a.tiles[w / a.NT];
    const int ne = (rec.z + kTM - 1) / kTM, off = w - rec.y * a.NT;
    const int nt = off / ne, m0 = (off % ne) * kTM;
    const int rows = min(kTM, rec.z - m0), pos0 = rec.w + m0;
    const uint64_t *ptr = a.table + static_cast<int64_t>(rec.x) * 6;
    if (rows > 48)
        grouped_tile<DOWN, TERMS, 4>(a, lds, nt, rows, pos0, ptr);
    else if (rows > 32)
        grouped_tile<DOWN, TERMS, 3>(a, lds, nt, rows, pos0, ptr);
    else if (rows > 16)
        grouped_tile<DOWN, TERMS, 2>(a, lds, nt, rows, pos0, ptr);
    else
        grouped_tile<DOWN, TERMS, 1>(a, lds, nt, rows, pos0, ptr);
}

// More than the default 64 KB of dynamic LDS (gfx950 has 160 KB per CU).
int grouped_prepare() {
    static const hipError_t rc = [] {
        const void *k[3] = {reinterpret_cast<const void *>(&grouped_gemm_kernel<false, 1>),
                            reinterpret_cast<const void *>(&grouped_gemm_kernel<false, 2>),
                            reinterpret_cast<const void *>(&grouped_gemm_kernel<true, 2>)};
        for (const void *f : k) {
            const hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
            if (e != hipSuccess) return e;
        }
        return hipSuccess;
    }();
    return check_hip(rc, "moe grouped: LDS size attribute");
}

// ------------------------------------------------------------------ combine
struct CombineArgs {
    const float *ypair;   // [T * k, H]
    const float *w;       // [T, k]
    void *out;            // [T, H]
    int T, H, k;
    int out_bf16;
};

// grid: (T, cdiv(H, 1024)); thread: 4 consecutive columns
__global__ __launch_bounds__(256) void combine_kernel(CombineArgs a) {
    const int t = blockIdx.x;
    const int c = (blockIdx.y * 256 + threadIdx.x) * 4;
    if (c >= a.H) return;
    float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int j = 0; j < a.k; ++j) {
        const float wj = a.w[t * a.k + j];
        const float4 v = *reinterpret_cast<const float4 *>(a.ypair + static_cast<int64_t>(t * a.k + j) * a.H + c);
        s.x = fmaf(wj, v.x, s.x);
        s.y = fmaf(wj, v.y, s.y);
        s.z = fmaf(wj, v.z, s.z);
        s.w = fmaf(wj, v.w, s.w);
    }
    const int64_t o = static_cast<int64_t>(t) * a.H + c;
    if (a.out_bf16) {
        uint16_t *p = static_cast<uint16_t *>(a.out) + o;
        p[0] = f32_to_bf16(s.x);
        p[1] = f32_to_bf16(s.y);
        p[2] = f32_to_bf16(s.z);
        p[3] = f32_to_bf16(s.w);
    } else {
        *reinterpret_cast<float4 *>(static_cast<float *>(a.out) + o) = s;
    }
}

// ------------------------------------------------------------------ host side
struct GroupedWs {
    size_t counts, base, perm, tiles, n_tiles, xt, act, ypair, total;
    int max_tiles;
    int64_t Hblk, Iblk;   // 128-element blocks of a two-term row
};

GroupedWs grouped_ws_layout(int64_t T, int64_t k, int64_t E, int64_t H, int64_t I) {
    GroupedWs L{};
    auto up = [](size_t v) { return (v + 255) & ~size_t(255); };
    const int64_t P = T * k;
    L.Hblk = cdiv(H, kBlk);
    L.Iblk = cdiv(I, kBlk);
    // every expert in use has at least one pair, and all its tiles but one are full
    L.max_tiles = static_cast<int>(cdiv(P, kTM) + std::min(P, E));
    size_t o = 0;
    L.counts = o, o += up(E * 4);
    L.base = o, o += up(E * 4);
    L.perm = o, o += up(P * 4);
    L.tiles = o, o += up(static_cast<size_t>(L.max_tiles) * sizeof(int4));
    L.n_tiles = o, o += up(4);
    L.xt = o, o += up(static_cast<size_t>(T) * L.Hblk * kBlk * 4);
    L.act = o, o += up(static_cast<size_t>(P) * L.Iblk * kBlk * 4);
    L.ypair = o, o += up(static_cast<size_t>(P) * H * 4);
    L.total = o;
    return L;
}

}  // namespace
}  // namespace k3

using namespace k3;

extern "C" int64_t k3_moe_grouped_workspace_size(int64_t T, int64_t top_k, int64_t n_experts, int64_t H, int64_t I) {
    if (T <= 0 || top_k <= 0 || n_experts <= 0 || H <= 0 || I <= 0) return 0;
    return static_cast<int64_t>(grouped_ws_layout(T, top_k, n_experts, H, I).total);
}

extern "C" int k3_moe_grouped_ffn(const void *x, int x_dtype, const int32_t *expert_idx, const float *expert_w,
                                  const void *expert_table, void *out, int out_dtype, int64_t T, int64_t H, int64_t I,
                                  int64_t n_experts, int64_t top_k, int act_kind, float beta, float linear_beta,
                                  void *workspace, int64_t workspace_bytes, void *stream) {
    if (!x || !expert_idx || !expert_w || !expert_table || !out || !workspace)
        return set_error(K3_ERR_NULL, "moe grouped: null pointer");
    if (x_dtype != K3_BF16 && x_dtype != K3_F32)
        return set_error(K3_ERR_DTYPE, "moe grouped: x must be bf16 or fp32 (x_dtype %d)", x_dtype);
    if (out_dtype != K3_F32 && out_dtype != K3_BF16) return set_error(K3_ERR_DTYPE, "moe grouped: out_dtype");
    if (act_kind != K3_ACT_SILU && act_kind != K3_ACT_SITU) return set_error(K3_ERR_SHAPE, "moe grouped: act_kind");
    if (T <= 0 || top_k <= 0 || top_k > 64 || n_experts <= 0 || n_experts > 1024)
        return set_error(K3_ERR_SHAPE, "moe grouped: T >= 1, 1 <= top_k <= 64, 1 <= n_experts <= 1024 required");
    if (H <= 0 || I <= 0 || H % 64 || I % 64)
        return set_error(K3_ERR_SHAPE, "moe grouped: H=%lld and I=%lld must be positive multiples of 64",
                         (long long)H, (long long)I);
    const GroupedWs L = grouped_ws_layout(T, top_k, n_experts, H, I);
    const int64_t P = T * top_k;
    const int64_t Hpad = cdiv(H, 256) * 256, Ipad = cdiv(I, 256) * 256;
    if (P >= (1ll << 30) || H * I / 2 >= (1ll << 31) || 3 * P * Ipad >= (1ll << 31) || 3 * T * Hpad >= (1ll << 31))
        return set_error(K3_ERR_SHAPE, "moe grouped: problem too large");
    if (workspace_bytes < static_cast<int64_t>(L.total))
        return set_error(K3_ERR_WORKSPACE, "moe grouped: workspace %lld < %zu bytes", (long long)workspace_bytes,
                         L.total);
    if (!aligned16(x) || !aligned16(workspace) || !aligned16(out))
        return set_error(K3_ERR_ALIGN, "moe grouped: x, out and workspace must be 16-byte aligned");
    auto st = static_cast<hipStream_t>(stream);
    char *ws = static_cast<char *>(workspace);

    GroupArgs g{};
    g.idx = expert_idx;
    g.P = static_cast<int>(P);
    g.E = static_cast<int>(n_experts);
    g.counts = reinterpret_cast<int32_t *>(ws + L.counts);
    g.base = reinterpret_cast<int32_t *>(ws + L.base);
    g.perm = reinterpret_cast<int32_t *>(ws + L.perm);
    g.tiles = reinterpret_cast<int4 *>(ws + L.tiles);
    g.n_tiles = reinterpret_cast<int32_t *>(ws + L.n_tiles);
    g.max_tiles = L.max_tiles;
    group_count_kernel<<<dim3(g.E), kScanThreads, 0, st>>>(g);
    group_plan_kernel<<<dim3(1), 1024, 0, st>>>(g);
    group_place_kernel<<<dim3(g.E), kScanThreads, 0, st>>>(g);
    int rc = check_hip(hipGetLastError(), "moe grouped: grouping launches");
    if (rc) return rc;

    rc = grouped_prepare();
    if (rc) return rc;
    const bool xf32 = x_dtype == K3_F32;
    if (xf32) {
        SplitArgs sa{};
        sa.x = static_cast<const float *>(x);
        sa.xt = reinterpret_cast<uint16_t *>(ws + L.xt);
        sa.T = static_cast<int>(T), sa.H = static_cast<int>(H), sa.Hblk = static_cast<int>(L.Hblk);
        split_x_kernel<<<dim3(static_cast<unsigned>(cdiv(T * (H / 8), 256))), 256, 0, st>>>(sa);
        rc = check_hip(hipGetLastError(), "moe grouped: x split launch");
        if (rc) return rc;
    }
    GemmArgs ma{};
    ma.table = static_cast<const uint64_t *>(expert_table);
    ma.perm = g.perm;
    ma.tiles = g.tiles;
    ma.n_tiles = g.n_tiles;
    ma.act = reinterpret_cast<uint16_t *>(ws + L.act);
    ma.act_row = static_cast<uint32_t>(L.Iblk * kBlk * 4);
    ma.ypair = reinterpret_cast<float *>(ws + L.ypair);
    ma.top_k = static_cast<int>(top_k);
    ma.act_kind = act_kind;
    ma.beta = beta;
    ma.lbeta = linear_beta;
    // gate/up: K = H, weight rows N = I, 128 intermediate indices per block
    ma.b = xf32 ? static_cast<const void *>(ws + L.xt) : x;
    ma.brow = static_cast<uint32_t>(xf32 ? L.Hblk * kBlk * 4 : H * 2);
    ma.b_bytes = static_cast<uint32_t>(T * ma.brow);   // below kOob: 3 T Hpad < 2^31
    ma.K = static_cast<int>(H);
    ma.N = static_cast<int>(I);
    ma.NT = static_cast<int>(cdiv(I, 128));
    auto grid = [&](int NT) { return dim3(static_cast<unsigned>(8 * cdiv(static_cast<int64_t>(L.max_tiles) * NT, 8))); };
    if (xf32)
        grouped_gemm_kernel<false, 2><<<grid(ma.NT), kThreads, kLds, st>>>(ma);
    else
        grouped_gemm_kernel<false, 1><<<grid(ma.NT), kThreads, kLds, st>>>(ma);
    rc = check_hip(hipGetLastError(), "moe grouped: gate/up launch");
    if (rc) return rc;
    // down: K = I, weight rows N = H, 256 output rows per block, B = the act terms
    ma.b = ma.act;
    ma.brow = ma.act_row;
    ma.K = static_cast<int>(I);
    ma.N = static_cast<int>(H);
    ma.NT = static_cast<int>(cdiv(H, 256));
    grouped_gemm_kernel<true, 2><<<grid(ma.NT), kThreads, kLds, st>>>(ma);
    rc = check_hip(hipGetLastError(), "moe grouped: down launch");
    if (rc) return rc;

    CombineArgs ca{ma.ypair, expert_w, out, static_cast<int>(T), static_cast<int>(H), static_cast<int>(top_k),
                   out_dtype == K3_BF16};
    combine_kernel<<<dim3(static_cast<unsigned>(T), static_cast<unsigned>(cdiv(H, 1024))), 256, 0, st>>>(ca);
    return check_hip(hipGetLastError(), "moe grouped: combine launch");
}
