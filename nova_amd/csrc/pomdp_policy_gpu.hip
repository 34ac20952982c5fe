// nova-mi355x: executing alpha-vector policies over many beliefs at once on one MI355X.
//
// 1. Value and action of k dense beliefs (src/pomdp/policies/pomdp_alpha_vectors.cpp:52-79 per
//    belief: V(b) = max_j Gamma_j . b over the r alphas, the action pi[j*] of the first
//    maximiser, V = -1e10 and action 0 when no alpha beats -1e10). Three arithmetic modes:
//      exact - every dot product summed over s = 0..n-1 with each product and sum rounded
//              separately, as the reference: V and the action equal nova's bit for bit. A
//              vector-ALU tile kernel: 64 beliefs x 64 alphas per workgroup, each lane a 4 x 4
//              block, both operands staged state-major in LDS 32 states at a time.
//      fp32  - the split GEMM of dense_gemm.h on the bf16 matrix cores (three bf16 parts of
//              each operand, six products, fp32 sums), its fp32 GEMM (v_mfma_f32_32x32x2_f32)
//              where the operands have no such parts.
//      bf16  - dense_score_bf16 of dense_gemm.h: bf16 operands in the k-blocked layout,
//              copied straight into LDS, fp32 accumulation (v_mfma_f32_32x32x16_bf16): about
//              3 significant digits per operand.
//    Calls of few beliefs run on the vector ALUs in every mode (alpha_value_few).
//    All modes write per-(belief, alpha tile) maxima that one merge kernel reduces in tile
//    order (the earlier tile wins ties, i.e. the first maximiser overall).
// 2. Belief updates of k (belief, action, observation) triples
//    (src/pomdp/utilities/pomdp_model_cpu.cpp:89-137 per triple): b'(s') = O[a,s',o] *
//    sum_s T[s,a,s'] b(s), normalised by its sum over s'. The sum over predecessors runs over a
//    list ordered by (s, successor slot) -- the order in which the reference's scatter adds to
//    b'(s') -- and the normaliser is summed serially over s' ascending, so b' equals nova's
//    bit for bit. Three kernels, four where many triples are tiled (belief_tiles lays their
//    beliefs out, belief_update_tiles forms 32 b' per list entry read): the unnormalised b'
//    (predecessor entries read coalesced, their products summed per s' from LDS, b gathered from
//    LDS, O from an observation-major copy built once per model), the normalisers (one serial
//    chain per triple fed through LDS), and the division. A triple whose normaliser is below
//    1e-9 in magnitude keeps the unnormalised b' and reports NOVA_WARNING_INVALID_BELIEF, as the
//    reference returns it.
#include <algorithm>
#include <climits>
#include <cstdint>
#include <cstring>
#include <mutex>
#include <vector>

#include <nova/amd/nova_amd.h>
#include <nova/pomdp/pomdp.h>

#include "dense_gemm.h"
#include "nova_hip.h"

namespace nova_amd {

namespace {

constexpr int kVT = 64;          // beliefs and alphas per exact tile
constexpr int kVS = 32;          // states per LDS step of the exact tile
constexpr int kVThreads = 256;   // 16 x 16 lanes, each a 4 x 4 block of (belief, alpha)

// Exact tile: partial first maxima of b_i . Gamma_j over the tile's alphas, j ascending, with
// strict '>' from -1e10 (alpha_vectors.cpp:64-76).
__global__ __launch_bounds__(kVThreads) void alpha_value_exact(unsigned k, unsigned n,
        unsigned r, const float *__restrict__ B, const float *__restrict__ G,
        float *__restrict__ partV, int *__restrict__ partJ)
{
    __shared__ __attribute__((aligned(16))) float bs[kVS][kVT + 4];
    __shared__ __attribute__((aligned(16))) float gs[kVS][kVT + 4];
    const unsigned i0 = blockIdx.x * kVT, j0 = blockIdx.y * kVT, t = threadIdx.x;
    const unsigned bi = t / 16, aj = t % 16;
    float acc[4][4];
#pragma unroll
    for (int x = 0; x < 4; x++)
#pragma unroll
        for (int y = 0; y < 4; y++)
            acc[x][y] = 0.0f;
    // stage 64 rows x 32 states of each operand, transposed to state-major; entries past n
    // (and rows past k or r) are zeros, whose products add +0 and leave every sum as is. The
    // next step's values are requested into registers before the current step's products,
    // so their latency hides behind the arithmetic.
    constexpr int kPer = kVT * kVS / kVThreads;      // values per lane and operand per step
    float bpre[kPer], gpre[kPer];
    auto loadStep = [&](unsigned s0) {
#pragma unroll
        for (int u = 0; u < kPer; u++) {
            const unsigned x = t + u * kVThreads, row = x / kVS, s = x % kVS;
            const bool inS = s0 + s < n;
            bpre[u] = (inS && i0 + row < k) ? B[(size_t)(i0 + row) * n + s0 + s] : 0.0f;
            gpre[u] = (inS && j0 + row < r) ? G[(size_t)(j0 + row) * n + s0 + s] : 0.0f;
        }
    };
    loadStep(0);
    for (unsigned s0 = 0; s0 < n; s0 += kVS) {
#pragma unroll
        for (int u = 0; u < kPer; u++) {
            const unsigned x = t + u * kVThreads, row = x / kVS, s = x % kVS;
            bs[s][row] = bpre[u];
            gs[s][row] = gpre[u];
        }
        __syncthreads();
        if (s0 + kVS < n)
            loadStep(s0 + kVS);
#pragma unroll 4
        for (int s = 0; s < kVS; s++) {
            const float4 bv = *reinterpret_cast<const float4 *>(&bs[s][bi * 4]);
            const float4 gv = *reinterpret_cast<const float4 *>(&gs[s][aj * 4]);
            const float b4[4] = {bv.x, bv.y, bv.z, bv.w};
            const float g4[4] = {gv.x, gv.y, gv.z, gv.w};
#pragma unroll
            for (int x = 0; x < 4; x++)
#pragma unroll
                for (int y = 0; y < 4; y++)
                    acc[x][y] = __fadd_rn(acc[x][y], __fmul_rn(g4[y], b4[x]));
        }
        __syncthreads();
    }
#pragma unroll
    for (int x = 0; x < 4; x++) {
        float bv = kLow;
        int bj = INT_MAX;
#pragma unroll
        for (int y = 0; y < 4; y++) {
            const unsigned j = j0 + aj * 4 + y;
            if (j < r && acc[x][y] > bv) {
                bv = acc[x][y];
                bj = (int)j;
            }
        }
        // the 16 lanes of this belief row are 16 consecutive lanes of one wave
        for (int off = 8; off >= 1; off >>= 1) {
            const float ov = __shfl_xor(bv, off, 16);
            const int oj = __shfl_xor(bj, off, 16);
            if (better(ov, oj, bv, bj)) {
                bv = ov;
                bj = oj;
            }
        }
        const unsigned i = i0 + bi * 4 + x;
        if (aj == 0 && i < k) {
            partV[(size_t)blockIdx.y * k + i] = bv;
            partJ[(size_t)blockIdx.y * k + i] = bj;
        }
    }
}

// Merge of the alpha tiles per belief, tile 0 first: V, the winning alpha (or -1) and its
// action (0 when none beat -1e10, as the reference leaves a). skip (nullable): when *skip is
// not 0 the tiles were left out, and there is nothing to merge.
__global__ __launch_bounds__(256) void alpha_value_merge(unsigned k, unsigned tiles,
        const float *__restrict__ partV, const int *__restrict__ partJ,
        const unsigned *__restrict__ pi, float *__restrict__ V, unsigned *__restrict__ act,
        int *__restrict__ jOut, const int *__restrict__ skip)
{
    const unsigned i = blockIdx.x * 256 + threadIdx.x;
    if (i >= k || (skip && *skip))
        return;
    float bv = kLow;
    int bj = INT_MAX;
    for (unsigned tl = 0; tl < tiles; tl++) {
        const float v = partV[(size_t)tl * k + i];
        const int j = partJ[(size_t)tl * k + i];
        if (better(v, j, bv, bj)) {
            bv = v;
            bj = j;
        }
    }
    const bool none = (bj == INT_MAX) || !(bv > kLow);
    V[i] = none ? kLow : bv;
    act[i] = none ? 0u : pi[bj];
    if (jOut)
        jOut[i] = none ? -1 : bj;
}

// The same for few beliefs: one wave per tile of 16 alphas x 4 X beliefs, each lane one alpha and
// X beliefs, so that a call of a few beliefs spreads over many CUs where alpha_value_exact has
// one workgroup per 64 alphas. A lane's sums are serial chains over the states (the reference's
// order), so what bounds a call is that chain and the loads that feed it: the wave requests the
// next CH states of its rows into registers before it sums the current CH from LDS (rows padded
// by 4 floats: the 16 alphas' 16-byte reads fall on distinct banks, the beliefs' are
// broadcasts). One wave per workgroup: its LDS needs no barrier, only the order of its own
// accesses. VEC: rows 16-byte aligned (n % 4 == 0).
constexpr unsigned kFewAlphas = 16;

// A load at a 32-bit byte offset from a uniform base (one address register a lane)
template <typename T>
__device__ __forceinline__ T load_at(const void *base, unsigned bytes)
{
    return *reinterpret_cast<const T *>(static_cast<const char *>(base) + bytes);
}

// PREC: the call's precision, 0 exact, 1 fp32 (each product and sum rounded once, by an FMA), 2
// operands rounded to bf16 on the way into LDS and fp32 sums of 16 products at a time, as the
// bf16 matrix instruction takes them (a chain of single products is 2.4 times as far from 64
// bits: n = 20,000: 1.8e-6 against 5.9e-7, the matrix instruction 7.2e-7). FAR: rows of more than
// 2^30 states (VEC rows are addressed that way at any size; without VEC it takes a tenth longer).
template <int X, int CH, bool VEC, int PREC, bool FAR>
__global__ __launch_bounds__(64) void alpha_value_few(unsigned k, unsigned n, unsigned r,
        const float *__restrict__ B, const float *__restrict__ G, float *__restrict__ partV,
        int *__restrict__ partJ)
{
    constexpr int kRows = (int)kFewAlphas + 4 * X, kStride = CH + 4;
    // a lane's loads per chunk: VEC takes float4s numbered row-major over the tile, else words
    constexpr int kAcross = VEC ? CH / 4 : CH;
    constexpr int kPer = kAcross * kRows / 64;
    __shared__ __attribute__((aligned(16))) float buf[kRows * kStride];
    const unsigned lane = threadIdx.x, al = lane % kFewAlphas, bl = lane / kFewAlphas;
    const unsigned j0 = blockIdx.y * kFewAlphas, i0 = blockIdx.x * 4 * X;
    // row q of the tile: alphas, then beliefs; rows past r or k repeat the last one
    auto rowOf = [&](unsigned q) {
        return q < kFewAlphas ? G + (size_t)min(j0 + q, r - 1) * n
                              : B + (size_t)min(i0 + (q - kFewAlphas), k - 1) * n;
    };
    float4 pre4[VEC ? kPer : 1];
    float pre[VEC ? 1 : kPer];
    // states past n are zeros in both operands: their products add +0
    auto load = [&](unsigned s0) {
#pragma unroll
        for (int u = 0; u < kPer; u++) {
            const unsigned e = u * 64 + lane;
            // a whole row per load or more: the same row in every lane, addressed from a scalar.
            // FAR: the chunk's start is part of the 64-bit base, as a 32-bit offset from the row's
            // start would wrap at 4 GB.
            const float *row = (kAcross >= 64 ? rowOf(u * 64 / kAcross) : rowOf(e / kAcross)) +
                               (FAR ? s0 : 0u);
            const unsigned in = e % kAcross * (VEC ? 4u : 1u), at = FAR ? in : s0 + in;
            if constexpr (VEC)
                pre4[u] = s0 + in < n ? load_at<float4>(row, at * 4u)
                                      : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            else
                pre[u] = s0 + in < n ? load_at<float>(row, at * 4u) : 0.0f;
        }
    };
    float acc[X];
#pragma unroll
    for (int x = 0; x < X; x++)
        acc[x] = 0.0f;
    load(0);
    for (unsigned s0 = 0; s0 < n; s0 += CH) {
#pragma unroll
        for (int u = 0; u < kPer; u++) {
            const unsigned e = u * 64 + lane;
            auto in = [](float v) { return PREC == 2 ? (float)(__bf16)v : v; };
            if constexpr (VEC)
                *reinterpret_cast<float4 *>(&buf[e / kAcross * kStride + e % kAcross * 4]) =
                    make_float4(in(pre4[u].x), in(pre4[u].y), in(pre4[u].z), in(pre4[u].w));
            else
                buf[e / kAcross * kStride + e % kAcross] = in(pre[u]);
        }
        __syncthreads();
        if (s0 + CH < n)
            load(s0 + CH);
        // blocks of 16 states; one belief per lane reads the next block from LDS before it sums
        // the current one (n = 5,000: 67 -> 60 us; two beliefs per lane lose more to the
        // registers this takes, 129 -> 141 us at n = 5,000, r = 1,024, k = 256)
        const unsigned cnt = min((unsigned)CH, (n - s0 + 15) / 16 * 16);
        float4 g[4], bb[X][4];
        auto read = [&](unsigned s, float4 (&gq)[4], float4 (&bq)[X][4]) {
#pragma unroll
            for (int v = 0; v < 4; v++) {
                gq[v] = *reinterpret_cast<const float4 *>(&buf[al * kStride + s + 4 * v]);
#pragma unroll
                for (int x = 0; x < X; x++)
                    bq[x][v] = *reinterpret_cast<const float4 *>(
                        &buf[(kFewAlphas + bl * X + x) * kStride + s + 4 * v]);
            }
        };
        auto sum = [&](const float4 (&gq)[4], const float4 (&bq)[X][4]) {
            float part[X];
#pragma unroll
            for (int x = 0; x < X; x++)
                part[x] = PREC == 2 ? 0.0f : acc[x];
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const float g4[4] = {gq[v].x, gq[v].y, gq[v].z, gq[v].w};
#pragma unroll
                for (int e = 0; e < 4; e++)
#pragma unroll
                    for (int x = 0; x < X; x++) {
                        const float b4[4] = {bq[x][v].x, bq[x][v].y, bq[x][v].z, bq[x][v].w};
                        part[x] = PREC == 0 ? __fadd_rn(part[x], __fmul_rn(g4[e], b4[e]))
                                            : __fmaf_rn(g4[e], b4[e], part[x]);
                    }
            }
#pragma unroll
            for (int x = 0; x < X; x++)
                acc[x] = PREC == 2 ? __fadd_rn(acc[x], part[x]) : part[x];
        };
        if constexpr (X == 1) {
            read(0, g, bb);
            for (unsigned s = 0; s < cnt; s += 32) {
                float4 g2[4], bb2[X][4];
                read(min(s + 16, (unsigned)CH - 16), g2, bb2);
                __builtin_amdgcn_sched_barrier(0);
                sum(g, bb);
                if (s + 16 < cnt) {
                    read(min(s + 32, (unsigned)CH - 16), g, bb);
                    __builtin_amdgcn_sched_barrier(0);
                    sum(g2, bb2);
                }
            }
        } else {
            for (unsigned s = 0; s < cnt; s += 16) {
                read(s, g, bb);
                sum(g, bb);
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int x = 0; x < X; x++) {
        const bool use = j0 + al < r && acc[x] > kLow;
        float bv = use ? acc[x] : kLow;
        int bj = use ? (int)(j0 + al) : INT_MAX;
        for (int off = 8; off >= 1; off >>= 1) {
            const float ov = __shfl_xor(bv, off, 16);
            const int oj = __shfl_xor(bj, off, 16);
            if (better(ov, oj, bv, bj)) {
                bv = ov;
                bj = oj;
            }
        }
        const unsigned i = i0 + bl * X + x;
        if (al == 0 && i < k) {
            partV[(size_t)blockIdx.y * k + i] = bv;
            partJ[(size_t)blockIdx.y * k + i] = bj;
        }
    }
}

// alpha_value_merge with one wave per belief, for few beliefs and many tiles.
__global__ __launch_bounds__(64) void alpha_value_merge_few(unsigned k, unsigned tiles,
        const float *__restrict__ partV, const int *__restrict__ partJ,
        const unsigned *__restrict__ pi, float *__restrict__ V, unsigned *__restrict__ act,
        int *__restrict__ jOut)
{
    const unsigned i = blockIdx.x;
    float bv = kLow;
    int bj = INT_MAX;
    for (unsigned tl = threadIdx.x; tl < tiles; tl += 64) {
        const float v = partV[(size_t)tl * k + i];
        const int j = partJ[(size_t)tl * k + i];
        if (better(v, j, bv, bj)) {
            bv = v;
            bj = j;
        }
    }
    for (int off = 32; off >= 1; off >>= 1) {
        const float ov = __shfl_xor(bv, off);
        const int oj = __shfl_xor(bj, off);
        if (better(ov, oj, bv, bj)) {
            bv = ov;
            bj = oj;
        }
    }
    if (threadIdx.x != 0)
        return;
    const bool none = (bj == INT_MAX) || !(bv > kLow);
    V[i] = none ? kLow : bv;
    act[i] = none ? 0u : pi[bj];
    if (jOut)
        jOut[i] = none ? -1 : bj;
}

template <int X, int CH, int PREC>
void launch_few(unsigned k, unsigned n, unsigned r, const float *B, const float *G, float *partV,
                int *partJ, hipStream_t st)
{
    const bool vec = n % 4 == 0 && ((reinterpret_cast<uintptr_t>(B) |
                                     reinterpret_cast<uintptr_t>(G)) & 15u) == 0;
    const dim3 g((k + 4 * X - 1) / (4 * X), (r + kFewAlphas - 1) / kFewAlphas);
    if (vec)
        hipLaunchKernelGGL((alpha_value_few<X, CH, true, PREC, true>), g, dim3(64), 0, st, k, n, r,
                           B, G, partV, partJ);
    else if (n <= 1u << 30)
        hipLaunchKernelGGL((alpha_value_few<X, CH, false, PREC, false>), g, dim3(64), 0, st, k, n,
                           r, B, G, partV, partJ);
    else
        hipLaunchKernelGGL((alpha_value_few<X, CH, false, PREC, true>), g, dim3(64), 0, st, k, n, r,
                           B, G, partV, partJ);
}

template <int PREC>
void launch_few_of(unsigned few, unsigned k, unsigned n, unsigned r, const float *B,
                   const float *G, float *partV, int *partJ, hipStream_t st)
{
    if (few == 1)
        launch_few<1, 256, PREC>(k, n, r, B, G, partV, partJ, st);
    else
        launch_few<2, 128, PREC>(k, n, r, B, G, partV, partJ, st);
}

// Beliefs per lane of alpha_value_few for a call, or 0 where the mode's own kernel is the faster:
// one while that gives at most 1,024 waves (one per SIMD), then two, until alpha_value_exact has
// a workgroup per CU and more. us of a call, 0 / 1 / 2 beliefs per lane: n = 5,000, r = 1,024:
// k = 4: 602 / 60 / 90; k = 256: 630 / 208 / 131; k = 2,048: 595 / 1,189 / 745. n = 20,000,
// r = 4,096: k = 1: 2,400 / 204 / 311; k = 64: 2,480 / 829 / 460; k = 256: 2,470 / 2,490 /
// 1,540; k = 512: 2,290 / 4,660 / 3,150. The same line serves fp32, whose GEMM has a workgroup
// per 256 x 256 block of C (us, the fp32 GEMM / the split GEMM / this: n = 20,000, r = 4,096,
// k = 16: 5,140 / 2,310 / 214; k = 256: 5,150 / 2,320 / 1,510; n = 1,000, r = 200, k = 4,096:
// 315 / 177 / 82). bf16 calls take it up to kFewBf16 beliefs (n = 20,000, r = 4,096: k = 8: 213,
// k = 64: 408 against 508 of the bf16 GEMM at any k up to 256).
// Short rows leave nothing to spread: exact calls of at most kFewShort states, and of many
// pairs (kFewShortPairs) in both directions, keep the square tiles (n = 50: k = 1,000,
// r = 1,200: 34 / 34; k = 18,750, r = 64: 29 / 34; k = 50,000, r = 20: 34 / 38; k = 9,375, r = 64:
// 29 / 28; k = 75,000, r = 16: 40 / 34; n = 100: k = 18,750, r = 64: 38 / 34).
// The partials of k >= kMergeWaves beliefs (at most 10 tiles each) are merged a lane per belief,
// fewer a wave per belief (us of a call, wave / lane: n = 50, k = 50,000, r = 20: 49 / 38;
// k = 8,192, r = 10: 24 / 22; k = 4,096, r = 300: 36 / 40).
constexpr size_t kFewPairs = 5u << 18;       // most (belief, alpha) pairs, 1.25 Mi
constexpr size_t kFewShortPairs = 9u << 16;  // of short rows
constexpr unsigned kFewShort = 64;
constexpr unsigned kFewBf16 = 64;
constexpr unsigned kFewStates = 1u << 31;    // most states (the kernel's 32-bit state counters)
constexpr unsigned kMergeWaves = 8192;

unsigned few_beliefs(unsigned n, unsigned k, unsigned r, int precision)
{
    if ((size_t)k * r > kFewPairs || r > 65535u * kFewAlphas ||       // (the grid's y extent)
            n > kFewStates ||
            (precision == 0 && n <= kFewShort && (size_t)k * r > kFewShortPairs && k >= 1024 &&
             r > kFewAlphas) ||
            (precision == 2 && (k > kFewBf16 || dense_legacy_bf16())))
        return 0;
    const size_t waves = (size_t)((k + 3) / 4) * ((r + kFewAlphas - 1) / kFewAlphas);
    return waves <= 1024 ? 1 : 2;
}

// Alphas per partial of the exact mode.
inline unsigned exact_tile(unsigned few) { return few ? kFewAlphas : (unsigned)kVT; }

// Partials and merge on the vector ALUs: the exact mode, and the others' calls of few beliefs.
void launch_exact(unsigned few, int precision, unsigned k, unsigned n, unsigned r, const float *B,
                  const float *G, const unsigned *pi, float *partV, int *partJ, float *V,
                  unsigned *act, int *jOut, hipStream_t st)
{
    const unsigned tiles = (r + exact_tile(few) - 1) / exact_tile(few);
    if (few == 0) {
        hipLaunchKernelGGL(alpha_value_exact, dim3((k + kVT - 1) / kVT, tiles), dim3(kVThreads),
                           0, st, k, n, r, B, G, partV, partJ);
        hipLaunchKernelGGL(alpha_value_merge, dim3((k + 255) / 256), dim3(256), 0, st, k, tiles,
                           partV, partJ, pi, V, act, jOut, (const int *)nullptr);
        return;
    }
    if (precision == 0)
        launch_few_of<0>(few, k, n, r, B, G, partV, partJ, st);
    else if (precision == 1)
        launch_few_of<1>(few, k, n, r, B, G, partV, partJ, st);
    else
        launch_few_of<2>(few, k, n, r, B, G, partV, partJ, st);
    if (k < kMergeWaves)
        hipLaunchKernelGGL(alpha_value_merge_few, dim3(k), dim3(64), 0, st, k, tiles, partV, partJ,
                           pi, V, act, jOut);
    else
        hipLaunchKernelGGL(alpha_value_merge, dim3((k + 255) / 256), dim3(256), 0, st, k, tiles,
                           partV, partJ, pi, V, act, jOut, (const int *)nullptr);
}

__global__ __launch_bounds__(256) void fill_ones(unsigned count, float *__restrict__ x)
{
    const unsigned i = blockIdx.x * 256 + threadIdx.x;
    if (i < count)
        x[i] = 1.0f;
}

// Belief updates in three kernels (four for many triples: belief_tiles, belief_update_tiles in
// the place of the first), each sum in the reference's order:
//   belief_update_batch: one workgroup per triple q; b is staged in LDS. Wave w takes blocks
//     of 64 consecutive states s'. The block's predecessor entries (contiguous in the lists)
//     are read 64 at a time, coalesced, and their products T * b(s) formed into the wave's LDS
//     scratch; lane t then adds the products of s' = block + t in list order, multiplies by
//     O[a,s',o] (from the observation-major copy Ot[a][o][s']) and writes the unnormalised
//     b'(s'). When n exceeds the LDS buffer b is read from global memory.
//   belief_norms: the normaliser of triple q, summed serially over s' by one lane; 16 triples
//     per workgroup, their rows streamed through double-buffered LDS by the other waves.
//   belief_divide: b'_q / c_q for the triples whose normaliser is usable.
constexpr int kUB = 1024;
constexpr int kUpdWaves = kUB / 64;
constexpr int kUpdScratch = 1024;                // product slots per wave
constexpr int kUpdLdsFloats = 40 * 1024 - kUpdWaves * kUpdScratch;   // 160 KB in all
constexpr int kUpdBatch = 8;                     // list entries per lane requested together

// IDX: the predecessor's index type, 16 bits for n <= 65,536 (6 bytes per list entry, not 8)
template <typename IDX>
__global__ __launch_bounds__(kUB) void belief_update_batch(unsigned n, unsigned m, unsigned z,
        const unsigned *__restrict__ pstart, const IDX *__restrict__ pS,
        const float *__restrict__ pT, const float *__restrict__ Ot, const float *__restrict__ B,
        const unsigned *__restrict__ rowOf, const unsigned *__restrict__ act,
        const unsigned *__restrict__ obs, float *__restrict__ Bp, int useLds,
        const unsigned *__restrict__ order)
{
    extern __shared__ float smem[];
    // order: the triples grouped by action, so that the workgroups running together on an XCD
    // stream the same action's predecessor list and find it in their L2
    const unsigned q = order ? order[blockIdx.x] : blockIdx.x;
    const unsigned t = threadIdx.x, lane = t % 64, w = t / 64;
    const unsigned a = act[q], o = obs[q];
    if (a >= m || o >= z)
        return;                                  // belief_norms reports it
    const float *b = B + (size_t)(rowOf ? rowOf[q] : q) * n;   // rowOf: belief row of triple q
    float *out = Bp + (size_t)q * n;
    float *row = smem;                                           // n floats when useLds
    float *scr = smem + (useLds ? n : 0) + w * kUpdScratch;
    if (useLds) {
        for (unsigned s = t; s < n; s += kUB)
            row[s] = b[s];
        __syncthreads();
    }
    const float *src = useLds ? row : b;
    const unsigned *ps = pstart + (size_t)a * (n + 1);
    const float *Oao = Ot + ((size_t)a * z + o) * n;
    for (unsigned s0 = w * 64; s0 < n; s0 += kUpdWaves * 64) {
        const unsigned s1 = min(s0 + 64, n), sp = s0 + lane;
        const unsigned xa = ps[s0], xb = ps[s1];
        const unsigned lo = sp < n ? ps[sp] : xb, hi = sp < n ? ps[sp + 1] : xb;
        float u = 0.0f;
        for (unsigned xs = xa; xs < xb; xs += kUpdScratch) {
            const unsigned xe = min(xs + (unsigned)kUpdScratch, xb);
            // the lane's entries of the chunk kUpdBatch at a time, their predecessors and
            // factors requested together (indices clamped into the chunk, the extra products
            // not stored)
            for (unsigned x0 = xs + lane; x0 < xe; x0 += 64 * kUpdBatch) {
                IDX si[kUpdBatch];
                float tv[kUpdBatch];
#pragma unroll
                for (int k = 0; k < kUpdBatch; k++) {
                    const unsigned x = min(x0 + 64u * k, xe - 1);
                    si[k] = pS[x];
                    tv[k] = pT[x];
                }
#pragma unroll
                for (int k = 0; k < kUpdBatch; k++) {
                    const unsigned x = x0 + 64u * k;
                    const float pr = __fmul_rn(tv[k], src[si[k]]);
                    if (x < xe)
                        scr[x - xs] = pr;
                }
            }
            // the wave's own LDS writes, then reads by other lanes of the wave
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            const unsigned e1 = min(hi, xe);
            for (unsigned x = max(lo, xs); x < e1; x++)
                u = __fadd_rn(u, scr[x - xs]);
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }
        if (sp < n)
            out[sp] = __fmul_rn(u, Oao[sp]);
    }
}

// The k triples grouped by action (a counting sort in one workgroup; invalid actions last).
// The order within an action is whatever the atomics give: each triple's result does not
// depend on when it runs. tiles (nullable) receives the groups cut into tiles of at most
// kTileT triples of one action, (action, first position in order, triples, 0); the entries
// past the last tile, up to maxTiles, get 0 triples.
constexpr unsigned kOrderMaxM = 4096;
constexpr size_t kOrderListBytes = (size_t)4 << 20;
constexpr unsigned kTileT = 32;

__global__ __launch_bounds__(1024) void order_by_action(unsigned k, unsigned m,
        const unsigned *__restrict__ act, unsigned *__restrict__ order, uint4 *__restrict__ tiles,
        unsigned maxTiles)
{
    __shared__ unsigned cnt[kOrderMaxM + 1], first[kOrderMaxM + 1];
    const unsigned t = threadIdx.x;
    for (unsigned x = t; x <= m; x += 1024)
        cnt[x] = 0;
    __syncthreads();
    for (unsigned q = t; q < k; q += 1024)
        atomicAdd(&cnt[min(act[q], m)], 1u);
    __syncthreads();
    if (t == 0) {
        unsigned run = 0, tile = 0;
        for (unsigned x = 0; x <= m; x++) {
            const unsigned c = cnt[x];
            cnt[x] = run;
            first[x] = tile;
            run += c;
            tile += (c + kTileT - 1) / kTileT;
        }
    }
    __syncthreads();
    if (tiles) {
        const unsigned used = first[m];
        for (unsigned x = t; x < m; x += 1024)
            for (unsigned q = cnt[x], i = first[x]; q < cnt[x + 1]; q += kTileT, i++)
                tiles[i] = make_uint4(x, q, min(kTileT, cnt[x + 1] - q), 0u);
        for (unsigned i = used + t; i < maxTiles; i += 1024)
            tiles[i] = make_uint4(0u, 0u, 0u, 0u);
    }
    __syncthreads();
    for (unsigned q = t; q < k; q += 1024)
        order[atomicAdd(&cnt[min(act[q], m)], 1u)] = q;
}

// Many updates: the beliefs of a tile of kTileT triples of one action are laid out state-major,
// BT[tile][s][triple], so that one predecessor entry (s, T) serves all of them with one
// 128-byte row. belief_update_batch re-reads the action's whole list (6 or 8 bytes an entry)
// for every belief; here a list is read once per tile and a belief costs 4 coalesced bytes an
// entry, from the L2 that holds its tile (n x 128 bytes). Sums run over the same lists in the
// same order, products and sums rounded as there.
constexpr unsigned kTileS = 128;         // states per workgroup of the two kernels
constexpr unsigned kTileThreads = 256;

__global__ __launch_bounds__(kTileThreads) void belief_tiles(unsigned n,
        const uint4 *__restrict__ tiles, const unsigned *__restrict__ order,
        const unsigned *__restrict__ rowOf, const float *__restrict__ B, float *__restrict__ BT)
{
    __shared__ float buf[kTileT][kTileS + 1];
    const uint4 tile = tiles[blockIdx.y];
    if (tile.z == 0)
        return;
    const unsigned t = threadIdx.x, s0 = blockIdx.x * kTileS;
    constexpr unsigned kPer = kTileT * kTileS / kTileThreads;
    float v[kPer];
#pragma unroll
    for (unsigned u = 0; u < kPer; u++) {
        const unsigned x = u * kTileThreads + t, i = x / kTileS, s = s0 + x % kTileS;
        v[u] = 0.0f;
        if (i < tile.z && s < n) {
            const unsigned q = order[tile.y + i];
            v[u] = B[(size_t)(rowOf ? rowOf[q] : q) * n + s];
        }
    }
#pragma unroll
    for (unsigned u = 0; u < kPer; u++) {
        const unsigned x = u * kTileThreads + t;
        buf[x / kTileS][x % kTileS] = v[u];
    }
    __syncthreads();
    float *out = BT + ((size_t)blockIdx.y * n + s0) * kTileT;
#pragma unroll
    for (unsigned u = 0; u < kPer; u++) {
        const unsigned x = u * kTileThreads + t, s = x / kTileT, i = x % kTileT;
        if (s0 + s < n)
            out[x] = buf[i][s];
    }
}

// The unnormalised updates of the tiles: 8 lanes per state s', each holding four triples; a
// lane walks the state's predecessors kTileE at a time (the next ones' indices and factors
// requested before this round's beliefs are summed), multiplies by O[a, s', o] and leaves the
// products in LDS, from where the triples' rows are written past the caches. At n = 20,000,
// ns = 8 a chunk of 48 tiles takes 133 us (7.4 TB/s of gathered rows, of which about 4.7 TB/s
// pass L2: the beliefs, O and the rows written, each as large); 16 triples a tile take 196 us per
// 48, staging the lists in LDS 160 us (fewer workgroups fit), 8 entries at a time 151 us. Workgroups are dealt to the XCDs
// in turn: workgroup b takes a tile of XCD b mod 8, so that the workgroups running together on
// an XCD share one tile's BT (spread = 8; a chunk of fewer than 8 tiles gives each to all XCDs,
// spread = 1). count tiles of the chunk.
constexpr unsigned kTileE = 4;
constexpr size_t kTileBytes = (size_t)128 << 20;     // most state-major beliefs of a chunk of tiles

template <typename IDX>
__global__ __launch_bounds__(kTileThreads) void belief_update_tiles(unsigned n, unsigned z,
        unsigned blocks, unsigned count, unsigned spread, const uint4 *__restrict__ tiles,
        const unsigned *__restrict__ order, const unsigned *__restrict__ pstart,
        const IDX *__restrict__ pS, const float *__restrict__ pT, const float *__restrict__ O,
        const unsigned *__restrict__ obs, const float *__restrict__ BT, float *__restrict__ Bp)
{
    __shared__ float buf[kTileT][kTileS + 1];
    __shared__ unsigned row[kTileT];         // the triple's row of Bp, or ~0 when it has none
    const unsigned b = blockIdx.x / spread, slot = b / blocks * spread + blockIdx.x % spread;
    if (slot >= count)
        return;
    const uint4 tile = tiles[slot];
    if (tile.z == 0)
        return;
    const unsigned t = threadIdx.x, s0 = b % blocks * kTileS, a = tile.x;
    constexpr unsigned kL = kTileT / 4;      // lanes per state
    const unsigned l = t % kL, first = 4 * l;
    unsigned o[4];
#pragma unroll
    for (unsigned e = 0; e < 4; e++) {
        // (an observation out of range: no row is written, belief_norms reports it)
        const unsigned ob = first + e < tile.z ? obs[order[tile.y + first + e]] : z;
        o[e] = min(ob, z - 1);
        if (t < kL)
            row[first + e] = ob < z ? order[tile.y + first + e] : ~0u;
    }
    const unsigned *ps = pstart + (size_t)a * (n + 1);
    const float *Oa = O + (size_t)a * n * z;
    const float4 *bt = reinterpret_cast<const float4 *>(BT + (size_t)slot * n * kTileT) + l;
    for (unsigned s = t / kL; s < kTileS; s += kTileThreads / kL) {
        const unsigned sp = s0 + s;
        if (sp >= n)
            break;
        const unsigned lo = ps[sp], hi = ps[sp + 1];
        float u[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        if (lo < hi) {
            IDX si[kTileE];
            float tv[kTileE];
            auto request = [&](unsigned x) {
#pragma unroll
                for (unsigned e = 0; e < kTileE; e++) {
                    const unsigned at = min(x + e, hi - 1);
                    si[e] = pS[at];
                    tv[e] = pT[at];
                }
            };
            request(lo);
            for (unsigned x = lo; x < hi; x += kTileE) {
                float4 bv[kTileE];
                float tc[kTileE];
#pragma unroll
                for (unsigned e = 0; e < kTileE; e++) {
                    bv[e] = bt[(size_t)si[e] * (kTileT / 4)];
                    tc[e] = tv[e];
                }
                if (x + kTileE < hi)
                    request(x + kTileE);
#pragma unroll
                for (unsigned e = 0; e < kTileE; e++)
                    if (x + e < hi) {
                        u[0] = __fadd_rn(u[0], __fmul_rn(tc[e], bv[e].x));
                        u[1] = __fadd_rn(u[1], __fmul_rn(tc[e], bv[e].y));
                        u[2] = __fadd_rn(u[2], __fmul_rn(tc[e], bv[e].z));
                        u[3] = __fadd_rn(u[3], __fmul_rn(tc[e], bv[e].w));
                    }
            }
        }
#pragma unroll
        for (unsigned e = 0; e < 4; e++)
            buf[first + e][s] = __fmul_rn(u[e], Oa[(size_t)sp * z + o[e]]);
    }
    __syncthreads();
    constexpr unsigned kPer = kTileT * kTileS / kTileThreads;
#pragma unroll
    for (unsigned v = 0; v < kPer; v++) {
        const unsigned x = v * kTileThreads + t, i = x / kTileS, s = x % kTileS;
        if (s0 + s < n && row[i] != ~0u)
            __builtin_nontemporal_store(buf[i][s], Bp + (size_t)row[i] * n + s0 + s);
    }
}

constexpr unsigned kNormT = 16;          // triples per workgroup of belief_norms
constexpr unsigned kNormC = 512;         // states per chunk
constexpr unsigned kNormLoaders = 256;   // lanes of waves 1-4, 32 values each per chunk

// The normaliser is one serial sum per triple: waves 1-4 stream chunks of the 16 rows into one
// buffer (coalesced, all 32 loads of a lane in flight together) while lanes 0-15 of wave 0 add
// the other buffer's chunk into their triple's sum, in order. What bounds it is that chain of
// adds: 16 values are read from LDS as four 16-byte words while the 16 before are added (one
// word at a time, each add waited for its own LDS read: 593 us for 16,384 triples of 20,000
// states, now 519 us, at 2.5 TB/s). Rows are padded to 516 floats so that the 16 lanes' reads fall on distinct
// banks; values past n are zeros, which leave the sum (never -0) as it is.
__global__ __launch_bounds__(64 + kNormLoaders) void belief_norms(unsigned n, unsigned m,
        unsigned z, unsigned k, const unsigned *__restrict__ act,
        const unsigned *__restrict__ obs, const float *__restrict__ Bp,
        float *__restrict__ norms, int *__restrict__ status)
{
    constexpr unsigned kPer = kNormT * kNormC / kNormLoaders;
    __shared__ __attribute__((aligned(16))) float buf[2][kNormT][kNormC + 4];
    const unsigned t = threadIdx.x, q0 = blockIdx.x * kNormT;
    // the loaders' values: requested one chunk before they are written to LDS, two before they
    // are summed
    float v[kPer];
    auto request = [&](unsigned c0) {
#pragma unroll
        for (unsigned u = 0; u < kPer; u++) {
            const unsigned e = (t - 64) + kNormLoaders * u, j = e / kNormC, i = e % kNormC;
            v[u] = (q0 + j < k && c0 + i < n) ? Bp[(size_t)(q0 + j) * n + c0 + i] : 0.0f;
        }
    };
    auto place = [&](unsigned which) {
#pragma unroll
        for (unsigned u = 0; u < kPer; u++) {
            const unsigned e = (t - 64) + kNormLoaders * u;
            buf[which][e / kNormC][e % kNormC] = v[u];
        }
    };
    if (t >= 64) {
        request(0);
        place(0);
        request(kNormC);
    }
    __syncthreads();
    float c = 0.0f;
    unsigned cur = 0;
    for (unsigned c0 = 0; c0 < n; c0 += kNormC, cur ^= 1) {
        if (t >= 64 && c0 + kNormC < n) {
            place(cur ^ 1);
            request(c0 + 2 * kNormC);        // (zeros past n)
        }
        if (t < kNormT) {
            const float4 *row = reinterpret_cast<const float4 *>(buf[cur][t]);
            const unsigned end = (min(kNormC, n - c0) + 15) / 16 * 4;
            float4 x[4];
#pragma unroll
            for (unsigned e = 0; e < 4; e++)
                x[e] = row[e];
            for (unsigned i = 0; i < end; i += 4) {
                float4 w[4];
                const unsigned next = min(i + 4, kNormC / 4 - 4);
#pragma unroll
                for (unsigned e = 0; e < 4; e++)
                    w[e] = row[next + e];
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (unsigned e = 0; e < 4; e++) {
                    c = __fadd_rn(c, x[e].x);
                    c = __fadd_rn(c, x[e].y);
                    c = __fadd_rn(c, x[e].z);
                    c = __fadd_rn(c, x[e].w);
                }
#pragma unroll
                for (unsigned e = 0; e < 4; e++)
                    x[e] = w[e];
            }
        }
        __syncthreads();
    }
    const unsigned q = q0 + t;
    if (t >= kNormT || q >= k)
        return;
    if (act[q] >= m || obs[q] >= z) {
        status[q] = NOVA_ERROR_INVALID_DATA;
        return;
    }
    norms[q] = c;
    // a normaliser below the tolerance leaves b' unnormalised (pomdp_model_cpu.cpp:125-130)
    status[q] = ((double)fabsf(c) < NOVA_FLT_ERR_TOL) ? NOVA_WARNING_INVALID_BELIEF
                                                      : NOVA_SUCCESS;
}

__global__ __launch_bounds__(256) void belief_divide(unsigned n, const float *__restrict__ norms,
        const int *__restrict__ status, float *__restrict__ Bp)
{
    const unsigned q = blockIdx.x;
    if (status[q] != NOVA_SUCCESS)
        return;
    const float c = norms[q];
    float *out = Bp + (size_t)q * n;
    for (unsigned sp = threadIdx.x; sp < n; sp += 256)
        out[sp] = __fdiv_rn(out[sp], c);
}

__global__ __launch_bounds__(256) void observation_major(unsigned n, unsigned z, size_t count,
        const float *__restrict__ O, float *__restrict__ Ot)
{
    for (size_t x = blockIdx.x * (size_t)256 + threadIdx.x; x < count;
            x += (size_t)gridDim.x * 256) {
        const size_t sp = x % n, ao = x / n;
        const size_t a = ao / z, o = ao % z;
        Ot[x] = O[(a * n + sp) * z + o];
    }
}

// A device buffer kept between calls and grown on demand (one per use, all devices share
// the process's current device; calls are serialised by the mutex of their use).
struct Arena {
    void *mem = nullptr;
    size_t bytes = 0;
    int device = -1;
};

int arena_get(Arena &A, size_t bytes, const char *fn, void *&out)
{
    int dev = 0;
    hipGetDevice(&dev);
    if (A.mem != nullptr && (A.bytes < bytes || A.device != dev)) {
        hipDeviceSynchronize();
        device_free(A.mem, fn, "policy workspace");
        A.mem = nullptr;
        A.bytes = 0;
    }
    if (A.mem == nullptr) {
        const int rc = device_alloc(&A.mem, bytes, fn, "policy workspace");
        if (rc != NOVA_SUCCESS)
            return rc;
        A.bytes = bytes;
        A.device = dev;
    }
    out = A.mem;
    return NOVA_SUCCESS;
}

std::mutex g_valueMutex;
Arena g_valueArena;
struct DenseShape {
    unsigned k = 0, n = 0, r = 0;
    int precision = -1;
    void *mem = nullptr;
} g_valueShape;

std::mutex g_updateMutex;
// The normalisers, the action order and the tiles of a batch of belief updates: 24 bytes a triple
// at most and kTileBytes. Given back, as the lists below, with the model (belief_update_release).
Arena g_updateArena;
// predecessor lists of the last model seen, keyed by its device arrays
struct PredLists {
    const void *dS = nullptr, *dT = nullptr, *dO = nullptr;
    unsigned long long generation = 0;      // model_generation(true) when built
    unsigned n = 0, m = 0, ns = 0, z = 0;
    void *mem = nullptr;
    size_t bytes = 0;
    unsigned *pstart = nullptr;
    int *pS = nullptr;                  // predecessors when n > 65,536
    unsigned short *pS16 = nullptr;     // predecessors when n <= 65,536
    float *pT = nullptr;
    float *Ot = nullptr;      // O observation-major: Ot[a][o][s'] = O[a][s'][o]
} g_pred;

inline size_t up256(size_t x) { return (x + 255) / 256 * 256; }

} // namespace

// Predecessor lists per action of p's model, (s, T[s,a,l]) for every valid successor entry,
// grouped by successor s' and ordered by (s, l) within each group, built on the host from p's
// host arrays; and the observation-major copy of O, built on the device. Kept until another
// model (other device arrays or sizes) is passed, or S, T or O are uploaded or released again.
static int pred_lists(const nova::POMDP *p, const char *fn)
{
    if (g_pred.mem != nullptr && g_pred.dS == p->d_S && g_pred.dT == p->d_T &&
            g_pred.dO == p->d_O && g_pred.n == p->n && g_pred.m == p->m && g_pred.ns == p->ns &&
            g_pred.z == p->z && g_pred.generation == model_generation(true))
        return NOVA_SUCCESS;
    const unsigned n = p->n, m = p->m, ns = p->ns;
    std::vector<unsigned> pstart((size_t)m * (n + 1), 0);
    for (unsigned s = 0; s < n; s++)
        for (unsigned a = 0; a < m; a++)
            for (unsigned l = 0; l < ns; l++) {
                const int sp = p->S[idx3(s, a, l, m, ns)];
                if (sp < 0)
                    break;
                pstart[(size_t)a * (n + 1) + sp + 1]++;
            }
    size_t total = 0;
    for (unsigned a = 0; a < m; a++) {
        unsigned *rowp = &pstart[(size_t)a * (n + 1)];
        rowp[0] = (unsigned)total;
        for (unsigned sp = 0; sp < n; sp++)
            rowp[sp + 1] += rowp[sp];
        total = rowp[n];
    }
    std::vector<int> pS(std::max<size_t>(total, 1));
    std::vector<float> pT(std::max<size_t>(total, 1));
    std::vector<unsigned> fill(pstart);
    for (unsigned s = 0; s < n; s++)
        for (unsigned a = 0; a < m; a++)
            for (unsigned l = 0; l < ns; l++) {
                const size_t x = idx3(s, a, l, m, ns);
                const int sp = p->S[x];
                if (sp < 0)
                    break;
                const unsigned at = fill[(size_t)a * (n + 1) + sp]++;
                pS[at] = (int)s;
                pT[at] = p->T[x];
            }
    if (g_pred.mem != nullptr) {
        hipDeviceSynchronize();
        device_free(g_pred.mem, fn, "predecessor lists");
        g_pred = PredLists();
    }
    const bool narrow = n <= 65536;
    std::vector<unsigned short> pS16(narrow ? pS.size() : 0);
    for (size_t x = 0; x < pS16.size(); x++)
        pS16[x] = (unsigned short)pS[x];
    const size_t idxBytes = narrow ? sizeof(unsigned short) : sizeof(int);
    const size_t b0 = up256(sizeof(unsigned) * pstart.size()), b1 = up256(idxBytes * pS.size());
    const size_t b2 = up256(sizeof(float) * pT.size());
    const size_t otCount = (size_t)m * p->z * n;
    const size_t bytes = b0 + b1 + b2 + up256(sizeof(float) * otCount);
    void *mem = nullptr;
    int rc = device_alloc(&mem, bytes, fn, "predecessor lists");
    if (rc != NOVA_SUCCESS)
        return rc;
    char *c = static_cast<char *>(mem);
    hipError_t e = hipMemcpy(c, pstart.data(), sizeof(unsigned) * pstart.size(),
                             hipMemcpyHostToDevice);
    if (e == hipSuccess)
        e = hipMemcpy(c + b0, narrow ? (const void *)pS16.data() : (const void *)pS.data(),
                      idxBytes * pS.size(), hipMemcpyHostToDevice);
    if (e == hipSuccess)
        e = hipMemcpy(c + b0 + b1, pT.data(), sizeof(float) * pT.size(), hipMemcpyHostToDevice);
    if (e != hipSuccess) {
        device_free(mem, fn, "predecessor lists");
        return hip_fail(e, fn, "Failed to copy the predecessor lists.",
                        NOVA_ERROR_MEMCPY_TO_DEVICE);
    }
    float *Ot = reinterpret_cast<float *>(c + b0 + b1 + b2);
    hipStream_t st = stream();
    hipLaunchKernelGGL(observation_major,
                       dim3((unsigned)std::min<size_t>((otCount + 255) / 256, 65536)), dim3(256),
                       0, st, n, p->z, otCount, p->d_O, Ot);
    e = hipGetLastError();
    if (e == hipSuccess)
        e = hipStreamSynchronize(st);
    if (e != hipSuccess) {
        device_free(mem, fn, "predecessor lists");
        return hip_fail(e, fn, "Failed to build the observation-major copy of O.",
                        NOVA_ERROR_KERNEL_EXECUTION);
    }
    g_pred.dS = p->d_S;
    g_pred.dT = p->d_T;
    g_pred.dO = p->d_O;
    g_pred.generation = model_generation(true);
    g_pred.n = n;
    g_pred.m = m;
    g_pred.ns = ns;
    g_pred.z = p->z;
    g_pred.mem = mem;
    g_pred.bytes = bytes;
    g_pred.pstart = reinterpret_cast<unsigned *>(c);
    if (narrow)
        g_pred.pS16 = reinterpret_cast<unsigned short *>(c + b0);
    else
        g_pred.pS = reinterpret_cast<int *>(c + b0);
    g_pred.pT = reinterpret_cast<float *>(c + b0 + b1);
    g_pred.Ot = Ot;
    return NOVA_SUCCESS;
}

} // namespace nova_amd

namespace nova_amd {

// Gives back the belief updates' lists and workspace when an array of the model they were built
// from is released (the lists are stale from then on).
void belief_update_release(const void *p)
{
    if (p == nullptr)
        return;
    std::lock_guard<std::mutex> lock(g_updateMutex);
    if (g_pred.mem == nullptr || (p != g_pred.dS && p != g_pred.dT && p != g_pred.dO))
        return;
    const char *fn = "belief_update_release";
    device_free(g_pred.mem, fn, "predecessor lists");
    g_pred = PredLists();
    device_free(g_updateArena.mem, fn, "policy workspace");
    g_updateArena = Arena();
}

// Whether a batch of updates goes through the tiles of kTileT triples: where one workgroup per
// triple is too slow a walk (n from 8,192 on) or the batch is large, and the actions' groups
// fill their tiles well enough (a tile costs about the same with 1 triple as with 32). us of a
// call, workgroup per triple / tiles: n = 20,000, m = 16: k = 1: 770 / 727, k = 33: 815 / 776,
// k = 128: 796 / 783, k = 1,024: 1,007 / 896, k = 16,384: 6,260 / 3,730; n = 100,000, m = 4:
// k = 1: 1,550 / 1,060, k = 1,000: 6,920 / 1,860; n = 1,000,000, m = 2: k = 1: 12,000 / 7,780,
// k = 256: 20,600 / 10,700; n = 10,000, m = 8: k = 1,024: 306 / 251; n = 3,001,
// m = 7: k = 512: 88 / 99, k = 4,096: 171 / 151; n = 500, m = 4: k = 16,384: 166 / 124.
static bool update_tiled(unsigned k, unsigned n, unsigned m, unsigned z)
{
    if (m > kOrderMaxM || (size_t)n * kTileT * 4 > kTileBytes ||
            (size_t)n * z >= ((size_t)1 << 30))      // (32-bit byte offsets)
        return false;
    return (n >= 8192 && (k >= 8 * m || m <= 16)) || (k >= 4096 && k >= 32 * m);
}

// tau(b, a, o) for k triples whose beliefs are rows rowOf[q] of B (rowOf null: row q), bit for
// bit nova's pomdp_belief_update_cpu; shared by the batched entry point and the GPU PEMA.
int belief_update_rows(const nova::POMDP *pomdp, unsigned k, const float *d_B,
                       const unsigned *d_rowOf, const unsigned *d_action,
                       const unsigned *d_observation, float *d_Bp, int *d_status,
                       const char *fn)
{
    const long long bad = first_bad_successor(pomdp->S, (size_t)pomdp->n * pomdp->m, pomdp->ns,
                                              pomdp->n);
    if (bad >= 0) {
        NOVA_ERR(fn, "A successor index lies outside [0, n).");
        return NOVA_ERROR_INVALID_DATA;
    }
    std::lock_guard<std::mutex> lock(g_updateMutex);
    int rc = pred_lists(pomdp, fn);
    if (rc != NOVA_SUCCESS)
        return rc;
    const unsigned n = pomdp->n, m = pomdp->m;
    // tiles of one action's triples: at most k and ceil(k / kTileT) + m of them, in chunks whose
    // state-major beliefs take at most kTileBytes (the grid's y extent bounds them too). Without
    // the memory for a chunk the triples go one by one.
    bool tiled = update_tiled(k, n, m, pomdp->z);
    const unsigned blocks = (n + kTileS - 1) / kTileS;
    const size_t tileBytes = sizeof(float) * kTileT * (size_t)n;
    const size_t normBytes = up256(sizeof(float) * (size_t)k);
    const size_t orderBytes = up256(sizeof(unsigned) * (size_t)k);
    unsigned maxTiles = (unsigned)std::min<size_t>(k, ((size_t)k + kTileT - 1) / kTileT + m);
    unsigned chunkTiles = (unsigned)std::min<size_t>(std::min(maxTiles, 65528u),
                                                     std::max<size_t>(kTileBytes / tileBytes, 1));
    if (chunkTiles > 8)
        chunkTiles = chunkTiles / 8 * 8;
    size_t listBytes = up256(sizeof(uint4) * (size_t)maxTiles);
    size_t chunkBytes = tileBytes * chunkTiles;
    if (tiled && g_updateArena.bytes < normBytes + orderBytes + listBytes + chunkBytes) {
        size_t freeBytes = 0, totalBytes = 0;
        tiled = hipMemGetInfo(&freeBytes, &totalBytes) == hipSuccess &&
                freeBytes + g_updateArena.bytes >=
                    normBytes + orderBytes + listBytes + chunkBytes + ((size_t)64 << 20);
    }
    void *mem = nullptr;
    if (tiled && arena_get(g_updateArena, normBytes + orderBytes + listBytes + chunkBytes, fn,
                           mem) != NOVA_SUCCESS) {
        (void)hipGetLastError();
        tiled = false;
    }
    if (!tiled) {
        maxTiles = chunkTiles = 0;
        listBytes = chunkBytes = 0;
        rc = arena_get(g_updateArena, normBytes + orderBytes, fn, mem);
        if (rc != NOVA_SUCCESS)
            return rc;
    }
    char *c = static_cast<char *>(mem);
    float *norms = reinterpret_cast<float *>(c);
    // without tiles, grouping by action pays only where the predecessor lists exceed an L2
    const bool grouped = tiled || (m <= kOrderMaxM &&
                                   (size_t)n * m * pomdp->ns * sizeof(float) > kOrderListBytes);
    unsigned *order = grouped ? reinterpret_cast<unsigned *>(c + normBytes) : nullptr;
    uint4 *tiles = tiled ? reinterpret_cast<uint4 *>(c + normBytes + orderBytes) : nullptr;
    float *BT = reinterpret_cast<float *>(c + normBytes + orderBytes + listBytes);
    hipStream_t st = stream();
    if (order)
        hipLaunchKernelGGL(order_by_action, dim3(1), dim3(1024), 0, st, k, m, d_action, order,
                           tiles, maxTiles);
    for (unsigned t0 = 0; t0 < maxTiles; t0 += chunkTiles) {
        const unsigned cnt = std::min(chunkTiles, maxTiles - t0);
        const unsigned spread = cnt >= 8 ? 8 : 1;
        const dim3 ug(blocks * ((cnt + spread - 1) / spread * spread));
        hipLaunchKernelGGL(belief_tiles, dim3(blocks, cnt), dim3(kTileThreads), 0, st, n,
                           tiles + t0, order, d_rowOf, d_B, BT);
        if (g_pred.pS16 != nullptr)
            hipLaunchKernelGGL(belief_update_tiles<unsigned short>, ug, dim3(kTileThreads), 0, st,
                               n, pomdp->z, blocks, cnt, spread, tiles + t0, order,
                               g_pred.pstart, g_pred.pS16, g_pred.pT, pomdp->d_O, d_observation,
                               BT, d_Bp);
        else
            hipLaunchKernelGGL(belief_update_tiles<int>, ug, dim3(kTileThreads), 0, st, n,
                               pomdp->z, blocks, cnt, spread, tiles + t0, order, g_pred.pstart,
                               g_pred.pS, g_pred.pT, pomdp->d_O, d_observation, BT, d_Bp);
    }
    const int useLds = n <= (unsigned)kUpdLdsFloats ? 1 : 0;
    const size_t lds = sizeof(float) * ((useLds ? n : 0) + (size_t)kUpdWaves * kUpdScratch);
    if (tiled) {
        // done above
    } else if (g_pred.pS16 != nullptr) {
        hipFuncSetAttribute((const void *)belief_update_batch<unsigned short>,
                            hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        hipLaunchKernelGGL(belief_update_batch<unsigned short>, dim3(k), dim3(kUB), lds, st, n,
                           m, pomdp->z, g_pred.pstart, g_pred.pS16, g_pred.pT, g_pred.Ot,
                           d_B, d_rowOf, d_action, d_observation, d_Bp, useLds, order);
    } else {
        hipFuncSetAttribute((const void *)belief_update_batch<int>,
                            hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        hipLaunchKernelGGL(belief_update_batch<int>, dim3(k), dim3(kUB), lds, st, n, m,
                           pomdp->z, g_pred.pstart, g_pred.pS, g_pred.pT, g_pred.Ot, d_B,
                           d_rowOf, d_action, d_observation, d_Bp, useLds, order);
    }
    hipLaunchKernelGGL(belief_norms, dim3((k + kNormT - 1) / kNormT), dim3(64 + kNormLoaders), 0, st, n,
                       pomdp->m, pomdp->z, k, d_action, d_observation, d_Bp, norms, d_status);
    hipLaunchKernelGGL(belief_divide, dim3(k), dim3(256), 0, st, n, norms, d_status, d_Bp);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess)
        e = hipStreamSynchronize(st);
    if (e != hipSuccess)
        return hip_fail(e, fn, "Kernel execution failed.", NOVA_ERROR_KERNEL_EXECUTION);
    return NOVA_SUCCESS;
}

// The fp32 mode on the bf16 matrix cores (dense_score_split). *done stays false when the
// operands cannot be split exactly or its workspace does not fit: the fp32 instructions do the
// call then.
static int value_split(unsigned n, unsigned r, const float *d_Gamma, const unsigned *d_pi,
                       unsigned k, const float *d_B, float *d_V, unsigned *d_action,
                       int *d_alpha, const char *fn, bool *done)
{
    hipStream_t st = stream();
    const unsigned rowTiles = (k + kGT - 1) / kGT, colTiles = (r + kGT - 1) / kGT;
    const unsigned kpad = (n + kGKPad - 1) / kGKPad * kGKPad;
    const size_t aRows = (size_t)rowTiles * kGT, gRows = (size_t)colTiles * kGT;
    const size_t bPart = up256((size_t)colTiles * k * sizeof(float));
    const size_t bA = up256(3 * aRows * kpad * sizeof(__bf16));
    const size_t bG = up256(3 * gRows * kpad * sizeof(__bf16));
    void *mem = nullptr;
    size_t freeBytes = 0, totalBytes = 0;
    const size_t bytes = 256 + 2 * bPart + bA + bG;
    if (g_valueArena.mem == nullptr || g_valueArena.bytes < bytes)
        if (hipMemGetInfo(&freeBytes, &totalBytes) != hipSuccess ||
                freeBytes + g_valueArena.bytes < bytes + ((size_t)64 << 20))
            return NOVA_SUCCESS;
    g_valueShape = DenseShape();      // the fp32 layout's padding is overwritten, or released
    if (arena_get(g_valueArena, bytes, fn, mem) != NOVA_SUCCESS) {
        (void)hipGetLastError();
        return NOVA_SUCCESS;
    }
    char *c = static_cast<char *>(mem);
    int *wild = reinterpret_cast<int *>(c);
    float *partV = reinterpret_cast<float *>(c + 256);
    int *partJ = reinterpret_cast<int *>(c + 256 + bPart);
    __bf16 *A = reinterpret_cast<__bf16 *>(c + 256 + 2 * bPart);
    __bf16 *G = reinterpret_cast<__bf16 *>(c + 256 + 2 * bPart + bA);
    hipFuncSetAttribute((const void *)dense_score_split,
                        hipFuncAttributeMaxDynamicSharedMemorySize, (int)kSplitLdsBytes);
    const auto blocks = [&](size_t rowsPad) {
        return dim3((unsigned)std::min<size_t>(
            (rowsPad * kpad / 16 + kGConvThreads - 1) / kGConvThreads, 65536));
    };
    hipError_t e = hipMemsetAsync(wild, 0, sizeof(int), st);
    hipLaunchKernelGGL(dense_split_convert, blocks(aRows), dim3(kGConvThreads), 0, st, n, kpad,
                       (size_t)k * n, aRows, d_B, A, wild);
    hipLaunchKernelGGL(dense_split_convert, blocks(gRows), dim3(kGConvThreads), 0, st, n, kpad,
                       (size_t)r * n, gRows, d_Gamma, G, wild);
    hipLaunchKernelGGL(dense_score_split, dim3(rowTiles * colTiles), dim3(kGThreads),
                       kSplitLdsBytes, st, k, r, kpad, rowTiles, colTiles,
                       (const __bf16 *)A, (const __bf16 *)G, partV, partJ, (const int *)wild);
    hipLaunchKernelGGL(alpha_value_merge, dim3((k + 255) / 256), dim3(256), 0, st, k, colTiles,
                       partV, partJ, d_pi, d_V, d_action, d_alpha, (const int *)wild);
    if (e == hipSuccess)
        e = hipGetLastError();
    int flag = 0;
    if (e == hipSuccess)
        e = hipMemcpyAsync(&flag, wild, sizeof(int), hipMemcpyDeviceToHost, st);
    if (e == hipSuccess)
        e = hipStreamSynchronize(st);
    if (e != hipSuccess)
        return hip_fail(e, fn, "Kernel execution failed.", NOVA_ERROR_KERNEL_EXECUTION);
    *done = flag == 0;
    return NOVA_SUCCESS;
}

} // namespace nova_amd

using namespace nova_amd;

extern "C" int nova_amd_alpha_vectors_value_and_action_gpu(unsigned int n, unsigned int r,
        const float *d_Gamma, const unsigned int *d_pi, unsigned int k, const float *d_B,
        int precision, float *d_V, unsigned int *d_action, int *d_alpha)
{
    NOVA_AMD_API_LOCK();
    const char *fn = "nova_amd_alpha_vectors_value_and_action_gpu";
    if (n == 0 || r == 0 || k == 0 || d_Gamma == nullptr || d_pi == nullptr ||
            d_B == nullptr || d_V == nullptr || d_action == nullptr || precision < 0 ||
            precision > 2 || (r + kVT - 1) / kVT > 65535u) {
        NOVA_ERR(fn, "Invalid arguments (n, r, k > 0, r <= 4,194,240; device arrays; "
                     "precision 0, 1 or 2).");
        return NOVA_ERROR_INVALID_DATA;
    }
    std::lock_guard<std::mutex> lock(g_valueMutex);
    hipStream_t st = stream();
    const unsigned few = few_beliefs(n, k, r, precision);
    const bool exact = precision == 0 || few != 0;       // on the vector ALUs
    const unsigned tileW = exact ? exact_tile(few) : (unsigned)kGT;
    const unsigned colTiles = (r + tileW - 1) / tileW;
    const unsigned rowTiles = (k + kGT - 1) / kGT;
    const size_t inSize = precision == 2 ? sizeof(__bf16) : sizeof(float);
    const unsigned kpad = (n + kGKPad - 1) / kGKPad * kGKPad;
    const size_t bPart = up256((size_t)colTiles * k * sizeof(float));
    size_t bytes = 2 * bPart;
    size_t bA = 0, bG = 0, bS = 0;
    void *mem = nullptr;
    if (!exact && precision == 1) {
        bool done = false;
        const int rcs = value_split(n, r, d_Gamma, d_pi, k, d_B, d_V, d_action, d_alpha, fn, &done);
        if (rcs != NOVA_SUCCESS || done)
            return rcs;
    }
    if (!exact) {
        bA = up256((size_t)rowTiles * kGT * kpad * inSize);
        bG = up256((size_t)colTiles * kGT * kpad * inSize);
        bS = up256(sizeof(float) * kpad);
        bytes += bA + bG + bS;
    }
    int rc = arena_get(g_valueArena, bytes, fn, mem);
    if (rc != NOVA_SUCCESS)
        return rc;
    char *c = static_cast<char *>(mem);
    float *partV = reinterpret_cast<float *>(c);
    int *partJ = reinterpret_cast<int *>(c + bPart);
    hipError_t e = hipSuccess;
    if (exact) {
        g_valueShape = DenseShape();   // the partials may overwrite the dense operands' padding
        launch_exact(few, precision, k, n, r, d_B, d_Gamma, d_pi, partV, partJ, d_V, d_action,
                     d_alpha, st);
    } else {
        void *A = c + 2 * bPart, *Gi = c + 2 * bPart + bA;
        float *ones = reinterpret_cast<float *>(c + 2 * bPart + bA + bG);
        // the zero padding of the row-major layouts survives between calls of one shape and
        // layout; another shape or layout clears it (the k-blocked layout is written whole)
        const bool blocked = precision == 2 && !dense_legacy_bf16();
        const int layout = blocked ? 3 : precision;
        const bool same = g_valueShape.mem == mem && g_valueShape.k == k &&
                          g_valueShape.n == n && g_valueShape.r == r &&
                          g_valueShape.precision == layout;
        if (!same) {
            e = hipMemsetAsync(A, 0, bA + bG, st);
            hipLaunchKernelGGL(fill_ones, dim3((kpad + 255) / 256), dim3(256), 0, st, kpad, ones);
            g_valueShape.mem = mem;
            g_valueShape.k = k;
            g_valueShape.n = n;
            g_valueShape.r = r;
            g_valueShape.precision = layout;
        }
        const size_t kn = (size_t)k * n, rn = (size_t)r * n;
        const unsigned ga = (unsigned)std::min<size_t>((kn + kGConvThreads - 1) / kGConvThreads,
                                                       65536);
        const unsigned gg = (unsigned)std::min<size_t>((rn + kGConvThreads - 1) / kGConvThreads,
                                                       65536);
        const dim3 sg(rowTiles * colTiles, 1);
        if (blocked) {
            // k-blocked operands, every padding element written by the conversion
            const size_t ta = (size_t)rowTiles * kGT * kpad, tg = (size_t)colTiles * kGT * kpad;
            const unsigned ca = (unsigned)std::min<size_t>(
                (ta / 8 + kGConvThreads - 1) / kGConvThreads, 65536);
            const unsigned cg = (unsigned)std::min<size_t>(
                (tg / 8 + kGConvThreads - 1) / kGConvThreads, 65536);
            hipFuncSetAttribute((const void *)dense_score_bf16,
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)kGDlLdsBytes);
            hipLaunchKernelGGL(dense_convert_blk, dim3(ca), dim3(kGConvThreads), 0, st, n, kpad,
                               kn, (size_t)rowTiles * kGT, d_B, static_cast<__bf16 *>(A));
            hipLaunchKernelGGL(dense_convert_blk, dim3(cg), dim3(kGConvThreads), 0, st, n, kpad,
                               rn, (size_t)colTiles * kGT, d_Gamma, static_cast<__bf16 *>(Gi));
            hipLaunchKernelGGL(dense_score_bf16, sg, dim3(kGThreads), kGDlLdsBytes, st, k, r,
                               kpad, 1u, 1u, rowTiles, colTiles, 0u, (size_t)0,
                               static_cast<const __bf16 *>(A), static_cast<const __bf16 *>(Gi),
                               partV, partJ);
        } else if (precision == 2) {
            hipFuncSetAttribute((const void *)dense_score<__bf16>,
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)kGLdsBytes);
            hipLaunchKernelGGL(dense_convert<__bf16>, dim3(ga), dim3(kGConvThreads), 0, st, n,
                               kpad, kn, d_B, static_cast<__bf16 *>(A));
            hipLaunchKernelGGL(dense_convert<__bf16>, dim3(gg), dim3(kGConvThreads), 0, st, n,
                               kpad, rn, d_Gamma, static_cast<__bf16 *>(Gi));
            hipLaunchKernelGGL(dense_score<__bf16>, sg, dim3(kGThreads), kGLdsBytes, st, k, r,
                               kpad, 1u, 1u, rowTiles, colTiles, static_cast<const __bf16 *>(A),
                               static_cast<const __bf16 *>(Gi), ones, partV, partJ);
        } else {
            hipFuncSetAttribute((const void *)dense_score<float>,
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)kGLdsBytes);
            hipLaunchKernelGGL(dense_convert<float>, dim3(ga), dim3(kGConvThreads), 0, st, n,
                               kpad, kn, d_B, static_cast<float *>(A));
            hipLaunchKernelGGL(dense_convert<float>, dim3(gg), dim3(kGConvThreads), 0, st, n,
                               kpad, rn, d_Gamma, static_cast<float *>(Gi));
            hipLaunchKernelGGL(dense_score<float>, sg, dim3(kGThreads), kGLdsBytes, st, k, r,
                               kpad, 1u, 1u, rowTiles, colTiles, static_cast<const float *>(A),
                               static_cast<const float *>(Gi), ones, partV, partJ);
        }
    }
    if (!exact)
        hipLaunchKernelGGL(alpha_value_merge, dim3((k + 255) / 256), dim3(256), 0, st, k,
                           colTiles, partV, partJ, d_pi, d_V, d_action, d_alpha,
                           (const int *)nullptr);
    if (e == hipSuccess)
        e = hipGetLastError();
    if (e == hipSuccess)
        e = hipStreamSynchronize(st);
    if (e != hipSuccess)
        return hip_fail(e, fn, "Kernel execution failed.", NOVA_ERROR_KERNEL_EXECUTION);
    return NOVA_SUCCESS;
}

extern "C" int nova_amd_belief_update_batch_gpu(const nova::POMDP *pomdp, unsigned int k,
        const float *d_B, const unsigned int *d_action, const unsigned int *d_observation,
        float *d_Bp, int *d_status)
{
    NOVA_AMD_API_LOCK();
    const char *fn = "nova_amd_belief_update_batch_gpu";
    if (pomdp == nullptr || pomdp->n == 0 || pomdp->ns == 0 || pomdp->m == 0 ||
            pomdp->z == 0 || pomdp->S == nullptr || pomdp->T == nullptr ||
            pomdp->d_S == nullptr || pomdp->d_O == nullptr || k == 0 || d_B == nullptr ||
            d_action == nullptr || d_observation == nullptr || d_Bp == nullptr ||
            d_status == nullptr) {
        NOVA_ERR(fn, "Invalid arguments (a device-resident POMDP with its host arrays, "
                     "k > 0, device arrays).");
        return NOVA_ERROR_INVALID_DATA;
    }
    return belief_update_rows(pomdp, k, d_B, nullptr, d_action, d_observation, d_Bp, d_status,
                              fn);
}

// ---- the exact value/action without allocation
//
// The per-(belief, alpha tile) partials of the exact path live in `scratch`, a static device
// array of kNoAllocScratchBytes that every GPU the library runs on holds until the process
// ends. Host code never passes the array's name to a kernel (on the host it is only a stand-in
// for the symbol): its device address is looked up once per device with
// hipGetSymbolAddress and kept in g_scratchDev. Every partial the merge reads is written by the
// tile kernel of the same call first, so nothing in it has to start at zero. The contents
// persist between calls; calls on one GPU share the array, and overlapping ones would race
// (the library lock serialises the calls of one process).
constexpr size_t kNoAllocScratchBytes = (size_t)16 << 20;
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

namespace {
constexpr int kScratchDevices = 64;
void *g_scratchDev[kScratchDevices];
hipError_t g_scratchErr[kScratchDevices];
std::once_flag g_scratchOnce[kScratchDevices];

// Device address of `scratch` on the current device (nullptr and an error message on failure).
void *scratch_address(const char *fn)
{
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess || dev < 0 || dev >= kScratchDevices) {
        hip_fail(e != hipSuccess ? e : hipErrorInvalidDevice, fn,
                 "No usable current device for the scratch array.", NOVA_ERROR_INVALID_DATA);
        return nullptr;
    }
    std::call_once(g_scratchOnce[dev], [dev]() {
        void *p = nullptr;
        g_scratchErr[dev] = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        g_scratchDev[dev] = g_scratchErr[dev] == hipSuccess ? p : nullptr;
    });
    if (g_scratchDev[dev] == nullptr)
        hip_fail(g_scratchErr[dev] != hipSuccess ? g_scratchErr[dev] : hipErrorInvalidSymbol, fn,
                 "Could not look up the device address of the scratch array.",
                 NOVA_ERROR_KERNEL_EXECUTION);
    return g_scratchDev[dev];
}
} // namespace

extern "C" int nova_amd_alpha_vectors_value_and_action_noalloc_gpu(unsigned int n,
        unsigned int r, const float *d_Gamma, const unsigned int *d_pi, unsigned int k,
        const float *d_B, float *d_V, unsigned int *d_action, int *d_alpha)
{
    NOVA_AMD_API_LOCK();
    const char *fn = "nova_amd_alpha_vectors_value_and_action_noalloc_gpu";
    if (n == 0 || r == 0 || k == 0 || d_Gamma == nullptr || d_pi == nullptr ||
            d_B == nullptr || d_V == nullptr || d_action == nullptr ||
            (r + kVT - 1) / kVT > 65535u) {
        NOVA_ERR(fn, "Invalid arguments (n, r, k > 0, r <= 4,194,240; device arrays).");
        return NOVA_ERROR_INVALID_DATA;
    }
    size_t colTiles = (r + kVT - 1) / kVT;
    size_t bPart = up256(colTiles * k * sizeof(float));
    if (2 * bPart > kNoAllocScratchBytes) {
        NOVA_ERR(fn, "ceil(r / 64) * k exceeds the 16 MiB scratch array (at most 2,097,152 "
                     "(belief, 64-alpha tile) partials per call).");
        return NOVA_ERROR_INVALID_DATA;
    }
    char *c = static_cast<char *>(scratch_address(fn));
    if (c == nullptr)
        return NOVA_ERROR_KERNEL_EXECUTION;
    // the narrower tiles of few beliefs have four times the partials: only where they fit too
    unsigned few = few_beliefs(n, k, r, 0);
    if (few) {
        colTiles = (r + kFewAlphas - 1) / kFewAlphas;
        if (2 * up256(colTiles * k * sizeof(float)) <= kNoAllocScratchBytes)
            bPart = up256(colTiles * k * sizeof(float));
        else
            few = 0;
    }
    hipStream_t st = stream();
    float *partV = reinterpret_cast<float *>(c);
    int *partJ = reinterpret_cast<int *>(c + bPart);
    launch_exact(few, 0, k, n, r, d_B, d_Gamma, d_pi, partV, partJ, d_V, d_action, d_alpha, st);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess)
        e = hipStreamSynchronize(st);
    if (e != hipSuccess)
        return hip_fail(e, fn, "Kernel execution failed.", NOVA_ERROR_KERNEL_EXECUTION);
    return NOVA_SUCCESS;
}
