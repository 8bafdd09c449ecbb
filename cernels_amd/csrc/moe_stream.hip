// Routed experts on packed weights where experts average few rows, so that a call is bound by streaming the selected
// experts' weights from HBM rather than by the matrix units (bf16 / fp16 MFMA, gfx950).
//
// The grouped GEMMs of moe_gemm_packed.hip keep one workgroup per CU on 256-row tiles; with a handful of rows per
// expert they leave most of the chip without work (one token of gpt-oss: 92 items on 256 CUs) and wait for an LDS
// stage and a barrier per 64 reduction columns. Here a workgroup owns one 32-column weight fragment of one expert and
// its four waves split the reduction: weights (1 KB per fragment and k-step, read once) and activation rows (L2) both go
// straight to registers, and no wave waits for another until the four partial sums meet in LDS at the end. Four such
// workgroups per CU keep 128 KB of weights in flight (a plain read of 126 MB reaches 5.9 TB/s with 64 KB in flight on
// 176 and more CUs, 4.2 TB/s on 88). What bounds it: HBM, 5.2-5.8 TB/s of weights in a launch of 130 MB and more.
// Tried and slower: workgroups of one wave 0-5%, of eight waves 2-25%, five of four waves per CU (at most 102 registers,
// which spill) 35%.
//
// Two forms share the first projection:
//   few    (T <= 32 tokens, at most 512 pairs, see few_supported): no route. Each workgroup finds its expert and that
//          expert's tokens from the indices by itself (rows are tokens). Up to 16 pairs the down kernel may sum every
//          expert's contribution to its 16 output columns (two launches, few_sums), else it writes a row per pair and the
//          combine sums them (three; the general path takes five).
//   tiles  (up to 512 tokens, at most 8 rows per expert on average): the route's list with M-tiles of 32 rows, then the
//          glu fixup and the combine as on the general path.
// Measured, whole op in us, general path -> here (seeded routing, weights of three layers in turn): gpt-oss shapes (H = F =
// 2880, E = 32, k = 4) T=1 85 -> 43, T=8 234 -> 195, T=32 299 -> 273, T=48 311 -> 297 (tiles); H=2048 F=512 E=513 k=11
// T=3 90 -> 58, T=28 293 -> 256 (tiles), T=128 580 -> 521, T=400 635 -> 599 (tiles); H=2048 F=768 E=128 k=8 T=1 82 -> 34,
// T=32 207 -> 183 (tiles), T=65 239 -> 221, T=128 245 -> 237 (tiles). Above 8 rows per expert the tiles form loses (12.5 rows:
// 245 -> 252): each wave fetches every row's 128-byte lines itself, where the general path shares them through LDS.
// Precision is the general path's: fp32 accumulation, glu in fp16 segments scaled where needed (moe_packed.h), fp16
// weights scaled per fragment, the routing weight and the sum over slots in fp32, one rounding to bf16.
#include <algorithm>
#include <climits>
#include <type_traits>

#include "moe_packed.h"
#include "moe_split.h"
#include "moe_tile.h"

namespace cmoe {

constexpr int kStWaves = 4, kStThreads = kStWaves * kWave;
constexpr int kStRows = 32;         // rows of an M-tile (one 32-row MFMA block)
constexpr int kFewMaxTokens = 32;   // one 32-row block: rows are tokens
constexpr int kFewMaxPairs = 512;
constexpr int kFewMaxExperts = 1024;  // bitmap of 32 words
constexpr int kFdWaves = 8, kFdThreads = kFdWaves * kWave;  // few: down workgroup with the sum over slots
constexpr int kFdStages = 4;
constexpr int kFdShare = 4;         // stages of a share at least (an expert of fewer is one share). A wave pays for each share it
                                   // begins and ends (the expert's place, a store to LDS): whole op with shares of 1 / 2 / 4
                                   // stages and more, 11 of 513 experts of H 2048 F 512 19.8 / 19.0 / 18.8 us; 230 layers 0.5%,
                                   // 1.8%, 2.3% faster than with equal parts of all experts' stages
constexpr int kFdMaxPairs = 16;    // above: rows per pair and the combine (few_sums)
constexpr int kFewMaxTopk = 64;    // few_select's division by K
// few_select: p / K as a product holds while the error p / 65536 stays below 1 / K; bit 14 of few_row lies above every pair
static_assert(kFewMaxPairs * kFewMaxTopk <= 65536 && kFewMaxPairs <= 0x4000 && kFewMaxTokens <= kWave);
constexpr int kTilesMaxTokens = 512;  // bounds the M-tiles of one popular expert, each of which streams its weights
constexpr int kTilesMaxRows = 8;      // rows per expert on average

struct StreamParams {
    const uint16_t* A;            // first projection: x [T, H]; down: glu fp16
    const uint16_t* B;            // packed weights of this projection
    const float* bias;            // first: [E, 2F]; few down: [E, H]; or null
    const int32_t* idx;           // few: [T, K]
    const void* route_w;          // [T, K]
    int types;                    // of idx and route_w (kPairsI64, kPairsBf16); tiles: 0
    const int32_t* sorted_pairs;  // tiles: the route's lists
    const int32_t* offsets;
    const int32_t* tile_offsets;
    const int32_t* tile_expert;
    const int32_t* meta;
    uint16_t* glu;                // few: row p of pair p; tiles: expert order
    unsigned char* Y;             // tiles down: 24-bit rows, row p of pair p
    uint16_t* out;                // few down: [T, H] bf16
    int8_t* gexp;                 // [F/16, p_cap] power of two of each 16-column glu segment
    int8_t* rsig;                 // tiles: rows with a scaled segment
    int32_t* sync;                // tiles: [1] = some segment is scaled
    const int8_t* wexp;           // down: [E, NF] power of two of each weight fragment
    int32_t* few_e;               // few: [U_max] the u-th smallest expert chosen, -1 past the last
    int16_t* few_row;             // few: [U_max, T] glu row (pair) of (expert u, token t), bit 14 if t names u again, -1: not chosen
    uint8_t* few_scaled;          // few: [U_max, NF of the first projection] some segment is scaled
    int T, K, E, H, F, NF, KS, u_max, nf1;
    int share_log;                // few down with the sum: an expert's stages are cut into 1 << share_log shares
    int p_cap, a_bytes, bias_interleaved;
};

// One wave's share of an item's reduction: stages [s0, s0 + n) of 64 columns, acc += W_frag * A_block (32 rows). Two stages
// are in flight, 8 KB of weights per wave; the last rounds are peeled so that no load sits behind a branch and the waits
// stay exact. ao: byte offset of this lane's row (and 8-column half) in A.
template <typename OpT>
__device__ __forceinline__ void stream_stages(__amdgpu_buffer_rsrc_t rw, uint32_t wo, int bs, __amdgpu_buffer_rsrc_t ra,
                                              uint32_t ao, int s0, int n, f32x16& acc) {
    u32x4 w[2][4], a[2][4];
    auto load = [&](int d, int s) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
            w[d][q] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rw, wo, (4 * s + q) * bs, 0));
#pragma unroll
        for (int q = 0; q < 4; ++q)
            a[d][q] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(ra, ao + 32 * q, s * kBK * 2, 0));
    };
    auto mul = [&](int d) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const OpT wq = __builtin_bit_cast(OpT, w[d][q]), aq = __builtin_bit_cast(OpT, a[d][q]);
            if constexpr (std::is_same_v<OpT, f16x8>) acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(wq, aq, acc, 0, 0, 0);
            else acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wq, aq, acc, 0, 0, 0);
        }
    };
    if (n <= 0) return;
    load(0, s0);
    load(1, s0 + min(1, n - 1));
    int s = 0;
    for (; s + 3 < n; s += 2) {
        mul(0);
        load(0, s0 + s + 2);
        mul(1);
        load(1, s0 + s + 3);
    }
    if (s + 2 < n) {  // three left
        mul(0);
        load(0, s0 + s + 2);
        mul(1);
        mul(0);
    } else {
        mul(0);
        if (s + 1 < n) mul(1);
    }
}

// The sum of the four waves' partial accumulators, by one wave.
__device__ __forceinline__ void sum_parts(const float (*part)[16][kWave], int lane, float (&v)[16]) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        float s = part[0][r][lane];
#pragma unroll
        for (int w = 1; w < kStWaves; ++w) s += part[w][r][lane];
        v[r] = s;
    }
}

// One 32-row block's glu of one weight fragment: element r of v is row lane & 31 (valid: an existing one, glu row gr),
// fragment column 8(r/4) + 4 half + r%4; bias: the fragment's 16 gate, then 16 up values (HAS_BIAS). Stores the fp16
// segment and its power of two; true on lanes whose segment is scaled.
template <int MODE, int ACT, bool HAS_BIAS, typename V>
__device__ __forceinline__ bool store_glu(const StreamParams& prm, const V& v, bool valid, long long gr, int fc, int half,
                                          const float* bias) {
    constexpr int NV = MODE == kModePkGateUp ? 8 : 16;  // glu columns per lane
    float g[NV];
    float m = 0.f;  // the segment's largest |glu| (a nan is passed over)
    if constexpr (MODE == kModePkGateUp) {
#pragma unroll
        for (int r = 0; r < 8; ++r) {
            float gv = v[r], uv = v[8 + r];
            if constexpr (HAS_BIAS) {
                const int col = 8 * (r >> 2) + 4 * half + (r & 3);
                gv += bias[col];
                uv += bias[16 + col];
            }
            g[r] = swiglu<ACT>(gv, uv);
            m = fmaxf(m, fabsf(g[r]));
        }
    } else {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            g[r] = act_plain<ACT>(v[r]);
            m = fmaxf(m, fabsf(g[r]));
        }
    }
    m = max_halves(m);  // both lanes of the row
    const int sg = glu_needs_scale(m) ? glu_scale_exp(m) : 0;  // 0 also for an all-zero segment
    const bool scaled = valid && sg != 0;
    if (__ballot(scaled) != 0ull) {  // rare
#pragma unroll
        for (int r = 0; r < NV; ++r) g[r] = __builtin_amdgcn_ldexpf(g[r], -sg);
    }
    if (valid) {  // lanes l and l ^ 32 hold the same row, so both run this or neither
        uint32_t h[NV / 2];
#pragma unroll
        for (int r = 0; r < NV / 2; ++r) h[r] = pack_f16x2(g[2 * r], g[2 * r + 1]);
        const int8_t se = (int8_t)(m == 0.f ? kGluAnyScale : sg);
        if constexpr (MODE == kModePkGateUp) {
            swap_halves(h[0], h[2]);  // lane l: columns 0-7, lane l + 32: columns 8-15
            swap_halves(h[1], h[3]);
            *reinterpret_cast<u32x4*>(prm.glu + gr * prm.F + 16 * fc + 8 * half) = u32x4{h[0], h[1], h[2], h[3]};
            if (half == 0) prm.gexp[(long long)fc * prm.p_cap + gr] = se;
        } else {
#pragma unroll
            for (int d = 0; d < 2; ++d) {  // lane l: columns 0-15, lane l + 32: columns 16-31
                swap_halves(h[d], h[4 + d]);
                swap_halves(h[2 + d], h[6 + d]);
            }
            u32x4* o = reinterpret_cast<u32x4*>(prm.glu + gr * prm.F + 32 * fc + 16 * half);
            o[0] = u32x4{h[0], h[1], h[4], h[5]};
            o[1] = u32x4{h[2], h[3], h[6], h[7]};
            prm.gexp[(long long)(2 * fc + half) * prm.p_cap + gr] = se;
        }
    }
    return scaled;
}

// 32 columns of a Y row as 24-bit floats: a lane holds columns 8i + 4 half + 0..3 (both half-waves active for the row); after
// the exchange lane l has columns 0-15 and lane l + 32 columns 16-31, 48 bytes each, at y.
template <typename V>
__device__ __forceinline__ void pack_y(const V& v, float ws, u32x4* y) {
    f24x4 q[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) q[i] = pack_f24x4(v[4 * i] * ws, v[4 * i + 1] * ws, v[4 * i + 2] * ws, v[4 * i + 3] * ws);
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        swap_halves(q[0].d[d], q[2].d[d]);
        swap_halves(q[1].d[d], q[3].d[d]);
    }
    y[0] = u32x4{q[0].d[0], q[0].d[1], q[0].d[2], q[2].d[0]};
    y[1] = u32x4{q[2].d[1], q[2].d[2], q[1].d[0], q[1].d[1]};
    y[2] = u32x4{q[1].d[2], q[3].d[0], q[3].d[1], q[3].d[2]};
}

// The same, straight to the Y row of pair p (fragment fc).
template <typename V>
__device__ __forceinline__ void store_y(unsigned char* Y, long long p, int H, int fc, int half, const V& v, float ws) {
    pack_y(v, ws, reinterpret_cast<u32x4*>(Y + (p * H + 32 * fc + 16 * half) * 3));
}

// few: the u-th smallest distinct expert of the indices (-1: fewer than u + 1), and in tokp[t] the first pair of token t that
// names it, with bit 16 set if further pairs of t do (INT_MAX: none). One wave by itself: its own LDS words (a wave's LDS
// operations run in order), no workgroup barrier.
__device__ __forceinline__ int few_select(const int32_t* __restrict__ idx, int types, int P, int E, int K, int u, int lane,
                                          uint32_t* bits, int* tokp) {
    int ev[kFewMaxPairs / kWave];
#pragma unroll
    for (int c = 0; c < kFewMaxPairs / kWave; ++c) {
        ev[c] = -1;
        if (kWave * c < P) {  // uniform
            const int p = lane + kWave * c;
            const int v = p < P ? pair_id(idx, types, p) : -1;
            ev[c] = (unsigned)v < (unsigned)E ? v : -1;
        }
    }
    if (lane < kFewMaxExperts / 32) bits[lane] = 0u;
    if (lane < kFewMaxTokens) tokp[lane] = INT_MAX;
#pragma unroll
    for (int c = 0; c < kFewMaxPairs / kWave; ++c)
        if (ev[c] >= 0) atomicOr(&bits[ev[c] >> 5], 1u << (ev[c] & 31));
    uint32_t bw = lane < kFewMaxExperts / 32 ? bits[lane] : 0u;
    const int cnt = __popc(bw);  // 0..32
    const uint64_t lt = lane == 0 ? 0ull : (~0ull >> (kWave - lane));
    int excl = 0;  // prefix sum over the lower lanes, bit by bit of cnt
#pragma unroll
    for (int b = 0; b < 6; ++b) excl += __popcll(__ballot((cnt >> b) & 1) & lt) << b;
    const bool holder = u >= excl && u < excl + cnt;  // at most one lane
    int eh = 0;
    if (holder) {
        for (int r = u - excl; r > 0; --r) bw &= bw - 1;
        eh = lane * 32 + __ffs(bw) - 1;
    }
    const uint64_t hb = __ballot(holder);
    if (hb == 0ull) return -1;
    const int e = __builtin_amdgcn_readlane(eh, __ffsll((unsigned long long)hb) - 1);
    const int magic = 65536 / K + 1;  // p / K = p * magic >> 16
#pragma unroll
    for (int c = 0; c < kFewMaxPairs / kWave; ++c)
        if (ev[c] == e) {
            const int p = lane + kWave * c;
            atomicMin(&tokp[(p * magic) >> 16], p);
        }
#pragma unroll
    for (int c = 0; c < kFewMaxPairs / kWave; ++c)
        if (ev[c] == e) {
            const int p = lane + kWave * c, t = (p * magic) >> 16;
            if ((tokp[t] & 0xffff) != p) atomicOr(&tokp[t], 0x10000);
        }
    return e;
}

// First projection: glu rows = act(A W1 (+ b1)) of one expert's rows and one weight fragment (16 glu columns for
// gate_up, 32 for the non-gated projection). grid: (NF, u_max) few, (NF, tiles) tiles; neighbours in x read
// neighbouring 1 KB pieces of one bundle.
template <int MODE, int ACT, bool HAS_BIAS, bool FEW>
__global__ __launch_bounds__(kStThreads, 4) void moe_stream_first_kernel(StreamParams prm) {
    __shared__ float part[kStWaves][16][kWave];
    __shared__ float s_bias[32];
    __shared__ uint32_t s_bits[FEW ? kStWaves : 1][kFewMaxExperts / 32];
    __shared__ int s_tokp[FEW ? kStWaves : 1][kFewMaxTokens];
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int lrow = lane & 31, half = lane >> 5;
    const int fc = blockIdx.x;
    const int nst = prm.H / kBK;
    const int s0 = wave * nst / kStWaves, n = (wave + 1) * nst / kStWaves - s0;

    int e, row_begin = 0, rows = 0;
    int my_pair = INT_MAX, again = 0;  // few: this lane's token's glu row, and whether the token names e again
    uint32_t ao;
    if constexpr (FEW) {
        e = few_select(prm.idx, prm.types, prm.T * prm.K, prm.E, prm.K, blockIdx.y, lane, s_bits[wave], s_tokp[wave]);
        if (e < 0) {  // the same in every wave
            if (fc == 0 && tid == 0) prm.few_e[blockIdx.y] = -1;
            if (tid == 0) prm.few_scaled[(long long)blockIdx.y * prm.NF + fc] = 0;
            return;
        }
        int tp = INT_MAX;
        if (lrow < prm.T) tp = s_tokp[wave][lrow];
        if (tp != INT_MAX) {
            my_pair = tp & 0xffff;
            again = tp >> 16;
        }
        // rows of tokens that did not choose e read the first such token's row and are dropped
        const uint64_t have = __ballot(my_pair != INT_MAX);
        const int t = my_pair != INT_MAX ? lrow : (__ffsll((unsigned long long)have) - 1) & 31;
        ao = (uint32_t)t * (uint32_t)(prm.H * 2) + 16u * half;
    } else {
        const int t = blockIdx.y;
        if (t >= prm.meta[0]) return;
        e = prm.tile_expert[t];
        const int t0 = prm.tile_offsets[e], seg0 = prm.offsets[e];
        tile_rows(t - t0, prm.tile_offsets[e + 1] - t0, prm.offsets[e + 1] - seg0, row_begin, rows);
        row_begin += seg0;
        const int pr = prm.sorted_pairs[row_begin + min(lrow, rows - 1)];
        ao = (uint32_t)(pr / prm.K) * (uint32_t)(prm.H * 2) + 16u * half;
    }
    float bv = 0.f;  // bias of the fragment's column tid % 32 (16 gate, then 16 up)
    if constexpr (HAS_BIAS) {
        const int f = (tid >> 4) & 1, col = 16 * fc + (tid & 15);
        const float* be = prm.bias + (long long)e * 2 * prm.F;
        bv = prm.bias_interleaved ? be[2 * col + f] : be[f * prm.F + col];
    }
    const int nw = min(8, prm.NF - 8 * (fc >> 3));
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(prm.B + packed_frag(e, fc, 0, prm.NF, prm.KS) * kPkFrag), (short)0, (prm.KS - 1) * nw * 1024 + 1024, kBufferWord3);
    const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void*)prm.A, (short)0, prm.a_bytes, kBufferWord3);
    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
    stream_stages<bf16x8>(rw, lane * 16u, nw * 1024, ra, ao, s0, n, acc);
#pragma unroll
    for (int r = 0; r < 16; ++r) part[wave][r][lane] = acc[r];
    if constexpr (HAS_BIAS) {
        if (tid < 32) s_bias[tid] = bv;
    }
    __syncthreads();
    if (wave != 0) return;

    // ---- epilogue: element r is row lane & 31, fragment column 8(r/4) + 4 half + r%4.
    float v[16];
    sum_parts(part, lane, v);
    bool valid;
    long long gr;
    if constexpr (FEW) {
        valid = my_pair != INT_MAX;
        gr = my_pair;
    } else {
        valid = lrow < rows;
        gr = row_begin + lrow;
    }
    const bool scaled = store_glu<MODE, ACT, HAS_BIAS>(prm, v, valid, gr, fc, half, s_bias);
    if constexpr (!FEW) {
        if (scaled) {
            if (half == 0) prm.rsig[gr] = 1;
            prm.sync[1] = 1;
        }
    }
    if constexpr (FEW) {
        const uint64_t sb = __ballot(scaled);
        const long long u = blockIdx.y;
        if (lane == 0) prm.few_scaled[u * prm.NF + fc] = sb != 0ull;
        if (fc == 0) {  // the lists that the down kernel walks
            if (lane == 0) prm.few_e[u] = e;
            if (lane < prm.T) prm.few_row[u * prm.T + lane] = (int16_t)(valid ? my_pair | again << 14 : -1);
        }
    }
}

// tiles: Y[p, 32 columns of fragment c] = w_p * (glu row . W2_e) for the rows of one M-tile, as 24-bit floats at the pair's
// own row. grid (NF, tiles).
__global__ __launch_bounds__(kStThreads, 4) void moe_stream_down_kernel(StreamParams prm) {
    __shared__ float part[kStWaves][16][kWave];
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int lrow = lane & 31, half = lane >> 5;
    const int fc = blockIdx.x, t = blockIdx.y;
    if (t >= prm.meta[0]) return;
    const int e = prm.tile_expert[t];
    const int t0 = prm.tile_offsets[e], seg0 = prm.offsets[e];
    int row_begin, rows;
    tile_rows(t - t0, prm.tile_offsets[e + 1] - t0, prm.offsets[e + 1] - seg0, row_begin, rows);
    row_begin += seg0;
    const int nst = prm.F / kBK;
    const int s0 = wave * nst / kStWaves, n = (wave + 1) * nst / kStWaves - s0;
    const int row = min(lrow, rows - 1);
    const long long p = prm.sorted_pairs[row_begin + row];
    const float ws = __builtin_amdgcn_ldexpf(static_cast<const float*>(prm.route_w)[p], prm.wexp[(long long)e * prm.NF + fc]);
    const int nw = min(8, prm.NF - 8 * (fc >> 3));
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(prm.B + packed_frag(e, fc, 0, prm.NF, prm.KS) * kPkFrag), (short)0, (prm.KS - 1) * nw * 1024 + 1024, kBufferWord3);
    const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void*)(prm.A + (long long)row_begin * prm.F), (short)0,
                                                                        rows * prm.F * 2, kBufferWord3);
    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
    stream_stages<f16x8>(rw, lane * 16u, nw * 1024, ra, (uint32_t)row * (uint32_t)(prm.F * 2) + 16u * half, s0, n, acc);
#pragma unroll
    for (int r = 0; r < 16; ++r) part[wave][r][lane] = acc[r];
    __syncthreads();
    if (wave != 0 || lrow >= rows) return;  // lanes l and l ^ 32 hold the same row
    float v[16];
    sum_parts(part, lane, v);
    store_y(prm.Y, p, prm.H, fc, half, v, ws);
}

// few: Y[p, 32 columns of fragment c] = w_p * (glu row . W2_e) for the tokens of the u-th expert, as 24-bit floats at the
// pair's own row. grid (NF, u_max).
__global__ __launch_bounds__(kStThreads, 4) void moe_few_down_rows_kernel(StreamParams prm) {
    __shared__ float part[kStWaves][16][kWave];
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int lrow = lane & 31, half = lane >> 5;
    const int fc = blockIdx.x;
    const long long u = blockIdx.y;
    const int e = prm.few_e[u];
    int fr = lrow < prm.T ? prm.few_row[u * prm.T + lrow] : -1;
    int flags = 0;
    for (int i = lane; i < prm.nf1; i += kWave) flags |= prm.few_scaled[u * prm.nf1 + i];
    if (e < 0) return;
    const bool any_scaled = __ballot(flags != 0) != 0ull;
    const uint64_t have = __ballot(fr >= 0);
    const int first = __builtin_amdgcn_readlane(fr, (__ffsll((unsigned long long)have) - 1) & 63);
    const bool valid = fr >= 0, again = valid && (fr & 0x4000);
    const int p = (valid ? fr : first) & 0x3fff;  // tokens without this expert read its first token's row and are dropped
    const int nst = prm.F / kBK;
    const int s0 = wave * nst / kStWaves, n = (wave + 1) * nst / kStWaves - s0;
    const int wx = prm.wexp[(long long)e * prm.NF + fc];
    int smax = 0;  // power of two of the glu row
    const float rw0 = pair_weight(prm.route_w, prm.types, p);
    const uint32_t ao = (uint32_t)p * (uint32_t)(prm.F * 2) + 16u * half;
    const int nw = min(8, prm.NF - 8 * (fc >> 3));
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(prm.B + packed_frag(e, fc, 0, prm.NF, prm.KS) * kPkFrag), (short)0, (prm.KS - 1) * nw * 1024 + 1024, kBufferWord3);
    const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void*)prm.A, (short)0, prm.a_bytes, kBufferWord3);
    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
    if (!any_scaled) {
        stream_stages<f16x8>(rw, lane * 16u, nw * 1024, ra, ao, s0, n, acc);
    } else {  // some segment of this expert's rows is scaled: every segment to its row's largest scale first
        smax = kGluAnyScale;
        for (int g = 0; g < prm.F / 16; ++g) smax = max(smax, (int)prm.gexp[(long long)g * prm.p_cap + p]);
        if (smax == kGluAnyScale) smax = 0;
        for (int ks = 4 * s0; ks < 4 * (s0 + n); ++ks) {  // a k-step is one 16-column segment
            const f16x8 wq = __builtin_bit_cast(f16x8, __builtin_amdgcn_raw_buffer_load_b128(rw, lane * 16u, ks * nw * 1024, 0));
            f16x8 aq = __builtin_bit_cast(f16x8, __builtin_amdgcn_raw_buffer_load_b128(ra, ao, ks * 32, 0));
            const int d = min(0, (int)prm.gexp[(long long)ks * prm.p_cap + p] - smax);
#pragma unroll
            for (int j = 0; j < 8; ++j) aq[j] = (_Float16)__builtin_amdgcn_ldexpf((float)aq[j], d);
            acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(wq, aq, acc, 0, 0, 0);
        }
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) part[wave][r][lane] = acc[r];
    __syncthreads();
    if (wave != 0 || !valid) return;  // lanes l and l ^ 32 hold the same row
    float v[16];
    sum_parts(part, lane, v);
    // The weight and the fragment's power come first, the row's power last, as on the general path: w 2^(wx + smax) in one factor
    // would be subnormal for rows of tiny glu (smax down to -126) whose products are not.
    auto store = [&](int pp, float w) {
        const float ws = __builtin_amdgcn_ldexpf(w, wx);
        if (!any_scaled) {
            store_y(prm.Y, pp, prm.H, fc, half, v, ws);
            return;
        }
        float y[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) y[r] = __builtin_amdgcn_ldexpf(v[r] * ws, smax);
        store_y(prm.Y, pp, prm.H, fc, half, y, 1.f);
    };
    store(p, rw0);
    if (again)  // further slots of the token that name the same expert
        for (int k = 0; k < prm.K; ++k) {
            const int pp = lrow * prm.K + k;
            if (pp != p && pair_id(prm.idx, prm.types, pp) == e) store(pp, pair_weight(prm.route_w, prm.types, pp));
        }
}

// few, at most kFdMaxPairs pairs: out[t, 16 columns] = bf16( sum over the slots k of t of w_k * (glu row . W2_e + b2_e) ), in slot
// order, which saves the combine's launch. grid H / 16: a workgroup takes one half of a 32-column weight fragment for all
// experts. An expert's 64-column stages are cut into up to kFdWaves shares whose number and bounds depend on F alone (kFdShare
// stages and more). The shares of all experts go round the waves, rotated by one from expert to expert (they differ
// by a stage); a wave walks its own with kFdStages stages in flight and leaves each one's partial sums in LDS (16x16x32 MFMA,
// tokens as columns). A thread per pair and column then adds the shares in order. So a row depends on its token and that
// token's slots alone: not on the other tokens of the call, nor on how the experts are numbered.
template <bool HAS_BIAS>
__global__ __launch_bounds__(kFdThreads) void moe_few_down_kernel(StreamParams prm) {
    const int T = prm.T, um = prm.u_max, P = prm.T * prm.K;  // all <= kFdMaxPairs
    __shared__ int s_e[kFdMaxPairs];
    __shared__ int s_id[kFdMaxPairs];                 // pairs' experts, -1: out of range
    __shared__ int s_row[kFdMaxPairs * kFdMaxPairs];  // [um, T] glu row, -1: not chosen
    __shared__ int s_max[kFdMaxPairs];                // where segments are scaled: the largest power of two of each glu row
    __shared__ __attribute__((aligned(16))) float s_part[kFdWaves][kFdMaxPairs][16];  // share, glu row, column
    __shared__ float s_y[kFdMaxPairs][16];            // slots' weighted rows
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int fc = blockIdx.x >> 1, hf = blockIdx.x & 1;  // weight fragment, its half
    const int l16 = lane & 15, grp = lane >> 4;

    const int my_e = tid < um ? prm.few_e[tid] : -1;
    int flags = 0;
    const int nfl = um * prm.nf1;
    for (int i = tid; i < nfl; i += kFdThreads) flags |= prm.few_scaled[i];
    if (tid < um * T) {
        const int r = prm.few_row[tid];
        s_row[tid] = r < 0 ? -1 : r & 0x3fff;
    }
    if (tid < um) s_e[tid] = my_e;
    if (tid < P) {
        const int e = pair_id(prm.idx, prm.types, tid);
        s_id[tid] = (unsigned)e < (unsigned)prm.E ? e : -1;
    }
    const int U = __builtin_amdgcn_readfirstlane(__syncthreads_count(my_e >= 0));  // the entries are a prefix
    const bool any_scaled = __syncthreads_or(flags) != 0;
    if (any_scaled) {
        if (tid < U * T && s_row[tid] >= 0) {
            const int p = s_row[tid];
            int smax = kGluAnyScale;
            for (int u = 0; u < prm.F / 16; ++u) smax = max(smax, (int)prm.gexp[(long long)u * prm.p_cap + p]);
            s_max[p] = smax == kGluAnyScale ? 0 : smax;
        }
        __syncthreads();
    }

    const int S = prm.F / kBK;  // stages per expert
    // share j of expert u is number (u << share_log) + (j - u) % shares of the list that goes round the waves; none is empty
    const int sl = prm.share_log, shares = 1 << sl, tasks = U << sl;
    auto share_of = [&](int t) { return (t + (t >> sl)) & (shares - 1); };
    auto bound = [&](int j) { return (j * S) >> sl; };
    int cnt = 0;  // this wave's stages
    for (int t = wave; t < tasks; t += kFdWaves) cnt += bound(share_of(t) + 1) - bound(share_of(t));
    const int nw = min(8, prm.NF - 8 * (fc >> 3)), bs = nw * 1024;
    const uint32_t wo = (uint32_t)((grp >> 1) * bs + (grp & 1) * 512 + (16 * hf + l16) * 16);
    const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void*)prm.A, (short)0, prm.a_bytes, kBufferWord3);
    const int t16 = min(l16, T - 1);

    // the epilogue's pair and column of this thread (the first 16 P threads)
    const int q = tid >> 4, c = tid & 15;
    const int eq = q < P ? s_id[q] : -1, e0 = max(eq, 0);
    int first = q;  // the glu row of the pair: the token's first pair that names the expert
    if (eq >= 0)
        for (int k = q / prm.K * prm.K; k < first; ++k)
            if (s_id[k] == eq) first = k;
    const int wx = prm.wexp[(long long)e0 * prm.NF + fc];
    const float wq = pair_weight(prm.route_w, prm.types, min(q, P - 1));
    float bq = 0.f;
    if constexpr (HAS_BIAS) bq = prm.bias[(long long)e0 * prm.H + 16 * blockIdx.x + c];

    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    constexpr int D = kFdStages;
    u32x4 w[D][2], a[D][2];

    auto run = [&](auto sc) {
        constexpr bool SC = decltype(sc)::value;
        // a walk over this wave's stages: stage s of [.., end) of share t
        struct Walk { int t, s, end; };
        auto settle = [&](Walk& k) {
            if (k.s == k.end && k.t + kFdWaves < tasks) {
                k.t += kFdWaves;
                k.s = bound(share_of(k.t));
                k.end = bound(share_of(k.t) + 1);
            }
        };
        Walk ld{wave, bound(share_of(wave)), bound(share_of(wave) + 1)};  // stage to load next
        Walk mu = ld;    // stage to multiply next
        int left = cnt;  // stages not loaded yet
        auto load = [&](int d) {
            const int u = ld.t >> sl, e = __builtin_amdgcn_readfirstlane(s_e[u]);
            const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
                (void*)(prm.B + packed_frag(e, fc, 0, prm.NF, prm.KS) * kPkFrag), (short)0, (prm.KS - 1) * bs + 1024, kBufferWord3);
            const uint32_t r = (uint32_t)max(0, s_row[u * T + t16]);  // a token without this expert: row 0, dropped
            const uint32_t ro = r * (uint32_t)(prm.F * 2) + 16u * grp;
#pragma unroll
            for (int i = 0; i < 2; ++i)
                w[d][i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rw, wo, (4 * ld.s + 2 * i) * bs, 0));
#pragma unroll
            for (int i = 0; i < 2; ++i)
                a[d][i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(ra, ro + 64 * i, ld.s * kBK * 2, 0));
            if (--left > 0) {  // past the last stage: the last one again, dropped
                ++ld.s;
                settle(ld);
            }
        };
        auto mul = [&](int d) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                f16x8 aq = __builtin_bit_cast(f16x8, a[d][i]);
                if constexpr (SC) {  // bring the segment to its row's scale
                    const int p = max(0, s_row[(mu.t >> sl) * T + t16]);
                    const int dd = (int)prm.gexp[(long long)(4 * mu.s + 2 * i + (grp >> 1)) * prm.p_cap + p] - s_max[p];
#pragma unroll
                    for (int j = 0; j < 8; ++j) aq[j] = (_Float16)__builtin_amdgcn_ldexpf((float)aq[j], min(dd, 0));
                }
                acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, w[d][i]), aq, acc, 0, 0, 0);
            }
            if (++mu.s == mu.end) {  // the share is whole
                const int p = l16 < T ? s_row[(mu.t >> sl) * T + l16] : -1;
                if (p >= 0) *reinterpret_cast<f32x4*>(&s_part[share_of(mu.t)][p][4 * grp]) = acc;
                acc = f32x4{0.f, 0.f, 0.f, 0.f};
                settle(mu);
            }
        };
        if (cnt > 0) {
#pragma unroll
            for (int d = 0; d < D; ++d) load(d);
        }
        for (int i = 0; i < cnt; i += D) {
#pragma unroll
            for (int d = 0; d < D; ++d) {
                if (i + d < cnt) mul(d);
                load(d);
            }
        }
    };
    if (any_scaled) run(std::true_type{});
    else run(std::false_type{});
    __syncthreads();
    if (eq >= 0) {
        float v = 0.f;
        for (int k = 0; k < shares; ++k) v += s_part[k][first][c];
        float y = v * __builtin_amdgcn_ldexpf(wq, wx);
        if (any_scaled) y = __builtin_amdgcn_ldexpf(y, s_max[first]);
        if constexpr (HAS_BIAS) y += wq * bq;
        s_y[q][c] = y;
    }
    __syncthreads();
    if (q < T) {  // now a token and column
        float s = 0.f;
        for (int k = 0; k < prm.K; ++k)
            if (s_id[q * prm.K + k] >= 0) s += s_y[q * prm.K + k][c];
        prm.out[(long long)q * prm.H + 16 * blockIdx.x + c] = f32_to_bf16_bits(s);
    }
}

// ---- mid: the packed GEMMs as one workgroup per item, two workgroups per CU ------------------------------------------------
// The persistent GEMMs of moe_gemm_packed.hip run one 8-wave workgroup per CU on items of up to 256 rows x 8 fragments. That
// is the best use of the matrix units while every CU has full items, but a CU multiplies nothing while its one workgroup
// stores an item and fills the pipe of the next, a last round that few items share costs as much as a full one, and items of
// fewer than 8 fragments leave waves idle. Here an item is a workgroup of its own, 128 rows x 8 fragments, and a CU holds two
// (64 KB LDS and 128 VGPRs for 8 waves each): the stores of one run under the MFMAs of the other. Which calls take it:
// mid_supported() in moe_gemm_packed.hip. Activations go through LDS (copied there by buffer_load .. lds, double buffered),
// weights straight to registers two 64-column groups ahead. First + second GEMM, persistent -> here (us): 8 non-gated experts
// of H 2048 F 5632, 1024 rows each, 251 + 282 -> 190 + 215 (0.71 -> 0.93 PFLOP/s); 513 experts of H 2048 F 512, 88 rows with Zipf 1.2
// skew, 304 + 236 -> 251 + 222; 128 of F 768, 21 rows, 146 + 85 -> 140 + 80 (5.5 TB/s of weights). Tried and slower over 60 to
// 150 shapes: items of 192 rows x 4 fragments, three per CU (-2% on average, up to 10% where rows cross 192), 256 x 4 (spills),
// 128 x 8 with four waves of two fragments (0-2%, 3% faster under skew); no s_setprio around the MFMAs 0.6%; no order of MFMAs
// and LDS reads 1%; five LDS reads ahead in place of three +0.3%, within the spread.
constexpr int kMidMB = 4, kMidBM = 32 * kMidMB;  // rows of an item
constexpr int kMidWaves = 8, kMidThreads = kMidWaves * kWave;
constexpr int kYRow = 96;  // bytes of a fragment's 32 columns of a Y row
constexpr int kMidGroups = 2;  // 64-column groups of an activation stage (32 KB)

// The k-loop of one wave: one weight fragment (rw) times NMB row blocks. Group g (64 columns) of the reduction sits in
// subtile g % kMidGroups of LDS buffer (g / kMidGroups) & 1; a stage is kMidGroups groups. Weight groups are loaded two
// groups ahead into slot g & 1, and a stage's activations while the stage before it is multiplied; past the end both load the
// last group again. buf(i): LDS buffer i, as an array of its own (a wait that the compiler adds before a read then covers the
// copies into that array only).
template <typename OpT, int NMB, typename Buf, typename CopyA>
__device__ __forceinline__ void mid_loop(__amdgpu_buffer_rsrc_t rw, uint32_t wo, int bs, __amdgpu_buffer_rsrc_t ra, int nG,
                                         int lane, Buf&& buf, CopyA&& copy_a, f32x16 (&acc)[kMidMB]) {
    constexpr int GS = kMidGroups;
    u32x4 w[2][4];
    auto load_w = [&](int d, int g) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
            w[d][q] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rw, wo, (4 * g + q) * bs, 0));
    };
    auto mul = [&](int d, const unsigned char* sub) {
        constexpr int NK = 4 * NMB, R = NMB < 3 ? 2 * NMB : 3;
        auto rd = [&](int k) {
            return *reinterpret_cast<const OpT*>(sub + lds_off((k % NMB) * 32 + (lane & 31), 2 * (k / NMB) + (lane >> 5)));
        };
        OpT af[R];
#pragma unroll
        for (int k = 0; k < R; ++k) af[k] = rd(k);
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int k = 0; k < NK; ++k) {
            const OpT wq = __builtin_bit_cast(OpT, w[d][k / NMB]);
            f32x16& c = acc[k % NMB];
            if constexpr (std::is_same_v<OpT, f16x8>) c = __builtin_amdgcn_mfma_f32_32x32x16_f16(wq, af[k % R], c, 0, 0, 0);
            else c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wq, af[k % R], c, 0, 0, 0);
            if (k + R < NK) af[k % R] = rd(k + R);
        }
        // each activation fragment's MFMA, then the LDS read that refills its registers, in that order
#pragma unroll
        for (int k = 0; k < NK; ++k) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            if (k + R < NK) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_setprio(0);
    };
    asm volatile("" ::: "memory");  // the caller's copies of the first stage are issued before these loads (see stage)
    load_w(0, 0);
    load_w(1, min(1, nG - 1));
    auto stage = [&](int g0, auto bc) {
        constexpr int B = decltype(bc)::value;
        // A stage issues its copies, then 4 GS weight loads, in this order (the clobbers keep it, and no load is ever dead):
        // with at most 4 GS operations in flight this wave's copies of the stage before have landed. After the barrier
        // every wave's have, and every wave's reads of the other buffer are done.
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0x0070 | 4 * GS);  // vmcnt(4 GS), lgkmcnt(0)
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        copy_a(ra, g0 + GS, std::integral_constant<int, 1 - B>{});
        asm volatile("" ::: "memory");
#pragma unroll
        for (int p = 0; p < GS; ++p) {
            const int g = g0 + p, d = p & 1;
            if (g < nG) mul(d, buf(bc) + p * kMidBM * 128);
            asm volatile("" ::: "memory");
            load_w(d, min(g + 2, nG - 1));
        }
    };
    // whole rounds of two stages: groups past the end are skipped (an early exit after the first stage, or a peeled tail,
    // made the compiler move weight registers whose loads were in flight)
    for (int g0 = 0; g0 < nG; g0 += 2 * GS) {
        stage(g0, std::integral_constant<int, 0>{});
        stage(g0 + GS, std::integral_constant<int, 1>{});
    }
#pragma unroll
    for (int d = 0; d < 2; ++d)
#pragma unroll
        for (int q = 0; q < 4; ++q) asm volatile("" ::"v"(w[d][q]));  // the loads past the end have a use
}

template <int MODE, int ACT, bool HAS_BIAS>
__global__ __launch_bounds__(kMidThreads, 4) void moe_mid_kernel(StreamParams prm, int n_tiles) {
    constexpr int GS = kMidGroups, FW = kMidWaves;
    constexpr bool kDown = MODE == kModePkDown;
    using OpT = std::conditional_t<kDown, f16x8, bf16x8>;
    __shared__ __attribute__((aligned(16))) unsigned char sA0[GS * kMidBM * 128];
    __shared__ __attribute__((aligned(16))) unsigned char sA1[GS * kMidBM * 128];
    __shared__ float s_bias[FW][32];
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int lrow = lane & 31, half = lane >> 5;
    // items of XCD x: one contiguous range of the list (M-tiles of an N-tile are neighbours)
    const int total = prm.meta[0] * n_tiles, per = ceil_div(total, 8);
    const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
    if (slot >= per || xcd * per + slot >= total) return;
    const WorkItem it = decode_item(xcd * per + slot, n_tiles, prm.tile_expert, prm.tile_offsets, prm.offsets);
    const int Kd = kDown ? prm.F : prm.H, nG = Kd / kBK;
    const bool active = FW * it.n_idx + wave < prm.NF;  // a wave past the last fragment multiplies the last one again, unstored
    const int fc = min(FW * it.n_idx + wave, prm.NF - 1);
    const int nmb = ceil_div(it.rows, 32);

    // activation copies: thread t takes chunk position t & 7 of rows t >> 3 and 64 + (t >> 3) of every subtile
    constexpr int RP = kMidThreads / 8, NR = kMidBM / RP;
    const int r0 = tid >> 3;
    uint32_t ao[NR];
#pragma unroll
    for (int i = 0; i < NR; ++i) {
        const int row = min(r0 + RP * i, it.rows - 1);
        const int chunk = (tid & 7) ^ swz(r0);
        uint32_t src;
        if constexpr (kDown) src = row;
        else src = prm.sorted_pairs[it.row_begin + row] / prm.K;
        ao[i] = src * (uint32_t)(Kd * 2) + 16u * chunk;
    }
    const void* abase = kDown ? (const void*)(prm.A + (long long)it.row_begin * Kd) : (const void*)prm.A;
    const __amdgpu_buffer_rsrc_t ra =
        __builtin_amdgcn_make_buffer_rsrc((void*)abase, (short)0, kDown ? it.rows * Kd * 2 : prm.a_bytes, kBufferWord3);
    using lds_bytes = __attribute__((address_space(3))) unsigned char*;
    auto sbuf = [&](auto bc) -> unsigned char* {
        if constexpr (decltype(bc)::value == 0) return sA0;
        else return sA1;
    };
    auto sbuf_lds = [&](auto bc) { return (lds_bytes)sbuf(bc); };
    auto copy_a = [&](__amdgpu_buffer_rsrc_t r, int g0, auto bc) {
#pragma unroll
        for (int p = 0; p < GS; ++p)
#pragma unroll
            for (int i = 0; i < NR; ++i) {
                const uint32_t o = ao[i];
                const int col = min(g0 + p, nG - 1) * kBK * 2, at = (p * kMidBM + RP * i + 8 * wave) * 128;
                __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)(sbuf_lds(bc) + at), 16, o, col,
                                                         0, 0);
            }
    };
    copy_a(ra, 0, std::integral_constant<int, 0>{});
    if constexpr (HAS_BIAS) {
        const int gu = (lane >> 4) & 1, col = 16 * fc + (lane & 15);
        const float* be = prm.bias + (long long)it.e * 2 * prm.F;
        if (lane < 32) s_bias[wave][lane] = prm.bias_interleaved ? be[2 * col + gu] : be[gu * prm.F + col];
    }
    const int nw = min(8, prm.NF - 8 * (fc >> 3));
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(prm.B + packed_frag(it.e, fc, 0, prm.NF, prm.KS) * kPkFrag), (short)0, (prm.KS - 1) * nw * 1024 + 1024, kBufferWord3);
    f32x16 acc[kMidMB];
#pragma unroll
    for (int mb = 0; mb < kMidMB; ++mb)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[mb][r] = 0.f;
    auto loop = [&](auto nc) {
        constexpr int NMB = decltype(nc)::value;
        mid_loop<OpT, NMB>(rw, lane * 16u, nw * 1024, ra, nG, lane, sbuf, copy_a, acc);
    };
    switch (nmb) {
        case 1: loop(std::integral_constant<int, 1>{}); break;
        case 2: loop(std::integral_constant<int, 2>{}); break;
        case 3: loop(std::integral_constant<int, 3>{}); break;
        case 4: loop(std::integral_constant<int, 4>{}); break;
        default: break;  // none (as the default, case 4 spills 58 registers)
    }
    // Down: rows of Y leave through LDS, 32 rows x 96 bytes of a wave's fragment at a time (in the first activation buffer), so
    // that consecutive lanes store consecutive bytes; straight from the accumulators a store is 64 pieces of 16 bytes, which
    // the L2 takes one by one. Down GEMM, without -> with (us): 513 experts of H 2048 F 512, 88 rows 294 -> 277; 8 of F 5632,
    // 1024 rows 223 -> 215, 550 rows 142 -> 136; 64 of H 1280 F 896, 469 rows 122 -> 112; 128 of F 768, 62 rows 94 -> 91.
    __shared__ int s_pair[kMidBM];
    __shared__ float s_w[kMidBM];
    if constexpr (kDown) {
        if (tid < it.rows) {
            const int p = prm.sorted_pairs[it.row_begin + tid];
            s_pair[tid] = p;
            s_w[tid] = static_cast<const float*>(prm.route_w)[p];
        }
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);  // the copies past the last stage land before the LDS is gone
    if constexpr (kDown) __syncthreads();
    if (!active) return;
    [[maybe_unused]] const float wsc = kDown ? __builtin_amdgcn_ldexpf(1.f, prm.wexp[(long long)it.e * prm.NF + fc]) : 1.f;
#pragma unroll
    for (int mb = 0; mb < kMidMB; ++mb) {
        if (mb >= nmb) break;
        const int row = 32 * mb + lrow;
        const bool valid = row < it.rows;
        const long long gr = it.row_begin + row;
        if constexpr (kDown) {
            static_assert(kMidWaves * 32 * kYRow <= kMidGroups * kMidBM * 128);
            unsigned char* st = sA0 + wave * 32 * kYRow;
            if (valid) pack_y(acc[mb], s_w[row] * wsc, reinterpret_cast<u32x4*>(st + lrow * kYRow + 48 * half));
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                const int c = 64 * i + lane, rr = 32 * mb + c / 6;
                const u32x4 v = *reinterpret_cast<const u32x4*>(st + 16 * c);
                if (rr < it.rows)
                    *reinterpret_cast<u32x4*>(prm.Y + ((long long)s_pair[rr] * prm.H + 32 * fc) * 3 + 16 * (c % 6)) = v;
            }
        } else {
            if (store_glu<MODE, ACT, HAS_BIAS>(prm, acc[mb], valid, gr, fc, half, s_bias[wave])) {
                if (half == 0) prm.rsig[gr] = 1;
                prm.sync[1] = 1;
            }
        }
    }
}

template <int MODE, int ACT, bool HAS_BIAS>
static void launch_mid_t(const StreamParams& q, int max_tiles, hipStream_t s) {
    const int nt = ceil_div(q.NF, kMidWaves);
    hipLaunchKernelGGL((moe_mid_kernel<MODE, ACT, HAS_BIAS>), dim3(8 * ceil_div(max_tiles * nt, 8)), dim3(kMidThreads), 0, s, q, nt);
}

int mid_tile_m() { return kMidBM; }

int stream_tile_m() { return kStRows; }

// Whether a call (that is not of the few form) takes the tiles form.
bool tiles_supported(int T, int K, int E) {
    return T <= kTilesMaxTokens && (long long)T * K <= (long long)kTilesMaxRows * E;
}

// Whether a call takes the few form: one 32-row block of tokens, experts that fit few_select's bitmap, lists that fit the
// down kernel's LDS. Above kFdMaxPairs pairs also a bound on the ids that the first projection reads: each of its workgroups
// (nf1 fragments of each chosen expert) goes through all of them, where the other forms sort them once. Against the tiles
// form, which takes most of these calls instead, the line is at 2^20 ids, against the grouped GEMMs at 600000. Whole op, few
// -> tiles (us): 22 tokens of 428 experts of H 192 F 1664, top-21 (20 M ids) 216 -> 147; 28 of 76 of H 576 F 3968, top-14
// (7.4 M) 257 -> 190; 32 of 128 of H 2048 F 768, top-8 (1.6 M) 177 -> 183; 32 of 32 of H = F = 2880, top-4 (0.74 M) 276 ->
// 282; few -> grouped: 30 tokens of 25 experts of H 1088 F 2112, top-16 (1.6 M) 109 -> 89; 32 of 14 of H 2816 F 1792, top-12
// (0.60 M) 119 -> 101; 20 of 12 of H 3648 F 3776, top-9 (0.51 M) 199 -> 200. Over 1150 shapes of up to 32 tokens the two
// lines are 0.4% off the better form on average, no line 2.5%. (So glu, one buffer in the down kernels, stays far below 2^31
// bytes there.)
bool few_supported(int T, int K, int E, int nf1) {
    const long long P = (long long)T * K;
    if (T > kFewMaxTokens || K > kFewMaxTopk || E > kFewMaxExperts || P > kFewMaxPairs) return false;
    return P <= kFdMaxPairs || nf1 * std::min<long long>(P, E) * P <= (tiles_supported(T, K, E) ? 1 << 20 : 600000);
}

// Whether the few form's down kernel sums over the slots itself, which saves the combine's launch. Its H / 16 workgroups walk
// all chosen experts one after the other, so with short rows of the result they stream less than the whole chip, for a time
// that goes with experts x F. Whole op, sum / rows and combine (us): 4 experts of H = F = 2880 35.8 / 37.3; 11 of H 2048 F
// 512 18.9 / 21.1; 6 of H 1280 F 896 15.7 / 17.0, 12 23.8 / 22.4; 14 of H 1280 F 640 20.8 / 23.0; 8 of H 896 F 1024 14.0 /
// 12.5; 8 of H 1472 F 2560 36.6 / 33.0; 2 of H 1664 F 3968 14.3 / 17.6. Over 500 shapes of up to 16 pairs this line is 0.2%
// off the better of both, the sum alone 3%, rows alone 10%. Above 16 pairs rows: 33 pairs of H 2048 F 768, the down kernel
// alone, 23.1 / 15.6 + 4.0.
bool few_sums(int T, int K, int E, int H, int F) {
    const long long P = (long long)T * K, um = std::min<long long>(P, E);
    return P <= kFdMaxPairs && (H >= 2048 || um <= 2 || um * F <= std::max(5000, 8 * H));
}

// Parts of the lists that the few form passes from its first to its second launch, at `lists`: um experts, um x T glu rows,
// um x nf1 flags, each to a multiple of 16 bytes.
static size_t few_part(size_t n) { return (n + 15) / 16 * 16; }

hipError_t launch_combine_h(const unsigned char* Y, const int32_t* idx, uint16_t* out, int T, int K, int E, int H,
                            const int32_t* sync, const int8_t* psig, const float* b2, const void* route_w,
                            hipStream_t s, int types);

template <bool FEW>
static void launch_stream_first(const StreamParams& q, int act, dim3 grid, hipStream_t s) {
#define CMOE_ST1(MODE, ACT, BIAS) hipLaunchKernelGGL((moe_stream_first_kernel<MODE, ACT, BIAS, FEW>), grid, dim3(kStThreads), 0, s, q)
    if (act == kActSilu) {
        if (q.bias) CMOE_ST1(kModePkGateUp, kActSilu, true);
        else CMOE_ST1(kModePkGateUp, kActSilu, false);
    } else if (act == kActGptOss) {
        if (q.bias) CMOE_ST1(kModePkGateUp, kActGptOss, true);
        else CMOE_ST1(kModePkGateUp, kActGptOss, false);
    } else if (act == kActGeluTanh) CMOE_ST1(kModePkUp, kActGeluTanh, false);
    else if (act == kActSiluPlain) CMOE_ST1(kModePkUp, kActSiluPlain, false);
    else CMOE_ST1(kModePkUp, kActRelu, false);
#undef CMOE_ST1
}

// gate_up -> down with the sum over slots, on stream s. Shapes were checked by the caller (few_supported).
hipError_t launch_few(const void* x, const void* w1p, const float* b1, const void* w2p, const float* b2, const int32_t* idx,
                      const void* route_w, int types, int T, int H, int F, int E, int K, int bias_interleaved, int act, void* out,
                      uint16_t* glu, int8_t* gexp, unsigned char* Y, unsigned char* lists, hipStream_t s, hipEvent_t* ev) {
    auto mark = [&](int i) { if (ev) (void)hipEventRecord(ev[i], s); };
    const int P = T * K, um = std::min(P, E);
    StreamParams q{};
    q.A = static_cast<const uint16_t*>(x);
    q.B = static_cast<const uint16_t*>(w1p);
    q.bias = b1;
    q.idx = idx;
    q.route_w = route_w;
    q.types = types;
    q.glu = glu;
    q.gexp = gexp;
    q.few_e = reinterpret_cast<int32_t*>(lists);
    q.few_row = reinterpret_cast<int16_t*>(lists + few_part((size_t)um * 4));
    q.few_scaled = reinterpret_cast<unsigned char*>(q.few_row) + few_part((size_t)um * T * 2);
    q.T = T; q.K = K; q.E = E; q.H = H; q.F = F;
    q.NF = q.nf1 = act_is_gated(act) ? F / 16 : F / 32;
    q.KS = H / 16;
    q.u_max = um;
    q.p_cap = P;
    q.a_bytes = T * H * 2;
    q.bias_interleaved = bias_interleaved;
    mark(0);
    mark(1);  // no route
    launch_stream_first<true>(q, act, dim3(q.NF, um), s);
    hipError_t st = hipGetLastError();
    if (st != hipSuccess) return st;
    mark(2);
    q.A = glu;
    q.a_bytes = P * F * 2;
    q.B = static_cast<const uint16_t*>(w2p);
    q.wexp = reinterpret_cast<const int8_t*>(static_cast<const uint16_t*>(w2p) + (long long)E * H * F);
    q.bias = b2;
    q.NF = H / 32;
    q.KS = F / 16;
    q.out = static_cast<uint16_t*>(out);
    while (2 << q.share_log <= kFdWaves && (F / kBK) >> (q.share_log + 1) >= kFdShare) ++q.share_log;
    if (!few_sums(T, K, E, H, F)) {
        q.Y = Y;
        hipLaunchKernelGGL(moe_few_down_rows_kernel, dim3(q.NF, um), dim3(kStThreads), 0, s, q);
        st = hipGetLastError();
        if (st != hipSuccess) return st;
        mark(3);
        st = launch_combine_h(Y, idx, static_cast<uint16_t*>(out), T, K, E, H, nullptr, nullptr, b2, route_w, s, types);
        mark(4);
        return st;
    }
    if (b2) hipLaunchKernelGGL((moe_few_down_kernel<true>), dim3(H / 16), dim3(kFdThreads), 0, s, q);
    else hipLaunchKernelGGL((moe_few_down_kernel<false>), dim3(H / 16), dim3(kFdThreads), 0, s, q);
    st = hipGetLastError();
    mark(3);
    mark(4);  // no combine
    return st;
}

// The two projections of the tiles form (mid: of moe_mid_kernel), between the route (M-tiles of stream_tile_m() or mid_tile_m()
// rows) and the fixup, and between the fixup and the combine. max_tiles bounds the M-tile list.
hipError_t launch_stream_gemm1(const void* x, const void* w1p, const float* b1, int T, int H, int F, int E, int K,
                               int bias_interleaved, int act, const int32_t* offsets, const int32_t* tile_offsets,
                               const int32_t* meta, const int32_t* sorted_pairs, const int32_t* tile_expert, int max_tiles, bool mid,
                               uint16_t* glu, int8_t* gexp, int8_t* rsig, int32_t* sync, hipStream_t s) {
    StreamParams q{};
    q.A = static_cast<const uint16_t*>(x);
    q.B = static_cast<const uint16_t*>(w1p);
    q.bias = b1;
    q.offsets = offsets; q.tile_offsets = tile_offsets; q.meta = meta; q.sorted_pairs = sorted_pairs; q.tile_expert = tile_expert;
    q.glu = glu;
    q.gexp = gexp;
    q.rsig = rsig;
    q.sync = sync;
    q.T = T; q.K = K; q.E = E; q.H = H; q.F = F;
    q.NF = act_is_gated(act) ? F / 16 : F / 32;
    q.KS = H / 16;
    q.p_cap = T * K;
    q.a_bytes = T * H * 2;
    q.bias_interleaved = bias_interleaved;
    if (mid) {
        if (act == kActSilu) {
            if (b1) launch_mid_t<kModePkGateUp, kActSilu, true>(q, max_tiles, s);
            else launch_mid_t<kModePkGateUp, kActSilu, false>(q, max_tiles, s);
        } else if (act == kActGptOss) {
            if (b1) launch_mid_t<kModePkGateUp, kActGptOss, true>(q, max_tiles, s);
            else launch_mid_t<kModePkGateUp, kActGptOss, false>(q, max_tiles, s);
        } else if (act == kActGeluTanh) launch_mid_t<kModePkUp, kActGeluTanh, false>(q, max_tiles, s);
        else if (act == kActSiluPlain) launch_mid_t<kModePkUp, kActSiluPlain, false>(q, max_tiles, s);
        else launch_mid_t<kModePkUp, kActRelu, false>(q, max_tiles, s);
        return hipGetLastError();
    }
    launch_stream_first<false>(q, act, dim3(q.NF, max_tiles), s);
    return hipGetLastError();
}

hipError_t launch_stream_gemm2(const uint16_t* glu, const void* w2p, const float* route_w, int T, int H, int F, int E, int K,
                               const int32_t* offsets, const int32_t* tile_offsets, const int32_t* meta,
                               const int32_t* sorted_pairs, const int32_t* tile_expert, int max_tiles, bool mid, unsigned char* Y,
                               hipStream_t s) {
    StreamParams q{};
    q.A = glu;
    q.B = static_cast<const uint16_t*>(w2p);
    q.wexp = reinterpret_cast<const int8_t*>(static_cast<const uint16_t*>(w2p) + (long long)E * H * F);
    q.route_w = route_w;
    q.offsets = offsets; q.tile_offsets = tile_offsets; q.meta = meta; q.sorted_pairs = sorted_pairs; q.tile_expert = tile_expert;
    q.Y = Y;
    q.T = T; q.K = K; q.E = E; q.H = H; q.F = F;
    q.NF = H / 32;
    q.KS = F / 16;
    q.p_cap = T * K;
    if (mid) {
        launch_mid_t<kModePkDown, kActSilu, false>(q, max_tiles, s);
        return hipGetLastError();
    }
    hipLaunchKernelGGL(moe_stream_down_kernel, dim3(q.NF, max_tiles), dim3(kStThreads), 0, s, q);
    return hipGetLastError();
}

}  // namespace cmoe
