// Fused MoE router: logits = x Wᵀ (+ b) rounded to bf16, then per-token expert selection, written
// straight in the form the experts op consumes (int32 ids, fp32 weights), plus the bf16 logits.
//
// Replaces the routers the reference runs inside its timed gpt-oss and qwen3 ops
// (src/kops/registry/gpt_oss_moe_experts.py:35, src/kops/registry/qwen3_next_moe_experts.py:28),
// i.e. transformers' GptOssTopKRouter (modeling_gpt_oss.py:126-130) and Qwen3NextTopKRouter
// (modeling_qwen3_next.py:766-775): bf16 F.linear, then
//   SOFTMAX_TOPK: probs = softmax_fp32(logits); top-k of probs; optional renormalisation; weights
//                 rounded to bf16 (the logits dtype);
//   TOPK_SOFTMAX: top-k of the logits; softmax over the k values, rounded to bf16.
// Ties (equal values, common with bf16 logits) go to the lower expert id; torch leaves their order
// unspecified. Output weights are the bf16 values widened to fp32, as the loaders' .float() casts.
//
// The logits GEMM ([T,H] x [E,H]ᵀ) runs on MFMA (bf16, fp32 accumulation).
//   E <= 64  (gpt-oss): one kernel. A workgroup owns 16 tokens and all experts; its waves split the
//            reduction, their partial sums meet in LDS (fixed order), and the same workgroup selects
//            for its 16 tokens. Many tokens with wide rows: 32 tokens on four waves and an LDS stage ring.
//   E > 64   (qwen3-next): up to 256 tokens the same split over workgroups of 16 tokens x 16 experts,
//            above that a 128-token x 64-expert tiled GEMM from LDS (stages of 64 k-columns copied
//            HBM -> LDS directly into a ring, one wait and one barrier per stage), writes the bf16
//            logits; then a selection kernel (one wave per token) reads them back.
// Selection: a lane holds experts lane, lane+64, ...; each expert becomes a 32-bit key (logit
// order, then lower id) and top-k is k rounds of a DPP wave maximum over the lanes' sorted heads.
#include <type_traits>

#include "moe_common.h"
#include "moe_tile.h"

namespace cmoe {

constexpr int kRtrThreads = 256;  // 4 waves
constexpr int kRtrMaxE = 1024;
constexpr int kRtrMaxK = 32;
constexpr int kRtrFusedMaxE = 64;
constexpr int kRtrSplitMaxT = 256;  // E > 64: tokens up to which the logits come from the split kernel (figures there)

constexpr int kRouterSoftmaxTopk = 0;
constexpr int kRouterTopkSoftmax = 1;

__device__ __forceinline__ float round_bf16(float f) { return bf16_bits_to_f32(f32_to_bf16_bits(f)); }

// ---- wave reductions over DPP: row_shr 1, 2, 4, 8 within rows of 16 lanes, then row_bcast 15 and
// 31 carry row results up; lane 63 ends with the reduction of all 64 lanes, read back as a uniform
// value. Lanes a DPP source does not reach contribute 0, the identity of both reductions below.
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ uint32_t dpp_or_zero(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROW_MASK, 0xf, false);
}

__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) {
    v = max(v, dpp_or_zero<0x111, 0xf>(v));
    v = max(v, dpp_or_zero<0x112, 0xf>(v));
    v = max(v, dpp_or_zero<0x114, 0xf>(v));
    v = max(v, dpp_or_zero<0x118, 0xf>(v));
    v = max(v, dpp_or_zero<0x142, 0xa>(v));
    v = max(v, dpp_or_zero<0x143, 0xc>(v));
    return __builtin_amdgcn_readlane(v, 63);
}

__device__ __forceinline__ float wave_sum_f32(float v) {
    v += __uint_as_float(dpp_or_zero<0x111, 0xf>(__float_as_uint(v)));
    v += __uint_as_float(dpp_or_zero<0x112, 0xf>(__float_as_uint(v)));
    v += __uint_as_float(dpp_or_zero<0x114, 0xf>(__float_as_uint(v)));
    v += __uint_as_float(dpp_or_zero<0x118, 0xf>(__float_as_uint(v)));
    v += __uint_as_float(dpp_or_zero<0x142, 0xa>(__float_as_uint(v)));
    v += __uint_as_float(dpp_or_zero<0x143, 0xc>(__float_as_uint(v)));
    return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), 63));
}

// Selection key: the bf16 logit mapped to an order-preserving 16-bit code (larger logit, larger
// code; -0 ranks as +0) in the high half, 0xffff - expert id in the low half, so that one unsigned
// max picks the largest logit and, among equal logits, the lowest id. Every real key is nonzero
// (the code of -inf is 0x007f); 0 marks "none".
__device__ __forceinline__ uint32_t order_key(float logit, int e) {
    uint32_t b = __float_as_uint(logit) >> 16;  // the logit is a bf16 value
    if (b == 0x8000u) b = 0u;
    const uint32_t o = (b & 0x8000u) ? (~b & 0xffffu) : (b | 0x8000u);
    return (o << 16) | (0xffffu - (uint32_t)e);
}
__device__ __forceinline__ float key_logit(uint32_t key) {
    const uint32_t o = key >> 16;
    return __uint_as_float(((o & 0x8000u) ? (o & 0x7fffu) : (~o & 0xffffu)) << 16);
}
__device__ __forceinline__ int key_expert(uint32_t key) { return (int)(0xffffu - (key & 0xffffu)); }

// Bitonic sort of N (a power of two) keys into descending order, in registers.
template <int N>
__device__ __forceinline__ void sort_desc(uint32_t (&a)[N]) {
#pragma unroll
    for (int k = 2; k <= N; k <<= 1)
#pragma unroll
        for (int j = k >> 1; j > 0; j >>= 1)
#pragma unroll
            for (int i = 0; i < N; ++i) {
                const int l = i ^ j;
                if (l > i) {
                    const uint32_t hi = max(a[i], a[l]), lo = min(a[i], a[l]);
                    const bool desc = (i & k) == 0;
                    a[i] = desc ? hi : lo;
                    a[l] = desc ? lo : hi;
                }
            }
}

// Selection for token t by one wave (all 64 lanes active). v[j] = bf16 logit of expert lane + 64 j.
// Output row t has K + S slots: the K chosen experts, then S shared-expert slots with ids E..E+S-1
// and weight bf16(sigmoid(gate_logit)) (the Qwen3-Next shared-expert gate, modeling_qwen3_next.py:794).
// The experts are chosen on the logits in both modes: softmax is strictly increasing, so the top-k
// of the probabilities is the top-k of the logits, and equal probabilities come only from equal
// logits. Each lane sorts its keys; round k takes the wave-wide maximum of the lanes' heads and the
// lane holding it pops its head. Lane k keeps the k-th key.
template <int MODE, int EJ>
__device__ __forceinline__ void select_token(const float (&v)[EJ], int lane, long long t, int E, int K, int renorm,
                                             int S, float gate_logit, int32_t* __restrict__ idx_out,
                                             float* __restrict__ w_out) {
    uint32_t key[EJ];
#pragma unroll
    for (int j = 0; j < EJ; ++j) key[j] = lane + kWave * j < E ? order_key(v[j], lane + kWave * j) : 0u;
    sort_desc<EJ>(key);
    uint32_t sel = 0u, top = 0u;
    for (int k = 0; k < K; ++k) {
        const uint32_t best = wave_max_u32(key[0]);
        if (k == 0) top = best;
        if (lane == k) sel = best;
        const bool pop = key[0] == best;
#pragma unroll
        for (int j = 0; j + 1 < EJ; ++j) key[j] = pop ? key[j + 1] : key[j];
        key[EJ - 1] = pop ? 0u : key[EJ - 1];
    }
    const float lmax = key_logit(top), lsel = key_logit(sel);
    float wt;
    if constexpr (MODE == kRouterSoftmaxTopk) {
        // p = exp(l - max) / sum over all experts of exp(l_j - max), the fp32 softmax
        float s = 0.f;
#pragma unroll
        for (int j = 0; j < EJ; ++j) s += lane + kWave * j < E ? __expf(v[j] - lmax) : 0.f;
        s = wave_sum_f32(s);
        const float p = lane < K ? __expf(lsel - lmax) / s : 0.f;
        wt = renorm ? p / wave_sum_f32(p) : p;
    } else {
        // softmax over the k selected logits; lmax is their maximum
        const float ex = lane < K ? __expf(lsel - lmax) : 0.f;
        wt = ex / wave_sum_f32(ex);
    }
    const int KO = K + S;
    if (lane < K) {
        idx_out[t * KO + lane] = key_expert(sel);
        w_out[t * KO + lane] = round_bf16(wt);
    } else if (lane < KO) {
        idx_out[t * KO + lane] = E + lane - K;
        w_out[t * KO + lane] = round_bf16(1.f / (1.f + __expf(-gate_logit)));
    }
}

// Stage ring of NW waves: a stage holds 64 k-columns of ROWS rows = tokens t0.. (rows [0, TM)) then experts
// e0.. (rows [TM, ROWS)), as 128-byte rows in the swizzled layout of lds_off. The copies go straight
// from HBM to LDS (global_load_lds_dwordx4): instruction i of a stage fills rows 8i..8i+7, lane l
// taking row 8i + l/8 and the chunk that the swizzle puts at position l % 8. Wave w issues
// instructions w, w+NW, ... (kPerWave each), from row pointers it computed once (recomputing them per stage cost more than
// the stage's MFMAs). Rows beyond T or E are clamped (their results are never stored); columns beyond H are clamped to
// H - 8 (their k-steps are skipped), so every address is inside x or W.
template <int ROWS, int TM, int NW>
struct StageRing {
    static constexpr int kStageBytes = ROWS * kBK * 2;
    static constexpr int kPerWave = ROWS / 8 / NW;
    static_assert(ROWS % (8 * NW) == 0, "the waves issue whole 8-row instructions");
    const uint16_t* src[kPerWave];
    int kmax[kPerWave];  // H - 8 from src's chunk

    __device__ __forceinline__ StageRing(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w, int t0, int e0, int T,
                                         int E, int H, int wave, int lane) {
#pragma unroll
        for (int j = 0; j < kPerWave; ++j) {
            const int row = 8 * (wave + NW * j) + (lane >> 3);
            const int chunk = (lane & 7) ^ swz(row);
            src[j] = (row < TM ? x + (long long)min(t0 + row, T - 1) * H : w + (long long)min(e0 + row - TM, E - 1) * H) + 8 * chunk;
            kmax[j] = H - 8 - 8 * chunk;
        }
    }
    __device__ __forceinline__ void issue(int st, uint32_t slot, int wave) const {
#pragma unroll
        for (int j = 0; j < kPerWave; ++j) dma16(src[j] + min(st * kBK, kmax[j]), slot + 1024u * (wave + NW * j));
    }
};

// Fragment of rows row0..row0+31 for k-step q of a stage: lane l reads row l % 32, 8 bf16 at
// k = 16 q + 8 (l / 32).
__device__ __forceinline__ bf16x8 lds_frag(const char* __restrict__ stage, int row0, int q, int lane) {
    return __builtin_bit_cast(bf16x8,
                              *reinterpret_cast<const u32x4*>(stage + lds_off(row0 + (lane & 31), 2 * q + (lane >> 5))));
}

// Stage pipeline: S-1 stages in flight; per stage one wait on this wave's own
// copies, one barrier that publishes the stage (and frees the slot read one stage earlier), then the
// copy of stage st + S - 1 into that slot, then compute(stage pointer, st).
template <int S, int ROWS, int TM, int NW, typename Compute>
__device__ __forceinline__ void stage_pipeline(char* ring, const uint16_t* __restrict__ x,
                                               const uint16_t* __restrict__ w, int t0, int e0, int T, int E, int H,
                                               int wave, int lane, Compute&& compute) {
    using R = StageRing<ROWS, TM, NW>;
    const R r(x, w, t0, e0, T, E, H, wave, lane);
    const int nst = ceil_div(H, kBK);
    const uint32_t base = lds_u32(ring);
#pragma unroll
    for (int s = 0; s < S - 1; ++s)
        if (s < nst) r.issue(s, base + s * R::kStageBytes, wave);
    int cur = 0, nxt = S - 1;  // ring slots of stages st and st + S - 1
    for (int st = 0; st < nst; ++st) {
        if (st + S - 2 < nst) wait_vmcnt<(S - 2) * R::kPerWave>();  // stages st+1 .. st+S-2 may stay in flight
        else wait_vmcnt<0>();
        __syncthreads();
        if (st + S - 1 < nst) r.issue(st + S - 1, base + nxt * R::kStageBytes, wave);
        compute(ring + cur * R::kStageBytes, st);
        cur = cur + 1 == S ? 0 : cur + 1;
        nxt = nxt + 1 == S ? 0 : nxt + 1;
    }
    __syncthreads();
}

// ---- logits of 16 tokens x 16 NE experts by one workgroup, its W waves splitting the reduction: 16x16x32 MFMA on
// fragments loaded straight to registers (a load covers 64 bytes of each of 16 rows), every load of a wave in flight at
// once, one barrier where the partial sums meet in LDS. Rows beyond T or ER are clamped (their results are dropped).
template <int NE, int W>
struct SplitLogits {
    static constexpr int kTokens = 16, kExperts = 16 * NE;
    float part[W][kTokens][kExperts + 4];  // + 4: rows 16 bytes off the bank period

    template <int C>
    __device__ __forceinline__ static void steps(const uint16_t* __restrict__ xr, const uint16_t* const (&wr)[NE], int k0,
                                                 int k1, f32x4 (&acc)[NE]) {
        for (int ks = k0; ks < k1; ks += C) {
            u32x4 a[C], b[C][NE];
#pragma unroll
            for (int c = 0; c < C; ++c) {
                const int k = 32 * min(ks + c, k1 - 1);
                a[c] = *reinterpret_cast<const u32x4*>(xr + k);
#pragma unroll
                for (int n = 0; n < NE; ++n) b[c][n] = *reinterpret_cast<const u32x4*>(wr[n] + k);
            }
#pragma unroll
            for (int c = 0; c < C; ++c) {
                if (ks + c >= k1) break;  // uniform
#pragma unroll
                for (int n = 0; n < NE; ++n)
                    acc[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, b[c][n]),
                                                                     __builtin_bit_cast(bf16x8, a[c]), acc[n], 0, 0, 0);
            }
        }
    }
    // part[wave] of this wave; the caller synchronises before sum()
    __device__ __forceinline__ void run(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w, int t0, int e0, int T,
                                        int ER, int H, int wave, int lane) {
        const int l16 = lane & 15, g = lane >> 4;
        const uint16_t* xr = x + (long long)min(t0 + l16, T - 1) * H + 8 * g;
        const uint16_t* wr[NE];
#pragma unroll
        for (int n = 0; n < NE; ++n) wr[n] = w + (long long)min(e0 + 16 * n + l16, ER - 1) * H + 8 * g;
        f32x4 acc[NE];
#pragma unroll
        for (int n = 0; n < NE; ++n) acc[n] = f32x4{0.f, 0.f, 0.f, 0.f};
        const int nks = H / 32, k0 = wave * nks / W, k1 = (wave + 1) * nks / W;
        if (k1 - k0 <= 4) steps<4>(xr, wr, k0, k1, acc);
        else steps<(NE > 2 ? 4 : 6)>(xr, wr, k0, k1, acc);
        if ((H & 31) && wave == W - 1) {  // the last 16 columns: the upper half of the k-step is zero
            const int k = 32 * nks - (g >= 2 ? 16 : 0);
            const u32x4 z = {0u, 0u, 0u, 0u};
            const u32x4 a = *reinterpret_cast<const u32x4*>(xr + k);
#pragma unroll
            for (int n = 0; n < NE; ++n) {
                const u32x4 b = *reinterpret_cast<const u32x4*>(wr[n] + k);
                acc[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, g >= 2 ? z : b),
                                                                 __builtin_bit_cast(bf16x8, g >= 2 ? z : a), acc[n], 0, 0, 0);
            }
        }
        // element r: expert 4 g + r of its block, token lane % 16
#pragma unroll
        for (int n = 0; n < NE; ++n) *reinterpret_cast<f32x4*>(&part[wave][l16][16 * n + 4 * g]) = acc[n];
    }
    __device__ __forceinline__ float sum(int tl, int el) const {
        float s = part[0][tl][el];
#pragma unroll
        for (int k = 1; k < W; ++k) s += part[k][tl][el];
        return s;
    }
};

// ---- E <= 64: logits + selection in one kernel; grid = ceil(T / 16). What bounds it is latency (a wave reads its whole
// share at once): 256 workgroups at T = 4096. Against 32 tokens per workgroup with four waves and an LDS stage ring (128
// workgroups, one barrier per 64 columns), us per launch: H = 2880 E = 32 T=1 12.0 -> 7.9, T=4096 18.0 -> 12.1; H = 2048
// E = 8 T=4096 14.1 -> 7.5; H = 2048 E = 64 T=2048 20.3 -> 13.8.
template <int MODE, int NE>
__global__ __launch_bounds__(NE <= 2 ? 1024 : 512) void moe_router_fused_kernel(
    const uint16_t* __restrict__ x, const uint16_t* __restrict__ w, const uint16_t* __restrict__ bias, int T, int H,
    int E, int K, int renorm, int S, int32_t* __restrict__ idx_out, float* __restrict__ w_out,
    uint16_t* __restrict__ logits_out) {
    constexpr int W = NE <= 2 ? 16 : 8, EN = 16 * NE;
    const int ER = E + (S > 0);  // rows of W and of a logits row: the experts, then the shared-expert gate
    __shared__ __align__(16) SplitLogits<NE, W> sl;
    __shared__ float s_logit[16][EN];
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int t0 = blockIdx.x * 16;
    sl.run(x, w, t0, 0, T, ER, H, wave, lane);
    __syncthreads();
    // logit = bf16(sum of the partial sums in wave order + b)
    for (int c = tid; c < 16 * EN; c += W * kWave) {
        const int tl = c / EN, e = c % EN;
        if (e >= ER) continue;
        const float b = bias != nullptr ? bf16_bits_to_f32(bias[e]) : 0.f;
        const float v = round_bf16(sl.sum(tl, e) + b);
        s_logit[tl][e] = v;
        if (t0 + tl < T) logits_out[(long long)(t0 + tl) * ER + e] = f32_to_bf16_bits(v);
    }
    __syncthreads();
    for (int tl = wave; tl < 16; tl += W) {
        if (t0 + tl >= T) break;  // uniform
        float v[1] = {lane < E ? s_logit[tl][min(lane, EN - 1)] : -INFINITY};
        select_token<MODE, 1>(v, lane, t0 + tl, E, K, renorm, S, S > 0 ? s_logit[tl][E] : 0.f, idx_out, w_out);
    }
}

// ---- E <= 64, many tokens: the same on 32 tokens per workgroup, four waves and an LDS stage ring (each stage's four k-steps one
// per wave), which reads W half as often and holds two workgroups per CU (one above 32 rows of W); grid = ceil(T / 32).
// A 16-token workgroup of 16 waves has a CU to itself, so the split kernel goes up in steps of 4096 tokens. us per launch, split
// -> ring: H = 2880 E = 32 T = 4096 13.5 -> 17.7, 5120 22.7 -> 17.7, 16384 43.0 -> 26.4; H = 4096 E = 64 T = 5120 43.6 -> 29.5; H =
// 2048 E = 64 T = 8192 24.5 -> 20.0, 10240 34.0 -> 37.3, 16384 45.0 -> 38.7; H = 1024 E = 32 T = 8192 9.1 -> 11.7, 16384 17.4 -> 14.7; E =
// 64 24.7 -> 27.9; H = 2880 E = 16 T = 8208 23.1 -> 18.0; H = 4096 E = 8 T = 32768 69.3 -> 73.1.
static bool ring_pays(int T, int H, int ER) {
    if (T <= 4096 || ER <= 8) return false;
    if (T <= 8192) return ER > 16 && H >= 2048;
    return H >= (ER > 32 ? 1536 : ER > 16 ? 1024 : 2048);
}

constexpr int kRtrRingStages = 8;
template <int MODE, int NT>  // NT = expert blocks of 32 (1 or 2)
__global__ __launch_bounds__(kRtrThreads) void moe_router_ring_kernel(
    const uint16_t* __restrict__ x, const uint16_t* __restrict__ w, const uint16_t* __restrict__ bias, int T, int H,
    int E, int K, int renorm, int S, int32_t* __restrict__ idx_out, float* __restrict__ w_out,
    uint16_t* __restrict__ logits_out) {
    constexpr int TM = 32, EN = 32 * NT, ROWS = TM + EN;
    const int ER = E + (S > 0);  // rows of W and of a logits row: the experts, then the shared-expert gate
    constexpr int kRing = kRtrRingStages * ROWS * kBK * 2;
    static_assert(4 * TM * EN * 4 <= kRing, "partial sums reuse the stage ring");
    __shared__ __align__(1024) char ring[kRing];
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int t0 = blockIdx.x * TM;

    f32x16 acc[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[n][r] = 0.f;
    // wave q takes k-step q of every stage; a k-step at or beyond H is skipped
    stage_pipeline<kRtrRingStages, ROWS, TM, 4>(ring, x, w, t0, 0, T, ER, H, wave, lane, [&](const char* sb, int st) {
        if (st * kBK + 16 * wave < H) {
            const bf16x8 a = lds_frag(sb, 0, wave, lane);
#pragma unroll
            for (int n = 0; n < NT; ++n)
                acc[n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, lds_frag(sb, TM + 32 * n, wave, lane), acc[n], 0, 0, 0);
        }
    });
    // partial sums of the four waves: element r is token 8(r/4) + 4(lane/32) + r%4, expert 32 n + lane % 32
    float(*part)[TM][EN] = reinterpret_cast<float(*)[TM][EN]>(ring);
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int r = 0; r < 16; ++r) part[wave][8 * (r >> 2) + 4 * (lane >> 5) + (r & 3)][32 * n + (lane & 31)] = acc[n][r];
    __syncthreads();
    // logit = bf16(((p0 + p1) + p2) + p3 + b); kept in slice 0 and written to logits_out
    for (int c = tid; c < TM * EN; c += kRtrThreads) {
        const int tl = c / EN, e = c % EN;
        if (e >= ER) continue;
        const float b = bias != nullptr ? bf16_bits_to_f32(bias[e]) : 0.f;
        const float v = round_bf16(((part[0][tl][e] + part[1][tl][e]) + part[2][tl][e]) + part[3][tl][e] + b);
        part[0][tl][e] = v;
        if (t0 + tl < T) logits_out[(long long)(t0 + tl) * ER + e] = f32_to_bf16_bits(v);
    }
    __syncthreads();
    for (int tl = wave; tl < TM; tl += 4) {
        if (t0 + tl >= T) break;  // uniform
        float v[1] = {lane < E ? part[0][tl][min(lane, EN - 1)] : -INFINITY};
        select_token<MODE, 1>(v, lane, t0 + tl, E, K, renorm, S, S > 0 ? part[0][tl][E] : 0.f, idx_out, w_out);
    }
}

// ---- E > 64, few tokens: logits of 16 tokens x 16 experts per workgroup, the shared-expert gate's row among them;
// grid = (ceil(ER / 16), ceil(T / 16)). Up to kRtrSplitMaxT tokens: H=2048 E=512 T=1 4.6 us against 19.3 of the tiled
// kernel (whose few workgroups walk 32 stages one after the other), T=256 12.7 / 15.6, T=512 20.2 / 15.6.
__global__ __launch_bounds__(1024) void moe_router_split_logits_kernel(const uint16_t* __restrict__ x,
                                                                       const uint16_t* __restrict__ w,
                                                                       const uint16_t* __restrict__ bias, int T, int H,
                                                                       int ER, uint16_t* __restrict__ logits_out) {
    __shared__ __align__(16) SplitLogits<1, 16> sl;
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int e0 = blockIdx.x * 16, t0 = blockIdx.y * 16;
    sl.run(x, w, t0, e0, T, ER, H, wave, lane);
    __syncthreads();
    const int tl = tid >> 4, e = e0 + (tid & 15);
    if (tid >= 256 || t0 + tl >= T || e >= ER) return;
    const float b = bias != nullptr ? bf16_bits_to_f32(bias[e]) : 0.f;
    logits_out[(long long)(t0 + tl) * ER + e] = f32_to_bf16_bits(sl.sum(tl, tid & 15) + b);
}

// ---- E > 64: tiled logits GEMM, 128 tokens x 64 experts per workgroup; grid = (ceil(T/128), ceil(E/64));
// logits rows are ldl apart (E + 1 with a shared-expert gate, whose logit the selection kernel adds). Eight waves, two
// per SIMD, one 32x32 block each: with four waves (two blocks each) the stage's LDS reads, copies and barrier were exposed
// on every SIMD. T=4096 H=2048 E=512: 22.1 -> 18.9 us with both; ring depths of 3 and 6 measured the same.
constexpr int kRtrTiledStages = 4;
constexpr int kRtrTiledWaves = 8;
__global__ __launch_bounds__(kRtrTiledWaves* kWave) void moe_router_logits_kernel(const uint16_t* __restrict__ x,
                                                                                  const uint16_t* __restrict__ w,
                                                                                  const uint16_t* __restrict__ bias, int T,
                                                                                  int H, int E, int ldl,
                                                                                  uint16_t* __restrict__ logits_out) {
    constexpr int TM = 128, EN = 64, ROWS = TM + EN;
    __shared__ __align__(1024) char ring[kRtrTiledStages * ROWS * kBK * 2];
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int t0 = blockIdx.x * TM, e0 = blockIdx.y * EN;
    const int wt = 32 * (wave >> 1), we = 32 * (wave & 1);  // this wave's token rows and expert rows

    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
    stage_pipeline<kRtrTiledStages, ROWS, TM, kRtrTiledWaves>(
        ring, x, w, t0, e0, T, E, H, wave, lane, [&](const char* sb, int st) {
            if (st * kBK + kBK <= H) {
                bf16x8 a[4], b[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    a[q] = lds_frag(sb, wt, q, lane);
                    b[q] = lds_frag(sb, TM + we, q, lane);
                }
#pragma unroll
                for (int q = 0; q < 4; ++q) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[q], b[q], acc, 0, 0, 0);
            } else {
                for (int q = 0; st * kBK + 16 * q < H; ++q)  // last stage of an H that is not a multiple of 64
                    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(lds_frag(sb, wt, q, lane), lds_frag(sb, TM + we, q, lane), acc,
                                                                  0, 0, 0);
            }
        });
    const int e = e0 + we + (lane & 31);
    if (e >= E) return;
    const float b = bias != nullptr ? bf16_bits_to_f32(bias[e]) : 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int t = t0 + wt + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
        if (t < T) logits_out[(long long)t * ldl + e] = f32_to_bf16_bits(acc[r] + b);
    }
}

// ---- E > 64: selection from the bf16 logits, one wave per token; grid = ceil(T / 4)
// With S > 0 and not gate_done the wave also computes the shared-expert gate logit, bf16(x_t . w_E (+ b_E)), as a dot
// product over H (16 bf16 per lane per step, fp32, DPP sum) and stores it in logits column E.
template <int MODE, int EJ>  // EJ = experts per lane = ceil(E / 64)
__global__ __launch_bounds__(kRtrThreads) void moe_router_select_kernel(
    uint16_t* __restrict__ logits, const uint16_t* __restrict__ x, const uint16_t* __restrict__ w,
    const uint16_t* __restrict__ bias, int T, int H, int E, int K, int renorm, int S, int gate_done,
    int32_t* __restrict__ idx_out, float* __restrict__ w_out) {
    const int lane = threadIdx.x & (kWave - 1);
    const int t = blockIdx.x * 4 + (int)(threadIdx.x / kWave);
    if (t >= T) return;  // uniform per wave
    uint16_t* row = logits + (long long)t * (E + (S > 0));
    float gate = 0.f;
    if (S > 0 && gate_done) {
        gate = bf16_bits_to_f32(row[E]);
    } else if (S > 0) {
        const uint16_t* xr = x + (long long)t * H;
        const uint16_t* gr = w + (long long)E * H;
        float acc = 0.f;
        for (int h = 8 * lane; h < H; h += 8 * kWave) {  // H % 16 == 0: whole 8-element chunks
            const u32x4 xa = *reinterpret_cast<const u32x4*>(xr + h);
            const u32x4 ga = *reinterpret_cast<const u32x4*>(gr + h);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                acc = fmaf(__uint_as_float(xa[q] << 16), __uint_as_float(ga[q] << 16), acc);
                acc = fmaf(__uint_as_float(xa[q] & 0xffff0000u), __uint_as_float(ga[q] & 0xffff0000u), acc);
            }
        }
        gate = round_bf16(wave_sum_f32(acc) + (bias != nullptr ? bf16_bits_to_f32(bias[E]) : 0.f));
        if (lane == 0) row[E] = f32_to_bf16_bits(gate);
    }
    float v[EJ];
#pragma unroll
    for (int j = 0; j < EJ; ++j) {
        const int e = lane + kWave * j;
        v[j] = e < E ? bf16_bits_to_f32(row[e]) : -INFINITY;
    }
    select_token<MODE, EJ>(v, lane, t, E, K, renorm, S, gate, idx_out, w_out);
}

int router_max_experts() { return kRtrMaxE; }
int router_max_topk() { return kRtrMaxK; }

template <int MODE>
static hipError_t launch_router_m(const uint16_t* x, const uint16_t* w, const uint16_t* bias, int T, int H, int E,
                                  int K, int renorm, int S, int32_t* idx, float* wt, uint16_t* logits, hipStream_t s) {
    const int ER = E + (S > 0);
    if (ER <= kRtrFusedMaxE && ring_pays(T, H, ER)) {
        const dim3 grid(ceil_div(T, 32)), block(kRtrThreads);
        if (ER <= 32)
            hipLaunchKernelGGL((moe_router_ring_kernel<MODE, 1>), grid, block, 0, s, x, w, bias, T, H, E, K, renorm, S, idx, wt, logits);
        else
            hipLaunchKernelGGL((moe_router_ring_kernel<MODE, 2>), grid, block, 0, s, x, w, bias, T, H, E, K, renorm, S, idx, wt, logits);
        return hipGetLastError();
    }
    if (ER <= kRtrFusedMaxE) {
        const dim3 grid(ceil_div(T, 16));
#define CMOE_RTF(NE) \
    hipLaunchKernelGGL((moe_router_fused_kernel<MODE, NE>), grid, dim3(NE <= 2 ? 1024 : 512), 0, s, x, w, bias, T, H, E, \
                       K, renorm, S, idx, wt, logits)
        if (ER <= 16) CMOE_RTF(1);
        else if (ER <= 32) CMOE_RTF(2);
        else CMOE_RTF(4);
#undef CMOE_RTF
        return hipGetLastError();
    }
    const int few = T <= kRtrSplitMaxT;
    if (few)
        hipLaunchKernelGGL(moe_router_split_logits_kernel, dim3(ceil_div(ER, 16), ceil_div(T, 16)), dim3(1024), 0, s, x, w,
                           bias, T, H, ER, logits);
    else
        hipLaunchKernelGGL(moe_router_logits_kernel, dim3(ceil_div(T, 128), ceil_div(E, 64)), dim3(kRtrTiledWaves * kWave), 0, s,
                           x, w, bias, T, H, E, ER, logits);
    const dim3 grid(ceil_div(T, 4));
    const int ej = ceil_div(E, kWave);
#define CMOE_RTR(EJ) \
    hipLaunchKernelGGL((moe_router_select_kernel<MODE, EJ>), grid, dim3(kRtrThreads), 0, s, logits, x, w, bias, T, H, \
                       E, K, renorm, S, few, idx, wt)
    if (ej <= 2) CMOE_RTR(2);
    else if (ej <= 4) CMOE_RTR(4);
    else if (ej <= 8) CMOE_RTR(8);
    else CMOE_RTR(16);
#undef CMOE_RTR
    return hipGetLastError();
}

// Shapes were checked by the caller: 1 <= K <= min(E, 32), 0 <= S <= 32, E + (S > 0) <= 1024,
// H % 16 == 0, T >= 1; W and bias have E + (S > 0) rows, logits is [T, E + (S > 0)] bf16, ids and
// weights are [T, K + S].
hipError_t launch_router(const uint16_t* x, const uint16_t* w, const uint16_t* bias, int T, int H, int E, int K,
                         int mode, int renorm, int S, int32_t* idx, float* wt, uint16_t* logits, hipStream_t s) {
    if (mode == kRouterSoftmaxTopk)
        return launch_router_m<kRouterSoftmaxTopk>(x, w, bias, T, H, E, K, renorm, S, idx, wt, logits, s);
    return launch_router_m<kRouterTopkSoftmax>(x, w, bias, T, H, E, K, renorm, S, idx, wt, logits, s);
}

}  // namespace cmoe
