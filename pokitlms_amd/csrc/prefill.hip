// prefill.hip -- batched routed-MoE prefill on gfx950 (MFMA grouped GEMM).
//
// The reference prefills a prompt one token at a time through the MoE block
// of src/qwen3_moe_runner.cpp:643-692 (the loop at :785-790), so every
// token's routes and output are those of a single-token pass.  Here the
// whole batch goes through six launches:
//
//  1. k_router_batch: the logit value S (the decode router's) and a rounding
//     bound B of every (token, expert) pair.
//  2. k_route_batch: one workgroup per token ranks the experts exactly as the
//     decode path does (certified wave ranking, exact serial fallback) and
//     writes ids and route weights.
//  3. k_group: one workgroup counts each expert's tokens and lays out
//     per-expert row ranges, a list of 64-row tiles and the assignments
//     (token * top_k + route) grouped by expert; its other workgroups split
//     x into the gate/up GEMM's operands meanwhile.
//  4. gate/up GEMM (expert_gemm.hip): per tile and 128 ffn rows, gate and up on
//     fp16 MFMA with the SwiGLU epilogue, which writes the activations already
//     split for the down GEMM.
//  5. down GEMM: per tile and 256 hidden rows; each output row goes to its
//     (token, route) slot.
//  6. k_combine: y = ((0 + p0*o0) + p1*o1) + ... per token in route order
//     (:688-690).
//
// Launch sizes depend only on the token count; tiles past the actual count
// exit at once, so the host never waits for the grouping.
#include <math.h>

#include "gemm_split.hpp"
#include "kquant.hpp"
#include "launch.hpp"
#include "route.hpp"

namespace pk {
namespace {

// ---------------------------------------------------------------------------
// 1. Batched router: per (token, expert) the value S of the decode router (the
// FP64 sum of the CPU's rounded FP32 products) and a bound B on the CPU's serial
// FP32 sum.
//
// A workgroup takes 16 tokens x 32 rows; its eight waves split K, and each lane of
// a wave sums 2 tokens x 4 rows over the wave's range, so a
// product costs its multiplication, the conversion and one FP64 add, and no
// scan across lanes is left (one row per wave with a scan and two FP64 adds per
// product: 275 us for 4096 tokens x 128 rows of 2048, 42 us for 512; so: 116
// and 21 us, bound by those three instructions; the ranking's second look at what
// the coarser bound leaves open adds 6 us).  The waves' operands pass
// through LDS parts of their own, ordered within the wave (wave_lds_order); the only
// barrier is before the waves' sums meet.
//
// The bound.  With T_i the exact prefix sums of the products p_i, the serial sum
// is within u (1 + 2^-10) sum_i |T_i| of S.  In a run of 16 products from prefix O
// to prefix O', |T_i| <= |O| + the |p| before i in the first half and |O'| + the
// |p| after i in the second, so the run's sum is at most 8 |O| + 8 |O'| + sum_j
// o_j |p_j| with o = 8 .. 1, 0 .. 7; and by Cauchy-Schwarz over the whole row
// sum_j o_j |p_j| <= |o w| |x|, two norms.  A wave's range starts at an offset that
// the earlier waves' sums give: |O| <= |offset| + |its own prefix|.  On
// router-like rows of 2048 this is 1.4 times the decode router's bound.

constexpr uint32_t kRtWaves = 8;                        // waves per workgroup, each a range of K
constexpr uint32_t kRtK = 32, kRtRow = kRtK + 4;        // K per stage; floats per staged row
struct RouterSums {
    double l, q;  // a wave's sum, and the sum of its |prefixes| at every 16th product
};

// Lane (i, j) of a wave takes tokens TT i .. and rows TE j ..: 8 TT tokens x 8 TE
// rows per workgroup.  2 x 4 where that makes two workgroups per CU, else 1 x 2
// (a wave's chain is a quarter as long: 512 tokens 33 -> 21 us, 77 tokens x 64
// rows of 1024 17 -> 6 us).  The first form spills seven registers of addresses, which
// a stage of 768 vector instructions reads back once; 32-bit offsets spill as many.
template <uint32_t TT, uint32_t TE>
__global__ __launch_bounds__(64 * kRtWaves, 4) void k_router_batch(MoePrefillArgs a) {
    constexpr uint32_t T = 8u * TT, R = 8u * TE, NL = TT + TE;
    __shared__ __attribute__((aligned(16))) union {
        float stage[kRtWaves][(T + R) * kRtRow];
        RouterSums part[kRtWaves][T * R];
    } sh;
    __shared__ float nx[kRtWaves][T], nw[kRtWaves][R];  // squared norms of each wave's range
    const uint32_t E = a.layer.n_experts, ER = E + a.layer.variant, H = a.layer.hidden;
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint32_t e0 = blockIdx.x * R, t0 = blockIdx.y * T;
    const uint32_t range = H / kRtWaves;  // a multiple of kRtK
    // staging: piece lane % 8 (4 floats) of rows lane / 8 + 8 i; rows past the end
    // repeat the last and write nothing
    const uint32_t pr = lane / 8u, pc = 4u * (lane % 8u);
    const float* src[NL];
#pragma unroll
    for (uint32_t i = 0; i < NL; ++i) {
        if (i < TT) {
            const uint32_t t = t0 + pr + 8u * i < a.tokens ? t0 + pr + 8u * i : a.tokens - 1u;
            src[i] = a.x + static_cast<uint64_t>(t) * H;
        } else {
            const uint32_t e = e0 + pr + 8u * (i - TT) < ER ? e0 + pr + 8u * (i - TT) : ER - 1u;
            src[i] = e < E ? a.layer.router + static_cast<uint64_t>(e) * H : a.layer.shared_router;
        }
        src[i] += wave * range + pc;
    }
    // o_j of this lane's four positions in a run of 16, plus 1 (and a little) for the
    // rounding of the products themselves
    float om[4];
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) {
        const uint32_t j = pc % 16u + i;
        om[i] = (j < 8u ? 8.0f - static_cast<float>(j) : static_cast<float>(j) - 8.0f) + 1.001f;
    }
    // stages of loads in flight: two, or one where registers would limit the waves
    constexpr uint32_t NS = TT == 1u ? 2u : 1u;
    rf32x4 v[NS][NL];
    auto load = [&](uint32_t set, uint32_t k) {
        const uint32_t kk = k < range ? k : range - kRtK;  // past the range: its last stage again
#pragma unroll
        for (uint32_t i = 0; i < NL; ++i) v[set][i] = *reinterpret_cast<const rf32x4*>(src[i] + kk);
    };
    float* st = sh.stage[wave];
    float sq[NL];
#pragma unroll
    for (uint32_t i = 0; i < NL; ++i) sq[i] = 0.0f;
    const uint32_t ti = TT * (lane / 8u), ej = TE * (lane % 8u);  // this lane's tokens and rows
    const float* xr = st + ti * kRtRow;
    const float* wr = st + (T + ej) * kRtRow;
    double l[TT][TE], q[TT][TE];
#pragma unroll
    for (uint32_t t = 0; t < TT; ++t)
#pragma unroll
        for (uint32_t e = 0; e < TE; ++e) l[t][e] = q[t][e] = 0.0;
#pragma unroll
    for (uint32_t i = 0; i < NS; ++i) load(i, i * kRtK);
    auto stage = [&](uint32_t set, uint32_t k) {
#pragma unroll
        for (uint32_t i = 0; i < NL; ++i) {
            *reinterpret_cast<rf32x4*>(st + (pr + 8u * i) * kRtRow + pc) = v[set][i];
#pragma unroll
            for (uint32_t c = 0; c < 4; ++c) {
                const float f = i < TT ? v[set][i][c] : v[set][i][c] * om[c];
                sq[i] = __builtin_fmaf(f, f, sq[i]);
            }
        }
        load(set, k + NS * kRtK);
        wave_lds_order();  // the lanes read each other's stores
#pragma unroll
        for (uint32_t c = 0; c < kRtK / 4u; ++c) {
            rf32x4 x[TT], w[TE];
#pragma unroll
            for (uint32_t t = 0; t < TT; ++t) x[t] = *reinterpret_cast<const rf32x4*>(xr + t * kRtRow + 4u * c);
#pragma unroll
            for (uint32_t e = 0; e < TE; ++e) w[e] = *reinterpret_cast<const rf32x4*>(wr + e * kRtRow + 4u * c);
#pragma unroll
            for (uint32_t i = 0; i < 4; ++i)
#pragma unroll
                for (uint32_t t = 0; t < TT; ++t)
#pragma unroll
                    for (uint32_t e = 0; e < TE; ++e)
                        l[t][e] += static_cast<double>(__fmul_rn(w[e][i], x[t][i]));
            if (c % 4u == 3u) {
#pragma unroll
                for (uint32_t t = 0; t < TT; ++t)
#pragma unroll
                    for (uint32_t e = 0; e < TE; ++e) q[t][e] += fabs(l[t][e]);
            }
        }
        wave_lds_order();  // and the next stage's stores overwrite what they read
    };
    uint32_t k = 0;
    for (; k + NS * kRtK <= range; k += NS * kRtK)
#pragma unroll
        for (uint32_t i = 0; i < NS; ++i) stage(i, k + i * kRtK);
    if (k < range) stage(0u, k);
#pragma unroll
    for (uint32_t i = 0; i < NL; ++i) {
        const float n = group_sum<8>(sq[i]);
        if (lane % 8u == 0u) (i < TT ? nx[wave][pr + 8u * i] : nw[wave][pr + 8u * (i - TT)]) = n;
    }
    __syncthreads();  // every wave is past its staged operands
#pragma unroll
    for (uint32_t t = 0; t < TT; ++t)
#pragma unroll
        for (uint32_t e = 0; e < TE; ++e) {
            RouterSums& p = sh.part[wave][(ti + t) * R + ej + e];
            p.l = l[t][e];
            p.q = q[t][e];
        }
    __syncthreads();
    static_assert(T * R <= 64u * kRtWaves, "at most one (token, row) per thread");
    if (threadIdx.x >= T * R) return;
    const uint32_t t = threadIdx.x / R, e = threadIdx.x % R;
    double S = 0.0, Q = 0.0;
    float xx = 0.0f, ww = 0.0f;
    const double run = static_cast<double>(range);
#pragma unroll
    for (uint32_t w = 0; w < kRtWaves; ++w) {
        const RouterSums p = sh.part[w][threadIdx.x];
        // 16 |L| per inner run end, 8 at the range's end, and its offset at both ends of each run
        Q += 16.0 * p.q - 8.0 * fabs(p.l) + run * fabs(S);
        S += p.l;
        xx += nx[w][t];
        ww += nw[w][e];
    }
    // the squares were rounded and summed in FP32 (2^-10 covers it) and may have
    // underflowed (2^-100 each); router_bound covers the rest, 2^-126 the products
    // below FP32's range
    const double slack = 8192.0 * 0x1p-100;
    const double P = (1.0 + 0x1p-10) * sqrt((static_cast<double>(xx) + slack) * (static_cast<double>(ww) + slack));
    if (t0 + t < a.tokens && e0 + e < ER) {
        const uint64_t at = static_cast<uint64_t>(t0 + t) * ER + e0 + e;
        a.row_sum[at] = S;
        a.row_bound[at] = router_bound(Q + P) + 0x1p-126;
    }
}

// ---------------------------------------------------------------------------
// 2. Per-token ranking, route weights and expert counts.

template <int NS>
__global__ __launch_bounds__(256) void k_route_batch(MoePrefillArgs A) {
    extern __shared__ __attribute__((aligned(16))) float xs[];  // [hidden]
    __shared__ FallbackShared<256> fb;
    __shared__ uint32_t s_sel[kMaxTopK];
    __shared__ uint32_t s_state, s_ncand, s_cand[kMaxExperts];
    __shared__ double s_lo, s_S[kMaxExperts], s_B[kMaxExperts];
    const uint32_t t = blockIdx.x, lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint32_t E = A.layer.n_experts, K = A.layer.top_k;
    MoeDecodeArgs a = A.layer;  // this token's view
    a.x = A.x + static_cast<uint64_t>(t) * a.hidden;
    a.row_sum = A.row_sum + static_cast<uint64_t>(t) * (E + a.variant);
    a.row_bound = A.row_bound + static_cast<uint64_t>(t) * (E + a.variant);
    a.ids = A.ids + static_cast<uint64_t>(t) * K;
    a.probs = A.probs + static_cast<uint64_t>(t) * K;
    a.status = A.status;

    const XRegs xr = load_x_regs(a.x, a.hidden);
    RouteData<NS> rd;
    if (wave == 0) rd = load_route_data<NS>(a);
    store_x_regs(xs, xr, a.hidden);
    WaveRoutes<NS> w;
    auto rank = [&] {  // wave 0
        w = wave_route<NS>(a, rd);
        if (lane == 0) {
#pragma unroll
            for (uint32_t r = 0; r < kMaxTopK; ++r) s_sel[r] = w.sel[r];
            s_state = !w.finite ? 2u : w.certified ? 0u : 1u;
            s_lo = w.lo_min_sel;
            s_ncand = 0u;
        }
    };
    if (wave == 0) rank();
    __syncthreads();
    uint32_t state = s_state;  // uniform
    if (state == 1u) {
        // The batched router's bound does not certify the ranking: form the decode
        // router's sum and bound of every expert whose interval reaches the selected
        // ones, and rank again.  An expert below them by the coarser bound is below
        // them by the finer one, so the decision is the decode path's.
        if (wave == 0) {
#pragma unroll
            for (int m = 0; m < NS; ++m) {
                const uint32_t e = lane + 64u * m;
                if (e < E) {
                    s_S[e] = rd.S[m];
                    s_B[e] = rd.B[m];
                    if (!(rd.S[m] + rd.B[m] < w.lo_min_sel)) s_cand[atomicAdd(&s_ncand, 1u)] = e;
                }
            }
        }
        __syncthreads();
        const uint32_t nc = s_ncand;
        for (uint32_t c = wave; c < nc; c += 4u) {
            const uint32_t e = s_cand[c];
            double S, B;
            router_row_sum_bound(a.router + static_cast<uint64_t>(e) * a.hidden, xs, a.hidden / 256u, S, B);
            if (lane == 0u) {
                s_S[e] = S;
                s_B[e] = B;
            }
        }
        __syncthreads();
        if (wave == 0) {
#pragma unroll
            for (int m = 0; m < NS; ++m) {
                const uint32_t e = lane + 64u * m;
                rd.S[m] = s_S[e < E ? e : 0u];
                rd.B[m] = s_B[e < E ? e : 0u];
            }
            rank();
        }
        __syncthreads();
        state = s_state;
    }
    if (state == 2u) {
        if (wave == 0) flag_router_error(a);
        return;
    }
    uint32_t sel[kMaxTopK];
    if (state == 1u) {  // rare: exact serial logits of the candidates
        exact_routes<4, 256>(a, s_S, s_B, s_lo, xs, fb, true);
        if (fb.bad) {
            if (wave == 0) flag_router_error(a);
            return;
        }
#pragma unroll
        for (uint32_t r = 0; r < kMaxTopK; ++r) sel[r] = r < K ? fb.sel[r] : 0u;
        if (wave == 0) {
#pragma unroll
            for (int m = 0; m < NS; ++m)
                w.logit[m] = lane + 64u * m < E ? static_cast<float>(fb.logit[lane + 64u * m]) : -INFINITY;
        }
    } else {
#pragma unroll
        for (uint32_t r = 0; r < kMaxTopK; ++r) sel[r] = s_sel[r];
    }
    if (wave == 0) write_routes<NS>(a, sel, w.logit);
}

// ---------------------------------------------------------------------------
// 3. The gate/up GEMM's operands (gemm_split.hpp): one wave takes a token's row,
// finds its largest magnitude, and writes the row's scale, the two fp16 halves
// of every value and, per 32 values, their sum (accumulated in FP64, rounded
// once).  hidden is a multiple of 256.

__device__ __forceinline__ void split_row(const float* __restrict__ x, uint32_t n,
                                          uint16_t* __restrict__ parts, float* __restrict__ sums,
                                          float* __restrict__ scale) {
    const uint32_t lane = threadIdx.x & 63u;
    float m = 0.0f;
    for (uint32_t i = 4u * lane; i < n; i += 256u) {
        const rf32x4 v = *reinterpret_cast<const rf32x4*>(x + i);
        m = fmaxf(fmaxf(m, fmaxf(fabsf(v.x), fabsf(v.y))), fmaxf(fabsf(v.z), fabsf(v.w)));
    }
    m = static_cast<float>(lane63(group_max<64>(static_cast<double>(m))));
    float s, inv;
    split_scale(m, s, inv);
    if (lane == 0u) *scale = s;
    // eight values per lane and round (the last round of an odd multiple of 256
    // is half empty: those lanes repeat the row's last values and do not store)
    for (uint32_t c = 8u * lane; c - 8u * lane < n; c += 512u) {
        const bool ok = c < n;
        const uint32_t k = ok ? c : n - 8u;
        const rf32x4 v0 = *reinterpret_cast<const rf32x4*>(x + k);
        const rf32x4 v1 = *reinterpret_cast<const rf32x4*>(x + k + 4u);
        double sum = (static_cast<double>(v0.x) + v0.y) + (static_cast<double>(v0.z) + v0.w) +
                     ((static_cast<double>(v1.x) + v1.y) + (static_cast<double>(v1.z) + v1.w));
        sum = group_sum<4>(sum);
        uint4 hi, lo;  // stored order 0, 2, 1, 3, 4, 6, 5, 7
        split_pair(v0.x * inv, v0.z * inv, hi.x, lo.x);
        split_pair(v0.y * inv, v0.w * inv, hi.y, lo.y);
        split_pair(v1.x * inv, v1.z * inv, hi.z, lo.z);
        split_pair(v1.y * inv, v1.w * inv, hi.w, lo.w);
        if (ok) {
            uint16_t* d = parts + (k / 32u) * 64u + k % 32u;
            *reinterpret_cast<uint4*>(d) = hi;
            *reinterpret_cast<uint4*>(d + 32u) = lo;
            if ((lane & 3u) == 3u) sums[k / 32u] = static_cast<float>(sum);
        }
    }
}

// ---------------------------------------------------------------------------
// 4. Grouping (workgroup 0, 1024 threads): per-expert counts from the
// ids (LDS atomics), row ranges, the 64-row tile list and the assignments
// (token * top_k + route) grouped by expert.  Tokens the router flagged
// (ids 0xffffffff) take no rows.

constexpr uint32_t kGroupThreads = 1024;

// Tiles of an expert with c rows: 64-row ones (the last may hold 33 to 64), and one
// of at most 32 rows for what is left; or, when that makes no more workgroups
// than the chip holds at once (kGemmSlots), 32-row tiles only, since the longest
// workgroup then sets the time (77 tokens, 64 experts and a shared one: gate/up
// 42 -> 33 us).  The list holds every 64-row tile first, so the GEMMs' longest
// workgroups start first and short ones fill the tail (512 tokens, skewed load:
// gate/up 128 -> 119 us).
__device__ __forceinline__ uint32_t big_tiles(uint32_t c, bool split) {
    return split ? 0u : c / 64u + (c % 64u > 32u ? 1u : 0u);
}
__device__ __forceinline__ uint32_t small_tiles(uint32_t c, bool split) {
    return split ? (c + 31u) / 32u : (c % 64u > 0u && c % 64u <= 32u) ? 1u : 0u;
}

// Workgroup 0 groups; the others split x into the gate/up GEMM's operands, a
// row per wave, while it does, since the grouping alone would leave the rest of
// the chip idle.
__global__ __launch_bounds__(kGroupThreads) void k_group(MoePrefillArgs a) {
    if (blockIdx.x > 0u) {
        const uint32_t t = (blockIdx.x - 1u) * (kGroupThreads / 64u) + (threadIdx.x >> 6);
        const uint64_t h = a.layer.hidden;
        if (t < a.tokens)
            split_row(a.x + t * h, a.layer.hidden, a.x_parts + t * h * 2u, a.x_sums + t * (h / 32u),
                      a.x_scale + t);
        return;
    }
    constexpr uint32_t NE = kMaxExperts + 1;  // + the shared expert (variant 1)
    __shared__ uint32_t cnt[NE], off[NE + 1], tb[NE], ts[NE], fill[NE], split32;
    const uint32_t E = a.layer.n_experts, K = a.layer.top_k, V = a.layer.variant, tid = threadIdx.x;
    const uint32_t EE = E + V, KR = K + V, n = a.tokens * K;
    if (tid < EE) {
        cnt[tid] = 0u;
        fill[tid] = 0u;
    }
    __syncthreads();
    for (uint32_t i = tid; i < n; i += kGroupThreads) {
        const uint32_t e = a.ids[i];
        if (e < E) atomicAdd(&cnt[e], 1u);
    }
    // the shared expert takes every token the router did not flag
    if (V)
        for (uint32_t t = tid; t < a.tokens; t += kGroupThreads)
            if (a.ids[t * K] < E) atomicAdd(&cnt[E], 1u);
    __syncthreads();
    if (tid < 64) {  // exclusive prefix of rows and tiles: PER experts a lane, one wave scan
        constexpr uint32_t PER = (NE + 63u) / 64u;
        uint32_t c[PER];
        double l32 = 0.0;  // integer sums, exact in FP64
#pragma unroll
        for (uint32_t k = 0; k < PER; ++k) {
            const uint32_t e = tid * PER + k;
            c[k] = e < EE ? cnt[e] : 0u;
            l32 += static_cast<double>(small_tiles(c[k], true));
        }
        const uint32_t t32 = static_cast<uint32_t>(lane63(wave_inclusive_scan(l32)));
        const bool split = t32 * a.tile_wgs <= kGemmSlots;  // uniform
        double lc = 0.0, lt = 0.0, ls = 0.0;
#pragma unroll
        for (uint32_t k = 0; k < PER; ++k) {
            lc += static_cast<double>(c[k]);
            lt += static_cast<double>(big_tiles(c[k], split));
            ls += static_cast<double>(small_tiles(c[k], split));
        }
        const double ic = wave_inclusive_scan(lc), it = wave_inclusive_scan(lt), is = wave_inclusive_scan(ls);
        uint32_t o = static_cast<uint32_t>(ic - lc), b = static_cast<uint32_t>(it - lt);
        uint32_t sm = static_cast<uint32_t>(lane63(it)) + static_cast<uint32_t>(is - ls);
#pragma unroll
        for (uint32_t k = 0; k < PER; ++k) {
            const uint32_t e = tid * PER + k;
            if (e < EE) {
                off[e] = o;
                tb[e] = b;
                ts[e] = sm;
            }
            o += c[k];
            b += big_tiles(c[k], split);
            sm += small_tiles(c[k], split);
        }
        if (tid == 63u) {
            off[EE] = static_cast<uint32_t>(ic);
            a.n_tiles[0] = static_cast<uint32_t>(it) + static_cast<uint32_t>(is);
            split32 = split ? 1u : 0u;
        }
    }
    __syncthreads();
    if (tid <= EE) a.offsets[tid] = off[tid];
    if (tid < EE) {
        const bool split = split32 != 0u;
        const uint32_t nb = big_tiles(cnt[tid], split), ns = small_tiles(cnt[tid], split);
        for (uint32_t j = 0; j < nb; ++j) a.tiles[tb[tid] + j] = (tid << 16) | kTileBig | (2u * j);
        for (uint32_t j = 0; j < ns; ++j) a.tiles[ts[tid] + j] = (tid << 16) | (2u * nb + j);
    }
    // grouped rows hold slots token * (top_k + variant) + route (the shared
    // expert is route top_k); the order inside a group is free: every row's
    // result is independent
    for (uint32_t i = tid; i < n; i += kGroupThreads) {
        const uint32_t e = a.ids[i];
        if (e < E) a.perm[off[e] + atomicAdd(&fill[e], 1u)] = (i / K) * KR + i % K;
    }
    if (V)
        for (uint32_t t = tid; t < a.tokens; t += kGroupThreads)
            if (a.ids[t * K] < E) a.perm[off[E] + atomicAdd(&fill[E], 1u)] = t * KR + K;
}

// ---------------------------------------------------------------------------
// 6. Ordered combine.

// Four consecutive outputs per thread (hidden is a multiple of 256), every
// route's loads issued before the ordered sums.
__global__ __launch_bounds__(256) void k_combine(MoePrefillArgs a) {
    const uint32_t t = blockIdx.x, i = (blockIdx.y * 256u + threadIdx.x) * 4u;
    const uint32_t K = a.layer.top_k, H = a.layer.hidden, E = a.layer.n_experts;
    const uint32_t V = a.layer.variant, KR = K + V;
    if (i >= H) return;
    bool ok = true;
    for (uint32_t r = 0; r < K; ++r) ok = ok && a.ids[t * K + r] < E;
    if (!ok) return;  // the router flagged this token
    rf32x4 o[kMaxTopK + 1];
    float p[kMaxTopK + 1];
#pragma unroll
    for (uint32_t r = 0; r < kMaxTopK + 1; ++r) {
        const uint32_t rr = r < KR ? r : 0u;  // routes past the last re-read route 0 (unused)
        o[r] = *reinterpret_cast<const rf32x4*>(a.out + (static_cast<uint64_t>(t) * KR + rr) * H + i);
        p[r] = r < K ? a.probs[t * K + rr] : 0.0f;
    }
    rf32x4 y = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (uint32_t r = 0; r < kMaxTopK; ++r) {
        if (r < K) {
            y.x = __fadd_rn(y.x, __fmul_rn(p[r], o[r].x));
            y.y = __fadd_rn(y.y, __fmul_rn(p[r], o[r].y));
            y.z = __fadd_rn(y.z, __fmul_rn(p[r], o[r].z));
            y.w = __fadd_rn(y.w, __fmul_rn(p[r], o[r].w));
        }
    }
    if (V) {  // mixer_output = moe_result + sigmoid(shared gate) * shared (src/qwen35_runner.cpp:752-761)
        const float g = sigmoid35(static_cast<float>(a.row_sum[static_cast<uint64_t>(t) * (E + 1u) + E]));
        rf32x4 sh = o[0];
#pragma unroll
        for (uint32_t r = 1; r < kMaxTopK + 1; ++r) sh = r == K ? o[r] : sh;
        y.x = __fadd_rn(y.x, __fmul_rn(g, sh.x));
        y.y = __fadd_rn(y.y, __fmul_rn(g, sh.y));
        y.z = __fadd_rn(y.z, __fmul_rn(g, sh.z));
        y.w = __fadd_rn(y.w, __fmul_rn(g, sh.w));
    }
    *reinterpret_cast<rf32x4*>(a.y + static_cast<uint64_t>(t) * H + i) = y;
}

// ---------------------------------------------------------------------------
// Host side.

bool prefill_type_ok(uint32_t t) {
    return t == T_Q4_K || t == T_Q5_K || t == T_Q6_K || t == T_Q8_0 || t == T_Q4_0 || t == T_Q4_1;
}

uint32_t ceil_div_u(uint32_t a, uint32_t b) { return (a + b - 1u) / b; }

}  // namespace

uint32_t moe_prefill_max_tiles(uint32_t tokens, uint32_t top_k, uint32_t n_experts) {
    const uint32_t pairs = tokens * top_k;
    // 64-row tiles, one partly filled per expert, or fewer 32-row tiles than kGemmSlots
    const uint32_t touched = n_experts < pairs ? n_experts : pairs;
    const uint32_t t64 = pairs / kGemmTileM + touched, t32 = pairs / 32u + touched;
    return t64 > kGemmSlots ? t64 : t32 < kGemmSlots ? t32 : kGemmSlots;
}

bool moe_prefill_supported(uint32_t gate_type, uint32_t up_type, uint32_t down_type,
                           uint32_t hidden, uint32_t ffn, uint32_t n_experts, uint32_t top_k,
                           uint32_t tokens, uint32_t variant) {
    if (variant > 1u) return false;
    if (gate_type != up_type || !prefill_type_ok(gate_type) || !prefill_type_ok(down_type))
        return false;
    if (tokens == 0 || tokens > kMaxPrefillTokens) return false;
    if (hidden % 256u || ffn % 256u || hidden / 256u > 32u) return false;
    switch (hidden / 256u) {
        case 2: case 4: case 8: case 12: case 16: case 24: case 32: break;
        default: return false;
    }
    // hidden and ffn are multiples of 256: whole 128-row blocks, 32- and 64-value stages

    return n_experts >= 1 && n_experts <= kMaxExperts && top_k >= 1 && top_k <= kMaxTopK &&
           top_k <= n_experts;
}

hipError_t launch_prefill_routing(const MoePrefillArgs& a, hipStream_t s) {
    const MoeDecodeArgs& L = a.layer;
    // 1. router
    const uint32_t ER = L.n_experts + L.variant;
    if (ceil_div_u(ER, 32u) * ceil_div_u(a.tokens, 16u) >= kGemmSlots)
        hipLaunchKernelGGL((k_router_batch<2, 4>), dim3(ceil_div_u(ER, 32u), ceil_div_u(a.tokens, 16u)),
                           dim3(64 * kRtWaves), 0, s, a);
    else
        hipLaunchKernelGGL((k_router_batch<1, 2>), dim3(ceil_div_u(ER, 16u), ceil_div_u(a.tokens, 8u)),
                           dim3(64 * kRtWaves), 0, s, a);
    // 2. ranking
    const size_t xlds = L.hidden * sizeof(float);
    switch (slots_for(L.n_experts)) {
        case 1: hipLaunchKernelGGL(k_route_batch<1>, dim3(a.tokens), dim3(256), xlds, s, a); break;
        case 2: hipLaunchKernelGGL(k_route_batch<2>, dim3(a.tokens), dim3(256), xlds, s, a); break;
        default: hipLaunchKernelGGL(k_route_batch<4>, dim3(a.tokens), dim3(256), xlds, s, a); break;
    }
    // 3. grouping
    const dim3 ggrid(1u + ceil_div_u(a.tokens, kGroupThreads / 64u));
    hipLaunchKernelGGL(k_group, ggrid, dim3(kGroupThreads), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_prefill_gate_up(const MoePrefillArgs& a, hipStream_t s) {
    return launch_expert_gate_up(a, s);
}

hipError_t launch_prefill_down(const MoePrefillArgs& a, hipStream_t s) {
    const MoeDecodeArgs& L = a.layer;
    const hipError_t err = launch_expert_down(a, s);
    if (err != hipSuccess) return err;
    hipLaunchKernelGGL(k_combine, dim3(a.tokens, ceil_div_u(L.hidden, 1024u)), dim3(256), 0, s, a);
    return hipGetLastError();
}

}  // namespace pk
