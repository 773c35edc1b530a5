// prompt.hip -- the fast mode's prompt in batches: up to kPromptTokens positions
// through every layer at once instead of one token step each.
//
// The reference feeds a prompt one token at a time through forward_into
// (src/qwen3_moe_runner.cpp:580-704, the loop at :785-790), and so did the fast
// mode's step graph: about nine dependent launches of a few microseconds per
// layer and token, each reading every weight for one row.  Here each layer takes
// the whole chunk: the projections as dense GEMMs (expert_gemm.hip with one
// expert), the q/k norms, RoPE and KV append per position, causal attention per
// (head, position), and the MoE block as the batched prefill.  The sums are the
// fast step's within FP32 reassociation, and the KV ring holds k and v from the
// same norm, RoPE and FP16 rounding.  The last prompt token stays a step, so
// logits and the first new token come from the step's kernels.
//
// A dense GEMM's tiles leave most of the chip idle on a short prompt (127 tokens:
// 32 tiles of 32 x 256 for the output projection), so K is split over workgroups
// until kGemmSlots are filled; the consumers add the parts in order.
//
// 4 layers of hidden 2048, 128 experts, 32 heads, 128 tokens and 8 new ones:
// 19.9 -> 2.8 ms (one token step per prompt token before).
#include <hip/hip_fp16.h>
#include <math.h>

#include "gemm_split.hpp"
#include "kquant.hpp"
#include "launch.hpp"
#include "route.hpp"

namespace pk {
namespace {

// One value per lane, 32 consecutive columns per half wave (one chunk of the dense
// GEMM's operand): the chunk's scale, the two fp16 halves and the sum.
__device__ __forceinline__ void split_chunk(float v, uint32_t lane, uint64_t chunk, uint16_t* parts,
                                            float* scales, float* sums) {
    uint32_t u = __float_as_uint(v) & 0x7fffffffu;
    u = max(u, dpp_u0max<0xb1>(u));
    u = max(u, dpp_u0max<0x4e>(u));
    u = max(u, dpp_u0max<0x141>(u));
    u = max(u, dpp_u0max<0x140>(u));
    const auto w = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    float s, inv;
    split_scale(__uint_as_float(max(w[0], w[1])), s, inv);
    const float x = v * inv;
    const _Float16 h = static_cast<_Float16>(x);
    const _Float16 l = static_cast<_Float16>(x - static_cast<float>(h));
    const double sum = group_sum<32>(static_cast<double>(v));
    const uint32_t ln = lane & 31u, at = (ln & 24u) | kPairOrder(ln & 7u);
    parts[chunk * 64u + at] = __builtin_bit_cast(uint16_t, h);
    parts[chunk * 64u + 32u + at] = __builtin_bit_cast(uint16_t, l);
    if (ln == 31u) {
        scales[chunk] = s;
        sums[chunk] = static_cast<float>(sum);
    }
}

// The dense GEMMs' tile list: one group of `n` rows in order.
__global__ __launch_bounds__(256) void k_prompt_tiles(uint32_t n, uint32_t big, uint32_t tiles_n,
                                                      uint32_t* tiles, uint32_t* n_tiles,
                                                      uint32_t* offsets, uint32_t* perm) {
    for (uint32_t i = threadIdx.x; i < n; i += 256u) perm[i] = i;
    for (uint32_t i = threadIdx.x; i < tiles_n; i += 256u) tiles[i] = big ? (kTileBig | (2u * i)) : i;
    if (threadIdx.x == 0u) {
        n_tiles[0] = tiles_n;
        offsets[0] = 0u;
        offsets[1] = n;
    }
}

// The sum of np (at most kMaxParts) parts in order, every load issued before the
// first add (parts past the last re-read it).
constexpr uint32_t kMaxParts = 8;
template <typename V>
__device__ __forceinline__ V sum_parts(const float* p, uint32_t np, uint64_t stride) {
    V v[kMaxParts];
#pragma unroll
    for (uint32_t i = 0; i < kMaxParts; ++i)
        v[i] = *reinterpret_cast<const V*>(p + (i < np ? i : np - 1u) * stride);
    V s = v[0];
#pragma unroll
    for (uint32_t i = 1; i < kMaxParts; ++i) s = i < np ? s + v[i] : s;
    return s;
}

// Row t: h += the sum of `np` delta parts (if any), x = RMSNorm(h) * w
// (src/rms_norm.cpp:9-27, the sum of squares reassociated), and with parts the
// split operand of x.  n a multiple of 256, at most 8192.
__global__ __launch_bounds__(256) void k_prompt_norm(float* h, const float* delta, uint32_t np,
                                                     uint64_t part_stride, const float* w, uint32_t n,
                                                     float eps, float* x, uint16_t* parts,
                                                     float* scales, float* sums) {
    __shared__ __attribute__((aligned(16))) float row[8192];
    __shared__ float red[4];
    const uint32_t t = blockIdx.x, tid = threadIdx.x;
    float* hr = h + static_cast<uint64_t>(t) * n;
    float ss = 0.0f;
    for (uint32_t i = 4u * tid; i < n; i += 1024u) {
        rf32x4 v = *reinterpret_cast<const rf32x4*>(hr + i);
        if (delta) {
            const rf32x4 d = sum_parts<rf32x4>(delta + static_cast<uint64_t>(t) * n + i, np, part_stride);
            v = v + d;
            *reinterpret_cast<rf32x4*>(hr + i) = v;
        }
        *reinterpret_cast<rf32x4*>(row + i) = v;
        ss += (v.x * v.x + v.y * v.y) + (v.z * v.z + v.w * v.w);
    }
    ss = lane63(group_sum<64>(ss));
    if ((tid & 63u) == 0u) red[tid >> 6] = ss;
    __syncthreads();
    const float total = (red[0] + red[1]) + (red[2] + red[3]);
    const float scale = 1.0f / sqrtf(total / static_cast<float>(n) + eps);
    for (uint32_t i = tid; i < n; i += 256u) {  // consecutive columns in consecutive lanes
        const float v = row[i] * scale * w[i];
        if (x) x[static_cast<uint64_t>(t) * n + i] = v;
        if (parts) split_chunk(v, tid & 63u, (static_cast<uint64_t>(t) * n + i) / 32u, parts, scales, sums);
    }
}

// Block (b, t): for b < heads, q head b of position t: RMSNorm, RoPE, to qr; else kv
// head b - heads: the same for k, and k and v as FP16 into the ring (the step's
// k_fast_attention: the sum of squares in the reference's serial order, so the
// ring holds the same bits).
template <int HD>
__global__ __launch_bounds__(HD) void k_prompt_qk(PromptArgs a, ModelLayer L) {
    __shared__ float sq[HD], red;
    constexpr uint32_t HALF = HD / 2u;
    const uint32_t b = blockIdx.x, t = blockIdx.y, d = threadIdx.x, dp = d % HALF;
    const uint32_t pos = a.m.state[0] + t;
    const bool isq = b < a.m.heads;
    const uint32_t head = isq ? b : b - a.m.heads;
    const float* src = isq ? a.q + static_cast<uint64_t>(t) * a.q_stride : a.k + static_cast<uint64_t>(t) * a.kv_stride;
    const uint64_t part = isq ? a.q_part : a.kv_part;
    const float v = sum_parts<float>(src + head * HD + d, a.qkv_parts, part);
    float vv = 0.0f;
    if (!isq) vv = sum_parts<float>(a.v + static_cast<uint64_t>(t) * a.kv_stride + head * HD + d, a.qkv_parts, part);
    sq[d] = __fmul_rn(v, v);
    __syncthreads();
    if (d == 0u) {
        float s = 0.0f;
        for (uint32_t i = 0; i < HD; ++i) s = __fadd_rn(s, sq[i]);
        red = s;
    }
    __syncthreads();
    const float scale = 1.0f / sqrtf(red / static_cast<float>(HD) + a.m.rms_eps);
    const float x = v * scale * (isq ? L.q_norm : L.k_norm)[d];
    sq[d] = x;
    __syncthreads();
    const float* cs = a.m.rope_table + static_cast<uint64_t>(pos) * HD;
    const float c0 = cs[dp], s0 = cs[HALF + dp];
    const float r = d < HALF ? x * c0 - sq[d + HALF] * s0 : x * c0 + sq[dp] * s0;
    if (isq) {
        a.qr[static_cast<uint64_t>(t) * a.m.heads * HD + head * HD + d] = r;
        return;
    }
    const uint64_t at = (static_cast<uint64_t>(pos % a.m.capacity) * a.m.kv_heads + head) * HD + d;
    L.kcache[at] = __half_as_ushort(__float2half_rn(r));
    L.vcache[at] = __half_as_ushort(__float2half_rn(vv));
}

__device__ __forceinline__ float wave_sum_f(float v) { return lane63(group_sum<64>(v)); }
__device__ __forceinline__ float wave_max_f(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
    return v;
}

// Block (h, t): head h of position t over the ring's positions 0 .. pos (the chunk
// is inside the window, so nothing has wrapped), and the output's split operand.
template <int HD>
__global__ __launch_bounds__(256) void k_prompt_attention(PromptArgs a, ModelLayer L) {
    extern __shared__ __attribute__((aligned(16))) float sc[];  // scores
    constexpr uint32_t LP = HD / 8, ST = 4u * (64u / LP), U = 4;
    __shared__ float qv[HD], part[ST][HD], red[2][4];
    const uint32_t h = blockIdx.x, t = blockIdx.y, tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint32_t kvh = h / (a.m.heads / a.m.kv_heads);
    const uint32_t n = a.m.state[0] + t + 1u;
    const uint64_t row_halves = static_cast<uint64_t>(a.m.kv_heads) * HD;
    if (tid < HD) qv[tid] = a.qr[static_cast<uint64_t>(t) * a.m.heads * HD + h * HD + tid];
    __syncthreads();
    // scores, one position per thread (four partial dots), and their maximum
    float m = -INFINITY;
    for (uint32_t i = tid; i < n; i += 256u) {
        const u32x4_t* kr = reinterpret_cast<const u32x4_t*>(L.kcache + i * row_halves + kvh * HD);
        float p[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 8
        for (int j = 0; j < HD / 8; ++j) {
            const u32x4_t w = kr[j];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float k0 = __half2float(__ushort_as_half(static_cast<uint16_t>(w[e] & 0xffffu)));
                const float k1 = __half2float(__ushort_as_half(static_cast<uint16_t>(w[e] >> 16)));
                p[2 * (e & 1)] = __builtin_fmaf(qv[8 * j + 2 * e], k0, p[2 * (e & 1)]);
                p[2 * (e & 1) + 1] = __builtin_fmaf(qv[8 * j + 2 * e + 1], k1, p[2 * (e & 1) + 1]);
            }
        }
        const float s = ((p[0] + p[1]) + (p[2] + p[3])) * a.m.attn_scale;
        sc[i] = s;
        m = fmaxf(m, s);
    }
    m = wave_max_f(m);
    if (lane == 0u) red[0][wave] = m;
    __syncthreads();
    const float mx = fmaxf(fmaxf(red[0][0], red[0][1]), fmaxf(red[0][2], red[0][3]));
    float den = 0.0f;
    for (uint32_t i = tid; i < n; i += 256u) {
        const float e = expf(sc[i] - mx);
        sc[i] = e;
        den += e;
    }
    den = wave_sum_f(den);
    if (lane == 0u) red[1][wave] = den;
    __syncthreads();
    const float inv = 1.0f / (red[1][0] + red[1][1] + red[1][2] + red[1][3]);
    // output: LP lanes hold one position's row, so the workgroup runs ST interleaved
    // streams of positions, U loads each before their first use
    const uint32_t stream = tid / LP, d0 = 8u * (tid % LP);
    float acc[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    const uint16_t* vb = L.vcache + kvh * HD + d0;
    for (uint32_t i0 = stream; i0 < n; i0 += ST * U) {
        u32x4_t raw[U];
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
            const uint32_t i = i0 + ST * u;
            raw[u] = *reinterpret_cast<const u32x4_t*>(vb + (i < n ? i : i0) * row_halves);
        }
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
            const uint32_t i = i0 + ST * u;
            const float p = i < n ? sc[i] : 0.0f;
            if (i < n) {
#pragma unroll
                for (uint32_t j = 0; j < 8; ++j)
                    acc[j] = __builtin_fmaf(p, __half2float(__ushort_as_half(static_cast<uint16_t>(
                                                   raw[u][j / 2] >> (16 * (j % 2))))), acc[j]);
            }
        }
    }
#pragma unroll
    for (uint32_t j = 0; j < 8; ++j) part[stream][d0 + j] = acc[j];
    __syncthreads();
    if (tid < HD) {
        float o = 0.0f;
        for (uint32_t k = 0; k < ST; ++k) o += part[k][tid];
        const uint64_t at = static_cast<uint64_t>(t) * a.m.heads * HD + h * HD + tid;
        split_chunk(o * inv, lane, at / 32u, a.op_parts, a.op_scale, a.op_sums);
    }
}

__global__ void k_prompt_advance(uint32_t* state, uint32_t n) {
    if (threadIdx.x == 0u) state[0] += n;
}

bool gemm_type(uint32_t t) {
    return t == T_Q4_K || t == T_Q5_K || t == T_Q6_K || t == T_Q8_0 || t == T_Q4_0 || t == T_Q4_1;
}

// W (n_out rows of `in`) times the chunk's split rows: out[part][t][n_out].
hipError_t dense(const PromptArgs& a, uint32_t type, const uint8_t* W, uint32_t n_out, uint32_t in,
                 float* out, uint32_t parts, hipStream_t s) {
    MoePrefillArgs g = a.moe;
    g.layer.down = W;
    g.layer.down_type = type;
    g.layer.hidden = n_out;
    g.layer.ffn = in;
    g.layer.n_experts = 1;
    g.layer.variant = 0;
    g.max_tiles = a.dense_tiles;
    g.tiles = a.d_tiles;
    g.n_tiles = a.d_tiles + a.dense_tiles;
    g.offsets = a.d_offsets;
    g.perm = a.d_perm;
    g.act_parts = a.op_parts;
    g.act_scale = a.op_scale;
    g.act_sums = a.op_sums;
    g.out = out;
    g.k_parts = parts;
    g.precise = 1;
    g.out_part = static_cast<uint64_t>(a.tokens) * n_out;
    return launch_expert_down(g, s);
}

// Workgroups along K for a dense GEMM of n_out rows: as many as fill the chip's slots.
uint32_t k_parts_for(uint32_t tiles, uint32_t n_out, uint32_t in) {
    const uint32_t wgs = tiles * (n_out / 256u), most = in / 256u < kMaxParts ? in / 256u : kMaxParts;
    const uint32_t p = wgs < kGemmSlots ? kGemmSlots / wgs : 1u;
    return p < most ? p : most;
}

uint32_t dense_rows(uint32_t tokens, uint32_t n_out) {  // rows per tile
    return (tokens + 31u) / 32u * (n_out / 256u) <= kGemmSlots ? 32u : 64u;
}

}  // namespace

bool prompt_supported(const ModelArgs& m, const ModelLayer* layers) {
    const uint32_t qd = m.heads * m.head_dim, kd = m.kv_heads * m.head_dim;
    if (m.exact || m.hidden % 256u || m.hidden > 8192u || qd % 256u || kd % 256u) return false;
    if (m.head_dim != 64u && m.head_dim != 128u && m.head_dim != 256u) return false;
    for (uint32_t l = 0; l < m.layers; ++l) {
        const MoeDecodeArgs& g = layers[l].moe;
        if (!gemm_type(layers[l].attn_type)) return false;
        if (!moe_prefill_supported(g.gate_type, g.up_type, g.down_type, g.hidden, g.ffn, g.n_experts,
                                   g.top_k, kPromptTokens))
            return false;
    }
    return true;
}

uint64_t prompt_scratch(const ModelArgs& m, const ModelLayer* layers, uint32_t tokens, uint8_t* base,
                        PromptArgs& a) {
    uint64_t at = 0;
    auto take = [&](auto*& p, uint64_t n) {
        using P = std::remove_reference_t<decltype(*p)>;
        p = reinterpret_cast<P*>(base + at);
        at += (n * sizeof(P) + 255u) / 256u * 256u;
    };
    const uint64_t T = tokens, qd = uint64_t(m.heads) * m.head_dim, kd = uint64_t(m.kv_heads) * m.head_dim;
    uint64_t E = 1, K = 1, F = 256;
    for (uint32_t l = 0; l < m.layers; ++l) {
        E = layers[l].moe.n_experts > E ? layers[l].moe.n_experts : E;
        K = layers[l].moe.top_k > K ? layers[l].moe.top_k : K;
        F = layers[l].moe.ffn > F ? layers[l].moe.ffn : F;
    }
    const uint64_t H = m.hidden, W = qd > H ? qd : H;
    // a projection's parts: tiles * (n_out / 256) * parts <= kGemmSlots, or one part
    const uint64_t slots = uint64_t(kGemmSlots) * 256u *
                           dense_rows(tokens, static_cast<uint32_t>(qd + 2 * kd > H ? qd + 2 * kd : H));
    auto parts_floats = [&](uint64_t n_out) { return T * n_out > slots ? T * n_out : slots; };
    a.m = m;
    take(a.h, T * H);
    take(a.x, T * H);
    take(a.y, T * H);
    take(a.qr, T * qd);
    take(a.proj, parts_floats(qd + 2 * kd) + parts_floats(kd) * 2u);
    take(a.attn_out, parts_floats(H));
    take(a.op_parts, 2 * T * W);
    take(a.op_scale, T * W / 32u);
    take(a.op_sums, T * W / 32u);
    take(a.d_tiles, (T + 31u) / 32u + 1u);
    take(a.d_offsets, 2);
    take(a.d_perm, T);
    MoePrefillArgs& g = a.moe;
    const uint64_t P = T * K;
    a.moe_tiles = moe_prefill_max_tiles(tokens, static_cast<uint32_t>(K), static_cast<uint32_t>(E));
    take(g.row_sum, T * E);
    take(g.row_bound, T * E);
    take(g.offsets, E + 1);
    take(g.tiles, a.moe_tiles + 1u);
    take(g.perm, P);
    take(g.x_parts, 2 * T * H);
    take(g.x_sums, T * H / 32u);
    take(g.x_scale, T);
    take(g.act_parts, 2 * P * F);
    take(g.act_sums, P * F / 32u);
    take(g.act_scale, P * F / 32u);
    take(g.out, P * H);
    take(g.ids, P);
    take(g.probs, P);
    return at;
}

hipError_t launch_prompt_chunk(PromptArgs a, const ModelLayer* layers, uint32_t tokens, uint32_t pos0,
                               hipStream_t s) {
    const ModelArgs& m = a.m;
    const uint32_t qd = m.heads * m.head_dim, kd = m.kv_heads * m.head_dim, H = m.hidden;
    hipError_t err;
    a.tokens = tokens;
    ModelArgs em = m;
    em.hidden_state = a.h;
    if ((err = launch_embed(em, tokens, m.hidden, s))) return err;
    // the tile list of the dense GEMMs: one for both, from the wider
    const uint32_t rows = dense_rows(tokens, qd + 2u * kd > H ? qd + 2u * kd : H);
    a.dense_tiles = (tokens + rows - 1u) / rows;
    hipLaunchKernelGGL(k_prompt_tiles, dim3(1), dim3(256), 0, s, tokens, rows == 64u ? 1u : 0u,
                       a.dense_tiles, a.d_tiles, a.d_tiles + a.dense_tiles, a.d_offsets, a.d_perm);
    const float* delta = nullptr;
    auto norm = [&](const float* d, uint32_t parts, const float* w, float* x, bool split) {
        hipLaunchKernelGGL(k_prompt_norm, dim3(tokens), dim3(256), 0, s, a.h, d, parts,
                           static_cast<uint64_t>(tokens) * H, w, H, m.rms_eps, x,
                           split ? a.op_parts : nullptr, a.op_scale, a.op_sums);
    };
    for (uint32_t l = 0; l < m.layers; ++l) {
        const ModelLayer& L = layers[l];
        norm(delta, 1u, L.attn_norm, nullptr, true);
        if (L.qkv) {  // q, k and v in one GEMM
            const uint32_t n = qd + 2u * kd;
            a.qkv_parts = k_parts_for(a.dense_tiles, n, H);
            a.q = a.proj;
            a.k = a.q + qd;
            a.v = a.k + kd;
            a.q_stride = a.kv_stride = n;
            a.q_part = a.kv_part = static_cast<uint64_t>(tokens) * n;
            if ((err = dense(a, L.attn_type, L.qkv, n, H, a.proj, a.qkv_parts, s))) return err;
        } else {
            a.qkv_parts = k_parts_for(a.dense_tiles, qd, H);
            float* q = a.proj;
            float* k = q + static_cast<uint64_t>(a.qkv_parts) * tokens * qd;
            float* v = k + static_cast<uint64_t>(a.qkv_parts) * tokens * kd;
            a.q = q;
            a.k = k;
            a.v = v;
            a.q_stride = qd;
            a.kv_stride = kd;
            a.q_part = static_cast<uint64_t>(tokens) * qd;
            a.kv_part = static_cast<uint64_t>(tokens) * kd;
            if ((err = dense(a, L.attn_type, L.q, qd, H, q, a.qkv_parts, s))) return err;
            if ((err = dense(a, L.attn_type, L.k, kd, H, k, a.qkv_parts, s))) return err;
            if ((err = dense(a, L.attn_type, L.v, kd, H, v, a.qkv_parts, s))) return err;
        }
        const dim3 gq(m.heads + m.kv_heads, tokens), ga(m.heads, tokens);
        const size_t lds = static_cast<size_t>(pos0 + tokens) * sizeof(float);
#define PK_PA(HD)                                                                              \
    case HD:                                                                                   \
        hipLaunchKernelGGL(k_prompt_qk<HD>, gq, dim3(HD), 0, s, a, L);                         \
        hipLaunchKernelGGL(k_prompt_attention<HD>, ga, dim3(256), lds, s, a, L);               \
        break;
        switch (m.head_dim) {
            PK_PA(64) PK_PA(128) PK_PA(256)
            default: return hipErrorInvalidValue;
        }
#undef PK_PA
        const uint32_t op = k_parts_for(a.dense_tiles, H, qd);
        if ((err = dense(a, L.attn_type, L.o, H, qd, a.attn_out, op, s))) return err;
        norm(a.attn_out, op, L.ffn_norm, a.x, false);
        MoePrefillArgs g = a.moe;
        g.layer = L.moe;
        g.tokens = tokens;
        g.max_tiles = moe_prefill_max_tiles(tokens, L.moe.top_k, L.moe.n_experts);
        g.tile_wgs = moe_prefill_tile_wgs(H, L.moe.ffn);
        g.n_tiles = g.tiles + g.max_tiles;
        g.x = a.x;
        g.y = a.y;
        g.status = L.moe.status;
        if ((err = launch_prefill_routing(g, s))) return err;
        if ((err = launch_prefill_gate_up(g, s))) return err;
        if ((err = launch_prefill_down(g, s))) return err;
        delta = a.y;
    }
    return launch_advance(m.state, tokens, s);
}

hipError_t launch_advance(uint32_t* state, uint32_t n, hipStream_t s) {
    hipLaunchKernelGGL(k_prompt_advance, dim3(1), dim3(64), 0, s, state, n);
    return hipGetLastError();
}

}  // namespace pk
