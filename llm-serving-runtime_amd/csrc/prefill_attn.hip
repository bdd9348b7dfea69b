// Causal attention of a prompt for gfx950: the prefill half of the block_paged attention hook
// (runtime/phase2/block_paged_attention.py:50-60, eager attention on the gathered K/V), which
// returns both the attention output and the whole weight matrix.
//
// Two passes over the keys in one launch, so that neither the scores nor unnormalised
// probabilities ever reach memory: pass 1 finds each row's maximum and sum, pass 2 recomputes the
// scores, writes p = exp2(score - max - log2(sum)) rounded to the element type as the weights and
// multiplies the same rounded values into V. The recomputed Q K^T costs 2 P S D flops per head; the
// eager chain moved the P x S matrix about eleven times (product, scale, mask, softmax, cast and
// second product), which is what bound it.
//
// A wave owns QT tiles of 16 query rows of one head and half of the keys: the workgroup stages two
// tiles of 64 tokens at a time in LDS, double buffered, K as rows and V transposed, four waves take
// the even tiles and four the same rows with the odd ones, and the pairs add up in LDS (the row's
// maximum and sum after pass 1, the output after pass 2). Scores are
// computed transposed (K rows as the A operand of v_mfma_f32_16x16x32, query rows as B), with the K
// rows of the two 16-token A tiles of 32 tokens taken in the order 8 * (r / 4) + r % 4 and that + 4:
// lane l then holds the scores of the eight consecutive tokens 8 * (l / 16) + [0, 8) of query row
// l % 16, which is the k order of the B operand of the same instruction. So p goes from the scores'
// registers into P.V with no exchange between lanes, and a lane stores 16 bytes of a weight row.
//
// The four waves of a key half take consecutive units of (row block, head of the kv-head's group),
// heads fastest: they share K and V, and their causal limits are close together. Later row blocks
// attend over more keys, so the heaviest workgroups are launched first.
//
// Bound by the weights' stores and by the exponentials, which do not overlap well: for the Llama-3-8B
// heads at 2048 tokens 99 us, of which 71 us remain without the stores (268 MB, 2.7 TB/s over the
// whole launch); the eager chain took 1.0 ms. Two workgroups of 4 waves per CU instead of one of 8
// with the keys split took 121 us there and 25 against 21 us for 509 of 685 tokens (a wave's own
// chain of load, product and softmax sets the pace).
#include <type_traits>

#include "common.h"
#include "elt.h"

namespace mx {
namespace prefill {

constexpr int kUnits = 4;           // units per workgroup
constexpr int kHalves = 2;          // key halves: waves per unit
constexpr int kThreads = kUnits * kHalves * 64;
constexpr int kTok = 64;            // tokens per tile
constexpr int kStep = kTok * kHalves;
constexpr int kVStride = kTok + 8;  // halfs per transposed V row: rows start 36 banks apart
constexpr int kCus = 256;
typedef uint32_t u32x4v __attribute__((ext_vector_type(4)));

struct Params {
    const _Float16* q;
    int64_t q_sb, q_sh, q_st;
    const _Float16* k;
    int64_t k_sb, k_sh, k_st;
    const _Float16* v;
    int64_t v_sb, v_sh, v_st;
    int Hkv, G, P, S;
    float scale_log2e;
    _Float16* out;      // [B, P, Hkv * G, D]
    _Float16* weights;  // [B, Hkv * G, P, S]
    int heads;          // B * Hkv
    int units;          // row blocks * G
    int wgs;            // workgroups per (row of the batch, kv-head)
};

template <int D, int QT, bool BF16, bool ALIGNED>
__global__ __launch_bounds__(kThreads, 2) void prefill_attn_kernel(Params p) {
    using E = Elt<BF16>;
    constexpr int KC = D / 32;          // 32-dim steps of a score
    constexpr int DT = D / 16;          // 16-dim output tiles
    constexpr int KS = D + 8;           // halfs per staged K row
    constexpr int KCH = kStep * D / 8 / kThreads;  // 16-byte K chunks per thread
    constexpr int QROWS = 16 * QT;
    constexpr int kTileK = kTok * KS, kTileV = D * kVStride;
    __shared__ __attribute__((aligned(16))) _Float16 ks[2][kHalves * kTileK];
    __shared__ __attribute__((aligned(16))) _Float16 vs[2][kHalves * kTileV];
    __shared__ float2 stat[kHalves][kUnits][QROWS];

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int half = wave / kUnits;
    const int lane = tid & 63, g = lane >> 4, r = lane & 15;

    const int head = blockIdx.x % p.heads, wg = p.wgs - 1 - blockIdx.x / p.heads;
    const int b = head / p.Hkv, kvh = head - b * p.Hkv;

    const int u_last = (wg * kUnits + kUnits < p.units ? wg * kUnits + kUnits : p.units) - 1;
    // A wave past the last unit repeats it and stores the same bytes to the same places.
    const int u = wg * kUnits + wave % kUnits < u_last ? wg * kUnits + wave % kUnits : u_last;
    const int row0 = u / p.G * QROWS, hq = kvh * p.G + u % p.G;
    const int off = p.S - p.P;                  // query row i sees tokens [0, i + off]
    const auto end_of = [&](int block_row0) {   // tokens the row block starting there attends over
        const int last = block_row0 + QROWS < p.P ? block_row0 + QROWS : p.P;
        return last + off;
    };
    const int wave_end = end_of(row0);
    const int steps = (end_of(u_last / p.G * QROWS) + kStep - 1) / kStep;

    // Query fragments: lane l holds dims 32 c + 8 (l / 16) + [0, 8) of row l % 16.
    half8v qf[QT][KC];
    int qpos[QT];
    const _Float16* qb = p.q + b * p.q_sb + hq * p.q_sh;
#pragma unroll
    for (int t = 0; t < QT; ++t) {
        // Rows past the prompt repeat its last row and store the same bytes to the same places.
        qpos[t] = row0 + 16 * t + r < p.P ? row0 + 16 * t + r : p.P - 1;
#pragma unroll
        for (int c = 0; c < KC; ++c)
            qf[t][c] = __builtin_bit_cast(half8v, *reinterpret_cast<const uint4*>(qb + qpos[t] * p.q_st + 32 * c + 8 * g));
    }

    const _Float16* kb = p.k + b * p.k_sb + kvh * p.k_sh;
    const _Float16* vb = p.v + b * p.v_sb + kvh * p.v_sh;
    // Loads are unconditional, so that a step's wait for the next one's loads never moves up to a
    // branch: rows past the last token load the last one (their scores are masked). Stages are passed by value: as captured arrays they
    // went to scratch memory.
    struct KStage {
        uint4 c[KCH];
    };
    struct VStage {
        half8v t[4];
    };
    auto load_k = [&](int step) {
        KStage st;
#pragma unroll
        for (int i = 0; i < KCH; ++i) {
            const int c = tid + i * kThreads, row = step * kStep + c / (D / 8);
            const uint32_t tok = row < p.S ? row : p.S - 1;
            st.c[i] = *reinterpret_cast<const uint4*>(kb + (tok * (uint32_t)p.k_st + c % (D / 8) * 8));
        }
        return st;
    };
    auto store_k = [&](int buf, const KStage st) {
#pragma unroll
        for (int i = 0; i < KCH; ++i) {
            const int c = tid + i * kThreads;
            *reinterpret_cast<uint4*>(&ks[buf][c / (D / 8) * KS + c % (D / 8) * 8]) = st.c[i];
        }
    };
    // V: a thread transposes 4 tokens x 8 dims (D 64: the last four waves repeat the first four).
    const int vt = (tid & 15) + 16 * ((tid >> 4) / (D / 8) % kHalves), vd = (tid >> 4) % (D / 8);
    auto load_v = [&](int step) {
        VStage st;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int row = step * kStep + 4 * vt + i;
            const uint32_t tok = row < p.S ? row : p.S - 1;
            st.t[i] = __builtin_bit_cast(half8v, *reinterpret_cast<const uint4*>(vb + (tok * (uint32_t)p.v_st + 8 * vd)));
        }
        return st;
    };
    auto store_v = [&](int buf, const VStage st) {
#pragma unroll
        for (int e = 0; e < 8; ++e)
            *reinterpret_cast<half4v*>(&vs[buf][(vt >> 4) * kTileV + (8 * vd + e) * kVStride + 4 * (vt & 15)]) =
                half4v{st.t[0][e], st.t[1][e], st.t[2][e], st.t[3][e]};
    };
    // Scores of the wave's tile of the step (tile = 2 * step + half), not yet scaled: s[h][t][i] is token tile * 64 + 32 h + 8 g + i of
    // row qpos[t], masked to -inf past the causal limit. MASK is false for the tiles that every row
    // of the wave sees whole: their code then has no branch, and the two halves overlap.
    auto scores = [&](auto mask, int tile, float (&s)[2][QT][8]) {
        float4v acc[2][QT][2];
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int t = 0; t < QT; ++t) acc[h][t][0] = acc[h][t][1] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
        const _Float16* row = &ks[(tile / kHalves) & 1][half * kTileK + (8 * (r >> 2) + (r & 3)) * KS + 8 * g];
#pragma unroll
        for (int c = 0; c < KC; ++c)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const _Float16* src = row + 32 * h * KS + 32 * c;
                const half8v a0 = __builtin_bit_cast(half8v, *reinterpret_cast<const uint4*>(src));
                const half8v a1 = __builtin_bit_cast(half8v, *reinterpret_cast<const uint4*>(src + 4 * KS));
#pragma unroll
                for (int t = 0; t < QT; ++t) {
                    acc[h][t][0] = E::mma32(a0, qf[t][c], acc[h][t][0]);
                    acc[h][t][1] = E::mma32(a1, qf[t][c], acc[h][t][1]);
                }
            }
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int t = 0; t < QT; ++t) {
                const int seen = qpos[t] + off - tile * kTok - 32 * h - 8 * g;  // i <= seen is visible
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const float v = acc[h][t][i >> 2][i & 3];
                    s[h][t][i] = !decltype(mask)::value || i <= seen ? v : -__builtin_huge_valf();
                }
            }
    };
    // Steps that every row of the workgroup sees whole (its first unit has the earliest rows). They
    // are walked in a loop of their own: with the masked tiles' conditional stores in the same loop
    // the wait for the next step's loads was a wait for every weight store as well.
    const int whole = (wg * kUnits / p.G * QROWS + off + 1) / kStep;

    // Pass 1. Every lane keeps the scaled maximum and the sum over its own tokens of each row; the four lanes
    // of a row meet after the last tile. The maximum starts at the lowest finite number, so that a
    // lane that has only seen masked tokens adds exp2(-inf) = 0 and no NaN.
    float m[QT], l[QT];
#pragma unroll
    for (int t = 0; t < QT; ++t) {
        m[t] = -3.4028235e38f;
        l[t] = 0.0f;
    }
    auto pass1 = [&](auto mask, int tile) {
        float s[2][QT][8];
        scores(mask, tile, s);
#pragma unroll
        for (int t = 0; t < QT; ++t) {
            float mx = s[0][t][0];
#pragma unroll
            for (int i = 1; i < 16; ++i) mx = fmaxf(mx, s[i >> 3][t][i & 7]);
            mx = fmaxf(m[t], mx * p.scale_log2e);
            float sum = 0.0f;
#pragma unroll
            for (int i = 0; i < 16; ++i)
                sum += __builtin_amdgcn_exp2f(__builtin_fmaf(s[i >> 3][t][i & 7], p.scale_log2e, -mx));
            l[t] = l[t] * __builtin_amdgcn_exp2f(m[t] - mx) + sum;
            m[t] = mx;
        }
    };
    store_k(0, load_k(0));
    __syncthreads();
    for (int step = 0; step < whole; ++step) {
        const KStage kn = load_k(step + 1);
        pass1(std::false_type{}, kHalves * step + half);
        store_k((step + 1) & 1, kn);
        __syncthreads();
    }
    for (int step = whole; step < steps; ++step) {
        const KStage kn = load_k(step + 1);
        const int tile = kHalves * step + half;
        if (tile * kTok < wave_end) pass1(std::true_type{}, tile);
        store_k((step + 1) & 1, kn);
        __syncthreads();
    }
    float bias[QT];  // p = exp2(score * scale_log2e + bias)
#pragma unroll
    for (int t = 0; t < QT; ++t) {
        const float mx = xor_max_16_32(m[t]);
        l[t] = xor_sum_16_32(l[t] * __builtin_amdgcn_exp2f(m[t] - mx));
        m[t] = mx;
        if (g == 0) stat[half][wave % kUnits][16 * t + r] = float2{m[t], l[t]};
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < QT; ++t) {
        const float2 other = stat[1 - half][wave % kUnits][16 * t + r];
        const float mx = fmaxf(m[t], other.x);
        const float sum = l[t] * __builtin_amdgcn_exp2f(m[t] - mx) + other.y * __builtin_amdgcn_exp2f(other.x - mx);
        bias[t] = -(mx + __builtin_amdgcn_logf(sum));
    }

    // Pass 2.
    float4v acc[DT][QT];
#pragma unroll
    for (int d = 0; d < DT; ++d)
#pragma unroll
        for (int t = 0; t < QT; ++t) acc[d][t] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
    const int64_t wrow = ((int64_t)b * p.Hkv * p.G + hq) * p.P;  // weight row of query row 0
    _Float16* wdst[QT];
#pragma unroll
    for (int t = 0; t < QT; ++t) wdst[t] = p.weights + (wrow + qpos[t]) * p.S + 8 * g;
    auto pass2 = [&](auto mask, int tile) {
        float s[2][QT][8];
        scores(mask, tile, s);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            half8v pr[QT];
#pragma unroll
            for (int t = 0; t < QT; ++t) {
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    pr[t][i] = E::round(__builtin_amdgcn_exp2f(__builtin_fmaf(s[h][t][i], p.scale_log2e, bias[t])));
                const int tok = tile * kTok + 32 * h;
                _Float16* dst = wdst[t] + tok;
                if (!decltype(mask)::value || tok + 8 * g + 8 <= p.S) {
                    if constexpr (ALIGNED) *reinterpret_cast<half8v*>(dst) = pr[t];
                    else __builtin_memcpy(dst, &pr[t], 16);
                } else if constexpr (!ALIGNED) {
#pragma unroll
                    for (int i = 0; i < 8; ++i)
                        if (tok + 8 * g + i < p.S) dst[i] = pr[t][i];
                }
            }
#pragma unroll
            for (int d = 0; d < DT; ++d) {
                const half8v a = __builtin_bit_cast(
                    half8v, *reinterpret_cast<const uint4*>(&vs[(tile / kHalves) & 1][half * kTileV + (16 * d + r) * kVStride + 32 * h + 8 * g]));
#pragma unroll
                for (int t = 0; t < QT; ++t) acc[d][t] = E::mma32(a, pr[t], acc[d][t]);
            }
        }
    };
    store_k(0, load_k(0));
    store_v(0, load_v(0));
    __syncthreads();
    for (int step = 0; step < whole; ++step) {
        const KStage kn = load_k(step + 1);
        const VStage vn = load_v(step + 1);
        pass2(std::false_type{}, kHalves * step + half);
        store_k((step + 1) & 1, kn);
        store_v((step + 1) & 1, vn);
        __syncthreads();
    }
    for (int step = whole; step < steps; ++step) {
        const KStage kn = load_k(step + 1);
        const VStage vn = load_v(step + 1);
        const int tile = kHalves * step + half;
        if (tile * kTok < wave_end) pass2(std::true_type{}, tile);
        store_k((step + 1) & 1, kn);
        store_v((step + 1) & 1, vn);
        __syncthreads();
    }
    // The odd tiles' half of the output joins the even tiles' through LDS (K is done with).
    static_assert(sizeof(ks) >= sizeof(float4v) * kUnits * DT * QT * 64, "output exchange");
    float4v* xch = reinterpret_cast<float4v*>(&ks[0][0]) + wave % kUnits * (DT * QT * 64) + lane;
    if (half == 1) {
#pragma unroll
        for (int d = 0; d < DT; ++d)
#pragma unroll
            for (int t = 0; t < QT; ++t) xch[(d * QT + t) * 64] = acc[d][t];
    }
    __syncthreads();

    // The weights of the tokens past the wave's last tile: 0, or NaN where the row's own are (the
    // softmax of a row with a NaN or a +inf score, or with none above -inf, whose bias is +inf, is NaN
    // at its masked tokens as well). Whole lines that nothing here reads again: stored with the
    // streaming policy, 113 -> 101 us for the Llama-3-8B heads at 2048 tokens. The weights' own stores,
    // half a line each, lost by it (121).
    const int zero0 = (wave_end + kTok - 1) / kTok * kTok;
    if (zero0 < p.S) {
        constexpr uint32_t kNan = BF16 ? 0x7fc07fc0u : 0x7e007e00u;
#pragma unroll
        for (int t = 0; t < QT; ++t)
            for (int i = half; i < 16; i += kHalves) {
                const int row = row0 + 16 * t + i;
                if (row >= p.P) break;
                const float bi = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, bias[t]), i));
                const uint32_t w = __builtin_fabsf(bi) < __builtin_huge_valf() ? 0u : kNan;
                const u32x4v fill{w, w, w, w};
                for (int tok = zero0 + 8 * lane; tok < p.S; tok += 512) {
                    _Float16* dst = p.weights + (wrow + row) * p.S + tok;
                    if constexpr (ALIGNED) {
                        __builtin_nontemporal_store(fill, reinterpret_cast<u32x4v*>(dst));
                    } else if (tok + 8 <= p.S) {
                        __builtin_memcpy(dst, &fill, 16);
                    } else {
                        for (int e = 0; tok + e < p.S; ++e) __builtin_memcpy(dst + e, &fill, 2);
                    }
                }
            }
    }
    if (half == 1) return;
    // Lane l holds dims 16 d + 4 (l / 16) + [0, 4) of row l % 16.
#pragma unroll
    for (int t = 0; t < QT; ++t) {
        _Float16* dst = p.out + (((int64_t)b * p.P + qpos[t]) * p.Hkv * p.G + hq) * D + 4 * g;
#pragma unroll
        for (int d = 0; d < DT; ++d) {
            const float4v sum = acc[d][t] + xch[(d * QT + t) * 64];
            half4v o;
#pragma unroll
            for (int i = 0; i < 4; ++i) o[i] = E::round(sum[i]);
            *reinterpret_cast<half4v*>(dst + 16 * d) = o;
        }
    }
}

template <int D, int QT, bool BF16>
static void launch(Params p, int64_t blocks, hipStream_t st) {
    p.units = (int)(blocks * p.G);
    p.wgs = (int)ceil_div(p.units, kUnits);
    const dim3 grid((unsigned)(p.wgs * p.heads)), block(kThreads);
    if (p.S % 8 == 0)
        hipLaunchKernelGGL((prefill_attn_kernel<D, QT, BF16, true>), grid, block, 0, st, p);
    else
        hipLaunchKernelGGL((prefill_attn_kernel<D, QT, BF16, false>), grid, block, 0, st, p);
}

// Two row tiles per wave (each K and V fragment read from LDS feeds two products) where that still
// gives every CU a workgroup, else one, which has twice the workgroups and half the work in each
// dependent step. Measured on MI355X, two against one: Llama-3-8B heads 2048 tokens 100 / 138 us,
// 1024 tokens (256 workgroups) 40.1 / 42.8, 512 tokens 25.0 / 20.1; Qwen2-0.5B heads 2048 tokens (224
// workgroups) 52.8 / 46.1, 509 of 685 tokens 32.1 / 21.4.
template <int D, bool BF16>
static void launch_qt(const Params& p, hipStream_t st) {
    const int64_t two = ceil_div(p.P, 32);
    if (ceil_div(two * p.G, kUnits) * p.heads >= kCus) launch<D, 2, BF16>(p, two, st);
    else launch<D, 1, BF16>(p, ceil_div(p.P, 16), st);
}

}  // namespace prefill
}  // namespace mx

using namespace mx;

extern "C" int mx_prefill_attn(const uint16_t* q, int64_t q_sb, int64_t q_sh, int64_t q_st, const uint16_t* k,
                               int64_t k_sb, int64_t k_sh, int64_t k_st, const uint16_t* v, int64_t v_sb, int64_t v_sh,
                               int64_t v_st, int32_t B, int32_t Hq, int32_t Hkv, int32_t P, int32_t S, int32_t D,
                               float scale, uint16_t* out, uint16_t* weights, uint32_t flags, void* stream) {
    clear_error();
    const char* what = "mx_prefill_attn";
    if (B < 0 || P < 0) return fail(MX_ERR_INVALID, "%s: B and P must be >= 0", what);
    if (B == 0 || P == 0) return MX_OK;
    if (!q || !k || !v || !out || !weights) return fail(MX_ERR_NULL, "%s: null pointer", what);
    if (Hkv <= 0 || Hq <= 0 || Hq % Hkv || S < P)
        return fail(MX_ERR_INVALID, "%s: need Hq a multiple of Hkv and S >= P (Hq=%d Hkv=%d P=%d S=%d)", what, Hq, Hkv, P, S);
    if (D != 64 && D != 128) return fail(MX_ERR_UNSUPPORTED, "%s: head_dim %d (64 or 128)", what, D);
    const float scale_log2e = scale * 1.4426950408889634f;
    if (!(scale >= 1.17549435e-38f) || scale_log2e > 3.4e38f)
        return fail(MX_ERR_UNSUPPORTED, "%s: scale must be positive and a normal fp32 number, also times log2(e)", what);
    if (flags & ~MX_PA_BF16) return fail(MX_ERR_INVALID, "%s: unknown flags", what);
    const int64_t strides[] = {q_sb, q_sh, q_st, k_sb, k_sh, k_st, v_sb, v_sh, v_st};
    for (int64_t s : strides)
        if (s % 8 || s < 0) return fail(MX_ERR_ALIGNMENT, "%s: strides must be multiples of 8 elements", what);
    if (!aligned(q, 16) || !aligned(k, 16) || !aligned(v, 16) || !aligned(out, 16) || !aligned(weights, 16))
        return fail(MX_ERR_ALIGNMENT, "%s: 16-byte alignment", what);
    // A token's row within a head is a 32-bit element offset.
    if ((int64_t)S * k_st > 0x7fffffff || (int64_t)S * v_st > 0x7fffffff)
        return fail(MX_ERR_UNSUPPORTED, "%s: K and V rows of a head must span less than 2^31 elements", what);
    // A launch holds fewer than 2^32 threads (that many workgroups only with two row tiles per wave,
    // see launch_qt). Indices of tokens, row blocks, units and workgroups then stay below 2^31.
    const int64_t wgs = (int64_t)B * Hkv * ceil_div(ceil_div((int64_t)P, 32) * (Hq / Hkv), prefill::kUnits);
    if (wgs > 0xffffffffll / prefill::kThreads || S > (1 << 30))
        return fail(MX_ERR_UNSUPPORTED, "%s: too many rows", what);
    prefill::Params p{};
    p.q = reinterpret_cast<const _Float16*>(q);
    p.q_sb = q_sb;
    p.q_sh = q_sh;
    p.q_st = q_st;
    p.k = reinterpret_cast<const _Float16*>(k);
    p.k_sb = k_sb;
    p.k_sh = k_sh;
    p.k_st = k_st;
    p.v = reinterpret_cast<const _Float16*>(v);
    p.v_sb = v_sb;
    p.v_sh = v_sh;
    p.v_st = v_st;
    p.Hkv = Hkv;
    p.G = Hq / Hkv;
    p.P = P;
    p.S = S;
    p.scale_log2e = scale_log2e;
    p.out = reinterpret_cast<_Float16*>(out);
    p.weights = reinterpret_cast<_Float16*>(weights);
    p.heads = B * Hkv;
    hipStream_t st = as_stream(stream);
    const bool bf16 = flags & MX_PA_BF16;
    if (D == 64) {
        if (bf16) prefill::launch_qt<64, true>(p, st);
        else prefill::launch_qt<64, false>(p, st);
    } else {
        if (bf16) prefill::launch_qt<128, true>(p, st);
        else prefill::launch_qt<128, false>(p, st);
    }
    return check_launch(what);
}
