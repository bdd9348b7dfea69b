// Int8 linear for many rows (a prompt, or a batch above the decode launches' 128 rows): one launch
// over all rows where the decode GEMM runs chunk after chunk of 128 rows and reads every weight
// once per chunk.
//
// A workgroup of 4 waves computes MT * 16 rows x 256 or 128 channels. Each wave owns NPW = 4 or 2
// n-tiles for all of the workgroup's rows, so a weight byte is loaded and dequantized once per
// workgroup, straight into the registers that the MFMAs read. x goes through LDS, its 16-byte chunks
// swapped round by the row's low three bits: the stores meet in no bank, a fragment read meets twice
// (rows r and r + 8; the counters call 4 of its 8 LDS cycles conflicts). Every fragment feeds NPW
// n-tiles. The products are taken transposed (weights as the A operand), so that a lane ends up with 4
// consecutive channels of one row and stores 8 bytes (16 of a split's partial). Stages are selected by
// compile-time indices in an unrolled loop: a copy between stages made the compiler wait for the loads
// where they were issued.
//
// Few workgroups per CU are bound by their own chain (barrier, x store, fragment reads, dequant,
// products), so each half k-tile's fragments and weights are made ready under the previous half's
// products: 0.47-0.60 -> 0.43-0.53 us per k-tile for one workgroup of 32 or 64 rows x 256 channels, and
// 0.25-0.34 us with 128 channels. Many are bound by the matrix cores together with what feeds them.
// Llama-3-8B gate||up at 2048 rows: 646-680 -> 416-445 us (707-744 -> 1081-1155 TFLOP/s; torch's fp16
// product of that size takes 418 us). The MFMAs and barriers alone take 272 us; without the dequant it
// would be 385, without the weight loads 323-360, without the x loads 374. Counters there: MFMA busy
// 59 %, 4.55 GB read out of L2 per call (10.4 TB/s), 71 % of the requests hits. Loads two or three
// k-tiles ahead measured the same, 8 waves per workgroup (128 x 512 or 256 x 256) 440-500 us: one barrier
// then holds the whole CU.
#include "w8a16_rows.h"

#include "w8a16_tiles.h"

namespace mx {
namespace w8a16 {

constexpr int kRowsWaves = 4;
constexpr int kRowsThreads = kRowsWaves * 64;
constexpr int rows_tiles(int npw) { return kRowsWaves * npw; }  // n-tiles per workgroup

// gridDim.y k ranges; with more than one, the scaled fp32 partial of each goes to
// partial[range][M][N] (no bias) for the split reduce.
template <int MT, int NPW, bool GU>
__global__ __launch_bounds__(kRowsThreads, 2) void gemm_rows_kernel(
    const uint16_t* __restrict__ x, int64_t xs, int M, const uint8_t* __restrict__ w, const uint16_t* __restrict__ scale,
    const uint16_t* __restrict__ bias, uint16_t* __restrict__ y, int64_t ys, int KT, int NT, int MB, bool wide,
    float* __restrict__ partial) {
    constexpr int ROWS = MT * 16;
    constexpr int XC = ROWS * 8 / kRowsThreads;  // 16-byte chunks of one x k-tile per thread
    static_assert(XC * kRowsThreads == ROWS * 8, "whole chunks per thread");
    constexpr bool AHEAD = MT < 8 || NPW < 4;  // fragments and dequant one half k-tile ahead
    __shared__ __attribute__((aligned(16))) _Float16 xl[AHEAD ? 3 : 2][ROWS * kTileK];

    // Consecutive workgroups go to the 8 XCDs in turn; each XCD takes a contiguous run of tiles,
    // row blocks first, so that the workgroups that share weights share an L2.
    const int total = gridDim.x, xcd = blockIdx.x & 7;
    const int tile = xcd * (total >> 3) + ((total & 7) < xcd ? (total & 7) : xcd) + (blockIdx.x >> 3);
    const int nb = tile / MB, row0 = (tile - nb * MB) * ROWS;
    const int k_lo = (int)((int64_t)blockIdx.y * KT / gridDim.y);
    const int nk = (int)((int64_t)(blockIdx.y + 1) * KT / gridDim.y) - k_lo;

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63, g = lane >> 4, r = lane & 15;
    const int nt0 = nb * rows_tiles(NPW) + wave * NPW;

    // x: thread chunk c = tid + u * 256 is chunk c % 8 of row c / 8; rows past M read the last one.
    const char* xb = reinterpret_cast<const char*>(x + (int64_t)row0 * xs + (int64_t)k_lo * kTileK);
    uint32_t xoff[XC];
    static_assert(kRowsThreads / 8 % 8 == 0, "a thread's rows share their low bits");
    const int xdst = (tid >> 3) * kTileK + (((tid & 7) ^ (tid >> 3 & 7)) * 8);
#pragma unroll
    for (int u = 0; u < XC; ++u) {
        const int c = tid + u * kRowsThreads, row = c >> 3, col = c & 7;
        const int last = M - 1 - row0;
        xoff[u] = 2u * ((uint32_t)(row < last ? row : last) * (uint32_t)xs + col * 8);
    }
    int wt[NPW];  // the wave's n-tiles; tiles past the last one read it and store nothing
#pragma unroll
    for (int p = 0; p < NPW; ++p) wt[p] = nt0 + p < NT ? nt0 + p : NT - 1;
    const uint32_t lane16 = (uint32_t)lane * 16;

    struct XStage {
        uint4 c[XC];
    };
    struct WStage {
        uint4 t[NPW];
    };
    auto load_x = [&](int j) {  // k-tiles past the range load its last one
        XStage s;
        const char* src = xb + (int64_t)(j < nk ? j : nk - 1) * (kTileK * 2);
#pragma unroll
        for (int u = 0; u < XC; ++u) s.c[u] = *reinterpret_cast<const uint4*>(src + xoff[u]);
        return s;
    };
    auto store_x = [&](int buf, const XStage s) {
#pragma unroll
        for (int u = 0; u < XC; ++u) *reinterpret_cast<uint4*>(&xl[buf][xdst + u * (kRowsThreads / 8 * kTileK)]) = s.c[u];
    };
    auto load_w = [&](int j) {
        WStage s;
        const int64_t first = (int64_t)(k_lo + (j < nk ? j : nk - 1)) * NT;
#pragma unroll
        for (int p = 0; p < NPW; ++p)
            s.t[p] = *reinterpret_cast<const uint4*>(w + (first + wt[p]) * 1024 + lane16);
        return s;
    };

    float4v acc[MT][NPW];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int p = 0; p < NPW; ++p) acc[mt][p] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
    const int frag = r * kTileK + (((2 * g) ^ (r & 7)) * 8);
    struct Frag {
        half8v a[MT];
    };
    struct Deq {
        half8v b[NPW];
    };
    // Half h of a k-tile: k = 16 g + 8 h + [0, 8) per lane.
    auto read = [&](int buf, int h) {
        Frag f;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) f.a[mt] = load_half8(&xl[buf][(frag ^ (8 * h)) + mt * 16 * kTileK]);
        return f;
    };
    auto deq = [&](const WStage s, int h) {
        Deq d;
#pragma unroll
        for (int p = 0; p < NPW; ++p) d.b[p] = h == 0 ? dequant8(s.t[p].x, s.t[p].y) : dequant8(s.t[p].z, s.t[p].w);
        return d;
    };
    auto mma = [&](const Frag f, const Deq d) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int p = 0; p < NPW; ++p)
                acc[mt][p] = __builtin_amdgcn_mfma_f32_16x16x32_f16(d.b[p], f.a[mt], acc[mt][p], 0, 0, 0);
    };

    if constexpr (AHEAD) {
        // While a half's products run, the next half's fragments are read and its weights dequantized,
        // across the barrier too: step j stores x k-tile j + 2 into the third buffer, so k-tile j + 1 is
        // readable throughout it. Slots are compile-time indices, the loop is unrolled U times.
        constexpr int WD = NPW < 4 ? 4 : 3, XD = NPW < 4 ? 2 : 1, U = NPW < 4 ? 12 : 3;
        static_assert(U % 3 == 0 && U % WD == 0 && U % XD == 0, "slots repeat every U steps");
        // The order within a half: two products, one fragment, a share of the dequant.
        auto mix = [&]() {
            constexpr int Q = MT * NPW / 2;
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                __builtin_amdgcn_sched_group_barrier(0x8, 2, 0);
                if (q < MT) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x2, 8 * NPW / Q + 1, 0);
            }
        };
        WStage ws[WD];
        XStage xst[XD];
        store_x(0, load_x(0));
        store_x(1, load_x(1));
#pragma unroll
        for (int u = 0; u < WD - 1; ++u) ws[u] = load_w(u);
#pragma unroll
        for (int u = 0; u < XD; ++u) xst[u] = load_x(2 + u);
        __syncthreads();
        Frag f0 = read(0, 0);
        Deq d0 = deq(ws[0], 0);
#define MX_ROWS_STEP(j, u)                                   \
    {                                                        \
        ws[((u) + WD - 1) % WD] = load_w((j) + WD - 1);      \
        const Frag f1 = read((u) % 3, 1);                    \
        const Deq d1 = deq(ws[(u) % WD], 1);                 \
        mma(f0, d0);                                         \
        mix();                                               \
        __builtin_amdgcn_sched_barrier(0);                   \
        store_x(((u) + 2) % 3, xst[(u) % XD]);               \
        xst[(u) % XD] = load_x((j) + 2 + XD);                \
        f0 = read(((u) + 1) % 3, 0);                         \
        d0 = deq(ws[((u) + 1) % WD], 0);                     \
        mma(f1, d1);                                         \
        mix();                                               \
        __builtin_amdgcn_sched_barrier(0);                   \
        __syncthreads();                                     \
    }
        int j = 0;
        for (; j + U <= nk; j += U) {
#pragma unroll
            for (int u = 0; u < U; ++u) MX_ROWS_STEP(j + u, u)
        }
#pragma unroll
        for (int u = 0; u < U - 1; ++u) {
            if (j + u < nk) MX_ROWS_STEP(j + u, u)
        }
#undef MX_ROWS_STEP
    } else {
        // 8 x 4 tiles per wave hold 128 accumulators: no registers for that. Step j stores x k-tile
        // j + 1 (loaded a step ago) into the other buffer, whose readers passed the last barrier,
        // issues the loads of the next stages and computes k-tile j, ahead of the other workgroup's
        // waves on the SIMD while they do the rest (4096 x 14336 at 4096 rows 413-415 against 421 us
        // without the priority; 6144 x 4096 there and gate||up 28672 x 4096 at 1100 rows the same).
        store_x(0, load_x(0));
        WStage w0 = load_w(0), w1;
        XStage xn = load_x(1);
        __syncthreads();
#define MX_ROWS_STEP(j, buf, cur, nxt)         \
    {                                          \
        store_x(1 - (buf), xn);                \
        nxt = load_w((j) + 1);                 \
        xn = load_x((j) + 2);                  \
        __builtin_amdgcn_sched_barrier(0);     \
        __builtin_amdgcn_s_setprio(1);         \
        mma(read(buf, 0), deq(cur, 0));        \
        mma(read(buf, 1), deq(cur, 1));        \
        __builtin_amdgcn_s_setprio(0);         \
        __builtin_amdgcn_sched_barrier(0);     \
        __syncthreads();                       \
    }
        int j = 0;
        for (; j + 1 < nk; j += 2) {
            MX_ROWS_STEP(j, 0, w0, w1)
            MX_ROWS_STEP(j + 1, 1, w1, w0)
        }
        if (j < nk) MX_ROWS_STEP(j, 0, w0, w1)
#undef MX_ROWS_STEP
    }

    // Lane (g, r) holds channels 4 g + [0, 4) of each n-tile for row r of each m-tile.
    const bool split = gridDim.y > 1;
#pragma unroll
    for (int p = 0; p < NPW; ++p) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int64_t n = (int64_t)wt[p] * kTileN + 4 * g + i;
            const float sc = h2f(scale, n), bi = bias && !split ? h2f(bias, n) : 0.0f;
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) acc[mt][p][i] = split ? acc[mt][p][i] * sc : acc[mt][p][i] * sc + bi;
        }
    }
    auto put = [&](uint16_t* dst, const uint16_t (&o)[4]) {
        if (wide) {
            *reinterpret_cast<uint2*>(dst) = uint2{o[0] | (uint32_t)o[1] << 16, o[2] | (uint32_t)o[3] << 16};
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) dst[i] = o[i];
        }
    };
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        const int m = row0 + mt * 16 + r;
        if constexpr (GU) {
            // Gate channels are lanes 0-31 of an n-tile, the matching up channels lanes 32-63: swapped
            // across a pair of n-tiles, every lane finishes four channels.
#pragma unroll
            for (int p = 0; p < NPW; p += 2) {
                uint16_t o[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    float gate = (float)(_Float16)pin_f32(acc[mt][p][i]), up = (float)(_Float16)pin_f32(acc[mt][p + 1][i]);
                    row_swap32(gate, up);
                    const _Float16 sg = (_Float16)silu_f32(gate);
                    o[i] = f2h_bits((float)sg * up);
                }
                const int nt = nt0 + p + (g >> 1);
                if (m < M && nt < NT) put(y + (int64_t)m * ys + nt * (kTileN / 2) + 4 * (g & 1), o);
            }
        } else {
#pragma unroll
            for (int p = 0; p < NPW; ++p) {
                if (m >= M || nt0 + p >= NT) continue;
                const int n = (nt0 + p) * kTileN + 4 * g;
                if (split) {
                    *reinterpret_cast<float4v*>(partial + ((int64_t)blockIdx.y * M + m) * (NT * kTileN) + n) = acc[mt][p];
                } else {
                    uint16_t o[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) o[i] = f2h_bits(pin_f32(acc[mt][p][i]));
                    put(y + (int64_t)m * ys + n, o);
                }
            }
        }
    }
}

template <int MT, int NPW, bool GU>
static void launch_rows_mt(int KS, const uint16_t* x, int64_t xs, int M, const uint8_t* w, const uint16_t* scale,
                           const uint16_t* bias, uint16_t* y, int64_t ys, int NT, int KT, float* partial, hipStream_t st) {
    const int MB = (int)ceil_div(M, MT * 16), NB = (int)ceil_div(NT, rows_tiles(NPW));
    const bool wide = aligned(y, 8) && ys % 4 == 0;
    hipLaunchKernelGGL((gemm_rows_kernel<MT, NPW, GU>), dim3((unsigned)(MB * NB), (unsigned)KS), dim3(kRowsThreads), 0, st, x, xs,
                       M, w, scale, bias, y, ys, KT, NT, MB, wide, partial);
}

// The tiles and k ranges of a launch, from what a k-tile costs a CU (us, measured on MI355X): alone on it
// a workgroup takes `alone` (its own chain), several share it at `shared` each; `fixed` covers launch,
// prologue and epilogue. Ranges add the fp32 partials, written and read again at about 4 TB/s, and the
// reduce launch. Narrow workgroups (2 n-tiles per wave, 128 channels) win where the wide ones leave CUs
// empty. Chosen against the 128-row chunks this replaced (us): 4096 x 14336 at 1531 rows 160-166 / 330 (96
// rows x 256 channels), at 256 rows 42 + reduce / 62 (128 x 128, 4 ranges); gate||up 28672 x 4096 at 2048
// rows 422 / 672 (96 x 256; 128 x 256 434), at 256 rows 65 / 83 (64 x 256), at 128 rows 41 / 44-46 (128 x
// 128), at 96 rows 35 / 43 (96 x 128); 1152 x 896 at 777 rows 8 / 74 (32 x 128); 6144 x 4096 at 512 rows 38 / 82
// (32 x 128).
RowsPlan plan_rows(int64_t M, int NT, int KT, size_t partial_bytes) {
    struct Shape {
        int mt, npw;
        float alone, shared, fixed;
    };
    constexpr Shape kShapes[] = {{2, 4, 0.43f, 0.31f, 4.7f},  {4, 4, 0.53f, 0.505f, 8.0f},  {6, 4, 0.62f, 0.68f, 11.0f},
                                 {8, 4, 1.00f, 0.97f, 14.3f}, {2, 2, 0.245f, 0.184f, 4.5f}, {4, 2, 0.34f, 0.31f, 6.0f},
                                 {6, 2, 0.41f, 0.44f, 7.7f},  {8, 2, 0.47f, 0.50f, 9.2f}};
    constexpr int kCus = 256;
    RowsPlan best{0, 0, 1};
    float best_us = 0.0f;
    for (const Shape& sh : kShapes)
        for (int ks = 1; ks <= 8; ks *= 2) {
            const float partial = (float)ks * M * NT * kTileN * sizeof(float);
            if (ks > 1 && (partial > (float)partial_bytes || KT / ks < 4)) break;
            const int64_t wgs = ceil_div(M, sh.mt * 16) * ceil_div(NT, rows_tiles(sh.npw)) * ks;
            const float per_cu = (float)ceil_div(wgs, kCus);
            const float tile_us = per_cu * sh.shared > sh.alone ? per_cu * sh.shared : sh.alone;
            const float us = tile_us * ceil_div(KT, ks) + sh.fixed + (ks > 1 ? 4.0f + 2 * partial / 4e6f : 0.0f);
            if (!best.MT || us < best_us) {
                best = RowsPlan{sh.mt, sh.npw, ks};
                best_us = us;
            }
        }
    return best;
}

bool rows_fit(int64_t M, int64_t xs, int NT) {
    // x rows of a workgroup are 32-bit byte offsets, workgroups and rows 32-bit counts.
    return M < (1 << 30) && xs < (1 << 23) && ceil_div(M, 32) * ceil_div(NT, rows_tiles(2)) < 0x7fffffff;
}

void launch_rows(bool gu, const RowsPlan& pl, const uint16_t* x, int64_t xs, int M, const uint8_t* w,
                 const uint16_t* scale, const uint16_t* bias, uint16_t* y, int64_t ys, int NT, int KT, float* partial,
                 hipStream_t st) {
#define MX_ROWS_SHAPE(T, P)                                                                                  \
    if (pl.MT == T && pl.NPW == P) {                                                                         \
        if (gu) launch_rows_mt<T, P, true>(1, x, xs, M, w, scale, bias, y, ys, NT, KT, nullptr, st);         \
        else launch_rows_mt<T, P, false>(pl.KS, x, xs, M, w, scale, bias, y, ys, NT, KT, partial, st);       \
    }
    MX_ROWS_SHAPE(2, 4)
    MX_ROWS_SHAPE(4, 4)
    MX_ROWS_SHAPE(6, 4)
    MX_ROWS_SHAPE(8, 4)
    MX_ROWS_SHAPE(2, 2)
    MX_ROWS_SHAPE(4, 2)
    MX_ROWS_SHAPE(6, 2)
    MX_ROWS_SHAPE(8, 2)
#undef MX_ROWS_SHAPE
}

}  // namespace w8a16
}  // namespace mx
