// Grouped LUT-GEMM for few tokens per expert (3 tokens and more, up to about
// 24 positions an expert): weights streamed straight to registers, looked up
// there, and multiplied on MFMA (16 x 16 x 32, gfx950).
//
// It stands between the decode GEMV kernels, which look every weight up again
// for each pass of one to four tokens and spend VALU dot products and cross-lane
// sums on them, and the prefill ring kernel, whose 256-row tiles through 150 KB
// of LDS leave one wave a SIMD.  What bounds it is HBM.  A CTA is 8 waves of 16
// weight rows (gate/up: 8 gate and 8 up rows, so the SwiGLU pair meets in one
// wave) and one work item: up to 16 NM positions of one expert.  Two CTAs a CU,
// 4 waves a SIMD.
//   K step: 128 columns.  Lane (n = l % 16, g = l / 16) holds columns 32g ..
//     32g + 31 of row n: BL4 16 code bytes, NestedLUT one 32-weight group, REF 32
//     code bytes; its block's table (or absmax) beside them.  The next two
//     steps are in flight while two are looked up, none of it through LDS.
//   Lookups: BL4 / NestedLUT by v_perm over the block's table as byte planes.
//     REF: the fp32 codebook in LDS, one copy per bank (32 KB, entry c of lane l
//     at 128 c + 4 (l % 32)): a lookup never meets another lane's bank, where 64
//     random entries of one copy take 6-8 cycles.
//   Activations: the item's rows, KC columns at a time, in LDS in fragment order
//     (a fragment read is 64 lanes x 16 consecutive bytes), for BL4 / NestedLUT
//     with every 8 columns in the order the lookups leave their weights in.
// Results leave the accumulators as runs of 4 outputs of one position.
//
// Before / here, us a layer (the GEMV kernels up to 32 tokens, the ring above):
// Qwen shape BL4 T = 32 / 64 / 256 145 / 185 / 195 -> 120 / 130 / 157, REF T = 19 / 64
// 143 / 231 -> 108 / 144, NestedLUT tiers T = 16 / 64 83 / 183 -> 73 / 111; Mixtral
// shape BL4 T = 16 / 64 576 / 408 -> 300 / 345 (4.7 TB/s at T = 16).
#include "common.h"
#include "kernels.h"
#include "lut_core.h"

using namespace lutmoe;
using lutmoe_host::StreamRoute;

namespace {

constexpr int kWaves = 8;

struct StreamArgs {
    lutmoe_weights w;
    const uint16_t* src;   // gate/up: x [T][K]; down: act [P][K]
    void* dst;             // gate/up: act bf16 [P][I]; down: y fp32 [P][M] per K split
    int64_t split_stride;  // floats between the K splits' y
    StreamRoute r;
};

// A weight array, uniform and in global memory (pointers that come from memory
// would otherwise be loaded from with flat loads).
typedef __attribute__((address_space(1))) const uint8_t* gbytes_t;
typedef __attribute__((address_space(1))) const uint32_t* gwords_t;
typedef __attribute__((address_space(1))) const u32x4_t* gquads_t;
__device__ __forceinline__ gbytes_t weight_array(const void* p) {
    const uint64_t v = (uint64_t)p;
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return (gbytes_t)(((uint64_t)hi << 32) | lo);
}
// N dwords at p
template <int N>
__device__ __forceinline__ void load_words(uint32_t (&d)[N], gbytes_t p) {
    if constexpr (N % 4 == 0) {
#pragma unroll
        for (int i = 0; i < N; i += 4) {
            const u32x4_t v = *(gquads_t)(p + 4 * i);
            d[i] = v[0];
            d[i + 1] = v[1];
            d[i + 2] = v[2];
            d[i + 3] = v[3];
        }
    } else {
#pragma unroll
        for (int i = 0; i < N; ++i) d[i] = ((gwords_t)p)[i];
    }
}

__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// One K step's weights of one lane, and their MFMA fragments.  B: code bits of
// a table format (BL4: 4).
template <int kFmt, int B>
struct Step {
    static constexpr bool kBl4 = kFmt == LUTMOE_FMT_BL4;
    static constexpr int kTab = (1 << B) / 2;      // table dwords of a block
    uint32_t c[B], t[kTab];

    // row_c / row_t: byte offsets of the lane's row; g: lane group (tail: g & 1)
    __device__ __forceinline__ void load(gbytes_t codes, gbytes_t tabs, uint32_t row_c, uint32_t row_t, int step,
                                         int g) {
        const uint32_t co = row_c + (uint32_t)(4 * step + g) * (4 * B);
        const uint32_t to = row_t + (uint32_t)(2 * step + (g >> 1)) * (4 * kTab);
        load_words(c, codes + co);
        load_words(t, tabs + to);
    }
    // the loaded words as values that appear here: the compiler then derives
    // nothing from them (and waits for them) before this point
    __device__ __forceinline__ void arrive() {
#pragma unroll
        for (int i = 0; i < B; ++i) asm volatile("" : "+v"(c[i]));
#pragma unroll
        for (int i = 0; i < kTab; ++i) asm volatile("" : "+v"(t[i]));
    }
    __device__ __forceinline__ void planes(uint32_t* lo, uint32_t* hi) const { table_planes<B>(t, lo, hi); }
    __device__ __forceinline__ bf16x8_t frag(const uint32_t* lo, const uint32_t* hi, int j) const {
        uint32_t w;
        if constexpr (kBl4) w = c[j];
        else w = nested_code8<B>(c[0], c[1], B >= 3 ? c[B >= 3 ? 2 : 0] : 0u, B >= 4 ? c[B >= 4 ? 3 : 0] : 0u, j);
        return __builtin_bit_cast(bf16x8_t, regtab_lookup8_eo<B>(lo, hi, w));
    }
};

struct RefStep {
    u32x4_t c[2];
    uint32_t am;
    __device__ __forceinline__ void load(const uint8_t* codes, const uint16_t* absmax, uint32_t row_c, uint32_t row32,
                                         uint32_t q32, uint32_t nb, int step, int g) {
        const uint32_t u = (uint32_t)(4 * step + g);
        c[0] = *reinterpret_cast<const u32x4_t*>(codes + row_c + 32 * u);
        c[1] = *reinterpret_cast<const u32x4_t*>(codes + row_c + 32 * u + 16);
        am = absmax[min((row32 + u) / q32, nb - 1u)];
    }
    __device__ __forceinline__ void arrive() {
        asm volatile("" : "+v"(c[0]), "+v"(c[1]), "+v"(am));
    }
    // 8 codes -> bf16(cb[c] * absmax), in column order (the product of two
    // bf16 values is exact in fp32; one rounding, as the reference dequantises)
    __device__ __forceinline__ bf16x8_t frag(uint32_t cbase, int j) const {
        const float a = bf16_to_f32(am);
        u32x4_t r;
#pragma unroll
        for (int d = 0; d < 2; ++d) {
            const uint32_t w = c[j >> 1][2 * (j & 1) + d];
            const uint32_t we = (w & 0x00ff00ffu) << 7;   // 128 * codes 0, 2 (16-bit fields)
            const uint32_t wo = (w >> 1) & 0x7f807f80u;   // 128 * codes 1, 3
            const float e0 = __uint_as_float(lds_ld32(add_word<0>(cbase, we)));
            const float o0 = __uint_as_float(lds_ld32(add_word<0>(cbase, wo)));
            const float e1 = __uint_as_float(lds_ld32(add_word<1>(cbase, we)));
            const float o1 = __uint_as_float(lds_ld32(add_word<1>(cbase, wo)));
            r[2 * d] = f32x2_to_bf16x2(e0 * a, o0 * a);
            r[2 * d + 1] = f32x2_to_bf16x2(e1 * a, o1 * a);
        }
        return __builtin_bit_cast(bf16x8_t, r);
    }
};

template <int kFmt, bool kGateUp, int NM>
__global__ __launch_bounds__(64 * kWaves, 4) void stream_kernel(StreamArgs A) {
    constexpr bool kRef = kFmt == LUTMOE_FMT_REF, kNested = kFmt == LUTMOE_FMT_NESTED;
    constexpr int KC = (kRef ? 1024 : 2048) / NM;   // columns of activations in LDS
    constexpr int KS = KC / 128;                    // their K steps
    static_assert(KS % 4 == 0, "a staging holds whole rounds of the K loop");
    __shared__ __attribute__((aligned(16))) uint8_t s_x[KC * 16 * NM * 2];
    __shared__ __attribute__((aligned(16))) float s_cb[kRef ? 256 * 32 : 4];
    const RouteChunks* ch = A.r.chunks;
    const int item = blockIdx.y;
    if (item >= __builtin_amdgcn_readfirstlane(ch->nchunk)) return;
    const int e = __builtin_amdgcn_readfirstlane(ch->ce[item]);
    const int p0 = __builtin_amdgcn_readfirstlane(ch->cp0[item]);
    const int n = __builtin_amdgcn_readfirstlane(ch->cn[item]);
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int ln = lane & 15, g = lane >> 4;
    const int M = A.w.rows, K = A.w.cols;
    const int I = M / 2;   // (gate/up)
    // K steps [st0, st0 + nst) of this CTA's K split
    const int nst_all = (K + 127) / 128, st0 = nst_all * (int)blockIdx.z / (int)gridDim.z;
    const int nst = nst_all * ((int)blockIdx.z + 1) / (int)gridDim.z - st0;
    const bool half_tail = (K & 64) != 0;   // the last step has 64 columns: groups 2, 3 past K
    // first output of the wave, and this lane's weight row
    const int o0 = (int)blockIdx.x * (kGateUp ? 64 : 128) + wv * (kGateUp ? 8 : 16);
    const uint32_t row = kGateUp ? (uint32_t)min(ln < 8 ? o0 + ln : I + o0 + ln - 8, M - 1)
                                 : (uint32_t)min(o0 + ln, M - 1);
    f32x4_t acc[NM];
#pragma unroll
    for (int m = 0; m < NM; ++m) acc[m] = f32x4_t{0.f, 0.f, 0.f, 0.f};

    // the item's source rows, one a lane (lane t: position t), read back by
    // lane index; every load of a staging round is issued before any is used
    int srow = p0 + min(lane, n - 1);
    if constexpr (kGateUp) srow = A.r.perm[srow] / A.r.ke;
    // the KC columns from step s0 of the item's activation rows -> LDS: 16-byte
    // piece q of position t (step q / 16, group, j) at fragment (step, j, t / 16),
    // lane 16 group + t % 16.  Rows past the item's n stay unwritten: they only
    // reach accumulator columns that are not stored.
    auto stage = [&](int step0) __attribute__((always_inline)) {
        const int s0 = st0 + step0;
        constexpr int kPieces = KC / 8;   // of a row; a wave's 64 lie in one row
        const int total = n * kPieces;
        for (int i0 = 0; i0 < total; i0 += 4 * 64 * kWaves) {
            u32x4_t v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int i = i0 + u * 64 * kWaves + tid;
                const int t = min(__builtin_amdgcn_readfirstlane(i / kPieces), n - 1);
                const int64_t r = __builtin_amdgcn_readlane(srow, t);
                const int col = min(128 * s0 + 8 * (i & (kPieces - 1)), K - 8);
                v[u] = *reinterpret_cast<const u32x4_t*>(A.src + r * K + col);
            }
            // landed here on every path (a load that a lane drops would be waited
            // for at the head of the K loop, in each of its rounds)
            asm volatile("" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]));
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int i = i0 + u * 64 * kWaves + tid;
                const int t = i / kPieces, q = i & (kPieces - 1);
                if (t < n) {
                    const bool in = 128 * s0 + 8 * q < K;   // past K: zero
                    const int f = ((q >> 4) * 4 + (q & 3)) * NM + (t >> 4), l = ((q >> 2) & 3) * 16 + (t & 15);
                    const u32x4_t x = kRef ? v[u] : eo_order(v[u]);
                    *reinterpret_cast<u32x4_t*>(s_x + (f * 64 + l) * 16) = in ? x : u32x4_t{0u, 0u, 0u, 0u};
                }
            }
        }
    };
    // step s (of the staged KS): the four fragments' MFMAs
    auto mma = [&](int s, int j, bf16x8_t w) __attribute__((always_inline)) {
#pragma unroll
        for (int m = 0; m < NM; ++m) {
            const bf16x8_t x = *reinterpret_cast<const bf16x8_t*>(
                s_x + ((((s & (KS - 1)) * 4 + j) * NM + m) * 64 + lane) * 16);
            acc[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, x, acc[m], 0, 0, 0);
        }
    };
    // the K loop: load(buffer, step, group), use(buffer, step, last step of 64).
    // Steps go in pairs (256 columns: a pair's loads touch whole 128-byte lines
    // of a row together), the next pair's loads issued before a pair is used.
    // The loop over pairs that have a next pair has no condition around its
    // loads, so the compiler's wait counts keep them in flight.
    // (Steps are counted from st0.)
    auto k_loop = [&](auto* buf, auto load, auto use) __attribute__((always_inline)) {
        auto load_pair = [&](int b, int s) __attribute__((always_inline)) {
            const int a0 = st0 + min(s, nst - 1), a1 = st0 + min(s + 1, nst - 1);
            load(buf[b], a0, half_tail && a0 == nst_all - 1 ? g & 1 : g);
            load(buf[b + 1], a1, half_tail && a1 == nst_all - 1 ? g & 1 : g);
            __builtin_amdgcn_sched_barrier(0);
        };
        auto use_step = [&](int b, int s, bool tail) __attribute__((always_inline)) {
            buf[b].arrive();
            use(buf[b], s, tail);
            __builtin_amdgcn_sched_barrier(0);
        };
        load_pair(0, 0);
        for (int c0 = 0; c0 < nst; c0 += KS) {
            if (c0) lds_barrier();   // every wave is done with the columns in LDS
            stage(c0);
            lds_barrier();
            const int c1 = min(c0 + KS, nst);
            int s0 = c0;
            for (; s0 + 4 <= c1 && s0 + 4 < nst; s0 += 4) {
                load_pair(2, s0 + 2);
                use_step(0, s0, false);
                use_step(1, s0 + 1, false);
                load_pair(0, s0 + 4);
                use_step(2, s0 + 2, false);
                use_step(3, s0 + 3, false);
            }
            // at most one round of 4 left (the last of K)
            if (s0 < c1) {
                if (s0 + 2 < nst) load_pair(2, s0 + 2);
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    if (s0 + u >= c1) break;
                    use_step(u, s0 + u, half_tail && st0 + s0 + u == nst_all - 1);
                }
            }
        }
    };
    const bf16x8_t zero = __builtin_bit_cast(bf16x8_t, u32x4_t{0u, 0u, 0u, 0u});
    if constexpr (kRef) {
        {   // the bank-private codebook copies: thread t writes half of entry t / 2
            const float c = bf16_to_f32(ref_codebook(A.w, e)[tid >> 1]);
#pragma unroll
            for (int i = 0; i < 4; ++i)
                *reinterpret_cast<f32x4_t*>(&s_cb[(tid >> 1) * 32 + (tid & 1) * 16 + 4 * i]) = f32x4_t{c, c, c, c};
        }
        const uint8_t* codes = (const uint8_t*)A.w.codes + (int64_t)e * M * K;
        const uint16_t* am = (const uint16_t*)A.w.tables + (int64_t)e * A.w.absmax_per_expert;
        const uint32_t q32 = (uint32_t)A.w.block_size / 32u, nb = (uint32_t)A.w.absmax_per_expert;
        const uint32_t cbase = lds_addr(s_cb) + 4u * (uint32_t)(lane & 31);
        RefStep buf[4];
        k_loop(buf,
               [&](RefStep& b, int s, int gg) __attribute__((always_inline)) {
                   b.load(codes, am, row * (uint32_t)K, row * (uint32_t)(K / 32), q32, nb, s, gg);
               },
               [&](RefStep& b, int s, bool tail) __attribute__((always_inline)) {
#pragma unroll
                   for (int j = 0; j < 4; ++j) {
                       bf16x8_t w = b.frag(cbase, j);
                       if (tail) w = g >= 2 ? zero : w;   // (lanes past K read other weights)
                       mma(s, j, w);
                   }
               });
    } else {
        auto run = [&](auto BC, gbytes_t codes, gbytes_t tabs) __attribute__((always_inline)) {
            constexpr int B = decltype(BC)::value;
            using St = Step<kFmt, B>;
            const uint32_t row_c = row * (uint32_t)(K / 8 * B), row_t = row * (uint32_t)(K / 64 * 4 * St::kTab);
            St buf[4];
            k_loop(buf,
                   [&](St& b, int s, int gg) __attribute__((always_inline)) { b.load(codes, tabs, row_c, row_t, s, gg); },
                   [&](St& b, int s, bool tail) __attribute__((always_inline)) {
                       uint32_t lo[(1 << B) / 4], hi[(1 << B) / 4];
                       b.planes(lo, hi);
                       if (tail && g >= 2) {   // lanes past K read another block: zero weights
#pragma unroll
                           for (int i = 0; i < (1 << B) / 4; ++i) lo[i] = hi[i] = 0u;
                       }
#pragma unroll
                       for (int j = 0; j < 4; ++j) mma(s, j, b.frag(lo, hi, j));
                   });
        };
        if constexpr (kNested) {
            const gbytes_t codes = weight_array(((const void* const*)A.w.codes)[e]);
            const gbytes_t tabs = weight_array(((const void* const*)A.w.tables)[e]);
            const int bits = __builtin_amdgcn_readfirstlane((int)A.w.tier_bits[e]);
            if (bits == 4) run(std::integral_constant<int, 4>{}, codes, tabs);
            else if (bits == 3) run(std::integral_constant<int, 3>{}, codes, tabs);
            else run(std::integral_constant<int, 2>{}, codes, tabs);
        } else {
            const int64_t per = (int64_t)M * (K / 2);
            run(std::integral_constant<int, 4>{}, weight_array((const uint8_t*)A.w.codes + e * per),
                weight_array((const uint8_t*)A.w.tables + e * per));
        }
    }
    // D: lane (position n, g), element i -> weight row 4g + i of the wave's 16
#pragma unroll
    for (int m = 0; m < NM; ++m) {
        const int t = 16 * m + ln;
        const int64_t p = p0 + t;
        if constexpr (kGateUp) {
            float a[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) a[i] = silu_mul(acc[m][i], from_upper_half(acc[m][i]));   // lanes < 32: gate, up
            if (t < n && g < 2 && o0 < I)
                *reinterpret_cast<u32x2_t*>((uint16_t*)A.dst + p * I + o0 + 4 * g) =
                    u32x2_t{f32x2_to_bf16x2(a[0], a[1]), f32x2_to_bf16x2(a[2], a[3])};
        } else if (t < n && o0 < M) {
            const float pw = A.r.pos_w ? A.r.pos_w[p] : A.r.pair_w[A.r.perm[p]];
            *reinterpret_cast<f32x4_t*>((float*)A.dst + blockIdx.z * A.split_stride + p * M + o0 + 4 * g) =
                f32x4_t{acc[m][0] * pw, acc[m][1] * pw, acc[m][2] * pw, acc[m][3] * pw};
        }
    }
}

template <bool kGateUp, int NM>
void stream_launch(const StreamArgs& A, dim3 grid, hipStream_t s) {
    const dim3 block(64 * kWaves);
    switch (A.w.format) {
        case LUTMOE_FMT_REF: hipLaunchKernelGGL((stream_kernel<LUTMOE_FMT_REF, kGateUp, NM>), grid, block, 0, s, A); break;
        case LUTMOE_FMT_NESTED: hipLaunchKernelGGL((stream_kernel<LUTMOE_FMT_NESTED, kGateUp, NM>), grid, block, 0, s, A); break;
        default: hipLaunchKernelGGL((stream_kernel<LUTMOE_FMT_BL4, kGateUp, NM>), grid, block, 0, s, A); break;
    }
}

// *ns: K splits allowed (down), and taken.
template <bool kGateUp>
int stream_dispatch(const StreamArgs& A, int* ns, hipStream_t s) {
    const int out = kGateUp ? A.w.rows / 2 : A.w.rows, per = kGateUp ? 64 : 128;
    const int cu = lutmoe_host::cu_count(), ncu = cu > 0 ? cu : 256;
    const int64_t ctas = (int64_t)((out + per - 1) / per) * A.r.max_chunks;
    // fewer CTAs than CUs and a long K: split it in two (below 4096 columns the
    // second y costs the combine about what the split gains)
    *ns = *ns >= 2 && ctas <= ncu && A.w.cols >= 4096 ? 2 : 1;
    const dim3 grid((out + per - 1) / per, A.r.max_chunks, *ns);
    if (A.r.positions > 16) stream_launch<kGateUp, 2>(A, grid, s);
    else stream_launch<kGateUp, 1>(A, grid, s);
    return lutmoe_host::check_launch();
}

}  // namespace

namespace lutmoe_host {

bool stream_supported(const lutmoe_moe_desc* d) {
    // 32-bit byte offsets within an expert
    for (const lutmoe_weights* w : {&d->w13, &d->w2}) {
        if ((int64_t)w->rows * w->cols >= (int64_t(1) << 32)) return false;
        if (w->format == LUTMOE_FMT_REF && (w->block_size % 32 || w->absmax_per_expert >= (int64_t(1) << 31)))
            return false;
    }
    return true;
}

int launch_stream_gate_up(const lutmoe_moe_desc* d, const uint16_t* x, const StreamRoute& r, uint16_t* act,
                          hipStream_t s) {
    int ns = 1;
    return stream_dispatch<true>(StreamArgs{d->w13, x, act, 0, r}, &ns, s);
}

int launch_stream_down(const lutmoe_moe_desc* d, const uint16_t* act, const StreamRoute& r, float* y, int64_t stride,
                       int max_split, int* nsplit, hipStream_t s) {
    *nsplit = max_split;
    return stream_dispatch<false>(StreamArgs{d->w2, act, y, stride, r}, nsplit, s);
}

}  // namespace lutmoe_host
