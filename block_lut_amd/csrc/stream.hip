// Grouped LUT-GEMM for few tokens per expert (3 tokens and more; past 32 tokens
// up to 27 positions an expert): weights streamed to registers, looked up
// there, and multiplied on MFMA (16 x 16 x 32, gfx950).
//
// It stands between the decode GEMV kernels, which look every weight up again
// for each pass of one to four tokens and spend VALU dot products and cross-lane
// sums on them, and the prefill ring kernel, whose 256-row tiles through 150 KB
// of LDS leave one wave a SIMD.  What bounds it is HBM where an expert is large
// (Mixtral shape gate/up 5.0 TB/s, the copy rate); at the Qwen shape (3.0-4.4
// TB/s) the VALU, issuing 46-57 % of a CU's busy time, and a grid of one or two
// rounds of the chip.  A CTA is 8 waves of 16
// weight rows (gate/up: 8 gate and 8 up rows, so the SwiGLU pair meets in one
// wave) and one work item: up to 16 NM positions of one expert.  Two CTAs a CU,
// 4 waves a SIMD.
//   K step: 128 columns.  Lane (n = l % 16, g = l / 16) looks up columns 32g ..
//     32g + 31 of row n: BL4 16 code bytes, NestedLUT one 32-weight group, REF 32
//     code bytes; its block's table (or absmax) beside them.  REF loads them
//     itself.  BL4 / NestedLUT rows are loaded in 16-byte pieces on consecutive
//     lanes, three steps ahead, and reach their lane through 2 KB of LDS that the
//     wave has to itself: 16 rows on consecutive lanes cost the address unit a
//     cache line a lane (Mixtral shape BL4 T = 16 / 64 352 / 385 -> 312 / 364 us
//     on one card, NestedLUT 283 / 365 -> 270 / 346, Qwen shape 1-4 % less).
//   Lookups: BL4 / NestedLUT by v_perm over the block's table as byte planes.
//     REF: the fp32 codebook in LDS, one copy per bank (32 KB, entry c of lane l
//     at 128 c + 4 (l % 32)): a lookup never meets another lane's bank, where 64
//     random entries of one copy take 6-8 cycles.
//   Activations: the item's rows, KC columns at a time, in LDS in fragment order
//     (a fragment read is 64 lanes x 16 consecutive bytes), for BL4 / NestedLUT
//     with every 8 columns in the order the lookups leave their weights in.
// Results leave the accumulators as runs of 4 outputs of one position.
//
// Before / here, us a layer (the GEMV kernels up to 32 tokens, the ring above;
// rotating layers, each pair of figures from one card, and cards differ by 5 %):
// Qwen shape BL4 T = 32 / 64 / 256 145 / 185 / 195 -> 119 / 129 / 155, REF T = 19 / 64
// 143 / 231 -> 108 / 144, NestedLUT tiers T = 16 / 64 83 / 183 -> 68 / 111; Mixtral
// shape BL4 T = 16 / 64 576 / 408 -> 299 / 341 (4.7 TB/s at T = 16).
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
typedef u32x4_t u32x4_a4_t __attribute__((aligned(4)));   // (3-bit codes and 2-bit tables: 8-byte aligned)
typedef __attribute__((address_space(1))) const u32x4_a4_t* gquads_t;
__device__ __forceinline__ gbytes_t weight_array(const void* p) {
    const uint64_t v = (uint64_t)p;
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return (gbytes_t)(((uint64_t)hi << 32) | lo);
}
__device__ __forceinline__ u32x4_t load16(gbytes_t p, uint32_t off) {
    return *(gquads_t)(p + off);
}
__device__ __forceinline__ u32x4_t lds_ld128(uint32_t a) {
    return *(__attribute__((address_space(3))) const u32x4_t*)a;
}
__device__ __forceinline__ void lds_st128(uint32_t a, u32x4_t v) {
    *(__attribute__((address_space(3))) u32x4_t*)a = v;
}

__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// Keeps a wave-uniform condition a branch (not selects on every path).
__device__ __forceinline__ void rare_branch() { asm volatile(""); }

constexpr int kSlotB = 2048;   // LDS bytes of a wave's K step of weights

// A wave's weights of one K step (16 rows x 128 columns) go global -> registers
// in 16-byte pieces of a row on consecutive lanes (a load of 16 bytes a lane
// from 16 different rows on consecutive lanes would take a cache line access
// per lane), then through the wave's LDS slot to the lane that looks them up:
// lane (n, g), columns 32g .. 32g + 31 of row n.  B: code bits (BL4: 4).
template <int B>
struct Weights {
    static constexpr int kTab = (1 << B) / 2;   // table dwords of a block
    static constexpr int CP = B, TP = kTab / 2; // 16-byte pieces of a row's codes / tables per step
    uint32_t off_c, off_t;      // this lane's pieces, from the step's first byte of the arrays
    uint32_t wr_c, wr_t;        // their LDS addresses
    uint32_t rd_c, rd_t[2];     // LDS addresses of lane (n, g)
    int cp, tp;
    struct Raw {
        u32x4_t c, t;
    };
    struct Step {
        uint32_t c[B], t[kTab];
    };
    static __device__ __forceinline__ int swz(int r) { return B == 4 ? (r >> 1) & 3 : 0; }

    // row(i): the weight row of the wave's row i
    template <class RowFn>
    __device__ __forceinline__ void init(int lane, int K, uint32_t slot, RowFn row) {
        const int cr = min(lane / CP, 15), tr = min(lane / TP, 15);
        cp = lane < 16 * CP ? lane % CP : CP - 1;   // (lanes past the pieces repeat the last)
        tp = lane < 16 * TP ? lane % TP : TP - 1;
        off_c = row(cr) * (uint32_t)(K / 8 * B) + 16u * (uint32_t)cp;
        off_t = row(tr) * (uint32_t)(K / 64 * 4 * kTab) + 16u * (uint32_t)tp;
        wr_c = slot + (uint32_t)(cr * 16 * CP + 16 * (cp ^ swz(cr)));
        wr_t = slot + 1024u + (uint32_t)(tr * 16 * TP + 16 * (tp ^ swz(tr)));
        const int n = lane & 15, g = lane >> 4;
        rd_c = slot + (uint32_t)(n * 16 * CP + (B == 4 ? 16 * (g ^ swz(n)) : 4 * B * g));
#pragma unroll
        for (int h = 0; h < 2; ++h)
            rd_t[h] = slot + 1024u +
                      (uint32_t)(n * 16 * TP + (B == 4 ? 16 * ((2 * (g >> 1) + h) ^ swz(n)) : 4 * kTab * (g >> 1)));
    }
    // tail: the step has 64 columns; pieces past the row's end start at its last
    // 16 bytes instead
    __device__ __forceinline__ void load(Raw& r, gbytes_t codes, gbytes_t tabs, int step, bool tail) const {
        // offsets from the arrays' starts (never below them: a wrapped 32-bit
        // offset would point 4 GiB past)
        uint32_t oc = off_c + (uint32_t)step * (16 * CP), ot = off_t + (uint32_t)step * (16 * TP);
        if (tail) {
            rare_branch();
            oc -= 16u * (uint32_t)cp - (uint32_t)min(16 * cp, 8 * B - 16);
            if constexpr (B > 2) {
                ot -= 16u * (uint32_t)tp - (uint32_t)min(16 * tp, 4 * kTab - 16);
            } else {   // 8 bytes of table left: the 16 that end there (never before the array)
                ot -= min(ot, 8u);
            }
        }
        r.c = load16(codes, oc);
        r.t = load16(tabs, ot);
    }
    // the loaded words as values that appear here: the compiler then derives
    // nothing from them (and waits for them) before this point
    static __device__ __forceinline__ void arrive(Raw& r) { asm volatile("" : "+v"(r.c), "+v"(r.t)); }
    __device__ __forceinline__ void store(const Raw& r, int step, bool tail) const {
        uint32_t c = wr_c, t = wr_t;
        u32x4_t tv = r.t;
        if (tail) {
            rare_branch();
            const int lane = (int)threadIdx.x & 63;
            const int cr = min(lane / CP, 15), tr = min(lane / TP, 15);
            const int cs = min(16 * cp, 8 * B - 16);   // byte start within the row's step
            c = wr_c - (uint32_t)(16 * (cp ^ swz(cr))) + (uint32_t)(B == 4 ? 16 * ((cs >> 4) ^ swz(cr)) : cs);
            if constexpr (B == 4) {
                t = wr_t - (uint32_t)(16 * (tp ^ swz(tr))) + (uint32_t)(16 * (min(tp, 1) ^ swz(tr)));
            } else if constexpr (B == 3) {
                t = wr_t - 16u * (uint32_t)tp;
            } else {
                if (off_t + (uint32_t)step * (16 * TP) >= 8u) tv = u32x4_t{tv[2], tv[3], tv[2], tv[3]};
            }
        }
        lds_st128(c, r.c);
        lds_st128(t, tv);
    }
    __device__ __forceinline__ void read(Step& s) const {
        if constexpr (B == 4) {
            const u32x4_t v = lds_ld128(rd_c), t0 = lds_ld128(rd_t[0]), t1 = lds_ld128(rd_t[1]);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                s.c[i] = v[i];
                s.t[i] = t0[i];
                s.t[4 + i] = t1[i];
            }
        } else {
#pragma unroll
            for (int i = 0; i < B; ++i) s.c[i] = lds_ld32(rd_c + 4 * i);
#pragma unroll
            for (int i = 0; i < kTab; ++i) s.t[i] = lds_ld32(rd_t[0] + 4 * i);
        }
    }
    // code dword of the lane's 8 columns j; kBl4: in column order as stored
    template <bool kBl4>
    static __device__ __forceinline__ uint32_t code(const Step& s, int j) {
        if constexpr (kBl4) return s.c[j];
        else return nested_code8<B>(s.c[0], s.c[1], B >= 3 ? s.c[B >= 3 ? 2 : 0] : 0u, B >= 4 ? s.c[B >= 4 ? 3 : 0] : 0u, j);
    }
};

// REF: 32 code bytes of its row a lane and step, straight to the lane that looks
// them up (a row's step is a whole cache line; through the slot was no faster,
// and slower where the codebook's lookups already fill the LDS).
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
    __shared__ __attribute__((aligned(16))) uint8_t s_w[kRef ? 16 : kWaves * kSlotB];
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
    // first output of the wave, and the weight row of its row i
    const int o0 = (int)blockIdx.x * (kGateUp ? 64 : 128) + wv * (kGateUp ? 8 : 16);
    auto row = [&](int i) __attribute__((always_inline)) {
        return (uint32_t)min(!kGateUp ? o0 + i : i < 8 ? o0 + i : I + o0 + i - 8, M - 1);
    };
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
    // Steps are counted from st0; the last one may have 64 columns.
    auto is_tail = [&](int s) __attribute__((always_inline)) { return half_tail && st0 + s == nst_all - 1; };
    // BL4 / NestedLUT: load(buffer, step) three steps ahead,
    // store(buffer, step) to the wave's slot one step ahead (behind the reads of
    // the step before, which the LDS serves in order), use(step, stored).  Every load
    // is unconditional (past the end: the last step again), so that the compiler's
    // wait counts keep them in flight, and the code is one round of 4 steps (the
    // first pass through it waits for its instructions).
    auto k_loop_staged = [&](auto* buf, auto load, auto store, auto use) __attribute__((always_inline)) {
        auto load_step = [&](int b, int s) __attribute__((always_inline)) {
            const int c = min(s, nst - 1);
            load(buf[b], st0 + c, is_tail(c));
            __builtin_amdgcn_sched_barrier(0);
        };
#pragma unroll
        for (int q = 0; q < 3; ++q) load_step(q, q);
        for (int c0 = 0; c0 < nst; c0 += KS) {
            if (c0) lds_barrier();   // every wave is done with the columns in LDS
            stage(c0);
            lds_barrier();
            if (c0 == 0) store(buf[0], st0, is_tail(0));
            const int c1 = min(c0 + KS, nst);
            for (int s0 = c0; s0 < c1; s0 += 4) {
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int s = s0 + u;
                    load_step((u + 3) & 3, s + 3);
                    if (s < c1) {
                        use(s, is_tail(s), [&]() __attribute__((always_inline)) {
                            const int c = min(s + 1, nst - 1);
                            store(buf[(u + 1) & 3], st0 + c, is_tail(c));
                        });
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            }
        }
    };
    // REF: steps in pairs, the next pair's loads issued before a pair is used.  The
    // loop over pairs that have a next pair has no condition around its loads or
    // its uses.  (The loop above measured 3-6 % more here.)
    auto k_loop_pairs = [&](auto* buf, auto load, auto use) __attribute__((always_inline)) {
        auto load_pair = [&](int b, int s) __attribute__((always_inline)) {
            const int a0 = st0 + min(s, nst - 1), a1 = st0 + min(s + 1, nst - 1);
            load(buf[b], a0, is_tail(a0 - st0));
            load(buf[b + 1], a1, is_tail(a1 - st0));
            __builtin_amdgcn_sched_barrier(0);
        };
        auto use_step = [&](int b, int s, bool tail) __attribute__((always_inline)) {
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
                    use_step(u, s0 + u, is_tail(s0 + u));
                }
            }
        }
    };
    const uint32_t slot = lds_addr(s_w) + (uint32_t)(wv * kSlotB);
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
        const uint32_t cbase = lds_addr(s_cb) + 4u * (uint32_t)(lane & 31), r = row(ln);
        const bf16x8_t zero = __builtin_bit_cast(bf16x8_t, u32x4_t{0u, 0u, 0u, 0u});
        RefStep buf[4];
        k_loop_pairs(buf,
               [&](RefStep& b, int step, bool tail) __attribute__((always_inline)) {
                   b.load(codes, am, r * (uint32_t)K, r * (uint32_t)(K / 32), q32, nb, step, tail ? g & 1 : g);
               },
               [&](RefStep& b, int s, bool tail) __attribute__((always_inline)) {
                   b.arrive();
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
            using Wt = Weights<B>;
            Wt W;
            W.init(lane, K, slot, row);
            typename Wt::Raw buf[4];
            k_loop_staged(buf, [&](typename Wt::Raw& b, int step, bool tail) __attribute__((always_inline)) { W.load(b, codes, tabs, step, tail); },
                   [&](typename Wt::Raw& b, int step, bool tail) __attribute__((always_inline)) {
                       W.arrive(b);
                       W.store(b, step, tail);
                   },
                   [&](int s, bool tail, auto next) __attribute__((always_inline)) {
                       typename Wt::Step st;
                       W.read(st);
                       next();
                       uint32_t lo[(1 << B) / 4], hi[(1 << B) / 4];
                       table_planes<B>(st.t, lo, hi);
                       if (tail) {   // lanes past K hold other tables: zero weights
                           rare_branch();
#pragma unroll
                           for (int i = 0; i < (1 << B) / 4; ++i) {
                               lo[i] = g >= 2 ? 0u : lo[i];
                               hi[i] = g >= 2 ? 0u : hi[i];
                           }
                       }
#pragma unroll
                       for (int j = 0; j < 4; ++j)
                           mma(s, j, __builtin_bit_cast(bf16x8_t, regtab_lookup8_eo<B, true>(lo, hi, Wt::template code<!kNested>(st, j))));
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
