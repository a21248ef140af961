// Dense bf16 shared expert of the MoE layer (gfx950).
//
// The reference keeps a model's shared experts unquantised: DeepseekV2MoE_LUT
// holds them as bf16 ColumnParallelLinear / RowParallelLinear layers and adds
// their output to the routed experts' (vllm_lut/moe_layer.py:186-200,
// 348-353); the HF blocks use dense DeepseekV2MLP / Qwen2MoeMLP
// (customized/deepseek.py:52-58, 111-115; customized/qwen.py:40-43, 96-100).
// Here that MLP runs beside the LUT experts on the same activations:
//   act_s[t] = bf16(silu(x[t] . Wg^T) * (x[t] . Wu^T))     W13s = [Wg; Wu] bf16 [2 Is][H]
//   y_s[t]   = w[t] * (act_s[t] . W2s^T)                    W2s bf16 [H][Is], fp32
// with w[t] = 1, or sigmoid(x[t] . shared_gate) (Qwen's shared_expert_gate),
// and y_s is added to each token's sum of routed experts by the kernel that
// writes the layer's output, before its one rounding.
//
// Three kernels, by the number of tokens T (the weights, 6 H Is bytes, are read
// once in each; 46 + 23 MB at H = 2048, Is = 5632):
//   T <= 4   dense_gemv_kernel: a wave owns 4 weight rows, v_dot2_f32_bf16.
//   T <= 32  dense_skinny_kernel: HBM-bound MFMA; a CTA owns 16 rows of the
//            output, its 8 waves split K, operands straight to registers.
//   else     dense_tile_kernel: MFMA tiles fed by LDS DMA; the down projection
//            split over K where its tiles would leave CUs idle.
// The token weights come from extra CTAs of the gate/up launch.
#include "common.h"
#include "kernels.h"
#include "lut_core.h"

using namespace lutmoe;

namespace {

constexpr int kDStep = 512;     // columns per lane step (64 lanes x 8)
constexpr int kDSteps = 4;      // steps in flight per row

// w[t] = sigmoid(x[t] . g) (fp32 sum of bf16 products), or 1 without a gate, by
// the calling wave.
struct TokenWeights {
    const uint16_t* g;   // NULL: 1
    float* w;            // NULL: none to compute
};
__device__ __forceinline__ void token_weight(const TokenWeights& tw, const uint16_t* x, int t, int H) {
    const float v = tw.g ? shared_gate_weight(x + (int64_t)t * H, tw.g, H) : 1.0f;
    if ((threadIdx.x & 63) == 0) tw.w[t] = v;
}

// TB tokens a pass.  kSwiGLU: W = W13s [2I][K], out = act_s bf16 [T][I];
// else W = W2s [M][K], out = y_s fp32 [T][M] times tokw[t].
template <int TB, bool kSwiGLU>
__global__ __launch_bounds__(256, 2) void dense_gemv_kernel(const uint16_t* __restrict__ W, int M, int K, int I,
                                                            const uint16_t* __restrict__ x, int T,
                                                            const float* __restrict__ tokw, void* __restrict__ out,
                                                            TokenWeights tw) {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int unit = blockIdx.x * 4 + wv;
    if (kSwiGLU && tw.w && blockIdx.x == gridDim.x - 1) {   // the last CTA: the token weights
        for (int t = wv; t < T; t += 4) token_weight(tw, x, t, K);
        return;
    }
    int rows[4];
    if constexpr (kSwiGLU) {
        const int i0 = 2 * unit;
        if (i0 >= I) return;
        rows[0] = i0;
        rows[1] = i0 + 1;
        rows[2] = I + i0;
        rows[3] = I + i0 + 1;
    } else {
        const int r0 = 4 * unit;
        if (r0 >= M) return;
#pragma unroll
        for (int r = 0; r < 4; ++r) rows[r] = min(r0 + r, M - 1);
    }
    const int nstep = (K + kDStep - 1) / kDStep;
    for (int t0 = 0; t0 < T; t0 += TB) {
        const int nt = min(TB, T - t0);
        float acc[4][TB];
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int t = 0; t < TB; ++t) acc[r][t] = 0.f;
        for (int s0 = 0; s0 < nstep; s0 += kDSteps) {
            // every load of kDSteps steps issued before any is used (columns
            // past K: the row's last 8 columns, their activations zeroed)
            u32x4_t wr[kDSteps][4], xr[kDSteps][TB];
#pragma unroll
            for (int s = 0; s < kDSteps; ++s) {
                const int col = min((s0 + s) * kDStep + 8 * lane, K - 8);
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    wr[s][r] = *reinterpret_cast<const u32x4_t*>(W + (int64_t)rows[r] * K + col);
#pragma unroll
                for (int t = 0; t < TB; ++t)
                    xr[s][t] = *reinterpret_cast<const u32x4_t*>(x + (int64_t)(t0 + min(t, nt - 1)) * K + col);
            }
#pragma unroll
            for (int s = 0; s < kDSteps; ++s) {
                const bool ok = (s0 + s) * kDStep + 8 * lane < K;
#pragma unroll
                for (int t = 0; t < TB; ++t) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const uint32_t xv = ok ? xr[s][t][j] : 0u;
#pragma unroll
                        for (int r = 0; r < 4; ++r) acc[r][t] = dot2_bf16(wr[s][r][j], xv, acc[r][t]);
                    }
                }
            }
        }
#pragma unroll
        for (int t = 0; t < TB; ++t) {
            if (t >= nt) break;
            const float v = wave_reduce4(acc[0][t], acc[1][t], acc[2][t], acc[3][t]);   // lane 16r: row r
            if constexpr (kSwiGLU) {
                const float u = from_upper_half(v);   // lanes 0 / 16: up rows 2 / 3
                if (lane == 0 || lane == 16)
                    ((uint16_t*)out)[(int64_t)(t0 + t) * I + rows[lane >> 4]] = (uint16_t)f32_to_bf16(silu_mul(v, u));
            } else {
                const int r = lane >> 4;
                if ((lane & 15) == 0 && 4 * unit + r < M)
                    ((float*)out)[(int64_t)(t0 + t) * M + 4 * unit + r] = v * tokw[t0 + t];
            }
        }
    }
}

// ------------------------------------------------- 5 to 32 tokens: MFMA, K split
// CTA = 16 output columns (gate/up: 16 gate and 16 up rows; down: 16 rows),
// all tokens in NMT tiles of 16.  Wave w takes the 64-column K steps w, w + 8,
// ..: lane (n = l % 16, g = l / 16) holds columns 16g .. 16g + 15 of row n in
// both operands (a permutation of k common to the two: each 128-byte line of a
// row is read whole), two 16x16x32 MFMAs per row tile, token tile and step.
// The waves' partial sums meet in LDS and are added in wave order.  H = 2048,
// Is = 5632, gate/up + down with the layer's other launches (7-10 us; in brackets
// the 4-token GEMV passes, which read the weights ceil(T / 4) times): T = 5 / 16 /
// 32 30.5 / 36.7 / 44.9 us (49.9 / 86.2 / 148.4).
// The line to the GEMV, us with it / here: at two tokens the GEMV is ahead (H = 2048,
// Is = 5632 22.8 / 25.9, 4096 x 512 12.5 / 17.7); at three and four neither is
// everywhere (four tokens: 2048 x 5632 33.5 / 30.7, 4096 x 14336 100 / 84, 512 x 256
// 16.4 / 14.2, but 2048 x 1408 18.4 / 19.1, 4096 x 512 19.4 / 21.9), and they stay
// with it; at five it would take two passes.
constexpr int kSkWaves = 8;
constexpr int kSkUnroll = 4;   // K steps in flight per wave

template <bool kGateUp, int NMT>
__global__ __launch_bounds__(64 * kSkWaves) void dense_skinny_kernel(const uint16_t* __restrict__ W,
                                                                     const uint16_t* __restrict__ src, int T, int H,
                                                                     int I, const float* __restrict__ tokw,
                                                                     void* __restrict__ dst, TokenWeights tw) {
    constexpr int NR = kGateUp ? 2 : 1;   // row tiles
    __shared__ f32x4_t s_p[kSkWaves][NR * NMT][64];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int K = kGateUp ? H : I;
    if (kGateUp && tw.w && blockIdx.x == gridDim.x - 1) {
        for (int t = wv; t < T; t += kSkWaves) token_weight(tw, src, t, H);
        return;
    }
    const int n0 = blockIdx.x * 16, n = lane & 15, g = lane >> 4;
    const uint16_t* wp[NR];
    const uint16_t* xp[NMT];
#pragma unroll
    for (int r = 0; r < NR; ++r) wp[r] = W + (int64_t)(n0 + n + (r ? I : 0)) * K + 16 * g;
#pragma unroll
    for (int m = 0; m < NMT; ++m) xp[m] = src + (int64_t)min(16 * m + n, T - 1) * K + 16 * g;
    f32x4_t acc[NR][NMT];
#pragma unroll
    for (int r = 0; r < NR; ++r)
#pragma unroll
        for (int m = 0; m < NMT; ++m) acc[r][m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    const int nkb = K / 64;
    for (int k0 = wv; k0 < nkb; k0 += kSkWaves * kSkUnroll) {
        bf16x8_t wf[kSkUnroll][NR][2], xf[kSkUnroll][NMT][2];
#pragma unroll
        for (int u = 0; u < kSkUnroll; ++u) {
            const int64_t c = 64 * (int64_t)min(k0 + kSkWaves * u, nkb - 1);   // past K: loaded, not used
#pragma unroll
            for (int r = 0; r < NR; ++r) {
                wf[u][r][0] = *reinterpret_cast<const bf16x8_t*>(wp[r] + c);
                wf[u][r][1] = *reinterpret_cast<const bf16x8_t*>(wp[r] + c + 8);
            }
#pragma unroll
            for (int m = 0; m < NMT; ++m) {
                xf[u][m][0] = *reinterpret_cast<const bf16x8_t*>(xp[m] + c);
                xf[u][m][1] = *reinterpret_cast<const bf16x8_t*>(xp[m] + c + 8);
            }
        }
        __builtin_amdgcn_sched_barrier(0);   // every load of the round before its MFMAs
#pragma unroll
        for (int u = 0; u < kSkUnroll; ++u) {
            if (k0 + kSkWaves * u >= nkb) break;
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int r = 0; r < NR; ++r)
#pragma unroll
                    for (int m = 0; m < NMT; ++m)
                        acc[r][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[u][r][j], xf[u][m][j], acc[r][m], 0, 0, 0);
        }
    }
#pragma unroll
    for (int r = 0; r < NR; ++r)
#pragma unroll
        for (int m = 0; m < NMT; ++m) s_p[wv][r * NMT + m][lane] = acc[r][m];
    __syncthreads();
    if (wv >= NMT) return;
    // wave m: token tile m.  D: lane (token = l % 16, g), element i -> row 4g + i
    f32x4_t sum[NR];
#pragma unroll
    for (int r = 0; r < NR; ++r) {
        sum[r] = s_p[0][r * NMT + wv][lane];
#pragma unroll
        for (int w = 1; w < kSkWaves; ++w) sum[r] += s_p[w][r * NMT + wv][lane];
    }
    const int t = 16 * wv + n;
    if (t >= T) return;
    if constexpr (kGateUp) {
        float a[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) a[i] = silu_mul(sum[0][i], sum[NR - 1][i]);
        *reinterpret_cast<u32x2_t*>((uint16_t*)dst + (int64_t)t * I + n0 + 4 * g) =
            u32x2_t{f32x2_to_bf16x2(a[0], a[1]), f32x2_to_bf16x2(a[2], a[3])};
    } else {
        const float w = tokw[t];
        f32x4_t v;
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = sum[0][i] * w;
        *reinterpret_cast<f32x4_t*>((float*)dst + (int64_t)t * H + n0 + 4 * g) = v;
    }
}

// ------------------------------------------------------- more tokens: MFMA tiles
// CTA (tile, K split z): BM = 64 NMW tokens x 128 weight rows (gate/up: 64
// intermediate indices, gate and up rows), 4 waves in 2 x 2,
// a wave NMW m-tiles of 32 tokens x 2 n-tiles of 32 rows.  K steps of 64
// columns go global -> LDS by 16-byte DMA through a ring of S stages (16-byte
// chunk c of row r at chunk c ^ swz(r)); a step's fragments are read one
// k-substep ahead of their MFMAs, the next step's first ones right after the
// barrier that lands its stage.
//
// Each eighth of the tiles runs on one XCD (a CTA's index modulo 8), row block by
// row block over a group of token blocks: the 32 tiles on its CUs at a time are
// about as many rows of weights as of tokens, which share its L2.  (All 16 or 32
// token blocks of a row block at once read a long batch's activations again for
// every two row blocks, or every one; against that H = 2048, Is = 5632, T = 4096 /
// 8192 360 / 781 -> 348 / 675 us, H = 4096 697 / 1489 -> 676 / 1305.)
//
// A tile's rate is set by how many CUs have one and by the bytes it pulls (50 to
// 60 GB/s a CU with all of them streaming), so few tokens take small tiles and the
// down projection (H / 128 row blocks, K = Is) is split over K: its partial
// rows are added by the kernel that writes the layer's output.  T = 333,
// H = 2048, Is = 5632 (the tile it replaces: 256 x 256, weights loaded per lane,
// no split), with the layer's other launches: 295 -> 84 us; T = 2048 385 -> 231.
constexpr int kDBN = 128;
constexpr int kDBK = 64;

__device__ __forceinline__ int d_swz(int r) { return ((r >> 1) ^ (r << 2)) & 7; }

// 16 bytes a lane from sbase + voff into LDS at m0 + 16 * lane; the load reads
// sbase as an SGPR pair and carries the 5 wait states a VALU write of it needs.
__device__ __forceinline__ void d_dma16(uint32_t voff, const void* sbase, uint32_t m0) {
    asm volatile("s_nop 4\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(voff), "s"(sbase), "{m0}"(m0) : "memory");
}
template <int kAfter>
__device__ __forceinline__ void d_wait_barrier() {
    static_assert(kAfter >= 0 && kAfter <= 63, "vmcnt range");
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kAfter) : "memory");
}

template <int NMW>
struct DTile {
    static constexpr int kBM = 64 * NMW;
    static constexpr int kStage = (kBM + kDBN) * kDBK * 2;
    static constexpr int kStages = NMW == 1 ? 6 : NMW == 2 ? 4 : 3;
    static constexpr int kLoads = (kBM + kDBN) / 32;   // DMAs per thread per stage
};

template <bool kGateUp, int NMW, bool kGroups>
__global__ __launch_bounds__(256, 1) void dense_tile_kernel(const uint16_t* __restrict__ W,
                                                            const uint16_t* __restrict__ src, int T, int H, int I,
                                                            const float* __restrict__ tokw, void* __restrict__ dst,
                                                            int nxb, int group, int64_t split_stride, TokenWeights tw) {
    using D = DTile<NMW>;
    constexpr int S = D::kStages, L = D::kLoads, kBM = D::kBM;
    __shared__ __attribute__((aligned(16))) uint8_t ring[S * D::kStage];
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int K = kGateUp ? H : I;
    const int nyb = (T + kBM - 1) / kBM, per = (nxb * nyb + 7) / 8;   // tiles per XCD
    if (kGateUp && (int)blockIdx.x >= 8 * per) {   // CTA past the tiles: 16 token weights
        for (int j = 0; j < 4; ++j) {
            const int t = 16 * ((int)blockIdx.x - 8 * per) + 4 * wv + j;
            if (t < T) token_weight(tw, src, t, H);
        }
        return;
    }
    const int tile = ((int)blockIdx.x & 7) * per + ((int)blockIdx.x >> 3);
    if (tile >= nxb * nyb) return;
    int y0 = 0, gy = nyb, in = tile;   // the group's first token block, their number, the tile in it
    if constexpr (kGroups) {
        y0 = tile / (group * nxb) * group;
        gy = min(group, nyb - y0);
        in -= y0 * nxb;
    }
    const int bx = in / gy, m0 = (y0 + in - bx * gy) * kBM;
    const int nk = K / kDBK, kb0 = nk * (int)blockIdx.z / (int)gridDim.z;
    const int nkb = nk * ((int)blockIdx.z + 1) / (int)gridDim.z - kb0;
    const int n0 = bx * (kGateUp ? kDBN / 2 : kDBN);
    const int nvalid = min(kBM, T - m0);

    // ---- loader: wave w, load j covers stage rows 8 (L w + j) .. +7 (tokens,
    // then weight rows); lane l the (l % 8 ^ swz)-th 16 bytes of row + l / 8.
    // Rows past the last token / weight row repeat it (their results are dropped)
    const uint8_t* a_base = (const uint8_t*)(src + (int64_t)m0 * K + kb0 * kDBK);
    const uint8_t* w_base = (const uint8_t*)(W + kb0 * kDBK);
    uint32_t off[L];
    bool is_w[L];
#pragma unroll
    for (int j = 0; j < L; ++j) {
        const int q = 8 * (L * wv + j), r = q + (lane >> 3);
        is_w[j] = q >= kBM;   // wave-uniform
        uint32_t row;
        if (!is_w[j]) {
            row = (uint32_t)min(r, nvalid - 1);
        } else if (kGateUp) {   // weight rows 0 .. 63 of the block: gate, 64 .. 127: up
            const int b = r - kBM, i = min(n0 + (b & 63), I - 1);
            row = (uint32_t)(b < 64 ? i : I + i);
        } else {
            row = (uint32_t)min(n0 + r - kBM, H - 1);
        }
        off[j] = 2u * (row * (uint32_t)K + 8u * (uint32_t)((lane & 7) ^ d_swz(r)));
    }
    const uint32_t l_ring = lds_addr(ring);
    auto issue = [&](int kb, int slot) __attribute__((always_inline)) {
        const uint32_t l0 = l_ring + (uint32_t)slot * D::kStage + (uint32_t)(L * wv) * 1024u;
#pragma unroll
        for (int j = 0; j < L; ++j)
            d_dma16(off[j], (is_w[j] ? w_base : a_base) + (int64_t)kb * (kDBK * 2), l0 + 1024u * j);
    };

    // ---- compute side: wave (wm, wn); lane (n = l % 32, h = l / 32)
    const int wm = wv & 1, wn = wv >> 1, bn = lane & 31, bh = lane >> 5;
    const int a_row = wm * 32 * NMW + bn;
    int w_row[2];   // stage rows of the n-tiles (gate/up: gate, up)
    w_row[0] = kBM + (kGateUp ? 32 * wn : 64 * wn) + bn;
    w_row[1] = w_row[0] + (kGateUp ? 64 : 32);
    f32x16_t acc[NMW][2];
#pragma unroll
    for (int m = 0; m < NMW; ++m)
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[m][q][i] = 0.f;
    auto frags = [&](int slot, int ks, bf16x8_t (&af)[NMW], bf16x8_t (&wf)[2]) __attribute__((always_inline)) {
        const uint8_t* st = ring + slot * D::kStage;
        const int c = 4 * bh + ks;
#pragma unroll
        for (int m = 0; m < NMW; ++m) {
            const int r = a_row + 32 * m;
            af[m] = *reinterpret_cast<const bf16x8_t*>(st + r * 128 + 16 * (c ^ d_swz(r)));
        }
#pragma unroll
        for (int q = 0; q < 2; ++q)
            wf[q] = *reinterpret_cast<const bf16x8_t*>(st + w_row[q] * 128 + 16 * (c ^ d_swz(w_row[q])));
    };
    // at most `after` stages issued later than the one needed may be in flight
    auto wait_stage = [&](int after) __attribute__((always_inline)) {
        if (S >= 6 && after >= 4) d_wait_barrier<(S >= 6 ? 4 : 0) * L>();
        else if (S >= 5 && after >= 3) d_wait_barrier<(S >= 5 ? 3 : 0) * L>();
        else if (S >= 4 && after >= 2) d_wait_barrier<(S >= 4 ? 2 : 0) * L>();
        else if (after >= 1) d_wait_barrier<L>();
        else d_wait_barrier<0>();
    };
    const int first = min(S, nkb);
    for (int k = 0; k < first; ++k) issue(k, k);
    // stage 0 landed (the S - 1 others may be in flight)
    if (first == S) d_wait_barrier<(S - 1) * L>();
    else d_wait_barrier<0>();
    bf16x8_t af[NMW], wf[2];
    frags(0, 0, af, wf);
    int slot = 0;
    for (int kb = 0; kb < nkb; ++kb) {
        const int nslot = slot == S - 1 ? 0 : slot + 1;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            bf16x8_t af_n[NMW], wf_n[2];
            if (ks < 3) {
                frags(slot, ks + 1, af_n, wf_n);
            } else if (kb + 1 < nkb) {
                // this slot's reads are done, stage kb + 1 has landed: refill
                wait_stage(min(S - 2, nkb - 2 - kb));
                if (kb + S < nkb) issue(kb + S, slot);
                frags(nslot, 0, af_n, wf_n);
            }
#pragma unroll
            for (int m = 0; m < NMW; ++m)
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    // gate/up: weights as the A operand (a lane holds runs of 4
                    // output columns of one token: 8-byte stores)
                    if constexpr (kGateUp)
                        acc[m][q] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[q], af[m], acc[m][q], 0, 0, 0);
                    else
                        acc[m][q] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[m], wf[q], acc[m][q], 0, 0, 0);
                }
            if (ks < 3 || kb + 1 < nkb) {
#pragma unroll
                for (int m = 0; m < NMW; ++m) af[m] = af_n[m];
                wf[0] = wf_n[0];
                wf[1] = wf_n[1];
            }
        }
        slot = nslot;
    }
    // ---- epilogue.  D: lane (n, h), element i -> row 8 (i / 4) + 4h + (i % 4)
    // of the A operand, column n of the B operand.
    if constexpr (kGateUp) {
        const int i0 = n0 + 32 * wn;
        if (i0 < I) {
#pragma unroll
            for (int m = 0; m < NMW; ++m) {
                const int r = a_row + 32 * m;
                if (r >= nvalid) continue;
                uint16_t* o = (uint16_t*)dst + (int64_t)(m0 + r) * I + i0 + 4 * bh;
#pragma unroll
                for (int gq = 0; gq < 4; ++gq) {
                    float a[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) a[i] = silu_mul(acc[m][0][4 * gq + i], acc[m][1][4 * gq + i]);
                    *reinterpret_cast<u32x2_t*>(o + 8 * gq) =
                        u32x2_t{f32x2_to_bf16x2(a[0], a[1]), f32x2_to_bf16x2(a[2], a[3])};
                }
            }
        }
    } else {
        float* y = (float*)dst + blockIdx.z * split_stride;
#pragma unroll
        for (int m = 0; m < NMW; ++m)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int r = wm * 32 * NMW + 32 * m + 8 * (i >> 2) + 4 * bh + (i & 3);
                if (r >= nvalid) continue;
                const float w = tokw[m0 + r];
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    const int h = n0 + 64 * wn + 32 * q + bn;
                    if (h < H) y[(int64_t)(m0 + r) * H + h] = acc[m][q][i] * w;
                }
            }
    }
}

constexpr int kSkMaxT = 32;

inline int dense_row_blocks(bool gate_up, int H, int I) {
    return gate_up ? (I + kDBN / 2 - 1) / (kDBN / 2) : (H + kDBN - 1) / kDBN;
}

// Tile height (m-tiles a wave) and K splits (at most max_split, of at least 4
// K steps each) of the tile kernel: the least number of rounds over the CUs
// times a tile's time.  Per K step a 64 / 128 / 256-token tile takes about
// 0.7 : 1 : 1.7 (it pulls 24 / 32 / 48 KB): gate/up at H = 2048, one round over
// the CUs, takes 12.5 / 19 / 32 us; the splits fill the last round.
struct DenseTiles {
    int nmw, ns;
};
inline DenseTiles dense_tiles(bool gate_up, int T, int H, int I, int max_split) {
    if (T <= kSkMaxT) return DenseTiles{0, 1};   // (dense_skinny_kernel)
    const int nxb = dense_row_blocks(gate_up, H, I), nk = (gate_up ? H : I) / kDBK;
    const int cu = lutmoe_host::cu_count(), ncu = cu > 0 ? cu : 256;
    DenseTiles best{1, 1};
    float best_cost = 0.f;
    for (int nmw = 1; nmw <= 4; nmw *= 2) {
        const int tiles = nxb * ((T + 64 * nmw - 1) / (64 * nmw));
        int ns = ncu / tiles;
        if (ns > nk / 4) ns = nk / 4;
        if (ns > max_split) ns = max_split;
        if (ns < 1) ns = 1;
        const float cost = (nmw == 1 ? 0.7f : nmw == 2 ? 1.f : 1.7f) * (float)((tiles * ns + ncu - 1) / ncu) / ns;
        if (best_cost == 0.f || cost < best_cost) {
            best = DenseTiles{nmw, ns};
            best_cost = cost;
        }
    }
    return best;
}

template <bool kSwiGLU>
int dense_gemv_launch(const uint16_t* W, int M, int K, int I, const uint16_t* x, int T, const float* tokw,
                      void* out, const TokenWeights& tw, hipStream_t s) {
    const int units = kSwiGLU ? (I + 1) / 2 : (M + 3) / 4;
    const dim3 grid((units + 3) / 4 + (kSwiGLU ? 1 : 0));
    if (T <= 1)
        hipLaunchKernelGGL((dense_gemv_kernel<1, kSwiGLU>), grid, dim3(256), 0, s, W, M, K, I, x, T, tokw, out, tw);
    else if (T == 2)
        hipLaunchKernelGGL((dense_gemv_kernel<2, kSwiGLU>), grid, dim3(256), 0, s, W, M, K, I, x, T, tokw, out, tw);
    else
        hipLaunchKernelGGL((dense_gemv_kernel<4, kSwiGLU>), grid, dim3(256), 0, s, W, M, K, I, x, T, tokw, out, tw);
    return lutmoe_host::check_launch();
}

template <bool kGateUp>
int dense_mfma_launch(const uint16_t* W, const uint16_t* src, int T, int H, int I, const float* tokw, void* dst,
                      const DenseTiles& tiles, const TokenWeights& tw, hipStream_t s) {
    if (!tiles.nmw) {
        const dim3 grid((kGateUp ? I : H) / 16 + (kGateUp ? 1 : 0)), block(64 * kSkWaves);
        if (T <= 16)
            hipLaunchKernelGGL((dense_skinny_kernel<kGateUp, 1>), grid, block, 0, s, W, src, T, H, I, tokw, dst, tw);
        else
            hipLaunchKernelGGL((dense_skinny_kernel<kGateUp, 2>), grid, block, 0, s, W, src, T, H, I, tokw, dst, tw);
        return lutmoe_host::check_launch();
    }
    const int nxb = dense_row_blocks(kGateUp, H, I);
    const int64_t stride = (int64_t)T * H;
    // groups of at least 4 blocks of 256 tokens and less than 8 (the smaller tiles have
    // few blocks; a kernel that finds its group takes 0.15 us longer, 2.5 at 333 tokens)
    const int nyb = (T + 64 * tiles.nmw - 1) / (64 * tiles.nmw), ng = tiles.nmw < 4 || nyb < 8 ? 1 : nyb / 4;
    const int group = (nyb + ng - 1) / ng;
    const dim3 grid(8 * ((nxb * nyb + 7) / 8 + (kGateUp ? (T + 127) / 128 : 0)), 1, tiles.ns);
#define LUTMOE_DENSE_TILE(NMW, GROUPS)                                                                               \
    hipLaunchKernelGGL((dense_tile_kernel<kGateUp, NMW, GROUPS>), grid, dim3(256), 0, s, W, src, T, H, I, tokw, dst, \
                       nxb, group, stride, tw)
    switch (ng > 1 ? 0 : tiles.nmw) {
        case 0: LUTMOE_DENSE_TILE(4, true); break;
        case 1: LUTMOE_DENSE_TILE(1, false); break;
        case 2: LUTMOE_DENSE_TILE(2, false); break;
        default: LUTMOE_DENSE_TILE(4, false); break;
    }
#undef LUTMOE_DENSE_TILE
    return lutmoe_host::check_launch();
}

}  // namespace

namespace lutmoe_host {

int launch_dense_gate_up(const lutmoe_moe_desc* d, const uint16_t* x, int T, uint16_t* act, float* tokw,
                         hipStream_t s) {
    const int H = d->hidden, I = d->dense_inter;
    const uint16_t* W = (const uint16_t*)d->dense_w13;
    const TokenWeights tw{(const uint16_t*)d->shared_gate, tokw};
    if (T <= 4) return dense_gemv_launch<true>(W, 2 * I, H, I, x, T, nullptr, act, tw, s);
    return dense_mfma_launch<true>(W, x, T, H, I, nullptr, act, dense_tiles(true, T, H, I, 1), tw, s);
}

int launch_dense_down(const lutmoe_moe_desc* d, const uint16_t* act, int T, const float* tokw, float* y,
                      int max_split, int* nsplit, hipStream_t s) {
    const int H = d->hidden, I = d->dense_inter;
    const uint16_t* W = (const uint16_t*)d->dense_w2;
    *nsplit = 1;
    if (T <= 4) return dense_gemv_launch<false>(W, H, I, I, act, T, tokw, y, TokenWeights{}, s);
    const DenseTiles tiles = dense_tiles(false, T, H, I, max_split);
    *nsplit = tiles.ns;
    return dense_mfma_launch<false>(W, act, T, H, I, tokw, y, tiles, TokenWeights{}, s);
}

}  // namespace lutmoe_host
