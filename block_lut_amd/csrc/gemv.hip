// Decode-time LUT-GEMV kernels (HBM-bound).
//
// Work unit: one wavefront owns 8 weight rows ("octet") and walks K in
// chunks of 512 columns.  In a chunk, lane l = 8*g + q covers 8 consecutive
// columns 64*g + 8*q .. +7 of block g, i.e.
//   BL4: one code dword (8 nibbles) per row and one dword of the block's
//        32-byte bf16 table -- codes and tables have the same byte offset
//        (K/2 bytes per row each), so both loads are 256-byte coalesced;
//   REF: one code dwordx2 (8 bytes) per row; the 256-entry codebook is
//        staged once per CTA in LDS as fp32 and the 128-element absmax is
//        factored out per lane ((sum x*cb) * absmax).
// BL4 tables go through a per-wave LDS slot (8 rows x 256 B) so that the
// lookup is one ds_read_u16 per weight at  slot + 32*g + 2*code; the two
// looked-up bf16 values of an element pair feed one v_dot2_f32_bf16 with the
// activation pair.  Partial sums are reduced across the wave at the end.
// These serve the single-matrix entry points (lutmoe_gemv, lut_gemv and
// launch_lut_gemv_kernel); the MoE layer's decode kernels are in decode.hip.
//
// Reference behaviour restated: lut_gemv_kernel
// (vllm_lut/cuda_lut_gemv.py:23-80).
#include "common.h"
#include "kernels.h"
#include "lut_core.h"

using namespace lutmoe;

namespace {

constexpr int kChunk = 512;          // columns per wave chunk
constexpr int kRows = 8;             // rows per wave
constexpr int kSlot = kRows * 256;   // LDS bytes per wave for BL4 tables

// ------------------------------------------------------------------ decoders

struct Bl4Dec {
    const uint8_t* codes;
    const uint8_t* tabs;
    int K;
    uint32_t cw[kRows], tw[kRows];

    __device__ __forceinline__ void set_expert(const lutmoe_weights& w, int e) {
        const int64_t per = (int64_t)w.rows * (w.cols / 2);
        codes = (const uint8_t*)w.codes + e * per;
        tabs = (const uint8_t*)w.tables + e * per;
        K = w.cols;
    }
    __device__ __forceinline__ void load(const int (&rows)[kRows], int c, int lane, bool ok) {
#pragma unroll
        for (int r = 0; r < kRows; ++r) {
            const int64_t off = (int64_t)rows[r] * (K / 2) + c * 256 + 4 * lane;
            cw[r] = ok ? *reinterpret_cast<const uint32_t*>(codes + off) : 0u;
            tw[r] = ok ? *reinterpret_cast<const uint32_t*>(tabs + off) : 0u;
        }
    }
    __device__ __forceinline__ void stage(uint8_t* slot, int lane) const {
#pragma unroll
        for (int r = 0; r < kRows; ++r) *reinterpret_cast<uint32_t*>(slot + r * 256 + 4 * lane) = tw[r];
    }
    template <int TB>
    __device__ __forceinline__ void dot(int r, const uint8_t* slot, int lane, const uint4 (&xq)[TB],
                                        int nt, float (&acc)[TB]) const {
        const uint8_t* tb = slot + r * 256 + ((lane >> 3) << 5);
        const uint32_t w = cw[r];
        const uint32_t we = (w << 1) & 0x1e1e1e1eu;
        const uint32_t wo = (w >> 3) & 0x1e1e1e1eu;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t lo = *reinterpret_cast<const uint16_t*>(tb + ((we >> (8 * j)) & 0xffu));
            const uint32_t hi = *reinterpret_cast<const uint16_t*>(tb + ((wo >> (8 * j)) & 0xffu));
            const uint32_t pr = lo | (hi << 16);
#pragma unroll
            for (int t = 0; t < TB; ++t) {
                if (t < nt) {
                    const uint32_t xv = j == 0 ? xq[t].x : j == 1 ? xq[t].y : j == 2 ? xq[t].z : xq[t].w;
                    acc[t] = dot2_bf16(pr, xv, acc[t]);
                }
            }
        }
    }
    // fp32 activations: each looked-up entry widened to fp32 (exact) and
    // multiplied with its activation by an fp32 FMA
    template <int TB>
    __device__ __forceinline__ void dot_f32(int r, const uint8_t* slot, int lane, const float (&xv)[TB][8],
                                            int nt, float (&acc)[TB]) const {
        const uint8_t* tb = slot + r * 256 + ((lane >> 3) << 5);
        const uint32_t w = cw[r];
        const uint32_t we = (w << 1) & 0x1e1e1e1eu;
        const uint32_t wo = (w >> 3) & 0x1e1e1e1eu;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float lo = bf16_to_f32(*reinterpret_cast<const uint16_t*>(tb + ((we >> (8 * j)) & 0xffu)));
            const float hi = bf16_to_f32(*reinterpret_cast<const uint16_t*>(tb + ((wo >> (8 * j)) & 0xffu)));
#pragma unroll
            for (int t = 0; t < TB; ++t) {
                if (t < nt) {
                    acc[t] = fmaf(xv[t][2 * j], lo, acc[t]);
                    acc[t] = fmaf(xv[t][2 * j + 1], hi, acc[t]);
                }
            }
        }
    }
};

struct RefDec {
    const uint8_t* codes;
    const uint16_t* absmax;
    const float* s_cb;   // LDS fp32 codebook
    int K;
    int64_t nb;          // absmax entries per expert
    int bs;
    uint2 cw[kRows];
    float am[kRows];

    __device__ __forceinline__ void set_expert(const lutmoe_weights& w, int e) {
        codes = (const uint8_t*)w.codes + (int64_t)e * w.rows * w.cols;
        absmax = (const uint16_t*)w.tables + (int64_t)e * w.absmax_per_expert;
        nb = w.absmax_per_expert;
        bs = w.block_size;
        K = w.cols;
    }
    __device__ __forceinline__ void load(const int (&rows)[kRows], int c, int lane, bool ok) {
#pragma unroll
        for (int r = 0; r < kRows; ++r) {
            const int64_t flat = (int64_t)rows[r] * K + c * kChunk + 8 * lane;
            cw[r] = ok ? *reinterpret_cast<const uint2*>(codes + flat) : make_uint2(0u, 0u);
            int64_t b = flat / bs;
            b = b < nb ? b : nb - 1;
            am[r] = ok ? bf16_to_f32(absmax[b]) : 0.f;
        }
    }
    __device__ __forceinline__ void stage(uint8_t*, int) const {}
    // lut_gemv's product order (x * cb) * absmax
    template <int TB>
    __device__ __forceinline__ void dot(int r, const uint8_t*, int, const uint4 (&xq)[TB], int nt,
                                        float (&acc)[TB]) const {
        float s[TB];
#pragma unroll
        for (int t = 0; t < TB; ++t) s[t] = 0.f;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const uint32_t word = j < 4 ? cw[r].x : cw[r].y;
            const float v = s_cb[(word >> (8 * (j & 3))) & 0xffu];
#pragma unroll
            for (int t = 0; t < TB; ++t) {
                if (t < nt) {
                    const uint32_t xp = (j >> 1) == 0 ? xq[t].x : (j >> 1) == 1 ? xq[t].y
                                       : (j >> 1) == 2 ? xq[t].z : xq[t].w;
                    const float xv = (j & 1) ? __uint_as_float(xp & 0xffff0000u) : __uint_as_float(xp << 16);
                    s[t] = fmaf(xv, v, s[t]);
                }
            }
        }
#pragma unroll
        for (int t = 0; t < TB; ++t) acc[t] = fmaf(s[t], am[r], acc[t]);
    }
    // fp32 activations, lut_gemv's product order (x * cb) * absmax
    template <int TB>
    __device__ __forceinline__ void dot_f32(int r, const uint8_t*, int, const float (&xv)[TB][8], int nt,
                                            float (&acc)[TB]) const {
        float s[TB];
#pragma unroll
        for (int t = 0; t < TB; ++t) s[t] = 0.f;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const uint32_t word = j < 4 ? cw[r].x : cw[r].y;
            const float cv = s_cb[(word >> (8 * (j & 3))) & 0xffu];
#pragma unroll
            for (int t = 0; t < TB; ++t)
                if (t < nt) s[t] = fmaf(xv[t][j], cv, s[t]);
        }
#pragma unroll
        for (int t = 0; t < TB; ++t) acc[t] = fmaf(s[t], am[r], acc[t]);
    }
};

template <class Dec>
__device__ __forceinline__ void init_cb(const lutmoe_weights&, int, float*) {}
template <>
__device__ __forceinline__ void init_cb<RefDec>(const lutmoe_weights& w, int e, float* s_cb) {
    const uint16_t* cb = ref_codebook(w, e);
    for (int i = threadIdx.x; i < 256; i += blockDim.x) s_cb[i] = bf16_to_f32(cb[i]);
}

template <class Dec>
__device__ __forceinline__ void bind_cb(Dec&, const float*) {}
template <>
__device__ __forceinline__ void bind_cb<RefDec>(RefDec& d, const float* s_cb) { d.s_cb = s_cb; }

// One chunk for the wave's 8 rows: load, stage, dot.
template <class Dec, int TB>
__device__ __forceinline__ void octet_chunk(Dec& dec, const int (&rows)[kRows], int c, int nblk_k,
                                            int lane, uint8_t* slot, const uint16_t* const (&xrow)[TB],
                                            int nt, float (&acc)[kRows][TB]) {
    const bool ok = (c * 8 + (lane >> 3)) < nblk_k;
    uint4 xq[TB];
#pragma unroll
    for (int t = 0; t < TB; ++t)
        xq[t] = (ok && t < nt) ? *reinterpret_cast<const uint4*>(xrow[t] + c * kChunk + 8 * lane)
                               : make_uint4(0u, 0u, 0u, 0u);
    dec.load(rows, c, lane, ok);
    dec.stage(slot, lane);
    wave_lds_sync();
    if (ok) {
#pragma unroll
        for (int r = 0; r < kRows; ++r) dec.template dot<TB>(r, slot, lane, xq, nt, acc[r]);
    }
    wave_lds_sync();
}

// The same for fp32 activations (8 floats a lane, two 16-byte loads).
template <class Dec, int TB>
__device__ __forceinline__ void octet_chunk_f32(Dec& dec, const int (&rows)[kRows], int c, int nblk_k,
                                                int lane, uint8_t* slot, const float* const (&xrow)[TB],
                                                int nt, float (&acc)[kRows][TB]) {
    const bool ok = (c * 8 + (lane >> 3)) < nblk_k;
    float xv[TB][8];
#pragma unroll
    for (int t = 0; t < TB; ++t) {
        float4 a = make_float4(0.f, 0.f, 0.f, 0.f), b = a;
        if (ok && t < nt) {
            a = *reinterpret_cast<const float4*>(xrow[t] + c * kChunk + 8 * lane);
            b = *reinterpret_cast<const float4*>(xrow[t] + c * kChunk + 8 * lane + 4);
        }
        xv[t][0] = a.x; xv[t][1] = a.y; xv[t][2] = a.z; xv[t][3] = a.w;
        xv[t][4] = b.x; xv[t][5] = b.y; xv[t][6] = b.z; xv[t][7] = b.w;
    }
    dec.load(rows, c, lane, ok);
    dec.stage(slot, lane);
    wave_lds_sync();
    if (ok) {
#pragma unroll
        for (int r = 0; r < kRows; ++r) dec.template dot_f32<TB>(r, slot, lane, xv, nt, acc[r]);
    }
    wave_lds_sync();
}

// -------------------------------------------------------- single-matrix GEMV

// y[t][row] for one expert; CTA = 4 waves, wave w owns rows 8*(4*bx + w) ..
// kXF32: x is fp32 [T][K] (else bf16).
template <class Dec, int TB, bool kXF32>
__global__ __launch_bounds__(256) void gemv_kernel(lutmoe_weights w, int expert,
                                                   const void* __restrict__ x, int T,
                                                   void* __restrict__ y, int y_dtype) {
    __shared__ __attribute__((aligned(16))) uint8_t s_slot[4 * kSlot];
    __shared__ float s_cb[256];
    init_cb<Dec>(w, expert, s_cb);
    __syncthreads();
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int M = w.rows, K = w.cols;
    const int row0 = (blockIdx.x * 4 + wv) * kRows;
    if (row0 >= M) return;
    int rows[kRows];
#pragma unroll
    for (int r = 0; r < kRows; ++r) rows[r] = min(row0 + r, M - 1);
    Dec dec;
    bind_cb(dec, s_cb);
    dec.set_expert(w, expert);
    const int nblk_k = K / kBlockBL;
    const int nch = (K + kChunk - 1) / kChunk;
    uint8_t* slot = s_slot + wv * kSlot;
    for (int tb = 0; tb < T; tb += TB) {
        const int nt = min(TB, T - tb);
        float acc[kRows][TB];
#pragma unroll
        for (int r = 0; r < kRows; ++r)
#pragma unroll
            for (int t = 0; t < TB; ++t) acc[r][t] = 0.f;
        if constexpr (kXF32) {
            const float* xrow[TB];
#pragma unroll
            for (int t = 0; t < TB; ++t) xrow[t] = (const float*)x + (int64_t)(tb + min(t, nt - 1)) * K;
            for (int c = 0; c < nch; ++c) octet_chunk_f32<Dec, TB>(dec, rows, c, nblk_k, lane, slot, xrow, nt, acc);
        } else {
            const uint16_t* xrow[TB];
#pragma unroll
            for (int t = 0; t < TB; ++t) xrow[t] = (const uint16_t*)x + (int64_t)(tb + min(t, nt - 1)) * K;
            for (int c = 0; c < nch; ++c) octet_chunk<Dec, TB>(dec, rows, c, nblk_k, lane, slot, xrow, nt, acc);
        }
#pragma unroll
        for (int r = 0; r < kRows; ++r) {
#pragma unroll
            for (int t = 0; t < TB; ++t) {
                const float v = wave_sum(acc[r][t]);
                if (lane == 0 && t < nt && row0 + r < M) {
                    const int64_t o = (int64_t)(tb + t) * M + row0 + r;
                    if (y_dtype == LUTMOE_DTYPE_F32) ((float*)y)[o] = v;
                    else ((uint16_t*)y)[o] = (uint16_t)f32_to_bf16(v);
                }
            }
        }
    }
}

// REF GEMV on the reference's raw tensors (lut_gemv, fused_lut_gemv).  A wave
// owns R rows; lane l takes columns kC*l .. kC*l + kC-1 of every 64*kC-column
// step, its codes, absmax and activations loaded for two steps before any is
// used.  The fp32 codebook sits in the wave's own LDS (no barrier between the
// waves).  kDeq: the dequantised weight bf16(cb * absmax) times x
// (fused_lut_gemv, vllm_lut/fused_kernel.py:13-46); otherwise lut_gemv's
// (x * cb) * absmax with the absmax factored out of a lane's columns.
//
// One matrix is a few MB, so what bounds it is the latency of one round of
// loads and how many waves issue them: 2 rows a wave (1408 waves at 2816
// rows) instead of 8: 2816 x 2048, one vector, 14.0 -> 4.1 us in a graph
// (5.9 MB, 1.4 TB/s from the Infinity Cache; a launch alone is about 2).
//
// kAligned: K and block_size multiples of 16, 16-byte loads of 16 columns, one
// absmax per lane and row step.  Else any K, block_size >= 8: 8 columns,
// unaligned loads, at most one absmax block boundary inside them, the row's
// last K % 8 columns element by element.
struct RefRows {
    const uint16_t* x;
    const uint8_t* idx;
    const uint16_t* cbh;    // bf16 codebook, or
    const float* cbf;       // fp32 codebook
    const uint16_t* absmax;
    void* y;
    int M, K, T, nb, bs, bs_shift, y_dtype;   // bs_shift: log2(bs), -1 if bs is no power of two
    uint32_t at;            // weights before row 0's first in idx and in absmax's first block (M K + at < 2^32)
};

__device__ __forceinline__ uint32_t ref_block(const RefRows& a, uint32_t flat) {
    return a.bs_shift >= 0 ? flat >> a.bs_shift : flat / (uint32_t)a.bs;
}

template <int R, int TB, bool kDeq, bool kAligned>
__global__ __launch_bounds__(256) void ref_gemv_rows_kernel(RefRows a) {
    constexpr int kC = kAligned ? 16 : 8;
    constexpr int kStep = 64 * kC;
    constexpr int kCW = kC / 4, kXW = kC / 2;   // code / activation dwords
    __shared__ float s_cb[4][256];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int row0 = (blockIdx.x * 4 + wv) * R;
    if (row0 >= a.M) return;
    float cbv[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
        cbv[i] = a.cbf ? a.cbf[4 * lane + i] : bf16_to_f32(a.cbh[4 * lane + i]);
    uint32_t flat0[R];
#pragma unroll
    for (int r = 0; r < R; ++r) flat0[r] = (uint32_t)min(row0 + r, a.M - 1) * (uint32_t)a.K + a.at;
    const float* cb = s_cb[wv];
    const int nwhole = a.K / kC;   // lane pieces of kC columns
    const int nb1 = a.nb - 1;
    for (int t0 = 0; t0 < a.T; t0 += TB) {
        const int nt = min(TB, a.T - t0);
        float acc[R][TB];
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int t = 0; t < TB; ++t) acc[r][t] = 0.f;
        for (int p0 = 0; p0 < nwhole; p0 += 128) {
            uint32_t cw[2][R][kCW], xw[2][TB][kXW];
            float am[2][R], am1[2][R];
            int split[2][R];   // columns of the piece in the first absmax block
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                // past the row's last piece: that piece again, its sums dropped
                const uint32_t c = (uint32_t)min(p0 + 64 * u + lane, nwhole - 1) * kC;
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const uint32_t f = flat0[r] + c;
                    __builtin_memcpy(cw[u][r], __builtin_assume_aligned(a.idx + f, kAligned ? 16 : 1), kC);
                    const uint32_t b = ref_block(a, f);
                    am[u][r] = bf16_to_f32(a.absmax[min((int)b, nb1)]);
                    if constexpr (!kAligned) {
                        split[u][r] = (int)min((b + 1) * (uint32_t)a.bs - f, 8u);
                        am1[u][r] = bf16_to_f32(a.absmax[min((int)b + 1, nb1)]);
                    }
                }
#pragma unroll
                for (int t = 0; t < TB; ++t)
                    __builtin_memcpy(xw[u][t], __builtin_assume_aligned(a.x + (int64_t)(t0 + min(t, nt - 1)) * a.K + c,
                                                                        kAligned ? 16 : 2), 2 * kC);
            }
            if (p0 == 0 && t0 == 0) {
                *reinterpret_cast<f32x4_t*>(&s_cb[wv][4 * lane]) = f32x4_t{cbv[0], cbv[1], cbv[2], cbv[3]};
                wave_lds_sync();
            }
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const bool ok = p0 + 64 * u + lane < nwhole;
                float s[R][TB];
#pragma unroll
                for (int r = 0; r < R; ++r)
#pragma unroll
                    for (int t = 0; t < TB; ++t) s[r][t] = 0.f;
#pragma unroll
                for (int j = 0; j < kC; ++j) {
                    float xv[TB];
#pragma unroll
                    for (int t = 0; t < TB; ++t) {
                        const uint32_t xp = xw[u][t][j >> 1];
                        xv[t] = (j & 1) ? __uint_as_float(xp & 0xffff0000u) : __uint_as_float(xp << 16);
                    }
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        float v = cb[(cw[u][r][j >> 2] >> (8 * (j & 3))) & 0xffu];
                        if constexpr (!kAligned) v *= j < split[u][r] ? am[u][r] : am1[u][r];
                        else if constexpr (kDeq) v *= am[u][r];
                        if constexpr (kDeq) v = bf16_to_f32(f32_to_bf16(v));
#pragma unroll
                        for (int t = 0; t < TB; ++t) s[r][t] = fmaf(xv[t], v, s[r][t]);
                    }
                }
#pragma unroll
                for (int r = 0; r < R; ++r)
#pragma unroll
                    for (int t = 0; t < TB; ++t) {
                        const float v = kAligned && !kDeq ? fmaf(s[r][t], am[u][r], acc[r][t]) : acc[r][t] + s[r][t];
                        acc[r][t] = ok ? v : acc[r][t];
                    }
            }
        }
        if constexpr (!kAligned) {
            if (nwhole == 0 && t0 == 0) {
                *reinterpret_cast<f32x4_t*>(&s_cb[wv][4 * lane]) = f32x4_t{cbv[0], cbv[1], cbv[2], cbv[3]};
                wave_lds_sync();
            }
            const int c = nwhole * kC + lane;
            if (c < a.K) {
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const uint32_t f = flat0[r] + (uint32_t)c;
                    float v = cb[a.idx[f]] * bf16_to_f32(a.absmax[min((int)ref_block(a, f), nb1)]);
                    if (kDeq) v = bf16_to_f32(f32_to_bf16(v));
#pragma unroll
                    for (int t = 0; t < TB; ++t)
                        acc[r][t] = fmaf(bf16_to_f32(a.x[(int64_t)(t0 + min(t, nt - 1)) * a.K + c]), v, acc[r][t]);
                }
            }
        }
#pragma unroll
        for (int t = 0; t < TB; ++t) {
            if (t >= nt) break;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const float v = wave_reduce(acc[r][t]);
                if (lane == r && row0 + r < a.M) {
                    const int64_t o = (int64_t)(t0 + t) * a.M + row0 + r;
                    if (a.y_dtype == LUTMOE_DTYPE_F32) ((float*)a.y)[o] = v;
                    else ((uint16_t*)a.y)[o] = (uint16_t)f32_to_bf16(v);
                }
            }
        }
    }
}

// Absmax blocks of fewer than 8 elements: one wave per row, scalar lanes.
template <bool kDeq>
__global__ __launch_bounds__(256) void ref_gemv_generic_kernel(RefRows a) {
    __shared__ float s_cb[256];
    s_cb[threadIdx.x] = a.cbf ? a.cbf[threadIdx.x] : bf16_to_f32(a.cbh[threadIdx.x]);
    __syncthreads();
    const int lane = threadIdx.x & 63;
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= a.M) return;
    for (int t = 0; t < a.T; ++t) {
        float acc = 0.f;
        for (int c = lane; c < a.K; c += 64) {
            const uint32_t flat = (uint32_t)row * (uint32_t)a.K + a.at + (uint32_t)c;
            const float xv = bf16_to_f32(a.x[(int64_t)t * a.K + c]);
            const float cv = s_cb[a.idx[flat]], av = bf16_to_f32(a.absmax[min((int)ref_block(a, flat), a.nb - 1)]);
            acc += kDeq ? xv * bf16_to_f32(f32_to_bf16(cv * av)) : xv * cv * av;
        }
        acc = wave_reduce(acc);
        if (lane == 0) {
            const int64_t o = (int64_t)t * a.M + row;
            if (a.y_dtype == LUTMOE_DTYPE_F32) ((float*)a.y)[o] = acc;
            else ((uint16_t*)a.y)[o] = (uint16_t)f32_to_bf16(acc);
        }
    }
}

inline int tb_for(int T) { return T <= 1 ? 1 : T <= 2 ? 2 : 4; }

}  // namespace

namespace lutmoe_host {

template <int R, bool kDeq, bool kAligned>
static void ref_gemv_rows_launch(const RefRows& a, hipStream_t s) {
    const dim3 grid((a.M + 4 * R - 1) / (4 * R)), block(256);
    switch (tb_for(a.T)) {
        case 1: hipLaunchKernelGGL((ref_gemv_rows_kernel<R, 1, kDeq, kAligned>), grid, block, 0, s, a); break;
        case 2: hipLaunchKernelGGL((ref_gemv_rows_kernel<R, 2, kDeq, kAligned>), grid, block, 0, s, a); break;
        default: hipLaunchKernelGGL((ref_gemv_rows_kernel<R, 4, kDeq, kAligned>), grid, block, 0, s, a); break;
    }
}

template <bool kDeq>
static int ref_gemv_dispatch(const RefRows& a, hipStream_t s) {
    const bool aligned = a.K % 16 == 0 && a.bs % 16 == 0 && ((uintptr_t)a.idx + a.at) % 16 == 0 && (uintptr_t)a.x % 16 == 0;
    if (aligned) ref_gemv_rows_launch<2, kDeq, true>(a, s);
    else if (a.bs >= 8) ref_gemv_rows_launch<2, kDeq, false>(a, s);
    else hipLaunchKernelGGL(ref_gemv_generic_kernel<kDeq>, dim3((a.M + 3) / 4), dim3(256), 0, s, a);
    return check_launch();
}

int launch_ref_gemv(const uint16_t* x, const uint8_t* idx, const uint16_t* cb_bf16,
                    const float* cb_f32, const uint16_t* absmax, void* y, int M, int K, int T,
                    int num_blocks, int block_size, int y_dtype, hipStream_t s, bool dequant) {
    const int shift = (block_size & (block_size - 1)) == 0 ? __builtin_ctz((unsigned)block_size) : -1;
    RefRows a{x, idx, cb_bf16, cb_f32, absmax, y, M, K, T, num_blocks, block_size, shift, y_dtype, 0};
    // The kernels count weights in 32 bits.  A larger matrix goes in ranges of
    // rows (the entry points with several vectors take fewer than 2^31 weights)
    const int64_t most = ((int64_t)1 << 32) - 1;
    if ((int64_t)M * K <= most) return dequant ? ref_gemv_dispatch<true>(a, s) : ref_gemv_dispatch<false>(a, s);
    if (T != 1) return LUTMOE_EUNSUPPORTED;
    const int64_t rows = (most - (block_size - 1)) / K;   // at least one: K, block_size < 2^31
    for (int64_t r0 = 0; r0 < M; r0 += rows) {
        const int64_t first = r0 * K, b0 = first / block_size < num_blocks ? first / block_size : num_blocks - 1;
        a.at = (uint32_t)(first % block_size);
        a.idx = idx + first - a.at;
        a.absmax = absmax + b0;   // (past the last block: that one for every weight)
        a.nb = num_blocks - (int)b0;
        a.M = (int)(M - r0 < rows ? M - r0 : rows);
        a.y = (char*)y + r0 * (y_dtype == LUTMOE_DTYPE_F32 ? 4 : 2);
        if (const int rc = dequant ? ref_gemv_dispatch<true>(a, s) : ref_gemv_dispatch<false>(a, s)) return rc;
    }
    return LUTMOE_OK;
}

template <class Dec, bool kXF32>
static int gemv_dispatch(const lutmoe_weights* w, int expert, const void* x, int T, void* y,
                         int y_dtype, hipStream_t s) {
    const dim3 grid((w->rows + 4 * kRows - 1) / (4 * kRows));
    switch (tb_for(T)) {
        case 1: hipLaunchKernelGGL((gemv_kernel<Dec, 1, kXF32>), grid, dim3(256), 0, s, *w, expert, x, T, y, y_dtype); break;
        case 2: hipLaunchKernelGGL((gemv_kernel<Dec, 2, kXF32>), grid, dim3(256), 0, s, *w, expert, x, T, y, y_dtype); break;
        default: hipLaunchKernelGGL((gemv_kernel<Dec, 4, kXF32>), grid, dim3(256), 0, s, *w, expert, x, T, y, y_dtype); break;
    }
    return check_launch();
}

int launch_bl4_gemv(const lutmoe_weights* w, int expert, const void* x, bool x_f32, int T, void* y,
                    int y_dtype, hipStream_t s) {
    if (w->format == LUTMOE_FMT_REF)
        return x_f32 ? gemv_dispatch<RefDec, true>(w, expert, x, T, y, y_dtype, s)
                     : gemv_dispatch<RefDec, false>(w, expert, x, T, y, y_dtype, s);
    return x_f32 ? gemv_dispatch<Bl4Dec, true>(w, expert, x, T, y, y_dtype, s)
                 : gemv_dispatch<Bl4Dec, false>(w, expert, x, T, y, y_dtype, s);
}


}  // namespace lutmoe_host
