// BL4 encoder on the GPU: per-64-weight-block k-means (k = 16), one
// wavefront per block, lane j holding weight j.
//
// The procedure is LUTQuantizer._train_kmeans (vllm_lut/quantizer.py:120-178)
// applied per block: Lloyd iterations with argmin |x - c| (first minimum),
// mean update leaving empty clusters unchanged, final sort, cast to the
// storage dtype (fp16), codes re-assigned against the stored codebook
// (quantize(), quantizer.py:292-296); in the final 16-means an empty cluster
// is re-seeded at the farthest member instead of being left in place.  Initialisation is a binary-splitting
// tree (4-means from the quantile start sorted[16i+8], then every cell split
// by 2-means twice) instead of a random pick, so CPU and GPU agree exactly.
// Cluster sums are the xor-butterfly over the 64 lanes (non-members add +0)
// and every lane divides the same uniform sum by the same count, so the
// result is bit-identical to the CPU restatement run in the same order.
#include "common.h"
#include "kernels.h"
#include "lut_core.h"

using namespace lutmoe;

namespace {

__device__ __forceinline__ float butterfly(float v) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v = v + __shfl_xor(v, off, kWave);
    return v;
}

template <int K>
__device__ __forceinline__ int argmin_abs(float x, const float (&c)[K]) {
    int best = 0;
    float bd = fabsf(x - c[0]);
#pragma unroll
    for (int i = 1; i < K; ++i) {
        const float dd = fabsf(x - c[i]);
        if (dd < bd) { bd = dd; best = i; }
    }
    return best;
}

template <int K>
__device__ __forceinline__ float pick(const float (&c)[K], int i) {
    float v = c[0];
#pragma unroll
    for (int q = 1; q < K; ++q) v = (i == q) ? c[q] : v;
    return v;
}

// Lloyd on the member lanes; c[] is uniform across the wave.  kReseed: after
// each mean update every empty cluster (index order) moves to the member
// farthest from its own centroid (lowest lane on ties, each lane once per
// iteration) when that distance is > 0.
template <int K, bool kReseed = false>
__device__ void lloyd(float x, bool member, float (&c)[K], int n_iter, int& assign) {
    const int lane = threadIdx.x & 63;
    assign = -1;
    for (int it = 0; it < n_iter; ++it) {
        const int a = member ? argmin_abs<K>(x, c) : -1;
        const bool changed = member && a != assign;
        assign = a;
        if (!__any(changed)) break;
        uint32_t empty = 0;
#pragma unroll
        for (int i = 0; i < K; ++i) {
            const bool in = member && assign == i;
            const float s = butterfly(in ? x : 0.0f);
            const int cnt = __popcll(__ballot(in));
            if (cnt) c[i] = s / (float)cnt;
            else empty |= 1u << i;
        }
        if (kReseed && empty) {
            bool taken = false;
#pragma unroll
            for (int i = 0; i < K; ++i) {
                if (!((empty >> i) & 1u)) continue;
                const float d = (member && !taken) ? fabsf(x - pick(c, assign)) : -1.0f;
                const float mx = wave_reduce_max(d);
                if (!(mx > 0.0f)) break;
                const int j = (int)__builtin_ctzll(__ballot(d == mx));
                c[i] = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), j));
                if (lane == j) taken = true;
            }
        }
    }
}

template <int K>
__device__ __forceinline__ void sort_small(float (&c)[K]) {
#pragma unroll
    for (int i = 1; i < K; ++i) {
        const float v = c[i];
        int j = i - 1;
        while (j >= 0 && c[j] > v) { c[j + 1] = c[j]; --j; }
        c[j + 1] = v;
    }
}

__device__ void split2(float x, bool member, float parent, int n_iter, float (&ch)[2]) {
    const bool any = __any(member);
    if (!any) { ch[0] = ch[1] = parent; return; }
    float lo = member ? x : INFINITY, hi = member ? x : -INFINITY;
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        lo = fminf(lo, __shfl_xor(lo, off, kWave));
        hi = fmaxf(hi, __shfl_xor(hi, off, kWave));
    }
    ch[0] = lo;
    ch[1] = hi;
    int a;
    lloyd<2>(x, member, ch, n_iter, a);
    if (ch[1] < ch[0]) { const float t = ch[0]; ch[0] = ch[1]; ch[1] = t; }
}


__global__ __launch_bounds__(256) void bl4_encode_kernel(const float* __restrict__ w,
                                                         int64_t nblocks, int n_iter,
                                                         uint8_t* __restrict__ codes,
                                                         uint16_t* __restrict__ tables) {
    __shared__ float s_x[4][64];
    __shared__ float s_sorted[4][64];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    for (int64_t b = (int64_t)blockIdx.x * 4 + wv; b < nblocks; b += (int64_t)gridDim.x * 4) {
        const float x = w[b * 64 + lane];
        s_x[wv][lane] = x;
        wave_lds_sync();
        int r = 0;
        for (int i = 0; i < 64; ++i) {
            const float xi = s_x[wv][i];
            r += (xi < x) || (xi == x && i < lane);
        }
        s_sorted[wv][r] = x;
        wave_lds_sync();
        float c2[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) c2[i] = s_sorted[wv][16 * i + 8];
        wave_lds_sync();
        int a2;
        lloyd<4>(x, true, c2, n_iter, a2);
        // order level-2 cells by centroid (stable insertion order of indices)
        int order[4] = {0, 1, 2, 3};
#pragma unroll
        for (int i = 1; i < 4; ++i) {
            const int v = order[i];
            int j = i - 1;
            while (j >= 0 && pick(c2, order[j]) > pick(c2, v)) { order[j + 1] = order[j]; --j; }
            order[j + 1] = v;
        }
        float c2s[4];
        int rank = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            c2s[i] = pick(c2, order[i]);
            rank = (order[i] == a2) ? i : rank;
        }
        a2 = rank;
        float c3[8];
#pragma unroll
        for (int j2 = 0; j2 < 4; ++j2) {
            float ch[2];
            split2(x, a2 == j2, c2s[j2], n_iter, ch);
            c3[j2] = ch[0];
            c3[j2 | 4] = ch[1];
        }
        int cell3;
        {
            const float two[2] = {pick(c3, a2), pick(c3, a2 | 4)};
            cell3 = a2 | (argmin_abs<2>(x, two) << 2);
        }
        float c[16];
#pragma unroll
        for (int k3 = 0; k3 < 8; ++k3) {
            float ch[2];
            split2(x, cell3 == k3, c3[k3], n_iter, ch);
            c[k3] = ch[0];
            c[k3 | 8] = ch[1];
        }
        int a16;
        lloyd<16, true>(x, true, c, n_iter, a16);
        sort_small<16>(c);
        float cf[16];
        uint32_t h_mine = 0;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const uint32_t h = f32_to_f16(c[i]);
            cf[i] = f16_to_f32(h);
            if (lane == i) h_mine = h;
        }
        const uint32_t code = (uint32_t)argmin_abs<16>(x, cf);
        const uint32_t nb = (uint32_t)__shfl_down((int)code, 1, kWave);
        if ((lane & 1) == 0) codes[b * 32 + (lane >> 1)] = (uint8_t)(code | (nb << 4));
        if (lane < 16) tables[b * 16 + lane] = (uint16_t)h_mine;
    }
}

// ---------------------------------------------------------------------------
// REF encoders.  Three rules, one kernel:
//   kEncode (the reference's encode_blocklut_kernel, vllm_lut/fast_encode.py:
//     22-72): bf16 weights; absmax = max |w| of the block (fp32, at least
//     1e-10); v = w / absmax (IEEE fp32 division); code = the nearest of 256
//     codebook entries by |v - c| in fp32, the first one on equal distances
//     (the codebook need not be sorted).
//   kQuantizer, LUTQuantizer.quantize (vllm_lut/quantizer.py:242-306, the
//     BLOCKLUT / NESTEDLUT branch; block_size = n is its global "LUT"
//     branch): absmax = max |w| in the weights' dtype, at least 1e-10 in that
//     dtype (:282-283); v = w / absmax, rounded to bf16 for bf16 weights (torch
//     divides bf16 tensors in fp32 and rounds the result, :284); code as
//     kEncode, among ncb entries (argmin, :293-296).
//   kMidpoints, the offload runtime's encoder (runtime/model_offload.py:
//     897-907): weights as fp32; absmax at least fp32(1e-12); v = w / absmax in
//     fp32; code = the number of midpoints fl32(fl32(c_i + c_{i+1}) / 2) of the
//     ascending codebook below v (np.searchsorted, side "left": a value on a
//     midpoint takes the lower entry, NaN the last).
// absmax is stored as bf16 (round to nearest even).
//
// Comparing a weight with every entry costs 3 VALU ops per entry and weight
// (2816 x 2048 weights, 256 entries: 142 us, 0.12 TB/s, VALU-bound).  Here a
// CTA sorts the entries once (LDS), equal ones kept once, and a weight reads by
// its bucket of 1024 over the entries' range which sorted values lie in that
// bucket, searches those (none to two of a trained codebook's) and steps to its
// neighbours: about 6 LDS reads and 45 VALU ops a weight (19 us for
// the same weights).  The result is the scan's, bit for bit: rounding is monotone, so the
// entries at the least rounded distance are a run of the sorted order around v;
// the run is walked and its lowest index taken.  Where runs can be long
// (codebooks whose spacing is lost in the distances' rounding) the CTA scans
// (187 us).  Equal entries walked as runs, and a crowded bucket searched one
// value after another, took 300 to 940 us (a tier's table, padded with its last
// entry: 495, now 20).
enum EncodeRule { kEncode = 0, kQuantizer = 1, kMidpoints = 2 };

constexpr int kEncThreads = 512;
constexpr int kEncBuckets = 1024;

struct EncTable {
    float raw[256];                  // entry values, NaN past the last
    float v[258];                    // [0] NaN, then the non-NaN values ascending, then NaN
    uint8_t idx[256];                // entry of each (the lowest of equal ones)
    uint32_t bucket[kEncBuckets];    // sorted values in lower buckets, and << 16 those in this one
    uint16_t rank[256];
    int wsum[4], crowded[4];
};

// Bucket of v: monotone in v (each step is, with NaN products taken as 0).
__device__ __forceinline__ int enc_bucket(float v, float lo, float scale) {
    return (int)fminf(fmaxf((v - lo) * scale, 0.f), (float)(kEncBuckets - 1));
}

// The entries sorted by value, equal ones once if `once`; returns their number
// (every thread of the CTA calls it, s.raw complete).  ascending: they are so,
// without NaN.
__device__ int enc_sort(EncTable& s, bool ascending, bool once) {
    static_assert(kEncThreads == 512, "two threads an entry");
    const int t = threadIdx.x, e = t & 255;
    const float c = s.raw[e];
    int r = 0;
    if (ascending) {
        r = t < 256 ? e : 0;
    } else {
        // rank of entry e, each thread counting one half of the entries: of the
        // ones before it those up to its value, of the ones after it those below
        const int e0 = __builtin_amdgcn_readfirstlane(e & ~63);   // the wave's first entry
        const int j0 = __builtin_amdgcn_readfirstlane(t & 256 ? 128 : 0), j1 = j0 + 128;
        auto count = [&](int a, int b, auto less) __attribute__((always_inline)) {
#pragma unroll 1
            for (int j = max(a, j0); j < min(b, j1); j += 8) {
                const f32x4_t u = *reinterpret_cast<const f32x4_t*>(&s.raw[j]);
                const f32x4_t w = *reinterpret_cast<const f32x4_t*>(&s.raw[j + 4]);
#pragma unroll
                for (int i = 0; i < 8; ++i) r += less(i < 4 ? u[i & 3] : w[i & 3], j + i);
            }
        };
        count(0, e0, [&](float u, int) { return u <= c; });
        count(e0, e0 + 64, [&](float u, int j) { return (u < c) | ((u == c) & (j < e)); });
        count(e0 + 64, 256, [&](float u, int) { return u < c; });
    }
    if (t >= 256) s.rank[e] = (uint16_t)r;
    if (t < 258) s.v[t] = __builtin_nanf("");
    int n = __syncthreads_count(t < 256 && c == c);
    if (t < 256 && c == c) {
        r += s.rank[e];
        s.v[r + 1] = c;
        s.idx[r] = (uint8_t)e;
    }
    __syncthreads();
    if (once) {
        const float val = t < 256 ? s.v[t + 1] : 0.f;
        const uint8_t id = s.idx[e];
        const bool keep = t < n && (t == 0 || s.v[t] != val);
        const int kept = __syncthreads_count(keep);
        const uint64_t b = __ballot(keep);
        if ((t & 63) == 0 && t < 256) s.wsum[t >> 6] = __popcll(b);
        __syncthreads();
        int p = __popcll(b & ((1ull << (t & 63)) - 1ull));
        for (int w = 0; w < (e >> 6); ++w) p += s.wsum[w];
        if (keep) {
            s.v[p + 1] = val;
            s.idx[p] = id;
        }
        if (t >= kept && t < n) s.v[t + 1] = __builtin_nanf("");
        n = kept;
        __syncthreads();
    }
    return n;
}

// Code of the normalised weight x.
template <int kRule>
__device__ __forceinline__ uint32_t enc_code(const EncTable& s, float x, float lo, float scale, int last, bool none) {
    if (x != x) return kRule == kMidpoints ? (uint32_t)last : 0u;
    const uint32_t bk = s.bucket[enc_bucket(x, lo, scale)];
    int pos = (int)(bk & 0xffffu), left = (int)(bk >> 16);   // of the bucket's values, those below x
    // neighbours: sorted value pos - 1 <= x < value pos (NaN: there is none)
    float vl = s.v[pos], vu = s.v[pos + left + 1];
    while (left > 0) {
        const int half = (left + 1) >> 1;
        const float u = s.v[pos + half];
        const bool below = kRule == kMidpoints ? u < x : u <= x;
        pos = below ? pos + half : pos;
        left = below ? left - half : half - 1;
        vl = below ? u : vl;
        vu = below ? vu : u;
    }
    if constexpr (kRule == kMidpoints) return (uint32_t)pos;
    const float dl = x - vl, du = vu - x;
    const float d = fminf(dl, du);
    if (none || !(d < INFINITY)) return 0u;   // the scan's start value stands
    uint32_t best = 255u;
    if (dl == d) {
        int j = pos;
        do best = min(best, (uint32_t)s.idx[--j]);
        while (x - s.v[j] == d);
    }
    if (du == d) {
        int j = pos;
        do best = min(best, (uint32_t)s.idx[j++]);
        while (s.v[j + 1] - x == d);
    }
    return best;
}

// The scan: the first of the m entries at the least distance from x.
__device__ __forceinline__ uint32_t enc_scan(const EncTable& s, float x, int m) {
    float bd = fabsf(x - s.raw[0]);
    uint32_t best = 0;
#pragma unroll 8
    for (int c = 1; c < m; ++c) {
        const float dd = fabsf(x - s.raw[c]);
        if (dd < bd) {
            bd = dd;
            best = (uint32_t)c;
        }
    }
    return best;
}

// kVec: blocks of 8 * 2^i <= 512 weights, 8 weights (16-byte loads) a lane;
// else any block size, one wave per block.
template <int kRule, bool kBf16In, bool kVec>
__global__ __launch_bounds__(kEncThreads) void ref_encode_kernel(const void* __restrict__ w,
                                                                 const float* __restrict__ cb, int ncb, int64_t n,
                                                                 int block_size, int64_t nblocks,
                                                                 uint8_t* __restrict__ codes,
                                                                 uint16_t* __restrict__ absmax) {
    __shared__ __attribute__((aligned(16))) EncTable s;
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    // values searched: the entries, or the midpoints between them (a midpoint
    // counts as often as it is there; halving is exact)
    constexpr bool once = kRule != kMidpoints;
    const int m = once ? ncb : ncb - 1;
    auto value = [&](int i) __attribute__((always_inline)) { return once ? cb[i] : (cb[i] + cb[i + 1]) * 0.5f; };
    const float mine = t < m ? value(t) : __builtin_nanf("");
    const float prev = t > 0 && t < m ? value(t - 1) : -INFINITY;
    // strictly ascending without NaN (as trained codebooks are): each value is in place
    if (t < 256) {
        s.raw[t] = mine;
        s.v[t + 1] = mine;
        s.idx[t] = (uint8_t)t;
        const uint64_t up = __ballot(t >= m || prev <= mine);
        const uint64_t strict = __ballot(t == 0 || t >= m || prev < mine);
        if (lane == 0) s.wsum[wv] = (~up == 0) + 2 * (~strict == 0);
    } else if (t < 258) {
        s.v[257 * (t - 256)] = __builtin_nanf("");
    }
    __syncthreads();
    const int order = s.wsum[0] & s.wsum[1] & s.wsum[2] & s.wsum[3];
    const bool in_place = order == 3 || (!once && order == 1);
    if (!in_place) __syncthreads();   // (wsum is used again)
    const int nv = in_place ? m : enc_sort(s, order & 1, once);
    const float v1 = nv ? s.v[1] : 0.f, d = nv ? s.v[nv] - v1 : 0.f;
    const bool spread = d > 0.f && d < INFINITY;   // (equal values or an infinite end: one bucket)
    const float lo = spread ? v1 : 0.f, scale = spread ? (float)kEncBuckets / d : 0.f;
    const bool none = kRule != kMidpoints && (nv == 0 || s.raw[0] != s.raw[0]);   // entry 0 NaN: nothing is nearer
    {   // buckets 2 t and 2 t + 1: values below them and below the next one
        int pos[3] = {0, 0, 0};
#pragma unroll
        for (int step = 128; step >= 1; step >>= 1)
#pragma unroll
            for (int i = 0; i < 3; ++i)
                if (pos[i] + step <= nv && enc_bucket(s.v[pos[i] + step], lo, scale) < 2 * t + i) pos[i] += step;
        // past the last bucket with values: all (the search stops at 255)
        if (!spread) {
            pos[0] = t ? nv : 0;
            pos[1] = nv;
        }
        if (!spread || t == kEncThreads - 1) pos[2] = nv;
        *reinterpret_cast<u32x2_t*>(&s.bucket[2 * t]) =
            u32x2_t{(uint32_t)(pos[0] | (pos[1] - pos[0]) << 16), (uint32_t)(pos[1] | (pos[2] - pos[1]) << 16)};
    }
    // |x| <= 1, so equal rounded distances are at most 2^-23 (1 + |v|) apart.  Where
    // nine values lie (twice) that close, whole runs of them can be equally far
    if (t < 256) {
        const float u = s.v[t + 1];
        const uint64_t c = __ballot(t + 8 < nv && s.v[t + 9] - u <= 0x1p-22f * (1.0f + fabsf(u)));
        if (lane == 0) s.crowded[wv] = c != 0;
    }
    __syncthreads();
    const bool scan = once && (s.crowded[0] | s.crowded[1] | s.crowded[2] | s.crowded[3]);
    // the clamp's bound in the dtype the reference clamps in
    const float floor_v = kRule == kMidpoints ? 1e-12f
                          : kRule == kQuantizer && kBf16In ? bf16_to_f32(f32_to_bf16(1e-10f)) : 1e-10f;
    auto norm = [&](float wx, float mx) __attribute__((always_inline)) {
        const float x = wx / mx;
        return kRule == kQuantizer && kBf16In ? bf16_to_f32(f32_to_bf16(x)) : x;
    };
    auto code_of = [&](float wx, float mx) __attribute__((always_inline)) {
        return enc_code<kRule>(s, norm(wx, mx), lo, scale, ncb - 1, none);
    };
    if (kVec && !scan) {
        const int lpb = block_size >> 3;   // lanes per block
        for (int64_t i0 = ((int64_t)blockIdx.x * kEncThreads + t) * 8; i0 - 8 * lane < n;
             i0 += (int64_t)gridDim.x * kEncThreads * 8) {
            float x[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) x[j] = 0.f;
            if (i0 + 8 <= n) {
                if constexpr (kBf16In) {
                    const u32x4_t v = *reinterpret_cast<const u32x4_t*>((const uint16_t*)w + i0);
#pragma unroll
                    for (int j = 0; j < 8; ++j) x[j] = bf16_to_f32((v[j >> 1] >> (16 * (j & 1))) & 0xffffu);
                } else {
                    const f32x4_t a = *reinterpret_cast<const f32x4_t*>((const float*)w + i0);
                    const f32x4_t b = *reinterpret_cast<const f32x4_t*>((const float*)w + i0 + 4);
#pragma unroll
                    for (int j = 0; j < 8; ++j) x[j] = j < 4 ? a[j] : b[j - 4];
                }
            } else {
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    if (i0 + j < n)
                        x[j] = kBf16In ? bf16_to_f32(((const uint16_t*)w)[i0 + j]) : ((const float*)w)[i0 + j];
            }
            float mx = 0.f;
#pragma unroll
            for (int j = 0; j < 8; ++j) mx = fmaxf(mx, fabsf(x[j]));
            for (int off = lpb >> 1; off >= 1; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off, kWave));
            mx = fmaxf(mx, floor_v);
            uint32_t c[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) c[j] = code_of(x[j], mx);
            if (i0 + 8 <= n) {
                *reinterpret_cast<u32x2_t*>(codes + i0) = u32x2_t{c[0] | c[1] << 8 | c[2] << 16 | c[3] << 24,
                                                                  c[4] | c[5] << 8 | c[6] << 16 | c[7] << 24};
            } else {
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    if (i0 + j < n) codes[i0 + j] = (uint8_t)c[j];
            }
            if ((lane & (lpb - 1)) == 0 && i0 < n) absmax[i0 / block_size] = (uint16_t)f32_to_bf16(mx);
        }
    } else {
        auto load = [&](int64_t i) __attribute__((always_inline)) {
            return kBf16In ? bf16_to_f32(reinterpret_cast<const uint16_t*>(w)[i]) : reinterpret_cast<const float*>(w)[i];
        };
        for (int64_t b = (int64_t)blockIdx.x * (kEncThreads / 64) + wv; b < nblocks;
             b += (int64_t)gridDim.x * (kEncThreads / 64)) {
            const int64_t start = b * block_size;
            const int len = (int)min((int64_t)block_size, n - start);
            float mx = 0.f;
            for (int i = lane; i < len; i += 64) mx = fmaxf(mx, fabsf(load(start + i)));
            mx = fmaxf(wave_reduce_max(mx), floor_v);
            if (scan) {
                for (int i = lane; i < len; i += 64) codes[start + i] = (uint8_t)enc_scan(s, norm(load(start + i), mx), m);
            } else {
                for (int i = lane; i < len; i += 64) codes[start + i] = (uint8_t)code_of(load(start + i), mx);
            }
            if (lane == 0) absmax[b] = (uint16_t)f32_to_bf16(mx);
        }
    }
}

// 1-D Lloyd k-means (LUTQuantizer._train_kmeans iterations,
// vllm_lut/quantizer.py:158-173): every sample joins its nearest centroid by
// |x - c| (the first one on equal distances, as argmin), then every centroid
// with members becomes their mean (one without members keeps its value).
// The assignment runs one thread per sample with the k <= 256 centroids in
// LDS; the update one CTA per centroid, which sums its members in a fixed
// order (strided by thread, then a fixed tree), so results do not depend on
// scheduling.
__global__ __launch_bounds__(256) void kmeans1d_assign_kernel(const float* __restrict__ x, int64_t n,
                                                              const float* __restrict__ cent, int k,
                                                              int32_t* __restrict__ asg) {
    __shared__ float s_c[256];
    if ((int)threadIdx.x < k) s_c[threadIdx.x] = cent[threadIdx.x];
    __syncthreads();
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const float v = x[i];
    float bd = fabsf(v - s_c[0]);
    int bj = 0;
    for (int j = 1; j < k; ++j) {
        const float d = fabsf(v - s_c[j]);
        if (d < bd) {
            bd = d;
            bj = j;
        }
    }
    asg[i] = bj;
}

__global__ __launch_bounds__(256) void kmeans1d_update_kernel(const float* __restrict__ x, int64_t n,
                                                              const int32_t* __restrict__ asg,
                                                              float* __restrict__ cent) {
    __shared__ float s_sum[256];
    __shared__ int s_cnt[256];
    const int j = blockIdx.x, t = threadIdx.x;
    float sum = 0.f;
    int cnt = 0;
    for (int64_t i = t; i < n; i += 256) {
        if (asg[i] == j) {
            sum += x[i];
            ++cnt;
        }
    }
    s_sum[t] = sum;
    s_cnt[t] = cnt;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if (t < h) {
            s_sum[t] += s_sum[t + h];
            s_cnt[t] += s_cnt[t + h];
        }
        __syncthreads();
    }
    if (t == 0 && s_cnt[0] > 0) cent[j] = s_sum[0] / (float)s_cnt[0];
}

}  // namespace

namespace lutmoe_host {

int launch_bl4_encode(const float* w, int64_t nblocks, int n_iter, uint8_t* codes,
                      uint16_t* tables, hipStream_t s) {
    int64_t ctas = (nblocks + 3) / 4;
    if (ctas > 65536) ctas = 65536;
    hipLaunchKernelGGL(bl4_encode_kernel, dim3((unsigned)ctas), dim3(256), 0, s, w, nblocks,
                       n_iter, codes, tables);
    return check_launch();
}

int launch_kmeans_1d(const float* x, int64_t n, float* cent, int k, int n_iter, int32_t* asg, hipStream_t s) {
    const unsigned grid = (unsigned)((n + 255) / 256);
    for (int it = 0; it < n_iter; ++it) {
        hipLaunchKernelGGL(kmeans1d_assign_kernel, dim3(grid), dim3(256), 0, s, x, n, cent, k, asg);
        int rc = check_launch();
        if (rc) return rc;
        hipLaunchKernelGGL(kmeans1d_update_kernel, dim3((unsigned)k), dim3(256), 0, s, x, n, asg, cent);
        if ((rc = check_launch())) return rc;
    }
    return LUTMOE_OK;
}

// CTAs of the encoders: building the sorted table takes a CTA about as long
// as 8 thousand weights, so the grid is no more than two CTAs of 8 waves per
// CU, which loop.
template <int kRule, bool kBf16In>
static int ref_encode_launch(const void* w, const float* codebook, int ncb, int64_t n, int block_size, uint8_t* codes,
                             uint16_t* absmax, hipStream_t s) {
    const int64_t nblocks = (n + block_size - 1) / block_size;
    // 8 weights a lane: whole lanes, a power of two of them per block, and
    // aligned 16-byte (codes: 8-byte) accesses
    const bool vec = block_size >= 8 && block_size <= 512 && (block_size & (block_size - 1)) == 0 &&
                     (uintptr_t)w % 16 == 0 && (uintptr_t)codes % 8 == 0;
    const int64_t per = kEncThreads * 8;
    const int64_t want = vec ? (n + per - 1) / per : (nblocks + kEncThreads / 64 - 1) / (kEncThreads / 64);
    const dim3 grid((unsigned)(want < 512 ? want : 512)), block(kEncThreads);
    if (vec)
        hipLaunchKernelGGL((ref_encode_kernel<kRule, kBf16In, true>), grid, block, 0, s, w, codebook, ncb, n,
                           block_size, nblocks, codes, absmax);
    else
        hipLaunchKernelGGL((ref_encode_kernel<kRule, kBf16In, false>), grid, block, 0, s, w, codebook, ncb, n,
                           block_size, nblocks, codes, absmax);
    return check_launch();
}

int launch_ref_quantize(const void* w, bool bf16_in, const float* codebook, int ncb, int64_t n, int block_size,
                        int rule, uint8_t* codes, uint16_t* absmax, hipStream_t s) {
    if (rule == LUTMOE_QRULE_QUANTIZER)
        return bf16_in ? ref_encode_launch<kQuantizer, true>(w, codebook, ncb, n, block_size, codes, absmax, s)
                       : ref_encode_launch<kQuantizer, false>(w, codebook, ncb, n, block_size, codes, absmax, s);
    return bf16_in ? ref_encode_launch<kMidpoints, true>(w, codebook, ncb, n, block_size, codes, absmax, s)
                   : ref_encode_launch<kMidpoints, false>(w, codebook, ncb, n, block_size, codes, absmax, s);
}

int launch_ref_encode(const uint16_t* w, const float* codebook, int64_t n, int block_size, uint8_t* codes,
                      uint16_t* absmax, hipStream_t s) {
    return ref_encode_launch<kEncode, true>(w, codebook, 256, n, block_size, codes, absmax, s);
}

}  // namespace lutmoe_host
