// ts_gemv.h -- projections of one or two rows (decode of one or two sequences): every weight row's dot
// products with all of them on the vector units, in f32, with the weights in any stored form
// (f16 rows of one or two planes, GGUF blocks).
//
// The matrix-core slices pad a row or two to 32, write 32-row partials for every slice and need a
// second kernel to add them.  Here eight lanes own one weight row: a lane takes 32 of every 256
// k (a GGUF block, or the 16 bytes of a K super-block's qs), so a wave's loads are 128 contiguous
// bytes per row, and R rows per lane share the x values it reads from LDS.  The four waves of a
// workgroup take every fourth 256 k and their sums are added through LDS in wave order, so a
// result is complete in one kernel and deterministic.
//
// x is used as it is (f32, no hi/lo split); products with f16 weights and with the integer codes
// are fused multiply-adds into f32, block scales are applied to the sum over the block.  The codes
// of Q4_0 and Q5_0 are taken signed (n - 8, n - 16, exact): with n alone and 8 or 16 times the sum
// of x subtracted, the two cancel and leave 1.5 to 2.4 times the error of the matrix-core slices.
//
// One row of Q4_K: 3072 -> 5120 (QKV) 11.6 + 6.2 us (slices + sum and append) -> 7.3 + 3.5 (this +
// append), 3072 -> 3072 with the residual 8.8 + 3.2 -> 5.8; launch and the x -> LDS -> sum chain
// bound both (memory needs 2 us).  Whole layers (projections and attention, 1000 cached
// positions): one row 1.2 to 1.9 times as fast over all weight forms, two rows 1.0 to 1.5; with
// four rows the LDS reads of x cost what the matrix cores save (0.91 to 1.11), with eight 0.57 to
// 0.75, so the slices keep those (kGemvRows).
#pragma once
#include "ts_kquant.h"

namespace ts {
namespace {

constexpr int kGemvRows = 2;    // most rows of x
constexpr int kGemvF16 = 0, kGemvF16x2 = 1;  // T besides the GGUF types
constexpr int kGemvLds = 32768; // bytes of x in LDS at a time

// Bytes of 256 k of one weight row (of the hi plane for two planes).
template <int T>
__host__ __device__ constexpr int gemv_bytes() {
    return T == kGemvF16 || T == kGemvF16x2 ? 512 : kq_bytes(T);
}

// A lane's share of 256 k of a weight row, as loaded.
template <int T>
struct GemvRaw {
    static constexpr int NW = T == kGemvF16 ? 16 : T == kGemvF16x2 ? 32 : T == kGgmlQ4K ? 8 : T == kGgmlQ5K ? 12
                            : T == kGgmlQ8_0 ? 9 : T == kGgmlQ5_0 ? 6 : 5;
    uint32_t w[NW];
};

// k of the lane's e-th weight inside its 256 (p = lane % 8).
template <int T>
__device__ constexpr int gemv_k(int p, int e) {
    if (T == kGemvF16 || T == kGemvF16x2) return 64 * (e / 8) + 8 * p + e % 8;
    if (T == kGgmlQ4K || T == kGgmlQ5K) return 64 * (p / 2) + 16 * (p % 2) + 32 * (e / 16) + e % 16;
    return 32 * p + e;
}

template <int T>
__device__ __forceinline__ void gemv_load(GemvRaw<T> &r, const uint8_t *at, size_t plane, int p) {
    auto put16 = [&](int i, const uint8_t *src) {
        const uint4 v = *reinterpret_cast<const uint4 *>(src);
        r.w[i] = v.x;
        r.w[i + 1] = v.y;
        r.w[i + 2] = v.z;
        r.w[i + 3] = v.w;
    };
    if constexpr (T == kGemvF16 || T == kGemvF16x2) {
#pragma unroll
        for (int i = 0; i < 4; i++) put16(4 * i, at + 128 * i + 16 * p);
        if constexpr (T == kGemvF16x2) {
#pragma unroll
            for (int i = 0; i < 4; i++) put16(16 + 4 * i, at + plane + 128 * i + 16 * p);
        }
    } else if constexpr (T == kGgmlQ4K || T == kGgmlQ5K) {
        put16(0, at + KQ<T>::QS + 16 * p);
        put16(4, at);
        if constexpr (T == kGgmlQ5K) put16(8, at + 16 + 16 * (p & 1));
    } else {
        // the block's dwords from the 4-byte boundary at or before it (its start is 2 past one for
        // odd blocks); the last block's read ends with the 256 k
        constexpr int BB = T == kGgmlQ8_0 ? 34 : T == kGgmlQ5_0 ? 22 : 18;
        const uint32_t *src = reinterpret_cast<const uint32_t *>(at + ((BB * p) & ~3));
#pragma unroll
        for (int i = 0; i < GemvRaw<T>::NW; i++) r.w[i] = src[i];
    }
}

// The share's weights as f32 integers (the codes, signed except in the K formats), w[e] at k
// gemv_k(p, e), and the factors that make the sum over them a result: a0 times it; in the K formats,
// with s0, s1 the sums over elements 0-15 and 16-31 and t0, t1 the sums of x over the same,
// a0 s0 + a1 s1 + c0 t0 + c1 t1.
template <int T>
struct GemvWeights {
    float w[32];
    float a0, a1, c0, c1;
};

template <int T>
__device__ __forceinline__ void gemv_decode(GemvWeights<T> &g, const GemvRaw<T> &r, int p) {
    static_assert(T != kGemvF16 && T != kGemvF16x2, "f16 rows need no decoding");
    auto ub = [](uint32_t v, int b) { return (float)((v >> (8 * b)) & 0xFFu); };
    if constexpr (T == kGgmlQ4K || T == kGgmlQ5K) {
        const int j = p >> 1;  // chunk: sub-blocks 2j (low nibbles) and 2j + 1 (high)
        const KqScales s = kq_scales(make_uint4(r.w[4], r.w[5], r.w[6], r.w[7]));
        const uint32_t sc = (j < 2 ? s.sc03 : s.sc47) >> (16 * (j & 1)), m = (j < 2 ? s.m03 : s.m47) >> (16 * (j & 1));
        const float d = (float)__builtin_bit_cast(_Float16, (uint16_t)(r.w[4] & 0xFFFFu));
        const float dm = -(float)__builtin_bit_cast(_Float16, (uint16_t)(r.w[4] >> 16));
        g.a0 = d * ub(sc, 0);
        g.a1 = d * ub(sc, 1);
        g.c0 = dm * ub(m, 0);
        g.c1 = dm * ub(m, 1);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            uint32_t lo = r.w[i] & 0x0F0F0F0Fu, hi = (r.w[i] >> 4) & 0x0F0F0F0Fu;
            if constexpr (T == kGgmlQ5K) {
                const uint32_t h = r.w[8 + i] >> (2 * j);
                lo |= (h & 0x01010101u) << 4;
                hi |= (h & 0x02020202u) << 3;
            }
#pragma unroll
            for (int b = 0; b < 4; b++) {
                g.w[4 * i + b] = ub(lo, b);
                g.w[16 + 4 * i + b] = ub(hi, b);
            }
        }
    } else {
        const bool odd = p & 1;
        // dword i of the block's bytes from offset 2 (behind d); d
        auto word = [&](int i) {
            return odd ? r.w[i + 1] : __builtin_amdgcn_alignbyte(r.w[i + 1], r.w[i], 2);
        };
        const uint32_t dbits = odd ? r.w[0] >> 16 : r.w[0] & 0xFFFFu;
        const float d = (float)__builtin_bit_cast(_Float16, (uint16_t)dbits);
        g.a0 = d;
        if constexpr (T == kGgmlQ8_0) {
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const uint32_t v = word(i);
#pragma unroll
                for (int b = 0; b < 4; b++) g.w[4 * i + b] = (float)(int8_t)(v >> (8 * b));
            }
        } else {
            constexpr float mid = T == kGgmlQ5_0 ? 16.0f : 8.0f;
            const uint32_t qh = T == kGgmlQ5_0 ? word(0) : 0u;
            constexpr int first = T == kGgmlQ5_0 ? 1 : 0;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const uint32_t v = word(first + i);
                uint32_t lo = v & 0x0F0F0F0Fu, hi = (v >> 4) & 0x0F0F0F0Fu;
                if constexpr (T == kGgmlQ5_0) {
                    // bits 4i .. 4i + 3 (elements 4i ..) and 16 + 4i .. to bit 4 of every byte
                    lo |= ((((qh >> (4 * i)) & 0xFu) * 0x00204081u) & 0x01010101u) << 4;
                    hi |= ((((qh >> (16 + 4 * i)) & 0xFu) * 0x00204081u) & 0x01010101u) << 4;
                }
#pragma unroll
                for (int b = 0; b < 4; b++) {
                    g.w[4 * i + b] = ub(lo, b) - mid;
                    g.w[16 + 4 * i + b] = ub(hi, b) - mid;
                }
            }
        }
    }
}

// Sums of MB rows of x (row m at x + min(m, M - 1) * ld, K long) with the weight rows row[0 ..
// R - 1] of this lane's eight-lane group, by the 4 waves of a workgroup: on return the
// lanes with p == 0 of wave 0 hold out[r][m].  plane: bytes from a row's hi plane to its lo plane.
// sx: dynamic LDS of min(K, kGemvLds / (4 MB)) * MB floats; red: [4][8 R][MB] floats.
template <int T, int MB, int R>
__device__ __forceinline__ void gemv_rows(float *sx, float *red, const float *x, int M, size_t ld, int K,
                                          const uint8_t *const (&row)[R], size_t plane, int tid,
                                          float (&out)[R][MB]) {
    const int wave = tid >> 6, lane = tid & 63, p = lane & 7;
    const int nsb = K / 256;
    constexpr int kSeg = kGemvLds / (1024 * MB);  // 256s of x in LDS at a time
    float acc[R][MB];
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int m = 0; m < MB; m++) acc[r][m] = 0.0f;
    // a ring of D 256s per row in flight: usually all that a wave has to read
    constexpr int D = GemvRaw<T>::NW * R > 32 ? 1 : GemvRaw<T>::NW * R > 16 ? 2 : 4;
    GemvRaw<T> ring[D][R];
    auto load = [&](GemvRaw<T> (&g)[R], int sb) {
        if (sb >= nsb) return;  // uniform
#pragma unroll
        for (int r = 0; r < R; r++) gemv_load<T>(g[r], row[r] + (size_t)sb * gemv_bytes<T>(), plane, p);
    };
#pragma unroll
    for (int u = 0; u < D; u++) load(ring[u], wave + 4 * u);
    for (int s0 = 0; s0 < nsb; s0 += kSeg) {
        const int n = min(kSeg, nsb - s0), seg = 256 * n;
        if (s0) __syncthreads();
        for (int i = 4 * tid; i < MB * seg; i += 1024) {
            const int m = MB == 1 ? 0 : i / seg, k = i - m * seg;
            *reinterpret_cast<float4 *>(sx + i) =
                *reinterpret_cast<const float4 *>(x + (size_t)min(m, M - 1) * ld + 256 * s0 + k);
        }
        __syncthreads();
        // (a segment is a multiple of 4 D 256s, or the last one)
        auto step = [&](auto uc, int sb) {
            constexpr int u = decltype(uc)::value;
            GemvRaw<T> raw[R];
#pragma unroll
            for (int r = 0; r < R; r++) raw[r] = ring[u][r];
            load(ring[u], sb + 4 * D);
            const float *xb = sx + 256 * (sb - s0);
            if constexpr (T == kGemvF16 || T == kGemvF16x2) {
                // a sum of its own for every plane of the 256 (one chain through the whole reduction,
                // both planes in it, had 1.1 to 1.3 times the slices' error from 3072 k on)
                constexpr int planes = T == kGemvF16x2 ? 2 : 1;
#pragma unroll
                for (int m = 0; m < MB; m++) {
                    float s[R][planes];
#pragma unroll
                    for (int r = 0; r < R; r++)
#pragma unroll
                        for (int q = 0; q < planes; q++) s[r][q] = 0.0f;
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const float *xk = xb + m * seg + 64 * i + 8 * p;
                        const float4 u = *reinterpret_cast<const float4 *>(xk), v = *reinterpret_cast<const float4 *>(xk + 4);
                        const float xv[8] = {u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
#pragma unroll
                        for (int r = 0; r < R; r++)
#pragma unroll
                            for (int e = 0; e < 8; e++)
#pragma unroll
                                for (int q = 0; q < planes; q++) {
                                    const half2_t h = __builtin_bit_cast(half2_t, raw[r].w[16 * q + 4 * i + e / 2]);
                                    s[r][q] = __builtin_fmaf((float)h[e & 1], xv[e], s[r][q]);
                                }
                    }
#pragma unroll
                    for (int r = 0; r < R; r++) acc[r][m] = acc[r][m] + (planes == 2 ? s[r][1] + s[r][0] : s[r][0]);
                }
            } else {
                constexpr bool K = T == kGgmlQ4K || T == kGgmlQ5K;
                GemvWeights<T> g[R];
#pragma unroll
                for (int r = 0; r < R; r++) gemv_decode<T>(g[r], raw[r], p);
#pragma unroll
                for (int m = 0; m < MB; m++) {
                    // K formats: a sum per sub-block; the others: four chains of eight k (two of sixteen
                    // have a tenth more error)
                    constexpr int NS = K ? 2 : 4;
                    float s[R][NS];
                    float t[2] = {0.0f, 0.0f};
#pragma unroll
                    for (int r = 0; r < R; r++)
#pragma unroll
                        for (int c = 0; c < NS; c++) s[r][c] = 0.0f;
#pragma unroll
                    for (int i = 0; i < 8; i++) {
                        const float4 u = *reinterpret_cast<const float4 *>(xb + m * seg + gemv_k<T>(p, 4 * i));
                        const float xv[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
                        for (int r = 0; r < R; r++)
#pragma unroll
                            for (int e = 0; e < 4; e++) {
                                float &sum = s[r][K ? i >> 2 : e];
                                sum = __builtin_fmaf(g[r].w[4 * i + e], xv[e], sum);
                            }
                        if constexpr (K) t[i >> 2] = t[i >> 2] + ((u.x + u.y) + (u.z + u.w));
                    }
#pragma unroll
                    for (int r = 0; r < R; r++) {
                        if constexpr (K) {
                            const float v = __builtin_fmaf(g[r].a1, s[r][1], g[r].a0 * s[r][0]);
                            acc[r][m] = acc[r][m] + __builtin_fmaf(g[r].c1, t[1], __builtin_fmaf(g[r].c0, t[0], v));
                        } else {
                            acc[r][m] = __builtin_fmaf(g[r].a0, (s[r][0] + s[r][1]) + (s[r][NS - 2] + s[r][NS - 1]), acc[r][m]);
                        }
                    }
                }
            }
        };
        for (int sb = s0 + wave; sb < s0 + n; sb += 4 * D) {
            step(std::integral_constant<int, 0>{}, sb);
            if constexpr (D > 1) {
                if (sb + 4 < s0 + n) step(std::integral_constant<int, 1>{}, sb + 4);
            }
            if constexpr (D > 2) {
                if (sb + 8 < s0 + n) step(std::integral_constant<int, 2>{}, sb + 8);
                if (sb + 12 < s0 + n) step(std::integral_constant<int, 3>{}, sb + 12);
            }
        }
    }
    // the eight lanes of a row, then the waves in order
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int m = 0; m < MB; m++) {
            float v = acc[r][m];
            v += dpp_f<0xB1>(v);   // quad_perm(1,0,3,2)
            v += dpp_f<0x4E>(v);   // quad_perm(2,3,0,1)
            v += dpp_f<0x141>(v);  // row_half_mirror: the other four of the eight
            out[r][m] = v;
            if (p == 0) red[(wave * 8 * R + R * (lane >> 3) + r) * MB + m] = v;
        }
    __syncthreads();
    if (wave == 0 && p == 0) {
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
            for (int m = 0; m < MB; m++) {
                float v = out[r][m];
#pragma unroll
                for (int w = 1; w < 4; w++) v += red[(w * 8 * R + R * (lane >> 3) + r) * MB + m];
                out[r][m] = v;
            }
    }
}

// Rows of x that the kernel of M rows is built for (a dead row repeats the last one).
inline int gemv_mb(int M) { return M <= 1 ? 1 : 2; }
// Weight rows per lane: two share the x reads once there is more than one row of x.
__host__ __device__ constexpr int gemv_r(int mb) { return mb == 1 ? 1 : 2; }
// Whether M rows of K take these kernels for N weight rows of form t.  Two rows of more than 6144 pass
// LDS in pieces that the slices do without: in us, slices then these, 2 x 12288 -> 4096: Q4_K 19.4,
// 22.4, Q5_K 22.0, 24.1, f16 28.5, 30.7; 2 x 8192 -> 10240 in two planes 82, 102.  With 8192 weight
// rows to share x they win all the same (8192 -> 8192: Q4_K 22.9, 20.4, f16 36.6, 33.6), and always
// where the slices are bound by decoding (Q8_0, Q4_0, Q5_0: 0.35 to 0.97 of their time).
inline bool gemv_fits(int t, int M, int K, int N) {
    if (M > kGemvRows || K % 256 != 0) return false;
    if (M == 1 || K <= 6144) return true;
    return t == kGgmlQ8_0 || t == kGgmlQ4_0 || t == kGgmlQ5_0 || (t != kGemvF16x2 && N >= 8192);
}
inline size_t gemv_lds(int mb, int K) { return std::min<size_t>((size_t)mb * K * 4, kGemvLds); }

// f(integral_constant<int, T>, integral_constant<int, MB>) for f16 rows of 1 or 2 planes (type 0 or
// 1) or a GGUF type.
template <typename F>
void gemv_dispatch(int t, int mb, F f) {
    auto rows = [&](auto tc) {
        if (mb == 1)
            f(tc, std::integral_constant<int, 1>{});
        else
            f(tc, std::integral_constant<int, 2>{});
    };
    if (t == kGemvF16)
        rows(std::integral_constant<int, kGemvF16>{});
    else if (t == kGemvF16x2)
        rows(std::integral_constant<int, kGemvF16x2>{});
    else
        kq_dispatch(t, rows);
}

}  // namespace
}  // namespace ts
